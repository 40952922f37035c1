// Batched pipeline: the dense kernels (dense.inc), persistent over a device queue
// of paths, then the plain pipeline's unordered tile stage over the paths that no
// dense instance holds.  With the dense kernels off the call is the plain pipeline
// itself, whose sums follow emission order.  (A one-wave-per-path ordered kernel
// that took these paths before, flattening, counting, emitting and committing a
// path's increments on one wave, is slower at every size measured: 61 glyphs of
// 12-48 px 666 us against 300, 10,000 of them 1,621 against 880, 300 of 12-120 px
// 4,174 against 387, one of 250 px 7,373 against 276.)
//
// Also here: the coverage adjoint (adjoint.inc, adjoint_large.inc), the single
// fill (single.inc) and the allocation-free dense chain.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "device_common.hpp"
#include "pipeline.hpp"
#include "raster_common.hpp"
#include "scan.hpp"

namespace ochre {

constexpr int F_LCAP = 8192;   // lines per path
constexpr int F_GRID = 32;     // tile grid side (256 px)
constexpr int F_TSTRIDE = 65;  // accumulator stride per tile (bank spread)
constexpr size_t F_SCRATCH = (size_t)F_LCAP * 32;  // per wave of the adjoint: its path's lines and their gradients
constexpr uint32_t F_INVALID = 0xffffffffu;

struct FusedIn {
    int64_t n_paths;
    const uint8_t* verbs;
    const int64_t* verb_off;
    const float* points;
    const int64_t* point_off;
    const float* weights;
    const int64_t* weight_off;
    const Xform* xf;
    int64_t n_points, n_weights;
    // when set, the queue runs over ids[0 .. *n_ids) (paths handed on by
    // k_dense) instead of 0 .. n_paths
    const uint32_t* ids = nullptr;
    const uint32_t* n_ids = nullptr;
    int64_t item_cap = F_LCAP;  // lines per chunk of commands over which a dense instance hands a path on
};

struct FusedOut {
    int16_t* tile_xy;
    uint8_t* tile_alpha;
    float* tile_cov;  // optional: pre-quantisation coverage min(|accum + area|, 1), 64 per tile
    int64_t tile_cap;
    int16_t* span_xy;
    uint16_t* span_w;
    int64_t span_cap;
    int64_t* pts;
    int32_t* ptc;
    int64_t* pss;
    int32_t* psc;
};

struct FusedCtl {
    uint32_t queue;     // path queue of the first kernel of the launch
    uint32_t deferred;  // paths over the kernel's limits (the adjoint, the single fill)
    uint32_t error;
    uint32_t dq;        // paths handed on by k_dense
    unsigned long long tiles;
    unsigned long long spans;
    uint32_t queue3;    // queue of the large-grid dense kernel
    uint32_t dq2;       // paths handed on by the second dense instance
    uint32_t queue4;    // queue of the third dense instance
    uint32_t dq3;       // paths handed on by the third dense instance
    uint32_t pad[52];
};

__global__ void k_fused_reset(FusedCtl* c) {
    if (threadIdx.x == 0) {
        c->queue = 0;
        c->deferred = 0;
        c->error = 0;
        c->dq = 0;
        c->tiles = 0;
        c->spans = 0;
        c->queue3 = 0;
        c->dq2 = 0;
        c->queue4 = 0;
        c->dq3 = 0;
    }
}

struct OpMax64 {
    __device__ int64_t operator()(int64_t a, int64_t b) const { return a > b ? a : b; }
};

__device__ inline V2 fload(const FusedIn& in, int64_t g, const Xform& X) {
    return apply(X, mk(in.points[2 * g], in.points[2 * g + 1]));
}

template <int TC>
struct LdsState {
    uint32_t occ[F_GRID];
    uint32_t row_rank[F_GRID + 1];
    struct {  // lines queued for a walk of the adjoint
        float4 line[2 * WAVE];
        uint16_t id[2 * WAVE];
    } q;
    // tsign is dead once spans are written; the accumulators live after that
    union {
        int32_t tsign[F_GRID * F_GRID];
        struct {
            float acc_a[TC * F_TSTRIDE];
            float acc_h[TC * F_TSTRIDE];
        } a;
        struct {  // fixed-point area / height sums of half a chunk (the coverage adjoint)
            unsigned long long fa[TC / 2 * 64];
            unsigned long long fh[TC / 2 * 64];
        } x;
    } u;
};

// Rank of tile (tx, ty) (grid-local) among the path's occupied tiles in
// row-major order.
template <class S>
__device__ inline uint32_t tile_rank(const S& s, int tx, int ty) {
    return s.row_rank[ty] + (uint32_t)__popc(s.occ[ty] & ((1u << tx) - 1u));
}

// Adjoint inputs/outputs (see adjoint.inc).  The target of path p is its
// tiles [tt_start[p], +tt_count[p]) (row-major, 64 f32 coverages each) and
// spans [ts_start[p], +ts_count[p]).
struct AdjArgs {
    const int64_t* tt_start;
    const int32_t* tt_count;
    const int16_t* t_xy;
    const float* t_cov;
    const int64_t* ts_start;
    const int32_t* ts_count;
    const int16_t* ts_xy;
    const uint16_t* ts_w;
    float* loss;      // [n_paths]
    float* d_points;  // [n_points * 2]
    float* d_xf;      // [n_paths * 6]
};

constexpr int A_TCAP = 256;   // tiles per path
constexpr int A_VCAP = 1024;  // commands per path
constexpr int A_PCAP = 4096;  // points per path
constexpr int A_SCAP = 1024;  // spans per path
constexpr size_t A_OFF_TILES = 0;                                            // float[A_TCAP][128]: g, G
constexpr size_t A_OFF_CMD = A_OFF_TILES + (size_t)A_TCAP * 128 * 4;         // float[A_VCAP][12]
constexpr size_t A_OFF_CMDOFF = A_OFF_CMD + (size_t)A_VCAP * 12 * 4;         // uint32[A_VCAP + 1]
constexpr size_t A_OFF_PCMD = A_OFF_CMDOFF + (size_t)(A_VCAP + 4) * 4;       // uint32[A_PCAP]
constexpr size_t A_OFF_SPANS = A_OFF_PCMD + (size_t)A_PCAP * 4;              // uint32[A_SCAP][2]
constexpr size_t A_OFF_L64 = (A_OFF_SPANS + (size_t)A_SCAP * 8 + 255) & ~(size_t)255;  // double2[F_LCAP][2]
constexpr size_t A_SCRATCH = A_OFF_L64 + (size_t)F_LCAP * 32;

template <int TC>
__device__ void adjoint_backward(const FusedIn& in, const AdjArgs& adj, FusedCtl* ctl, uint8_t* sc, uint8_t* asc,
                                 LdsState<TC>& s, int64_t p, uint32_t L, uint32_t NT, uint32_t NS, int32_t tx0,
                                 int32_t ty0, int32_t GW, int32_t GH);

// The adjoint evaluates its forward in path-local device coordinates: the
// transform's offset less a tile-aligned origin (the first point's tile), so
// that f32 coordinates stay small.  At 1000 px an f32 coordinate carries
// ~6e-5 px of rounding, enough to move a pixel's |v| across the clamp at 1
// relative to the exact coverage; local coordinates cut that tenfold.  A
// whole-tile shift leaves the pixel and tile grid unchanged, and the
// derivatives with respect to the offset are those of the original one.
// (ox, oy) is the origin in tiles.
__device__ inline Xform adjoint_local_xform(const FusedIn& in, int64_t p, int32_t* ox, int32_t* oy) {
    Xform X = in.xf[p];
    *ox = *oy = 0;
    const int64_t pb = in.point_off[p];
    if (in.point_off[p + 1] > pb) {
        const V2 w = apply(X, mk(in.points[2 * pb], in.points[2 * pb + 1]));
        if (fabsf(w.x) < 1.0e6f && fabsf(w.y) < 1.0e6f) {
            *ox = (int32_t)floorf(w.x * 0.125f);
            *oy = (int32_t)floorf(w.y * 0.125f);
            X.ox -= (float)(*ox * TILE);
            X.oy -= (float)(*oy * TILE);
        }
    }
    return X;
}

// One path of the adjoint, on one wave: its lines (to the wave's scratch), its
// occupied tiles and spans as the f32 forward has them, then adjoint_backward.
template <int TC>
__device__ void adjoint_path(const FusedIn& in, FusedCtl* ctl, uint32_t* deferred, uint8_t* sc, LdsState<TC>& s,
                             int64_t p, const AdjArgs& adj, uint8_t* asc) {
    const int lane = threadIdx.x;
    float4* lines = reinterpret_cast<float4*>(sc);

    const int64_t vb = in.verb_off[p], ve = in.verb_off[p + 1];
    const int64_t pb = in.point_off[p], pe = in.point_off[p + 1];
    const int64_t wb = in.weight_off[p], we = in.weight_off[p + 1];
    if (ve - vb > A_VCAP || pe - pb > A_PCAP) {  // over one wave's limits whatever its lines are
        if (lane == 0) deferred[atomicAdd(&ctl->deferred, 1u)] = (uint32_t)p;  // (the adjoint's large path)
        return;
    }
    int32_t aox = 0, aoy = 0;
    const Xform X = adjoint_local_xform(in, p, &aox, &aoy);

    // ---------------------------------------------------------- flatten
    uint32_t L = 0;
    uint32_t cpts = 0, ccon = 0;
    int64_t cmove = -1;
    bool overflow = false;
    bool bad = false, flat_bad = false;
    BoxAcc box;
    bool any_line = false;
    for (int64_t cb = vb; cb < ve; cb += WAVE) {
        const int64_t i = cb + lane;
        const bool valid = i < ve;
        int verb = valid ? in.verbs[i] : (int)CLOSE;
        int np = verb_points(verb);
        bool lane_bad = valid && np < 0;
        if (np < 0) np = 0;
        const uint32_t np_incl = wave_incl_scan((uint32_t)np, OpAdd());
        const uint32_t cc = (valid && verb == CONIC) ? 1u : 0u;
        const uint32_t cc_incl = wave_incl_scan(cc, OpAdd());
        const int64_t g = pb + cpts + (np_incl - (uint32_t)np);
        const int64_t mv = (valid && verb == MOVE) ? g : (int64_t)-1;
        const int64_t mv_incl = wave_incl_scan(mv, OpMax64());
        int64_t mv_excl = shfl_up_any(mv_incl, 1);
        if (lane == 0) mv_excl = -1;
        mv_excl = mv_excl > cmove ? mv_excl : cmove;
        Cmd c;
        c.verb = verb;
        c.path = (int32_t)p;
        c.last_in_path = (i == ve - 1);
        c.bad = false;
        if (valid && g + np > pe) lane_bad = true;
        if (valid && !lane_bad) {
            // static indices keep the command in registers
            if (np > 0) c.pt[0] = fload(in, g, X);
            if (np > 1) c.pt[1] = fload(in, g + 1, X);
            if (np > 2) c.pt[2] = fload(in, g + 2, X);
            c.w = 0.0f;
            if (verb == CONIC) {
                int64_t wi = wb + ccon + (cc_incl - 1);
                if (wi < we) c.w = in.weights[wi];
                else lane_bad = true;
            }
            c.start = g > pb ? fload(in, g - 1, X) : mk(0.0f, 0.0f);
            c.first = mv_excl >= 0 ? fload(in, mv_excl, X) : mk(0.0f, 0.0f);
        }
        // A certain overflow of the line list, from the curves' steps alone
        // (t advances by at most dt + 1e-7 per step of the flatten loop): the
        // path is handed on before any of its curves is evaluated here.
        uint32_t lower = 0;
        if (valid && !lane_bad && (verb == QUAD || verb == CUBIC)) {
            const float dt = verb == QUAD ? quad_dt(c.start, c.pt[0], c.pt[1])
                                          : cubic_dt(c.start, c.pt[0], c.pt[1], c.pt[2]);
            const float est = 0.99f / (dt + 1e-7f);
            if (est > 0.0f) lower = est >= (float)F_LCAP ? (uint32_t)F_LCAP + 1u : (uint32_t)est;
        }
        const uint32_t lower_tot = __shfl(wave_incl_scan(lower, OpAdd()), WAVE - 1, WAVE);
        if (L + lower_tot > (uint32_t)F_LCAP) {
            if (lane == 0) deferred[atomicAdd(&ctl->deferred, 1u)] = (uint32_t)p;  // (the adjoint's large path)
            return;
        }
        uint32_t n = 0;
        if (valid && !lane_bad) {
            bool ok = command_lines(c, [&](V2 a, V2 b) {
                n++;
                box.add(a);
                box.add(b);
            });
            if (!ok) flat_bad = true;
        }
        if (n) any_line = true;
        const uint32_t n_incl = wave_incl_scan(n, OpAdd());
        const uint32_t chunk_total = __shfl(n_incl, WAVE - 1, WAVE);
        if (__ballot(lane_bad)) bad = true;
        if (!overflow && L + chunk_total > (uint32_t)F_LCAP) overflow = true;
        if (!overflow && valid && !lane_bad && n) {
            uint32_t o = L + n_incl - n;
            command_lines(c, [&](V2 a, V2 b) { lines[o++] = make_float4(a.x, a.y, b.x, b.y); });
        }
        if (valid && i - vb < A_VCAP) {
            reinterpret_cast<uint32_t*>(asc + A_OFF_CMDOFF)[i - vb] = L + n_incl - n;
            if (i == ve - 1) reinterpret_cast<uint32_t*>(asc + A_OFF_CMDOFF)[i - vb + 1] = L + n_incl;
            for (int k = 0; k < np; k++)
                if (g - pb + k < A_PCAP) reinterpret_cast<uint32_t*>(asc + A_OFF_PCMD)[g - pb + k] = (uint32_t)(i - vb);
        }
        L += chunk_total;
        cpts += __shfl(np_incl, WAVE - 1, WAVE);
        ccon += __shfl(cc_incl, WAVE - 1, WAVE);
        const int64_t last_mv = shfl_any(mv_incl, WAVE - 1);
        cmove = last_mv > cmove ? last_mv : cmove;
    }
    if (bad || (cpts != (uint32_t)(pe - pb))) {
        if (lane == 0) atomicOr(&ctl->error, (uint32_t)ERR_INPUT);
        return;
    }
    if (__ballot(flat_bad)) {
        if (lane == 0) atomicOr(&ctl->error, (uint32_t)ERR_FLATTEN);
        return;
    }
    // path bounding box of all line end points
    const bool has_lines = __ballot(any_line) != 0;
    const bool full = __ballot(box.full) != 0;
    float bminx = box.minx, bminy = box.miny, bmaxx = box.maxx, bmaxy = box.maxy;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        bminx = fminf(bminx, __shfl_xor(bminx, d, WAVE));
        bminy = fminf(bminy, __shfl_xor(bminy, d, WAVE));
        bmaxx = fmaxf(bmaxx, __shfl_xor(bmaxx, d, WAVE));
        bmaxy = fmaxf(bmaxy, __shfl_xor(bmaxy, d, WAVE));
    }
    int32_t tx0 = 0, ty0 = 0, GW = 0, GH = 0;
    if (has_lines && !full && bminx <= bmaxx)
        grid_from_box(true, false, (int32_t)floorf(bminx), (int32_t)floorf(bminy), (int32_t)floorf(bmaxx),
                      (int32_t)floorf(bmaxy), &tx0, &ty0, &GW, &GH);
    if (overflow || full || GW > F_GRID || GH > F_GRID) {
        if (lane == 0) deferred[atomicAdd(&ctl->deferred, 1u)] = (uint32_t)p;  // (the adjoint's large path)
        return;
    }

    // ------------------------------------------------------- count walk
    for (int k = lane; k < F_GRID * F_GRID; k += WAVE) s.u.tsign[k] = 0;
    if (lane < F_GRID) s.occ[lane] = 0;
    __syncthreads();
    bool bbox_err = false, walk_err = false;
    {
        // a lane per line at tile granularity (line_tiles: the tiles, tile-row
        // crossings and increments from the DDA's two crossing-parameter
        // chains); a line it does not cover is walked pixel by pixel
        auto mark = [&](int32_t tx, int32_t ty) {
            const int lx = tx - tx0, ly = ty - ty0;
            if ((unsigned)lx < (unsigned)GW && (unsigned)ly < (unsigned)GH) atomicOr(&s.occ[ly], 1u << lx);
            else bbox_err = true;
        };
        auto cross = [&](int32_t tx, int32_t ty, int sign) {
            const int lx = tx - tx0, ly = ty - ty0;
            if ((unsigned)lx < (unsigned)GW && (unsigned)ly < (unsigned)GH) atomicAdd(&s.u.tsign[ly * F_GRID + lx], sign);
            else bbox_err = true;
        };
        for (uint32_t line = (uint32_t)lane; line < L; line += WAVE) {
            const float4 ln = lines[line];
            const V2 a = mk(ln.x, ln.y), point = mk(ln.z, ln.w);
            if (line_tiles(a, point, mark, cross)) continue;
            if (veq(point, a)) continue;  // rasterizer.rs:73
            Dda d;
            dda_init(d, a, point);
            int16_t ty_prev = div8(d.y), cur_tx = div8(d.x), cur_ty = ty_prev;
            mark(cur_tx, cur_ty);
            for (uint32_t steps = 0;;) {
                bool term = dda_step(d);
                if (term) {  // rasterizer.rs:118-121
                    d.x = f2i16(floorf(point.x));
                    d.y = f2i16(floorf(point.y));
                }
                const int16_t ty = div8(d.y);
                if (ty != ty_prev) {  // rasterizer.rs:123-131
                    cross(div8(d.x), ty_prev < ty ? ty_prev : ty, (int)(int8_t)(int16_t)(ty - ty_prev));
                    ty_prev = ty;
                }
                if (!term && ++steps >= WALK_LIMIT) {
                    walk_err = true;
                    term = true;
                }
                if (term) break;
                const int16_t tx = div8(d.x);
                if (tx != cur_tx || ty != cur_ty) {
                    cur_tx = tx;
                    cur_ty = ty;
                    mark(tx, ty);
                }
            }
        }
    }
    __syncthreads();
    if (__ballot(bbox_err) || __ballot(walk_err)) {
        if (lane == 0) atomicOr(&ctl->error, __ballot(bbox_err) ? (uint32_t)ERR_BBOX : (uint32_t)ERR_FLATTEN);
        return;
    }

    // --------------------------------------------- tiles, spans, output
    // lane = tile row
    const bool row_lane = lane < GH;
    const uint32_t row_tiles = row_lane ? (uint32_t)__popc(s.occ[lane]) : 0u;
    const uint32_t rt_incl = wave_incl_scan(row_tiles, OpAdd());
    if (row_lane) s.row_rank[lane] = rt_incl - row_tiles;
    const uint32_t NT = __shfl(rt_incl, WAVE - 1, WAVE);
    int32_t row_sum = 0;
    if (row_lane)
        for (int x = 0; x < GW; x++) row_sum += s.u.tsign[lane * F_GRID + x];
    const int32_t rs_incl = wave_incl_scan(row_sum, OpAdd());
    const int32_t w_before = rs_incl - row_sum;  // winding of all crossings in earlier rows
    // spans (rasterizer.rs:252-264): between consecutive tiles of a row
    uint32_t row_spans = 0;
    if (row_lane) {
        int32_t wnd = w_before, w_prev = 0, prev = -1;
        const uint32_t o = s.occ[lane];
        for (int x = 0; x < GW; x++) {
            wnd += s.u.tsign[lane * F_GRID + x];
            if ((o >> x) & 1u) {
                if (prev >= 0 && x > prev + 1 && w_prev != 0) row_spans++;
                prev = x;
                w_prev = wnd;
            }
        }
    }
    const uint32_t rsp_incl = wave_incl_scan(row_spans, OpAdd());
    const uint32_t NS = __shfl(rsp_incl, WAVE - 1, WAVE);
    if (NT > (uint32_t)A_TCAP || NS > (uint32_t)A_SCAP) {
        if (lane == 0) deferred[atomicAdd(&ctl->deferred, 1u)] = (uint32_t)p;  // the large path
        return;
    }
    if (row_lane && row_spans) {
        uint32_t si = rsp_incl - row_spans;
        int32_t wnd = w_before, w_prev = 0, prev = -1;
        const uint32_t o = s.occ[lane];
        uint32_t* sp = reinterpret_cast<uint32_t*>(asc + A_OFF_SPANS);
        for (int x = 0; x < GW; x++) {
            wnd += s.u.tsign[lane * F_GRID + x];
            if ((o >> x) & 1u) {
                if (prev >= 0 && x > prev + 1 && w_prev != 0) {
                    sp[2 * si] = (uint32_t)lane;                                  // grid row
                    sp[2 * si + 1] = (uint32_t)(prev + 1) | ((uint32_t)x << 16);  // tile columns [a, b)
                    si++;
                }
                prev = x;
                w_prev = wnd;
            }
        }
    }
    // (the adjoint takes its coverage from the f64 geometry: emitting and
    // committing the f32 increments in front of it was half of its walks,
    // 1,447 -> 1,137 us on 4,096 paths of 16 cubics)
    adjoint_backward<TC>(in, adj, ctl, sc, asc, s, p, L, NT, NS, tx0, ty0, GW, GH);
}

#include "adjoint.inc"
#include "adjoint_large.inc"
#include "dense.inc"
#include "single.inc"

// ---------------------------------------------- deferred paths -> plain

// Gathers the deferred paths into a compact segment input, gridDim.y workgroups
// to a path (one per path left 24 paths of 60,000 points to 24 of the CUs: 122 ->
// 7 us).
__global__ void k_gather_paths(FusedIn in, const uint32_t* ids, uint32_t n, const int64_t* dst_voff,
                               const int64_t* dst_poff, const int64_t* dst_woff, uint8_t* verbs, float* points,
                               float* weights, Xform* xf) {
    for (uint32_t k = blockIdx.x; k < n; k += gridDim.x) {
        const int64_t p = ids[k];
        const int64_t vb = in.verb_off[p], nv = in.verb_off[p + 1] - vb;
        const int64_t pb = in.point_off[p], np = in.point_off[p + 1] - pb;
        const int64_t wb = in.weight_off[p], nw = in.weight_off[p + 1] - wb;
        const int64_t i0 = (int64_t)blockIdx.y * blockDim.x + threadIdx.x, st = (int64_t)gridDim.y * blockDim.x;
        for (int64_t i = i0; i < nv; i += st) verbs[dst_voff[k] + i] = in.verbs[vb + i];
        for (int64_t i = i0; i < 2 * np; i += st) points[2 * dst_poff[k] + i] = in.points[2 * pb + i];
        for (int64_t i = i0; i < nw; i += st) weights[dst_woff[k] + i] = in.weights[wb + i];
        if (i0 == 0) xf[k] = in.xf[p];
    }
}

__global__ void k_scatter_ranges(const uint32_t* ids, uint32_t n, const int64_t* ts, const int32_t* tc,
                                 const int64_t* ss, const int32_t* scn, int64_t tbase, int64_t sbase, int64_t* pts,
                                 int32_t* ptc, int64_t* pss, int32_t* psc) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t p = ids[k];
    pts[p] = ts[k] + tbase;
    ptc[p] = tc[k];
    pss[p] = ss[k] + sbase;
    psc[p] = scn[k];
}

struct BatchedState {
    DBuf scratch, ascratch, ctl, deferred, dense_ids, dense_ids2, dense_ids3, d_sizes, d_pack;
    DBuf adj_bin, adj_ids;       // the adjoint's path order
    DBuf large_cmd, large_grid;  // the large-path adjoint's scratch
    DBuf g_verbs, g_points, g_weights, g_xf, g_ts, g_tc, g_ss, g_sc;
    // graph of (reset, dense kernels) for the last argument set
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<uint8_t> graph_key, last_key;
    ~BatchedState() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};

// The plain pipeline in passes of bounded scratch: a call that took the batched
// pipeline's fixed scratch before must not need the plain one's tens of gigabytes
// for a large batch.  About 0.8 GB at the first limits, 0.1 GB at the second,
// which a pass falls back to when memory is short; a single path over them still
// gets the context's own limits.
static int run_plain_bounded(Context* ctx, const SegInput& in, OutputDesc& out, hipStream_t s) {
    const OutputDesc asked = out;
    SegInput si = in;
    si.own_ranges = true;
    int st = run_plain(ctx, si, out, s, false, (int64_t)1 << 23, (int64_t)1 << 24);
    if (st == -2) {
        (void)hipGetLastError();
        out = asked;
        st = run_plain(ctx, si, out, s, false, (int64_t)1 << 20, (int64_t)1 << 21);
    }
    return st;
}

// The handed-on paths' command, point and weight counts.
struct DeferSize {
    int64_t path, nv, np, nw;
};
__global__ void k_defer_sizes(FusedIn in, const uint32_t* ids, uint32_t n, DeferSize* out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int64_t p = ids[k];
    out[k] = DeferSize{p, in.verb_off[p + 1] - in.verb_off[p], in.point_off[p + 1] - in.point_off[p],
                       in.weight_off[p + 1] - in.weight_off[p]};
}

static bool few_paths(const Context* ctx, int64_t n_paths, int cus) { return ctx->dense_large && n_paths <= cus; }

bool few_paths_route(const Context* ctx, int64_t n_paths) {
    int cus = 0;
    return ctx->dense && n_paths > 0 &&
           hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) == hipSuccess &&
           few_paths(ctx, n_paths, cus);
}

int run_batched(Context* ctx, const SegInput& in, OutputDesc& out, hipStream_t s, bool use_graph) {
    if (!ctx->batched) ctx->batched = new BatchedState();
    BatchedState* B = reinterpret_cast<BatchedState*>(ctx->batched);
    const int64_t NP = in.n_paths;
    out.n_tiles = out.n_spans = 0;
    if (NP <= 0) return 0;
    if (!ctx->dense) return run_plain_bounded(ctx, in, out, s);
    int dev = 0;
    HIPCHK_RET(hipGetDevice(&dev));
    int cus = 0;
    HIPCHK_RET(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHK_RET(B->ctl.ensure(sizeof(FusedCtl)));
    if (!ctx->host_pinned) HIPCHK_RET(hipHostMalloc(&ctx->host_pinned, 4096));
    FusedIn fi;
    fi.n_paths = NP;
    fi.verbs = in.verbs;
    fi.verb_off = in.seg_verb_off;
    fi.points = in.points;
    fi.point_off = in.seg_point_off;
    fi.weights = in.weights;
    fi.weight_off = in.seg_weight_off;
    fi.xf = in.seg_xf;
    fi.n_points = in.n_points;
    fi.n_weights = in.n_weights;
    FusedOut fo;
    fo.tile_xy = out.tile_xy;
    fo.tile_alpha = out.tile_alpha;
    fo.tile_cov = out.tile_cov;
    fo.tile_cap = out.tile_capacity;
    fo.span_xy = out.span_xy;
    fo.span_w = out.span_w;
    fo.span_cap = out.span_capacity;
    fo.pts = out.path_tile_start;
    fo.ptc = out.path_tile_count;
    fo.pss = out.path_span_start;
    fo.psc = out.path_span_count;
    FusedCtl* ctl = B->ctl.as<FusedCtl>();
    const int dnw = ctx->dense_waves == 2 ? 2 : (ctx->dense_waves == 8 ? 8 : 4);
    const int n_groups = std::max(1, cus * std::max(1, ctx->dense_groups_per_cu));
    const int n_small = cus * std::max(0, ctx->dense_small_groups);
    const int n_large = ctx->dense_large ? cus : 0;
    // The dense instances run one after another, each over the paths the one
    // before handed on: [small grids, 32 tiles] -> 64 tiles -> [256 tiles], or the
    // 256-tile one alone over few paths; what is
    // left goes to the plain pipeline.
    enum { D_SMALL, D_MAIN, D_LARGE, D_FEW };
    int stages[3], n_stages = 0;
    // With a CU for every path, each gets 16 waves of the 256-tile instance and one
    // launch: a path's latency is all there is (61 glyphs of 12-48 px 81 -> 68 us a
    // call, 256 of them 91 -> 71, 61 of 60-120 px 264 -> 238; at 512 paths, two to a
    // CU one after the other, 95 -> 108).
    // Its chunks are of 1,024 commands, four of the 64-tile instance's, and hold four
    // times the lines (200 paths of 1,000 cubics and 20,000 lines in 36 tiles: 279 us
    // a call, handed on for their 8,192 lines a chunk 602; one of them 262 / 346).
    if (few_paths(ctx, NP, cus)) {
        stages[n_stages++] = D_FEW;
    } else {
        if (n_small) stages[n_stages++] = D_SMALL;
        stages[n_stages++] = D_MAIN;
        if (n_large) stages[n_stages++] = D_LARGE;
    }
    HIPCHK_RET(B->dense_ids.ensure((size_t)NP * 4));
    if (n_stages > 1) HIPCHK_RET(B->dense_ids2.ensure((size_t)NP * 4));
    if (n_stages > 2) HIPCHK_RET(B->dense_ids3.ensure((size_t)NP * 4));
    uint32_t* lists[3] = {B->dense_ids.as<uint32_t>(), B->dense_ids2.as<uint32_t>(), B->dense_ids3.as<uint32_t>()};
    uint32_t* counts[3] = {&ctl->dq, &ctl->dq2, &ctl->dq3};
    uint32_t* queues[3] = {&ctl->queue, &ctl->queue3, &ctl->queue4};
    FusedIn fin[3] = {fi, fi, fi};  // stage i reads fin[i]
    if (stages[0] == D_FEW) fin[0].item_cap = 4 * (int64_t)F_LCAP;
    for (int i = 1; i < n_stages; i++) {
        fin[i].ids = lists[i - 1];
        fin[i].n_ids = counts[i - 1];
    }
    uint32_t* deferred = lists[n_stages - 1];
    const bool timing = ctx->timing;
    if (timing) {
        for (auto& e : ctx->ev)
            if (!e) HIPCHK_RET(hipEventCreate(&e));
    }
    // timing without a graph brackets the dense kernels with events
    auto enqueue = [&](hipStream_t st, bool ev) {
        hipLaunchKernelGGL(k_fused_reset, dim3(1), dim3(64), 0, st, ctl);
        if (ev) (void)hipEventRecord(ctx->ev[0], st);
        for (int i = 0; i < n_stages; i++) {
            const FusedIn& f = fin[i];
            if (stages[i] == D_FEW)
                hipLaunchKernelGGL((k_dense<16, 256>), dim3((unsigned)NP), dim3(16 * WAVE), 0, st, f, fo, ctl,
                                   queues[i], lists[i], counts[i]);
            else if (stages[i] == D_SMALL)
                hipLaunchKernelGGL((k_dense<2, 32>), dim3(n_small), dim3(2 * WAVE), 0, st, f, fo, ctl, queues[i],
                                   lists[i], counts[i]);
            else if (stages[i] == D_LARGE)
                hipLaunchKernelGGL((k_dense<8, 256>), dim3(n_large), dim3(8 * WAVE), 0, st, f, fo, ctl, queues[i],
                                   lists[i], counts[i]);
            else if (dnw == 2)
                hipLaunchKernelGGL((k_dense<2, 64>), dim3(n_groups), dim3(2 * WAVE), 0, st, f, fo, ctl, queues[i],
                                   lists[i], counts[i]);
            else if (dnw == 8)
                hipLaunchKernelGGL((k_dense<8, 64>), dim3(n_groups), dim3(8 * WAVE), 0, st, f, fo, ctl, queues[i],
                                   lists[i], counts[i]);
            else
                hipLaunchKernelGGL((k_dense<4, 64>), dim3(n_groups), dim3(4 * WAVE), 0, st, f, fo, ctl, queues[i],
                                   lists[i], counts[i]);
        }
        if (ev) (void)hipEventRecord(ctx->ev[1], st);
    };
    // A graph is captured where a call repeats the arguments of the one before it:
    // capturing and instantiating costs about 90 us, more than the launches it
    // saves, which calls with new buffers each would pay every time.
    bool replay = false;
    if (use_graph) {
        std::vector<uint8_t> key(sizeof(fi) + sizeof(fo) + 40, 0);
        uint8_t* at = key.data();
        auto put = [&](const void* p, size_t n) {
            memcpy(at, p, n);
            at += n;
        };
        put(&fi, sizeof(fi));
        put(&fo, sizeof(fo));
        put(lists, sizeof(lists));
        put(&dnw, 4);
        put(&n_groups, 4);
        put(&n_small, 4);
        put(&n_large, 4);  // (and the path count, in fi: they decide the stages)
        replay = B->exec && key == B->graph_key;
        if (!replay && key == B->last_key) {
            if (B->exec) (void)hipGraphExecDestroy(B->exec);
            if (B->graph) (void)hipGraphDestroy(B->graph);
            B->exec = nullptr;
            B->graph = nullptr;
            hipStream_t cs;
            HIPCHK_RET(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
            HIPCHK_RET(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
            enqueue(cs, false);
            hipError_t e = hipStreamEndCapture(cs, &B->graph);
            (void)hipStreamDestroy(cs);
            HIPCHK_RET(e);
            HIPCHK_RET(hipGraphInstantiate(&B->exec, B->graph, nullptr, nullptr, 0));
            B->graph_key = key;
            replay = true;
        }
        B->last_key = key;
    }
    if (replay) {
        if (timing) HIPCHK_RET(hipEventRecord(ctx->ev[0], s));
        HIPCHK_RET(hipGraphLaunch(B->exec, s));
        if (timing) HIPCHK_RET(hipEventRecord(ctx->ev[1], s));
    } else {
        enqueue(s, timing);
    }
    HIPCHK_RET(hipGetLastError());
    FusedCtl* hc = reinterpret_cast<FusedCtl*>(reinterpret_cast<uint8_t*>(ctx->host_pinned) + 1024);
    HIPCHK_RET(hipMemcpyAsync(hc, ctl, sizeof(FusedCtl), hipMemcpyDeviceToHost, s));
    HIPCHK_RET(hipStreamSynchronize(s));
    if (timing) {
        // graph: the whole launch; direct: the dense kernels
        float ms = 0;
        if (replay) {
            HIPCHK_RET(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
            auto& t = ctx->timings["batched_graph"];
            t.first += ms;
            t.second += 1;
        } else {
            HIPCHK_RET(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
            auto& t = ctx->timings["k_dense"];
            t.first += ms;
            t.second += 1;
        }
    }
    if (hc->error & ERR_INPUT) return -1;
    if (hc->error & ERR_FLATTEN) return -5;
    if (hc->error & ERR_BBOX) return -3;
    const int64_t Tf = (int64_t)hc->tiles, Sf = (int64_t)hc->spans;
    const uint32_t nd = n_stages == 1 ? hc->dq : (n_stages == 2 ? hc->dq2 : hc->dq3);
    int64_t Tp = 0, Sp = 0;
    int st = 0;
    if (nd > 0) {
        // compact the deferred paths and run the plain pipeline on them
        HIPCHK_RET(B->d_sizes.ensure((size_t)nd * sizeof(DeferSize)));
        hipLaunchKernelGGL(k_defer_sizes, dim3((nd + 255) / 256), dim3(256), 0, s, fi, deferred, nd,
                           B->d_sizes.as<DeferSize>());
        HIPCHK_RET(hipGetLastError());
        std::vector<DeferSize> sz(nd);
        HIPCHK_RET(hipMemcpyAsync(sz.data(), B->d_sizes.p, (size_t)nd * sizeof(DeferSize), hipMemcpyDeviceToHost, s));
        HIPCHK_RET(hipStreamSynchronize(s));
        std::sort(sz.begin(), sz.end(), [](const DeferSize& x, const DeferSize& y) { return x.path < y.path; });
        // offsets of the compact batch and the paths, in one upload: voff, poff, woff | ids
        const size_t no = (size_t)nd + 1;
        std::vector<int64_t> pack(3 * no + (nd + 1) / 2, 0);
        int64_t *dv = pack.data(), *dp = dv + no, *dw = dp + no;
        uint32_t* ids = reinterpret_cast<uint32_t*>(dw + no);
        for (uint32_t k = 0; k < nd; k++) {
            dv[k + 1] = dv[k] + sz[k].nv;
            dp[k + 1] = dp[k] + sz[k].np;
            dw[k + 1] = dw[k] + sz[k].nw;
            ids[k] = (uint32_t)sz[k].path;
        }
        HIPCHK_RET(B->g_verbs.ensure(std::max<int64_t>(dv[nd], 1)));
        HIPCHK_RET(B->g_points.ensure(std::max<int64_t>(dp[nd], 1) * 8));
        HIPCHK_RET(B->g_weights.ensure(std::max<int64_t>(dw[nd], 1) * 4));
        HIPCHK_RET(B->d_pack.ensure(pack.size() * 8));
        HIPCHK_RET(B->g_xf.ensure(nd * sizeof(Xform)));
        HIPCHK_RET(B->g_ts.ensure(nd * 8));
        HIPCHK_RET(B->g_tc.ensure(nd * 4));
        HIPCHK_RET(B->g_ss.ensure(nd * 8));
        HIPCHK_RET(B->g_sc.ensure(nd * 4));
        HIPCHK_RET(hipMemcpyAsync(B->d_pack.p, pack.data(), pack.size() * 8, hipMemcpyHostToDevice, s));
        const int64_t* g_voff = B->d_pack.as<int64_t>();
        const int64_t *g_poff = g_voff + no, *g_woff = g_poff + no;
        deferred = reinterpret_cast<uint32_t*>(B->d_pack.as<int64_t>() + 3 * no);
        const uint32_t slices = std::max<uint32_t>(1, std::min<uint32_t>(64, 4096 / nd));
        hipLaunchKernelGGL(k_gather_paths, dim3(std::min<uint32_t>(nd, 4096), slices), dim3(256), 0, s, fi, deferred, nd,
                           g_voff, g_poff, g_woff, B->g_verbs.as<uint8_t>(), B->g_points.as<float>(),
                           B->g_weights.as<float>(), B->g_xf.as<Xform>());
        HIPCHK_RET(hipGetLastError());
        SegInput si;
        si.n_segs = nd;
        si.n_paths = nd;
        si.verbs = B->g_verbs.as<uint8_t>();
        si.points = B->g_points.as<float>();
        si.weights = B->g_weights.as<float>();
        si.seg_verb_off = g_voff;
        si.seg_point_off = g_poff;
        si.seg_weight_off = g_woff;
        si.seg_xf = B->g_xf.as<Xform>();
        si.n_verbs = dv[nd];
        si.n_points = dp[nd];
        si.n_weights = dw[nd];
        si.own_ranges = true;
        OutputDesc od;
        const bool room = Tf <= out.tile_capacity && Sf <= out.span_capacity;
        od.tile_xy = out.tile_xy + (room ? 2 * Tf : 0);
        od.tile_alpha = out.tile_alpha + (room ? 64 * Tf : 0);
        od.tile_cov = out.tile_cov ? out.tile_cov + (room ? 64 * Tf : 0) : nullptr;
        od.tile_capacity = room ? out.tile_capacity - Tf : 0;
        od.span_xy = out.span_xy + (room ? 2 * Sf : 0);
        od.span_w = out.span_w + (room ? Sf : 0);
        od.span_capacity = room ? out.span_capacity - Sf : 0;
        od.path_tile_start = B->g_ts.as<int64_t>();
        od.path_tile_count = B->g_tc.as<int32_t>();
        od.path_span_start = B->g_ss.as<int64_t>();
        od.path_span_count = B->g_sc.as<int32_t>();
        // under the dense kernels' 1-LSB contract the handed-on paths take the
        // unordered tile stage
        st = run_plain(ctx, si, od, s, true);
        Tp = od.n_tiles;
        Sp = od.n_spans;
        if (st == 0) {
            hipLaunchKernelGGL(k_scatter_ranges, dim3((nd + 255) / 256), dim3(256), 0, s, deferred, nd,
                               od.path_tile_start, od.path_tile_count, od.path_span_start, od.path_span_count, Tf,
                               Sf, out.path_tile_start, out.path_tile_count, out.path_span_start,
                               out.path_span_count);
            HIPCHK_RET(hipGetLastError());
        } else if (st != -4) {
            return st;
        }
    }
    out.n_tiles = Tf + Tp;
    out.n_spans = Sf + Sp;
    if ((hc->error & ERR_CAPACITY) || out.n_tiles > out.tile_capacity || out.n_spans > out.span_capacity) return -4;
    return st;
}

// The large-path adjoint of path p, of nv commands and np points (one path over
// the whole device; see adjoint_large.inc).  `hp`: 2 KiB of pinned host memory
// for the read-back.  The call's error word (in the control block at the start
// of large_cmd, whose room for every path of the call the caller has ensured)
// keeps what the last passes of a path report; the caller reads it once.
constexpr size_t AL_CTL_BYTES = 256;  // box[4], nt, err, acc[8]
static size_t al_command_bytes(int64_t nv, int64_t np) {
    return AL_CTL_BYTES + 3 * ((size_t)nv * 8 + 256) + ((size_t)(nv + 1) * 4 + 256) + 2 * ((size_t)np * 4 + 256) +
           ((size_t)nv * 48 + 256);
}
static int al_status(uint32_t err) {
    if (err & ERR_INPUT) return -1;
    if (err & ERR_FLATTEN) return -5;
    if (err & ERR_CAPACITY) return -7;  // coordinates beyond the 16-bit pixel range
    if (err & ERR_BBOX) return -3;
    return 0;
}
static int run_adjoint_large(const FusedIn& fi, const AdjArgs& a, int64_t p, int64_t nv, int64_t np, hipStream_t s,
                             BatchedState* B, uint8_t* hp) {
    if (nv < 0 || np < 0) return -1;
    // command scratch: box, nt, err, acc | cg, cmv, cw | cl | pcmd | closer | slot
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    size_t o = AL_CTL_BYTES;
    const size_t o_cg = o;
    o = al(o + (size_t)nv * 8);
    const size_t o_cmv = o;
    o = al(o + (size_t)nv * 8);
    const size_t o_cw = o;
    o = al(o + (size_t)nv * 8);
    const size_t o_cl = o;
    o = al(o + (size_t)(nv + 1) * 4);
    const size_t o_pcmd = o;
    o = al(o + (size_t)np * 4);
    const size_t o_closer = o;
    o = al(o + (size_t)np * 4);
    const size_t o_slot = o;
    o = al(o + (size_t)nv * 48);
    uint8_t* c = B->large_cmd.as<uint8_t>();
    LargeAdj A;
    memset(&A, 0, sizeof(A));
    A.cg = reinterpret_cast<int64_t*>(c + o_cg);
    A.cmv = reinterpret_cast<int64_t*>(c + o_cmv);
    A.cw = reinterpret_cast<int64_t*>(c + o_cw);
    A.cl = reinterpret_cast<uint32_t*>(c + o_cl);
    A.pcmd = reinterpret_cast<uint32_t*>(c + o_pcmd);
    A.closer = reinterpret_cast<uint32_t*>(c + o_closer);
    A.slot = reinterpret_cast<float*>(c + o_slot);
    A.box = reinterpret_cast<unsigned*>(c);
    A.nt = reinterpret_cast<uint32_t*>(c + 16);
    A.err = reinterpret_cast<uint32_t*>(c + 20);
    A.acc = reinterpret_cast<double*>(c + 64);
    HIPCHK_RET(hipMemsetAsync(A.box, 0xff, 8, s));        // min x, min y
    HIPCHK_RET(hipMemsetAsync(A.box + 2, 0, 12, s));      // max x, max y, nt
    HIPCHK_RET(hipMemsetAsync(A.acc, 0, 8 * 8, s));
    // a wave per workgroup where a thread's work is long and threads are few (a
    // command, a line): 1,400 commands or 30,000 lines then reach every CU
    const int T = 256;
    const unsigned gv = (unsigned)std::max<int64_t>(1, (nv + WAVE - 1) / WAVE);
    hipLaunchKernelGGL(k_al_cmds, dim3(1), dim3(1024), 0, s, fi, p, A);
    hipLaunchKernelGGL(k_al_count, dim3(gv), dim3(WAVE), 0, s, fi, p, A);
    hipLaunchKernelGGL(k_al_scan, dim3(1), dim3(1024), 0, s, fi, p, A);
    HIPCHK_RET(hipGetLastError());
    uint32_t* hc = reinterpret_cast<uint32_t*>(hp + 64);
    HIPCHK_RET(hipMemcpyAsync(hc, A.cl + nv, 4, hipMemcpyDeviceToHost, s));
    HIPCHK_RET(hipMemcpyAsync(hc + 1, A.box, 24, hipMemcpyDeviceToHost, s));  // box[4], nt, err
    HIPCHK_RET(hipStreamSynchronize(s));
    if (const int st = al_status(hc[6])) return st;
    const int64_t L = hc[0];
    if (L >= AL_MAX_LINES) return -7;
    int32_t tx0 = 0, ty0 = 0, GW = 0, GH = 0;
    if (L > 0)
        grid_from_box(true, false, (int32_t)floorf(unord_f(hc[1])), (int32_t)floorf(unord_f(hc[2])),
                      (int32_t)floorf(unord_f(hc[3])), (int32_t)floorf(unord_f(hc[4])), &tx0, &ty0, &GW, &GH);
    const int64_t tiles = (int64_t)GW * GH;
    if (tiles > AL_MAX_TILES) return -7;
    const int32_t ow = (GW + 31) / 32;
    // line and grid scratch
    o = 0;
    const size_t o_l32 = o;
    o = al(o + (size_t)L * 16);
    const size_t o_l64 = o;
    o = al(o + (size_t)L * 32);
    const size_t o_dl = o;
    o = al(o + (size_t)L * 16);
    const size_t o_occ = o;
    o = al(o + (size_t)ow * GH * 4);
    const size_t o_fa = o;
    o = al(o + (size_t)tiles * 64 * 8);
    const size_t o_fh = o;
    o = al(o + (size_t)tiles * 64 * 8);
    const size_t o_ts = o;
    o = al(o + (size_t)tiles * 4);
    const size_t o_span = o;
    o = al(o + (size_t)tiles);
    const size_t o_g = o;
    o = al(o + (size_t)tiles * 64 * 4);
    const size_t o_G = o;
    o = al(o + (size_t)tiles * 64 * 4);
    HIPCHK_RET(B->large_grid.ensure(std::max<size_t>(o, 256)));
    uint8_t* gbuf = B->large_grid.as<uint8_t>();
    A.l32 = reinterpret_cast<float4*>(gbuf + o_l32);
    A.l64 = reinterpret_cast<double2*>(gbuf + o_l64);
    A.dl = reinterpret_cast<float4*>(gbuf + o_dl);
    A.occ = reinterpret_cast<uint32_t*>(gbuf + o_occ);
    A.fa = reinterpret_cast<unsigned long long*>(gbuf + o_fa);
    A.fh = reinterpret_cast<unsigned long long*>(gbuf + o_fh);
    A.tsign = reinterpret_cast<int32_t*>(gbuf + o_ts);
    A.span = gbuf + o_span;
    A.g = reinterpret_cast<float*>(gbuf + o_g);
    A.G = reinterpret_cast<float*>(gbuf + o_G);
    A.tx0 = tx0;
    A.ty0 = ty0;
    A.GW = GW;
    A.GH = GH;
    A.ow = ow;
    if (o_g > o_occ) HIPCHK_RET(hipMemsetAsync(gbuf + o_occ, 0, o_g - o_occ, s));  // occ, sums, crossings, spans
    const unsigned gl = (unsigned)std::max<int64_t>(1, (L + WAVE - 1) / WAVE);
    const unsigned gp = (unsigned)std::max<int64_t>(1, (np + AL_GT - 1) / AL_GT);
    hipLaunchKernelGGL(k_al_lines, dim3(gv), dim3(WAVE), 0, s, fi, p, A);
    if (L > 0) hipLaunchKernelGGL(k_al_fwd, dim3(gl), dim3(WAVE), 0, s, L, A);
    hipLaunchKernelGGL(k_al_spans, dim3(1), dim3(1024), 0, s, A);
    if (GH > 0) hipLaunchKernelGGL(k_al_rows, dim3(GH), dim3(512), 0, s, fi, A, a, p);
    // target tiles: one thread each (their count is the caller's, bounded by its capacity)
    hipLaunchKernelGGL(k_al_target, dim3(4096), dim3(T), 0, s, fi, A, a, p);
    if (L > 0) hipLaunchKernelGGL(k_al_bwd, dim3(gl), dim3(WAVE), 0, s, L, A);
    hipLaunchKernelGGL(k_al_cmd_bwd, dim3(gv), dim3(WAVE), 0, s, fi, p, A);
    if (np > 0) hipLaunchKernelGGL(k_al_gather, dim3(gp), dim3(AL_GT), 0, s, fi, p, A, a);
    hipLaunchKernelGGL(k_al_final, dim3(1), dim3(1), 0, s, A, a, p);
    HIPCHK_RET(hipGetLastError());
    return 0;
}

int run_adjoint(Context* ctx, const SegInput& in, const AdjTarget& tgt, float* loss, float* d_points, float* d_xf,
                hipStream_t s, int waves_per_cu, int gran, int tiles_per_chunk) {
    if (!ctx->batched) ctx->batched = new BatchedState();
    BatchedState* B = reinterpret_cast<BatchedState*>(ctx->batched);
    const int64_t NP = in.n_paths;
    if (NP <= 0) return 0;
    int dev = 0, cus = 0;
    HIPCHK_RET(hipGetDevice(&dev));
    HIPCHK_RET(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int n_waves = std::max(1, cus * std::max(1, waves_per_cu));
    HIPCHK_RET(B->scratch.ensure((size_t)n_waves * F_SCRATCH));
    HIPCHK_RET(B->ascratch.ensure((size_t)n_waves * A_SCRATCH));
    HIPCHK_RET(B->ctl.ensure(sizeof(FusedCtl)));
    if (!ctx->host_pinned) HIPCHK_RET(hipHostMalloc(&ctx->host_pinned, 4096));
    FusedIn fi;
    fi.n_paths = NP;
    fi.verbs = in.verbs;
    fi.verb_off = in.seg_verb_off;
    fi.points = in.points;
    fi.point_off = in.seg_point_off;
    fi.weights = in.weights;
    fi.weight_off = in.seg_weight_off;
    fi.xf = in.seg_xf;
    fi.n_points = in.n_points;
    fi.n_weights = in.n_weights;
    AdjArgs a;
    a.tt_start = tgt.tile_start;
    a.tt_count = tgt.tile_count;
    a.t_xy = tgt.tile_xy;
    a.t_cov = tgt.tile_cov;
    a.ts_start = tgt.span_start;
    a.ts_count = tgt.span_count;
    a.ts_xy = tgt.span_xy;
    a.ts_w = tgt.span_w;
    a.loss = loss;
    a.d_points = d_points;
    a.d_xf = d_xf;
    FusedCtl* ctl = B->ctl.as<FusedCtl>();
    const uint32_t g = (uint32_t)std::max(1, gran);
    hipLaunchKernelGGL(k_fused_reset, dim3(1), dim3(64), 0, s, ctl);
    if (NP > n_waves) {  // (up to a path per wave all start at once)
        HIPCHK_RET(B->adj_bin.ensure((size_t)NP));
        HIPCHK_RET(B->adj_ids.ensure((size_t)NP * 4));
        hipLaunchKernelGGL(k_adj_weigh, dim3((uint32_t)((NP + 3) / 4)), dim3(256), 0, s, fi, B->adj_bin.as<uint8_t>());
        hipLaunchKernelGGL(k_adj_order, dim3(1), dim3(1024), 0, s, B->adj_bin.as<uint8_t>(), NP,
                           B->adj_ids.as<uint32_t>());
        fi.ids = B->adj_ids.as<uint32_t>();
    }
    if (ctx->timing) {
        if (!ctx->ev[0]) HIPCHK_RET(hipEventCreate(&ctx->ev[0]));
        if (!ctx->ev[1]) HIPCHK_RET(hipEventCreate(&ctx->ev[1]));
        HIPCHK_RET(hipEventRecord(ctx->ev[0], s));
    }
    HIPCHK_RET(B->deferred.ensure((size_t)NP * 4));
    uint32_t* large = B->deferred.as<uint32_t>();
    if (tiles_per_chunk <= 16)
        hipLaunchKernelGGL(k_adjoint<16>, dim3(n_waves), dim3(WAVE), 0, s, fi, a, ctl, B->scratch.as<uint8_t>(),
                           B->ascratch.as<uint8_t>(), g, large);
    else
        hipLaunchKernelGGL(k_adjoint<32>, dim3(n_waves), dim3(WAVE), 0, s, fi, a, ctl, B->scratch.as<uint8_t>(),
                           B->ascratch.as<uint8_t>(), g, large);
    HIPCHK_RET(hipGetLastError());
    if (ctx->timing) HIPCHK_RET(hipEventRecord(ctx->ev[1], s));
    FusedCtl* hc = reinterpret_cast<FusedCtl*>(reinterpret_cast<uint8_t*>(ctx->host_pinned) + 1024);
    HIPCHK_RET(hipMemcpyAsync(hc, ctl, sizeof(FusedCtl), hipMemcpyDeviceToHost, s));
    HIPCHK_RET(hipStreamSynchronize(s));
    if (ctx->timing) {
        float ms = 0;
        HIPCHK_RET(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
        auto& t = ctx->timings["k_adjoint"];
        t.first += ms;
        t.second += 1;
    }
    if (hc->error & ERR_INPUT) return -1;
    if (hc->error & ERR_FLATTEN) return -5;
    if (hc->error & ERR_BBOX) return -3;
    if (hc->error & ERR_CAPACITY) return -7;
    // the paths over one wave's limits, one at a time over the whole device
    const uint32_t n_large = hc->deferred;
    if (n_large) {
        HIPCHK_RET(B->large_grid.ensure((size_t)n_large * sizeof(AlSize)));
        AlSize* dsz = B->large_grid.as<AlSize>();
        hipLaunchKernelGGL(k_al_sizes, dim3((n_large + 255) / 256), dim3(256), 0, s, fi, large, n_large, dsz);
        HIPCHK_RET(hipGetLastError());
        std::vector<AlSize> sz(n_large);
        HIPCHK_RET(hipMemcpyAsync(sz.data(), dsz, (size_t)n_large * sizeof(AlSize), hipMemcpyDeviceToHost, s));
        HIPCHK_RET(hipStreamSynchronize(s));
        std::sort(sz.begin(), sz.end(), [](const AlSize& x, const AlSize& y) { return x.path < y.path; });
        size_t room = 0;
        for (const AlSize& z : sz) room = std::max(room, al_command_bytes(std::max<int64_t>(z.nv, 0), std::max<int64_t>(z.np, 0)));
        HIPCHK_RET(B->large_cmd.ensure(room));
        HIPCHK_RET(hipMemsetAsync(B->large_cmd.p, 0, AL_CTL_BYTES, s));
        uint8_t* hp = reinterpret_cast<uint8_t*>(ctx->host_pinned) + 2048;
        for (const AlSize& z : sz) {
            const int st = run_adjoint_large(fi, a, z.path, z.nv, z.np, s, B, hp);
            if (st) return st;
        }
        uint32_t* he = reinterpret_cast<uint32_t*>(hp);
        HIPCHK_RET(hipMemcpyAsync(he, B->large_cmd.as<uint8_t>() + 20, 4, hipMemcpyDeviceToHost, s));
        HIPCHK_RET(hipStreamSynchronize(s));
        return al_status(*he);
    }
    return 0;
}

// ------------------------------------------- one path, no host round trip
//
// A Rasterizer's single fill: k_single (one workgroup of sixteen waves) resets
// the control block itself, writes the output and the counts wherever `out`
// and `ctl` (SMALL_CTL_BYTES) point, and nothing synchronises.  The drop-in
// finish points both at pinned host memory mapped into the device's address
// space, so that no copy follows the launch; after the caller's
// synchronisation small_batch_result reads the counts.  A path over the
// kernel's limits is only counted as deferred (the caller reruns it through
// run_batched, which handles it).
static_assert(sizeof(FusedCtl) == SMALL_CTL_BYTES, "control block size");

int launch_single_fill(const SegInput& in, const OutputDesc& out, void* ctl, hipStream_t s) {
    if (in.n_paths != 1) return -1;
    FusedIn fi;
    fi.n_paths = 1;
    fi.verbs = in.verbs;
    fi.verb_off = in.seg_verb_off;
    fi.points = in.points;
    fi.point_off = in.seg_point_off;
    fi.weights = in.weights;
    fi.weight_off = in.seg_weight_off;
    fi.xf = in.seg_xf;
    fi.n_points = in.n_points;
    fi.n_weights = in.n_weights;
    FusedOut fo;
    fo.tile_xy = out.tile_xy;
    fo.tile_alpha = out.tile_alpha;
    fo.tile_cov = out.tile_cov;
    fo.tile_cap = out.tile_capacity;
    fo.span_xy = out.span_xy;
    fo.span_w = out.span_w;
    fo.span_cap = out.span_capacity;
    fo.pts = out.path_tile_start;
    fo.ptc = out.path_tile_count;
    fo.pss = out.path_span_start;
    fo.psc = out.path_span_count;
    hipLaunchKernelGGL(k_single, dim3(1), dim3(S_NT), 0, s, fi, fo, reinterpret_cast<FusedCtl*>(ctl));
    HIPCHK_RET(hipGetLastError());
    return 0;
}

SmallBatchResult small_batch_result(const void* host_ctl) {
    const FusedCtl* hc = reinterpret_cast<const FusedCtl*>(host_ctl);
    SmallBatchResult r;
    r.tiles = (int64_t)hc->tiles;
    r.spans = (int64_t)hc->spans;
    r.deferred = hc->deferred;
    r.status = (hc->error & ERR_INPUT) ? -1 : (hc->error & ERR_FLATTEN) ? -5 : (hc->error & ERR_BBOX) ? -3
               : (hc->error & ERR_CAPACITY) ? -4 : 0;
    return r;
}

// ------------------------------------------------ the dense chain alone
//
// The dense 64-tile instance over every path, then the 256-tile instance over
// the paths it hands on, with control memory (DENSE_CTL_BYTES: queues,
// counters, error bits) and the handed-on list (n_paths entries) supplied by
// the caller: nothing is allocated.  Paths the 256-tile instance hands on are
// counted, not listed.
static_assert(sizeof(FusedCtl) == DENSE_CTL_BYTES, "control block size");

int launch_dense_chain(const SegInput& in, const OutputDesc& out, uint8_t* ctl_mem, uint32_t* ids, hipStream_t s) {
    const int64_t NP = in.n_paths;
    if (NP <= 0) return 0;
    int dev = 0, cus = 0;
    HIPCHK_RET(hipGetDevice(&dev));
    HIPCHK_RET(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    FusedCtl* ctl = reinterpret_cast<FusedCtl*>(ctl_mem);
    FusedIn fi;
    fi.n_paths = NP;
    fi.verbs = in.verbs;
    fi.verb_off = in.seg_verb_off;
    fi.points = in.points;
    fi.point_off = in.seg_point_off;
    fi.weights = in.weights;
    fi.weight_off = in.seg_weight_off;
    fi.xf = in.seg_xf;
    fi.n_points = in.n_points;
    fi.n_weights = in.n_weights;
    FusedOut fo;
    fo.tile_xy = out.tile_xy;
    fo.tile_alpha = out.tile_alpha;
    fo.tile_cov = out.tile_cov;
    fo.tile_cap = out.tile_capacity;
    fo.span_xy = out.span_xy;
    fo.span_w = out.span_w;
    fo.span_cap = out.span_capacity;
    fo.pts = out.path_tile_start;
    fo.ptc = out.path_tile_count;
    fo.pss = out.path_span_start;
    fo.psc = out.path_span_count;
    FusedIn f2 = fi;  // the 256-tile instance runs over the 64-tile one's hand-ons
    f2.ids = ids;
    f2.n_ids = &ctl->dq;
    hipLaunchKernelGGL(k_fused_reset, dim3(1), dim3(64), 0, s, ctl);
    hipLaunchKernelGGL((k_dense<4, 64>), dim3(cus * 4), dim3(4 * WAVE), 0, s, fi, fo, ctl, &ctl->queue, ids,
                       &ctl->dq);
    hipLaunchKernelGGL((k_dense<16, 256>), dim3(cus), dim3(16 * WAVE), 0, s, f2, fo, ctl, &ctl->queue3,
                       (uint32_t*)nullptr, &ctl->dq2);
    HIPCHK_RET(hipGetLastError());
    return 0;
}

int finish_dense_chain(const uint8_t* ctl_mem, OutputDesc& out, hipStream_t s) {
    FusedCtl hc;
    HIPCHK_RET(hipMemcpyAsync(&hc, ctl_mem, sizeof(FusedCtl), hipMemcpyDeviceToHost, s));
    HIPCHK_RET(hipStreamSynchronize(s));
    if (hc.error & ERR_INPUT) return -1;
    if (hc.error & ERR_FLATTEN) return -5;
    if (hc.error & ERR_BBOX) return -3;
    out.n_tiles = (int64_t)hc.tiles;
    out.n_spans = (int64_t)hc.spans;
    if ((hc.error & ERR_CAPACITY) || out.n_tiles > out.tile_capacity || out.n_spans > out.span_capacity) return -4;
    if (hc.dq2) return -7;
    return 0;
}

}  // namespace ochre
