// The plain five-stage pipeline (gfx950):
//   (a) flatten      k_flatten<false> counts lines per command, a device scan
//                    allocates slots, k_flatten<true> writes them
//   (b) binning      k_dda<false>/<true> walk each line's DDA and emit one
//                    sort entry per tile run and per tile-row crossing,
//                    keyed (path, tile_y, tile_x); k_rs_* radix-sort them
//   (c) accumulation k_tile_rows: one wave per tile row; a lane per run
//                    replays the row's runs, then the runs are added in
//                    sorted order, a lane per increment, into LDS sums
//   (d) row scan     the carry (rasterizer.rs:233-250) folded across the
//                    lanes of each pixel row, and the winding of the tile-row
//                    crossings (rasterizer.rs:252-261)
//   (e) compaction   k_tile_counts counts tiles and spans per tile row; they
//                    are written at the scanned offsets
// References: glowcoil/ochre src/path.rs:41-109, src/rasterizer.rs:61-268.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cmath>
#include <cstring>
#include <vector>

#include "device_common.hpp"
#include "pipeline.hpp"
#include "radix_sort.hpp"
#include "raster_common.hpp"
#include "scan.hpp"

namespace ochre {

// ----------------------------------------------------------------- utils

hipError_t DBuf::ensure(size_t need) {
    if (need <= bytes && p) return hipSuccess;
    size_t nb = std::max<size_t>(need + need / 4, 4096);
    if (p) {
        hipError_t e = hipFree(p);
        p = nullptr;
        bytes = 0;
        if (e != hipSuccess) return e;
    }
    hipError_t e = hipMalloc(&p, nb);
    if (e != hipSuccess) {
        p = nullptr;
        return e;
    }
    bytes = nb;
    return hipSuccess;
}

DBuf::~DBuf() {
    if (p) (void)hipFree(p);
}

AtlasState::~AtlasState() {
    if (host) (void)hipHostFree(host);
}

StrokeBuffers::~StrokeBuffers() {
    if (host) (void)hipHostFree(host);
}

Context::~Context() {
    if (host_pinned) (void)hipHostFree(host_pinned);
    for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
    for (auto& e : side_ev)
        if (e) (void)hipEventDestroy(e);
    if (own_stream) (void)hipStreamDestroy(own_stream);
}

int map_hip_error(hipError_t e) {
    if (e == hipSuccess) return 0;
    if (e == hipErrorOutOfMemory) return -2;
    return -3;
}

hipError_t ensure_scan_capacity(Context* ctx, int64_t n) {
    int64_t blocks = std::max<int64_t>(1, (n + SCAN_TILE - 1) / SCAN_TILE);
    return ctx->scan_partials.ensure((size_t)blocks * 16);
}

template <typename T, typename Op, typename Load, typename Store>
static hipError_t launch_scan(Context* ctx, int64_t n, Load load, Store store, Op op, T identity, T* total,
                              hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (n <= SCAN_TILE) {
        hipLaunchKernelGGL((k_scan_single<T, Op, Load, Store>), dim3(1), dim3(SCAN_NT), 0, s, load, store, n, op,
                           identity, total);
        return hipGetLastError();
    }
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if ((size_t)nb * sizeof(T) > ctx->scan_partials.bytes) return hipErrorInvalidValue;
    T* partials = ctx->scan_partials.as<T>();
    hipLaunchKernelGGL((k_scan_reduce<T, Op, Load>), dim3((uint32_t)nb), dim3(SCAN_NT), 0, s, load, n, partials, op,
                       identity);
    hipLaunchKernelGGL((k_scan_partials<T, Op>), dim3(1), dim3(SCAN_NT), 0, s, partials, nb, op, identity, total);
    hipLaunchKernelGGL((k_scan_down<T, Op, Load, Store>), dim3((uint32_t)nb), dim3(SCAN_NT), 0, s, load, store, n,
                       (const T*)partials, op, identity);
    return hipGetLastError();
}

template <typename T>
__global__ void k_fill(T* p, int64_t n, T v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

template <typename T>
static void fill(T* p, int64_t n, T v, hipStream_t s) {
    if (n <= 0) return;
    int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_fill<T>, dim3((uint32_t)blocks), dim3(256), 0, s, p, n, v);
}

static inline uint32_t bits_for(uint64_t n) {  // smallest b with (1 << b) >= n
    uint32_t b = 0;
    while (b < 63 && (1ull << b) < n) b++;
    return b;
}

// --------------------------------------------------- (a) command prologue

struct CmdAcc {
    uint32_t pts;
    uint32_t conics;
    int32_t move;
    uint32_t pad;
};
struct OpCmd {
    __device__ CmdAcc operator()(CmdAcc a, CmdAcc b) const {
        return CmdAcc{a.pts + b.pts, a.conics + b.conics, a.move > b.move ? a.move : b.move, 0u};
    }
};
struct LoadCmd {
    const uint8_t* verbs;
    __device__ CmdAcc operator()(int64_t i) const {
        int v = verbs[i];
        int np = verb_points(v);
        return CmdAcc{(uint32_t)(np < 0 ? 0 : np), v == CONIC ? 1u : 0u, v == MOVE ? (int32_t)i : -1, 0u};
    }
};
struct StoreCmd {
    CmdAcc* out;
    __device__ void operator()(int64_t i, CmdAcc excl, CmdAcc) const { out[i] = excl; }
};

// Largest index s in [0, n) with arr[s] <= v (arr non-decreasing, arr[lo] <= v).
__device__ inline int64_t seg_search(const int64_t* arr, int64_t n, int64_t v, int64_t lo = 0) {
    int64_t hi = n;
    while (hi - lo > 1) {
        int64_t mid = (lo + hi) >> 1;
        if (arr[mid] <= v) lo = mid;
        else hi = mid;
    }
    return lo;
}

// seg_search for consecutive v on consecutive lanes: the wave's first lane (its
// v is the smallest) searches once, on uniform addresses; the others step on
// from its segment, mostly by none or one, doubling the step where a wave spans
// many segments.
__device__ inline int64_t seg_search_wave(const int64_t* arr, int64_t n, int64_t v) {
    const uint32_t v_lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
    const uint32_t v_hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    int64_t lo = seg_search(arr, n, (int64_t)(((uint64_t)v_hi << 32) | v_lo));
    for (int64_t step = 1; lo + 1 < n && arr[lo + 1] <= v; step *= 2) {
        const int64_t to = lo + step < n ? lo + step : n - 1;
        if (arr[to] > v) return seg_search(arr, to, v, lo);
        lo = to;
    }
    return lo;
}

__device__ inline V2 load_point(const SegInput& in, int64_t g, int64_t s) {
    V2 p = mk(in.points[2 * g], in.points[2 * g + 1]);
    if (in.seg_raw && in.seg_raw[s]) return p;
    return apply(in.seg_xf[s], p);
}

// Command i, of segment s.
__device__ inline Cmd resolve_cmd(const SegInput& in, const CmdAcc* scan, int64_t i, int64_t s) {
    Cmd c;
    int64_t p = in.seg_path ? in.seg_path[s] : s;
    int64_t fs = in.path_seg_off ? in.path_seg_off[p] : p;
    int64_t ls = in.path_seg_off ? in.path_seg_off[p + 1] : p + 1;
    int64_t vb = in.seg_verb_off[fs], ve = in.seg_verb_off[ls];
    int64_t pb = in.seg_point_off[fs];
    CmdAcc a = scan[i];
    // the point and weight cursors, and the ends of what they may reach; the
    // scanned ones count from the arrays' start, a path's own from its first verb
    CmdAcc base{0, 0, -1, 0};
    int64_t p0 = 0, w0 = 0, p_end = in.n_points, w_end = in.n_weights;
    if (in.own_ranges) {
        base = scan[vb];
        p0 = pb;
        p_end = in.seg_point_off[s + 1];
        w0 = in.seg_weight_off[s];
        w_end = in.seg_weight_off[s + 1];
    }
    const int64_t g = p0 + (a.pts - base.pts);
    c.path = (int32_t)p;
    c.verb = in.verbs[i];
    c.last_in_path = (i == ve - 1);
    int np = verb_points(c.verb);
    c.bad = np < 0;
    if (np < 0) np = 0;
    if (in.own_ranges) {
        if (c.last_in_path && g + np != p_end) c.bad = true;
    } else if (i == in.seg_verb_off[s] && (g != in.seg_point_off[s] || (int64_t)a.conics != in.seg_weight_off[s])) {
        c.bad = true;
    }
    if (g + np > p_end) {
        c.bad = true;
        np = 0;
    }
    // static indices keep the command in registers
    if (np > 0) c.pt[0] = load_point(in, g, s);
    if (np > 1) c.pt[1] = load_point(in, g + 1, s);
    if (np > 2) c.pt[2] = load_point(in, g + 2, s);
    c.w = 0.0f;
    if (c.verb == CONIC) {
        const int64_t wi = w0 + (a.conics - base.conics);
        if (wi < w_end) c.w = in.weights[wi];
        else c.bad = true;
    }
    if (g > p_end) {  // (bad already)
        c.start = mk(0.0f, 0.0f);
    } else if (g > pb) {
        int64_t sp = (g - 1 >= in.seg_point_off[s]) ? s : seg_search(in.seg_point_off, in.n_segs, g - 1);
        c.start = load_point(in, g - 1, sp);
    } else {
        c.start = mk(0.0f, 0.0f);
    }
    if (a.move >= vb) {
        int64_t ms = a.move >= in.seg_verb_off[s] ? s : seg_search(in.seg_verb_off, in.n_segs, a.move);
        const int64_t gm = p0 + (scan[a.move].pts - base.pts);
        if (gm < p_end) c.first = load_point(in, gm, ms);
        else c.bad = true;
    } else {
        c.first = mk(0.0f, 0.0f);
    }
    return c;
}

// Whether command i belongs to a path (own ranges may leave some before and after).
__device__ inline bool in_paths(const SegInput& in, int64_t i) {
    return i < in.n_verbs &&
           (!in.own_ranges || (i >= in.seg_verb_off[0] && i < in.seg_verb_off[in.n_segs]));
}

// The paths' boxes, empty.  A path of its own range without verbs has no points either.
__global__ void k_path_init(SegInput in, PathBox* box, Counters* cnt) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= in.n_paths) return;
    box[p] = PathBox{INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, 0, {0, 0, 0}};
    if (in.own_ranges && in.seg_verb_off[p] == in.seg_verb_off[p + 1] && in.seg_point_off[p] != in.seg_point_off[p + 1])
        atomicOr(&cnt->error, (uint32_t)ERR_INPUT);
}

struct FlattenArgs {
    SegInput in;
    const CmdAcc* scan;
    uint32_t* cmd_lines;
    uint32_t* cmd_seg;  // the command's segment: count pass to emit pass
    const uint32_t* cmd_line_off;
    float4* lines;
    uint32_t* line_path;
    PathBox* box;
    Counters* cnt;
};

// A command of the emit pass's block, for the threads that make its lines:
// its points, a curve's step, and command_lines' decomposition of its lines
// (a Move's implicit close or a Line's own line, a curve's segments, the
// path's final close).
struct FlatCmd {
    float2 start, p0, p1, p2, first;
    float dt;
    uint32_t info;  // verb | segments << 4 (up to FLATTEN_LIMIT) | own << 30 | close << 31
    uint32_t path;
};

// The emit pass: FL_CMDS commands per workgroup of FL_NT threads.  A thread per
// command resolves it (a conic's lines it writes itself); then a thread per line
// makes its line, each wave a run of consecutive lines, so that consecutive
// threads write consecutive lines and a curve segment's start is its left
// neighbour's end.  Bound by latency, not by the 20 bytes it writes per line: a
// segment's parameter is a chain of additions (t accumulated the reference's
// way), so the command's thread keeps every 8th value of it and a segment adds on
// from there; 64 commands per workgroup instead of 256 (a blob's commands make 30
// to 80 lines each) give four times the waves, and the count
// pass leaves each command's segment.  24 blobs: 318 -> 51 us, 10,000 glyphs:
// 64 -> 53 us, 61 glyphs: 22 -> 10 us (128 commands per workgroup: 59, 43, 12).
constexpr int FL_CMDS = 64, FL_NT = 256;
constexpr int FL_CK = 16, FL_CK_STEP = 8;  // t after 0, 8, .. 120 steps

template <bool EMIT>
__global__ __launch_bounds__(256) void k_flatten(FlattenArgs a) {
    const int64_t i = blockIdx.x * (int64_t)(EMIT ? FL_CMDS : 256) + threadIdx.x;
    const bool in_range = i < a.in.n_verbs && (!EMIT || threadIdx.x < FL_CMDS);
    if (EMIT) {
        __shared__ FlatCmd fc[FL_CMDS];
        __shared__ uint32_t foff[FL_CMDS + 1];
        __shared__ float ck[FL_CMDS][FL_CK + 1];  // (+ 1: the commands' rows in different banks)
        const int t = threadIdx.x;
        const int64_t i0 = (int64_t)blockIdx.x * FL_CMDS;
        const int nb = (int)min<int64_t>((int64_t)FL_CMDS, a.in.n_verbs - i0);
        if (in_range) {
            foff[t] = a.cmd_line_off[i];
            if (t == nb - 1) foff[nb] = foff[t] + a.cmd_lines[i];
            fc[t].info = 0xfu;  // no lines
        }
        if (in_range && in_paths(a.in, i)) {
            const Cmd c = resolve_cmd(a.in, a.scan, i, a.cmd_seg[i]);
            const uint32_t o = foff[t];
            FlatCmd f;
            f.start = make_float2(c.start.x, c.start.y);
            f.p0 = make_float2(c.pt[0].x, c.pt[0].y);
            f.p1 = make_float2(c.pt[1].x, c.pt[1].y);
            f.p2 = make_float2(c.pt[2].x, c.pt[2].y);
            f.first = make_float2(c.first.x, c.first.y);
            f.dt = 0.0f;
            f.path = (uint32_t)c.path;
            uint32_t own = 0, nseg = 0;
            V2 last = c.start, first = c.first;
            if (c.bad) {
                f.info = 0xfu;  // no lines (the count pass reported it)
            } else if (c.verb == CONIC) {
                uint32_t q = o;
                command_lines(c, [&](V2 p0, V2 p1) {
                    a.lines[q] = make_float4(p0.x, p0.y, p1.x, p1.y);
                    a.line_path[q] = (uint32_t)c.path;
                    q++;
                });
                f.info = (uint32_t)CONIC;
            } else {
                if (c.verb == MOVE) {
                    own = veq(last, first) ? 0u : 1u;
                    last = first = c.pt[0];
                } else if (c.verb == LINE) {
                    own = 1u;
                    last = c.pt[0];
                } else if (c.verb == QUAD || c.verb == CUBIC) {
                    const bool cubic = c.verb == CUBIC;
                    f.dt = cubic ? cubic_dt(last, c.pt[0], c.pt[1], c.pt[2]) : quad_dt(last, c.pt[0], c.pt[1]);
                    // the lines counted, less the close after them
                    last = cubic ? cubic_at(1.0f, last, c.pt[0], c.pt[1], c.pt[2]) : quad_at(1.0f, last, c.pt[0], c.pt[1]);
                }
                const uint32_t close = (c.last_in_path && !veq(last, first)) ? 1u : 0u;
                if (c.verb == QUAD || c.verb == CUBIC) {
                    nseg = a.cmd_lines[i] - close;
                    float tt = 0.0f;
                    for (uint32_t k = 0; k < min(nseg, (uint32_t)(FL_CK * FL_CK_STEP)); k++) {
                        if (k % FL_CK_STEP == 0) ck[t][k / FL_CK_STEP] = tt;
                        tt = fminf(tt + f.dt, 1.0f);
                    }
                }
                f.info = (uint32_t)c.verb | (nseg << 4) | (own << 30) | (close << 31);
            }
            fc[t] = f;
        }
        __syncthreads();
        if (nb <= 0) return;
        const uint32_t l0 = foff[0], l1 = foff[nb];
        const int lane = t & (WAVE - 1);
        const uint32_t per = ((l1 - l0 + FL_NT - 1) / FL_NT) * WAVE;  // lines per wave
        const uint32_t w0 = l0 + (uint32_t)(t / WAVE) * per, w1 = min(l1, w0 + per);
        V2 prev = mk(0.0f, 0.0f);  // the end of the line before the wave's next 64
        for (uint32_t b = w0; b < w1; b += WAVE) {
            const uint32_t q = b + (uint32_t)lane;
            const bool valid = q < w1;
            int lo = 0, hi = nb - 1;  // the last command with foff <= q (it has lines)
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (foff[mid] <= q) lo = mid;
                else hi = mid - 1;
            }
            const FlatCmd f = fc[lo];
            const int verb = (int)(f.info & 0xfu);
            const uint32_t j = q - foff[lo], nseg = (f.info >> 4) & 0x3ffffffu, own = (f.info >> 30) & 1u;
            const V2 c0 = mk(f.start.x, f.start.y), fp = mk(f.first.x, f.first.y);
            const V2 c1 = mk(f.p0.x, f.p0.y), c2 = mk(f.p1.x, f.p1.y), c3 = mk(f.p2.x, f.p2.y);
            const bool cubic = verb == CUBIC, curve = cubic || verb == QUAD;
            auto at = [&](float u) { return cubic ? cubic_at(u, c0, c1, c2, c3) : quad_at(u, c0, c1, c2); };
            V2 pa = c0, pb = fp;
            float tp = 1.0f, tt = 1.0f;
            if (curve) {
                if (j < nseg) {  // segment j: t accumulated the reference's way (path.rs:49-74)
                    uint32_t k = min(j / FL_CK_STEP, (uint32_t)(FL_CK - 1));
                    tp = tt = ck[lo][k];
                    for (k *= FL_CK_STEP; k <= j; k++) {
                        tp = tt;
                        tt = fminf(tt + f.dt, 1.0f);
                    }
                    pb = at(tt);
                }
            } else if (own && j == 0) {  // a Move's implicit close, or a Line
                pb = verb == MOVE ? fp : c1;
            } else if (verb == LINE) {  // the path's final close, from a Line's point or the command's start (a Close)
                pa = c1;
            }
            // a later segment (or a curve's final close) starts where the line before it ends
            const V2 left = mk(__shfl_up(pb.x, 1, WAVE), __shfl_up(pb.y, 1, WAVE));
            if (curve && j > 0) {
                pa = lane == 0 ? prev : left;
                if (lane == 0 && b == w0) pa = at(tp);
            }
            prev = mk(__shfl(pb.x, WAVE - 1, WAVE), __shfl(pb.y, WAVE - 1, WAVE));
            if (valid && verb != CONIC && verb != 0xf) {  // (a conic's are written above; a bad command has none)
                a.lines[q] = make_float4(pa.x, pa.y, pb.x, pb.y);
                a.line_path[q] = f.path;
            }
        }
        return;
    }
    // count pass: lines per command, and a box holding the path's lines (from
    // the commands' control points: command_count).  A path's commands are
    // contiguous, so the wave reduces the box per path (segmented by path) and
    // one lane per path segment does the atomics.
    int32_t key = -1;
    uint32_t n = 0, flags = 0;
    BoxAcc box;
    if (in_range && !in_paths(a.in, i)) {
        a.cmd_lines[i] = 0;
    } else if (in_range) {
        const int64_t sg = seg_search_wave(a.in.seg_verb_off, a.in.n_segs, i);
        a.cmd_seg[i] = (uint32_t)sg;
        Cmd c = resolve_cmd(a.in, a.scan, i, sg);
        key = c.path;
        if (c.bad) {
            atomicOr(&a.cnt->error, (uint32_t)ERR_INPUT);
        } else {
            const bool ok = command_count(c, n, [&](V2 q) { box.add(q); });
            if (!ok) atomicOr(&a.cnt->error, (uint32_t)ERR_FLATTEN);
        }
        a.cmd_lines[i] = n;
        if (n > 0) flags = box.full ? (uint32_t)(BOX_FULL | BOX_LINES) : (uint32_t)BOX_LINES;
    }
    int32_t mnx = INT32_MAX, mny = INT32_MAX, mxx = INT32_MIN, mxy = INT32_MIN;
    if (n > 0 && box.minx <= box.maxx) {
        mnx = (int32_t)floorf(box.minx);
        mny = (int32_t)floorf(box.miny);
        mxx = (int32_t)floorf(box.maxx);
        mxy = (int32_t)floorf(box.maxy);
    }
    const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int32_t k2 = __shfl_up(key, d, WAVE);
        const uint32_t f2 = __shfl_up(flags, d, WAVE);
        const int32_t a0 = __shfl_up(mnx, d, WAVE), a1 = __shfl_up(mny, d, WAVE);
        const int32_t a2 = __shfl_up(mxx, d, WAVE), a3 = __shfl_up(mxy, d, WAVE);
        if (lane >= d && k2 == key) {
            flags |= f2;
            mnx = min(mnx, a0);
            mny = min(mny, a1);
            mxx = max(mxx, a2);
            mxy = max(mxy, a3);
        }
    }
    const int32_t knext = __shfl_down(key, 1, WAVE);
    const bool seg_end = lane == WAVE - 1 || knext != key;
    if (key >= 0 && seg_end && flags) {
        PathBox* b = &a.box[key];
        atomicOr(&b->flags, flags);
        if (mnx <= mxx) {
            atomicMin(&b->minx, mnx);
            atomicMin(&b->miny, mny);
            atomicMax(&b->maxx, mxx);
            atomicMax(&b->maxy, mxy);
        }
    }
}

__global__ void k_path_grid(const PathBox* box, PathGrid* grid, uint32_t* rows, int64_t n_paths, Counters* cnt) {
    int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= n_paths) return;
    PathBox b = box[p];
    PathGrid g;
    grid_from_box((b.flags & BOX_LINES) != 0, (b.flags & BOX_FULL) != 0, b.minx, b.miny, b.maxx, b.maxy, &g.tx0,
                  &g.ty0, &g.w, &g.h);
    if (b.flags & BOX_LINES) atomicMax(&cnt->max_w, (uint32_t)g.w);
    g.row_base = 0;
    grid[p] = g;
    rows[p] = (uint32_t)g.h + 1;  // + one row that carries the empty-path tile
}

struct LoadU32 {
    const uint32_t* p;
    __device__ uint32_t operator()(int64_t i) const { return p[i]; }
};
struct StoreU32 {
    uint32_t* p;
    __device__ void operator()(int64_t i, uint32_t excl, uint32_t) const { p[i] = excl; }
};
struct StoreRowBase {
    PathGrid* g;
    __device__ void operator()(int64_t i, uint32_t excl, uint32_t) const { g[i].row_base = excl; }
};

// A sort entry's value: bit 31 a tile-row crossing (its sign in the low byte).
// Else a run: the one that starts a line has no record (its replay starts where
// the line does), its value is the line; a later run's is its record's index
// with RT_REC set.  (Replaying
// every run from its line's start instead of keeping records measured slower:
// the extra steps cost more than the records' writes and gathers.)
constexpr uint32_t RT_REC = 0x40000000u;

// walk_line's run and entry counts (CountSink) without the walk, for the lines
// chain_walk_ok covers (rasterizer.rs:72-140).
// Each step moves one pixel along x or y, taking the smaller of the two
// crossing parameters, and the walk ends at the first parameter it takes
// that equals 1.  Each axis' parameters form a chain of their own (c, min(c +
// step, 1), ...) whatever the interleaving, so every value below 1 of both
// chains is taken before the end: the walk's last pixel before the end is its
// start moved by nx along x and ny along y (the chains' values below 1).  A
// step changes one tile coordinate by at most one, so the runs are 1 + the
// tile-x and tile-y changes, and the tile-row crossings are the tile-y changes
// plus one when the end-point snap (:118-121) lands in another tile row.
// Returns false for the lines it does not cover.
__device__ inline bool line_counts(V2 last, V2 point, uint32_t& runs, uint32_t& entries) {
    if (!chain_walk_ok(last, point)) return false;
    runs = entries = 0;
    if (veq(point, last)) return true;  // rasterizer.rs:73
    Dda d;
    dda_init(d, last, point);
    int32_t nx = 0, ny = 0;
    for (float c = d.col_t1; c < 1.0f; c = fminf(c + d.x_step, 1.0f)) nx++;
    for (float c = d.row_t1; c < 1.0f; c = fminf(c + d.y_step, 1.0f)) ny++;
    const int32_t x0 = d.x, y0 = d.y;
    const int32_t xl = x0 + (int32_t)d.x_dir * nx, yl = y0 + (int32_t)d.y_dir * ny;
    const uint32_t ty_changes = (uint32_t)abs((yl >> 3) - (y0 >> 3));
    runs = 1u + (uint32_t)abs((xl >> 3) - (x0 >> 3)) + ty_changes;
    const int32_t ty_end = (int32_t)f2i16(floorf(point.y)) >> 3;
    entries = runs + ty_changes + (ty_end != (yl >> 3) ? 1u : 0u);
    return true;
}

struct CountSink {
    uint32_t runs = 0, entries = 0;
    __device__ void run(int16_t, int16_t, bool, const Dda&) {
        runs++;
        entries++;
    }
    __device__ void crossing(int16_t, int16_t, int8_t) { entries++; }
    Counters* cnt;
    __device__ void limit() { atomicOr(&cnt->error, (uint32_t)ERR_FLATTEN); }
};

struct EmitSink {
    uint32_t line;
    uint32_t entry, run_idx;
    PathGrid g;
    uint32_t xbits;
    uint32_t* keys;
    uint32_t* vals;
    RunRec* recs;
    Counters* cnt;
    __device__ bool key_of(int16_t tx, int16_t ty, uint32_t* k) {
        uint32_t lx = (uint32_t)((int32_t)tx - g.tx0);
        uint32_t ly = (uint32_t)((int32_t)ty - g.ty0);
        if (lx >= (uint32_t)g.w || ly >= (uint32_t)g.h) {
            atomicOr(&cnt->error, (uint32_t)ERR_BBOX);
            return false;
        }
        *k = ((g.row_base + ly) << xbits) | lx;
        return true;
    }
    __device__ void run(int16_t tx, int16_t ty, bool start, const Dda& d) {
        uint32_t k = 0;
        key_of(tx, ty, &k);
        keys[entry] = k;
        if (start) {
            vals[entry] = line;
            entry++;
            return;
        }
        vals[entry] = run_idx | RT_REC;
        RunRec r;
        r.line = line;
        r.xy = (uint32_t)(uint16_t)d.x | ((uint32_t)(uint16_t)d.y << 16);
        r.row_t1 = d.row_t1;
        r.col_t1 = d.col_t1;
        recs[run_idx] = r;
        entry++;
        run_idx++;
    }
    __device__ void limit() {}
    __device__ void crossing(int16_t tx, int16_t ty, int8_t sign) {
        uint32_t k = 0;
        key_of(tx, ty, &k);
        keys[entry] = k;
        vals[entry] = 0x80000000u | (uint32_t)(uint8_t)sign;
        entry++;
    }
};

struct DdaArgs {
    const float4* lines;
    const uint32_t* line_path;
    int64_t n_lines;
    uint64_t* line_cnt;        // count pass: (records << 32) | entries per line, read by the emit pass
    const PathGrid* grid;
    uint32_t xbits;
    uint32_t* keys;
    uint32_t* vals;
    RunRec* recs;
    Counters* cnt;
    uint64_t* blk_entries;     // count pass: the entries of each block's lines
    uint64_t* blk_cnt;         // count pass: each block's (records << 32) | entries; emit pass: exclusive offsets
};


// Line offsets: the count pass leaves each line's packed (runs, entries)
// count and each block's sum; the blocks' sums are scanned, and the emit pass
// adds a block-local scan of its lines' counts (no device-wide scan over the
// lines).  A block's packed sum cannot carry between the halves: 256 lines of
// at most WALK_LIMIT entries each.
template <bool EMIT>
__global__ __launch_bounds__(256) void k_dda(DdaArgs a) {
    int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    __shared__ unsigned long long part[4];
    if (!EMIT) {
        unsigned long long e = 0, c = 0;
        if (l < a.n_lines) {
            float4 L = a.lines[l];
            CountSink s;
            s.cnt = a.cnt;
            if (!line_counts(mk(L.x, L.y), mk(L.z, L.w), s.runs, s.entries))
                walk_line(mk(L.x, L.y), mk(L.z, L.w), s);
            const uint32_t recs = s.runs ? s.runs - 1u : 0u;  // no record for the first run
            c = ((uint64_t)recs << 32) | s.entries;
            a.line_cnt[l] = c;
            e = s.entries;
        }
        // the 64-bit total of the block's entries (k_sum_u64 adds the blocks):
        // the packed block offsets are scanned in 32-bit halves, which wrap
        // silently past 2^32
        for (int o = 32; o > 0; o >>= 1) {
            e += __shfl_xor(e, o);
            c += __shfl_xor(c, o);
        }
        __shared__ unsigned long long cpart[4];
        if ((threadIdx.x & 63) == 0) {
            part[threadIdx.x >> 6] = e;
            cpart[threadIdx.x >> 6] = c;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            a.blk_entries[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
            a.blk_cnt[blockIdx.x] = cpart[0] + cpart[1] + cpart[2] + cpart[3];
        }
        return;
    }
    const uint64_t c = l < a.n_lines ? a.line_cnt[l] : 0ull;
    unsigned long long btotal;
    const uint64_t off = a.blk_cnt[blockIdx.x] +
                         block_excl_scan<256, unsigned long long>(c, OpAdd(), 0ull, part, &btotal);
    if (l >= a.n_lines) return;
    float4 L = a.lines[l];
    {
        EmitSink s;
        s.line = (uint32_t)l;
        s.entry = (uint32_t)off;
        s.run_idx = (uint32_t)(off >> 32);
        s.g = a.grid[a.line_path[l]];
        s.xbits = a.xbits;
        s.keys = a.keys;
        s.vals = a.vals;
        s.recs = a.recs;
        s.cnt = a.cnt;
        if (!walk_line_tiles(mk(L.x, L.y), mk(L.z, L.w), s)) walk_line(mk(L.x, L.y), mk(L.z, L.w), s);
    }
}

// *out += sum of a[0, n): a grid of at most 256 blocks, one atomic each.
__global__ __launch_bounds__(256) void k_sum_u64(const uint64_t* a, int64_t n, unsigned long long* out) {
    unsigned long long v = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        v += a[i];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __shared__ unsigned long long part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, part[0] + part[1] + part[2] + part[3]);
}

struct LoadU64 {
    const uint64_t* p;
    __device__ uint64_t operator()(int64_t i) const { return p[i]; }
};
struct StoreU64 {
    uint64_t* p;
    __device__ void operator()(int64_t i, uint64_t excl, uint64_t) const { p[i] = excl; }
};

// ------------------------------------------------ tile rows

// Inclusive scan restarting at every lane with head set.
__device__ inline int32_t seg_incl_scan(int32_t v, bool head) {
    const int lane = lane_id();
    int f = head ? 1 : 0;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        int32_t ov = __shfl_up(v, d, WAVE);
        int of = __shfl_up(f, d, WAVE);
        if (lane >= d && !f) v = ov + v;
        if (lane >= d) f |= of;
    }
    return v;
}

// The crossing sign of an entry's value (0 for a run).
__device__ inline int32_t entry_sign(uint32_t v) { return v >> 31 ? (int32_t)(int8_t)(v & 0xffu) : 0; }

// Each tile row's entries among the sorted ones and its crossing sum, in one
// pass over the entries.  A tile's entries are found again by the two tile
// kernels, from the keys of the 64 entries that a wave has in hand: tables of the
// distinct keys (their first entry, whether they hold a run, their crossing sum)
// took a device-wide scan, two zeroed arrays and a pass of their own, 410 us for
// the 20 million entries of 24 blobs against 36 us for this kernel.
constexpr int RTAB_ITEMS = 8;  // entries per lane
__global__ __launch_bounds__(256) void k_row_table(const uint32_t* keys, const uint32_t* vals, int64_t R,
                                                   uint32_t xbits, uint32_t* row_begin, uint32_t* row_end,
                                                   int32_t* row_sign) {
    const int lane = lane_id();
    const int64_t w = (int64_t)blockIdx.x * 4 + threadIdx.x / WAVE;
    int64_t i = w * (WAVE * RTAB_ITEMS) + lane;
    if (i - lane >= R) return;
    uint32_t left = i - lane > 0 ? keys[i - lane - 1] >> xbits : 0xffffffffu;  // the row before the wave's next entry
    uint32_t acc_row = 0;  // crossing sums of the row the last entries were in, per lane
    int32_t acc = 0;
    auto flush = [&]() {
        for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, WAVE);
        if (lane == 0 && acc) atomicAdd(&row_sign[acc_row], acc);
        acc = 0;
    };
#pragma unroll
    for (int k = 0; k < RTAB_ITEMS; k++, i += WAVE) {
        if (i - lane >= R) break;
        const bool valid = i < R;
        const uint32_t row = valid ? keys[i] >> xbits : 0xfffffffeu;
        const int32_t sg = valid ? entry_sign(vals[i]) : 0;
        uint32_t prev = __shfl_up(row, 1, WAVE);
        if (lane == 0) prev = left;
        const bool head = valid && row != prev;
        if (head) {
            row_begin[row] = (uint32_t)i;
            if (prev != 0xffffffffu) row_end[prev] = (uint32_t)i;
        }
        if (i == R - 1) row_end[row] = (uint32_t)R;
        const uint32_t r0 = __builtin_amdgcn_readfirstlane(row);
        if (__ballot(valid && row != r0) == 0) {  // one row
            if (r0 != acc_row) {
                if (__ballot(acc != 0)) flush();
                acc_row = r0;
            }
            acc += sg;
        } else if (__ballot(sg != 0)) {
            const int32_t sum = seg_incl_scan(sg, head || lane == 0);
            const uint32_t next = __shfl_down(row, 1, WAVE);
            if (valid && (lane == WAVE - 1 || next != row) && sum) atomicAdd(&row_sign[row], sum);
        }
        left = __shfl(row, WAVE - 1, WAVE);
    }
    if (__ballot(acc != 0)) flush();
}

// Per path: winding entering each tile row (the running sum of all earlier
// crossings, rasterizer.rs:253-260), the row -> path map, and the
// empty-path tile (rasterizer.rs:193-198: no increments still emits one
// all-zero tile at (0, 0)).  A wave per path, a lane per tile row: a thread per
// path took its rows one dependent load after another, 161 us for 24 paths of
// up to 600 rows against 14 now (10,000 paths of about 6 rows: 5.2 us).
constexpr int PR_WAVES = 4;  // paths per workgroup
__global__ __launch_bounds__(PR_WAVES * WAVE) void k_path_rows(const PathGrid* grid, int64_t n_paths,
                                                               const uint32_t* row_begin, const uint32_t* row_end,
                                                               const int32_t* row_sign, int32_t* row_wb,
                                                               uint32_t* row_path, uint64_t* row_cnt) {
    const int lane = lane_id();
    const int64_t p = blockIdx.x * (int64_t)PR_WAVES + threadIdx.x / WAVE;
    if (p >= n_paths) return;
    const PathGrid g = grid[p];
    int32_t running = 0;
    bool nonempty = false;
    for (int b = 0; b < g.h; b += WAVE) {
        const uint32_t row = g.row_base + (uint32_t)(b + lane);
        const bool valid = b + lane < g.h;
        const int32_t v = valid ? row_sign[row] : 0;
        const int32_t incl = wave_incl_scan(v, OpAdd());
        if (valid) {
            row_wb[row] = running + incl - v;
            row_path[row] = (uint32_t)p;
        }
        nonempty |= __ballot(valid && row_end[row] > row_begin[row]) != 0;
        running += __shfl(incl, WAVE - 1, WAVE);
    }
    if (lane == 0) {
        const uint32_t filler = g.row_base + (uint32_t)g.h;
        row_path[filler] = (uint32_t)p;
        row_cnt[filler] = nonempty ? 0ull : (1ull << 32);
    }
}

// ----------------------------------------- (c)(d)(e) tile rows, one wave each

struct TileArgs {
    const PathGrid* grid;
    const uint32_t* row_path;
    const uint32_t* row_begin;  // the row's entries
    const uint32_t* row_end;
    const int32_t* row_wb;
    int64_t n_rows;
    const uint32_t* keys;     // sorted entries
    const uint32_t* vals;
    uint32_t xbits;
    const RunRec* recs;
    const float4* lines;
    uint64_t* row_cnt;        // count pass output
    const uint64_t* row_off;  // emit pass input: (tiles << 32) | spans exclusive offsets
    uint32_t* long_rows;      // count pass output: the longest rows from the front, other long ones from the back
    uint32_t* n_long;         // [0] longest, [1] other long
    int16_t* tile_xy;
    uint8_t* tile_alpha;
    float* tile_cov;          // optional pre-quantisation coverage, 64 per tile
    int16_t* span_xy;
    uint16_t* span_w;
    Counters* cnt;
};

__device__ inline uint32_t rl(uint32_t v, int j) { return (uint32_t)__builtin_amdgcn_readlane((int)v, j); }

// The bins (rasterizer.rs:193-213) of a tile row's sorted entries, 64 at a time,
// one after another: the row's open bin and winding, and the previous tile.  All
// of it is uniform.  step(key, vals of the wave's entries, n of them) calls
// part(j0, j1) for each bin's entries that hold a run and tile(x) where a bin with
// runs ends (after its last part), span(x, width) before it where the gap to the
// previous tile is filled (rasterizer.rs:252-264).
struct RowBins {
    int32_t winding;       // after all entries so far
    bool open = false, open_run = false, have_prev = false;
    int32_t open_x = 0, open_w = 0;  // the open bin's x in the grid, the winding after its entries
    int32_t prev_x = 0, prev_w = 0;

    template <class Tile, class Span>
    __device__ void close(Tile&& tile, Span&& span) {
        if (open && open_run) {
            if (have_prev && open_x > prev_x + 1 && prev_w != 0) span(prev_x + 1, open_x - prev_x - 1);
            tile(open_x);
            have_prev = true;
            prev_x = open_x;
            prev_w = open_w;
        }
        open = false;
    }
    template <class Part, class Tile, class Span>
    __device__ void step(uint32_t key, uint32_t val, uint32_t n, uint32_t xmask, Part&& part, Tile&& tile,
                         Span&& span) {
        const int lane = lane_id();
        const bool valid = (uint32_t)lane < n;
        const uint64_t runs = __ballot(valid && !(val >> 31));
        const uint32_t before = __shfl_up(key, 1, WAVE);
        uint64_t heads = __ballot(valid && (lane == 0 || key != before));
        int32_t wsum = valid ? entry_sign(val) : 0;
        const bool cross = __ballot(wsum != 0) != 0;
        if (cross) wsum = wave_incl_scan(wsum, OpAdd());
        heads &= heads - 1;  // the starts after the first
        uint32_t j0 = 0;
        while (j0 < n) {
            const uint32_t j1 = heads ? (uint32_t)__builtin_ctzll(heads) : n;
            heads &= heads - 1;
            const int32_t x = (int32_t)(rl(key, (int)j0) & xmask);
            if (open && x != open_x) close(tile, span);
            if (!open) {
                open = true;
                open_run = false;
                open_x = x;
            }
            if (((runs >> j0) << (64u - (j1 - j0))) != 0) {
                open_run = true;
                part(j0, j1);
            }
            open_w = winding + (cross ? (int32_t)rl((uint32_t)wsum, (int)j1 - 1) : 0);
            j0 = j1;
        }
        winding = open_w;
    }
};

// Count pass of the tile stage: tiles and spans per tile row, one wave per row,
// RowBins' rules with a lane per entry: a tile starts at the first run of a bin,
// and the tile before it is the bin of the last run before the bin's entries (in
// the wave's 64 entries, or carried from the ones before).  (RowBins here, bin
// after bin in scalar code, measured 222 us against 143 on 24 blobs.)
constexpr int TC_ROWS = 4;   // rows per workgroup
constexpr uint32_t TR_LONG = 32 * WAVE, TR_LONGEST = 96 * WAVE;  // entries of a long row (see k_tile_rows)
constexpr int TC_AHEAD = 4;  // steps of 64 entries loaded ahead
__global__ __launch_bounds__(TC_ROWS * WAVE) void k_tile_counts(TileArgs a) {
    const int lane = lane_id();
    const uint64_t lt = lanemask_lt();
    const uint32_t xmask = (1u << a.xbits) - 1;
    for (int64_t row = (int64_t)blockIdx.x * TC_ROWS + threadIdx.x / WAVE; row < a.n_rows;
         row += (int64_t)gridDim.x * TC_ROWS) {
        const PathGrid G = a.grid[a.row_path[row]];
        if (row - (int64_t)G.row_base >= G.h) continue;  // the empty-path row (k_path_rows)
        const uint32_t eb = __builtin_amdgcn_readfirstlane(a.row_begin[row]);
        const uint32_t ee = __builtin_amdgcn_readfirstlane(a.row_end[row]);
        int32_t winding = __builtin_amdgcn_readfirstlane(a.row_wb[row]);
        uint32_t nt = 0, ns = 0;
        // the last tile before the entries in hand, and the bin they may continue
        bool have_prev = false, open_run = false;
        int32_t prev_x = 0, prev_w = 0, open_x = -1;
        auto load = [&](const uint32_t* p, uint32_t b, uint32_t none) {
            return b + (uint32_t)lane < ee ? p[b + (uint32_t)lane] : none;
        };
        auto step = [&](uint32_t b, uint32_t key, uint32_t v) {
            const int32_t x = (int32_t)(key & xmask);
            const uint32_t n = min((uint32_t)WAVE, ee - b);
            const bool valid = (uint32_t)lane < n, run = valid && !(v >> 31);
            int32_t w = valid ? entry_sign(v) : 0;
            w = winding + (__ballot(w != 0) ? wave_incl_scan(w, OpAdd()) : 0);
            const int32_t left_x = __shfl_up(x, 1, WAVE);
            const uint64_t heads = __ballot(valid && (lane == 0 || x != left_x)), runs = __ballot(run);
            const int my = 63 - __clzll((long long)(heads & (lt | (1ull << lane))));  // the start of my bin's entries
            // w after the bin that lane r's entry is in
            auto bin_end = [&](int r) {
                const uint64_t later = heads & (r == 63 ? 0ull : ~0ull << (r + 1));
                return later ? (int)__builtin_ctzll(later) - 1 : (int)n - 1;
            };
            const bool cont = (int32_t)rl((uint32_t)x, 0) == open_x;  // the first bin continues the one before
            const int32_t w0 = (int32_t)rl((uint32_t)w, bin_end(0));
            if (open_run && !cont) {  // it has ended: the last tile
                have_prev = true;
                prev_x = open_x;
                prev_w = winding;
            }
            const uint64_t below = (1ull << my) - 1ull;  // entries of earlier bins
            const bool starts = run && (runs & lt & ~below) == 0 && !(my == 0 && cont && open_run);
            const uint64_t before = runs & below;
            const int r = before ? 63 - __clzll((long long)before) : 0;
            const int32_t rx = __shfl(x, r, WAVE), rw = __shfl(w, bin_end(r), WAVE);
            const bool from_open = my > 0 && cont && open_run;
            const bool hp = before || from_open || have_prev;
            const int32_t px = before ? rx : (from_open ? open_x : prev_x);
            const int32_t pw = before ? rw : (from_open ? w0 : prev_w);
            nt += (uint32_t)__popcll(__ballot(starts));
            ns += (uint32_t)__popcll(__ballot(starts && hp && x > px + 1 && pw != 0));
            // the last bin stays open; the last tile before it
            const int last = (int)rl((uint32_t)my, (int)n - 1);
            if (last > 0) {
                const bool l_before = (runs & ((1ull << last) - 1ull)) != 0, l_open = cont && open_run;
                prev_x = (int32_t)rl((uint32_t)px, (int)n - 1);
                prev_w = (int32_t)rl((uint32_t)pw, (int)n - 1);
                have_prev = l_before || l_open || have_prev;
            }
            open_run = (runs >> last) != 0 || (last == 0 && cont && open_run);
            open_x = (int32_t)rl((uint32_t)x, (int)n - 1);
            winding = (int32_t)rl((uint32_t)w, (int)n - 1);
        };
        // TC_AHEAD steps' entries loaded together, the next ones while they are taken
        uint32_t key[TC_AHEAD], val[TC_AHEAD];
        auto load_all = [&](uint32_t b) {
#pragma unroll
            for (int k = 0; k < TC_AHEAD; k++) {
                key[k] = load(a.keys, b + (uint32_t)(k * WAVE), 0u);
                val[k] = load(a.vals, b + (uint32_t)(k * WAVE), 0x80000000u);
            }
        };
        load_all(eb);
        for (uint32_t b = eb; b < ee; b += TC_AHEAD * WAVE) {
            uint32_t ck[TC_AHEAD], cv[TC_AHEAD];
#pragma unroll
            for (int k = 0; k < TC_AHEAD; k++) {
                ck[k] = key[k];
                cv[k] = val[k];
            }
            load_all(b + TC_AHEAD * WAVE);
#pragma unroll
            for (int k = 0; k < TC_AHEAD; k++)
                if (b + (uint32_t)(k * WAVE) < ee) step(b + (uint32_t)(k * WAVE), ck[k], cv[k]);
        }
        if (lane == 0) {
            a.row_cnt[row] = ((uint64_t)nt << 32) | ns;
            if (ee - eb >= TR_LONGEST) a.long_rows[atomicAdd(&a.n_long[0], 1u)] = (uint32_t)row;
            else if (ee - eb >= TR_LONG) a.long_rows[a.n_rows - 1 - atomicAdd(&a.n_long[1], 1u)] = (uint32_t)row;
        }
    }
}

// Emit pass of the tile stage: one wave per tile row, walking the row's
// bins (rasterizer.rs:213-265) in key order.  The row's sort entries
// are taken TR_BLOCK at a time and each lane replays one run into LDS: its
// increments, and its bit in the `hit` words of the pixels it visits.  A run stays
// inside one 8x8 tile and its walk moves one pixel along one axis per step, always
// in the same direction along that axis, so it has at most 15 increments, at
// distinct pixels, and along it x + y (its directions along x and y alike) or
// x - y (unlike) moves by one per step: that is the increment's slot, which a pixel
// knows of itself, given the run's bit in the block's mask of alike ones.  No map
// from pixel to step is kept or read.  Each lane then owns a pixel of the tile and
// adds, for the set bits of
// its hit words among the tile's runs, in sorted order, the increments found
// there to its register sums, so every pixel's f32 sums follow the sorted order
// exactly (rasterizer.rs:221-228), with no read-modify-write through LDS.  At
// the end of a tile the row carry is folded across the 8 lanes of each pixel row
// in x order, the alphas quantised and stored (rasterizer.rs:230-250), and a span
// is written where the previous tile of the row is more than one tile to the
// left and the winding after it is non-zero (rasterizer.rs:252-264).
//
// Bound: VALU issue of the replays and, for a row alone on its SIMD, the chain of
// dependent loads (entry, record, line) and steps.  So: 64 runs replayed at once
// (a wave's worth; 32 left half the lanes idle), 8.2 KB of LDS per wave instead
// of 6 KB for 32 runs (no 64-byte pixel map to clear, fill and search per run), a
// pixel visits only the runs that hit it (the most hits of a tile's pixels, about
// 4, instead of its runs, about 11), the next block's records and lines load
// while this one is added, and the carry moves by DPP instead of eight LDS
// permutes.
// Measured against the 32-run kernel with maps: 120 -> 43 us on a line of 61
// glyphs, 422 -> 180 us on 10,000 glyphs (VALU-bound), 2,684 ->
// 560 us on 24 star blobs of 1,000-20,000 cubics.
constexpr int TR_SLOTS = 15;  // increments per run
constexpr int TR_BLOCK = WAVE;  // runs replayed per block

// The first tile row of a workgroup of a row kernel (rows first_row +
// k * gridDim.x).  Neighbouring tile rows gather the same lines and run
// records: runs of ROW_CHUNK consecutive rows go to the workgroups of one XCD
// (workgroups are dealt round-robin over the eight XCDs by id), so that the
// second gather hits that XCD's L2; the runs themselves go round-robin over
// the XCDs, which keeps their loads even.  Grids that are a multiple of
// 8 * ROW_CHUNK only (row_grid); others take rows in id order.
constexpr int ROW_CHUNK = 16;
__device__ inline int64_t xcd_first_row() {
    if (gridDim.x % (8u * ROW_CHUNK) != 0) return blockIdx.x;
    const int64_t j = blockIdx.x / 8u;  // the workgroup's place among its XCD's
    return ((j / ROW_CHUNK) * 8 + (int64_t)(blockIdx.x % 8u)) * ROW_CHUNK + j % ROW_CHUNK;
}
static inline uint32_t row_grid(int64_t rows, int64_t cap) {
    int64_t g = std::min<int64_t>(rows, cap);
    if (g >= 8 * ROW_CHUNK) g -= g % (8 * ROW_CHUNK);
    return (uint32_t)g;
}

// The increments of a run from the DDA state at its first one (p0: that
// increment's start point) into their slots from inc[0] on, `dir` apart, and the
// run's bit into the hit words of its pixels.  FAST: every active lane's line is
// one that FastWalk covers.  The pixel within the tile is two nibbles (y above x);
// leaving 0..7 on either axis sets a nibble's top bit.
template <bool FAST>
__device__ inline void tr_replay_steps(float2* inc, int dir, uint32_t* hit, uint32_t bit, Dda& d, V2 p0, bool finite,
                                       Counters* cnt) {
    uint32_t at = (uint32_t)(((d.y & 7) << 4) | (d.x & 7));
    const uint32_t xd = (uint32_t)(int32_t)d.x_dir, yd = (uint32_t)((int32_t)d.y_dir * 16);
    auto put = [&](float area, float height) {
        *inc = make_float2(area, height);
        inc += dir;
        atomicOr(&hit[at - ((at >> 4) << 3)], bit);
    };
    if constexpr (FAST) {
        FastWalk w;
        w.init(d, p0);
        for (;;) {  // (at most 15 steps: each moves one pixel on, the same way along its axis)
            float area, height;
            bool y;
            const bool end = w.step(area, height, y);
            put(area, height);
            at += y ? yd : xd;
            if (end || (at & 0x88u)) break;
        }
        return;
    }
    bool ended = false;
    for (int k = 0; k < TR_SLOTS; k++) {
        float area, height;
        dda_increment_carried(d, p0, finite, area, height);
        put(area, height);
        at += d.row_t1 < d.col_t1 ? yd : xd;
        if (dda_step(d) || (at & 0x88u)) {
            ended = true;
            break;
        }
    }
    if (!ended) atomicOr(&cnt->error, (uint32_t)ERR_REPLAY);
}

// A wave's LDS accesses before and after this point stay in their order (they
// are executed in order; this holds the compiler to it).
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int CTRL>
__device__ inline float dpp_f(float old, float v) {
    return __uint_as_float(dpp<CTRL>(__float_as_uint(old), __float_as_uint(v)));
}

// PAIRED: the long rows, two waves each, a block apart: one replays block i while
// the other adds block i - 1 and writes its tiles, one barrier per block.  Rows vary
// (24 blobs: 1,480 runs on average, 11,900 at most), a row's blocks run one after
// another, and a wave alone on its SIMD issues an instruction only every 9 cycles:
// with a wave per row the longest row took as long as the whole kernel, at 1.6
// waves per SIMD on average.  The longest of them start first.  The other rows, a
// wave each, run in a launch beside it.
struct TrBuf {
    float2 inc[TR_BLOCK * TR_SLOTS];
    uint32_t hit[2][64];       // pixel p, bit j: run 32 w + j visits p
    unsigned long long alike;  // the runs whose slots are x + y
};

template <bool PAIRED>
__global__ __launch_bounds__(PAIRED ? 2 * WAVE : WAVE) void k_tile_rows(TileArgs a, uint32_t n_longest) {
    __shared__ TrBuf buf[PAIRED ? 2 : 1];
    const int lane = threadIdx.x & (WAVE - 1);
    // Lane -> pixel: 16 lanes hold two pixel rows interleaved, so that a move of
    // two lanes is the next pixel of the same row and the first two lanes, which
    // have no source, keep the carry.
    const uint32_t px = (uint32_t)(lane >> 1) & 7u, py = (uint32_t)((lane >> 4) << 1) | (uint32_t)(lane & 1);
    const uint32_t pix = (py << 3) | px, slot_alike = px + py, slot_unlike = px + 7u - py;
    const uint32_t xmask = (1u << a.xbits) - 1;
    const bool replays = !PAIRED || threadIdx.x < WAVE, adds = !PAIRED || threadIdx.x >= WAVE;
    int64_t row = xcd_first_row();
    if (PAIRED) row = a.long_rows[blockIdx.x < n_longest ? blockIdx.x : a.n_rows - 1 - (blockIdx.x - n_longest)];
    for (; row < a.n_rows; row += PAIRED ? a.n_rows : (int64_t)gridDim.x) {
        const PathGrid G = a.grid[a.row_path[row]];
        if (row - (int64_t)G.row_base >= G.h) continue;  // the empty-path row (k_path_out)
        const uint32_t eb = __builtin_amdgcn_readfirstlane(a.row_begin[row]);
        const uint32_t ee = __builtin_amdgcn_readfirstlane(a.row_end[row]);
        if (ee <= eb || (ee - eb >= TR_LONG) != PAIRED) continue;
        const int32_t ty = G.ty0 + (int32_t)(row - (int64_t)G.row_base);
        const uint64_t off = a.row_off[row];
        const uint32_t row_tiles = (uint32_t)(off >> 32), row_spans = (uint32_t)off;
        RowBins bins;
        bins.winding = __builtin_amdgcn_readfirstlane(a.row_wb[row]);
        float carry = 0.0f;  // of the lane's pixel row, in its first lane
        uint32_t nt = 0, ns = 0;
        float pa = 0.0f, ph = 0.0f;  // this pixel's sums of the open tile
        uint32_t h0 = 0, h1 = 0;     // this pixel's hit words of the block
        uint64_t alike = 0;
        const float2* inc = nullptr;
        // two hits at a time: their reads are in flight together
        auto add_runs = [&](uint32_t h, uint32_t al, uint32_t lo, uint32_t hi, const float2* incs) {
            uint32_t m = h & (0xffffffffu << lo) & (0xffffffffu >> (32u - hi));
            auto at = [&](uint32_t r) {
                return incs[r * (uint32_t)TR_SLOTS + ((al >> r) & 1u ? slot_alike : slot_unlike)];
            };
            while (m) {
                const uint32_t r1 = (uint32_t)__ffs((int)m) - 1u;
                m &= m - 1u;
                const uint32_t r2 = m ? (uint32_t)__ffs((int)m) - 1u : r1;
                const float2 v1 = at(r1), v2 = at(r2);
                pa = pa + v1.x;
                ph = ph + v1.y;
                if (m) {
                    pa = pa + v2.x;
                    ph = ph + v2.y;
                }
                m &= m - 1u;
            }
        };
        // a bin's runs of this block, added in sorted order
        auto part = [&](uint32_t j0, uint32_t j1) {
            if (j0 < 32u) add_runs(h0, (uint32_t)alike, j0, min(j1, 32u), inc);
            if (j1 > 32u)
                add_runs(h1, (uint32_t)(alike >> 32), j0 > 32u ? j0 - 32u : 0u, j1 - 32u, inc + 32 * TR_SLOTS);
        };
        auto span = [&](int32_t x, int32_t w) {
            if (lane == 0) {
                const uint32_t si = row_spans + ns;
                a.span_xy[2 * si] = (int16_t)((G.tx0 + x) * TILE);
                a.span_xy[2 * si + 1] = (int16_t)(ty * TILE);
                a.span_w[si] = (uint16_t)((uint16_t)w * (uint16_t)TILE);
            }
            ns++;
        };
        int32_t txy = 0;
        auto store_xy = [&](uint32_t n) {  // of the last n tiles
            if ((uint32_t)lane < n) {
                int16_t* xy = a.tile_xy + 2 * (size_t)(row_tiles + nt - n + (uint32_t)lane);
                xy[0] = (int16_t)txy;
                xy[1] = (int16_t)(ty * TILE);
            }
        };
        auto tile = [&](int32_t x) {
            // (d)(e) the fold along each pixel row: after k moves the lanes of
            // pixels 0..k hold ((carry + h0) + h1) ..., the later ones not yet
            float mine = carry, t = carry + ph;
#pragma unroll
            for (int k = 1; k < TILE; k++) {
                mine = dpp_f<DPP_ROW_SHR2>(carry, t);
                t = mine + ph;
            }
            carry = dpp_f<DPP_ROW_ROR2>(t, t);
            const float cov = fabsf(mine + pa);
            const uint32_t ti = row_tiles + nt;
            if (a.tile_cov) a.tile_cov[(size_t)ti * 64 + pix] = fminf(cov, 1.0f);
            a.tile_alpha[(size_t)ti * 64 + pix] = (uint8_t)(uint32_t)fminf(cov * 256.0f, 255.0f);
            pa = 0.0f;
            ph = 0.0f;
            // the tiles' coordinates wait in lanes, stored 64 at a time
            if (lane == (int)(nt & (WAVE - 1))) txy = (G.tx0 + x) * TILE;
            nt++;
            if ((nt & (WAVE - 1)) == 0) store_xy(WAVE);
        };
        // the entries of a block, their records and lines
        auto load = [&](const uint32_t* p, uint32_t b, uint32_t none) {
            return b + (uint32_t)lane < ee ? p[b + (uint32_t)lane] : none;
        };
        auto load_rec = [&](uint32_t v) {  // (bit 31 of its line: the line's first run)
            if ((v >> 30) == 1u) return a.recs[v & (RT_REC - 1u)];
            return RunRec{v | 0x80000000u, 0, 0.0f, 0.0f};
        };
        auto load_line = [&](uint32_t v, const RunRec& r) {
            return v >> 31 ? make_float4(0, 0, 0, 0) : a.lines[r.line & 0x7fffffffu];
        };
        // each level of a block's loads has a block's time: entries three blocks
        // ahead, records two, lines one
        uint32_t k1 = load(a.keys, eb, 0u), v1 = load(a.vals, eb, 0x80000000u);
        uint32_t k2 = load(a.keys, eb + TR_BLOCK, 0u), v2 = load(a.vals, eb + TR_BLOCK, 0x80000000u);
        uint32_t k3 = load(a.keys, eb + 2 * TR_BLOCK, 0u), v3 = load(a.vals, eb + 2 * TR_BLOCK, 0x80000000u);
        RunRec r1{}, r2{};
        float4 l1{};
        if (replays) {
            r1 = load_rec(v1);
            r2 = load_rec(v2);
            l1 = load_line(v1, r1);
        }
        uint32_t key = 0, v = 0, key0 = 0, v0 = 0;  // of the block replayed, and of the one before
        const uint32_t n_blk = (ee - eb + TR_BLOCK - 1) / TR_BLOCK;
        for (uint32_t i = 0; i < n_blk + (PAIRED ? 1u : 0u); i++) {
            const uint32_t b = eb + i * TR_BLOCK;
            key0 = key;
            v0 = v;
            key = k1;
            v = v1;
            k1 = k2;
            v1 = v2;
            k2 = k3;
            v2 = v3;
            k3 = load(a.keys, b + 3 * TR_BLOCK, 0u);
            v3 = load(a.vals, b + 3 * TR_BLOCK, 0x80000000u);
            if (replays && i < n_blk) {
                // (c) replay the block's entries, one run per lane
                TrBuf& B = buf[PAIRED ? i & 1u : 0u];
                const RunRec r = r1;
                const float4 L = l1;
                r1 = r2;
                l1 = load_line(v1, r1);
                r2 = load_rec(v2);
                B.hit[0][lane] = 0;
                B.hit[1][lane] = 0;
                wave_lds_order();
                bool al = false;
                if (!(v >> 31)) {
                    Dda d;
                    const V2 last = mk(L.x, L.y), point = mk(L.z, L.w);
                    if (r.line >> 31) {
                        dda_init(d, last, point);
                    } else {
                        dda_consts(d, last, point);
                        d.x = (int16_t)(r.xy & 0xffffu);
                        d.y = (int16_t)(r.xy >> 16);
                        d.row_t1 = r.row_t1;
                        d.col_t1 = r.col_t1;
                        d.t0 = 0.0f;
                        dda_step(d);
                    }
                    const bool finite = line_finite(last, point);
                    const V2 p0 = dda_point(d, d.t0);
                    // (a direction is 0 only where a coordinate is not finite: that axis takes no step)
                    al = d.x_dir == d.y_dir || d.x_dir == 0 || d.y_dir == 0;
                    const int dir = d.x_dir ? d.x_dir : d.y_dir;
                    float2* out = B.inc + lane * TR_SLOTS + (al ? (d.x & 7) + (d.y & 7) : (d.x & 7) + 7 - (d.y & 7));
                    uint32_t* hw = B.hit[lane >> 5];
                    const uint32_t bit = 1u << (lane & 31);
                    if (__ballot(!fast_walk_ok(last, point)) == 0) tr_replay_steps<true>(out, dir, hw, bit, d, p0, finite, a.cnt);
                    else tr_replay_steps<false>(out, dir, hw, bit, d, p0, finite, a.cnt);
                }
                alike = __ballot(al);
                if (PAIRED && lane == 0) B.alike = alike;
                wave_lds_order();
            }
            if (adds && (!PAIRED || i > 0)) {
                const TrBuf& B = buf[PAIRED ? (i - 1u) & 1u : 0u];
                inc = B.inc;
                h0 = B.hit[0][pix];
                h1 = B.hit[1][pix];
                if (PAIRED) {
                    const unsigned long long w = B.alike;
                    alike = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(w >> 32)) << 32) |
                            (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)w);
                }
                const uint32_t b0 = PAIRED ? b - TR_BLOCK : b;
                bins.step(PAIRED ? key0 : key, PAIRED ? v0 : v, min((uint32_t)TR_BLOCK, ee - b0), xmask, part, tile,
                          span);
                wave_lds_order();
            }
            if (PAIRED) __syncthreads();
        }
        if (adds) {
            bins.close(tile, span);
            store_xy(nt & (WAVE - 1));
        }
    }
}

// ------------------------------------------- unordered tile stage (batched)
// For the large paths the batched pipeline hands on: instead of the radix
// sort, the sort entries are bucketed by (tile row, window of UW tiles) with
// no order inside a bucket, and each window's runs are replayed into LDS sums
// with float atomics, in arrival order — alpha within 1 LSB of the ordered
// result where a sum sits on a quantisation boundary, as in the dense kernels;
// the tile and span sets, which are integer, are exact.  One workgroup per tile
// row walks the row's windows left to right, carrying the winding, the last
// tile and the per-pixel-row height carry across them.
constexpr int UW = 32;   // tiles per window
constexpr int UWS = 65;  // accumulator slots per tile's sums (one of padding)
static_assert(UW <= WAVE && UW % 32 == 0, "a window is at most one wave of tiles, in 32-bit occupancy words");

struct LoadNWin {
    const PathGrid* g;
    __device__ uint32_t operator()(int64_t p) const { return (uint32_t)g[p].h * (((uint32_t)g[p].w + UW - 1) / UW); }
};

// row -> path and the row's first window bucket (a wave per path, as k_path_rows)
__global__ __launch_bounds__(PR_WAVES * WAVE) void k_rows_setup(const PathGrid* grid, int64_t n_paths,
                                                                const uint32_t* pwbase, uint32_t* row_path,
                                                                uint32_t* row_wbase) {
    const int64_t p = blockIdx.x * (int64_t)PR_WAVES + threadIdx.x / WAVE;
    if (p >= n_paths) return;
    const PathGrid g = grid[p];
    const uint32_t nwin = ((uint32_t)g.w + UW - 1) / UW;
    for (int r = lane_id(); r <= g.h; r += WAVE) {  // the last one is the empty-path row
        row_path[g.row_base + (uint32_t)r] = (uint32_t)p;
        row_wbase[g.row_base + (uint32_t)r] = pwbase[p] + (uint32_t)r * nwin;
    }
}

__device__ inline uint32_t entry_bucket(uint32_t key, uint32_t xbits, const uint32_t* row_wbase) {
    return row_wbase[key >> xbits] + ((key & ((1u << xbits) - 1u)) / UW);
}

// Bucketing: each workgroup takes BK_ITEMS entries per thread, consecutive
// entries on consecutive lanes.  The entries are in emission order (the runs
// and crossings of neighbouring lines along a contour), so consecutive ones
// mostly share a bucket: in each wave only the first lane of a run of equal
// buckets inserts the run's length into an LDS hash table (open addressing,
// room for every entry), and a bucket gets one global atomic per workgroup.
constexpr int BK_NT = 256;
constexpr int BK_ITEMS = 8;
constexpr int BK_HBITS = 11;
constexpr int BK_HS = 1 << BK_HBITS;  // == BK_NT * BK_ITEMS
constexpr uint32_t BK_EMPTY = 0xffffffffu;
static_assert(BK_HS >= BK_NT * BK_ITEMS, "the bucket hash must hold every entry of a workgroup");

struct BucketLds {
    uint32_t key[BK_HS];
    uint32_t cnt[BK_HS];
    uint32_t aux[BK_HS];  // histogram: the bucket's tile row; scatter: the workgroup's first slot in the bucket
    int32_t sgn[BK_HS];   // histogram: the bucket's crossing sum
};

__device__ inline uint64_t lanemask_le() { return lanemask_lt() | (1ull << (threadIdx.x & (WAVE - 1))); }

// Inserts n entries of bucket b; returns the bucket's slot and the first
// entry's rank within the workgroup.  Terminates: the table has room for
// every entry of the workgroup, hence for every distinct bucket.
__device__ inline uint32_t bucket_insert(BucketLds& h, uint32_t b, uint32_t n, uint32_t* rank) {
    uint32_t slot = (b * 2654435761u) >> (32 - BK_HBITS);
    for (;;) {
        const uint32_t old = atomicCAS(&h.key[slot], BK_EMPTY, b);
        if (old == BK_EMPTY || old == b) {
            *rank = atomicAdd(&h.cnt[slot], n);
            return slot;
        }
        slot = (slot + 1) & (BK_HS - 1);
    }
}

// One wave's 64 consecutive entries (the valid ones a prefix of the lanes):
// the slot of each entry's bucket and its rank within the workgroup.
__device__ inline void bucket_wave(BucketLds& h, bool valid, uint32_t b, uint32_t* slot, uint32_t* rank,
                                   uint32_t* head_row, uint32_t row) {
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t prev = __shfl_up(b, 1, WAVE);
    const bool head = valid && (lane == 0 || prev != b);
    const uint64_t hm = __ballot(head);
    const int nvalid = __popcll(__ballot(valid));
    uint32_t sl = 0, rk = 0;
    if (head) {
        const uint64_t above = hm & ~lanemask_le();
        const int next = above ? __ffsll((unsigned long long)above) - 1 : nvalid;
        sl = bucket_insert(h, b, (uint32_t)(next - lane), &rk);
        if (head_row) head_row[sl] = row;
    }
    const int hl = valid ? 63 - __clzll((long long)(hm & lanemask_le())) : lane;
    *slot = __shfl(sl, hl, WAVE);
    *rank = __shfl(rk, hl, WAVE) + (uint32_t)(lane - hl);
}

template <bool HIST>
__device__ inline void bucket_init(BucketLds& h) {
    for (int k = threadIdx.x; k < BK_HS; k += BK_NT) {
        h.key[k] = BK_EMPTY;
        h.cnt[k] = 0;
        if (HIST) h.sgn[k] = 0;
    }
}

// Bucket sizes, and the crossing sum of every tile row.
__global__ __launch_bounds__(BK_NT) void k_bucket_hist(const uint32_t* keys, const uint32_t* vals, int64_t R,
                                                       uint32_t xbits, const uint32_t* row_wbase, uint32_t* bcnt,
                                                       int32_t* row_sign) {
    __shared__ BucketLds h;
    bucket_init<true>(h);
    __syncthreads();
    const int64_t e0 = (int64_t)blockIdx.x * BK_NT * BK_ITEMS + threadIdx.x;
    uint32_t kk[BK_ITEMS], vv[BK_ITEMS];
#pragma unroll
    for (int u = 0; u < BK_ITEMS; u++) {
        const int64_t e = e0 + (int64_t)u * BK_NT;
        kk[u] = e < R ? keys[e] : 0u;
        vv[u] = e < R ? vals[e] : 0u;
    }
#pragma unroll
    for (int u = 0; u < BK_ITEMS; u++) {
        const bool valid = e0 + (int64_t)u * BK_NT < R;
        const uint32_t row = kk[u] >> xbits;
        const uint32_t b = valid ? entry_bucket(kk[u], xbits, row_wbase) : BK_EMPTY;
        uint32_t slot, rank;
        bucket_wave(h, valid, b, &slot, &rank, h.aux, row);
        if (valid && (vv[u] >> 31)) {
            const int sg = (int)(int8_t)(vv[u] & 0xffu);
            if (sg) atomicAdd(&h.sgn[slot], sg);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < BK_HS; k += BK_NT) {
        if (h.key[k] == BK_EMPTY) continue;
        atomicAdd(&bcnt[h.key[k]], h.cnt[k]);
        if (h.sgn[k]) atomicAdd(&row_sign[h.aux[k]], h.sgn[k]);
    }
}

// Scatter into the buckets: one cursor atomic per bucket per workgroup.
__global__ __launch_bounds__(BK_NT) void k_bucket_scatter(const uint32_t* keys, const uint32_t* vals, int64_t R,
                                                          uint32_t xbits, const uint32_t* row_wbase, uint32_t* bcur,
                                                          uint32_t* okeys, uint32_t* ovals) {
    __shared__ BucketLds h;
    bucket_init<false>(h);
    __syncthreads();
    const int64_t e0 = (int64_t)blockIdx.x * BK_NT * BK_ITEMS + threadIdx.x;
    uint32_t kk[BK_ITEMS], vv[BK_ITEMS], slot[BK_ITEMS], rank[BK_ITEMS];
#pragma unroll
    for (int u = 0; u < BK_ITEMS; u++) {
        const int64_t e = e0 + (int64_t)u * BK_NT;
        kk[u] = e < R ? keys[e] : 0u;
        vv[u] = e < R ? vals[e] : 0u;
    }
#pragma unroll
    for (int u = 0; u < BK_ITEMS; u++) {
        const bool valid = e0 + (int64_t)u * BK_NT < R;
        const uint32_t b = valid ? entry_bucket(kk[u], xbits, row_wbase) : BK_EMPTY;
        bucket_wave(h, valid, b, &slot[u], &rank[u], nullptr, 0u);
        if (!valid) slot[u] = BK_EMPTY;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < BK_HS; k += BK_NT)
        if (h.key[k] != BK_EMPTY) h.aux[k] = atomicAdd(&bcur[h.key[k]], h.cnt[k]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BK_ITEMS; u++) {
        if (slot[u] != BK_EMPTY) {
            const uint32_t o = h.aux[slot[u]] + rank[u];
            okeys[o] = kk[u];
            ovals[o] = vv[u];
        }
    }
}

// Per path: the winding entering each row, and the empty-path tile (a wave per
// path, as k_path_rows).
__global__ __launch_bounds__(PR_WAVES * WAVE) void k_path_rows_u(const PathGrid* grid, int64_t n_paths,
                                                                 const uint32_t* pwbase, const uint32_t* bbeg,
                                                                 const int32_t* row_sign, int32_t* row_wb,
                                                                 uint64_t* row_cnt) {
    const int lane = lane_id();
    const int64_t p = blockIdx.x * (int64_t)PR_WAVES + threadIdx.x / WAVE;
    if (p >= n_paths) return;
    const PathGrid g = grid[p];
    int32_t running = 0;
    for (int b = 0; b < g.h; b += WAVE) {
        const uint32_t row = g.row_base + (uint32_t)(b + lane);
        const bool valid = b + lane < g.h;
        const int32_t v = valid ? row_sign[row] : 0;
        const int32_t incl = wave_incl_scan(v, OpAdd());
        if (valid) row_wb[row] = running + incl - v;
        running += __shfl(incl, WAVE - 1, WAVE);
    }
    if (lane == 0) {
        const uint32_t nwin = ((uint32_t)g.w + UW - 1) / UW;
        const bool nonempty = bbeg[pwbase[p] + (uint32_t)g.h * nwin] > bbeg[pwbase[p]];
        row_cnt[g.row_base + (uint32_t)g.h] = nonempty ? 0ull : (1ull << 32);
    }
}

struct RowTileArgs {
    const PathGrid* grid;
    const uint32_t* row_path;
    const uint32_t* row_wbase;
    const int32_t* row_wb;
    int64_t n_rows;
    const uint32_t* bbeg;  // bucket starts (n_buckets + 1)
    const uint32_t* keys;  // bucketed entries
    const uint32_t* vals;
    uint32_t xbits;
    const RunRec* recs;
    const float4* lines;
    uint64_t* row_cnt;        // count pass output
    const uint64_t* row_off;  // emit pass input
    int16_t* tile_xy;
    uint8_t* tile_alpha;
    float* tile_cov;  // optional pre-quantisation coverage, 64 per tile
    int16_t* span_xy;
    uint16_t* span_w;
    Counters* cnt;
};

constexpr int RT_NW = 4;
constexpr int RT_NT = RT_NW * WAVE;
constexpr int RT_ROWS = TILE / RT_NW;  // pixel rows whose carry each wave takes
static_assert(RT_ROWS * RT_NW == TILE && RT_ROWS <= 2, "the carry takes one or two pixel rows per wave");
constexpr int RT_U = 2;  // entries per thread whose loads are issued together

// The window's per-pixel sums are fixed point (fx_of: 64-bit integers in units of
// 2^-30): the sums of the increments, each truncated at 2^-30, are then exact, so
// that the decoded f32 sum is the correctly rounded sum of the increments,
// independent of arrival order.  A window of a full-range path (coordinates that may
// be huge or non-finite) or with 2^22 entries or more keeps f32 atomics in the slots'
// low words instead.
constexpr uint32_t RT_FX_MAX_ENTRIES = 1u << 22;  // (a pixel takes at most one increment per run)

template <bool EMIT>
struct RowLds {
    long long acc_a[EMIT ? UW * UWS : 2];  // tile t, pixel p at t * UWS + p
    long long acc_h[EMIT ? UW * UWS : 2];
    int32_t tsign[UW];
    uint32_t occ[UW / 32];
    uint8_t tlist[UW];  // the window's occupied tiles in x order
    float rtot[EMIT ? UW * 8 : 1];  // per (occupied tile, pixel row): height total, then incoming carry
    uint32_t nt, ns, nocc;
};

// The increments of a run into a window's fixed-point sums (xb: the first slot of
// its tile).  Such a window's path is within +-HUGE_COORD, so FastWalk covers its
// lines.
template <bool WIDE, bool EMIT>
__device__ inline void rt_replay_fx(RowLds<EMIT>& s, const Dda& d, V2 p0, uint32_t xb, uint32_t at, uint32_t xd,
                                    uint32_t yd) {
    FastWalk w;
    w.init(d, p0);
    for (;;) {  // (at most 15 steps: each moves one pixel on, the same way along its axis)
        float area, height;
        bool y;
        const bool end = w.step(area, height, y);
        const uint32_t px = xb + at - ((at >> 4) << 3);
        atomicAdd(reinterpret_cast<unsigned long long*>(&s.acc_a[px]), fx_of<WIDE>(area));
        atomicAdd(reinterpret_cast<unsigned long long*>(&s.acc_h[px]), fx_of<WIDE>(height));
        at += y ? yd : xd;
        if (end || (at & 0x88u)) break;
    }
}

// Replays a run (x: its tile within the window) into the window's LDS sums, in
// arrival order.
template <bool EMIT>
__device__ inline void rt_replay_run(RowLds<EMIT>& s, uint32_t x, const RunRec& rr, const float4& L, bool fx,
                                     Counters* cnt) {
    Dda d;
    const V2 last = mk(L.x, L.y), point = mk(L.z, L.w);
    if (rr.line >> 31) {
        dda_init(d, last, point);
    } else {
        dda_consts(d, last, point);
        d.x = (int16_t)(rr.xy & 0xffffu);
        d.y = (int16_t)(rr.xy >> 16);
        d.row_t1 = rr.row_t1;
        d.col_t1 = rr.col_t1;
        d.t0 = 0.0f;
        dda_step(d);
    }
    V2 p0 = dda_point(d, d.t0);
    // the pixel within the run's tile as two nibbles, y above x: leaving 0..7 on
    // either axis sets a nibble's top bit
    uint32_t at = (uint32_t)(((d.y & 7) << 4) | (d.x & 7));
    const uint32_t xd = (uint32_t)(int32_t)d.x_dir, yd = (uint32_t)((int32_t)d.y_dir * 16);
    const uint32_t xb = x * (uint32_t)UWS;
    if (fx) {  // (a step along an axis is 1 / the line's length there)
        if (__ballot(fminf(d.x_step, d.y_step) < 1.0f / FX_NARROW_PX) == 0) rt_replay_fx<false>(s, d, p0, xb, at, xd, yd);
        else rt_replay_fx<true>(s, d, p0, xb, at, xd, yd);
        return;
    }
    const bool finite = line_finite(last, point);
    bool ended = false;
    for (int k = 0; k < 16; k++) {
        float area, height;
        dda_increment_carried(d, p0, finite, area, height);
        const uint32_t px = xb + at - ((at >> 4) << 3);
        atomicAdd(reinterpret_cast<float*>(&s.acc_a[px]), area);
        atomicAdd(reinterpret_cast<float*>(&s.acc_h[px]), height);
        at += d.row_t1 < d.col_t1 ? yd : xd;
        if (dda_step(d) || (at & 0x88u)) {
            ended = true;
            break;
        }
    }
    if (!ended) atomicOr(&cnt->error, (uint32_t)ERR_REPLAY);
}

// RT_U entries per thread of a window (entries e0 + u * RT_NT), with their
// run records and lines, loaded level by level (each level's loads in flight
// together).  The emit pass loads the next window's first batch while the
// current window's ranks, carries and quantisation run.
struct RtBatch {
    uint32_t kk[RT_U], vv[RT_U];
    RunRec rr[RT_U];
    float4 L[RT_U];
};
__device__ inline void rt_load_keys(RtBatch& b, const RowTileArgs& a, uint32_t e0, uint32_t ee) {
#pragma unroll
    for (int u = 0; u < RT_U; u++) {
        const uint32_t e = e0 + (uint32_t)(u * RT_NT);
        b.kk[u] = e < ee ? a.keys[e] : 0u;
        b.vv[u] = e < ee ? a.vals[e] : 0x80000000u;
    }
}
// An entry's value: bit 31 a crossing (its sign in the low byte); else a
// run record's index with RT_REC set, or the line whose first run it is.
__device__ inline void rt_load_recs(RtBatch& b, const RowTileArgs& a) {
#pragma unroll
    for (int u = 0; u < RT_U; u++) {
        b.rr[u].line = (b.vv[u] & (RT_REC - 1u)) | 0x80000000u;  // a line's first run: replayed from its start
        b.rr[u].xy = 0;
        b.rr[u].row_t1 = b.rr[u].col_t1 = 0.0f;
        if ((b.vv[u] >> 30) == 1u) b.rr[u] = a.recs[b.vv[u] & (RT_REC - 1u)];
    }
}
__device__ inline void rt_load_lines(RtBatch& b, const RowTileArgs& a) {
#pragma unroll
    for (int u = 0; u < RT_U; u++)
        b.L[u] = !(b.vv[u] >> 31) ? a.lines[b.rr[u].line & 0x7fffffffu] : make_float4(0, 0, 0, 0);
}

// One batch of a window's entries: occupancy (into the thread's bits, reduced
// per wave after the window's pass: every run of a wave would otherwise hit the
// one occupancy word) and crossing sums from the keys, and (emit pass) the
// runs replayed.
static_assert(UW == 32, "one occupancy word per window");
template <bool EMIT>
__device__ inline void rt_entries(RowLds<EMIT>& s, const RtBatch& b, uint32_t e0, uint32_t ee, uint32_t xmask,
                                  int32_t x0, bool fx, Counters* cnt, uint32_t& occ_bits) {
#pragma unroll
    for (int u = 0; u < RT_U; u++) {
        if (e0 + (uint32_t)(u * RT_NT) >= ee) break;
        const uint32_t x = (b.kk[u] & xmask) - (uint32_t)x0;
        if (b.vv[u] >> 31) {
            const int sg = (int)(int8_t)(b.vv[u] & 0xffu);
            if (sg) atomicAdd(&s.tsign[x], sg);
        } else {
            occ_bits |= 1u << x;
            if constexpr (EMIT) rt_replay_run(s, x, b.rr[u], b.L[u], fx, cnt);
        }
    }
}

template <bool EMIT>
__global__ __launch_bounds__(RT_NT) void k_row_tiles(RowTileArgs a) {
    __shared__ __align__(16) RowLds<EMIT> s;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wid = tid / WAVE;
    const uint32_t xmask = (1u << a.xbits) - 1u;
    const uint64_t lt = lanemask_lt();
    if constexpr (EMIT) {
        // The window sums start at zero: cleared here once, and after each
        // window the quantisation clears the slots it read (runs only add into
        // their own, occupied, tiles).
        constexpr int n16 = (int)sizeof(s.acc_a) / 16;  // 16 bytes at a time
        static_assert(sizeof(s.acc_a) % 16 == 0, "16-byte clears");
        float4* za = reinterpret_cast<float4*>(s.acc_a);
        float4* zh = reinterpret_cast<float4*>(s.acc_h);
        for (int k = tid; k < n16; k += RT_NT) {
            za[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            zh[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        __syncthreads();
    }
    const int64_t grid_n = gridDim.x;
    for (int64_t row = xcd_first_row(); row < a.n_rows; row += grid_n) {
        const PathGrid G = a.grid[a.row_path[row]];
        const int32_t r = (int32_t)(row - (int64_t)G.row_base);
        if (r >= G.h) continue;  // the empty-path row
        const int32_t ty = G.ty0 + r;
        const uint32_t nwin = ((uint32_t)G.w + UW - 1) / UW;
        const uint32_t b0 = a.row_wbase[row];
        uint32_t row_tiles = 0, row_spans = 0;
        if (EMIT) {
            const uint64_t off = a.row_off[row];
            row_tiles = (uint32_t)(off >> 32);
            row_spans = (uint32_t)off;
        }
        // wave 0's running state along the row
        int32_t winding = a.row_wb[row];
        bool have_prev = false;
        int32_t prev_x = 0, prev_w = 0;
        uint32_t nt = 0, ns = 0;
        float carry0 = 0.0f, carry1 = 0.0f;  // wave w: the height carries of pixel rows RT_ROWS * w + j
        // the first window holding entries (a window with none has no run
        // and no crossing)
        uint32_t wi = 0, eb = a.bbeg[b0], ee = a.bbeg[b0 + 1];
        while (ee == eb && ++wi < nwin) {
            eb = ee;
            ee = a.bbeg[b0 + wi + 1];
        }
        RtBatch nb;       // the first batch of window wi, when pf
        bool pf = false;
        while (wi < nwin) {
            // the next window holding entries
            uint32_t wn = wi + 1, nbeg = ee, nend = ee;
            while (wn < nwin) {
                nend = a.bbeg[b0 + wn + 1];
                if (nend != nbeg) break;
                wn++;
            }
            const bool has_next = EMIT && wn < nwin;
            const int32_t x0 = (int32_t)(wi * UW);
            const bool fx = G.w < 8192 && ee - eb < RT_FX_MAX_ENTRIES;  // fixed-point sums (see RowLds)
            if (tid < UW) s.tsign[tid] = 0;
            if (tid < UW / 32) s.occ[tid] = 0;
            __syncthreads();
            // one pass over the window's entries, a batch at a time
            uint32_t e0 = eb + (uint32_t)tid, occ_bits = 0;
            if (pf) {
                rt_entries(s, nb, e0, ee, xmask, x0, fx, a.cnt, occ_bits);
                e0 += RT_U * RT_NT;
            }
            for (; e0 < ee; e0 += RT_U * RT_NT) {
                RtBatch b;
                rt_load_keys(b, a, e0, ee);
                if constexpr (EMIT) {
                    rt_load_recs(b, a);
                    rt_load_lines(b, a);
                }
                rt_entries(s, b, e0, ee, xmask, x0, fx, a.cnt, occ_bits);
            }
            for (int o = 1; o < WAVE; o <<= 1) occ_bits |= __shfl_xor(occ_bits, o, WAVE);
            if (lane == 0 && occ_bits) atomicOr(&s.occ[0], occ_bits);
            __syncthreads();
            if (has_next) rt_load_keys(nb, a, nbeg + (uint32_t)tid, nend);
            if (wid == 0) {
                // lane = tile x0 + lane: ranks, the winding after each tile,
                // and the spans between consecutive tiles (rasterizer.rs:252-264)
                const bool occ = lane < UW && ((s.occ[lane >> 5] >> (lane & 31)) & 1u);
                const int32_t incl = wave_incl_scan(lane < UW ? s.tsign[lane] : 0, OpAdd());
                const int32_t w_at = winding + incl;
                const uint64_t om = __ballot(occ);
                const uint64_t below = om & lt;
                int32_t px = prev_x, pw = prev_w;
                bool hp = have_prev;
                const int pl = below ? 63 - __clzll((long long)below) : 0;
                const int32_t w_pl = __shfl(w_at, pl, WAVE);
                if (below) {
                    px = x0 + pl;
                    pw = w_pl;
                    hp = true;
                }
                const int32_t gx = x0 + lane;
                const bool span = occ && hp && gx > px + 1 && pw != 0;
                const uint64_t sm = __ballot(span);
                if (EMIT && span) {
                    const uint32_t si = row_spans + ns + (uint32_t)__popcll(sm & lt);
                    a.span_xy[2 * si] = (int16_t)((G.tx0 + px + 1) * TILE);
                    a.span_xy[2 * si + 1] = (int16_t)(ty * TILE);
                    a.span_w[si] = (uint16_t)((uint16_t)(gx - px - 1) * (uint16_t)TILE);
                }
                if (EMIT && occ) s.tlist[__popcll(om & lt)] = (uint8_t)lane;
                if (om) {
                    const int last = 63 - __clzll((long long)om);
                    prev_x = x0 + last;
                    prev_w = __shfl(w_at, last, WAVE);
                    have_prev = true;
                }
                winding = __shfl(w_at, WAVE - 1, WAVE);
                if (lane == 0) {
                    s.nt = nt;
                    s.nocc = (uint32_t)__popcll(om);
                }
                nt += (uint32_t)__popcll(om);
                ns += (uint32_t)__popcll(sm);
            }
            if constexpr (EMIT) {
                __syncthreads();
                if (has_next) rt_load_recs(nb, a);
                const uint32_t nocc = s.nocc, nt_w = s.nt;
                // The height carry: wave w takes RT_ROWS pixel rows from RT_ROWS * w,
                // lane k the window's k-th occupied tile, which folds its row's 8
                // heights into an in-tile prefix and a total; a wave scan over
                // the tiles' totals gives each tile its incoming carry, and the
                // quantise adds the two.  (Regrouping the row's f32 sums this way
                // moves a pixel's carry by a few ulps: within the 1-LSB contract.)
#pragma unroll
                for (int j = 0; j < RT_ROWS; j++) {
                    const int prow = RT_ROWS * wid + j;
                    float tot = 0.0f;
                    if ((uint32_t)lane < nocc) {
                        const int base = (int)s.tlist[lane] * UWS + prow * 8;
                        float* fh = reinterpret_cast<float*>(s.acc_h);  // the slots' low words
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            const float h = fx ? fx_to_f(s.acc_h[base + k])
                                               : fh[2 * (base + k)];
                            fh[2 * (base + k)] = tot;
                            tot += h;
                        }
                    }
                    const float incl = wave_incl_scan(tot, OpAdd());
                    const float up = __shfl_up(incl, 1, WAVE);
                    const float excl = lane ? up : 0.0f;
                    float& carry = j ? carry1 : carry0;
                    if ((uint32_t)lane < nocc) s.rtot[lane * 8 + prow] = carry + excl;
                    carry += __shfl(incl, WAVE - 1, WAVE);
                }
                __syncthreads();
                if (has_next) rt_load_lines(nb, a);
                for (uint32_t item = (uint32_t)tid; item < nocc * 16u; item += RT_NT) {
                    // item -> (the occupied tile of rank item / 16, 4 pixels)
                    const uint32_t rk = item >> 4, quad = item & 15u;
                    const int t = s.tlist[rk];
                    const int base = t * UWS + (int)quad * 4;
                    uint32_t word = 0;
                    const uint64_t ti = (uint64_t)row_tiles + nt_w + rk;
                    const float cin = s.rtot[rk * 8 + (quad >> 1)];  // pixel row quad / 2
                    const float* fh = reinterpret_cast<const float*>(s.acc_h);
                    const float* fa = reinterpret_cast<const float*>(s.acc_a);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float av = fx ? fx_to_f(s.acc_a[base + k])
                                            : fa[2 * (base + k)];
                        const float v = (cin + fh[2 * (base + k)]) + av;
                        word |= (uint32_t)fminf(fabsf(v) * 256.0f, 255.0f) << (8 * k);
                        if (a.tile_cov) a.tile_cov[ti * 64 + quad * 4 + (uint32_t)k] = fminf(fabsf(v), 1.0f);
                        s.acc_a[base + k] = 0;  // cleared for the next window
                        s.acc_h[base + k] = 0;
                    }
                    reinterpret_cast<uint32_t*>(a.tile_alpha + ti * 64)[quad] = word;
                    if (quad == 0) {
                        a.tile_xy[2 * ti] = (int16_t)((G.tx0 + x0 + t) * TILE);
                        a.tile_xy[2 * ti + 1] = (int16_t)(ty * TILE);
                    }
                }
            }
            __syncthreads();
            pf = has_next;
            wi = wn;
            eb = nbeg;
            ee = nend;
        }
        if (!EMIT && tid == 0) a.row_cnt[row] = ((uint64_t)nt << 32) | ns;
    }
}

// Per-path output ranges and the empty-path tile.
__global__ void k_path_out(const PathGrid* grid, int64_t n_paths, const uint64_t* row_off, const uint64_t* total,
                           int64_t* tstart, int32_t* tcount, int64_t* sstart, int32_t* scount, int16_t* tile_xy,
                           uint8_t* tile_alpha, float* tile_cov, int64_t tile_base, int64_t span_base) {
    int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= n_paths) return;
    PathGrid g = grid[p];
    uint64_t b = row_off[g.row_base];
    uint64_t e = (p + 1 < n_paths) ? row_off[grid[p + 1].row_base] : *total;
    uint64_t fb = row_off[g.row_base + g.h];
    tstart[p] = tile_base + (int64_t)(b >> 32);
    tcount[p] = (int32_t)((e >> 32) - (b >> 32));
    sstart[p] = span_base + (int64_t)(uint32_t)b;
    scount[p] = (int32_t)((uint32_t)e - (uint32_t)b);
    if ((e >> 32) - (fb >> 32) == 1) {  // the empty-path tile
        uint64_t ti = fb >> 32;
        tile_xy[2 * ti] = 0;
        tile_xy[2 * ti + 1] = 0;
        uint4* dst = reinterpret_cast<uint4*>(tile_alpha + ti * 64);
        for (int k = 0; k < 4; k++) dst[k] = make_uint4(0, 0, 0, 0);
        if (tile_cov)
            for (int k = 0; k < 64; k++) tile_cov[ti * 64 + k] = 0.0f;
    }
}

// ------------------------------------------------------------- host driver

#define HIPCHK(x) HIPCHK_RET(x)

static inline uint32_t grid_for(int64_t n, int bs) { return (uint32_t)((n + bs - 1) / bs); }

struct HostTotals {
    uint32_t lines;
    uint32_t error;
    uint32_t max_w;
    uint32_t rows;
    uint64_t dda;     // (runs << 32) | entries
    uint32_t windows;  // of the unordered tile stage
    uint32_t pad;
    uint32_t n_long[2];  // long rows of the ordered one (TileArgs::n_long); read with out
    uint64_t out;     // (tiles << 32) | spans
    uint64_t entries;
};

// Internal status of one pass: the input is over the per-pass limits.
constexpr int ST_SPLIT = -100;

// Folds a pass's error bits into the call's word: the emit kernels report a
// replay overrun (ERR_REPLAY) after the host's last read of the pass's
// counters, which the next pass clears.
__global__ void k_fold_error(const Counters* cnt, uint32_t* call_error) {
    if (threadIdx.x == 0 && cnt->error) atomicOr(call_error, cnt->error);
}

struct StoreBucketStart {
    uint32_t* beg;
    uint32_t* cur;
    __device__ void operator()(int64_t i, uint32_t excl, uint32_t) const {
        beg[i] = excl;
        cur[i] = excl;
    }
};

static int run_plain_pass(Context* ctx, const SegInput& in, OutputDesc& out, hipStream_t s, bool unordered) {
    const int64_t V = in.n_verbs;
    const int64_t NP = in.n_paths;
    if (NP <= 0) {
        out.n_tiles = out.n_spans = 0;
        return 0;
    }
    if (V >= (1ll << 31) || in.n_points >= (1ll << 32)) {
        ctx->split_ratio = std::max((double)V / (double)(1ll << 31), (double)in.n_points / (double)(1ll << 32));
        return ST_SPLIT;
    }
    HIPCHK(ctx->counters.ensure(256));
    HIPCHK(ctx->totals.ensure(256));
    if (!ctx->host_pinned) HIPCHK(hipHostMalloc(&ctx->host_pinned, 4096));
    Counters* cnt = ctx->counters.as<Counters>();
    uint64_t* tot = ctx->totals.as<uint64_t>();  // [0] lines, [1] rows, [2] dda, [3] long rows, [4] out, [6] windows
    HostTotals* ht = reinterpret_cast<HostTotals*>(ctx->host_pinned);
    fill<uint32_t>(reinterpret_cast<uint32_t*>(cnt), 64, 0u, s);
    fill<uint64_t>(tot, 32, 0ull, s);

    HIPCHK(ensure_scan_capacity(ctx, std::max<int64_t>({V, NP, 1})));

    // ---- (a) flatten
    HIPCHK(ctx->cmd_scan.ensure(std::max<int64_t>(V, 1) * sizeof(CmdAcc)));
    HIPCHK(ctx->cmd_lines.ensure(std::max<int64_t>(V, 1) * 4));
    HIPCHK(ctx->cmd_seg.ensure(std::max<int64_t>(V, 1) * 4));
    HIPCHK(ctx->cmd_line_off.ensure(std::max<int64_t>(V, 1) * 4));
    HIPCHK(ctx->path_box.ensure(NP * sizeof(PathBox)));
    HIPCHK(ctx->path_grid.ensure(NP * sizeof(PathGrid)));
    HIPCHK(ctx->path_rows.ensure(NP * 4));
    CmdAcc* cscan = ctx->cmd_scan.as<CmdAcc>();
    PathBox* box = ctx->path_box.as<PathBox>();
    hipLaunchKernelGGL(k_path_init, dim3(grid_for(NP, 256)), dim3(256), 0, s, in, box, cnt);
    HIPCHK(launch_scan<CmdAcc>(ctx, V, LoadCmd{in.verbs}, StoreCmd{cscan}, OpCmd(), CmdAcc{0, 0, -1, 0},
                               (CmdAcc*)nullptr, s));
    FlattenArgs fa;
    fa.in = in;
    fa.scan = cscan;
    fa.cmd_lines = ctx->cmd_lines.as<uint32_t>();
    fa.cmd_seg = ctx->cmd_seg.as<uint32_t>();
    fa.cmd_line_off = ctx->cmd_line_off.as<uint32_t>();
    fa.box = box;
    fa.cnt = cnt;
    fa.lines = nullptr;
    fa.line_path = nullptr;
    if (V > 0) {
        hipLaunchKernelGGL(k_flatten<false>, dim3(grid_for(V, 256)), dim3(256), 0, s, fa);
        HIPCHK(launch_scan<uint32_t>(ctx, V, LoadU32{fa.cmd_lines}, StoreU32{ctx->cmd_line_off.as<uint32_t>()},
                                     OpAdd(), 0u, reinterpret_cast<uint32_t*>(&tot[0]), s));
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(&ht->lines, &tot[0], 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(&ht->error, &cnt->error, 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (ht->error & ERR_INPUT) return -1;
    if (ht->error & ERR_FLATTEN) return -5;
    const int64_t L = ht->lines;
    if (L > ctx->pass_lines) {
        ctx->split_ratio = (double)L / (double)ctx->pass_lines;
        return ST_SPLIT;
    }

    HIPCHK(ctx->lines.ensure(std::max<int64_t>(L, 1) * 16));
    HIPCHK(ctx->line_path.ensure(std::max<int64_t>(L, 1) * 4));
    HIPCHK(ctx->line_cnt.ensure(std::max<int64_t>(L, 1) * 8));
    HIPCHK(ensure_scan_capacity(ctx, std::max<int64_t>(L, 1)));
    fa.lines = ctx->lines.as<float4>();
    fa.line_path = ctx->line_path.as<uint32_t>();
    if (V > 0) hipLaunchKernelGGL(k_flatten<true>, dim3(grid_for(V, FL_CMDS)), dim3(FL_NT), 0, s, fa);
    PathGrid* grid = ctx->path_grid.as<PathGrid>();
    hipLaunchKernelGGL(k_path_grid, dim3(grid_for(NP, 256)), dim3(256), 0, s, box, grid,
                       ctx->path_rows.as<uint32_t>(), NP, cnt);
    HIPCHK(launch_scan<uint32_t>(ctx, NP, LoadU32{ctx->path_rows.as<uint32_t>()}, StoreRowBase{grid}, OpAdd(), 0u,
                                 reinterpret_cast<uint32_t*>(&tot[1]), s));
    DdaArgs da;
    da.lines = fa.lines;
    da.line_path = fa.line_path;
    da.n_lines = L;
    da.line_cnt = ctx->line_cnt.as<uint64_t>();
    da.grid = grid;
    da.cnt = cnt;
    da.xbits = 0;
    da.keys = da.vals = nullptr;
    da.recs = nullptr;
    const int64_t nblk = (int64_t)grid_for(std::max<int64_t>(L, 1), 256);
    HIPCHK(ctx->dda_blk.ensure((size_t)nblk * 16));
    da.blk_entries = ctx->dda_blk.as<uint64_t>();
    da.blk_cnt = da.blk_entries + nblk;
    if (L > 0) {
        hipLaunchKernelGGL(k_dda<false>, dim3(grid_for(L, 256)), dim3(256), 0, s, da);
        hipLaunchKernelGGL(k_sum_u64, dim3(std::min<uint32_t>(grid_for(nblk, 256), 256)), dim3(256), 0, s,
                           da.blk_entries, nblk, &cnt->entries);
        HIPCHK(launch_scan<uint64_t>(ctx, nblk, LoadU64{da.blk_cnt}, StoreU64{da.blk_cnt}, OpAdd(), 0ull, &tot[2], s));
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(&ht->rows, &tot[1], 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(&ht->dda, &tot[2], 8, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(&ht->max_w, &cnt->max_w, 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(&ht->error, &cnt->error, 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(&ht->entries, &cnt->entries, 8, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (ht->error & ERR_FLATTEN) return -5;
    // entries >= runs (every run record is also a sort entry), so below the
    // limit both 32-bit halves of the packed total are exact
    if (ht->entries > (uint64_t)ctx->pass_entries) {
        ctx->split_ratio = (double)ht->entries / (double)ctx->pass_entries;
        return ST_SPLIT;
    }
    const int64_t R = (int64_t)(uint32_t)ht->dda;
    const int64_t RUNS = (int64_t)(ht->dda >> 32);
    const int64_t ROWS = ht->rows;
    const uint32_t xbits = std::max<uint32_t>(1, bits_for(std::max<uint32_t>(ht->max_w, 1)));
    const uint32_t rbits = bits_for((uint64_t)ROWS);
    if (xbits + rbits > 32) {
        ctx->split_ratio = 2.0;
        return ST_SPLIT;
    }
    const uint32_t kbits = xbits + rbits;

    // ---- (b) binning + sort
    HIPCHK(ctx->keys[0].ensure(std::max<int64_t>(R, 1) * 4));
    HIPCHK(ctx->keys[1].ensure(std::max<int64_t>(R, 1) * 4));
    HIPCHK(ctx->vals[0].ensure(std::max<int64_t>(R, 1) * 4));
    HIPCHK(ctx->vals[1].ensure(std::max<int64_t>(R, 1) * 4));
    HIPCHK(ctx->records.ensure(std::max<int64_t>(RUNS, 1) * sizeof(RunRec)));
    const int rs_bits = rs_digit_bits((int)kbits);
    const int64_t rs_tile = (int64_t)rs_threads(rs_bits, rs_items(R)) * rs_items(R);
    const uint32_t rs_blocks = (uint32_t)std::max<int64_t>(1, (R + rs_tile - 1) / rs_tile);
    if (!unordered) HIPCHK(ctx->rs_counts.ensure(((size_t)rs_blocks << rs_bits) * 4));
    HIPCHK(ensure_scan_capacity(ctx, std::max<int64_t>({unordered ? 1 : (int64_t)rs_blocks << rs_bits, ROWS, 1})));
    da.xbits = xbits;
    da.keys = ctx->keys[0].as<uint32_t>();
    da.vals = ctx->vals[0].as<uint32_t>();
    da.recs = ctx->records.as<RunRec>();
    if (L > 0) hipLaunchKernelGGL(k_dda<true>, dim3(grid_for(L, 256)), dim3(256), 0, s, da);
    if (unordered) {
        // ---- window buckets instead of the sort
        uint32_t* keys0 = ctx->keys[0].as<uint32_t>();
        uint32_t* vals0 = ctx->vals[0].as<uint32_t>();
        HIPCHK(ctx->u_pwbase.ensure((size_t)NP * 4));
        HIPCHK(ctx->u_rwbase.ensure((size_t)ROWS * 4));
        HIPCHK(ctx->row_path.ensure(ROWS * 4));
        HIPCHK(ctx->row_sign.ensure(ROWS * 4));
        HIPCHK(ctx->row_wb.ensure(ROWS * 4));
        HIPCHK(ctx->row_cnt.ensure(ROWS * 8));
        HIPCHK(ctx->row_off.ensure(ROWS * 8));
        uint32_t* pwbase = ctx->u_pwbase.as<uint32_t>();
        uint32_t* rwbase = ctx->u_rwbase.as<uint32_t>();
        uint32_t* nb_dev = reinterpret_cast<uint32_t*>(&tot[6]);
        HIPCHK(launch_scan<uint32_t>(ctx, NP, LoadNWin{grid}, StoreU32{pwbase}, OpAdd(), 0u, nb_dev, s));
        hipLaunchKernelGGL(k_rows_setup, dim3(grid_for(NP, PR_WAVES)), dim3(PR_WAVES * WAVE), 0, s, grid, NP, pwbase,
                           ctx->row_path.as<uint32_t>(), rwbase);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(&ht->windows, nb_dev, 4, hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        const int64_t NB = ht->windows;
        HIPCHK(ctx->u_bcnt.ensure((size_t)std::max<int64_t>(NB, 1) * 4));
        HIPCHK(ctx->u_bbeg.ensure((size_t)(NB + 1) * 4));
        HIPCHK(ctx->u_bcur.ensure((size_t)std::max<int64_t>(NB, 1) * 4));
        HIPCHK(ensure_scan_capacity(ctx, std::max<int64_t>({NB, ROWS, 1})));
        uint32_t* bcnt = ctx->u_bcnt.as<uint32_t>();
        uint32_t* bbeg = ctx->u_bbeg.as<uint32_t>();
        uint32_t* bcur = ctx->u_bcur.as<uint32_t>();
        fill<uint32_t>(bcnt, std::max<int64_t>(NB, 1), 0u, s);
        fill<int32_t>(ctx->row_sign.as<int32_t>(), ROWS, 0, s);
        const uint32_t bk_blocks = grid_for(R, BK_NT * BK_ITEMS);
        if (R > 0)
            hipLaunchKernelGGL(k_bucket_hist, dim3(bk_blocks), dim3(BK_NT), 0, s, keys0, vals0, R, xbits, rwbase,
                               bcnt, ctx->row_sign.as<int32_t>());
        if (NB > 0)
            HIPCHK(launch_scan<uint32_t>(ctx, NB, LoadU32{bcnt}, StoreBucketStart{bbeg, bcur}, OpAdd(), 0u, bbeg + NB,
                                         s));
        else
            fill<uint32_t>(bbeg, 1, 0u, s);
        if (R > 0)
            hipLaunchKernelGGL(k_bucket_scatter, dim3(bk_blocks), dim3(BK_NT), 0, s, keys0, vals0, R, xbits, rwbase,
                               bcur, ctx->keys[1].as<uint32_t>(), ctx->vals[1].as<uint32_t>());
        hipLaunchKernelGGL(k_path_rows_u, dim3(grid_for(NP, PR_WAVES)), dim3(PR_WAVES * WAVE), 0, s, grid, NP, pwbase, bbeg,
                           ctx->row_sign.as<int32_t>(), ctx->row_wb.as<int32_t>(), ctx->row_cnt.as<uint64_t>());
        RowTileArgs ra;
        ra.grid = grid;
        ra.row_path = ctx->row_path.as<uint32_t>();
        ra.row_wbase = rwbase;
        ra.row_wb = ctx->row_wb.as<int32_t>();
        ra.n_rows = ROWS;
        ra.bbeg = bbeg;
        ra.keys = ctx->keys[1].as<uint32_t>();
        ra.vals = ctx->vals[1].as<uint32_t>();
        ra.xbits = xbits;
        ra.recs = ctx->records.as<RunRec>();
        ra.lines = ctx->lines.as<float4>();
        ra.row_cnt = ctx->row_cnt.as<uint64_t>();
        ra.row_off = ctx->row_off.as<uint64_t>();
        ra.tile_xy = out.tile_xy;
        ra.tile_alpha = out.tile_alpha;
        ra.tile_cov = out.tile_cov;
        ra.span_xy = out.span_xy;
        ra.span_w = out.span_w;
        ra.cnt = cnt;
        const uint32_t row_blocks = row_grid(ROWS, 1 << 16);
        hipLaunchKernelGGL(k_row_tiles<false>, dim3(row_blocks), dim3(RT_NT), 0, s, ra);
        HIPCHK(launch_scan<uint64_t>(ctx, ROWS, LoadU64{ra.row_cnt}, StoreU64{ctx->row_off.as<uint64_t>()}, OpAdd(),
                                     0ull, &tot[4], s));
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(&ht->out, &tot[4], 8, hipMemcpyDeviceToHost, s));
        HIPCHK(hipMemcpyAsync(&ht->error, &cnt->error, 4, hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        if (ht->error & (ERR_BBOX | ERR_REPLAY)) return -3;
        const int64_t T = (int64_t)(ht->out >> 32);
        const int64_t S = (int64_t)(uint32_t)ht->out;
        out.n_tiles = T;
        out.n_spans = S;
        if (T > out.tile_capacity || S > out.span_capacity) return -4;
        if (ctx->timing) {
            // pass statistics beside the kernel times: lines, sort entries,
            // runs, tile rows, windows and the windows holding entries
            std::vector<uint32_t> bc((size_t)NB);
            if (NB > 0) HIPCHK(hipMemcpyAsync(bc.data(), bcnt, (size_t)NB * 4, hipMemcpyDeviceToHost, s));
            HIPCHK(hipStreamSynchronize(s));
            int64_t used = 0;
            for (uint32_t c : bc) used += c != 0;
            const std::pair<const char*, int64_t> st[] = {{"pass.lines", L},   {"pass.entries", R},
                                                         {"pass.runs", RUNS},  {"pass.rows", ROWS},
                                                         {"pass.windows", NB}, {"pass.windows_used", used}};
            for (const auto& kv : st) {
                auto& t = ctx->timings[kv.first];
                t.first += (double)kv.second;
                t.second += 1;
            }
            if (!ctx->ev[0]) HIPCHK(hipEventCreate(&ctx->ev[0]));
            if (!ctx->ev[1]) HIPCHK(hipEventCreate(&ctx->ev[1]));
            HIPCHK(hipEventRecord(ctx->ev[0], s));
        }
        hipLaunchKernelGGL(k_row_tiles<true>, dim3(row_blocks), dim3(RT_NT), 0, s, ra);
        if (ctx->timing) HIPCHK(hipEventRecord(ctx->ev[1], s));
        hipLaunchKernelGGL(k_path_out, dim3(grid_for(NP, 256)), dim3(256), 0, s, grid, NP, ra.row_off,
                           (const uint64_t*)&tot[4], out.path_tile_start, out.path_tile_count, out.path_span_start,
                           out.path_span_count, out.tile_xy, out.tile_alpha, out.tile_cov, out.tile_base, out.span_base);
        hipLaunchKernelGGL(k_fold_error, dim3(1), dim3(64), 0, s, cnt, ctx->call_error.as<uint32_t>());
        HIPCHK(hipGetLastError());
        if (ctx->timing) {
            HIPCHK(hipEventSynchronize(ctx->ev[1]));
            float ms = 0;
            HIPCHK(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
            auto& t = ctx->timings["k_row_tiles"];
            t.first += ms;
            t.second += 1;
        }
        return 0;
    }
    int cur = 0;
    uint32_t* rsc = ctx->rs_counts.as<uint32_t>();
    auto sort_pass = [&](auto bits, auto items, int shift) -> hipError_t {
        constexpr int B = decltype(bits)::value, I = decltype(items)::value;
        uint32_t *kin = ctx->keys[cur].as<uint32_t>(), *vin = ctx->vals[cur].as<uint32_t>();
        hipLaunchKernelGGL((k_rs_count<B, I>), dim3(rs_blocks), dim3(rs_threads(B, I)), 0, s, kin, R, shift, rsc, rs_blocks);
        const hipError_t e = launch_scan<uint32_t>(ctx, (int64_t)rs_blocks << B, LoadU32{rsc}, StoreU32{rsc}, OpAdd(),
                                                   0u, (uint32_t*)nullptr, s);
        if (e != hipSuccess) return e;
        // values are the entry payloads (a run, or crossing sign with bit 31)
        hipLaunchKernelGGL((k_rs_scatter<B, I>), dim3(rs_blocks), dim3(rs_threads(B, I)), 0, s, kin, vin, R, shift, rsc,
                           rs_blocks, ctx->keys[cur ^ 1].as<uint32_t>(), ctx->vals[cur ^ 1].as<uint32_t>());
        cur ^= 1;
        return hipSuccess;
    };
    using B8 = std::integral_constant<int, 8>;
    using B10 = std::integral_constant<int, 10>;
    using Large = std::integral_constant<int, RS_ITEMS_LARGE>;
    using Small = std::integral_constant<int, RS_ITEMS_SMALL>;
    const bool rs_small = rs_items(R) == RS_ITEMS_SMALL;
    for (int shift = 0; shift < (int)kbits && R > 0; shift += rs_bits) {
        if (rs_bits == 10)
            HIPCHK(rs_small ? sort_pass(B10(), Small(), shift) : sort_pass(B10(), Large(), shift));
        else
            HIPCHK(rs_small ? sort_pass(B8(), Small(), shift) : sort_pass(B8(), Large(), shift));
    }
    const uint32_t* skeys = ctx->keys[cur].as<uint32_t>();
    const uint32_t* svals = ctx->vals[cur].as<uint32_t>();

    // ---- tile rows
    HIPCHK(ctx->row_begin.ensure(ROWS * 4));
    HIPCHK(ctx->row_end.ensure(ROWS * 4));
    HIPCHK(ctx->row_sign.ensure(ROWS * 4));
    HIPCHK(ctx->row_wb.ensure(ROWS * 4));
    HIPCHK(ctx->row_path.ensure(ROWS * 4));
    HIPCHK(ctx->row_cnt.ensure(ROWS * 8));
    HIPCHK(ctx->row_off.ensure(ROWS * 8));
    uint32_t* row_begin = ctx->row_begin.as<uint32_t>();
    uint32_t* row_end = ctx->row_end.as<uint32_t>();
    fill<uint32_t>(row_begin, ROWS, 0u, s);
    fill<uint32_t>(row_end, ROWS, 0u, s);
    fill<int32_t>(ctx->row_sign.as<int32_t>(), ROWS, 0, s);
    if (R > 0)
        hipLaunchKernelGGL(k_row_table, dim3(grid_for(R, 256 * RTAB_ITEMS)), dim3(256), 0, s, skeys, svals, R, xbits,
                           row_begin, row_end, ctx->row_sign.as<int32_t>());
    hipLaunchKernelGGL(k_path_rows, dim3(grid_for(NP, PR_WAVES)), dim3(PR_WAVES * WAVE), 0, s, grid, NP, row_begin,
                       row_end, ctx->row_sign.as<int32_t>(), ctx->row_wb.as<int32_t>(), ctx->row_path.as<uint32_t>(),
                       ctx->row_cnt.as<uint64_t>());
    TileArgs ta;
    ta.grid = grid;
    ta.row_path = ctx->row_path.as<uint32_t>();
    ta.row_begin = row_begin;
    ta.row_end = row_end;
    ta.row_wb = ctx->row_wb.as<int32_t>();
    ta.n_rows = ROWS;
    ta.keys = skeys;
    ta.xbits = xbits;
    ta.vals = svals;
    ta.recs = ctx->records.as<RunRec>();
    ta.lines = ctx->lines.as<float4>();
    ta.row_cnt = ctx->row_cnt.as<uint64_t>();
    ta.row_off = ctx->row_off.as<uint64_t>();
    ta.tile_xy = out.tile_xy;
    ta.tile_alpha = out.tile_alpha;
    ta.tile_cov = out.tile_cov;
    ta.span_xy = out.span_xy;
    ta.span_w = out.span_w;
    ta.cnt = cnt;
    HIPCHK(ctx->long_rows.ensure(ROWS * 4));
    ta.long_rows = ctx->long_rows.as<uint32_t>();
    ta.n_long = reinterpret_cast<uint32_t*>(&tot[3]);
    const uint32_t tile_blocks = (uint32_t)std::min<int64_t>((ROWS + TC_ROWS - 1) / TC_ROWS, 1 << 20);
    hipLaunchKernelGGL(k_tile_counts, dim3(tile_blocks), dim3(TC_ROWS * WAVE), 0, s, ta);
    HIPCHK(launch_scan<uint64_t>(ctx, ROWS, LoadU64{ta.row_cnt}, StoreU64{ctx->row_off.as<uint64_t>()}, OpAdd(),
                                 0ull, &tot[4], s));
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(ht->n_long, &tot[3], 16, hipMemcpyDeviceToHost, s));  // and out
    HIPCHK(hipMemcpyAsync(&ht->error, &cnt->error, 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (ht->error & (ERR_BBOX | ERR_REPLAY)) return -3;
    const int64_t T = (int64_t)(ht->out >> 32);
    const int64_t S = (int64_t)(uint32_t)ht->out;
    out.n_tiles = T;
    out.n_spans = S;
    if (T > out.tile_capacity || S > out.span_capacity) return -4;

    // ---- (c)(d)(e)
    if (ctx->timing) {
        if (!ctx->ev[0]) HIPCHK(hipEventCreate(&ctx->ev[0]));
        if (!ctx->ev[1]) HIPCHK(hipEventCreate(&ctx->ev[1]));
        HIPCHK(hipEventRecord(ctx->ev[0], s));
    }
    const uint32_t n_long = ht->n_long[0] + ht->n_long[1];
    if (n_long) {
        // beside each other: the long rows alone leave the chip half empty
        if (!ctx->own_stream) HIPCHK(hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking));
        for (auto& e : ctx->side_ev)
            if (!e) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        HIPCHK(hipEventRecord(ctx->side_ev[0], s));
        HIPCHK(hipStreamWaitEvent(ctx->own_stream, ctx->side_ev[0], 0));
        hipLaunchKernelGGL(k_tile_rows<true>, dim3(n_long), dim3(2 * WAVE), 0, ctx->own_stream, ta, ht->n_long[0]);
    }
    hipLaunchKernelGGL(k_tile_rows<false>, dim3(row_grid(ROWS, 1 << 20)), dim3(WAVE), 0, s, ta, 0u);
    if (n_long) {
        hipError_t e = hipEventRecord(ctx->side_ev[1], ctx->own_stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(s, ctx->side_ev[1], 0);
        if (e != hipSuccess) {  // nothing of the call runs on after it
            (void)hipStreamSynchronize(ctx->own_stream);
            return map_hip_error(e);
        }
    }
    if (ctx->timing) HIPCHK(hipEventRecord(ctx->ev[1], s));
    hipLaunchKernelGGL(k_path_out, dim3(grid_for(NP, 256)), dim3(256), 0, s, grid, NP, ta.row_off,
                       (const uint64_t*)&tot[4], out.path_tile_start, out.path_tile_count, out.path_span_start,
                       out.path_span_count, out.tile_xy, out.tile_alpha, out.tile_cov, out.tile_base, out.span_base);
    hipLaunchKernelGGL(k_fold_error, dim3(1), dim3(64), 0, s, cnt, ctx->call_error.as<uint32_t>());
    HIPCHK(hipGetLastError());
    if (ctx->timing) {
        HIPCHK(hipEventSynchronize(ctx->ev[1]));
        float ms = 0;
        HIPCHK(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
        auto& t = ctx->timings["k_tile_rows"];
        t.first += ms;
        t.second += 1;
    }
    return 0;
}

// Offsets of paths [p0, p0 + n] rebased to the range's first verb, point and
// weight, packed as three arrays of n + 1.
__global__ void k_rebase_offsets(const int64_t* voff, const int64_t* poff, const int64_t* woff, int64_t p0, int64_t n,
                                 int64_t* dst) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i > n) return;
    dst[i] = voff[p0 + i] - voff[p0];
    dst[n + 1 + i] = poff[p0 + i] - poff[p0];
    dst[2 * (n + 1) + i] = woff[p0 + i] - woff[p0];
}

// The emit-phase error bits of a call (folded in by k_fold_error after each
// pass), read back once the call's work is queued: a replay overrun makes the
// call fail with -3 instead of returning truncated alpha.
static int check_call_error(Context* ctx, int st, hipStream_t s) {
    if (st != 0 && st != -4) return st;
    uint32_t* h = reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(ctx->host_pinned) + 2048);
    HIPCHK(hipMemcpyAsync(h, ctx->call_error.p, 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (*h & (ERR_BBOX | ERR_REPLAY)) return -3;
    return st;
}

int run_plain(Context* ctx, const SegInput& in, OutputDesc& out, hipStream_t s, bool unordered, int64_t pass_lines,
              int64_t pass_entries) {
    HIPCHK(ctx->call_error.ensure(256));
    if (!ctx->host_pinned) HIPCHK(hipHostMalloc(&ctx->host_pinned, 4096));
    fill<uint32_t>(ctx->call_error.as<uint32_t>(), 1, 0u, s);
    // a pass within the asked limits; one path over them, within the context's (and,
    // in the batched call, at least OWN_MIN_LINES and OWN_MIN_ENTRIES)
    auto pass = [&](const SegInput& si, OutputDesc& od) {
        ctx->pass_lines = pass_lines ? std::min(pass_lines, ctx->max_lines) : ctx->max_lines;
        ctx->pass_entries = pass_entries ? std::min(pass_entries, ctx->max_entries) : ctx->max_entries;
        const int rc = run_plain_pass(ctx, si, od, s, unordered);
        const int64_t lines = si.own_ranges ? std::max(ctx->max_lines, OWN_MIN_LINES) : ctx->max_lines;
        const int64_t entries = si.own_ranges ? std::max(ctx->max_entries, OWN_MIN_ENTRIES) : ctx->max_entries;
        if (rc != ST_SPLIT || si.n_paths > 1 || (ctx->pass_lines >= lines && ctx->pass_entries >= entries)) return rc;
        ctx->pass_lines = lines;
        ctx->pass_entries = entries;
        return run_plain_pass(ctx, si, od, s, unordered);
    };
    int st = pass(in, out);
    if (st != ST_SPLIT) return check_call_error(ctx, st, s);
    // Paths are independent Rasterizers: rasterise path ranges one after
    // another, each range's tiles and spans following the previous range's.
    if (in.path_seg_off || in.seg_path || in.n_paths < 2) return -7;
    const int64_t NP = in.n_paths;
    std::vector<int64_t> voff(NP + 1), poff(NP + 1), woff(NP + 1);
    HIPCHK(hipMemcpyAsync(voff.data(), in.seg_verb_off, (NP + 1) * 8, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(poff.data(), in.seg_point_off, (NP + 1) * 8, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(woff.data(), in.seg_weight_off, (NP + 1) * 8, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    HIPCHK(ctx->split_off.ensure((size_t)3 * (NP + 1) * 8));
    int64_t* roff = ctx->split_off.as<int64_t>();

    // ranges still to do, the next one at the back; a range over the limits is
    // cut into pieces of about equal verb counts, sized from how far the
    // failed pass was over
    std::vector<std::pair<int64_t, int64_t>> todo;
    auto cut = [&](int64_t p0, int64_t p1) {
        const int k = (int)std::min<double>(std::ceil(std::max(2.0, 1.25 * ctx->split_ratio)), (double)(p1 - p0));
        std::vector<int64_t> cuts{p0};
        const int64_t v0 = voff[p0], vr = voff[p1] - v0;
        for (int i = 1; i < k; i++) {
            const int64_t target = v0 + (int64_t)((double)vr * i / k);
            int64_t c = std::lower_bound(voff.begin() + p0, voff.begin() + p1, target) - voff.begin();
            if (c > cuts.back() && c < p1) cuts.push_back(c);
        }
        if (cuts.size() == 1) cuts.push_back(p0 + (p1 - p0) / 2);
        cuts.push_back(p1);
        for (size_t i = cuts.size() - 1; i > 0; i--) todo.push_back({cuts[i - 1], cuts[i]});
    };
    cut(0, NP);
    int64_t T = 0, S = 0;
    bool room = true;
    while (!todo.empty()) {
        const int64_t p0 = todo.back().first, p1 = todo.back().second;
        todo.pop_back();
        const int64_t n = p1 - p0;
        hipLaunchKernelGGL(k_rebase_offsets, dim3(grid_for(n + 1, 256)), dim3(256), 0, s, in.seg_verb_off,
                           in.seg_point_off, in.seg_weight_off, p0, n, roff);
        HIPCHK(hipGetLastError());
        SegInput si;
        si.n_segs = n;
        si.n_paths = n;
        si.verbs = in.verbs + voff[p0];
        si.points = in.points + 2 * poff[p0];
        si.weights = in.weights ? in.weights + woff[p0] : nullptr;
        si.seg_verb_off = roff;
        si.seg_point_off = roff + (n + 1);
        si.seg_weight_off = roff + 2 * (n + 1);
        si.seg_xf = in.seg_xf + p0;
        si.seg_raw = in.seg_raw ? in.seg_raw + p0 : nullptr;
        si.n_verbs = voff[p1] - voff[p0];
        si.n_points = poff[p1] - poff[p0];
        si.n_weights = woff[p1] - woff[p0];
        si.own_ranges = in.own_ranges;
        OutputDesc od;
        od.tile_xy = out.tile_xy + (room ? 2 * T : 0);
        od.tile_alpha = out.tile_alpha + (room ? 64 * T : 0);
        od.tile_cov = out.tile_cov ? out.tile_cov + (room ? 64 * T : 0) : nullptr;
        od.tile_capacity = room ? out.tile_capacity - T : 0;
        od.span_xy = out.span_xy + (room ? 2 * S : 0);
        od.span_w = out.span_w + (room ? S : 0);
        od.span_capacity = room ? out.span_capacity - S : 0;
        od.path_tile_start = out.path_tile_start + p0;
        od.path_tile_count = out.path_tile_count + p0;
        od.path_span_start = out.path_span_start + p0;
        od.path_span_count = out.path_span_count + p0;
        od.tile_base = out.tile_base + T;
        od.span_base = out.span_base + S;
        st = pass(si, od);
        if (st == ST_SPLIT) {
            if (n < 2) return -7;
            cut(p0, p1);
            continue;
        }
        if (st == -4) room = false;
        else if (st) return st;
        T += od.n_tiles;
        S += od.n_spans;
    }
    out.n_tiles = T;
    out.n_spans = S;
    return check_call_error(ctx, (room && T <= out.tile_capacity && S <= out.span_capacity) ? 0 : -4, s);
}

}  // namespace ochre
