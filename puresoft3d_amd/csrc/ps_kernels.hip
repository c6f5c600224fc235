// ps_kernels.hip -- gfx950 kernels of the sort-middle raster path.
//
//  setup   : one thread per triangle: vertex twin, 1/w divide, back-face cull,
//            z reject, pushVertex/pushTriangle row-range and edge choice
//            (drawvao.cpp:36-63, vertthrd.cpp, rasterizer.cpp:122-283)
//  rows    : exclusive scan of the row counts, and the triangle of every
//            64th row item
//  span    : one thread per (triangle,row), its triangle searched from that
//            table: span ends, clamping and the
//            depth / correction-factor start and step (drawvao.cpp:66-110,
//            interp.cpp:26-80); counts, per tile, the pieces (bin chunks) of
//            the spans and the waves that have pieces there
//  tiles   : exclusive scan of the per-tile counts: each tile's piece and
//            run ranges
//  segment : one thread per span walks it and writes its pieces; a wave's
//            pieces of one tile form one run of consecutive pieces, placed by
//            one atomic on the tile's counter
//  raster  : one wave per tile of 64 bins (a bin is a row piece of chunk_w
//            pixels); the wave puts its tile's runs in wave order, which is
//            submission order, and takes the pieces 64 at a time, one per
//            lane, keeping each pixel's depth and winner in LDS
//            (fragthrd.cpp:208-252); depth test -1 < z && z - d < -1e-4
//  shade   : one thread per pixel whose last colour-writing depth-test pass
//            is known: re-derives that span's varyings, walks them serially
//            to the pixel, runs the FP twin and writes BGRA8.
//  The depth test is order dependent, so per pixel the fragments are applied
//  strictly in submission order; no atomics touch depth or colour.
#include <type_traits>

#include "ps_kernels.h"
#include "ps_procs.h"

#define PS_WAVE 64

// An overflow is noted twice: in the counters, where it stops the later kernels
// of the log, and in the host's word for the logged command (pinned memory),
// so that no copy has to follow every flush.
__device__ __forceinline__ void ps_overflow(PsCounters* c, int bits, int* flag)
{
    atomicOr(&c->overflow, bits);
    __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ bool ps_poisoned(const PsCounters* c)
{
    return *((volatile const int*)&c->overflow) != 0;
}
// Kernels read the flag together with their first loads that stay in bounds
// whatever an overflow left behind, and test it before the first store or
// the first load whose address depends on the flush's device-side sizes:
// the flag's round trip then overlaps those loads instead of preceding them.

__device__ __forceinline__ uint64_t ps_lt_mask()
{
    return __lanemask_lt();
}

// the flush got past every overflow check: its pending statistics become
// committed (blocks 0..63 of the raster launch take the stripes between them)
__device__ __forceinline__ void ps_commit_pending(PsCounters* c)
{
    if (blockIdx.x >= PS_STRIPES || threadIdx.x >= PS_ST_N) return;
    for (int s = blockIdx.x; s < PS_STRIPES; s += gridDim.x) {
        unsigned long long v = c->pend[s][threadIdx.x];
        if (v) {
            atomicAdd(&c->stat[s][threadIdx.x], v);
            c->pend[s][threadIdx.x] = 0;
        }
    }
}

// The last view whose base is at most t (t the same in the whole wave, every
// lane active): 64 bases at a time, one per lane, so that up to 64 views cost
// one load, where a binary search makes a chain of six.
template <typename Base>
__device__ __forceinline__ int ps_find_view(int n, int64_t t, Base base)
{
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = n;   // views[lo] is at or below t; hi == n or views[hi] above it
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) / 64, p = lo + lane * step;
        const int c = __popcll(__ballot(p < hi && base(p) <= t));
        lo += (c - 1) * step;
        hi = min(hi, lo + step);
    }
    return lo;
}

__device__ __forceinline__ int ps_view_of_tile(const PsFrame& f, int64_t t)
{
    return ps_find_view(f.n_views, t, [&](int v) { return f.views[v].tile_base; });
}

__device__ __forceinline__ int ps_view_of_stile(const PsFrame& f, int64_t t)
{
    return ps_find_view(f.n_views, t, [&](int v) { return f.views[v].stile_base; });
}

// Rows of a padded winner plane start 32 bytes aligned, so that a raster lane
// stores its chunk in one instruction.
__device__ __forceinline__ int64_t ps_winner_at(const PsFrame& f, const PsView& V, int x, int y)
{
    return (int64_t)y * PS_WINNER_PITCH(V.W, f.winner_pad) + x;
}

// Workgroups are dealt to the 8 XCDs round-robin (workgroup b runs on XCD
// b % 8), and each XCD has its own L2.  This maps workgroups to logical
// indices so that each XCD gets runs of G consecutive indices: neighbouring
// screen tiles then share texels and triangle records in one L2, while the
// runs still alternate over the XCDs (contiguous eighths leave XCDs idle
// where the screen is empty).  A bijection on [0, n) whatever the dispatch:
// whole groups of 8G are permuted within, the tail keeps its order.
template <int G>
__device__ __forceinline__ int64_t ps_xcd_remap(int64_t b, int64_t n)
{
    const int64_t s = b / (8 * G), j = b - s * (8 * G);
    if ((s + 1) * (8 * G) > n) return b;
    return s * (8 * G) + (j & 7) * G + (j >> 3);
}

// the programme of a triangle's draw
__device__ __forceinline__ int ps_tri_prog(const PsTri& t) { return (int)(t.vflags >> 4); }

// the first of the two texcoord varyings the mip-level gradients use (-1: none)
template <class P> __device__ constexpr int ps_grad_iu()
{
    if constexpr (P::GRAD) return P::IU;
    else return -1;
}

// f(draw record): when every active lane of the wave uses the same draw, the
// record is addressed through a wave-uniform index, so its fields come in
// with scalar loads instead of one vector load per lane
template <typename F>
__device__ __forceinline__ void ps_with_draw(const PsDraw* __restrict__ draws, int di, F&& f)
{
    int d0 = __builtin_amdgcn_readfirstlane(di);
    if (__all(di == d0)) f(draws[d0]);
    else f(draws[di]);
}

// Wave-wide min / max / inclusive sum over 64 lanes with DPP row operations
// (no LDS crossbar round trips).  Control codes of GFX9 DPP: quad_perm
// 0x00-0xff, row_shr:n 0x110+n, row_mirror 0x140, row_half_mirror 0x141,
// row_bcast:15 0x142, row_bcast:31 0x143.
#define PS_DPP(v, ctrl, rmask, bound) \
    __builtin_amdgcn_update_dpp(0u, (v), (ctrl), (rmask), 0xf, (bound))

// the minimum, the same in every lane
// a tile start without the heavy-tile mark (bit 63)
#define PS_TS(x) ((x) & 0x7fffffffffffffffull)

__device__ __forceinline__ uint32_t ps_wave_min(uint32_t v)
{
    // within rows of 16: quad swaps, then the half-row and row mirrors
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, false));  // row_half_mirror
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xf, 0xf, false));  // row_mirror
    // the four row minima
    const uint32_t r0 = __builtin_amdgcn_readlane(v, 0), r1 = __builtin_amdgcn_readlane(v, 16);
    const uint32_t r2 = __builtin_amdgcn_readlane(v, 32), r3 = __builtin_amdgcn_readlane(v, 48);
    return min(min(r0, r1), min(r2, r3));
}

__device__ __forceinline__ uint32_t ps_wave_max(uint32_t v)
{
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xf, 0xf, false));
    const uint32_t r0 = __builtin_amdgcn_readlane(v, 0), r1 = __builtin_amdgcn_readlane(v, 16);
    const uint32_t r2 = __builtin_amdgcn_readlane(v, 32), r3 = __builtin_amdgcn_readlane(v, 48);
    return max(max(r0, r1), max(r2, r3));
}

// inclusive prefix sum over the lanes (every lane of the wave active)
__device__ __forceinline__ uint32_t ps_wave_incl_scan(uint32_t v)
{
    v += PS_DPP(v, 0x111, 0xf, true);   // row_shr:1, zero from outside the row
    v += PS_DPP(v, 0x112, 0xf, true);   // row_shr:2
    v += PS_DPP(v, 0x114, 0xf, true);   // row_shr:4
    v += PS_DPP(v, 0x118, 0xf, true);   // row_shr:8
    v += PS_DPP(v, 0x142, 0xa, false);  // row_bcast:15 into rows 1 and 3
    v += PS_DPP(v, 0x143, 0xc, false);  // row_bcast:31 into rows 2 and 3
    return v;
}

// keeps the compiler from moving LDS accesses across: the LDS operations of a
// wave are performed in order
__device__ __forceinline__ void ps_lds_turn()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// inclusive scan over each group of G (16 or 32) lanes
template <int G>
__device__ __forceinline__ uint32_t ps_group_incl_scan(uint32_t v)
{
    v += PS_DPP(v, 0x111, 0xf, true);
    v += PS_DPP(v, 0x112, 0xf, true);
    v += PS_DPP(v, 0x114, 0xf, true);
    v += PS_DPP(v, 0x118, 0xf, true);
    if constexpr (G == 32) v += PS_DPP(v, 0x142, 0xa, false);
    return v;
}

// a wave's statistic (lane values whose wave total fits 32 bits, every lane
// active): into the committed counters (pending = false) or the flush's
// pending ones; one atomic per wave, on a per-block stripe
__device__ __forceinline__ void ps_wave_add(PsCounters* c, int field, uint32_t v, bool pending = false)
{
    const uint32_t tot = __builtin_amdgcn_readlane(ps_wave_incl_scan(v), 63);
    if ((threadIdx.x & (PS_WAVE - 1)) == 0 && tot)
        atomicAdd(pending ? &c->pend[blockIdx.x & (PS_STRIPES - 1)][field] : &c->stat[blockIdx.x & (PS_STRIPES - 1)][field],
                  (unsigned long long)tot);
}

// the same for 64-bit lane values, into the committed counters
__device__ __forceinline__ void ps_wave_add64(PsCounters* c, int field, unsigned long long v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, PS_WAVE);
    if ((threadIdx.x & (PS_WAVE - 1)) == 0 && v) atomicAdd(&c->stat[blockIdx.x & (PS_STRIPES - 1)][field], v);
}

// The tiles a span's pieces fall in: tiles g0 .. g1 (consecutive tile
// indices of one tile row), chunk range cx0 .. cx1 of the row.
struct PsSpanTiles {
    uint32_t g0, g1;
    int cx0, cx1, tx0;
};

// The chunk width, tile rows and tile columns are powers of two
// (psgpu_tiling_set) and y, x1, x2 are not negative, so the divisions are
// shifts (a division by a run-time divisor costs a dozen instructions).
__device__ __forceinline__ PsSpanTiles ps_span_tiles(int64_t tile_base, int n_tiles_x, int tile_rows, int tile_cols,
                                                     int chunk_w, int y, int x1, int x2)
{
    const int cs = __builtin_ctz((unsigned)chunk_w), ts = __builtin_ctz((unsigned)tile_cols);
    const int rs = __builtin_ctz((unsigned)tile_rows);
    PsSpanTiles s;
    s.cx0 = x1 >> cs;
    s.cx1 = x2 >> cs;
    s.tx0 = s.cx0 >> ts;
    s.g0 = (uint32_t)(tile_base + (int64_t)(y >> rs) * n_tiles_x + s.tx0);
    s.g1 = s.g0 + (uint32_t)((s.cx1 >> ts) - s.tx0);
    return s;
}

// the chunks [lo, hi] of the span inside tile k (g0 <= k <= g1)
__device__ __forceinline__ void ps_span_tile_chunks(const PsSpanTiles& s, int tile_cols, uint32_t k, int& lo, int& hi)
{
    int tx = s.tx0 + (int)(k - s.g0);
    lo = max(s.cx0, tx * tile_cols);
    hi = min(s.cx1, tx * tile_cols + tile_cols - 1);
}

// The distinct tiles of the wave's spans, in increasing order, up to 64 at a
// time: lane j receives the j-th tile (bk) and the wave's pieces in it (bn);
// returns how many.  cur is the lane's next tile (0xffffffff: none left) and
// moves on past the batch.  Every lane of the wave calls it.  A span's tiles
// are consecutive, so taking the smallest pending tile each round visits each
// (wave, tile) pair exactly once.
__device__ __forceinline__ int ps_wave_tile_batch(const PsSpanTiles& s, int tile_cols, uint32_t& cur, uint32_t& bk,
                                                  uint32_t& bn)
{
    const int lane = threadIdx.x & (PS_WAVE - 1);
    bk = 0xffffffffu;
    bn = 0;
    int j = 0;
    for (; j < PS_WAVE; j++) {
        const uint32_t k = ps_wave_min(cur);
        if (k == 0xffffffffu) break;
        const bool m = cur == k;
        int lo = 0, hi = -1;
        if (m) ps_span_tile_chunks(s, tile_cols, k, lo, hi);
        const uint32_t n = __builtin_amdgcn_readlane(ps_wave_incl_scan((uint32_t)(hi - lo + 1)), 63);
        if (lane == j) { bk = k; bn = n; }
        if (m) cur = k < s.g1 ? k + 1 : 0xffffffffu;
    }
    return j;
}

// ---------------------------------------------------------------------------
// fills (graph friendly: no hipMemset nodes)
// ---------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* p, int64_t n, uint32_t v, const PsCounters* c)
{
    if (c && ps_poisoned(c)) return;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// a clear command: fill f = blockIdx.y; clear4 (fbo.cpp:332-346) is a fill of
// rows 0 .. height-2, clear16 (fbo.cpp:348-371) one of the whole buffer.
// Rows without padding form one run, stored four values per thread; otherwise
// work items are pieces of 1024 values of one row (a 4 KiB stride keeps the
// row's alignment), and inside a piece the 16-byte aligned middle is stored
// four values per thread.
#define FILL_PIECE 1024
__device__ __forceinline__ void ps_fill(const PsFill& fl)
{
    const uint4 v4 = make_uint4(fl.value, fl.value, fl.value, fl.value);
    if (fl.scan == fl.width) {
        // rows without padding are one run: four values per thread, grid-stride
        const int64_t n = fl.rows * fl.width;
        uint32_t* p = fl.ptr;
        int64_t head = (int64_t)(((16u - ((uintptr_t)p & 15u)) & 15u) / 4);
        if (head > n) head = n;
        const int64_t nvec = (n - head) / 4, tail0 = head + nvec * 4;
        if (blockIdx.x == 0 && (int64_t)threadIdx.x < head) p[threadIdx.x] = fl.value;
        if (blockIdx.x == 0 && tail0 + (int64_t)threadIdx.x < n) p[tail0 + threadIdx.x] = fl.value;
        uint4* q = (uint4*)(p + head);
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * blockDim.x)
            q[i] = v4;
        return;
    }
    const int64_t npc = (fl.width + FILL_PIECE - 1) / FILL_PIECE;
    const int64_t total = fl.rows * npc;
    for (int64_t k = blockIdx.x; k < total; k += gridDim.x) {
        int64_t y = k / npc, x0 = (k - y * npc) * FILL_PIECE;
        int64_t n = fl.width - x0 < FILL_PIECE ? fl.width - x0 : FILL_PIECE;
        uint32_t* p = fl.ptr + y * fl.scan + x0;
        int head = (int)(((16u - ((uintptr_t)p & 15u)) & 15u) / 4);
        if (head > n) head = (int)n;
        int64_t nvec = (n - head) / 4;
        int64_t tail0 = head + nvec * 4;
        if ((int)threadIdx.x < head) p[threadIdx.x] = fl.value;
        if ((int64_t)threadIdx.x < nvec) ((uint4*)(p + head))[threadIdx.x] = v4;
        if (tail0 + threadIdx.x < n) p[tail0 + threadIdx.x] = fl.value;
    }
}

__global__ void __launch_bounds__(256) k_fills(const PsFill* __restrict__ fills, const PsCounters* c)
{
    if (c && ps_poisoned(c)) return;
    ps_fill(fills[blockIdx.y]);
}

// a few fills come as kernel arguments, without a copy of their records
__global__ void __launch_bounds__(256) k_few_fills(PsFewFills fills, const PsCounters* c)
{
    if (c && ps_poisoned(c)) return;
    ps_fill(fills.f[blockIdx.y]);
}

// The end of the log, one wave: what the host waits for (the overflow flag, the
// sizes and the sums of the statistics) goes to its pinned memory, and unless
// the log is to be replayed everything is zero again for the next one.
__global__ void __launch_bounds__(64) k_finish(PsCounters* c, uint32_t* sizes, PsFinish* out, int reset)
{
    const int lane = threadIdx.x;
    const int overflow = c->overflow;
    unsigned long long sum[PS_ST_N];
#pragma unroll
    for (int f = 0; f < PS_ST_N; f++) {
        sum[f] = c->stat[lane][f];
        for (int o = 32; o > 0; o >>= 1) sum[f] += __shfl_xor(sum[f], o, 64);
    }
    if (lane < 4) out->sizes[lane] = sizes[lane];
    if (lane == 0) {
        out->overflow = overflow;
#pragma unroll
        for (int f = 0; f < PS_ST_N; f++) out->sum[f] = (long long)sum[f];
    }
    if (overflow && !reset) return;
#pragma unroll
    for (int f = 0; f < PS_ST_N; f++) c->stat[lane][f] = c->pend[lane][f] = 0;
    if (lane == 0) c->overflow = 0;
    if (lane < 4) sizes[lane] = 0;
}


// ---------------------------------------------------------------------------
// setup
// ---------------------------------------------------------------------------
// Draw of triangle t (the last draw with tri_start <= t; draws are sorted by
// tri_start and every t is covered).  The lanes' triangles lie in
// [t0, t0 + 63], t0 that of lane 0.  While more than 63 draws remain, a
// 64-way search (lane j loads pivot lo + j * step) narrows them to the
// interval holding t0's draw.  The last step loads the 63 draws from lo on
// into lanes 0..62 and the next one into lane 63: each lane's draw is then
// the last of those starting at or before its t, found from ballots and
// read lanes without another load, unless a lane's t reaches the draw after
// the 63 (then it steps on).  So one dependent load for up to 63 draws, two
// for up to 4,032.
__device__ __forceinline__ int ps_find_draw_wave(const PsDraw* __restrict__ draws, int nd, int64_t t)
{
    const int lane = threadIdx.x & 63;
    const int64_t t0 = (int64_t)__builtin_amdgcn_readfirstlane((int)(t >> 32)) << 32 |
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)t);
    int lo = 0, hi = nd;
    while (hi - lo > 63) {
        const int step = (hi - lo + 63) / 64;
        const int p = lo + lane * step;
        const bool le = p < hi && draws[p].tri_start <= t0;
        const int cnt = __popcll(__ballot(le));   // pivot 0 (lo) is always <= t0
        // pivots below cnt are <= t0: t0's draw is in [lo + (cnt-1)*step, lo + cnt*step)
        const int nhi = lo + cnt * step;
        lo = lo + (cnt - 1) * step;
        hi = nhi < hi ? nhi : hi;
    }
    const int p = lo + lane;
    const int64_t sp = p < nd ? draws[p].tri_start : INT64_MAX;
    // draws lo .. lo+62 starting in (t0, t] for some lane
    const uint64_t later = __ballot(lane < 63 && sp > t0 && sp <= t0 + 63) ;
    int d = lo + __popcll(__ballot(lane < 63 && sp <= t0)) - 1;
    for (uint64_t m = later; m;) {
        const int b = __builtin_ctzll(m);
        m &= m - 1;
        const int64_t sb = (int64_t)__builtin_amdgcn_readlane((int)(sp >> 32), b) << 32 |
                           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)sp, b);
        if (t >= sb) d = lo + b;
    }
    // the draw after the 63 starts at or before some lane's t: step on
    const int64_t s63 = (int64_t)__builtin_amdgcn_readlane((int)(sp >> 32), 63) << 32 |
                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)sp, 63);
    if (s63 <= t0 + 63)
        while (d + 1 < nd && draws[d + 1].tri_start <= t) d++;
    return d;
}

// row_part: the block's row total, for the scan of the row counts.  At least three waves per SIMD: a 1080p frame's 200k
// triangles make only about three per SIMD, and the bound of four left the
// Blinn-Phong instantiation at 128 VGPRs with a 12-byte spill.
// PROG 0: flushes of several programmes, each wave running through those of its
// triangles (the programmes that shade in the raster walk have their own
// flushes).  A launch a programme went over all triangles each time: four
// programmes at 1366x768, 38 + 4 us for the row totals -> 14.7, shading
// likewise 49 -> 25, the frame 77 -> 59.  A flush of one programme keeps its
// own instantiation, whose code and registers are that programme's alone.
#define PS_SETUP_PROGS(X)                                                                            \
    X(PSGPU_PROC_DEF01) X(PSGPU_PROC_DEF02) X(PSGPU_PROC_DEF03) X(PSGPU_PROC_DEF04)                  \
    X(PSGPU_PROC_DEF05) X(PSGPU_PROC_LAMBERT) X(PSGPU_PROC_BLINN) X(PSGPU_PROC_SHADOWED)
template <int PROG, bool SHARE>
__global__ void __launch_bounds__(128, 3) k_setup(const PsDraw* __restrict__ draws, int nd, int64_t T, PsTri* __restrict__ tris,
                                               float* __restrict__ vary, int nvs, float* __restrict__ grads,
                                               uint32_t* __restrict__ nrows, uint32_t* __restrict__ row_part,
                                               PsCounters* cnt, const PsView* __restrict__ views)
{
    extern __shared__ float su[];   // per wave: the varyings of its 64 triangles, 3*nvs floats each
    __shared__ uint32_t wrows[2];
    int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    bool live = t < T;
    int di = ps_find_draw_wave(draws, nd, live ? t : T - 1);
    unsigned culled = 0, zrej = 0, dropped = 0;
    uint32_t myrows = 0;
    const int lane = threadIdx.x & 63, n3 = 3 * nvs;
    float* wl = su + (size_t)(threadIdx.x & ~63) * n3;
    bool stage = false;
    auto triangle = [&](auto k, const PsDraw& d) {
    constexpr int K = decltype(k)::value;
    typedef PsProc<K> P;
    if (live && d.prog == K) {
        const int W = views[d.view].W, H = views[d.view].H;
        int64_t lt = t - d.tri_start;
        float pos[3][4];
        float u[3][P::NV > 0 ? P::NV : 1];
        float rw[3], z[3];
        bool pieces = false;
        const bool skip = SHARE && ps_shares_varyings(K) && d.vary_skip;
#pragma unroll
        for (int v = 0; v < 3; v++) {
            if (skip) ps_vp_pos(d, lt * 3 + v, pos[v], u[v], ps_grad_iu<P>());
            else P::vp(d, lt * 3 + v, pos[v], u[v]);
            // perspective division (vertthrd.cpp:37-47)
            float r = 1.0f / pos[v][3];
            pos[v][0] *= r; pos[v][1] *= r; pos[v][2] *= r; pos[v][3] *= r;
            z[v] = pos[v][2];
            rw[v] = r;
        }
        uint32_t n = 0;
        PsTri tr;
        bool keep = true;
        if ((d.behavior & PSGPU_FACE_CULLING) && ps_back_face(pos[0], pos[1], pos[2])) { keep = false; culled = 1; }
        if (keep) {
            // drawvao.cpp:51-56
#pragma unroll
            for (int v = 0; v < 3; v++)
                if (pos[v][2] < -1.0f || pos[v][2] > 1.0f) keep = false;
            if (!keep) zrej = 1;
        }
        if (keep) {
            // pushVertex (rasterizer.cpp:122-139)
            const int hw = W / 2, hh = H / 2;
            float vx[3], vy[3];
            bool bad = false;
#pragma unroll
            for (int v = 0; v < 3; v++) {
                vy[v] = ((float)hh * pos[v][1]) + (float)hh;
                vx[v] = ((float)hw * pos[v][0]) + (float)hw;
                // rows outside the int range make the reference read rows it
                // never wrote (or crash); the triangle is dropped
                if (!(vy[v] >= -2147483648.0f && vy[v] < 2147483648.0f)) bad = true;
            }
            int first = ps_cvt_i32(vy[0]), last = first;
#pragma unroll
            for (int v = 1; v < 3; v++) {
                if (vy[v] > (float)last) last = ps_cvt_i32(vy[v]);
                else if (vy[v] < (float)first) first = ps_cvt_i32(vy[v]);
            }
            if (first >= H || last < 0) { first = 0; last = -1; }
            if (first < 0) first = 0;
            if (last >= H) last = H - 1;
            if (bad || first == last) { keep = false; dropped = 1; }
            if (keep) {
                uint32_t code;
                int split = H;
                if (vy[0] == vy[1]) {
                    code = (vx[0] < vx[1]) ? (0u | (1u << 2) | (2u << 4)) : (1u | (0u << 2) | (2u << 4));
                } else if (vy[0] == vy[2]) {
                    code = (vx[0] < vx[2]) ? (0u | (2u << 2) | (1u << 4)) : (2u | (0u << 2) | (1u << 4));
                } else if (vy[1] == vy[2]) {
                    code = (vx[1] < vx[2]) ? (1u | (2u << 2) | (0u << 4)) : (2u | (1u << 2) | (0u << 4));
                } else {
                    int top, bottom, third = 2;
                    if (vy[0] > vy[1]) { top = 0; bottom = 1; } else { top = 1; bottom = 0; }
                    if (ps_sel3(vy, top) < ps_sel3(vy, third)) { int s = top; top = third; third = s; }
                    else if (ps_sel3(vy, bottom) > ps_sel3(vy, third)) { int s = bottom; bottom = third; third = s; }
                    PsEdge tt = ps_edge(vx, vy, top, third), tb = ps_edge(vx, vy, top, bottom);
                    float y3 = ps_sel3(vy, third);
                    bool left = ps_edge_eval(tb, y3) > ps_edge_eval(tt, y3);
                    code = (uint32_t)top | ((uint32_t)bottom << 2) | ((uint32_t)third << 4) | 64u | (left ? 128u : 0u);
                    // last row of the lower half: processTriangle's iyMax for yMax = third.y
                    split = y3 > (float)(H - 1) ? H - 1 : ps_cvt_i32(y3);
                }
#pragma unroll
                for (int v = 0; v < 3; v++) { tr.vx[v] = vx[v]; tr.vy[v] = vy[v]; tr.rw[v] = rw[v]; tr.z[v] = z[v]; }
                tr.first = first;
                tr.nrows = last - first + 1;
                tr.split = split;
                tr.code = code | ((uint32_t)di << 8);
                tr.view = d.view;
                tr.vflags = (uint32_t)(d.behavior & 3) | (d.writes_colour ? 4u : 0u) | (uint32_t)K << 4;
                tr.vary = (int)t + d.vary_delta;
                tr.pad = 0;
                n = (uint32_t)(last - first + 1);
                // a triangle without rows has no spans: nothing reads its records
                // (rows can lie outside the vertices' y range, where edges
                // extrapolate, so no x range test is safe here)
                pieces = n > 0;
                if (pieces) tris[t] = tr;
                if (!SHARE && pieces) {   // staged: the wave stores whole triangles below
#pragma unroll
                    for (int v = 0; v < 3; v++)
#pragma unroll
                        for (int k = 0; k < P::NV; k++) wl[lane * n3 + v * nvs + k] = u[v][k];
                }
                if constexpr (P::GRAD) if (pieces) {   // screen gradients for the mip level, once per triangle
                    float g[6];
                    ps_tri_grad(tr, u[0], u[1], u[2], P::IU, g);
                    float4* go = (float4*)(grads + t * 8);
                    go[0] = make_float4(g[0], g[1], g[2], g[3]);
                    go[1] = make_float4(g[4], g[5], 0.0f, 0.0f);
                }
            }
        }
        nrows[t] = n;
        myrows = n;
        // varyings of triangles with rows, or of all when other views read them
        stage = SHARE ? !skip && (pieces || d.vary_all) : pieces;
        if (SHARE && stage) {
#pragma unroll
            for (int v = 0; v < 3; v++)
#pragma unroll
                for (int k = 0; k < P::NV; k++) wl[lane * n3 + v * nvs + k] = u[v][k];
        }
    }
    };
    ps_with_draw(draws, di, [&](const PsDraw& d) {
        if constexpr (PROG != 0) {
            triangle(std::integral_constant<int, PROG>(), d);
        } else {
#define SU_ONE(K) triangle(std::integral_constant<int, K>(), d);
            PS_SETUP_PROGS(SU_ONE)
#undef SU_ONE
        }
    });
    // varyings of the wave's staged triangles: the wave's slots are one
    // contiguous block of 64 * 3*nvs floats, stored 16 bytes per lane and
    // instruction.  A float is written only when its triangle staged; floats
    // past NV of a staged vertex receive what the LDS holds, and nothing reads
    // them.
    const uint64_t m = __ballot(stage);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (m) {
        const int64_t tw = t - lane;
        const int nf = (int)min((int64_t)PS_WAVE, T - tw) * n3;   // the wave's floats
        const float rn3 = 1.0f / (float)n3;   // (f + 0.5) * rn3 floors to f / n3 exactly for f < 64 * 60
        float* dst = vary + tw * n3;
        auto staged = [&](int f) { return (m >> (int)(((float)f + 0.5f) * rn3)) & 1ull; };
        for (int f = lane * 4; f < nf; f += 4 * PS_WAVE) {
            if (f + 4 <= nf && staged(f) && staged(f + 3)) {
                *(float4*)(dst + f) = *(const float4*)(wl + f);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (f + j < nf && staged(f + j)) dst[f + j] = wl[f + j];
            }
        }
    }
    ps_wave_add(cnt, PS_ST_CULLED, culled, true);
    ps_wave_add(cnt, PS_ST_ZREJ, zrej, true);
    ps_wave_add(cnt, PS_ST_DROPPED, dropped, true);
    const uint32_t w = __builtin_amdgcn_readlane(ps_wave_incl_scan(myrows), 63);
    if (lane == 0) wrows[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x == 0) row_part[blockIdx.x] = wrows[0] + wrows[1];
}

// ---------------------------------------------------------------------------
// exclusive scans of the tiles' counts (two 32-bit counts side by side) and of
// the triangles' row counts; out[n] = total
// ---------------------------------------------------------------------------
#define SCAN_ITEMS 16
#define SCAN_BLOCK (256 * SCAN_ITEMS)

// Most heavy tiles a flush of n tiles lists: no more than a third of them can
// hold three times the mean.  At 1,024 a 3840x2160 frame's list was full and
// half its longest tiles began 30 us into the kernel, which they ended at
// 64 us; with all of them listed, and whole chunks stored at once, at 45.
#define PS_HEAVY_MAX 4096
__host__ __device__ __forceinline__ int64_t ps_heavy_cap(int64_t n) { return n / 3 + 1 < PS_HEAVY_MAX ? n / 3 + 1 : PS_HEAVY_MAX; }

// Pieces that make a tile heavy: three times the flush's mean per tile (at
// least 96), not counting those of waves that hold a wide span (k_span).  The flush's pieces are k_span's 64-bit count in the pending
// statistics: ps_pend_pieces loads one stripe per lane,
// ps_wave_sum64 adds the wave's stripes.
__device__ __forceinline__ unsigned long long ps_pend_pieces(const PsCounters* c)
{
    static_assert(PS_STRIPES == 64, "one stripe per lane");
    return c->pend[threadIdx.x & 63][PS_ST_SEGS];
}

__device__ __forceinline__ unsigned long long ps_wave_sum64(unsigned long long x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// the wave's pieces rounded down to multiples of 256 (plenty for a
// threshold): a 32-bit DPP scan instead of 64-bit shuffles
__device__ __forceinline__ unsigned long long ps_pend_approx(unsigned long long stripe)
{
    const uint32_t p256 = (uint32_t)min(stripe >> 8, (unsigned long long)0x3ffffff);
    return (unsigned long long)__builtin_amdgcn_readlane(ps_wave_incl_scan(p256), 63) << 8;
}

__device__ __forceinline__ uint32_t ps_heavy_min(unsigned long long pieces, int64_t n_tiles)
{
    const unsigned long long h = 3 * pieces / (unsigned long long)(n_tiles > 0 ? n_tiles : 1);
    return (uint32_t)min(max(h, 96ull), 0xffffffffull);
}

// inclusive wave scan of the two 32-bit halves separately (the packed counts
// never carry from the low half)
__device__ __forceinline__ unsigned long long ps_wave_incl_scan2(unsigned long long v)
{
    return (unsigned long long)ps_wave_incl_scan((uint32_t)v) |
           ((unsigned long long)ps_wave_incl_scan((uint32_t)(v >> 32)) << 32);
}

__device__ __forceinline__ unsigned long long ps_readlane64(unsigned long long v, int lane)
{
    return (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((uint32_t)v, lane) |
           ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((uint32_t)(v >> 32), lane) << 32);
}

// exclusive scan of one value per thread over a block of four waves
__device__ __forceinline__ unsigned long long ps_block_excl_scan(unsigned long long v, unsigned long long* lds,
                                                                 unsigned long long& total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long x = ps_wave_incl_scan2(v);
    if (lane == 63) lds[wave] = x;
    __syncthreads();
    unsigned long long wbase = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const unsigned long long l = lds[w];
        wbase += (w < wave) ? l : 0ull;
        total += l;
    }
    __syncthreads();
    return wbase + x - v;
}

// Wave-striped ownership: the wave owns items [wbase, wbase + 64 * SCAN_ITEMS),
// in groups of 128; in group g the lane owns the two consecutive items
// wbase + g * 128 + lane * 2 + j, so each group is one coalesced 16-byte load
// or store per lane.
__device__ __forceinline__ void ps_load_items(const unsigned long long* in, int64_t wbase, int64_t n, unsigned long long* v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g = 0; g < SCAN_ITEMS / 2; g++) {
        const int64_t i = wbase + (int64_t)g * 128 + lane * 2;
        if (i + 2 <= n) {
            const ulonglong2 u = *(const ulonglong2*)(in + i);
            v[g * 2] = u.x;
            v[g * 2 + 1] = u.y;
        } else {
            v[g * 2] = i < n ? in[i] : 0ull;
            v[g * 2 + 1] = 0ull;
        }
    }
}

// Heavy tiles among the lane's items (wave-striped as above): those of at
// least heavy_min pieces.
__device__ __forceinline__ uint32_t ps_heavy_count(int64_t wbase, int64_t n, const unsigned long long* v, uint32_t heavy_min)
{
    const int lane = threadIdx.x & 63;
    uint32_t nh = 0;
#pragma unroll
    for (int g = 0; g < SCAN_ITEMS / 2; g++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int64_t i = wbase + (int64_t)g * 128 + lane * 2 + j;
            nh += (i < n && (uint32_t)v[g * 2 + j] >= heavy_min) ? 1u : 0u;
        }
    return nh;
}

// The lane's first slot in the heavy list for its nh heavy tiles, reserved
// with one atomic per wave on heavy[0] (0xffffffff: the wave has none).
__device__ __forceinline__ uint32_t ps_heavy_reserve(uint32_t nh, uint32_t* heavy)
{
    const int lane = threadIdx.x & 63;
    const uint32_t incl = ps_wave_incl_scan(nh);
    const uint32_t tot = __builtin_amdgcn_readlane(incl, 63);
    if (!tot) return 0xffffffffu;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(heavy, tot);
    return __builtin_amdgcn_readlane(base, 0) + incl - nh;
}

// The wave's exclusive prefix of its items (from `run` on) into out.  With a
// heavy list (hslot given) it also lists the tiles of at least heavy_min pieces
// in heavy[1 ..], the lane's from slot hslot on (up to hcap are listed), and
// marks the listed ones with bit 63 of their start.
__device__ __forceinline__ void ps_store_scan(unsigned long long* out, int64_t wbase, int64_t n, const unsigned long long* v,
                                              unsigned long long run, uint32_t heavy_min, uint32_t* heavy, uint32_t hslot,
                                              uint32_t hcap)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g = 0; g < SCAN_ITEMS / 2; g++) {
        const unsigned long long v1 = v[g * 2 + 1], sum = v[g * 2] + v1;
        const unsigned long long x = ps_wave_incl_scan2(sum);
        const int64_t i = wbase + (int64_t)g * 128 + lane * 2;
        unsigned long long o[2] = {run + x - sum, run + x - v1};
#pragma unroll
        for (int j = 0; j < 2; j++)
            if (hslot != 0xffffffffu && i + j < n && (uint32_t)v[g * 2 + j] >= heavy_min) {
                if (hslot < hcap) {
                    heavy[1 + hslot] = (uint32_t)(i + j);
                    o[j] |= 1ull << 63;
                }
                hslot++;
            }
        if (i + 2 <= n) *(ulonglong2*)(out + i) = make_ulonglong2(o[0], o[1]);
        else if (i < n) out[i] = o[0];
        run += ps_readlane64(x, 63);
    }
}

// the head of list `lane` of the wide waves
__device__ __forceinline__ unsigned long long ps_wide_head(const unsigned long long* wide)
{
    static_assert(PS_WIDE_LISTS == 64, "one list per lane");
    return wide[PS_WIDE_STEP * (threadIdx.x & 63)];
}

// The tile scan adds 32-bit piece counts: when the flush's pieces, which k_span
// also counts in 64 bits into the pending statistics, do not fit, it reports
// the largest total and flags an overflow, so that the flush is split; so it
// does when they are more than seg_cap.  Called by the 64 lanes of one wave;
// head: the lane's of the wide lists.
__device__ __forceinline__ void ps_scan_total(unsigned long long tot, int64_t n, unsigned long long* out, uint32_t* total_out,
                                              unsigned long long head, unsigned long long* wide, int64_t seg_cap, PsCounters* c,
                                              int* flag, unsigned long long pieces)
{
    const int lane = threadIdx.x & 63;
    const uint32_t waves = (uint32_t)(head & PS_WIDE_COUNT), mine = (uint32_t)(head >> 20);
    const uint32_t w = ps_wave_incl_scan(waves), p = ps_wave_incl_scan(mine);
    wide[PS_WIDE_BEFORE + lane] = (unsigned long long)(w - waves) | (unsigned long long)(p - mine) << 32;
    if (lane == 63) wide[PS_WIDE_BEFORE + 64] = (unsigned long long)w | (unsigned long long)p << 32;
    if (lane != 63) return;
    out[n] = tot;
    // (a sum that wrapped has more than 2^32 pieces)
    const bool fits = pieces == (unsigned long long)(uint32_t)tot + p && pieces <= 0xffffffffull;
    const uint32_t total = fits ? (uint32_t)pieces : 0xffffffffu;
    *total_out = total;
    atomicMax(total_out + 2, total);
    if (!fits || (int64_t)pieces > seg_cap) ps_overflow(c, 1, flag);
}

__global__ void __launch_bounds__(256) k_scan_reduce(const unsigned long long* __restrict__ in, int64_t n,
                                                     unsigned long long* __restrict__ partial, const PsCounters* c)
{
    __shared__ unsigned long long lds[4];
    const int64_t wbase = blockIdx.x * (int64_t)SCAN_BLOCK + (int64_t)(threadIdx.x >> 6) * (64 * SCAN_ITEMS);
    unsigned long long s = 0;
    if (!ps_poisoned(c) && wbase < n) {
        unsigned long long v[SCAN_ITEMS];
        ps_load_items(in, wbase, n, v);
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; i++) s += v[i];
    }
    unsigned long long tot;
    ps_block_excl_scan(s, lds, tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// sum of partial[0, end) over a 256-thread block
__device__ __forceinline__ unsigned long long ps_block_sum_prefix(const unsigned long long* partial, int end,
                                                                  unsigned long long* lds)
{
    unsigned long long s = 0;
#pragma unroll 8
    for (int i = threadIdx.x; i < end; i += 256) s += partial[i];
    unsigned long long tot;
    ps_block_excl_scan(s, lds, tot);
    return tot;
}

// block b: prefix of the partial sums before it (one per block of items),
// then the block's own scan.  Block 0 also writes the total.  The overflow flag
// is tested only before the first store: the loads stay in bounds either way,
// so its round trip overlaps theirs.
__global__ void __launch_bounds__(256) k_scan_final(const unsigned long long* __restrict__ in, int64_t n,
                                                    const unsigned long long* __restrict__ partial, int nb,
                                                    unsigned long long* __restrict__ out, uint32_t* total_out,
                                                    unsigned long long* wide, int64_t seg_cap, PsCounters* c, uint32_t* heavy,
                                                    int* flag)
{
    __shared__ unsigned long long lds[4];
    const bool poisoned = ps_poisoned(c);
    const unsigned long long pend = ps_pend_pieces(c);
    const bool totals = blockIdx.x == 0 && threadIdx.x < 64;   // the wave that writes them
    const unsigned long long head = totals ? ps_wide_head(wide) : 0ull;
    const int64_t wbase = blockIdx.x * (int64_t)SCAN_BLOCK + (int64_t)(threadIdx.x >> 6) * (64 * SCAN_ITEMS);
    unsigned long long v[SCAN_ITEMS];
    ps_load_items(in, wbase, n, v);
    unsigned long long total = 0, before = 0;
    if (blockIdx.x == 0) total = ps_block_sum_prefix(partial, nb, lds);
    else before = ps_block_sum_prefix(partial, blockIdx.x, lds);
    if (poisoned) return;
    const unsigned long long pieces = ps_wave_sum64(pend);
    if (totals) ps_scan_total(total, n, out, total_out, head, wide, seg_cap, c, flag, pieces);
    unsigned long long s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) s += v[i];
    unsigned long long tot;
    // the waves before this one: the block scan of the lane sums, taken at lane 0
    const unsigned long long wpre = ps_block_excl_scan(s, lds, tot);
    uint32_t hm = 0xffffffffu, hslot = 0xffffffffu;
    if (heavy) {
        hm = ps_heavy_min(ps_pend_approx(pend), n);
        hslot = ps_heavy_reserve(ps_heavy_count(wbase, n, v, hm), heavy);
    }
    ps_store_scan(out, wbase, n, v, before + ps_readlane64(wpre, 0), hm, heavy, hslot, (uint32_t)ps_heavy_cap(n));
}

// One pass for tile counts up to SCAN_DIRECT_MAX.  Blocks of 16 waves; each
// lane owns two adjacent tiles (one 16-byte load), so a block covers
// DIRECT_BLOCK tiles and a wave needs one wave scan.  Block b adds the counts
// before its own tiles directly (up to 8 16-byte loads per thread in flight
// at a time, one round trip below 16k tiles) and counts the heavy tiles among
// them on the way, so each lane knows its slots in the heavy list without
// atomics (the list is in tile order).  The waves combine their totals in
// one LDS exchange; the last block writes the totals.
#define DIRECT_BLOCK 2048
#define SCAN_DIRECT_MAX (32 * DIRECT_BLOCK)
struct PsDirectWave {
    unsigned long long pre, own;   // counts before the block (the wave's share), the wave's own tiles
    uint32_t hpre, hown;           // heavy tiles among them
};
__global__ void __launch_bounds__(1024) k_scan_direct(const unsigned long long* __restrict__ in, int64_t n,
                                                      unsigned long long* __restrict__ out, uint32_t* total_out,
                                                      unsigned long long* wide, int64_t seg_cap, PsCounters* c,
                                                      uint32_t* heavy, int* flag)
{
    typedef unsigned long long T;
    __shared__ PsDirectWave xw[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // tested before the first store: every load stays in bounds either way,
    // so the flag's round trip overlaps theirs
    const bool poisoned = ps_poisoned(c);
    const int64_t b0 = blockIdx.x * (int64_t)DIRECT_BLOCK;
    const int64_t i = b0 + 2 * (int64_t)threadIdx.x;   // the lane's tiles i, i + 1
    const T a = in[min(i, n - 1)], b = in[min(i + 1, n - 1)];
    // tiles before the block: 8 loads per chunk, addresses past b0 clamped
    // (b0 - 2, a multiple of DIRECT_BLOCK less 2) and their values dropped
    const int nk = (int)(b0 / DIRECT_BLOCK);   // 16-byte loads per thread in all
    ulonglong2 u[8];
    auto chunk_load = [&](int k0) {
#pragma unroll
        for (int k = 0; k < 8; k++)
            u[k] = *(const ulonglong2*)(in + min(((int64_t)(k0 + k) * 1024 + threadIdx.x) * 2, b0 - 2));
    };
    if (nk > 0) chunk_load(0);
    const unsigned long long pend = ps_pend_pieces(c);   // after the loads: one wait covers them all
    const bool totals = blockIdx.x == gridDim.x - 1 && wave == 0;   // the wave that writes them
    const unsigned long long head = totals ? ps_wide_head(wide) : 0ull;
    const uint32_t hm = heavy ? ps_heavy_min(ps_pend_approx(pend), n) : 0xffffffffu;
    T pre = 0;
    uint32_t hpre = 0;
    for (int k0 = 0; k0 < nk; k0 += 8) {
        if (k0 > 0) chunk_load(k0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const bool ok = k0 + k < nk;
            const T x = ok ? u[k].x : 0ull, y = ok ? u[k].y : 0ull;
            pre += x + y;
            hpre += ((uint32_t)x >= hm ? 1u : 0u) + ((uint32_t)y >= hm ? 1u : 0u);   // hm >= 96: dropped values never count
        }
    }
    if (poisoned) return;
    const T va = i < n ? a : 0ull, vb = i + 1 < n ? b : 0ull;
    const uint32_t ha = (uint32_t)va >= hm ? 1u : 0u, hb = (uint32_t)vb >= hm ? 1u : 0u;
    // the wave's inclusive scans of its own tiles and heavy marks, and its
    // totals before the block
    const T own = ps_wave_incl_scan2(va + vb);
    const uint32_t hown = ps_wave_incl_scan(ha + hb);
    const T pre_w = ps_wave_incl_scan2(pre);
    const uint32_t hpre_w = ps_wave_incl_scan(hpre);
    if (lane == 63) xw[wave] = PsDirectWave{pre_w, own, hpre_w, hown};
    __syncthreads();
    T before = 0, woff = 0, btot = 0;
    uint32_t hbefore = 0, hwoff = 0, hbtot = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) {
        const PsDirectWave e = xw[w];
        before += e.pre;
        hbefore += e.hpre;
        woff += w < wave ? e.own : 0ull;
        hwoff += w < wave ? e.hown : 0u;
        btot += e.own;
        hbtot += e.hown;
    }
    T r = before + woff + own - (va + vb);                 // tile i's start
    uint32_t hs = hbefore + hwoff + hown - (ha + hb);      // its first heavy slot
    T oa = r, ob = r + va;
    if (heavy) {
        const uint32_t hcap = (uint32_t)ps_heavy_cap(n);
        if (ha && hs < hcap) { heavy[1 + hs] = (uint32_t)i; oa |= 1ull << 63; }
        hs += ha;
        if (hb && hs < hcap) { heavy[1 + hs] = (uint32_t)(i + 1); ob |= 1ull << 63; }
    }
    if (i + 2 <= n) {
        *(ulonglong2*)(out + i) = make_ulonglong2(oa, ob);
    } else if (i < n) {
        out[i] = oa;
    }
    if (totals) {
        ps_scan_total(before + btot, n, out, total_out, head, wide, seg_cap, c, flag, ps_wave_sum64(pend));
        if (heavy && lane == 0) heavy[0] = hbefore + hbtot;
    }
}

// Row scan from per-block partial sums (partial i sums items [i * pgran,
// (i + 1) * pgran), pgran dividing SCAN_BLOCK): blocks of 16 waves, each lane
// owning four adjacent items (one 16-byte load), so a block covers
// SCAN_BLOCK items and a wave needs one wave scan.  Block b adds the partials
// before it (two loads per thread below 2048 of them), the waves combine in
// one LDS exchange, and the last block writes the total.
struct PsRowWave {
    uint32_t pre, own;
};
__global__ void __launch_bounds__(1024) k_scan_parts(const uint32_t* __restrict__ in, int64_t n,
                                                     const uint32_t* __restrict__ partial, int pgran,
                                                     uint32_t* __restrict__ out, uint32_t* total_out,
                                                     uint32_t* __restrict__ bstart, int64_t bcap, unsigned long long* wide)
{
    __shared__ PsRowWave xw[16];
    if (blockIdx.x == 0 && threadIdx.x < PS_WIDE_LISTS) wide[PS_WIDE_STEP * threadIdx.x] = 0;   // for k_span
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i = blockIdx.x * (int64_t)SCAN_BLOCK + 4 * (int64_t)threadIdx.x;   // items i .. i + 3
    uint32_t v[4];
    if (i + 4 <= n) {
        const uint4 q = *(const uint4*)(in + i);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = in[min(i + j, n - 1)];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = i + j < n ? v[j] : 0u;
    }
    const int np = blockIdx.x * (SCAN_BLOCK / pgran);   // partials before the block
    uint32_t pre = 0;
#pragma unroll 4
    for (int k = threadIdx.x; k < np; k += 1024) pre += partial[k];
    const uint32_t sum = v[0] + v[1] + v[2] + v[3];
    const uint32_t own = ps_wave_incl_scan(sum);
    const uint32_t pre_w = ps_wave_incl_scan(pre);
    if (lane == 63) xw[wave] = PsRowWave{pre_w, own};
    __syncthreads();
    uint32_t before = 0, woff = 0, btot = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) {
        const PsRowWave e = xw[w];
        before += e.pre;
        woff += w < wave ? e.own : 0u;
        btot += e.own;
    }
    uint32_t r = before + woff + own - sum;
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) { o[j] = r; r += v[j]; }
    // the triangle of every 64th row item: item 64b lies in item i + j's rows
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (i + j >= n) break;
        const int64_t b1 = min(((int64_t)o[j] + v[j] + 63) >> 6, bcap);
        for (int64_t b = ((int64_t)o[j] + 63) >> 6; b < b1; b++) bstart[b] = (uint32_t)(i + j);
    }
    if (i + 4 <= n) {
        *(uint4*)(out + i) = make_uint4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i + j < n) out[i + j] = o[j];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        out[n] = before + btot;
        *total_out = before + btot;
        atomicMax(total_out + 2, before + btot);
    }
}

// Triangle of row item i: the t with row_off[t] <= i < row_off[t + 1]
// (row_off is the exclusive scan of the row counts, row_off[T] = R).  The
// wave finds the triangle of its lowest unresolved item with a 64-way search
// over row_off (64 pivots per step, a few dependent loads), holds the next 64
// row starts one per lane, and every lane counts those at or below its own
// item with a 6-step search over the lanes.  Lanes whose item lies beyond
// that window go round again from the lowest of them, so every round
// resolves at least one lane and runs of triangles without rows are jumped.
// All lanes of the wave call it; i0 is the wave's first item.
// Flushes that search hold fewer than 2^31 triangles and R < 2^26 row items,
// so the arithmetic is 32-bit.  hint, when not negative, is the triangle of
// item i0 and hint_hi that of item i0 + 64 (the row scan's table of every
// 64th item's triangle): the first round then takes the 64 row starts after
// hint without a search, and a later one searches only up to hint_hi.
__device__ __forceinline__ int ps_row_tri(const uint32_t* __restrict__ row_off, int T, uint32_t R, uint32_t i0, int hint,
                                          int hint_hi)
{
    const int lane = threadIdx.x & 63;
    const uint32_t i = i0 + lane;
    int found = -1;
    uint64_t pend = __ballot(i < R);
    const int lo0 = hint > 0 ? hint : 0;
    const int hi0 = hint >= 0 && hint_hi >= 0 ? hint_hi + 1 : T;
    bool guess = hint >= 0;
    while (pend) {
        const uint32_t tgt = i0 + __builtin_ctzll(pend);
        int lo = lo0, hi = guess ? lo0 + 1 : hi0;   // row_off[lo] <= tgt; hi == T or row_off[hi] > tgt
        guess = false;
        while (hi - lo > 1) {
            const int step = (hi - lo + 63) >> 6;
            const int p = lo + lane * step;
            const bool le = p < hi && row_off[p] <= tgt;
            const int c = __popcll(__ballot(le));
            const int nhi = lo + c * step;
            lo += (c - 1) * step;
            hi = nhi < hi ? nhi : hi;
        }
        const int we = lo + 1 + lane;
        const uint32_t e = we <= T ? row_off[we] : 0xffffffffu;   // above every item (R < 2^26)
        int pos = 0;   // row starts of the window at or below i: 0..63, or 64 past it
#pragma unroll
        for (int st = 32; st >= 1; st >>= 1) {
            const uint32_t v = (uint32_t)__shfl((int)e, pos + st - 1, 64);
            if (v <= i) pos += st;
        }
        if ((uint32_t)__builtin_amdgcn_readlane((int)e, 63) <= i) pos = 64;
        if (found < 0 && i < R && i >= tgt && pos < 64) found = lo + pos;
        pend = __ballot(found < 0 && i < R);
    }
    return found;
}

// ---------------------------------------------------------------------------
// span setup
// ---------------------------------------------------------------------------
// Spans at least this long keep varying checkpoints at each later piece, so
// that shading never replays more than about this many pixels; shorter spans
// are replayed from x1.
#define PS_CK_MIN 48
__device__ __forceinline__ bool ps_span_has_ck(const PsSpan& sp) { return sp.x2 - sp.x1 + 1 >= PS_CK_MIN; }

#define SPAN_BINS 512
// The spans of a wave of span items whose longest has at least this many pixels
// are placed by k_segments span by span, with a lane per accumulator instead of
// a span per lane.
// This is also where spans start to keep varying checkpoints, so only those
// waves carry varyings (24 to 96 measure alike; below 40 a small sphere's
// frame, whose spans are mostly that long, loses 3 us).
#define PS_WIDE_MIN PS_CK_MIN
#define PS_TC_RUN (1ull << 32)
// called by every lane of the wave; n: the lane's span's pixels, if it has one
__device__ __forceinline__ bool ps_wave_wide(bool has, uint32_t n) { return __any(has && n >= PS_WIDE_MIN); }

// Also counts, per tile, the pieces in it and the waves (of 64 span items) that
// have some there, each of which writes them as one run: tcnt[t] += pieces |
// waves << 32.  Waves that hold a wide span count their runs only
// and go on the lists `wide`; their pieces lie after those of all other waves.
// Eight waves per SIMD (64 VGPRs, no spill): at seven the 256-view batch's span
// pass took 1.55 ms instead of 1.21.
__global__ void __launch_bounds__(256, 8) k_span(const PsTri* __restrict__ tris,
                                              const uint32_t* __restrict__ row_off, const uint32_t* __restrict__ bstart,
                                              int64_t T, int64_t cap,
                                              PsSpan* __restrict__ spans, unsigned long long* __restrict__ tcnt,
                                              const PsView* __restrict__ views, int n_views, int chunk_w, int tile_rows,
                                              int tile_cols, uint32_t* heavy, unsigned long long* wide, PsCounters* cnt, int* flag)
{
    // per wave: piece counts of the tiles [kmin, kmin + SPAN_BINS) its spans touch
    __shared__ uint32_t bins_all[4][SPAN_BINS];
    uint32_t* bins = bins_all[threadIdx.x >> 6];
    const int lane = threadIdx.x & (PS_WAVE - 1);
    const bool poisoned = ps_poisoned(cnt);
    const int64_t R = row_off[T];
    // the only view of a one-view flush, read once (otherwise each triangle's)
    int64_t tb1 = 0;
    int ntx1 = 0, W1 = 0;
    if (n_views == 1) { tb1 = views[0].tile_base; ntx1 = views[0].n_tiles_x; W1 = views[0].W; }
    if (poisoned) return;
    if (heavy && blockIdx.x == 0 && threadIdx.x == 0) heavy[0] = 0;   // the two-pass tile scan lists heavy tiles atomically
    if (R > cap) {   // more rows than span records: flag it, write nothing
        if (threadIdx.x == 0 && blockIdx.x == 0) ps_overflow(cnt, 1, flag);
        return;
    }
    uint32_t all_spans = 0, all_pieces = 0, all_frags = 0;   // the lane's statistics, added up once per wave
    for (int64_t base = blockIdx.x * (int64_t)blockDim.x; base < R; base += (int64_t)gridDim.x * blockDim.x) {
        int64_t i = base + threadIdx.x;
        uint32_t nspan = 0, nfrag = 0;
        // the item's triangle, searched in row_off from the row scan's table
        const int64_t i0 = base + (threadIdx.x & ~63);
        const bool tab = i0 < R;
        const int tw = ps_row_tri(row_off, (int)T, (uint32_t)R, (uint32_t)i0, tab ? (int)bstart[i0 >> 6] : -1,
                                  tab && i0 + 64 < R ? (int)bstart[(i0 >> 6) + 1] : -1);
        PsSpanTiles st = {};
        bool has = false;
        if (i < R) {
            const int t = tw;
            const PsTri tr = tris[t];
            int64_t vtb = tb1;
            int vntx = ntx1, W = W1;
            if (n_views != 1) { const PsView& v = views[tr.view]; vtb = v.tile_base; vntx = v.n_tiles_x; W = v.W; }
            int row = tr.first + (int)(i - (int64_t)row_off[t]);
            PsEdge L, Rr;
            ps_row_edges(tr, row, L, Rr);
            int left = ps_cvt_i32(ps_edge_eval(L, (float)row) + 0.5f);
            int right = ps_cvt_i32(ps_edge_eval(Rr, (float)row) + 0.5f);
            PsSpan sp;
            sp.tri = -1;
            if (left != right) {   // drawvao.cpp:72-75
                nspan = 1;
                int x1 = left < 0 ? 0 : left;
                int x2 = right >= W ? W - 1 : right;
                if (x1 <= x2) {
                    PsSpanGeom g;
                    ps_span_geom(tr, row, left, right, L, Rr, g);
                    ps_span_vis(tr, g, sp.cf2, sp.cf2_step, sp.pz, sp.pz_step);
                    sp.tri = t;
                    sp.y = row | (int)((tr.vflags & 3u) << 24) | (int)(((tr.vflags >> 2) & 1u) << 28);
                    sp.x1 = x1;
                    sp.x2 = x2;
                    nfrag = (uint32_t)(x2 - x1 + 1);
                    st = ps_span_tiles(vtb, vntx, tile_rows, tile_cols, chunk_w, row, x1, x2);
                    has = true;
                }
            }
            spans[i] = sp;
        }
        const uint32_t npieces = has ? (uint32_t)(st.cx1 - st.cx0 + 1) : 0u;
        all_spans += nspan;
        all_pieces += npieces;
        all_frags += nfrag;
        const bool in_wide = ps_wave_wide(has, nfrag);
        if (in_wide) {
            const uint32_t n = __builtin_amdgcn_readlane(ps_wave_incl_scan(npieces), 63);
            if (lane == 0) {
                const uint32_t w = (uint32_t)(i0 >> 6), l = w % PS_WIDE_LISTS;
                const unsigned long long old = atomicAdd(wide + PS_WIDE_STEP * l, (unsigned long long)n << 20 | 1ull);
                wide[PS_WIDE_REC + PS_WIDE_PER(cap) * l + (int64_t)(old & PS_WIDE_COUNT)] = w | (old >> 20) << 32;
            }
        }
        // per tile of the wave's spans: its pieces there and one run.  When
        // the wave's tiles lie within SPAN_BINS of each other (about nine
        // tiles of one or two tile rows, typically), the lanes add their
        // pieces into LDS bins and one atomic per touched bin follows;
        // otherwise the wave visits its tiles in rounds (lane j adds the
        // j-th tile's counts, so a batch of tiles is one atomic), or, if it
        // holds a wide span, counts one run for each tile that some span covers.
        const uint32_t kmin = ps_wave_min(has ? st.g0 : 0xffffffffu);
        const uint32_t kmax = ps_wave_max(has ? st.g1 : 0u);
        if (kmin != 0xffffffffu && kmax - kmin < (uint32_t)SPAN_BINS) {
            const uint32_t nbin = kmax - kmin + 1;
            for (uint32_t b = lane; b < nbin; b += PS_WAVE) bins[b] = 0;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (has)
                for (uint32_t k = st.g0; k <= st.g1; k++) {
                    int lo, hi;
                    ps_span_tile_chunks(st, tile_cols, k, lo, hi);
                    atomicAdd(&bins[k - kmin], (uint32_t)(hi - lo + 1));
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            for (uint32_t b = lane; b < nbin; b += PS_WAVE) {
                const uint32_t c = bins[b];
                if (c) atomicAdd(&tcnt[kmin + b], in_wide ? PS_TC_RUN : (unsigned long long)c | PS_TC_RUN);
            }
            // the next iteration clears the bins only after every lane read them
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else if (in_wide) {
            // Tile row by tile row, 64 tiles at a time: each span marks in LDS
            // where it begins and ends, and sums along the row tell the tiles
            // that some span covers.  (In rounds a wave across a 1080p screen
            // makes 540: 68 us for two triangles, now 11.  Each span looking
            // through the others of its row took 84 us where this takes 37,
            // 1080p terrain in tiles of 1x64, and 243 against 32, the demo
            // scene in them.)
            const uint32_t base_t = st.g0 - (uint32_t)st.tx0;
            const int first_t = st.tx0, last_t = st.tx0 + (int)(st.g1 - st.g0);
            for (uint64_t todo = __ballot(has); todo;) {
                const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)base_t, __builtin_ctzll(todo));
                const bool in_row = has && base_t == r;
                todo &= ~__ballot(in_row);
                const int from = (int)ps_wave_min(in_row ? (uint32_t)first_t : 0xffffffffu), to = (int)ps_wave_max(in_row ? (uint32_t)last_t : 0u);
                for (int w0 = from; w0 <= to; w0 += PS_WAVE) {
                    bins[lane] = 0;
                    ps_lds_turn();
                    if (in_row && first_t < w0 + PS_WAVE && last_t >= w0) {
                        atomicAdd(&bins[max(first_t - w0, 0)], 1u);
                        if (last_t + 1 < w0 + PS_WAVE) atomicAdd(&bins[last_t + 1 - w0], 0xffffffffu);
                    }
                    ps_lds_turn();
                    if (ps_wave_incl_scan(bins[lane])) atomicAdd(&tcnt[r + (uint32_t)(w0 + lane)], PS_TC_RUN);
                    ps_lds_turn();
                }
            }
        } else {
            uint32_t cur = has ? st.g0 : 0xffffffffu;
            for (;;) {
                uint32_t bk, bn;
                const int nb = ps_wave_tile_batch(st, tile_cols, cur, bk, bn);
                if (lane < nb) atomicAdd(&tcnt[bk], (unsigned long long)bn | PS_TC_RUN);
                if (nb < PS_WAVE) break;
            }
        }
    }
    ps_wave_add(cnt, PS_ST_SPANS, all_spans, true);
    ps_wave_add(cnt, PS_ST_SEGS, all_pieces, true);
    ps_wave_add(cnt, PS_ST_FRAGS, all_frags, true);
}

// ---------------------------------------------------------------------------
// segments: (bin key, span) pairs
// ---------------------------------------------------------------------------
// One thread per span: the span's pieces per bin chunk, in order.  The walk
// from x1 applies the serial `+= step` of the pixel loop (interp.cpp:82-92)
// pixel by pixel, so each piece starts with exactly the accumulators the
// reference holds at its first pixel; wide spans of colour-writing draws also
// keep the varying accumulators at each later piece.
// Placement, in the waves without a wide span: the wave visits its tiles in
// increasing order, SG_BATCH at a time.  Per tile, each lane's pieces go after those of the lanes before it
// (offsets kept in LDS), and lane j reserves the j-th tile's run of
// consecutive pieces with one atomic on the tile's counter (counting down
// from k_span's count), all lanes at once.  Then every lane walks its pieces
// of the batch's tiles into their slots; a span's tiles are consecutive in
// the visit order, so each walk goes on from tile to tile.
#define SG_BATCH 16
// The record of a run of n pieces from `first` on, the one that a tile with
// `left` runs still to take and runs up to `end` takes; false if it has none
// left or the pieces lie outside.
__device__ __forceinline__ bool ps_put_run(const PsFrame& f, uint32_t left, unsigned long long end, uint32_t first, uint32_t n,
                                           uint32_t wave_id, int64_t cap)
{
    if (left == 0u || (uint64_t)first + n > (uint64_t)cap) return false;
    *(uint2*)(f.runs + 2 * (size_t)((uint32_t)(end >> 32) - left)) = make_uint2(first, wave_id << 12 | (n - 1u));
    return true;
}

// Takes a run of n pieces of tile k off the tile's counter and writes its
// record.  The tile's pieces that k_span counted are those of its runs in the
// order they are taken; returns the run's first.  The counts must cover the run
// (they always do: both kernels visit the same tiles); 0xffffffff, and the
// flag set, if they do not: never write outside.
__device__ __forceinline__ uint32_t ps_take_run(const PsFrame& f, unsigned long long* tcnt, uint32_t k, uint32_t n,
                                                uint32_t wave_id, int64_t cap, PsCounters* cnt, int* flag)
{
    const unsigned long long left = atomicAdd(&tcnt[k], 0ull - (n | PS_TC_RUN));
    const unsigned long long end = PS_TS(f.tstart[k + 1]);
    const uint32_t first = (uint32_t)end - (uint32_t)left;
    const uint32_t slot = (uint32_t)(end >> 32) - (uint32_t)(left >> 32);
    if ((uint32_t)left < n || (uint32_t)(left >> 32) == 0u || (uint64_t)first + n > (uint64_t)cap) {
        ps_overflow(cnt, 2, flag);
        return 0xffffffffu;
    }
    f.runs[2 * (size_t)slot] = first;  // two stores: as one, 123 us where this takes 119 (32 views)
    f.runs[2 * (size_t)slot + 1] = wave_id << 12 | (n - 1u);
    return first;
}

// Spans of the listed waves (those that hold a wide span): G (16 or 32) lanes
// a span, each carrying one accumulator, so that a span of n pixels takes n
// dependent adds whatever its varyings, and the spans of a listed wave spread
// over as many waves of the grid.  With a span per lane, a lane stepped up to
// 22 accumulators a pixel while the lanes whose spans lie in other tile rows
// waited: 24 objects and a full-view quad at 1366x768 took 2,830 us, now 38
// (1920x1080 terrain with spans of over 1,000 pixels, 8-pixel tiles: 93 -> 33);
// what is left is the chain of a span's loads and adds.
// Lane j of the group holds word j of the span's piece records (PsSeg: 2 is
// cf2, 3 the depth numerator) and, from 8 on, varying j - 8, so a piece is one
// store.
// A wave's pieces of a tile are one run here too, although its spans are
// placed by waves that know nothing of each other: a listed wave's pieces are
// one block (its first piece is on the list), ordered by tile row, tile and
// span, so that the place of each follows from the chunks that the wave's 64
// spans cover, one per lane.  The first span in a tile writes the run's record.
// (A run for each span, placed among the tile's own pieces, made eight of one,
// and sorting them was most of the raster kernel: 48 triangle pairs across
// 1920x1080 1,514 us there, now 279; frames of 4,000 triangles of 60 to 240
// pixels 1,150 -> 647, of 200,000 small ones with each fifth 60 pixels wide
// 3,470 -> 1,580.)
template <int G>
__device__ __forceinline__ void ps_wide_spans(const PsSpan* __restrict__ spans, int64_t R, const PsFrame& f,
                                              const PsTri* __restrict__ tris, const PsDraw* __restrict__ draws,
                                              const float* __restrict__ vary, int nvs, const unsigned long long* __restrict__ wide,
                                              int64_t wide_per, uint32_t listed, uint32_t narrow, int64_t tb1,
                                              int ntx1, unsigned long long* __restrict__ tcnt, PsSeg* __restrict__ segs,
                                              float* __restrict__ ck, int64_t cap, uint32_t* lds, PsCounters* cnt, int* flag)
{
    constexpr int SPW = 64 / G;
    static_assert(SPW * (G + 1) <= 4 * PS_WAVE && 6 * PS_WAVE <= SG_BATCH * PS_WAVE, "the wave's LDS");
    const int lane = threadIdx.x & (PS_WAVE - 1), j = lane & (G - 1), grp = lane & ~(G - 1);
    const int CW = f.chunk_w, TC = f.tile_cols, cw_shift = __builtin_ctz((unsigned)CW), tc_shift = __builtin_ctz((unsigned)TC);
    // what is before list `lane` waits in LDS, out of the registers
    uint2* before_list = (uint2*)(lds + PS_WAVE * 4);
    before_list[lane] = *(const uint2*)(wide + PS_WIDE_BEFORE + lane);
    const uint32_t units = listed * G;
    // the first unit goes to the first wave that has fewer items than the one
    // before it (or none), when the rest of the kernel deals them out
    const uint32_t stride = gridDim.x * (blockDim.x / PS_WAVE), less = (uint32_t)((R + PS_WAVE - 1) / PS_WAVE) % stride;
    const uint32_t id = blockIdx.x * (blockDim.x / PS_WAVE) + threadIdx.x / PS_WAVE;
    for (uint32_t u = id >= less ? id - less : id + stride - less; u < units; u += stride) {
        ps_lds_turn();
        const uint2 bl = before_list[lane];
        const int l = __popcll(__ballot(bl.x <= u / G)) - 1;   // the last list that begins at or before it
        const unsigned long long rec = wide[PS_WIDE_REC + wide_per * l + (u / G - (uint32_t)__builtin_amdgcn_readlane((int)bl.x, l))];
        const uint32_t wave_id = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)rec);
        const uint32_t block0 = narrow + (uint32_t)__builtin_amdgcn_readlane((int)bl.y, l) +
                                (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(rec >> 32));
        const int sub = (int)(u % G) * SPW, in_wave = sub + grp / G;
        const int64_t i0 = (int64_t)wave_id * PS_WAVE;
        PsSpan sp;   // the group's span
        sp.tri = -1;
        if (i0 + in_wave < R) sp = spans[i0 + in_wave];
        const bool has = sp.tri >= 0;
        if (!__any(has)) continue;
        int nv = 0;
        bool need_ck = false;
        uint32_t word = 0;          // what the lane stores of each piece, where it does not change
        float v = 0.0f, step = 0.0f;
        if (has) {
            const int y = sp.y & 0xffffff;
            need_ck = (sp.x2 >> cw_shift) > (sp.x1 >> cw_shift) && ((sp.y >> 28) & 1) && ps_span_has_ck(sp);
            const uint32_t flags = ((uint32_t)(sp.y >> 24) & 3u) << 26 | ((uint32_t)(sp.y >> 28) & 1u) << 28;
            if (j == 0) word = (uint32_t)(i0 + in_wave) | flags;
            if (j == 2) { v = sp.cf2; step = sp.cf2_step; }
            if (j == 3) { v = sp.pz; step = sp.pz_step; }
            if (j == 4) word = __float_as_uint(sp.cf2_step);
            if (j == 5) word = __float_as_uint(sp.pz_step);
            if (j == 6) word = (uint32_t)y;
            if (need_ck) {
                const PsTri tr = tris[sp.tri];
                const PsDraw& d = draws[tr.code >> 8];
                nv = d.nv;
                PsEdge L, Rr;
                ps_row_edges(tr, y, L, Rr);
                int left = ps_cvt_i32(ps_edge_eval(L, (float)y) + 0.5f);
                int right = ps_cvt_i32(ps_edge_eval(Rr, (float)y) + 0.5f);
                PsSpanGeom g;
                ps_span_geom(tr, y, left, right, L, Rr, g);
                if (j >= 8 && j - 8 < nv) {
                    const float* u0 = vary + (int64_t)tr.vary * 3 * nvs + (j - 8);
                    ps_span_varyings_n<1>(g, u0, u0 + nvs, u0 + 2 * nvs, &v, &step, 1);
                }
            }
        }
        // the listed wave's spans, one per lane: first tile of the tile row
        // (0xffffffff: no span) and chunks, cx0 | cx1 + 1 << 16
        uint32_t row = 0xffffffffu, chunks = 0;
        {
            int ln = lane;
            asm volatile("" : "+v"(ln));   // or its address is kept in registers all along
            PsSpan one;
            one.tri = -1;
            if (i0 + ln < R) one = spans[i0 + ln];
            int64_t vtb = tb1;
            int vntx = ntx1;
            if (f.n_views != 1) {
                // triangles come view by view: one view if the first and the
                // last have the same
                const uint64_t m = __ballot(one.tri >= 0);
                const int va = tris[__builtin_amdgcn_readlane(one.tri, __builtin_ctzll(m))].view;
                const int vb = tris[__builtin_amdgcn_readlane(one.tri, 63 - __builtin_clzll(m))].view;
                const PsView& V = f.views[va == vb || one.tri < 0 ? va : tris[one.tri].view];
                vtb = V.tile_base;
                vntx = V.n_tiles_x;
            }
            if (one.tri >= 0) {
                const PsSpanTiles st = ps_span_tiles(vtb, vntx, f.tile_rows, TC, CW, one.y & 0xffffff, one.x1, one.x2);
                row = st.g0 - (uint32_t)st.tx0;
                chunks = (uint32_t)st.cx0 | (uint32_t)(st.cx1 + 1) << 16;
            }
        }
        const uint32_t np = (chunks >> 16) - (chunks & 0xffffu);
        // of the group's span: its tile row, and the first piece there
        uint32_t seg0 = 0, row0 = 0;
#pragma unroll
        for (int k = 0; k < SPW; k++) {
            const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)row, sub + k);
            const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)ps_wave_incl_scan(row < r ? np : 0u), 63);
            if (grp == k * G) {
                seg0 = block0 + before;
                row0 = r;
            }
        }
        PsSpanTiles st = {};
        int nt = 0;
        if (has) {
            st = ps_span_tiles(row0, 0, f.tile_rows, TC, CW, 0, sp.x1, sp.x2);
            nt = (int)(st.g1 - st.g0) + 1;
        }
        const bool acc = j == 2 || j == 3 || j >= 8;
        // the lane's words of consecutive pieces lie `next` words apart; a
        // whole chunk further, the pixel range and the checkpointed piece's
        // own index move by `move`
        const int next = j < 8 ? (int)(sizeof(PsSeg) / 4) : f.ck_stride;
        const uint32_t move = j == 1 ? (uint32_t)CW * 0x10001u : (j == 7 && need_ck) ? 1u : 0u;
        const int maxnt = (int)ps_wave_max((uint32_t)nt);
        for (int q0 = 0; q0 < maxnt; q0 += G) {
            // Lane j: in the span's tile q0 + j, the pieces that the listed
            // wave's spans have there, those of the spans before this one, and
            // the first of them all.  A span's pieces per tile, from one column
            // to the next, change at its first and last tile only, so the spans
            // (one per lane) add four changes each for every group's tile row,
            // all spans' in the lower half of a word and the earlier ones' in
            // the upper (at most 4,096 pieces each), and sums along the columns
            // give the rest.  (Span by span it was 130 cycles for each of up to
            // 63 others.)
            for (int i = lane; i < SPW * (G + 1); i += PS_WAVE) lds[i] = 0;
            ps_lds_turn();
            uint32_t first = seg0;
#pragma unroll 1
            for (int k = 0; k < SPW; k++) {
                const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)row, sub + k);
                const int w0 = __builtin_amdgcn_readlane(st.tx0, k * G) + q0;
                const bool in_row = row == r && np != 0;
                const int lo = (int)(chunks & 0xffffu), hi = (int)(chunks >> 16), t0 = lo >> tc_shift, t1 = (hi - 1) >> tc_shift;
                // those before the first of these tiles
                const uint32_t left = (uint32_t)__builtin_amdgcn_readlane(
                    (int)ps_wave_incl_scan(in_row ? (uint32_t)(min(max(w0 * TC, lo), hi) - lo) : 0u), 63);
                if (grp == k * G) first += left;
                if (!in_row) continue;
                const int nl = (t0 + 1) * TC - lo, nr = hi - t1 * TC;
                const uint32_t both = lane < sub + k ? 0x10001u : 1u;
                const int at[4] = {t0, t0 + 1, t1, t1 + 1}, change[4] = {nl, TC - nl, nr - TC, -nr};
                uint32_t* row_k = lds + k * (G + 1);
#pragma unroll
                for (int i = 0; i < 4; i++)   // [G]: beyond these tiles
                    atomicAdd(row_k + min(max(at[i] - w0, 0), G), (uint32_t)change[i] * both);
            }
            ps_lds_turn();
            const uint32_t sums = ps_group_incl_scan<G>(lds[grp / G * (G + 1) + j]), here = sums & 0xffffu, earlier = sums >> 16;
            first += ps_group_incl_scan<G>(here) - here;
            ps_lds_turn();
            // the first span in a tile takes the run; its record is written after
            // the pieces, which need not wait for the counter
            const bool takes = q0 + j < nt && earlier == 0;
            uint32_t left = 0;
            if (takes) left = (uint32_t)(atomicAdd(&tcnt[st.g0 + (uint32_t)(q0 + j)], 0ull - PS_TC_RUN) >> 32);
            first += earlier;
            for (int q = q0; q < min(q0 + G, maxnt); q++) {
                const uint32_t s = (uint32_t)__shfl((int)first, grp + (q - q0), PS_WAVE);
                if (q >= nt) continue;
                int lo, hi;
                ps_span_tile_chunks(st, TC, st.g0 + (uint32_t)q, lo, hi);
                uint32_t* at = j < 8 ? (uint32_t*)(segs + s) + j : (uint32_t*)ck + (int64_t)s * f.ck_stride + (j - 8);
                const bool begins = lo == st.cx0;
                bool on = j < 8 || (j - 8 < nv && !begins);   // the span's first piece keeps no checkpoint
                if (j == 1) word = (uint32_t)max(sp.x1, lo * CW) | (uint32_t)min(sp.x2, lo * CW + CW - 1) << 16;
                if (j == 7) word = need_ck && !begins ? (s | PS_SEG_CK) : (uint32_t)sp.tri;
                int n = hi - lo + 1;
                if (begins) {   // on to the next chunk's first pixel
                    if (on) *at = acc ? __float_as_uint(v) : word;
                    const int x = (st.cx0 + 1) * CW;
                    for (int k = sp.x1; k < x; k++) v += step;
                    at += next;
                    on = j < 8 || j - 8 < nv;
                    if (j == 1) word = (uint32_t)x | (uint32_t)(x + CW - 1) << 16;
                    if (j == 7 && need_ck) word = (s + 1u) | PS_SEG_CK;
                    n--;
                }
                const bool ends = n > 0 && hi == st.cx1;
                if (ends) n--;
                if (on) {   // the other lanes carry nothing
                    auto whole = [&](int adds) {
                        *at = acc ? __float_as_uint(v) : word;
                        at += next;
                        word += move;
#pragma unroll
                        for (int k = 0; k < adds; k++) v += step;
                    };
                    auto tile = [&](int adds) {
                        for (; n >= 4; n -= 4) { whole(adds); whole(adds); whole(adds); whole(adds); }
                        for (; n > 0; n--) whole(adds);
                    };
                    if (CW == 2) tile(2);
                    else if (CW == 4) tile(4);
                    else if (CW == 8) tile(8);
                    else
                        for (; n > 0; n--) {
                            whole(1);
                            for (int k = 1; k < CW; k++) v += step;
                        }
                }
                if (ends) {
                    if (j == 1) word = (word & 0xffffu) | (uint32_t)sp.x2 << 16;
                    if (on) *at = acc ? __float_as_uint(v) : word;
                }
            }
            if (takes && !ps_put_run(f, left, PS_TS(f.tstart[st.g0 + (uint32_t)(q0 + j) + 1]), first, here, wave_id, cap))
                ps_overflow(cnt, 2, flag);
        }
    }
}

// G: lanes of a wide span, 8 and one per varying float.  Spans per lane carry
// two accumulators: with the varyings beside them the kernel took 96 VGPRs
// (five waves per SIMD) for 14 floats and 149 for 20.
template <int G>
__global__ void __launch_bounds__(256, 6) k_segments(const PsSpan* __restrict__ spans, const uint32_t* __restrict__ row_off,
                                                  int64_t T, PsFrame f, const PsTri* __restrict__ tris,
                                                  const PsDraw* __restrict__ draws, const float* __restrict__ vary, int nvs,
                                                  unsigned long long* __restrict__ tcnt, PsSeg* __restrict__ segs,
                                                  float* __restrict__ ck, int64_t cap, const unsigned long long* __restrict__ wide, int64_t wide_per,
                                                  PsCounters* cnt, int* flag)
{
    __shared__ uint32_t rel_all[4][SG_BATCH][PS_WAVE];   // per wave: [iteration][lane] offset in the run
    const bool poisoned = ps_poisoned(cnt);
    const int64_t R = row_off[T];
    const uint32_t narrow = (uint32_t)f.tstart[f.n_tiles];   // pieces of the waves that are not listed
    const uint32_t listed = (uint32_t)wide[PS_WIDE_BEFORE + PS_WIDE_LISTS];
    int64_t tb1 = 0;   // the only view of a one-view flush, read once
    int ntx1 = 0;
    if (f.n_views == 1) { tb1 = f.views[0].tile_base; ntx1 = f.views[0].n_tiles_x; }
    if (poisoned) return;   // also if there are more pieces than cap
    if (listed)
        ps_wide_spans<G>(spans, R, f, tris, draws, vary, nvs, wide, wide_per, listed, narrow, tb1, ntx1, tcnt, segs, ck, cap,
                         &rel_all[threadIdx.x >> 6][0][0], cnt, flag);
    const int CW = f.chunk_w, TC = f.tile_cols;
    const int lane = threadIdx.x & (PS_WAVE - 1);
    uint32_t (*rel)[PS_WAVE] = rel_all[threadIdx.x >> 6];
    for (int64_t base = blockIdx.x * (int64_t)blockDim.x; base < R; base += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = base + threadIdx.x;
        const uint32_t wave_id = (uint32_t)((base + (threadIdx.x & ~(PS_WAVE - 1))) >> 6);
        PsSpan sp;
        sp.tri = -1;
        if (i < R) sp = spans[i];
        const bool has = sp.tri >= 0;
        if (ps_wave_wide(has, (uint32_t)(sp.x2 - sp.x1 + 1))) continue;   // placed above
        PsSpanTiles st = {};
        int y = 0;
        uint32_t flags = 0;
        if (has) {
            // the triangle only for a flush of several views (its view)
            int64_t vtb = tb1;
            int vntx = ntx1;
            if (f.n_views != 1) {
                const PsView& v = f.views[tris[sp.tri].view];
                vtb = v.tile_base;
                vntx = v.n_tiles_x;
            }
            y = sp.y & 0xffffff;
            flags = ((uint32_t)(sp.y >> 24) & 3u) << 26 | ((uint32_t)(sp.y >> 28) & 1u) << 28;
            st = ps_span_tiles(vtb, vntx, f.tile_rows, TC, CW, y, sp.x1, sp.x2);
        }
        float cf2 = sp.cf2, pz = sp.pz;
        int x = sp.x1;
        int cx = st.cx0;                     // the lane's next chunk
        uint32_t cur = has ? st.g0 : 0xffffffffu;
        for (;;) {
            // the batch's tiles: lane j takes the j-th (bk) and its pieces (bn);
            // each lane notes its offset in the runs of its tiles, and which
            // iterations those are (consecutive: jt0 .. jt0 + ntb - 1)
            uint32_t bk = 0xffffffffu, bn = 0;
            int nb = 0, jt0 = -1, ntb = 0;
            for (; nb < SG_BATCH; nb++) {
                const uint32_t k = ps_wave_min(cur);
                if (k == 0xffffffffu) break;
                const bool m = cur == k;
                int lo = 0, hi = -1;
                if (m) ps_span_tile_chunks(st, TC, k, lo, hi);
                const uint32_t n = (uint32_t)(hi - lo + 1);
                const uint32_t incl = ps_wave_incl_scan(n);
                const uint32_t tot = __builtin_amdgcn_readlane(incl, 63);
                if (lane == nb) { bk = k; bn = tot; }
                if (m) {
                    rel[nb][lane] = incl - n;
                    if (jt0 < 0) jt0 = nb;
                    ntb++;
                    cur = k < st.g1 ? k + 1 : 0xffffffffu;
                }
            }
            if (nb == 0) break;
            uint32_t first = 0xffffffffu;
            if (lane < nb) first = ps_take_run(f, tcnt, bk, bn, wave_id, cap, cnt, flag);
            // every lane walks its pieces of the batch's tiles
            const int maxtb = __builtin_amdgcn_readfirstlane(ps_wave_max((uint32_t)ntb));
            for (int q = 0; q < maxtb; q++) {
                const int jj = jt0 + q;
                const uint32_t run0 = __shfl(first, jj < 0 ? 0 : jj, PS_WAVE);
                if (q < ntb && run0 != 0xffffffffu) {
                    uint32_t s = run0 + rel[jj][lane];
                    const int hi = min(st.cx1, cx | (TC - 1));   // the tile's last chunk of the span (cx >= 0, TC a power of two)
                    for (; cx <= hi; cx++, s++) {
                        const int xa = max(sp.x1, cx * CW), xb = min(sp.x2, cx * CW + CW - 1);
                        for (; x < xa; x++) {
                            cf2 += sp.cf2_step;
                            pz += sp.pz_step;
                        }
                        PsSeg sg;
                        sg.si = (uint32_t)i | flags;
                        sg.xab = (uint32_t)xa | ((uint32_t)xb << 16);
                        sg.cf2 = cf2;
                        sg.pz = pz;
                        sg.cst = sp.cf2_step;
                        sg.pst = sp.pz_step;
                        sg.y = y;
                        sg.win = (uint32_t)sp.tri;
                        segs[s] = sg;
                    }
                }
            }
            if (nb < SG_BATCH) break;
        }
    }
}

// ---------------------------------------------------------------------------
// tile lists: the runs of a tile in submission order
// ---------------------------------------------------------------------------
// For each lane's keys key[0 .. Q): how many of the n keys they are compared
// with lie below.  Those are held one per lane in `other` (lanes from n on are
// not looked at); each is read from its lane by a constant index, so a key
// costs a read lane and Q compares and adds, without a cross-lane round trip
// (a bitonic network makes two in each of up to 21 dependent steps).
template <int Q>
__device__ __forceinline__ void ps_count_below(const uint32_t* key, uint32_t other, uint32_t n, uint32_t* rank)
{
#pragma unroll
    for (int g = 0; g < 64; g += 8) {
        if ((uint32_t)g >= n) break;
#pragma unroll
        for (int i = g; i < g + 8; i++) {
            const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)other, i);   // 0xffffffff past the last: below none
#pragma unroll
            for (int q = 0; q < Q; q++) rank[q] += o < key[q] ? 1u : 0u;
        }
    }
}

// sorts one (key, value) pair per lane by key over lanes [0, n); the keys are
// distinct, those of the lanes from n on are 0xffffffff
__device__ __forceinline__ void ps_sort_lanes(uint32_t& key, uint32_t& val, uint32_t n)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t rank = 0;
    ps_count_below<1>(&key, key, n, &rank);
    const int to = (int)(lane < n ? rank : lane) * 4;
    key = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)key);
    val = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)val);
}

// The runs of a tile are written in the order their atomics happened.  Ordered
// by wave they give the tile's pieces in submission order: wave order is span
// order, and inside a run the pieces are in span order.
//
// Window of up to 64 runs from run w0 on, one per lane: rbase = the run's
// first piece, rv = the list position of that piece (0xffffffff past the last
// run), vhi = the list position where the window ends.  A tile of at most 64
// runs is sorted here; longer lists of n_list pieces come ordered by
// ps_order_runs, with each run's key replaced by its list position.
__device__ __forceinline__ void ps_run_window(const uint32_t* rl, uint32_t nr, uint32_t w0, uint32_t n_list,
                                              uint32_t& rbase, uint32_t& rv, uint32_t& vhi)
{
    const uint32_t j = w0 + (threadIdx.x & 63);
    const uint32_t nw = min(nr - w0, 64u);
    if (nr <= 64) {
        uint32_t key = j < nr ? rl[2 * j + 1] : 0xffffffffu;
        rbase = j < nr ? rl[2 * j] : 0u;
        ps_sort_lanes(key, rbase, nw);
        const uint32_t c = j < nr ? (key & 0xfffu) + 1u : 0u;
        const uint32_t incl = ps_wave_incl_scan(c);
        rv = j < nr ? incl - c : 0xffffffffu;
        vhi = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    } else {
        rbase = j < nr ? rl[2 * j] : 0u;
        rv = j < nr ? rl[2 * j + 1] : 0xffffffffu;
        vhi = w0 + nw < nr ? rl[2 * (w0 + nw) + 1] : n_list;
    }
}

// A tile with more than PS_LDS_RUNS runs: one wave sorts them by wave (LSD
// radix, 7-bit digits of the wave index above the smallest, ping-ponging
// between the tile's parts a and b of the two run arrays), then replaces each
// run's key by the list position of its first piece.  cnt128: 128 words of
// the wave's LDS.  Returns the array that holds the result; n_list: the pieces.
__device__ uint32_t* ps_order_runs(uint32_t* a, uint32_t* b, uint32_t nr, uint32_t* cnt128, uint32_t& n_list)
{
    const int lane = threadIdx.x & 63;
    const uint64_t lt = ps_lt_mask();
    uint32_t mn = 0xffffffffu, mx = 0;
    for (uint32_t j = lane; j < nr; j += 64) {
        const uint32_t w = a[2 * j + 1] >> 12;
        mn = min(mn, w);
        mx = max(mx, w);
    }
    mn = ps_wave_min(mn);
    mx = ps_wave_max(mx);
    const int bits = mx > mn ? 32 - __clz(mx - mn) : 0;
    for (int shift = 0; shift < bits; shift += 7) {
        cnt128[lane] = 0;
        cnt128[lane + 64] = 0;
        __builtin_amdgcn_wave_barrier();
        for (uint32_t j = lane; j < nr; j += 64)
            atomicAdd(&cnt128[(((a[2 * j + 1] >> 12) - mn) >> shift) & 127u], 1u);
        __builtin_amdgcn_wave_barrier();
        {
            const uint32_t c0 = cnt128[2 * lane], c1 = cnt128[2 * lane + 1];
            const uint32_t ex = ps_wave_incl_scan(c0 + c1) - c0 - c1;
            __builtin_amdgcn_wave_barrier();
            cnt128[2 * lane] = ex;
            cnt128[2 * lane + 1] = ex + c0;
            __builtin_amdgcn_wave_barrier();
        }
        for (uint32_t j0 = 0; j0 < nr; j0 += 64) {
            const uint32_t j = j0 + lane;
            const bool valid = j < nr;
            const uint32_t e0 = valid ? a[2 * j] : 0u, e1 = valid ? a[2 * j + 1] : 0u;
            const uint32_t dig = valid ? (((e1 >> 12) - mn) >> shift) & 127u : 0u;
            uint64_t same = __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < 7; bit++) {
                const uint64_t m = __ballot((dig >> bit) & 1u);
                same &= ((dig >> bit) & 1u) ? m : ~m;
            }
            const uint32_t before = (uint32_t)__popcll(same & lt);
            const uint32_t cur = cnt128[dig];
            __builtin_amdgcn_wave_barrier();
            if (valid) {
                b[2 * (cur + before)] = e0;
                b[2 * (cur + before) + 1] = e1;
                if (before == 0) cnt128[dig] = cur + (uint32_t)__popcll(same);
            }
            __builtin_amdgcn_wave_barrier();
        }
        __threadfence();   // the next pass reads what this one wrote
        uint32_t* t = a; a = b; b = t;
    }
    uint32_t carry = 0;
    for (uint32_t j0 = 0; j0 < nr; j0 += 64) {
        const uint32_t j = j0 + lane;
        const uint32_t c = j < nr ? (a[2 * j + 1] & 0xfffu) + 1u : 0u;
        const uint32_t incl = ps_wave_incl_scan(c);
        if (j < nr) a[2 * j + 1] = carry + incl - c;
        carry += __builtin_amdgcn_readlane(incl, 63);
    }
    __threadfence();
    n_list = carry;
    return a;
}

// ---------------------------------------------------------------------------
// raster: ordered depth test per bin
// ---------------------------------------------------------------------------
// LDS of one wave of the raster kernels: the runs of a tile of 65 to
// PS_LDS_RUNS runs in order (first piece, list position), which run starts at
// each position of a batch, a spare pixel per lane, then depth and winner (or
// colour) of the tile's pixels, pixel k of lane l's chunk at [k * 64 + l]
#define PS_LDS_RUNS 256
#define RA_PIX_WORDS(cw) (PS_LDS_RUNS * 2 + 64 + 64 * 2 + (cw) * 64 * 2)

// The runs of a tile of 65 to PS_LDS_RUNS runs, sorted by wave and with each
// key replaced by the list position of the run's first piece, into the wave's
// LDS: every key is counted against all of them (1 us for 128 runs), where
// sorting them in global memory takes several dependent passes over it
// (11 to 38 us, the longest part of the tiles that end the kernel).
__device__ __forceinline__ void ps_sort_runs_lds(const uint32_t* rl, uint32_t nr, uint2* out, uint32_t& n_list)
{
    constexpr int Q = PS_LDS_RUNS / 64;
    const uint32_t lane = threadIdx.x & 63;
    uint32_t key[Q], val[Q], rank[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const uint32_t j = q * 64 + lane;
        const uint2 r = j < nr ? *(const uint2*)(rl + 2 * j) : make_uint2(0u, 0xffffffffu);
        val[q] = r.x;
        key[q] = r.y;
        rank[q] = 0;
    }
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (nr > 64u * q) ps_count_below<Q>(key, key[q], min(nr - 64u * q, 64u), rank);
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (q * 64 + lane < nr) out[rank[q]] = make_uint2(val[q], (key[q] & 0xfffu) + 1u);
    ps_lds_turn();
    uint32_t carry = 0;
    for (uint32_t j0 = 0; j0 < nr; j0 += 64) {
        const uint32_t j = j0 + lane;
        const uint2 r = j < nr ? out[j] : make_uint2(0u, 0u);
        const uint32_t incl = ps_wave_incl_scan(r.y);
        if (j < nr) out[j].y = carry + incl - r.y;
        carry += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    }
    n_list = carry;
    ps_lds_turn();
}

// inclusive maximum over the lanes
__device__ __forceinline__ uint32_t ps_wave_incl_max(uint32_t v)
{
    v = max(v, (uint32_t)PS_DPP(v, 0x111, 0xf, true));
    v = max(v, (uint32_t)PS_DPP(v, 0x112, 0xf, true));
    v = max(v, (uint32_t)PS_DPP(v, 0x114, 0xf, true));
    v = max(v, (uint32_t)PS_DPP(v, 0x118, 0xf, true));
    v = max(v, (uint32_t)PS_DPP(v, 0x142, 0xa, false));
    v = max(v, (uint32_t)PS_DPP(v, 0x143, 0xc, false));
    return v;
}

// A lane's run of n (at most N) words at p, in the widest accesses that its
// length and alignment allow: whole runs of rows 16 bytes aligned (8 for two
// words) go in one instruction.
template <int N>
__device__ __forceinline__ void ps_load_run(const uint32_t* p, int n, uint32_t* v)
{
    constexpr int A = N >= 4 ? 16 : 4 * N;
    if (n == N && ((uintptr_t)p & (A - 1)) == 0) {
        if constexpr (N >= 4) {
#pragma unroll
            for (int k = 0; k < N; k += 4) {
                const uint4 q = *(const uint4*)(p + k);
                v[k] = q.x; v[k + 1] = q.y; v[k + 2] = q.z; v[k + 3] = q.w;
            }
        } else if constexpr (N == 2) {
            const uint2 q = *(const uint2*)p;
            v[0] = q.x; v[1] = q.y;
        } else {
            v[0] = p[0];
        }
    } else {
#pragma unroll
        for (int k = 0; k < N; k++) v[k] = k < n ? p[k] : 0u;
    }
}

template <int N>
__device__ __forceinline__ void ps_store_run(uint32_t* p, int n, const uint32_t* v)
{
    constexpr int A = N >= 4 ? 16 : 4 * N;
    if (n == N && ((uintptr_t)p & (A - 1)) == 0) {
        if constexpr (N >= 4) {
#pragma unroll
            for (int k = 0; k < N; k += 4) *(uint4*)(p + k) = make_uint4(v[k], v[k + 1], v[k + 2], v[k + 3]);
        } else if constexpr (N == 2) {
            *(uint2*)p = make_uint2(v[0], v[1]);
        } else {
            p[0] = v[0];
        }
    } else {
#pragma unroll
        for (int k = 0; k < N; k++)
            if (k < n) p[k] = v[k];
    }
}

// One wave per tile; the wave takes the tile's pieces 64 at a time, one per
// lane, in submission order.  Each lane evaluates its own piece's depths, so
// the divisions run on full waves whatever chunk the pieces fall in, and the
// order-dependent test is resolved per pixel in rounds: among the lanes whose
// piece covers pixel k of the same chunk, the one with r such lanes before it
// goes in round r, against the depth the rounds before it left in LDS.  A
// batch takes one round unless its pieces overlap.  While every piece of the
// batch tests depth, a pixel's depth only falls, so a fragment that fails
// against the depth at the batch's start fails in its turn too and takes no
// round.
// The walk this replaced (each lane its chunk's pieces, one after the other,
// from lists split in LDS) ran as long as the fullest of the 64 chunks.  What
// bounds it is a wave's chain of LDS and cross-lane latencies, some 3,000
// cycles a batch; its own work per pixel is small.  Before and after, default
// tiles: 3840x2160 terrain (2.8M pieces) 113 -> 45 us, 32 views of 256^2 to
// 1024^2 (3.7M) 158 -> 77, 515x389 (86k, as long as its longest tile) 37 ->
// 21; 1920x1080 in 16x8 tiles (1.1M) 33 -> 22.
// KCW: the chunk width when it is 1, 2, 4 or 8 (a batch's pixels are then
// unrolled and share their rounds), else 0: of a chunk of 16 pixels or more a
// piece covers so few that rounds over all of them mostly pass lanes by, and
// each lane walks the batch's pieces of its own chunk instead.  1920x1080
// terrain in 16x8 tiles 209 -> 184 us, 64x4 726 -> 339; a lane's pieces from
// lists split in LDS took 201 and 417.
template <bool DEBUG, int KCW>
__global__ void __launch_bounds__(512, 5) k_raster(const PsSpan* __restrict__ spans, const PsSeg* __restrict__ segs,
                         const PsTri* __restrict__ tris, const PsDraw* __restrict__ draws, PsFrame f, int64_t n_tiles,
                         PsCounters* cnt)
{
    extern __shared__ uint32_t lds[];
    const bool poisoned = ps_poisoned(cnt);
    const int CW = KCW ? KCW : f.chunk_w;
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int waves = blockDim.x >> 6;
    // neighbouring tiles share an L2; with a heavy-tile list, the first
    // waves take the listed tiles (they start first, so the
    // longest walks do not end the kernel), the others every unlisted tile
    // (the list and the marks are in bounds, stale or not)
    int64_t tile = ps_xcd_remap<4>(blockIdx.x, gridDim.x) * (int64_t)waves + wave;
    bool skip = false;
    if (f.heavy) {
        const int64_t hcap = ps_heavy_cap(n_tiles);
        if (tile < hcap) {
            const uint32_t listed = min(f.heavy[0], (uint32_t)hcap);
            const uint32_t t = f.heavy[1 + tile];
            skip = tile >= listed;
            tile = t;
        } else {
            tile -= hcap;
            skip = tile >= n_tiles || (f.tstart[min(tile, n_tiles)] >> 63);
        }
    }
    if (poisoned) return;
    ps_commit_pending(cnt);
    if (skip || tile >= n_tiles) return;
    uint2* lruns = (uint2*)(lds + (size_t)wave * RA_PIX_WORDS(CW));
    uint32_t* starts = (uint32_t*)(lruns + PS_LDS_RUNS);
    uint2* spare = (uint2*)(starts + 64) + lane;
    uint2* pix = (uint2*)(starts + 64) + 64;   // x: depth bits, y: winner code

    const int cw_shift = __builtin_ctz((unsigned)CW), tc_shift = __builtin_ctz((unsigned)f.tile_cols);
    const PsView& V = f.views[ps_view_of_tile(f, tile)];
    int64_t ltile = tile - V.tile_base;
    // a view has fewer than 2^31 tiles; tile_cols is a power of two
    const uint32_t lt32 = (uint32_t)ltile, ntx = (uint32_t)V.n_tiles_x;
    int ty = (int)(lt32 / ntx), tx = (int)(lt32 - (uint32_t)ty * ntx);
    int y = ty * f.tile_rows + (lane >> tc_shift);
    int X0 = (tx * f.tile_cols + (lane & (f.tile_cols - 1))) * CW;
    const int VW = V.W;
    const int ncol = y < V.H && X0 < VW ? min(CW, VW - X0) : 0;
    float* drow = V.depth + (int64_t)y * V.depth_scan;
    // a clear fused into the flush: the tile starts from its value, and the
    // whole tile is written back
    const bool dclear = V.dclear != 0;
    // the tile's runs in submission order, up to 64 at a time (one per lane)
    const unsigned long long ta = PS_TS(f.tstart[tile]), tb = PS_TS(f.tstart[tile + 1]);
    const uint32_t r0 = (uint32_t)(ta >> 32), nr = (uint32_t)(tb >> 32) - r0;
    const uint32_t* rl = f.runs + 2 * (size_t)r0;
    const bool in_lds = nr > 64 && nr <= PS_LDS_RUNS;
    uint32_t n_list = 0;   // the tile's pieces, where the runs are sorted here
    if (in_lds) ps_sort_runs_lds(rl, nr, lruns, n_list);
    else if (nr > 64) rl = ps_order_runs(f.runs + 2 * (size_t)r0, f.runs2 + 2 * (size_t)r0, nr, (uint32_t*)lruns, n_list);
    if constexpr (KCW > 0) {
        uint32_t d[KCW];
        if (dclear) {
#pragma unroll
            for (int k = 0; k < KCW; k++) d[k] = __float_as_uint(V.dclear_value);
        } else {
            ps_load_run<KCW>((const uint32_t*)drow + X0, ncol, d);
        }
#pragma unroll
        for (int k = 0; k < KCW; k++) pix[k * 64 + lane] = make_uint2(d[k], 0xffffffffu);
    } else {
        for (int k = 0; k < ncol; k++)
            pix[k * 64 + lane] = make_uint2(__float_as_uint(dclear ? V.dclear_value : drow[X0 + k]), 0xffffffffu);
    }
    uint32_t passes = 0;   // the lane's; a list has at most 2^31 pieces of 64 pixels
    bool dirty = dclear;
    ps_lds_turn();
    for (uint32_t w0 = 0; w0 < nr; w0 += 64) {
        // the window's runs, one per lane: list position of the first piece
        // (0xffffffff past the last run), and what to add to a list position
        // in the run to get its piece
        uint32_t rbase, rv, vhi;
        if (in_lds) {
            const uint32_t j = w0 + lane;
            const uint2 r = j < nr ? lruns[j] : make_uint2(0u, 0xffffffffu);
            rbase = r.x;
            rv = r.y;
            vhi = w0 + 64 < nr ? lruns[w0 + 64].y : n_list;
        } else {
            ps_run_window(rl, nr, w0, n_list, rbase, rv, vhi);
        }
        const uint32_t vlo = (uint32_t)__builtin_amdgcn_readlane((int)rv, 0), delta = rbase - rv;
        // the records of the next batch are in flight while one is tested.  A
        // batch's pieces: each run that starts in it marks its first position,
        // a running maximum over the positions gives every lane its run.
        uint4 ran, rbn;
        uint32_t run = 0;   // one more than the run of the last position before the batch
        auto gather = [&](uint32_t c) {
            starts[lane] = 0;
            ps_lds_turn();
            if (rv - c < 64u) starts[rv - c] = (uint32_t)lane + 1u;
            ps_lds_turn();
            const uint32_t m = max(ps_wave_incl_max(starts[lane]), run);
            ps_lds_turn();
            run = (uint32_t)__builtin_amdgcn_readlane((int)m, 63);
            const uint32_t e = c + lane;
            const uint32_t pp = e + (uint32_t)__builtin_amdgcn_ds_bpermute((int)(m - 1u) * 4, (int)delta);
            const uint4* p = (const uint4*)(segs + (e < vhi ? pp : 0u));
            ran = p[0];
            rbn = p[1];
        };
        gather(vlo);
        for (uint32_t cb = vlo; cb < vhi; cb += 64) {
            const uint4 ra = ran, rb = rbn;
            const bool valid = cb + lane < vhi;
            if (cb + 64 < vhi) gather(cb + 64);
            // the piece's chunk in the tile and its pixels [a, b] of it
            const int xa = (int)(ra.y & 0xffffu), pcx = xa >> cw_shift;
            const int key = (((int)rb.z & (f.tile_rows - 1)) << tc_shift) | (pcx & (f.tile_cols - 1));
            const int a = xa - (pcx << cw_shift), b = valid ? (int)(ra.y >> 16) - (pcx << cw_shift) : -1;
            const bool test = (ra.x >> 26) & PSGPU_TEST_DEPTH, upd = (ra.x >> 26) & PSGPU_UPDATE_DEPTH, wc = (ra.x >> 28) & 1;
            const uint32_t wcode = rb.w;
            float cf2 = __uint_as_float(ra.z), pz = __uint_as_float(ra.w);
            const float cst = __uint_as_float(rb.x), pst = __uint_as_float(rb.y);
            uint32_t th = 0;
            int tid = 0;
            if (DEBUG && valid) {
                int tri = (wcode & PS_SEG_CK) ? spans[segs[wcode & ~PS_SEG_CK].si & PS_SEG_SPAN_MASK].tri : (int)wcode;
                const PsDraw& d = draws[tris[tri].code >> 8];
                tid = (int)(d.id_base + (tri - d.tri_start));
                uint32_t h = (uint32_t)tid;
                h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
                th = h;
            }
            // lanes of the same chunk; with wide chunks, those of the chunk
            // that is the lane's
            const int of = KCW ? key : lane;
            uint64_t same = KCW ? ~0ull : __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < 6; bit++) {
                const uint64_t m = __ballot((key >> bit) & 1);
                same &= ((of >> bit) & 1) ? m : ~m;
            }
            const bool all_test = __all(test || !valid);
            // candidates before this lane at the same pixel
            auto rank_of = [&](bool cand) {
                const uint64_t m = same & __ballot(cand);
                return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            };
            // the lane's depth at pixel k, interpolateNextStep (interp.cpp:82-92)
            auto depth_at = [&](bool in) {
                const float r = 1.0f / cf2, z = pz * r;
                cf2 = in ? cf2 + cst : cf2;
                pz = in ? pz + pst : pz;
                return z;
            };
            // fragthrd.cpp:216-237 against the pixel's depth and winner
            auto fragment = [&](bool turn, int k, float z, uint2 cur) {
                const float d = test ? __uint_as_float(cur.x) : 1.0f;
                const bool pass = turn & (z - d < -0.0001f);
                if (upd) cur.x = __float_as_uint(z);
                if (wc) cur.y = wcode;
                // a fragment that fails, or whose turn it is not, goes to the
                // lane's own spare slot: selecting the address costs less
                // than masking the store
                *(pass ? pix + k * 64 + key : spare) = cur;
                passes += pass ? 1u : 0u;
                dirty |= pass & upd;
                if (DEBUG && pass) {
                    const int64_t at = (int64_t)(int)rb.z * VW + ((pcx << cw_shift) + k);
                    atomicAdd(&f.dbg_pcount[at], 1);
                    atomicXor(&f.dbg_phash[at], th);
                    f.dbg_last[at] = tid;
                }
            };
            auto drawn = [&](int k) {   // every rasterised fragment, passing or not
                const int64_t at = (int64_t)(int)rb.z * VW + ((pcx << cw_shift) + k);
                atomicAdd(&f.dbg_rcount[at], 1);
                atomicXor(&f.dbg_rhash[at], th);
            };
            if constexpr (KCW > 0) {
                // every lane evaluates every pixel of the chunk, so that the
                // divisions and the LDS reads overlap
                float z[KCW];
                uint2 cur[KCW];
                bool cand[KCW];
                int rank[KCW], last = 0;
#pragma unroll
                for (int k = 0; k < KCW; k++) cur[k] = pix[k * 64 + key];
#pragma unroll
                for (int k = 0; k < KCW; k++) {
                    const bool in = (k >= a) & (k <= b);
                    z[k] = depth_at(in);
                    if (DEBUG && in) drawn(k);
                    cand[k] = in & (-1.0f < z[k]) & (!all_test | (z[k] - __uint_as_float(cur[k].x) < -0.0001f));
                }
#pragma unroll
                for (int k = 0; k < KCW; k++) {
                    rank[k] = rank_of(cand[k]);
                    last = cand[k] ? max(last, rank[k]) : last;
                }
#pragma unroll
                for (int k = 0; k < KCW; k++) fragment(cand[k] & (rank[k] == 0), k, z[k], cur[k]);
                if (DEBUG) __threadfence();   // the last pass of a pixel is stored last
                ps_lds_turn();
                for (int r = 1; __any(last >= r); r++) {
#pragma unroll
                    for (int k = 0; k < KCW; k++) cur[k] = pix[k * 64 + key];
#pragma unroll
                    for (int k = 0; k < KCW; k++) fragment(cand[k] & (rank[k] == r), k, z[k], cur[k]);
                    if (DEBUG) __threadfence();
                    ps_lds_turn();
                }
            } else {
                // each lane walks the pieces of its own chunk, one after the
                // other, four pixels at a time
                const int ends = a | b << 8 | (int)(ra.x >> 26) << 16;
                int k = 1, last = 0, how = 0, code = 0, hash = 0, id = 0;
                float f2 = 0.0f, zn = 0.0f, f2s = 0.0f, zns = 0.0f;
                auto from = [](int j, int v) { return __builtin_amdgcn_ds_bpermute(j * 4, v); };
                auto fromf = [&](int j, float v) { return __int_as_float(from(j, __float_as_int(v))); };
                while (__any((same != 0) | (k <= last))) {
                    const bool take = (k > last) & (same != 0);
                    if (__any(take)) {
                        const int j = __builtin_ctzll(same | 1ull << 63);
                        const int e = from(j, ends), wj = from(j, (int)wcode);
                        const float g0 = fromf(j, cf2), g1 = fromf(j, pz), g2 = fromf(j, cst), g3 = fromf(j, pst);
                        const int hj = DEBUG ? from(j, (int)th) : 0, ij = DEBUG ? from(j, tid) : 0;
                        if (take) {
                            k = e & 0xff; last = e >> 8 & 0xff; how = e >> 16;
                            code = wj; f2 = g0; zn = g1; f2s = g2; zns = g3; hash = hj; id = ij;
                            same &= same - 1;
                        }
                    }
                    uint2 cur[4];
                    float z[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) cur[j] = pix[min(k + j, CW - 1) * 64 + lane];
#pragma unroll
                    for (int j = 0; j < 4; j++) {   // interpolateNextStep (interp.cpp:82-92)
                        const float r = 1.0f / f2;
                        z[j] = zn * r;
                        f2 += f2s;
                        zn += zns;
                    }
#pragma unroll
                    for (int j = 0; j < 4; j++) {   // fragthrd.cpp:216-237
                        const float dd = how & PSGPU_TEST_DEPTH ? __uint_as_float(cur[j].x) : 1.0f;
                        const bool in = k + j <= last, pass = in & (-1.0f < z[j]) & (z[j] - dd < -0.0001f);
                        if (how & PSGPU_UPDATE_DEPTH) cur[j].x = __float_as_uint(z[j]);
                        if (how & 4) cur[j].y = (uint32_t)code;
                        if (pass) pix[(k + j) * 64 + lane] = cur[j];
                        passes += pass ? 1u : 0u;
                        dirty |= pass & ((how & PSGPU_UPDATE_DEPTH) != 0);
                        if (DEBUG && in) {
                            const int64_t at = (int64_t)y * VW + X0 + k + j;
                            f.dbg_rcount[at] += 1;
                            f.dbg_rhash[at] ^= (uint32_t)hash;
                            if (pass) {
                                f.dbg_pcount[at] += 1;
                                f.dbg_phash[at] ^= (uint32_t)hash;
                                f.dbg_last[at] = id;
                            }
                        }
                    }
                    k += 4;
                }
                ps_lds_turn();
            }
        }
    }
    const bool write_depth = __any(dirty);
    uint32_t* wrow = (uint32_t*)V.winner + ps_winner_at(f, V, 0, y);
    if constexpr (KCW > 0) {
        uint32_t d[KCW], w[KCW];
#pragma unroll
        for (int k = 0; k < KCW; k++) {
            const uint2 p = pix[k * 64 + lane];
            d[k] = p.x;
            w[k] = p.y;
        }
        if (write_depth) ps_store_run<KCW>((uint32_t*)drow + X0, ncol, d);
        ps_store_run<KCW>(wrow + X0, ncol, w);
    } else {
        for (int k = 0; k < ncol; k++) {
            const uint2 p = pix[k * 64 + lane];
            if (write_depth) drow[X0 + k] = __uint_as_float(p.x);
            wrow[X0 + k] = p.y;
        }
    }
    ps_wave_add64(cnt, PS_ST_SHADED, passes);
}

// ---------------------------------------------------------------------------
// raster with the FP in the ordered walk: programmes that blend or discard
// ---------------------------------------------------------------------------
// A discarded fragment leaves the depth unchanged and a blended one depends
// on the colour beneath it, so neither can be deferred to one shading pass
// per pixel.  As in k_raster the wave takes the tile's pieces 64 at a time,
// one per lane; depth and colour of the tile stay in LDS.  What the programme
// gives for a fragment does not depend on the order, only whether it counts
// does: each lane runs the programme for the pixels of its piece, if a fragment
// of the batch can pass, and the order is resolved per pixel in rounds
// afterwards.
// What bounds it is issue on the SIMDs that hold the layer's tiles, some
// 25,000 cycles a batch with two waves each: a fragment takes five texture
// reads and 400 instructions, and the pieces fill 2.3 of their 4 pixels.  Before
// (each lane its chunk's pieces, one after the other, and a piece's pixels one
// after the other) and after, a layer over a 960x540 scene: blended 57 -> 30
// us, discarding 35 -> 17.  Unrolled over the chunk (KCW) the texture reads of
// its pixels overlap: 34 -> 30 and 21 -> 17; other widths go through its
// pixels in turn (KCW 0), but of 64 pixels each lane walks the pieces of its own
// chunk, as in k_raster: 64x64 tiles 643 -> 502 us (32x32 1,134 -> 1,264, 16x16
// 592 -> 688 the frame, since a batch's pieces lie in few chunks and lanes
// without one shade along).
template <int PROG, bool DEBUG, int KCW>
__global__ void __launch_bounds__(512) k_raster_imm(const PsSpan* __restrict__ spans, const PsSeg* __restrict__ segs,
                         const PsTri* __restrict__ tris, const PsDraw* __restrict__ draws, PsFrame f, int64_t n_tiles,
                         PsCounters* cnt, const float* __restrict__ vary, int nvs, const float* __restrict__ ck)
{
    typedef PsProc<PROG> P;
    constexpr int NV = P::NV;
    constexpr bool COLOUR = PROG == PSGPU_PROC_CLOUD;   // the other one only discards
    extern __shared__ uint32_t lds[];
    if (ps_poisoned(cnt)) return;
    ps_commit_pending(cnt);
    constexpr bool UNROLL = KCW > 0 && KCW <= 4, OWN = KCW > 4;
    const int CW = KCW ? KCW : f.chunk_w;
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int waves = blockDim.x >> 6;
    int64_t tile = ps_xcd_remap<4>(blockIdx.x, gridDim.x) * (int64_t)waves + wave;   // neighbouring tiles share an L2
    if (tile >= n_tiles) return;
    uint2* lruns = (uint2*)(lds + (size_t)wave * RA_PIX_WORDS(CW));
    uint32_t* starts = (uint32_t*)(lruns + PS_LDS_RUNS);
    uint2* spare = (uint2*)(starts + 64) + lane;
    uint2* pix = (uint2*)(starts + 64) + 64;   // x: depth bits, y: colour

    const int cw_shift = __builtin_ctz((unsigned)CW), tc_shift = __builtin_ctz((unsigned)f.tile_cols);
    const PsView& V = f.views[ps_view_of_tile(f, tile)];
    int64_t ltile = tile - V.tile_base;
    // a view has fewer than 2^31 tiles; tile_cols is a power of two
    const uint32_t lt32 = (uint32_t)ltile, ntx = (uint32_t)V.n_tiles_x;
    int ty = (int)(lt32 / ntx), tx = (int)(lt32 - (uint32_t)ty * ntx);
    int y = ty * f.tile_rows + (lane >> tc_shift);
    int X0 = (tx * f.tile_cols + (lane & (f.tile_cols - 1))) * CW;
    const int VW = V.W;
    const int ncol = y < V.H && X0 < VW ? min(CW, VW - X0) : 0;
    float* drow = V.depth + (int64_t)y * V.depth_scan;
    uint32_t* crow = V.colour + (V.colour_top_down ? (int64_t)(V.colour_h - 1 - y) : (int64_t)y) * V.colour_scan;
    // a clear fused into the flush: the tile starts from its value, and the
    // whole tile is written back
    const bool dclear = V.dclear != 0;
    // the tile's runs in submission order, up to 64 at a time (one per lane)
    const unsigned long long ta = PS_TS(f.tstart[tile]), tb = PS_TS(f.tstart[tile + 1]);
    const uint32_t r0 = (uint32_t)(ta >> 32), nr = (uint32_t)(tb >> 32) - r0;
    if (nr == 0 && !dclear) return;
    const uint32_t* rl = f.runs + 2 * (size_t)r0;
    const bool in_lds = nr > 64 && nr <= PS_LDS_RUNS;
    uint32_t n_list = 0;   // the tile's pieces, where the runs are sorted here
    if (in_lds) ps_sort_runs_lds(rl, nr, lruns, n_list);
    else if (nr > 64) rl = ps_order_runs(f.runs + 2 * (size_t)r0, f.runs2 + 2 * (size_t)r0, nr, (uint32_t*)lruns, n_list);
    // the chunk as the flush finds it, to write back what it changes
    uint32_t d0[UNROLL ? KCW : 1], c0[UNROLL ? KCW : 1];
    if constexpr (UNROLL) {
        ps_load_run<KCW>((const uint32_t*)drow + X0, ncol, d0);
#pragma unroll
        for (int k = 0; k < KCW; k++) c0[k] = 0;
        if (COLOUR) ps_load_run<KCW>(crow + X0, ncol, c0);
#pragma unroll
        for (int k = 0; k < KCW; k++) pix[k * 64 + lane] = make_uint2(dclear ? __float_as_uint(V.dclear_value) : d0[k], c0[k]);
    } else {
        for (int k = 0; k < ncol; k++)
            pix[k * 64 + lane] = make_uint2(__float_as_uint(dclear ? V.dclear_value : drow[X0 + k]), COLOUR ? crow[X0 + k] : 0u);
    }
    uint32_t passes = 0;   // the lane's; a list has at most 2^31 pieces of 64 pixels
    ps_lds_turn();
    for (uint32_t w0 = 0; w0 < nr; w0 += 64) {
        // the window's runs, one per lane: list position of the first piece
        // (0xffffffff past the last run), and what to add to a list position
        // in the run to get its piece
        uint32_t rbase, rv, vhi;
        if (in_lds) {
            const uint32_t j = w0 + lane;
            const uint2 r = j < nr ? lruns[j] : make_uint2(0u, 0xffffffffu);
            rbase = r.x;
            rv = r.y;
            vhi = w0 + 64 < nr ? lruns[w0 + 64].y : n_list;
        } else {
            ps_run_window(rl, nr, w0, n_list, rbase, rv, vhi);
        }
        const uint32_t vlo = (uint32_t)__builtin_amdgcn_readlane((int)rv, 0), delta = rbase - rv;
        uint32_t run = 0;   // one more than the run of the last position before the batch
        for (uint32_t cb = vlo; cb < vhi; cb += 64) {
            // the batch's pieces, as k_raster gathers them
            starts[lane] = 0;
            ps_lds_turn();
            if (rv - cb < 64u) starts[rv - cb] = (uint32_t)lane + 1u;
            ps_lds_turn();
            const uint32_t m = max(ps_wave_incl_max(starts[lane]), run);
            ps_lds_turn();
            run = (uint32_t)__builtin_amdgcn_readlane((int)m, 63);
            const uint32_t e = cb + lane;
            const bool valid = e < vhi;
            const uint32_t pp = e + (uint32_t)__builtin_amdgcn_ds_bpermute((int)(m - 1u) * 4, (int)delta);
            uint4 ra = make_uint4(0, 0, 0, 0), rb = make_uint4(0, 0, 0, 0);
            float vs[NV > 0 ? NV : 1], vt[NV > 0 ? NV : 1];
#pragma unroll
            for (int i = 0; i < NV; i++) vs[i] = vt[i] = 0.0f;
            int di = 0, tri = 0;
            if (valid) {
                const uint4* p = (const uint4*)(segs + pp);
                ra = p[0];
                rb = p[1];
                // the span's varyings at the piece's first pixel: from its
                // checkpoint or by the serial walk from x1 (interp.cpp:82-92),
                // as the deferred shading does
                const PsSpan sp = spans[ra.x & PS_SEG_SPAN_MASK];
                tri = sp.tri;
                const PsTri tr = tris[tri];
                di = (int)(tr.code >> 8);
                const int py = (int)rb.z, xa = (int)(ra.y & 0xffffu);
                PsEdge Le, Re;
                ps_row_edges(tr, py, Le, Re);
                int left = ps_cvt_i32(ps_edge_eval(Le, (float)py) + 0.5f);
                int right = ps_cvt_i32(ps_edge_eval(Re, (float)py) + 0.5f);
                PsSpanGeom g;
                ps_span_geom(tr, py, left, right, Le, Re, g);
                const float* u0 = vary + (int64_t)tr.vary * 3 * nvs;
                ps_span_varyings<NV>(g, u0, u0 + nvs, u0 + 2 * nvs, vs, vt);
                int xs = sp.x1;
                if (xa > sp.x1 && ps_span_has_ck(sp) && ((ra.x >> 28) & 1)) {
                    const float* cp = ck + (int64_t)pp * f.ck_stride;
#pragma unroll
                    for (int i = 0; i < NV; i++) vs[i] = cp[i];
                    xs = xa;
                }
                for (int xx = xs; xx < xa; xx++) {
#pragma unroll
                    for (int i = 0; i < NV; i++) vs[i] = vs[i] + vt[i];
                }
            }
            // the piece's chunk in the tile and its pixels [a, b] of it
            const int xa = (int)(ra.y & 0xffffu), pcx = xa >> cw_shift;
            const int key = (((int)rb.z & (f.tile_rows - 1)) << tc_shift) | (pcx & (f.tile_cols - 1));
            const int a = xa - (pcx << cw_shift), b = valid ? (int)(ra.y >> 16) - (pcx << cw_shift) : -1;
            const bool test = (ra.x >> 26) & PSGPU_TEST_DEPTH, upd = (ra.x >> 26) & PSGPU_UPDATE_DEPTH, wc = (ra.x >> 28) & 1;
            float cf2 = __uint_as_float(ra.z), pz = __uint_as_float(ra.w);
            const float cst = __uint_as_float(rb.x), pst = __uint_as_float(rb.y);
            const PsDraw& d = draws[di];
            const bool blend = COLOUR && (d.behavior & PSGPU_ALPHABLEND) != 0;
            uint32_t th = 0;
            int tid = 0;
            if (DEBUG && valid) {
                tid = (int)(d.id_base + (tri - d.tri_start));
                uint32_t h = (uint32_t)tid;
                h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
                th = h;
            }
            // lanes of the same chunk; with wide chunks, those of the chunk
            // that is the lane's
            const int of = OWN ? lane : key;
            uint64_t same = OWN ? __ballot(valid) : ~0ull;
#pragma unroll
            for (int bit = 0; bit < 6; bit++) {
                const uint64_t bm = __ballot((key >> bit) & 1);
                same &= ((of >> bit) & 1) ? bm : ~bm;
            }
            const bool all_test = __all(test || !valid);
            // candidates before this lane at the same pixel
            auto rank_of = [&](bool cand) {
                const uint64_t cm = same & __ballot(cand);
                return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(cm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)cm, 0));
            };
            // the lane's depth at pixel k, interpolateNextStep (interp.cpp:82-92)
            auto depth_at = [&](bool in, float& r) {
                r = 1.0f / cf2;
                const float z = pz * r;
                cf2 = in ? cf2 + cst : cf2;
                pz = in ? pz + pst : pz;
                return z;
            };
            auto can_pass = [&](bool in, float z, uint2 cur) {
                return in & (-1.0f < z) & (!all_test | (z - __uint_as_float(cur.x) < -0.0001f));
            };
            // the programme at the lane's pixel, and the step to the next.
            // Texture reads clamp their coordinates, so lanes without a
            // fragment run along.
            auto shade = [&](bool in, float r, uint32_t& col) {
                float v[NV > 0 ? NV : 1];
#pragma unroll
                for (int i = 0; i < NV; i++) {
                    v[i] = vs[i] * r;
                    vs[i] = in ? vs[i] + vt[i] : vs[i];
                }
                col = 0;
                return P::fpi(d, v, col);
            };
            auto drawn = [&](int k) {   // every rasterised fragment, passing or not
                const int64_t at = (int64_t)(int)rb.z * VW + ((pcx << cw_shift) + k);
                atomicAdd(&f.dbg_rcount[at], 1);
                atomicXor(&f.dbg_rhash[at], th);
            };
            // fragthrd.cpp:216-237 against the pixel as the rounds before left
            // it; the FP runs on a pass, and a discarded fragment leaves depth
            // as it was (fragthrd.cpp:227-236)
            auto fragment = [&](bool turn, int k, float z, int fr, uint32_t col, uint2 cur) {
                const float dd = test ? __uint_as_float(cur.x) : 1.0f;
                const bool pass = turn & (z - dd < -0.0001f);
                const bool depth = pass & upd & (fr != 2), paint = COLOUR & pass & wc & (fr == 1);
                if (depth) cur.x = __float_as_uint(z);
                if (paint) cur.y = blend ? ps_blend4(cur.y, col) : col;   // FBOBridge::write4 (fragthrd.cpp:70-82)
                *(depth | paint ? pix + k * 64 + key : spare) = cur;
                passes += pass ? 1u : 0u;
                if (DEBUG && pass) {
                    const int64_t at = (int64_t)(int)rb.z * VW + ((pcx << cw_shift) + k);
                    atomicAdd(&f.dbg_pcount[at], 1);
                    atomicXor(&f.dbg_phash[at], th);
                    f.dbg_last[at] = tid;
                }
            };
            if constexpr (UNROLL) {
                float z[KCW], r[KCW];
                uint2 cur[KCW];
                bool cand[KCW], some = false;
                int rank[KCW], fr[KCW], last = 0;
                uint32_t col[KCW];
#pragma unroll
                for (int k = 0; k < KCW; k++) cur[k] = pix[k * 64 + key];
#pragma unroll
                for (int k = 0; k < KCW; k++) {
                    const bool in = (k >= a) & (k <= b);
                    z[k] = depth_at(in, r[k]);
                    if (DEBUG && in) drawn(k);
                    cand[k] = can_pass(in, z[k], cur[k]);
                    some |= cand[k];
                }
                if (!__any(some)) continue;
#pragma unroll
                for (int k = 0; k < KCW; k++) fr[k] = shade((k >= a) & (k <= b), r[k], col[k]);
#pragma unroll
                for (int k = 0; k < KCW; k++) {
                    rank[k] = rank_of(cand[k]);
                    last = cand[k] ? max(last, rank[k]) : last;
                }
                for (int q = 0;;) {
#pragma unroll
                    for (int k = 0; k < KCW; k++) fragment(cand[k] & (rank[k] == q), k, z[k], fr[k], col[k], cur[k]);
                    if (DEBUG) __threadfence();   // the last pass of a pixel is stored last
                    ps_lds_turn();
                    q++;
                    if (!__any(last >= q)) break;
#pragma unroll
                    for (int k = 0; k < KCW; k++) cur[k] = pix[k * 64 + key];
                }
            } else if constexpr (OWN) {
                // each lane walks the pieces of its own chunk, one after the other
                const int ends = a | b << 8 | (int)(ra.x >> 26) << 16;
                int k = 1, last = 0, how = 0, dj = 0;
                float f2 = 0.0f, zn = 0.0f, f2s = 0.0f, zns = 0.0f;
                float ws[NV > 0 ? NV : 1], wt[NV > 0 ? NV : 1];
#pragma unroll
                for (int i = 0; i < NV; i++) ws[i] = wt[i] = 0.0f;
                auto from = [](int j, int v) { return __builtin_amdgcn_ds_bpermute(j * 4, v); };
                auto fromf = [&](int j, float v) { return __int_as_float(from(j, __float_as_int(v))); };
                while (__any((same != 0) | (k <= last))) {
                    const bool take = (k > last) & (same != 0);
                    if (__any(take)) {
                        const int j = __builtin_ctzll(same | 1ull << 63);
                        const int e = from(j, ends), g = from(j, di);
                        const float g0 = fromf(j, cf2), g1 = fromf(j, pz), g2 = fromf(j, cst), g3 = fromf(j, pst);
                        if (take) {
                            k = e & 0xff; last = e >> 8 & 0xff; how = e >> 16;
                            dj = g; f2 = g0; zn = g1; f2s = g2; zns = g3;
                            same &= same - 1;
                        }
#pragma unroll
                        for (int i = 0; i < NV; i++) {
                            const float s0 = fromf(j, vs[i]), s1 = fromf(j, vt[i]);
                            ws[i] = take ? s0 : ws[i];
                            wt[i] = take ? s1 : wt[i];
                        }
                    }
                    uint2* at = pix + min(k, CW - 1) * 64 + lane;
                    uint2 cur = *at;
                    const float r = 1.0f / f2, z = zn * r, dd = how & PSGPU_TEST_DEPTH ? __uint_as_float(cur.x) : 1.0f;
                    const bool pass = (k <= last) & (-1.0f < z) & (z - dd < -0.0001f);
                    if (__any(pass)) {
                        const PsDraw& dr = draws[dj];
                        float v[NV > 0 ? NV : 1];
#pragma unroll
                        for (int i = 0; i < NV; i++) v[i] = ws[i] * r;
                        uint32_t col = 0;
                        const int fr = P::fpi(dr, v, col);
                        const bool depth = pass & ((how & PSGPU_UPDATE_DEPTH) != 0) & (fr != 2);
                        const bool paint = COLOUR & pass & ((how & 4) != 0) & (fr == 1);
                        if (depth) cur.x = __float_as_uint(z);
                        if (paint) cur.y = (dr.behavior & PSGPU_ALPHABLEND) ? ps_blend4(cur.y, col) : col;
                        if (depth | paint) *at = cur;
                    }
                    passes += pass ? 1u : 0u;
                    f2 += f2s;
                    zn += zns;
#pragma unroll
                    for (int i = 0; i < NV; i++) ws[i] += wt[i];
                    k++;
                }
                ps_lds_turn();
            } else {
                for (int k = 0; k < CW; k++) {
                    const bool in = k >= a && k <= b;
                    if (!__any(in)) continue;
                    float r;
                    uint32_t col;
                    const float z = depth_at(in, r);
                    if (DEBUG && in) drawn(k);
                    const bool cand = can_pass(in, z, pix[k * 64 + key]);
                    const int fr = shade(in, r, col);
                    const int rank = rank_of(cand);
                    for (int q = 0; __any(cand && rank >= q); q++) {
                        fragment(cand && rank == q, k, z, fr, col, pix[k * 64 + key]);
                        if (DEBUG) __threadfence();
                        ps_lds_turn();
                    }
                }
            }
        }
    }
    // the colours that changed, then the depths of chunks in which one did
    bool dirty = dclear;
    if constexpr (UNROLL) {
        uint32_t dv[KCW];
#pragma unroll
        for (int k = 0; k < KCW; k++) {
            const uint2 q = pix[k * 64 + lane];
            dv[k] = q.x;
            dirty |= k < ncol && q.x != d0[k];
            if (COLOUR && k < ncol && q.y != c0[k]) crow[X0 + k] = q.y;
        }
        if (dirty) ps_store_run<KCW>((uint32_t*)drow + X0, ncol, dv);
    } else {
        // (one texture may be both targets)
        for (int k = 0; k < ncol; k++) dirty |= pix[k * 64 + lane].x != __float_as_uint(drow[X0 + k]);
        for (int k = 0; COLOUR && k < ncol; k++) {
            const uint32_t c = pix[k * 64 + lane].y;
            if (c != crow[X0 + k]) crow[X0 + k] = c;
        }
        if (dirty)
            for (int k = 0; k < ncol; k++) drow[X0 + k] = __uint_as_float(pix[k * 64 + lane].x);
    }
    ps_wave_add64(cnt, PS_ST_SHADED, passes);
}

// ---------------------------------------------------------------------------
// shade: deferred FP of the last colour-writing pass per pixel
// ---------------------------------------------------------------------------
// The winner plane names the triangle, so most pixels go winner -> triangle
// -> (draw, varyings) and re-derive the span's start (x1, cf2) from the
// triangle exactly as k_span did; only pixels of a piece with a varying
// checkpoint read that piece and its span first.
// a pixel of the programme, from its winner: the triangle, and of a piece with a
// checkpoint (from_ck) its index wi, first pixel xa and factor cfa there
template <int PROG>
__device__ __forceinline__ void ps_shade_pixel(const PsView& V, int x, int y, int64_t crow, int tri, const PsTri& tr, bool from_ck,
                                               uint32_t wi, int xa, float cfa, const float* __restrict__ ck, int ck_stride,
                                               const float* __restrict__ vary, int nvs, const float* __restrict__ grads,
                                               const PsDraw* __restrict__ draws)
{
    typedef PsProc<PROG> P;
    const int di = (int)(tr.code >> 8);
    PsEdge L, R;
    ps_row_edges(tr, y, L, R);
    int left = ps_cvt_i32(ps_edge_eval(L, (float)y) + 0.5f);
    int right = ps_cvt_i32(ps_edge_eval(R, (float)y) + 0.5f);
    PsSpanGeom g;
    ps_span_geom(tr, y, left, right, L, R, g);
    float cf2, cf2_step, pz, pz_step;
    ps_span_vis(tr, g, cf2, cf2_step, pz, pz_step);
    const float* u0 = vary + (int64_t)tr.vary * 3 * nvs;
    float vs[P::NV > 0 ? P::NV : 1], vt[P::NV > 0 ? P::NV : 1];
    ps_span_varyings<P::NV>(g, u0, u0 + nvs, u0 + 2 * nvs, vs, vt);
    // from the span's first pixel (leftClamped), or from the checkpoint,
    // the serial walk on to the pixel
    int xs = left < 0 ? 0 : left;
    if (from_ck) {
        const float* c = ck + (int64_t)wi * ck_stride;
#pragma unroll
        for (int i = 0; i < P::NV; i++) vs[i] = c[i];
        xs = xa;
        cf2 = cfa;
    }
    for (int k = xs; k < x; k++) {
        cf2 += cf2_step;
#pragma unroll
        for (int i = 0; i < P::NV; i++) vs[i] = vs[i] + vt[i];
    }
    float r = 1.0f / cf2;
    float in[P::NV > 0 ? P::NV : 1];
#pragma unroll
    for (int i = 0; i < P::NV; i++) in[i] = vs[i] * r;
    if constexpr (PROG == PSGPU_PROC_BLINN) {
        if (V.gbuf) {   // geometry buffer of the visible fragment (rows bottom-up)
            float4* gp = (float4*)(V.gbuf + ((int64_t)y * V.W + x) * 12);
            gp[0] = make_float4(in[6], in[7], in[8], 1.0f);
            gp[1] = make_float4(in[9], in[10], in[11], 0.0f);
            gp[2] = make_float4(in[12], in[13], 0.0f, 0.0f);
        }
    }
    float grad[6] = {0, 0, 0, 0, 0, 0};
    if constexpr (P::GRAD) {
        const float4* gi = (const float4*)(grads + (int64_t)tri * 8);
        float4 g0 = gi[0], g1 = gi[1];
        grad[0] = g0.x; grad[1] = g0.y; grad[2] = g0.z; grad[3] = g0.w; grad[4] = g1.x; grad[5] = g1.y;
    }
    // The programme, with the draw of the whole wave where it has only one: the
    // record's fields then come in with scalar loads and the branches on them
    // are scalar.  The index is opaque before it is made uniform: knowing it
    // equal to di, the compiler would index with di after all.  The geometry
    // stays out of the two branches, which spill with it.  Six waves per SIMD:
    // seven spill three registers for Blinn-Phong, 13 for its shadowed form.
    // Terrain 3840x2160 190 -> 176 us, 1920x1080 50 -> 46, 32 views 288 -> 267,
    // shadowed 1280x720 31.5 -> 27.9 (a loop over the wave's draws, one copy of
    // the code: 168, 50, 265, 38; waves of several draws on a list for a second
    // kernel: 168 + 20, 45 + 11, 270, 29 + 10).
    // What bounds the kernel is instruction issue, 90% of its time: some 1,280
    // per wave, a third of them the span's start and the walk to the pixel,
    // which neighbours share.  A lane per run of neighbours that leaves each
    // pixel its accumulators in LDS issues a quarter less, but its barriers
    // cost more (182 us against 176).  With ps_rsqrt and ps_texel_pair 160 us,
    // 44, 251, 28.0.
    uint32_t c;
    bool hit;
    if (__ballot(di != __builtin_amdgcn_readfirstlane(di)) == 0) {
        int du = di;
        asm volatile("" : "+v"(du));
        hit = P::fp(draws[__builtin_amdgcn_readfirstlane(du)], in, r, grad, c);
    } else {
        hit = P::fp(draws[di], in, r, grad, c);
    }
    if (hit) V.colour[crow * V.colour_scan + x] = c;
    else if (crow < V.cclear_rows) V.colour[crow * V.colour_scan + x] = V.cclear_value;
}

// PROG 0: every programme, each wave running through those of its pixels (see
// k_setup)
#define PS_SHADE_PROGS(X)                                                                            \
    X(PSGPU_PROC_DEF01) X(PSGPU_PROC_DEF02) X(PSGPU_PROC_DEF03) X(PSGPU_PROC_DEF04)                  \
    X(PSGPU_PROC_LAMBERT) X(PSGPU_PROC_BLINN) X(PSGPU_PROC_SHADOWED)
template <int PROG>
__global__ void __launch_bounds__(256, 6) k_shade(const PsSpan* __restrict__ spans, const PsSeg* __restrict__ segs,
                                               const float* __restrict__ ck, const PsTri* __restrict__ tris,
                                               const float* __restrict__ vary, int nvs, const float* __restrict__ grads,
                                               const PsDraw* __restrict__ draws, PsFrame f, const PsCounters* cnt)
{
    const bool poisoned = ps_poisoned(cnt);
    const int64_t lb = ps_xcd_remap<4>(blockIdx.x, gridDim.x);
    const PsView& V = f.views[ps_view_of_stile(f, lb)];
    int64_t st = lb - V.stile_base;
    // a view has fewer than 2^31 shading blocks
    const uint32_t st32 = (uint32_t)st, nsx = (uint32_t)V.n_stiles_x;
    int sy = (int)(st32 / nsx), sx = (int)(st32 - (uint32_t)sy * nsx);
    int x = sx * 16 + (threadIdx.x & 15);
    int y = sy * 16 + (threadIdx.x >> 4);
    if (x >= V.W || y >= V.H) return;
    const int64_t crow = V.colour_top_down ? (int64_t)(V.colour_h - 1 - y) : (int64_t)y;
    int w = V.winner[ps_winner_at(f, V, x, y)];
    if (poisoned) return;
    if (w == -1) {   // no fragment colours the pixel: a fused clear of its row, if any, is all it gets
        if (crow < V.cclear_rows) V.colour[crow * V.colour_scan + x] = V.cclear_value;
        return;
    }
    // a piece with a checkpoint: its first pixel xa carries the accumulators
    // as the serial walk from x1 leaves them
    const bool from_ck = (uint32_t)w & PS_SEG_CK;
    const uint32_t wi = (uint32_t)w & ~PS_SEG_CK;
    int tri = (int)wi, xa = 0;
    float cfa = 0.0f;
    if (from_ck) {
        const PsSeg sg = segs[wi];
        tri = spans[sg.si & PS_SEG_SPAN_MASK].tri;
        xa = (int)(sg.xab & 0xffffu);
        cfa = sg.cf2;
    }
    const PsTri tr = tris[tri];
    const int prog = ps_tri_prog(tr);
#define SH_PIXEL(K) \
    ps_shade_pixel<K>(V, x, y, crow, tri, tr, from_ck, wi, xa, cfa, ck, f.ck_stride, vary, nvs, grads, draws)
    if constexpr (PROG != 0) {
        if (prog == PROG) SH_PIXEL(PROG);
    } else {
#define SH_ONE(K) if (prog == K) SH_PIXEL(K);
        PS_SHADE_PROGS(SH_ONE)
#undef SH_ONE
    }
#undef SH_PIXEL
}

// ---------------------------------------------------------------------------
// mip chain: rounded 2x2 mean, level l-1 -> l
// ---------------------------------------------------------------------------
// One block takes a 64 x 64 square of the source level through up to six
// levels: each of their texels depends on that square alone, since a level
// halves rounding down (an odd last column or row is not read), and a side of
// one texel is its own pair.  The levels stay in LDS between the steps, so the
// chain reads its source once and a texture of up to 4,096 texels a side takes
// two launches, for all its layers at once; one launch per level and layer
// spent its time between launches (six layers of 1024^2: 60 launches, 217 to
// 222 us; now 2 of 5 to 8 us, 22 with the wait at their end).
__device__ __forceinline__ uint32_t ps_mean4(uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
    const uint32_t m = 0x00ff00ffu, r = 0x00020002u;   // two 16-bit sums a word
    const uint32_t e = ((a & m) + (b & m) + (c & m) + (d & m) + r) >> 2 & m;
    const uint32_t o = ((a >> 8 & m) + (b >> 8 & m) + (c >> 8 & m) + (d >> 8 & m) + r) >> 2 & m;
    return e | o << 8;
}

// E: bytes a texel (4 or 1)
template <int E>
__global__ void __launch_bounds__(256) k_mips(uint8_t* __restrict__ data, int64_t layer_bytes, PsMips m)
{
    __shared__ uint32_t lv[2][32 * 32];
    uint8_t* base = data + (int64_t)blockIdx.y * layer_bytes;
    const int nx = (m.w + 63) / 64, by = blockIdx.x / nx;
    const int t = threadIdx.x, ox = (blockIdx.x - by * nx) * 64, oy = by * 64;
    auto side = [](int n, int l) { return max(1, n >> l); };
    auto store = [&](int l, int x, int y, uint32_t v) {   // local texel (x, y) of level l of the block
        const int w = side(m.w, l), gx = (ox >> l) + x, gy = (oy >> l) + y;
        if (gx >= w || gy >= side(m.h, l)) return;
        uint8_t* p = base + m.off[l] + ((int64_t)gy * w + gx) * E;
        if constexpr (E == 4) *(uint32_t*)p = v;
        else *p = (uint8_t)v;
    };
    // level 1 from memory: a thread takes two texels, four source columns wide
    const bool vec = E == 4 && (m.w & 3) == 0 && ((uintptr_t)(base + m.off[0]) & 15) == 0;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int u = t + q * 256, x = u % 16 * 2, y = u / 16;   // of level 1 in the block
        const int gx = ox + 2 * x, gy0 = oy + 2 * y, gy1 = min(gy0 + 1, m.h - 1);
        uint32_t a[4] = {0, 0, 0, 0}, b[4] = {0, 0, 0, 0};
        if (gx < m.w && gy0 < m.h) {
            const uint8_t* r0 = base + m.off[0] + ((int64_t)gy0 * m.w + gx) * E;
            const uint8_t* r1 = base + m.off[0] + ((int64_t)gy1 * m.w + gx) * E;
            if (vec) {
                const uint4 p = *(const uint4*)r0, s = *(const uint4*)r1;
                a[0] = p.x; a[1] = p.y; a[2] = p.z; a[3] = p.w;
                b[0] = s.x; b[1] = s.y; b[2] = s.z; b[3] = s.w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int c = min(gx + k, m.w - 1) - gx;   // past the row: the last texel, which only a side of one reads
                    a[k] = E == 4 ? *(const uint32_t*)(r0 + c * E) : r0[c];
                    b[k] = E == 4 ? *(const uint32_t*)(r1 + c * E) : r1[c];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t v = ps_mean4(a[2 * k], a[2 * k + 1], b[2 * k], b[2 * k + 1]);
            lv[1][y * 32 + x + k] = v;
            store(1, x + k, y, v);
        }
    }
#pragma unroll
    for (int l = 2; l <= 6; l++) {
        if (l > m.levels) return;
        __syncthreads();
        const int n = 64 >> l, stride = 64 >> (l - 1);
        const uint32_t* src = lv[(l - 1) & 1];
        if (t < n * n) {
            const int x = t % n, y = t / n;
            // a side of one texel above this level: its only column (row)
            const int x1 = side(m.w, l - 1) == 1 ? 0 : 2 * x + 1, y1 = side(m.h, l - 1) == 1 ? 0 : 2 * y + 1;
            const uint32_t v = ps_mean4(src[2 * y * stride + 2 * x], src[2 * y * stride + x1], src[y1 * stride + 2 * x],
                                        src[y1 * stride + x1]);
            lv[l & 1][y * n + x] = v;
            store(l, x, y, v);
        }
    }
}

__global__ void k_selftest(int op, const float* a, const float* b, float* out, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float r = 0.0f;
    switch (op) {
    case 0: r = a[i] / b[i]; break;
    case 1: r = sqrtf(a[i]); break;
    case 2: r = 1.0f / a[i]; break;
    case 3: r = (float)ps_cvt_i32(a[i]); break;
    case 4: r = floorf(a[i]); break;
    case 5: r = (float)(int)ps_cvt_u32(a[i]); break;
    case 6: r = ps_log2(a[i]); break;
    case 7: r = a[i]; break;   // plain copy: 4 bytes read + 4 written per element
    case 8: case 9: {           // wrapped texel pair (v, v + 1) modulo m; int bits in and out
        int v = __float_as_int(a[i]), m = __float_as_int(b[i]), c0, c1;
        ps_clamp_pair(1, m, v, c0, c1);
        r = __int_as_float(op == 8 ? c0 : c1);
        break;
    }
    case 10: r = (float)ps_sse_pack_byte(a[i]); break;
    case 11: r = ps_rsqrt(a[i]); break;
    case 12: case 13: {         // texel pair of a whole coordinate, m the last texel, wrapped where the sign bit of m is set
        int m = __float_as_int(b[i]), c0, c1;
        ps_texel_pair(m < 0, m & 0x7fffffff, a[i], c0, c1);
        r = __int_as_float(op == 12 ? c0 : c1);
        break;
    }
    }
    out[i] = r;
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
static inline int gsz(int64_t n, int b) { int64_t g = (n + b - 1) / b; return (int)(g < 1 ? 1 : g); }

void psk_fill_u32(hipStream_t s, uint32_t* p, int64_t n, uint32_t v, const PsCounters* c)
{
    if (n <= 0) return;
    int g = gsz(n, 256); if (g > 4096) g = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3(g), dim3(256), 0, s, p, n, v, c);
}

int64_t psk_fill_pieces(int64_t rows, int64_t width) { return rows * ((width + FILL_PIECE - 1) / FILL_PIECE); }

void psk_fills(hipStream_t s, const PsFill* fills, int n, int64_t max_pieces, const PsCounters* c)
{
    if (n <= 0) return;
    int64_t g = max_pieces < 1 ? 1 : max_pieces; if (g > 4096) g = 4096;
    hipLaunchKernelGGL(k_fills, dim3((unsigned)g, n), dim3(256), 0, s, fills, c);
}

void psk_few_fills(hipStream_t s, const PsFewFills& fills, int n, int64_t max_pieces, const PsCounters* c)
{
    if (n <= 0) return;
    int64_t g = max_pieces < 1 ? 1 : max_pieces; if (g > 4096) g = 4096;
    hipLaunchKernelGGL(k_few_fills, dim3((unsigned)g, n), dim3(256), 0, s, fills, c);
}

void psk_finish(hipStream_t s, PsCounters* c, uint32_t* sizes, PsFinish* out, bool reset)
{
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(64), 0, s, c, sizes, out, reset ? 1 : 0);
}


int psk_setup_block() { return 128; }

void psk_setup(hipStream_t s, int prog, bool share, const PsDraw* draws, int nd, int64_t T, PsTri* tris, float* vary, int nvs,
               float* grads, uint32_t* nrows, uint32_t* row_part, PsCounters* cnt, const PsView* views)
{
    dim3 g(gsz(T, 128)), b(128);
    size_t lds = (size_t)128 * 3 * nvs * sizeof(float);
#define SU_CASE(K)                                                                                                  \
    case K:                                                                                                         \
        if (share && (K == 0 || ps_shares_varyings(K)))                                                                         \
            hipLaunchKernelGGL((k_setup<K, true>), g, b, lds, s, draws, nd, T, tris, vary, nvs, grads, nrows, row_part, cnt, views); \
        else                                                                                                        \
            hipLaunchKernelGGL((k_setup<K, false>), g, b, lds, s, draws, nd, T, tris, vary, nvs, grads, nrows, row_part, cnt, views); \
        break;
    switch (prog) {
    SU_CASE(0) PS_SETUP_PROGS(SU_CASE) SU_CASE(PSGPU_PROC_CLOUD) SU_CASE(PSGPU_PROC_CLOUD_SHADOW)
    }
#undef SU_CASE
}

int psk_scan_blocks(int64_t cap) { return gsz(cap, SCAN_BLOCK); }


void psk_scan_parts(hipStream_t s, const uint32_t* in, int64_t n, uint32_t* out, const uint32_t* parts, int pgran,
                    uint32_t* total_out, uint32_t* bstart, int64_t bcap, unsigned long long* wide)
{
    hipLaunchKernelGGL(k_scan_parts, dim3(psk_scan_blocks(n)), dim3(1024), 0, s, in, n, parts, pgran, out, total_out,
                       bstart, bcap, wide);
}

int psk_heavy_cap() { return PS_HEAVY_MAX; }

void psk_scan_tiles(hipStream_t s, const unsigned long long* tcnt, int64_t n, unsigned long long* tstart,
                    unsigned long long* partial, uint32_t* total_out, unsigned long long* wide, int64_t seg_cap, PsCounters* c,
                    uint32_t* heavy, int* flag)
{
    if (n <= SCAN_DIRECT_MAX) {
        hipLaunchKernelGGL(k_scan_direct, dim3(gsz(n, DIRECT_BLOCK)), dim3(1024), 0, s, tcnt, n, tstart,
                           total_out, wide, seg_cap, c, heavy, flag);
        return;
    }
    int nb = psk_scan_blocks(n);
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(256), 0, s, tcnt, n, partial, c);
    hipLaunchKernelGGL(k_scan_final, dim3(nb), dim3(256), 0, s, tcnt, n, partial, nb, tstart, total_out, wide, seg_cap, c, heavy, flag);
}


void psk_span(hipStream_t s, const PsTri* tris, const uint32_t* row_off, const uint32_t* bstart, int64_t T,
              PsSpan* spans, unsigned long long* tcnt, const PsView* views, int n_views, int chunk_w, int tile_rows,
              int64_t cap, uint32_t* heavy, unsigned long long* wide, PsCounters* cnt, int* flag)
{
    int g = gsz(cap, 256); if (g > 2048) g = 2048;
    const int tile_cols = 64 / tile_rows;
    hipLaunchKernelGGL(k_span, dim3(g), dim3(256), 0, s, tris, row_off, bstart, T, cap, spans, tcnt, views, n_views,
                       chunk_w, tile_rows, tile_cols, heavy, wide, cnt, flag);
}

void psk_segments(hipStream_t s, const PsSpan* spans, const uint32_t* row_off, int64_t T, const PsFrame& f,
                  const PsTri* tris, const PsDraw* draws, const float* vary, int nvs, unsigned long long* tcnt, PsSeg* segs,
                  float* ck, int64_t span_cap, int64_t seg_cap, const unsigned long long* wide, PsCounters* cnt, int* flag)
{
    int g = gsz(span_cap, 256); if (g > 2048) g = 2048;
#define SG_LAUNCH(G)                                                                                                  \
    hipLaunchKernelGGL(k_segments<G>, dim3(g), dim3(256), 0, s, spans, row_off, T, f, tris, draws, vary, nvs, tcnt,   \
                       segs, ck, seg_cap, wide, PS_WIDE_PER(span_cap), cnt, flag)
    static_assert(PS_MAX_NV <= 24, "a lane per varying float beside the 8 of the record");
    if (nvs <= 8) SG_LAUNCH(16);
    else SG_LAUNCH(32);
#undef SG_LAUNCH
}

// the tilings taken and refused go by 1,024 words a wave beside the pixels,
// which the kernels stay below
size_t psk_raster_lds(int chunk_w, int waves)
{
    static_assert(RA_PIX_WORDS(0) <= 1024, "a tiling that is taken fits");
    return (size_t)waves * (chunk_w * 64 * 2 + 1024) * 4;
}

void psk_raster(hipStream_t s, bool debug, const PsSpan* spans, const PsSeg* segs, const PsTri* tris, const PsDraw* draws,
                const PsFrame& f, int waves_per_group, PsCounters* cnt)
{
    int64_t n_tiles = f.n_tiles;
    const int cw = f.chunk_w;
    const bool known = cw == 1 || cw == 2 || cw == 4 || cw == 8;
    size_t lds = (size_t)waves_per_group * RA_PIX_WORDS(cw) * 4;
    dim3 g(gsz(n_tiles + (f.heavy ? ps_heavy_cap(n_tiles) : 0), waves_per_group)), b(64 * waves_per_group);
#define RA_LAUNCH(D, K) hipLaunchKernelGGL((k_raster<D, K>), g, b, lds, s, spans, segs, tris, draws, f, n_tiles, cnt)
    switch (known ? cw : 0) {
    case 1: if (debug) RA_LAUNCH(true, 1); else RA_LAUNCH(false, 1); break;
    case 2: if (debug) RA_LAUNCH(true, 2); else RA_LAUNCH(false, 2); break;
    case 4: if (debug) RA_LAUNCH(true, 4); else RA_LAUNCH(false, 4); break;
    case 8: if (debug) RA_LAUNCH(true, 8); else RA_LAUNCH(false, 8); break;
    default: if (debug) RA_LAUNCH(true, 0); else RA_LAUNCH(false, 0); break;
    }
#undef RA_LAUNCH
}

void psk_raster_imm(hipStream_t s, int prog, bool debug, const PsSpan* spans, const PsSeg* segs, const PsTri* tris,
                    const PsDraw* draws, const PsFrame& f, int waves_per_group, PsCounters* cnt, const float* vary, int nvs,
                    const float* ck)
{
    int64_t n_tiles = f.n_tiles;
    size_t lds = (size_t)waves_per_group * RA_PIX_WORDS(f.chunk_w) * 4;
    dim3 g(gsz(n_tiles, waves_per_group)), b(64 * waves_per_group);
#define RI_LAUNCH(P, D, K)                                                                                           \
    hipLaunchKernelGGL((k_raster_imm<P, D, K>), g, b, lds, s, spans, segs, tris, draws, f, n_tiles, cnt, vary, nvs, ck)
#define RI_CASE(P)                                                                                                   \
    case P:                                                                                                          \
        if (debug) RI_LAUNCH(P, true, 0);                                                                            \
        else if (f.chunk_w == 4) RI_LAUNCH(P, false, 4);                                                             \
        else if (f.chunk_w == 64) RI_LAUNCH(P, false, 64);                                                           \
        else RI_LAUNCH(P, false, 0);                                                                                 \
        break;
    switch (prog) {
    RI_CASE(PSGPU_PROC_CLOUD) RI_CASE(PSGPU_PROC_CLOUD_SHADOW)
    default: break;
    }
#undef RI_CASE
#undef RI_LAUNCH
}

void psk_shade(hipStream_t s, int prog, const PsSpan* spans, const PsSeg* segs, const float* ck, const PsTri* tris,
               const float* vary, int nvs, const float* grads, const PsDraw* draws, const PsFrame& f, const PsCounters* cnt)
{
    dim3 g((unsigned)f.n_stiles), b(256);
#define SH_CASE(K) case K: hipLaunchKernelGGL(k_shade<K>, g, b, 0, s, spans, segs, ck, tris, vary, nvs, grads, draws, f, cnt); break;
    switch (prog) {
    SH_CASE(0) PS_SHADE_PROGS(SH_CASE)
    default: break;
    }
#undef SH_CASE
}

void psk_mips(hipStream_t s, uint8_t* data, int64_t layer_bytes, int layers, int elem, const PsMips& m)
{
    const dim3 g((unsigned)((m.w + 63) / 64) * (unsigned)((m.h + 63) / 64), layers);
    if (elem == 4) hipLaunchKernelGGL(k_mips<4>, g, dim3(256), 0, s, data, layer_bytes, m);
    else hipLaunchKernelGGL(k_mips<1>, g, dim3(256), 0, s, data, layer_bytes, m);
}

void psk_selftest(hipStream_t s, int op, const float* a, const float* b, float* out, int n)
{
    hipLaunchKernelGGL(k_selftest, dim3(gsz(n, 256)), dim3(256), 0, s, op, a, b, out, n);
}
