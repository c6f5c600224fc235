// ps_adjoint.hip -- differentiable texture sampling and shading on a geometry
// buffer, forward and hand-written adjoint (psgpu_diff_forward/_backward).
//
// Model, per covered pixel p with geometry (N, wp, u, v):
//   n = N/|N|, L = norm(light - wp), E = norm(camera - wp), H = norm(L + E)
//   lam = max(n.L, 0), s = max(n.H, 0), spec = s > 0 ? ks * s^e : 0
//   T = sum_k w_k * tex[texel_k]        (bilinear, 4 texels, wrapping)
//   c = a * T * lam + spec              (per RGB channel)
// Adjoint, with g = dLoss/dc:
//   dLoss/dtex[texel_k] += a * lam * w_k * g       (atomics: texels are shared)
//   dLoss/da            += sum_c g_c * T_c * lam
//   dLoss/de            += sum_c g_c * spec * ln(s)
// Visibility is the geometry buffer's: it does not move with the parameters.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include "../../include/psgpu.h"

namespace {

struct DiffArgs {
    int W, H, tw, th;
    float light[3], camera[3];
    float ks;
};

struct Geo {
    bool covered;
    float lam, s, spec, u, v;
};

// lam and s from 64-bit sums and roots, rounded once, for both passes: a pixel
// whose highlight the image has is one whose highlight the gradients have.
// In FP32 the normalisations round unit vectors' lengths to one side, the
// exponent multiplies that, and the bias it leaves in the image (some 1e-7)
// was the largest part of the parameter gradients' error, which sum
// differences to a target over the whole image (1237x891: 1.0e-6 to 1.7e-6,
// now 0.1e-6 to 1.2e-6, the rounding of their own atomics); and where the
// half vector grazes the surface, the sign of s was that of the rounding.  The
// passes are bound by reading the geometry and by their atomics, and take as
// long as with FP32 sums (1237x891: 12 and 34 us, 512^2: 5 and 26).
__device__ __forceinline__ Geo geometry(const DiffArgs& A, const float* __restrict__ gbuf, int64_t p, float e)
{
    Geo g;
    const float4* gp = (const float4*)(gbuf + p * 12);
    const float4 g0 = gp[0], g1 = gp[1], g2 = gp[2];
    g.covered = g0.w != 0.0f;
    if (!g.covered) return g;
    const double n[3] = {g0.x, g0.y, g0.z}, at[3] = {g1.x, g1.y, g1.z};
    double L[3], E[3], H[3];
    auto dot = [](const double* u, const double* v) { return (u[0] * v[0] + u[1] * v[1]) + u[2] * v[2]; };
#pragma unroll
    for (int k = 0; k < 3; k++) { L[k] = (double)A.light[k] - at[k]; E[k] = (double)A.camera[k] - at[k]; }
    const double rn = rsqrt(dot(n, n)), rl = rsqrt(dot(L, L)), re = rsqrt(dot(E, E));
#pragma unroll
    for (int k = 0; k < 3; k++) H[k] = L[k] * rl + E[k] * re;
    const float lam = (float)(dot(n, L) * rl * rn), s = (float)(dot(n, H) * rsqrt(dot(H, H)) * rn);
    g.lam = lam > 0.0f ? lam : 0.0f;
    g.s = s > 0.0f ? s : 0.0f;
    g.spec = g.s > 0.0f ? A.ks * powf(g.s, e) : 0.0f;
    g.u = g2.x;
    g.v = g2.y;
    return g;
}

// bilinear footprint: texel j covers u = j/tw; wrapping addresses.  (ix, iy)
// is its first texel, (ax, ay) the weights of the second ones.
__device__ __forceinline__ void footprint_at(const DiffArgs& A, float u, float v, int& ix, int& iy, float& ax, float& ay)
{
    float fx = u * (float)A.tw, fy = v * (float)A.th;
    if (!(fabsf(fx) < 1073741824.0f)) fx = 0.0f;
    if (!(fabsf(fy) < 1073741824.0f)) fy = 0.0f;
    float x0 = floorf(fx), y0 = floorf(fy);
    ax = fx - x0;
    ay = fy - y0;
    ix = (int)x0 % A.tw;
    iy = (int)y0 % A.th;
    if (ix < 0) ix += A.tw;
    if (iy < 0) iy += A.th;
}

__device__ __forceinline__ void footprint_texels(const DiffArgs& A, int ix, int iy, float ax, float ay, int64_t* idx, float* w)
{
    int ix1 = ix + 1 == A.tw ? 0 : ix + 1, iy1 = iy + 1 == A.th ? 0 : iy + 1;
    idx[0] = (int64_t)iy * A.tw + ix;
    idx[1] = (int64_t)iy * A.tw + ix1;
    idx[2] = (int64_t)iy1 * A.tw + ix;
    idx[3] = (int64_t)iy1 * A.tw + ix1;
    w[0] = (1.0f - ax) * (1.0f - ay);
    w[1] = ax * (1.0f - ay);
    w[2] = (1.0f - ax) * ay;
    w[3] = ax * ay;
}

__device__ __forceinline__ void footprint(const DiffArgs& A, float u, float v, int64_t* idx, float* w)
{
    int ix, iy;
    float ax, ay;
    footprint_at(A, u, v, ix, iy, ax, ay);
    footprint_texels(A, ix, iy, ax, ay, idx, w);
}

__global__ void __launch_bounds__(256) k_diff_forward(DiffArgs A, const float* __restrict__ gbuf,
                                                      const float* __restrict__ tex, const float* __restrict__ params,
                                                      float* __restrict__ out)
{
    int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= (int64_t)A.W * A.H) return;
    float a = params[0], e = params[1];
    Geo g = geometry(A, gbuf, p, e);
    float c[3] = {0.0f, 0.0f, 0.0f};
    if (g.covered) {
        int64_t idx[4];
        float w[4];
        footprint(A, g.u, g.v, idx, w);
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            float t = ((w[0] * tex[idx[0] * 3 + ch] + w[1] * tex[idx[1] * 3 + ch]) + w[2] * tex[idx[2] * 3 + ch]) +
                      w[3] * tex[idx[3] * 3 + ch];
            c[ch] = a * t * g.lam + g.spec;
        }
    }
    out[p * 3 + 0] = c[0];
    out[p * 3 + 1] = c[1];
    out[p * 3 + 2] = c[2];
}

// The backward pass takes the image in tiles of 32 x 32 pixels, a block of
// eight waves each, and adds up a tile's texel gradients in LDS before they go
// to memory.  Neighbouring pixels share texels (the footprints of 1,024 pixels
// cover about as many texels where a texel is as wide as a pixel, a handful
// where one is magnified), and what does go out is a rectangle of the texture,
// whose atomics take whole cache lines: 12 scattered atomics a pixel, and two
// per wave on the one line of the parameters, were all of the time.
// LDS float atomics take some two cycles a lane, so contributions to the same
// texels are added up before them: a thread's two pixels, one above the other,
// and then the lanes of a quad.
// Blocks go over the tiles in turn and keep the parameter sums in registers:
// one atomic a block for each.  (The texture gradients of a frame cost the
// same with half the threads a block, but twice the atomics on the parameters
// round their sums twice as often.)  A texture that fits LDS stays there over
// all of a block's tiles.  A tile whose texels do not fit (more than about 1.7
// texels a pixel, or torn apart) scatters its own: going wave by wave instead,
// a part of the tile at a time, takes longer.
// 512^2 image and 1024^2 texture 120 -> 29 us, 1237x891 and 250x130 834 -> 37;
// reading the geometry, texels and gradients takes 8 and 18 of them, the rest
// is the chain of reductions and barriers of a tile and its LDS atomics.
const int kTileW = 32, kTileH = 32, kDiffThreads = 512, kDiffWaves = kDiffThreads / 64;
const int kLdsTexels = 3400;   // 40 KiB
// Images of up to so many pixels (see k_diff_backward_small), and of up to so
// many a texel and beside them: of few texels all waves share some.
// In tiles and there, us: 8x8 texels, 40^2 pixels 9.8 and 8.2, 64^2 9.8 and
// 11.3; 16x16, 80^2 10.7 and 9.6, 128^2 11.0 and 13.5; 32x32, 181x140 12.4 and
// 11.9.  The same texture magnified until 181x140 pixels lie in four texels
// takes 11.4 and 13.1, and more beyond; 200^2 pixels with a texel each 25 and 13.
const int64_t kSmallPixels = 32768, kSmallPerTexel = 24, kSmallBeside = 1024;
const int kSmallTile = 16, kSmallThreads = kSmallTile * kSmallTile;

// Whether the texture stays in LDS: with the first column and row again at the
// end, so that footprints need not wrap there either.
__host__ __device__ __forceinline__ bool whole_in_lds(const DiffArgs& A)
{
    return ((int64_t)A.tw + 1) * ((int64_t)A.th + 1) <= kLdsTexels;
}

// the wave's minimum, in every lane
__device__ __forceinline__ int wave_min(int v)
{
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, false));    // quad_perm [1,0,3,2]
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, false));    // quad_perm [2,3,0,1]
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, false));   // row_half_mirror
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x140, 0xf, 0xf, false));   // row_mirror
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// a texture coordinate in the texture moved by half its size n, so that its
// ends lie in the middle
__device__ __forceinline__ int half_round(int v, int n) { return v < n / 2 ? v + (n - n / 2) : v - n / 2; }

// A rectangle of texels: columns x .. x + w - 1 and rows y .. y + h - 1 of the
// texture as it lies or (mx, my) moved by half its width (height), whichever is
// smaller: one of them is not torn where the coordinates wrap.  The second
// texels of the footprints included; w is 0 where nothing is covered.
struct TexRect {
    int x, y, w, h;
    bool mx, my;
    __device__ int64_t texels() const { return (int64_t)w * h; }
};

__device__ __forceinline__ TexRect tex_rect(const int* e)
{
    TexRect r = {0, 0, 0, 0, false, false};
    if (e[0] == INT_MAX) return r;
    r.mx = -e[6] - e[4] < -e[2] - e[0];
    r.my = -e[7] - e[5] < -e[3] - e[1];
    r.x = r.mx ? e[4] : e[0];
    r.y = r.my ? e[5] : e[1];
    r.w = -(r.mx ? e[6] : e[2]) - r.x + 2;
    r.h = -(r.my ? e[7] : e[3]) - r.y + 2;
    return r;
}

// the value that lane ^ X has
template <int X>
__device__ __forceinline__ int lane_xor(int v)
{
    if (X == 1) return __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, false);   // quad_perm [1,0,3,2]
    if (X == 2) return __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, false);   // quad_perm [2,3,0,1]
    return __shfl_xor(v, X, 64);
}

// One step of adding up the lanes' contributions: lanes whose key equals that
// of lane ^ X take both, and the upper of the two drops out (key -1).  Called
// by every lane.
template <int X>
__device__ __forceinline__ void merge_lanes(int& key, float* c, bool upper)
{
    // read before any branch: a lane switched off by one would read as 0
    const int other = lane_xor<X>(key);
    const bool same = (other == key) & (key >= 0);
    if (!__any(same)) return;
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const float o = __int_as_float(lane_xor<X>(__float_as_int(c[k])));
        c[k] = same ? c[k] + o : c[k];
    }
    if (same && upper) key = -1;
}

__global__ void __launch_bounds__(kDiffThreads) k_diff_backward(DiffArgs A, const float* __restrict__ gbuf,
                                                               const float* __restrict__ tex, const float* __restrict__ params,
                                                               const float* __restrict__ gout, float* __restrict__ gtex,
                                                               float* __restrict__ gparams, int tiles_x, int64_t n_tiles)
{
    __shared__ float acc[kLdsTexels * 3];   // the texels' sums; all zero between tiles
    // of each wave's pixels: smallest texel column and row, and the largest
    // ones' negatives: [0..3] of the coordinates, [4..7] of the coordinates
    // half a texture further
    __shared__ int ext[kDiffWaves][8];
    __shared__ double sums[2][kDiffWaves];
    const int t = threadIdx.x, wave = t >> 6;
    const float a = params[0], e = params[1];
    const bool whole = whole_in_lds(A);
    double ga = 0.0, ge = 0.0;   // sums over many pixels: the terms are FP32
    for (int k = t; k < kLdsTexels * 3; k += kDiffThreads) acc[k] = 0.0f;
#pragma unroll 1
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int ty = (int)(tile / tiles_x), tx = (int)(tile - (int64_t)ty * tiles_x);
        const int x = tx * kTileW + (t & (kTileW - 1));
        // the thread's pixels q = 0, 1: (x, y + q)
        bool covered[2];
        int ix[2], iy[2];
        float ax[2], ay[2], gc[2][3];
        int lo[8];
#pragma unroll
        for (int k = 0; k < 8; k++) lo[k] = INT_MAX;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int y = ty * kTileH + t / kTileW * 2 + q;
            covered[q] = false;
            ix[q] = iy[q] = 0;
            if (x >= A.W || y >= A.H) continue;
            const int64_t p = (int64_t)y * A.W + x;
            const Geo g = geometry(A, gbuf, p, e);
            covered[q] = g.covered;
            if (!g.covered) continue;
            int64_t idx[4];
            float w[4];
            footprint_at(A, g.u, g.v, ix[q], iy[q], ax[q], ay[q]);
            footprint_texels(A, ix[q], iy[q], ax[q], ay[q], idx, w);
            const float go[3] = {gout[p * 3], gout[p * 3 + 1], gout[p * 3 + 2]};
            const float al = a * g.lam;
#pragma unroll
            for (int ch = 0; ch < 3; ch++) {
                float s = ((w[0] * tex[idx[0] * 3 + ch] + w[1] * tex[idx[1] * 3 + ch]) + w[2] * tex[idx[2] * 3 + ch]) +
                          w[3] * tex[idx[3] * 3 + ch];
                ga += (double)(go[ch] * s * g.lam);
                gc[q][ch] = go[ch] * al;
            }
            if (g.s > 0.0f) ge += (double)(((go[0] + go[1]) + go[2]) * g.spec * logf(g.s));
            const int sx = half_round(ix[q], A.tw), sy = half_round(iy[q], A.th);
            lo[0] = min(lo[0], ix[q]); lo[1] = min(lo[1], iy[q]); lo[2] = min(lo[2], -ix[q]); lo[3] = min(lo[3], -iy[q]);
            lo[4] = min(lo[4], sx); lo[5] = min(lo[5], sy); lo[6] = min(lo[6], -sx); lo[7] = min(lo[7], -sy);
        }
        if (!whole) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int m = wave_min(lo[k]);
                if ((t & 63) == 0) ext[wave][k] = m;
            }
        }
        __syncthreads();
        TexRect r = {0, 0, A.tw + 1, A.th + 1, false, false};
        if (!whole) {
            int e8[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                e8[k] = ext[0][k];
#pragma unroll
                for (int w = 1; w < kDiffWaves; w++) e8[k] = min(e8[k], ext[w][k]);
            }
            r = tex_rect(e8);
        }
        if (r.texels() <= kLdsTexels) {
            int key[2];
            float c[2][12];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int cx = r.mx ? half_round(ix[q], A.tw) : ix[q], cy = r.my ? half_round(iy[q], A.th) : iy[q];
                key[q] = covered[q] ? (cy - r.y) * r.w + (cx - r.x) : -1;
                const float w[4] = {(1.0f - ax[q]) * (1.0f - ay[q]), ax[q] * (1.0f - ay[q]), (1.0f - ax[q]) * ay[q], ax[q] * ay[q]};
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int ch = 0; ch < 3; ch++)
                        c[q][k * 3 + ch] = covered[q] && gc[q][ch] != 0.0f && w[k] != 0.0f ? gc[q][ch] * w[k] : 0.0f;
            }
            if (key[0] == key[1]) {
#pragma unroll
                for (int k = 0; k < 12; k++) c[0][k] += c[1][k];
                key[1] = -1;
            }
#pragma unroll
            for (int q = 0; q < 2; q++) {
                merge_lanes<1>(key[q], c[q], t & 1);
                merge_lanes<2>(key[q], c[q], t & 2);
            }
#pragma unroll
            for (int q = 0; q < 2; q++) {
                if (key[q] < 0) continue;
                float* at = acc + key[q] * 3;
                const int down = r.w * 3;
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int ch = 0; ch < 3; ch++)
                        if (c[q][k * 3 + ch] != 0.0f)
                            unsafeAtomicAdd(at + ((k & 1) ? 3 : 0) + ((k & 2) ? down : 0) + ch, c[q][k * 3 + ch]);
            }
            if (!whole || tile + gridDim.x >= n_tiles) {
                __syncthreads();
                // the rectangle's rows, consecutive threads on consecutive
                // floats, at the texture's own columns and rows
                const int x0 = r.mx ? r.x + A.tw / 2 : r.x, y0 = r.my ? r.y + A.th / 2 : r.y;
                const int row = r.w * 3, n = row * r.h;
                if (n > 0) {
                    const int dr = kDiffThreads / row, dc = kDiffThreads - dr * row;
                    int y = t / row, f = t - y * row;
                    for (int k = t; k < n; k += kDiffThreads) {
                        const float v = acc[k];
                        acc[k] = 0.0f;
                        if (v != 0.0f) {
                            const int tc = f / 3;
                            int gx = x0 + tc, gy = y0 + y;   // below twice the texture's size
                            gx = gx >= A.tw ? gx - A.tw : gx;
                            gy = gy >= A.th ? gy - A.th : gy;
                            unsafeAtomicAdd(gtex + ((int64_t)gy * A.tw + gx) * 3 + (f - tc * 3), v);
                        }
                        f += dc;
                        y += dr;
                        if (f >= row) { f -= row; y++; }
                    }
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                if (!covered[q]) continue;
                int64_t idx[4];
                float w[4];
                footprint_texels(A, ix[q], iy[q], ax[q], ay[q], idx, w);
#pragma unroll
                for (int ch = 0; ch < 3; ch++)
                    if (gc[q][ch] != 0.0f) {
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            if (w[k] != 0.0f) unsafeAtomicAdd(gtex + idx[k] * 3 + ch, gc[q][ch] * w[k]);
                    }
            }
        }
        __syncthreads();   // the next tile writes its extents
    }
    // the block's sums, one atomic for each parameter
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ga += __shfl_xor(ga, o, 64);
        ge += __shfl_xor(ge, o, 64);
    }
    if ((t & 63) == 0) { sums[0][t >> 6] = ga; sums[1][t >> 6] = ge; }
    __syncthreads();
    if (t < 2) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kDiffWaves; w++) s += sums[t][w];
        unsafeAtomicAdd(gparams + t, (float)s);
    }
}

// The same for an image of few pixels, which would leave most CUs without a
// tile (64x64 pixels: four tiles), each tile a chain of extents, LDS sums and a
// pass over its rectangle.  Here a thread has one pixel and adds its gradients
// to the texture itself, after those of pixels with the same texels were added
// up: in the wave's 8 x 8 pixels by halves (the lanes are in Morton order, and
// a step without equals costs one comparison), then the first lanes of the
// block's waves.  Bound by the latency of the loads and of 12 scattered atomics
// a lane; where the texture is magnified so far that waves share texels, by
// the atomics on those.
// 64x64 pixels and a 250x130 texture 18.6 us in tiles, 5.6 here (without
// adding up 5.3, but 123 where all of the image lies in four texels: 8 here,
// 10 in tiles); 40x40 and 1024^2 17.8 and 7.1, 181x140 18.2 and 9.7.
__global__ void __launch_bounds__(kSmallThreads) k_diff_backward_small(DiffArgs A, const float* __restrict__ gbuf,
                                                             const float* __restrict__ tex, const float* __restrict__ params,
                                                             const float* __restrict__ gout, float* __restrict__ gtex,
                                                             float* __restrict__ gparams, int blocks_x)
{
    __shared__ double sums[2][kSmallThreads / 64];
    __shared__ int first[kSmallThreads / 64];      // key and contributions of each wave's first lane
    __shared__ float firsts[kSmallThreads / 64][12];
    const int t = threadIdx.x;
    const int by = (int)blockIdx.x / blocks_x, bx = (int)blockIdx.x - by * blocks_x;
    // the lane's bits are those of x and y in turn: lanes 4, 16 and 64 of a
    // kind are squares of pixels
    const int x = bx * kSmallTile + (t >> 6 & 1) * 8 + ((t & 1) | (t >> 1 & 2) | (t >> 2 & 4));
    const int y = by * kSmallTile + (t >> 7) * 8 + ((t >> 1 & 1) | (t >> 2 & 2) | (t >> 3 & 4));
    double ga = 0.0, ge = 0.0;
    int key = -1;
    int64_t idx[4] = {0, 0, 0, 0};
    float c[12];
#pragma unroll
    for (int k = 0; k < 12; k++) c[k] = 0.0f;
    if (x < A.W && y < A.H) {
        const int64_t p = (int64_t)y * A.W + x;
        const float a = params[0], e = params[1];
        const Geo g = geometry(A, gbuf, p, e);
        if (g.covered) {
            float w[4];
            footprint(A, g.u, g.v, idx, w);
            key = (int)idx[0];
            const float go[3] = {gout[p * 3], gout[p * 3 + 1], gout[p * 3 + 2]};
            const float al = a * g.lam;
#pragma unroll
            for (int ch = 0; ch < 3; ch++) {
                const float s = ((w[0] * tex[idx[0] * 3 + ch] + w[1] * tex[idx[1] * 3 + ch]) + w[2] * tex[idx[2] * 3 + ch]) +
                                w[3] * tex[idx[3] * 3 + ch];
                ga += (double)(go[ch] * s * g.lam);
                const float gc = go[ch] * al;
#pragma unroll
                for (int k = 0; k < 4; k++) c[k * 3 + ch] = gc != 0.0f && w[k] != 0.0f ? gc * w[k] : 0.0f;
            }
            if (g.s > 0.0f) ge = (double)(((go[0] + go[1]) + go[2]) * g.spec * logf(g.s));
        }
    }
    merge_lanes<1>(key, c, t & 1);
    merge_lanes<2>(key, c, t & 2);
    merge_lanes<4>(key, c, t & 4);
    merge_lanes<8>(key, c, t & 8);
    merge_lanes<16>(key, c, t & 16);
    merge_lanes<32>(key, c, t & 32);
    if ((t & 63) == 0) {
        first[t >> 6] = key;
#pragma unroll
        for (int k = 0; k < 12; k++) firsts[t >> 6][k] = c[k];
    } else if (key >= 0) {
#pragma unroll
        for (int k = 0; k < 12; k++)
            if (c[k] != 0.0f) unsafeAtomicAdd(gtex + idx[k / 3] * 3 + k % 3, c[k]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ga += __shfl_xor(ga, o, 64);
        ge += __shfl_xor(ge, o, 64);
    }
    if ((t & 63) == 0) { sums[0][t >> 6] = ga; sums[1][t >> 6] = ge; }
    __syncthreads();
    if (t < 12) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kSmallThreads / 64; w++) {
            const int k = first[w];
            if (k < 0) continue;
            v += firsts[w][t];
            if (w + 1 < kSmallThreads / 64 && first[w + 1] == k) continue;
            int ix = k % A.tw, iy = k / A.tw;
            if ((t / 3 & 1) && ++ix == A.tw) ix = 0;
            if (t >= 6 && ++iy == A.th) iy = 0;
            if (v != 0.0f) unsafeAtomicAdd(gtex + ((int64_t)iy * A.tw + ix) * 3 + t % 3, v);
            v = 0.0f;
        }
    } else if (t >= 64 && t < 66) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kSmallThreads / 64; w++) s += sums[t - 64][w];
        unsafeAtomicAdd(gparams + t - 64, (float)s);
    }
}

int make_args(const psgpu_diff_desc* d, DiffArgs& A)
{
    if (!d || d->width < 1 || d->height < 1 || d->tex_w < 1 || d->tex_h < 1) return PSGPU_ERR_INVALID;
    A.W = d->width; A.H = d->height; A.tw = d->tex_w; A.th = d->tex_h;
    for (int k = 0; k < 3; k++) { A.light[k] = d->light[k]; A.camera[k] = d->camera[k]; }
    A.ks = d->ks;
    return PSGPU_OK;
}

}  // namespace

// These kernels keep no state of their own and touch only the buffers they
// are given; they run on the caller's stream (NULL is HIP's null stream).
extern "C" int psgpu_diff_forward(psgpu_ctx* ctx, const psgpu_diff_desc* desc, const float* gbuf, const float* tex,
                                  const float* params, float* out_rgb, void* stream)
{
    DiffArgs A;
    if (!ctx || !gbuf || !tex || !params || !out_rgb || make_args(desc, A)) return PSGPU_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    int64_t n = (int64_t)A.W * A.H;
    hipLaunchKernelGGL(k_diff_forward, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, A, gbuf, tex, params, out_rgb);
    return hipGetLastError() == hipSuccess ? PSGPU_OK : PSGPU_ERR_DEVICE;
}

extern "C" int psgpu_diff_backward(psgpu_ctx* ctx, const psgpu_diff_desc* desc, const float* gbuf, const float* tex,
                                   const float* params, const float* grad_out, float* grad_tex, float* grad_params,
                                   void* stream)
{
    DiffArgs A;
    if (!ctx || !gbuf || !tex || !params || !grad_out || !grad_tex || !grad_params || make_args(desc, A))
        return PSGPU_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    const int64_t pixels = (int64_t)A.W * A.H, texels = (int64_t)A.tw * A.th;
    if (pixels <= kSmallPixels && texels <= INT_MAX && pixels <= kSmallBeside + kSmallPerTexel * texels) {
        const int blocks_x = (A.W + kSmallTile - 1) / kSmallTile, blocks_y = (A.H + kSmallTile - 1) / kSmallTile;
        hipLaunchKernelGGL(k_diff_backward_small, dim3((unsigned)(blocks_x * blocks_y)), dim3(kSmallThreads), 0, s, A, gbuf, tex, params,
                           grad_out, grad_tex, grad_params, blocks_x);
        return hipGetLastError() == hipSuccess ? PSGPU_OK : PSGPU_ERR_DEVICE;
    }
    const int tiles_x = (int)(((int64_t)A.W + kTileW - 1) / kTileW);
    const int64_t n_tiles = tiles_x * (((int64_t)A.H + kTileH - 1) / kTileH);
    // two blocks a CU; one where every block adds to the whole of a small texture
    const int64_t most = whole_in_lds(A) ? 256 : 512;
    hipLaunchKernelGGL(k_diff_backward, dim3((unsigned)(n_tiles < most ? n_tiles : most)), dim3(kDiffThreads), 0, s, A, gbuf,
                       tex, params, grad_out, grad_tex, grad_params, tiles_x, n_tiles);
    return hipGetLastError() == hipSuccess ? PSGPU_OK : PSGPU_ERR_DEVICE;
}
