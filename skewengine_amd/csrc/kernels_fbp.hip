// kernels_fbp.hip -- standard parallel-beam geometry (no reference code; the
// counterpart of the reference's skew-space Radon, src/kernelRADN.h:212-259,
// in the 725-bin geometry of the benchmark configurations):
//
//   image   n x n on [-1,1]^2, pixel pitch delta = 2/n, row 0 at y = +1;
//   angles  theta_a (host table of cos/sin);
//   bins    s_k = (k - (ndet-1)/2) * delta.
//
//   project     p(a,k) = delta * sum_t f(s_k cos - t sin, s_k sin + t cos),
//               t on a delta grid of nt = ndet samples, f bilinear (zero
//               outside); the image is cut into tiles staged in LDS, each
//               tile's share of every ray summed there, the shares added in
//               tile order;
//   filter      q(a,k) = sum_k' p(a,k') h(k-k'), h = delta * Ram-Lak
//               (h0 = 1/(4 delta^2), odd m: -1/(m^2 pi^2 delta^2), even: 0) or
//               learned taps, as a GEMM with a Toeplitz matrix on the FP32
//               matrix cores;
//   backproject f(x,y) = (pi/nang) sum_a q(a, s(x,y)), linear in s.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "fbp.h"

namespace ske {

// Sample i of the ray of bin offset s at angle (c, sn) in pixel coordinates
// (u: column, v: row): with t = (i - half) delta,
// u = (s c - t sn + 1)/delta - 1/2 = U0 - i sn and
// v = (1 - s sn - t c)/delta - 1/2 = V0 - i c, so a sample costs two fma.
// Its bilinear base pixel is (floor v, floor u); it reads (v, u) .. (v+1,
// u+1), zero outside the image.  In exact arithmetic, with P = k - det_c,
// Q = half - i and m = n/2 - 1/2: u - m = P c + Q sn, v - m = -P sn + Q c.
struct RayCoord {
    float u0, v0;
};
// inv = 1 / delta (IEEE division)
__device__ __forceinline__ RayCoord ray_coord(const FbpGeom& g, float s, float c, float sn, float inv) {
    const float half = 0.5f * (float)(g.nt - 1);
    return RayCoord{((s * c + 1.0f) * inv - 0.5f) + half * sn, ((1.0f - s * sn) * inv - 0.5f) + half * c};
}

// The projector in LDS tiles.  A sample contributes only if one of its taps
// is an image pixel, i.e. its base pixel lies in [-1, n)^2; that square is
// cut into ntx x ntx tiles of side ts (ProjTiling).  A workgroup stages one
// tile of S slices, interleaved -- base pixels and their right/lower
// neighbours, (ts+1)^2 x S values, zero outside the image -- in LDS once, then
// for each angle of its chunk sums, per bin, the samples whose base pixel lies
// in the tile: every sample is counted in exactly one tile, with the position
// and bilinear weights the direct sampling gives.  The partial sums go to
// part[slice][angle][tile][k - klo]; k_fbp_project_sum adds each ray's
// partials in tile order.  Bins and samples a tile can hold are bounded with
// margins (tile_krange, sample_range) and every sample is tested exactly.
//
// The kernel is bound by VALU issue (23 of a sample's 30 instructions found
// its position and weights) and then by LDS: with S = 4 slices these serve
// four slices, and a slice adds four products and a quarter of four 16-byte
// reads.  16 x 512^2, 180 angles: 624 us with one slice per workgroup, 371 with
// four.  A single slice keeps larger tiles (fewer samples lost at tile
// edges: 79% of a pass are inside, 65% at the four-slice size); both fit LDS
// twice per CU, so that one workgroup stages while the other sums.
template <int S>
struct PtCfg {
    static constexpr int kMax = S == 1 ? kPtMax1 : kPtMax4;  // largest tile side
    // LDS row pitch (pixels), >= kMax + 1; S = 4: 4 modulo 16, so that the 4 x 4
    // base pixels of a read cycle's lanes fall on distinct banks
    static constexpr int kPitch = S == 1 ? 136 : 68;
    static constexpr int kUnroll = 4;                        // samples of a lane in flight
};
constexpr int kPtWaves = 8;
constexpr int kPtKB = 16;               // bins per work item (lanes of a pass along the bins)
constexpr int kPtIB = 64 / kPtKB;      // samples per pass along the ray
// Lane -> (bin, sample) of a pass.  A 16-byte LDS read serves the 4-lane blocks
// {0,3,5,6}, {1,2,4,7}, {8,11,13,14}, {9,10,12,15} in one cycle each, i.e.
// blocks b with equal b3 and equal parity of b2 b1 b0: the block's two low bits
// are the sample, b3 and the parity the upper bits of the bin, so that a cycle
// reads a compact patch of four bins x four samples.  Lanes of one bin differ
// by xor 20 and 24, those of one sample by xor 1, 2, 16, 32.
__device__ __forceinline__ int pt_bin(int lane) {
    const int b = lane >> 2;
    return (lane & 3) + 4 * ((b ^ (b >> 1) ^ (b >> 2)) & 1) + 8 * (b >> 3);
}
__device__ __forceinline__ int pt_sample(int lane) { return (lane >> 2) & 3; }

// Bins [klo, khi] whose rays can sample a base pixel of [x0, x1) x [y0, y1):
// P = (u - m) c - (v - m) sn over the corners, two bins of margin.
__device__ __forceinline__ void tile_krange(const FbpGeom& g, float c, float sn, int x0, int x1, int y0, int y1,
                                            int& klo, int& khi) {
    const float m = 0.5f * (float)g.n - 0.5f;
    const float ua = (float)x0 - m, ub = (float)x1 - m, va = (float)y0 - m, vb = (float)y1 - m;
    const float p0 = ua * c - va * sn, p1 = ub * c - va * sn, p2 = ua * c - vb * sn, p3 = ub * c - vb * sn;
    const float pmin = fminf(fminf(p0, p1), fminf(p2, p3)), pmax = fmaxf(fmaxf(p0, p1), fmaxf(p2, p3));
    klo = max((int)floorf(pmin + g.det_c) - 2, 0);
    khi = min((int)ceilf(pmax + g.det_c) + 2, g.ndet - 1);
}

// Samples [ilo, ihi] of bin offset P whose base pixel can lie in the tile:
// the line's chord through the tile's square widened by one pixel (Q from
// both slabs, rs = 1/sn and rc = 1/c rounded), two samples of margin; empty:
// ihi < ilo.
__device__ __forceinline__ void sample_range(const FbpGeom& g, float c, float sn, float rc, float rs, float P, int x0,
                                             int x1, int y0, int y1, int& ilo, int& ihi) {
    const float m = 0.5f * (float)g.n - 0.5f;
    const float X0 = (float)x0 - m - 1.0f, X1 = (float)x1 - m + 1.0f;
    const float Y0 = (float)y0 - m - 1.0f, Y1 = (float)y1 - m + 1.0f;
    float qlo = -1e30f, qhi = 1e30f;
    const float pc = P * c, ps = P * sn;
    if (fabsf(sn) > 1e-6f) {  // u - m = P c + Q sn in [X0, X1]
        const float q1 = (X0 - pc) * rs, q2 = (X1 - pc) * rs;
        qlo = fmaxf(qlo, fminf(q1, q2));
        qhi = fminf(qhi, fmaxf(q1, q2));
    } else if (pc < X0 || pc > X1) {
        qhi = qlo - 1.0f;
    }
    if (fabsf(c) > 1e-6f) {  // v - m = -P sn + Q c in [Y0, Y1]
        const float q1 = (Y0 + ps) * rc, q2 = (Y1 + ps) * rc;
        qlo = fmaxf(qlo, fminf(q1, q2));
        qhi = fminf(qhi, fmaxf(q1, q2));
    } else if (-ps < Y0 || -ps > Y1) {
        qhi = qlo - 1.0f;
    }
    ilo = 0;
    ihi = -1;
    if (qhi >= qlo) {
        const float half = 0.5f * (float)(g.nt - 1);
        ilo = max((int)floorf(half - qhi) - 2, 0);
        ihi = min((int)ceilf(half - qlo) + 2, g.nt - 1);
    }
}

// One workgroup per (tile, chunk of `chunk` angles, group of S slices).  Work
// items are (angle, block of kPtKB bins) of the chunk, taken by the waves in
// turn; lane (kb, ib) = (pt_bin, pt_sample) sums the samples ilo + ib,
// ilo + ib + kPtIB, ... of bin k0 + kb over the union of the block's sample
// ranges (a kPtKB x kPtIB block of (bin, sample) points a pass: a compact
// rotated patch of base pixels), kUnroll passes in flight; then the kPtIB
// lanes of a bin are added in a fixed butterfly order.
template <int S>
__global__ __launch_bounds__(64 * kPtWaves, 2) void k_fbp_project_tiles(const float* __restrict__ img,
                                                                              float* __restrict__ part,
                                                                              const float2* __restrict__ cs, FbpGeom g,
                                                                              ProjTiling pt, int chunk, int batch) {
    using F = PtCfg<S>;
    typedef float vec __attribute__((ext_vector_type(S)));
    // the tile, then two rows of zeros: what a sample outside the tile reads
    __shared__ __align__(16) float L[(F::kMax + 3) * F::kPitch * S];
    const int T = blockIdx.x, b0 = (int)blockIdx.z * S;
    const int x0 = -1 + (T % pt.ntx) * pt.ts, y0 = -1 + (T / pt.ntx) * pt.ts;
    const int x1 = min(x0 + pt.ts, g.n), y1 = min(y0 + pt.ts, g.n);  // base pixels [x0, x1) x [y0, y1)
    const int side = pt.ts + 1;
    for (int e = threadIdx.x; e < side * side; e += blockDim.x) {
        const int r = e / side, q = e - r * side;
        const int y = y0 + r, x = x0 + q;
        const bool in = y >= 0 && y < g.n && x >= 0 && x < g.n;
        vec v;
#pragma unroll
        for (int s = 0; s < S; s++)
            v[s] = (in && b0 + s < batch) ? img[((size_t)(b0 + s) * g.n + y) * g.n + x] : 0.0f;
        *(vec*)(L + (r * F::kPitch + q) * S) = v;
    }
    for (int e = threadIdx.x; e < 2 * F::kPitch * S; e += blockDim.x) L[(F::kMax + 1) * F::kPitch * S + e] = 0.0f;
    __syncthreads();
    const int lane = threadIdx.x & 63, kb = pt_bin(lane), ib = pt_sample(lane);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int a0 = blockIdx.y * chunk, na = min(chunk, g.nang - a0);
    const float inv = 1.0f / g.delta;
    // a base pixel (y, x) lies in the tile iff |x - xm| <= xh and |y - ym| <= yh (halves of integers: exact)
    const float xm = 0.5f * (float)(x0 + x1 - 1), xh = 0.5f * (float)(x1 - 1 - x0);
    const float ym = 0.5f * (float)(y0 + y1 - 1), yh = 0.5f * (float)(y1 - 1 - y0);
    // pixel (y, x) of the image at byte lt + (y * kPitch + x) * 4 S (below 2^24: exact in float)
    const float lt = -(float)((y0 * F::kPitch + x0) * 4 * S);
    constexpr int kZero = (F::kMax + 1) * F::kPitch * 4 * S;  // byte offset of the zeros
    int item = wave;  // flat index over (angle, bin block) pairs of the chunk
    int base = 0;     // items of the angles before aa
    for (int aa = 0; aa < na; ++aa) {
        const int a = a0 + aa;
        const float2 t2 = cs[a];
        const float c = t2.x, sn = t2.y;
        const float rc = 1.0f / c, rs = 1.0f / sn;  // used only where |c|, |sn| > 1e-6
        int klo, khi;
        tile_krange(g, c, sn, x0, x1, y0, y1, klo, khi);
        const int nkb = khi >= klo ? (khi - klo + kPtKB) / kPtKB : 0;
        for (; item < base + nkb; item += kPtWaves) {
            const int k = klo + kPtKB * (item - base) + kb;
            const bool kin = k <= khi;
            const float P = (float)k - g.det_c;
            int i0, i1;
            sample_range(g, c, sn, rc, rs, P, x0, x1, y0, y1, i0, i1);
            if (!kin) i1 = i0 - 1;
            int lo = i1 >= i0 ? i0 : INT_MAX, hi = i1 >= i0 ? i1 : INT_MIN;
#pragma unroll
            for (const int off : {1, 2, 16, 32}) {
                lo = min(lo, __shfl_xor(lo, off, 64));
                hi = max(hi, __shfl_xor(hi, off, 64));
            }
            const RayCoord ro = ray_coord(g, P * g.delta, c, sn, inv);
            vec acc;
#pragma unroll
            for (int s = 0; s < S; s++) acc[s] = 0.0f;
            // kU samples fi, fi + kPtIB, ...: branch-free, so that their reads
            // are in flight together; a sample outside the tile reads zeros
            auto samples = [&](auto ku_tag, float fi) {
                constexpr int kU = decltype(ku_tag)::value;
                vec ta[kU], tb[kU], tc[kU], td[kU];
                float wa[kU], wb[kU], wc[kU], wd[kU];
#pragma unroll
                for (int q = 0; q < kU; ++q) {
                    const float f = fi + (float)(kPtIB * q);
                    const float u = __builtin_fmaf(-f, sn, ro.u0), v = __builtin_fmaf(-f, c, ro.v0);
                    const float fu = floorf(u), fv = floorf(v);
                    const bool in = kin & (fabsf(fu - xm) <= xh) & (fabsf(fv - ym) <= yh);
                    const float at = __builtin_fmaf(fv, (float)(4 * S * F::kPitch), __builtin_fmaf(fu, (float)(4 * S), lt));
                    const char* r = (const char*)L + (in ? (int)at : kZero);
                    ta[q] = *(const vec*)r;
                    tb[q] = *(const vec*)(r + 4 * S);
                    tc[q] = *(const vec*)(r + F::kPitch * 4 * S);
                    td[q] = *(const vec*)(r + (F::kPitch + 1) * 4 * S);
                    const float wu = u - fu, wv = v - fv;
                    wd[q] = wu * wv;
                    wc[q] = wv - wd[q];
                    wb[q] = wu - wd[q];
                    wa[q] = (1.0f - wu) - wc[q];
                }
#pragma unroll
                for (int q = 0; q < kU; ++q)
#pragma unroll
                    for (int s = 0; s < S; s++)
                        acc[s] = __builtin_fmaf(
                            wa[q], ta[q][s],
                            __builtin_fmaf(wb[q], tb[q][s],
                                           __builtin_fmaf(wc[q], tc[q][s], __builtin_fmaf(wd[q], td[q][s], acc[s]))));
            };
            if (lo <= hi) {
                int i = lo + ib;
                float fi = (float)i;  // i, exactly (below 2^24)
                constexpr int kU = F::kUnroll;
                for (; i + (kU - 1) * kPtIB <= hi; i += kU * kPtIB, fi += (float)(kU * kPtIB))
                    samples(std::integral_constant<int, kU>(), fi);
                for (; i <= hi; i += kPtIB, fi += (float)kPtIB) samples(std::integral_constant<int, 1>(), fi);
            }
#pragma unroll
            for (int s = 0; s < S; s++) {
                float v = acc[s];
                v += __shfl_xor(v, 20, 64);
                v += __shfl_xor(v, 24, 64);
                if (ib == 0 && kin && b0 + s < batch)
                    part[(((size_t)(b0 + s) * g.nang + a) * pt.ntx * pt.ntx + T) * pt.kw + (k - klo)] = v;
            }
        }
        base += nkb;
    }
}

// sino(a, k) = delta * the sum of the partials of the tiles its ray crosses,
// in tile order.  One workgroup per (angle, slice): the tiles' bin ranges are
// found once, in LDS (each thread found them for its bin: half the time).
constexpr int kPtTilesMax = 1024;  // tiles whose ranges one pass keeps
__global__ __launch_bounds__(256) void k_fbp_project_sum(const float* __restrict__ part, float* __restrict__ sino,
                                                         const float2* __restrict__ cs, FbpGeom g, ProjTiling pt) {
    __shared__ int2 range[kPtTilesMax];
    const int a = blockIdx.x, b = blockIdx.y;
    const float2 t2 = cs[a];
    const int nt2 = pt.ntx * pt.ntx;
    const float* const p = part + ((size_t)b * g.nang + a) * nt2 * pt.kw;
    for (int k0 = 0; k0 < g.ndet; k0 += 1024) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int T0 = 0; T0 < nt2; T0 += kPtTilesMax) {
            __syncthreads();
            for (int T = T0 + (int)threadIdx.x; T < min(T0 + kPtTilesMax, nt2); T += 256) {
                const int x0 = -1 + (T % pt.ntx) * pt.ts, y0 = -1 + (T / pt.ntx) * pt.ts;
                int2 r;
                tile_krange(g, t2.x, t2.y, x0, min(x0 + pt.ts, g.n), y0, min(y0 + pt.ts, g.n), r.x, r.y);
                range[T - T0] = r;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int k = k0 + 256 * q + (int)threadIdx.x;
                if (k0 + 256 * q >= g.ndet) break;  // uniform
                const int n = min(kPtTilesMax, nt2 - T0);
                int T = 0;
                for (; T + 8 <= n; T += 8) {  // eight tiles' reads in flight, added in tile order
                    float v[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        const int2 r = range[T + u];
                        v[u] = 0.0f;
                        if (k >= r.x && k <= r.y) v[u] = p[(size_t)(T0 + T + u) * pt.kw + (k - r.x)];
                    }
#pragma unroll
                    for (int u = 0; u < 8; u++) acc[q] += v[u];
                }
                for (; T < n; ++T) {
                    const int2 r = range[T];
                    if (k >= r.x && k <= r.y) acc[q] += p[(size_t)(T0 + T) * pt.kw + (k - r.x)];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = k0 + 256 * q + (int)threadIdx.x;
            if (k < g.ndet) sino[((size_t)b * g.nang + a) * g.ndet + k] = acc[q] * g.delta;
        }
    }
}

// The filter as a GEMM on the matrix cores: Q = P T over the sinogram rows
// P (rows x ndet), with the Toeplitz T[k'][k] = h[k - k' + ndet - 1], in
// FP32 (v_mfma_f32_16x16x4_f32: fp32 products, fp32 accumulation).  A
// workgroup owns 16 rows and kFiltTiles 16-column output tiles; each of its
// waves keeps kFiltNB tiles in flight, so one A fragment feeds kFiltNB
// MFMAs.  K runs in chunks of up to kFiltKC: the chunk's 16 rows (zero past
// ndet and past the last row) and the window of taps its B fragments read
// (zero outside [0, 2 ndet - 1)) are staged in LDS.  Lane layout: A[i][k]
// at lane i + 16k, B[k][j] at lane j + 16k, D[i][j] at lane j + 16(i/4),
// register i%4.
typedef float f32x4 __attribute__((ext_vector_type(4)));
// B[k][j] of output tile u at step q is the tap 16 u - q past the wave's first,
// so B(u, q) = B(u - 1, q - 16): of the kFiltNB fragments of a step one is new,
// the others were read four steps (16 k) before.
constexpr int kFiltNB = 3;                    // output tiles per wave
constexpr int kFiltTiles = 4 * kFiltNB;       // output tiles per workgroup (4 waves)
constexpr int kFiltKC = 384;                  // K chunk (a multiple of 16)
// Row pitch of the staged rows: the 16 rows of an A fragment, two words apart,
// fall on distinct banks (a multiple of 32: all on one bank).
constexpr int kFiltPitch = kFiltKC + 2;
// Bound by the matrix cores at two to four workgroups per CU (27 KB of LDS,
// five fit): 192 columns a workgroup, so that 2,880 rows of 725 bins give 720
// workgroups for 256 CUs.  256 columns, five LDS reads for four MFMAs and a
// division per staged value: 58 us; now 36 (20 at the FP32 matrix rate);
// 3,840 rows 61 -> 48 us.
__global__ __launch_bounds__(256) void k_fbp_filter_mfma(const float* __restrict__ sino, float* __restrict__ filt,
                                                         const float* __restrict__ taps, int ndet, int rows) {
    __shared__ float P[16 * kFiltPitch];              // rows r0.., columns kc..kc+kFiltKC
    __shared__ float hw[kFiltTiles * 16 + kFiltKC];   // taps window of the chunk
    const int r0 = blockIdx.x * 16;
    const int c0 = blockIdx.y * kFiltTiles * 16;  // first output column of this workgroup
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, kk = lane >> 4;
    f32x4 acc[kFiltNB];
#pragma unroll
    for (int u = 0; u < kFiltNB; u++) acc[u] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    // the chunk's rows: thread t holds row t / 16, columns t % 16 + 16 e; the next
    // chunk's are loaded while this one's are multiplied
    constexpr int kE = kFiltKC / 16;
    float next[kE];
    const int lr = threadIdx.x >> 4, lc = threadIdx.x & 15;
    const float* src = sino + (size_t)(r0 + lr) * ndet;
    const int have = r0 + lr < rows ? ndet : 0;
    auto load = [&](int kc) {
#pragma unroll
        for (int e = 0; e < kE; e++) {
            const int k = kc + lc + 16 * e;
            next[e] = k < have ? src[k] : 0.0f;
        }
    };
    load(0);
    for (int kc = 0; kc < ndet; kc += kFiltKC) {
        const int kl = min(kFiltKC, (ndet - kc + 15) & ~15);
        __syncthreads();  // the previous chunk's reads are done
#pragma unroll
        for (int e = 0; e < kE; e++) P[lr * kFiltPitch + lc + 16 * e] = next[e];
        // column n = c0 + m (m < 16 kFiltTiles) at k' = kc + q (q < kl) needs
        // h[n - k' + ndet - 1], stored at hw[m - q + kl - 1]
        const int hbase = c0 + ndet - kc - kl;
        for (int y = threadIdx.x; y < kFiltTiles * 16 + kl; y += 256) {
            const int idx = hbase + y;
            hw[y] = (idx >= 0 && idx < 2 * ndet - 1) ? taps[idx] : 0.0f;
        }
        __syncthreads();
        if (kc + kFiltKC < ndet) load(kc + kFiltKC);
        if (c0 + 16 * kFiltNB * wave < ndet) {  // wave-uniform
            const float* pa = P + i * kFiltPitch + kk;
            const float* pb = hw + 16 * wave * kFiltNB + i - kk + kl - 1;
            float bf[4][kFiltNB];  // B(u, q) for q = 16 t + 4 v at bf[v][u]
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int u = 0; u < kFiltNB - 1; u++) bf[v][u] = pb[16 * (u + 1) - 4 * v];
            for (int q = 0; q < kl; q += 16) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int u = kFiltNB - 1; u > 0; u--) bf[v][u] = bf[v][u - 1];
                    bf[v][0] = pb[-q - 4 * v];
                    const float a = pa[q + 4 * v];
#pragma unroll
                    for (int u = 0; u < kFiltNB; u++)
                        acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bf[v][u], acc[u], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < kFiltNB; u++) {
        const int col = c0 + 16 * (wave * kFiltNB + u) + i;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = r0 + 4 * kk + r;
            if (row < rows && col < ndet) filt[(size_t)row * ndet + col] = acc[u][r];
        }
    }
}

// One thread per pixel, one workgroup per 16 x 16 pixel tile.  A tile
// projects onto at most 16*sqrt(2) + 2 < 25 consecutive bins of any angle,
// so per angle only a 32-bin window of the filtered row, starting at
// floor(projection of the tile centre) - 16, is staged in LDS (zeros outside
// the detector, which is what the bounds test of the linear interpolation
// gives); angles go in chunks of up to kBpChunk.
constexpr int kBpWin = 32;
constexpr int kBpChunk = 128;
__global__ __launch_bounds__(256) void k_fbp_backproject(const float* __restrict__ filt, float* __restrict__ img,
                                                         const float2* __restrict__ cs, FbpGeom g, float scale) {
    __shared__ float q[kBpChunk * kBpWin];
    __shared__ float2 csi[kBpChunk];  // (cos, sin) / delta of each angle of the chunk
    __shared__ int base[kBpChunk];    // window offset: aa * kBpWin - first bin of the window
    const int i0 = blockIdx.y * 16, j0 = blockIdx.x * 16;
    const int j = j0 + (threadIdx.x & 15);
    const int i = i0 + (threadIdx.x >> 4);
    const int b = blockIdx.z;
    const bool in = i < g.n && j < g.n;
    const float x = ((float)j + 0.5f) * g.delta - 1.0f;
    const float y = 1.0f - ((float)i + 0.5f) * g.delta;
    const float xc = ((float)j0 + 8.0f) * g.delta - 1.0f;
    const float yc = 1.0f - ((float)i0 + 8.0f) * g.delta;
    const float inv = 1.0f / g.delta;
    const float* fb = filt + (size_t)b * g.nang * g.ndet;
    float acc = 0.0f;
    for (int a0 = 0; a0 < g.nang; a0 += kBpChunk) {
        const int na = min(kBpChunk, g.nang - a0);
        __syncthreads();
        for (int t = threadIdx.x; t < na; t += blockDim.x) {
            const float2 t2 = cs[a0 + t];
            const float2 ci = make_float2(t2.x * inv, t2.y * inv);
            csi[t] = ci;
            // bin position of the tile centre, as the pixels compute theirs
            const float kc = __builtin_fmaf(xc, ci.x, __builtin_fmaf(yc, ci.y, g.det_c));
            base[t] = t * kBpWin - ((int)floorf(kc) - kBpWin / 2);
        }
        __syncthreads();
        for (int t = threadIdx.x; t < na * kBpWin; t += blockDim.x) {
            const int aa = t / kBpWin;
            const int k = (t % kBpWin) - (base[aa] - aa * kBpWin);
            q[t] = (k >= 0 && k < g.ndet) ? fb[(size_t)(a0 + aa) * g.ndet + k] : 0.0f;
        }
        __syncthreads();
        if (in) {
            for (int aa = 0; aa < na; ++aa) {
                const float2 ci = csi[aa];
                const float kf = __builtin_fmaf(x, ci.x, __builtin_fmaf(y, ci.y, g.det_c));
                const float fk = floorf(kf);
                const float w = kf - fk;
                const int r = (int)fk + base[aa];  // aa * kBpWin + [4, 28): the tile radius is < 12 bins
                const float v0 = q[r];
                const float v1 = q[r + 1];
                acc += __builtin_fmaf(w, v1 - v0, v0);
            }
        }
    }
    if (in) img[(size_t)b * g.n * g.n + (size_t)i * g.n + j] = acc * scale;
}

// Four slices at a time: one workgroup per tile of 32 x 8 PX pixels, a thread
// owns PX pixels (eight rows apart) of the four slices.  The windows (W bins)
// stand in LDS as pairs (q[k], q[k + 1] - q[k]); a pixel-angle's position,
// fraction and address serve the four slices, whose pairs are two 16-byte
// reads, and a slice adds one FMA lerp and an add.  The values and their order
// over the angles are k_fbp_backproject's, bit for bit.
// Lanes: a 16-byte read's cycle (pt_bin above) covers 4 x 4 pixels, whose bins
// lie within seven of each other: no bank conflicts at any angle.
// Angles go in chunks of CH, a wave staging every fourth angle; with kAhead
// the next chunk's windows are loaded into registers meanwhile.  Bound by LDS
// latency and VALU issue at four waves per SIMD.  16 slices of 512^2, 180
// angles: 192 -> 109 us; 64 slices, 60 angles: 279 -> 147 us.
template <int PX>
struct BpCfg {
    // >= 2 (half diagonal + 2): 15.5 and 4 PX - 0.5 pixels from the centre
    static constexpr int kW = PX == 4 ? 48 : 40;
    static constexpr bool kAhead = PX == 4;
    static constexpr int kChunk = kAhead ? 16 : 32;  // angles per staging
};
template <int PX>
__global__ __launch_bounds__(256) void k_fbp_backproject4(const float* __restrict__ filt, float* __restrict__ img,
                                                          const float2* __restrict__ cs, FbpGeom g, float scale,
                                                          int batch) {
    using F = BpCfg<PX>;
    constexpr int W = F::kW, CH = F::kChunk;
    __shared__ __align__(16) float q[2][CH * W * 4];  // slices 0, 1 and 2, 3 of a bin
    __shared__ __align__(16) float4 meta[CH];         // cos/delta, sin/delta, window offset aa * W - first bin (int bits)
    const int i0 = blockIdx.y * 8 * PX, j0 = blockIdx.x * 32;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int p16 = pt_bin(lane);  // the lane's 4 x 4 block (8, 4) and column in it (2, 1)
    const int j = j0 + 8 * wave + (p16 & 3) + 4 * (p16 >> 3);
    const int i = i0 + pt_sample(lane) + (p16 & 4);  // and i + 8, i + 16, ...
    const int b0 = (int)blockIdx.z * 4;
    const float x = ((float)j + 0.5f) * g.delta - 1.0f;
    float y[PX];
#pragma unroll
    for (int p = 0; p < PX; p++) y[p] = 1.0f - ((float)(i + 8 * p) + 0.5f) * g.delta;
    const float xc = ((float)j0 + 16.0f) * g.delta - 1.0f;
    const float yc = 1.0f - ((float)i0 + 4.0f * PX) * g.delta;
    const float inv = 1.0f / g.delta;
    float acc[PX][4];
#pragma unroll
    for (int p = 0; p < PX; p++)
#pragma unroll
        for (int s = 0; s < 4; s++) acc[p][s] = 0.0f;
    // lane order of the staging: slice fastest, so a bin's pairs are written side by side
    constexpr int kE = (W + 15) / 16, kA = 4;  // 16 bins a pass; four angles of a wave at a time
    const int ls = lane & 3, lw = lane >> 2;
    const bool in = b0 + ls < batch;
    float v0[kA][kE], v1[kA][kE];
    auto first_bin = [&](float cx, float cy) {
        // bin position of the tile centre, as the pixels compute theirs
        const float kc = __builtin_fmaf(xc, cx, __builtin_fmaf(yc, cy, g.det_c));
        return (int)floorf(kc) - W / 2;
    };
    auto load = [&](int a0) {  // angles a0 + wave, a0 + wave + 4, ...
#pragma unroll
        for (int c = 0; c < kA; c++) {
            const int a = a0 + wave + 4 * c;
            if (a >= g.nang) break;  // wave-uniform
            const float2 t2 = cs[a];
            const int k = first_bin(t2.x * inv, t2.y * inv) + lw;
            const float* row = filt + ((size_t)(b0 + ls) * g.nang + a) * g.ndet;
#pragma unroll
            for (int e = 0; e < kE; e++) {
                const int ke = k + 16 * e;
                v0[c][e] = (in && ke >= 0 && ke < g.ndet) ? row[ke] : 0.0f;
                v1[c][e] = (in && ke + 1 >= 0 && ke + 1 < g.ndet) ? row[ke + 1] : 0.0f;
            }
        }
    };
    auto store = [&](int a0, int t0, int na) {  // to the chunk's places t0 + wave, ...
#pragma unroll
        for (int c = 0; c < kA; c++) {
            const int aa = t0 + wave + 4 * c;
            if (aa >= na) break;  // wave-uniform
            if (lane == 0) {
                const float2 t2 = cs[a0 + aa];
                const float cx = t2.x * inv, cy = t2.y * inv;
                meta[aa] = make_float4(cx, cy, __int_as_float(aa * W - first_bin(cx, cy)), 0.0f);
            }
#pragma unroll
            for (int e = 0; e < kE; e++) {
                const int w = lw + 16 * e;
                if (W % 16 == 0 || w < W)
                    *(float2*)(q[ls >> 1] + (aa * W + w) * 4 + 2 * (ls & 1)) = make_float2(v0[c][e], v1[c][e] - v0[c][e]);
            }
        }
    };
    static_assert(!F::kAhead || CH == 4 * kA, "one load per chunk");
    if (F::kAhead) load(0);
    for (int a0 = 0; a0 < g.nang; a0 += CH) {
        const int na = min(CH, g.nang - a0);
        __syncthreads();
        if (F::kAhead) {
            store(a0, 0, na);
        } else {
            for (int t0 = 0; t0 < na; t0 += 4 * kA) {
                load(a0 + t0);
                store(a0, t0, na);
            }
        }
        __syncthreads();
        if (F::kAhead && a0 + CH < g.nang) load(a0 + CH);
#pragma unroll (PX == 4 ? 2 : 4)
        for (int aa = 0; aa < na; ++aa) {
            const float4 m = meta[aa];
#pragma unroll
            for (int p = 0; p < PX; p++) {
                const float kf = __builtin_fmaf(x, m.x, __builtin_fmaf(y[p], m.y, g.det_c));
                const float fk = floorf(kf);
                const float w = kf - fk;
                const int r = (int)fk + __float_as_int(m.z);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const f32x4 v = *(const f32x4*)(q[h] + r * 4);
                    acc[p][2 * h] += __builtin_fmaf(w, v[1], v[0]);
                    acc[p][2 * h + 1] += __builtin_fmaf(w, v[3], v[2]);
                }
            }
        }
    }
#pragma unroll
    for (int p = 0; p < PX; p++)
#pragma unroll
        for (int s = 0; s < 4; s++)
            if (i + 8 * p < g.n && j < g.n && b0 + s < batch)
                img[((size_t)(b0 + s) * g.n + i + 8 * p) * g.n + j] = acc[p][s] * scale;
}

// Angles per projector workgroup: at most kPtAngles (they share the tile's
// staging, which costs about as much as two of them), at least three, as few
// as give three workgroups per CU.
static int proj_chunk(const FbpGeom& g, const ProjTiling& pt, int groups) {
    const long long wgs = (long long)g.nang * pt.ntx * pt.ntx * groups;
    return (int)std::max(3LL, std::min((long long)kPtAngles, wgs / 768));
}

template <int S>
static hipError_t project_t(const float* img, float* part, float* sino, const float2* cs, const FbpGeom& g, int batch,
                            hipStream_t s) {
    const ProjTiling pt = proj_tiling(g.n, S);
    if (pt.ts < 1 || pt.ts > PtCfg<S>::kMax || pt.ntx * pt.ts < g.n + 1) return hipErrorInvalidValue;
    const int groups = (batch + S - 1) / S, chunk = proj_chunk(g, pt, groups);
    hipLaunchKernelGGL(k_fbp_project_tiles<S>,
                       dim3((unsigned)(pt.ntx * pt.ntx), (unsigned)((g.nang + chunk - 1) / chunk), (unsigned)groups),
                       dim3(64 * kPtWaves), 0, s, img, part, cs, g, pt, chunk, batch);
    hipLaunchKernelGGL(k_fbp_project_sum, dim3((unsigned)g.nang, (unsigned)batch), dim3(256), 0, s, part, sino, cs, g,
                       pt);
    return hipGetLastError();
}

// Four slices at a time, the last group with empty slices; where one group
// fills the card, a single last slice goes by itself (it takes 0.4 of a group).
// Batches whose partial sums do not fit `part` at once go through it in turn.
hipError_t launch_fbp_project(const float* img, float* part, size_t part_floats, float* sino, const float2* cs,
                              const FbpGeom& g, int batch, hipStream_t s) {
    const ProjTiling pt = proj_tiling(g.n, 4);
    const bool fills = (long long)pt.ntx * pt.ntx * ((g.nang + kPtAngles - 1) / kPtAngles) >= 512;
    const int fit = (int)std::min((size_t)batch, part_floats / proj_part_floats(g.n, g.nang, 1, 4));
    int four = batch == 1 ? 0 : (batch % 4 == 1 && fills) ? batch - 1 : batch;
    if (fit < std::min(four, 4)) four = 0;
    const int step = fit >= four ? std::max(four, 1) : fit & ~3;
    for (int b = 0; b < four; b += step) {
        const hipError_t e = project_t<4>(img + (size_t)b * g.n * g.n, part, sino + (size_t)b * g.nang * g.ndet, cs, g,
                                          std::min(step, four - b), s);
        if (e != hipSuccess) return e;
    }
    if (four == batch) return hipSuccess;
    return project_t<1>(img + (size_t)four * g.n * g.n, part, sino + (size_t)four * g.nang * g.ndet, cs, g,
                        batch - four, s);
}

hipError_t launch_fbp_filter(const float* sino, float* filt, const float* taps, const FbpGeom& g, int batch,
                             hipStream_t s) {
    const int rows = batch * g.nang;
    const dim3 grid((unsigned)((rows + 15) / 16), (unsigned)((g.ndet + 16 * kFiltTiles - 1) / (16 * kFiltTiles)));
    hipLaunchKernelGGL(k_fbp_filter_mfma, grid, dim3(256), 0, s, sino, filt, taps, g.ndet, rows);
    return hipGetLastError();
}

// Four slices at a time where that leaves at least three workgroups per CU
// (four pixels a thread), or eight (one pixel); otherwise, and for a remainder
// of one or two slices, a slice at a time (136^2, 13 slices, 324 angles: 39 us
// against 67 by fours).
hipError_t launch_fbp_backproject(const float* filt, float* img, const float2* cs, const FbpGeom& g, int batch,
                                  float scale, hipStream_t s) {
    int four = batch % 4 == 3 ? batch : batch - batch % 4;
    const unsigned t32 = (unsigned)(g.n + 31) / 32, t8 = (unsigned)(g.n + 7) / 8, t16 = (unsigned)(g.n + 15) / 16;
    const unsigned groups = (unsigned)(four + 3) / 4;
    if ((size_t)t32 * t32 * groups >= 768)
        hipLaunchKernelGGL(k_fbp_backproject4<4>, dim3(t32, t32, groups), dim3(256), 0, s, filt, img, cs, g, scale,
                           four);
    else if ((size_t)t32 * t8 * groups >= 2048)
        hipLaunchKernelGGL(k_fbp_backproject4<1>, dim3(t32, t8, groups), dim3(256), 0, s, filt, img, cs, g, scale,
                           four);
    else
        four = 0;
    if (four < batch)
        hipLaunchKernelGGL(k_fbp_backproject, dim3(t16, t16, (unsigned)(batch - four)), dim3(256), 0, s,
                           filt + (size_t)four * g.nang * g.ndet, img + (size_t)four * g.n * g.n, cs, g, scale);
    return hipGetLastError();
}

}  // namespace ske
