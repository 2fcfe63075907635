// kernels_blur.hip -- cepstral blur operator (src/kernelBLUR.h:267-302,
// lineCepstrum :153-228, select_subarray :69-85, getBlurParameter2 :88-110)
// on gfx950, FP64 throughout like the reference.
//
// Per skewed cell j of row r the reference takes the 64-sample window
// S(r, j-32 .. j+31) (zero outside [first,last)), X = DFT64/8, the log power
// of bins 0..31, C = DFT32/sqrt(32) of those logs, v_k = -min(0, Re C_k) for
// k < 16 and a peak rule on v, times 1e4.
//
// Layout: one wave per skewed row; the row is staged in LDS with 64 zeros of
// guard band on each side (which is exactly the window's zero fill).  Lane l
// owns a contiguous segment of cells.  It computes the 32 needed bins of the
// segment's first window and then slides the window one cell at a
// time: X_k(j+1) = e^{+2 pi i k/64} (X_k(j) + (x[j+32] - x[j-32])/8).  A
// segment is at most 16 cells, so rounding drift stays at the 1e-15 level.
// Re C_k is the cosine sum of the real log spectrum L_n, which is what the
// reference's complex DFT of a real input yields in its real part.  The peak
// rule reads k = 4 .. 15 only, and cos(2 pi k n/32) is the same for n and
// 32 - n, so the sums run over E_n = L_n + L_{32-n}, taken as one logarithm of
// the product of two powers, and over F_n = E_n + E_{16-n} for even k, G_n =
// E_n - E_{16-n} for odd k (even k once more by 8): 17 logarithms and about 90
// operations a cell instead of 32 and 384.
#include "device_common.h"
#include "launch.h"

namespace ske {

// Natural log of a double: x = m 2^e with m in [1, 2); the top 8 fraction
// bits i of m pick c_i ~ 1/(1 + (i + 1/2)/256) from the table (doubled in LDS,
// for m/2), so that u = m c_i - 1 (one fma) has |u| < 2^-9, and
//     log x = e ln2 + (-log c_i) + log1p(u),
//     log1p(u) = u - u^2/2 + u^3/3 - u^4/4 + u^5/5   (the rest < 2^-55).
// -log c_i and ln 2 (as a double-double) come from the host in extended
// precision.  x = 0 gives -inf like the libm log.  `lt` = the table in LDS.
__device__ __forceinline__ double fast_log(double x, const double* lt) {
    const double mant = __builtin_amdgcn_frexp_mant(x);  // [0.5, 1)
    const int ex = __builtin_amdgcn_frexp_exp(x) - 1;
    const int i = (int)((uint32_t)(__double_as_longlong(mant) >> 44) & 0xFFu);
    const double c = lt[2 * i], t = lt[2 * i + 1];
    const double u = __builtin_fma(mant, c, -1.0);
    const double q = __builtin_fma(u, __builtin_fma(u, __builtin_fma(u, 0.2, -0.25), 1.0 / 3.0), -0.5);
    const double p = __builtin_fma(u * u, q, u);
    const double e = (double)ex;
    const double r = __builtin_fma(e, lt[513], t + p);
    const double y = __builtin_fma(e, lt[512], r);
    return x == 0.0 ? -INFINITY : y;
}

// tab layout (double): [0,128): cos/sin(2 pi t/64) interleaved; [128,160): cos(2 pi t/32);
// from kLogTab the log table of fast_log.
__global__ __launch_bounds__(64) void k_op_blur(const SecDesc* __restrict__ secs, const RowWork* __restrict__ work,
                                                const float* __restrict__ in4, const int* __restrict__ target,
                                                const float* __restrict__ weight, const uint32_t* __restrict__ fl,
                                                const float* __restrict__ Sbuf, const double* __restrict__ tab,
                                                float* __restrict__ arena, int p_maxL) {
    extern __shared__ float lds[];
    float* row = lds + kPad;
    double* lt = reinterpret_cast<double*>(lds) + ((size_t)(p_maxL + 2 * kPad) + 1) / 2;  // after the row
    double* tws = lt + 514;  // cos, sin of 2 pi k/64, k < 32
    for (int t = threadIdx.x; t < 514; t += 64) {
        const double x = tab[kLogTab + t];
        lt[t] = t < 512 && !(t & 1) ? 2.0 * x : x;  // 2 c_i, T_i, ln 2
    }
    tws[threadIdx.x] = tab[threadIdx.x];
    const RowWork w = work[blockIdx.x];
    const SecDesc sd = secs[w.sec];
    const int r = w.row;
    const uint32_t v = fl[sd.rows + r];
    const int f = fl_first(v);
    const int L = fl_last(v) - f;
    if (L <= 0) return;
    stage_row(row, sd, r, f, L, in4, target, weight, Sbuf);
    __syncthreads();

    const int lane = threadIdx.x;
    const int seg = (L + 63) >> 6;
    const int c0 = lane * seg;
    const int c1 = min(c0 + seg, L);
    if (c0 >= c1) return;
    float* so = arena + sd.so + (size_t)r * sd.dim_i + f;

    // cos(pi t/16), t = 1 .. 7
    const double c16[9] = {1.0, tab[129], tab[130], tab[131], tab[132], tab[133], tab[134], tab[135], 0.0};
    // The first window's bins 0 .. 31: z_m = x_{2m} + i x_{2m+1}, a 32-point DFT
    // of z by five radix-2 stages in registers (Z_k at the bit-reversed place
    // of k), then X_k = (Z_k + Z*_{32-k})/2 - i e^{-2 pi i k/64} (Z_k - Z*_{32-k})/2.
    double Xr[32], Xi[32];
    {
        double zr[32], zi[32];
        // 1/8 of the transform and 1/2 of the split
#pragma unroll
        for (int m = 0; m < 32; ++m) {
            zr[m] = (double)row[c0 - 32 + 2 * m] * 0.0625;
            zi[m] = (double)row[c0 - 31 + 2 * m] * 0.0625;
        }
#pragma unroll
        for (int st = 0; st < 5; ++st) {
            const int len = 32 >> st, half = len >> 1;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int l = q & (half - 1), a = (q - l) * 2 + l, b = a + half, t = l << st;  // twiddle e^{-2 pi i t/32}
                const double ur = zr[a] - zr[b], ui = zi[a] - zi[b];
                zr[a] += zr[b];
                zi[a] += zi[b];
                if (t == 0) {
                    zr[b] = ur;
                    zi[b] = ui;
                } else if (t == 8) {  // -i
                    zr[b] = ui;
                    zi[b] = -ur;
                } else {
                    const double cr = t < 8 ? c16[t] : -c16[16 - t], sr = t < 8 ? c16[8 - t] : c16[t - 8];
                    zr[b] = __builtin_fma(ur, cr, ui * sr);
                    zi[b] = __builtin_fma(ui, cr, -(ur * sr));
                }
            }
        }
        auto rev = [](int k) { return (k & 1) << 4 | (k & 2) << 2 | (k & 4) | (k & 8) >> 2 | (k & 16) >> 4; };
        Xr[0] = 2.0 * (zr[0] + zi[0]);
        Xi[0] = 0.0;
        Xr[16] = 2.0 * zr[rev(16)];
        Xi[16] = -2.0 * zi[rev(16)];
#pragma unroll
        for (int k = 1; k < 16; ++k) {
            const int p = rev(k), q = rev(32 - k);
            const double er = zr[p] + zr[q], ei = zi[p] - zi[q];  // Z_k + Z*_{32-k}
            const double fr = zr[p] - zr[q], fi = zi[p] + zi[q];  // Z_k - Z*_{32-k}
            const double cr = tws[2 * k], sr = tws[2 * k + 1];
            // -i (cr - i sr)(fr + i fi) = (fi cr - fr sr) - i (fr cr + fi sr)
            const double gr = __builtin_fma(fi, cr, -(fr * sr)), gi = __builtin_fma(fr, cr, fi * sr);
            Xr[k] = er + gr;
            Xi[k] = ei - gi;
            Xr[32 - k] = er - gr;  // the same pair conjugated, e^{-2 pi i (32-k)/64} = -(cr + i sr)
            Xi[32 - k] = -ei - gi;
        }
    }
    const double inv_sqrt32 = 0.17677669529663687;  // 1/sqrt(32)
    for (int c = c0; c < c1; ++c) {
        asm volatile("" ::: "memory");  // the twiddles are read in every pass (as registers they would spill)
        // one cell on (past the last cell the row's guard band)
        const double delta = ((double)row[c + 32] - (double)row[c - 32]) * 0.125;
        // power of bin k of this window, then the bin of the next one
        auto power = [&](int k) {
            const double p = Xr[k] * Xr[k] + Xi[k] * Xi[k];
            const double cr = tws[2 * k], sr = tws[2 * k + 1];
            const double a = Xr[k] + delta, b = Xi[k];
            Xr[k] = __builtin_fma(a, cr, -(b * sr));
            Xi[k] = __builtin_fma(a, sr, b * cr);
            return p;
        };
        const double p0 = Xr[0] * Xr[0];
        Xr[0] += delta;  // bin 0 is real and does not turn
        const double l0 = fast_log(p0, lt), l16 = fast_log(power(16), lt);
        const double e8 = fast_log(power(8) * power(24), lt);
        double F[8];                                         // F_1 .. F_7
        double o5 = 0, o7 = 0, o9 = 0, o11 = 0, o13 = 0, o15 = 0;  // sums over G_n = E_n - E_{16-n}, k odd
        auto odd = [&](int n, double g) {
            // cos(pi k n/16) = +-cos(pi m/16), m = 0 .. 8, by the quadrant of k n mod 32
            auto term = [&](int k, double& o) {
                const int m = (k * n) & 31, q = m > 16 ? 32 - m : m, r = q > 8 ? 16 - q : q;
                if (r < 8) o = __builtin_fma(q > 8 ? -g : g, c16[r], o);
            };
            term(5, o5);
            term(7, o7);
            term(9, o9);
            term(11, o11);
            term(13, o13);
            term(15, o15);
        };
#pragma unroll
        for (int n = 1; n < 8; ++n) {
            const double e = fast_log(power(n) * power(32 - n), lt);        // E_n
            const double e2 = fast_log(power(16 - n) * power(16 + n), lt);  // E_{16-n}
            F[n] = e + e2;
            odd(n, e - e2);
        }
        const double h1 = F[1] + F[7], h2 = F[2] + F[6], h3 = F[3] + F[5];
        const double j1 = F[1] - F[7], j2 = F[2] - F[6], j3 = F[3] - F[5];
        const double s = l0 + l16, d = l0 - l16, A = s + e8, B = s - e8;
        const double A4 = A - F[4], h13 = h1 - h3;
        const double B1 = __builtin_fma(-c16[4], j2, B), B2 = __builtin_fma(c16[4], j2, B);
        const double j6 = __builtin_fma(c16[6], j1, -(c16[2] * j3)), j14 = __builtin_fma(c16[2], j1, c16[6] * j3);
        double vv[16];
        vv[4] = __builtin_fma(c16[4], h13, A4);
        vv[5] = d + o5;
        vv[6] = B1 + j6;
        vv[7] = d + o7;
        vv[8] = (A + F[4]) - h2;
        vv[9] = d + o9;
        vv[10] = B1 - j6;
        vv[11] = d + o11;
        vv[12] = __builtin_fma(-c16[4], h13, A4);
        vv[13] = d + o13;
        vv[14] = B2 - j14;
        vv[15] = d + o15;
#pragma unroll
        for (int k = 4; k < 16; ++k) vv[k] = fmax(-(vv[k] * inv_sqrt32), 0.0);  // -std::min(0.0, C)
        // getBlurParameter2(v, 16): first i >= 5 with v[i] > v[i-1]; the
        // value is max(v[i-1], v[i+1..15]) (v[i] itself is skipped).
        double V = 0.0, top = 0.0;  // top = max(v[i+1..15], 0): v >= 0
#pragma unroll
        for (int i = 15; i >= 5; --i) {
            V = vv[i] > vv[i - 1] ? fmax(vv[i - 1], top) : V;
            top = fmax(top, vv[i]);
        }
        so[c] = (float)(V * 10000);
    }
}

hipError_t launch_op_blur(const DevPlan& p, const float* in4, const float* Sbuf, float* arena, const double* tab,
                          hipStream_t s) {
    if (p.nwork == 0) return hipSuccess;
    const size_t row_floats = ((size_t)(p.maxL + 2 * kPad) + 1) / 2 * 2;  // keep the log table 8-byte aligned
    const size_t lds = sizeof(float) * row_floats + sizeof(double) * (514 + 64);
    hipLaunchKernelGGL(k_op_blur, dim3(p.nwork), dim3(64), lds, s, p.secs, p.work, in4, p.target, p.weight, p.fl,
                       Sbuf, tab, arena, p.maxL);
    return hipGetLastError();
}

}  // namespace ske
