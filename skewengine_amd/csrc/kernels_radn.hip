// kernels_radn.hip -- Radon operator (src/kernelRADN.h:212-258) on gfx950:
// the global transform (LRT=false) and the local one (LRT=true, pointRadon
// :114-182).
//
//   rowsum : P_r = sum_j S(r,j) of every skewed row in double (the
//            reference sums in double too, kernelRADN.h:227-232).
//   filter : one workgroup per sector.  P is zero-padded to H2 = 2^ceil(log2 H)
//            in LDS and filtered with the reference's own transform: the
//            radix-2 decimation-in-frequency FFT of src/helper.h:59-106 with
//            its twiddles (repeated complex products, precomputed on the host
//            by the same recurrence), the one-sided ramp k/H for k <= H/2
//            (kernelRADN.h:247), and ifft = conj o fft o conj / H2
//            (helper.h:108-114).  Butterflies of one stage are independent,
//            so the parallel stage computes exactly the reference's values.
//   The smear back (kernelRADN.h:252-257) is folded into the deskew, which
//   reads q_r for every cell of row r in [first, last).
#include <limits.h>

#include "device_common.h"
#include "launch.h"

namespace ske {

// The rows of a materialised skewInput (the per-sector calls).
__global__ __launch_bounds__(256) void k_radn_rowsum(const SecDesc* __restrict__ secs,
                                                     const RowWork* __restrict__ work, int nwork,
                                                     const uint32_t* __restrict__ fl,
                                                     const float* __restrict__ Sbuf, double* __restrict__ P) {
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= nwork) return;
    const int lane = threadIdx.x & 63;
    const RowWork w = work[item];
    const SecDesc sd = secs[w.sec];
    const uint32_t v = fl[sd.rows + w.row];
    const int f = fl_first(v), l = fl_last(v);
    double acc = 0.0;
    for (int j = f + lane; j < l; j += 64) acc += (double)Sbuf[(size_t)w.row * sd.dim_i + j];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) P[sd.q + w.row] = acc;
}

// The fused row sums (no materialised skewInput): one wave per 63
// consecutive skewed rows of one sector, lane = row (lane 0 the row before).  Each lane adds
// S(r, j) over its own [first, last) in ascending j in double -- the
// reference's own order (kernelRADN.h:227-232), so P is the reference's sum
// bit for bit -- with S(r, j) computed as skew_cell does.  The two taps of
// cell (r, j) lie in column j of the oriented copy, rows r - t_j - 1 and
// r - t_j; a column of one oriented copy is a row of another (the partner,
// read backwards for types 0 and 3):
//   type 0: in0[a][j] = in2[j][dimy-1-a]        type 1: in1[a][j] = in3[dimy-1-j][a]
//   type 2: in2[a][j] = in0[dimy-1-j][a]        type 3: in3[a][j] = in2[dimx-1-j][dimy-1-a]
// so at every j the 64 lanes' taps are 64 consecutive floats of one row and
// t_j, w_j are wave-uniform (scalar loads).  A lane loads the tap of row r - t_j
// and takes that of row r - t_j - 1 from the lane before, whose row is r - 1.
// The tap's byte offset is A + B j + C t_j + D: three sector constants and a
// per-lane term.  The wave walks the union of its rows' ranges; cells
// outside a lane's own range are read but add zero (acc + 0 = acc: acc is
// never -0).
constexpr int kColsUnroll = 8;
// Columns [j0, j1) of the walk, adding to acc.  Unless kInner (every lane inside
// its range and both taps inside the image) the lane's own [f, l) and the taps'
// rows are tested.  The
// first tap's value is w * x1 without the reference's 0 + (it differs only
// in the sign of a zero, which no later sum can see: acc is never -0).
template <bool kInner>
__device__ __forceinline__ void rowsum_cols_span(const int* __restrict__ tt, const float* __restrict__ ww,
                                                 __amdgpu_buffer_rsrc_t src, int A, int B, int C, int D, int r,
                                                 int dim_o, int f, int l, int j0, int j1, double& acc) {
    auto cell = [&](int j, int t, float w, unsigned tap) -> float {
        // row r - t, and from the lane before row r - 1 - t
        const float x0 = __uint_as_float(tap);
        const float x1 = __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)tap, 0x138, 0xf, 0xf, true));
        if (kInner) return w * x1 + (1.0f - w) * x0;
        const int i0 = r - t;
        const float s = ((unsigned)(i0 - 1) < (unsigned)dim_o) ? w * x1 : 0.0f;
        const float v = ((unsigned)i0 < (unsigned)dim_o) ? s + (1.0f - w) * x0 : s;
        return (unsigned)(j - f) < (unsigned)(l - f) ? v : 0.0f;
    };
    auto load = [&](int j, int t) -> unsigned {
        return __builtin_amdgcn_raw_buffer_load_b32(src, A + B * j + C * t + D, 0, 0);
    };
    int j = j0;
    for (; j + kColsUnroll <= j1; j += kColsUnroll) {
        int t[kColsUnroll];
        float w[kColsUnroll];
        unsigned pr[kColsUnroll];
#pragma unroll
        for (int u = 0; u < kColsUnroll; ++u) {
            t[u] = tt[j + u];
            w[u] = ww[j + u];
        }
#pragma unroll
        for (int u = 0; u < kColsUnroll; ++u) pr[u] = load(j + u, t[u]);
#pragma unroll
        for (int u = 0; u < kColsUnroll; ++u) acc += (double)cell(j + u, t[u], w[u], pr[u]);
    }
    for (; j < j1; ++j) {
        const int t = tt[j];
        acc += (double)cell(j, t, ww[j], load(j, t));
    }
}

// The walk over [lo, hi): columns [ia, ib) without tests.
__device__ __forceinline__ double rowsum_cols_walk(const int* __restrict__ tt, const float* __restrict__ ww,
                                                   __amdgpu_buffer_rsrc_t src, int A, int B, int C, int D, int r,
                                                   int dim_o, int f, int l, int lo, int hi, int ia, int ib) {
    double acc = 0.0;
    if (ia < ib) {
        rowsum_cols_span<false>(tt, ww, src, A, B, C, D, r, dim_o, f, l, lo, ia, acc);
        rowsum_cols_span<true>(tt, ww, src, A, B, C, D, r, dim_o, f, l, ia, ib, acc);
        rowsum_cols_span<false>(tt, ww, src, A, B, C, D, r, dim_o, f, l, ib, hi, acc);
    } else {
        rowsum_cols_span<false>(tt, ww, src, A, B, C, D, r, dim_o, f, l, lo, hi, acc);
    }
    return acc;
}

//
// Bound by VALU (about 18 operations a column with the tests, 9 without) and by
// L2 misses: the 64 lanes' taps are one partner row, and a miss in any of a
// pass's eight rows stalls the wave.  Workgroups go to the eight XCDs
// in turn, so runs of up to 23 sectors (an image's 180 over all eight; nearly
// always one partner copy) are laid on one XCD, whose L2 then serves them: 8 x
// 955^2 passes 1,498 -> 855 us.  A run is as long as gives every XCD one: with 23
// always, a share of 23 sectors ran on one XCD (1600^2: 199 us, now 114; 46
// sectors 208 and 126; without runs 130 and 128).  A workgroup is one wave: rows of a sector differ in
// length by up to 8 times, and waves that share a workgroup leave their slots
// to the next one only together.  16 x 512^2: 500 -> 387 us for both; columns
// without tests and one load a tap: 387 -> 323 (one 512^2 image 53 -> 43).  Not
// faster: scalar offsets with two or three taps per load (unaligned wide
// loads), passes in flight from tables held in lanes (540 to 670 us), 32
// columns a pass for a single image (59).
constexpr int kXcdSectors = 23, kRowsumWaves = 1, kRowsumRows = 63;
__global__ __launch_bounds__(64 * kRowsumWaves) void k_radn_rowsum_cols(const SecDesc* __restrict__ secs,
                                                          const float* __restrict__ in4,
                                                          const int* __restrict__ target,
                                                          const float* __restrict__ weight,
                                                          const uint32_t* __restrict__ fl, double* __restrict__ P,
                                                          int nsec, int nblk, int run) {
    const int at = blockIdx.x >> 3, k = at / nblk;
    const int si = (k / run * 8 + (int)(blockIdx.x & 7)) * run + k % run;
    if (si >= nsec) return;
    const SecDesc sd = secs[si];
    const int r0 = ((at - k * nblk) * kRowsumWaves + (threadIdx.x >> 6)) * kRowsumRows;
    if (r0 >= sd.H) return;  // wave-uniform
    const int lane = threadIdx.x & 63;
    const int r = r0 + lane - 1;  // lane 0 only loads its tap for lane 1
    const bool live = lane > 0 && r < sd.H;
    int f = 0, l = 0;
    if (live) {
        const uint32_t v = fl[sd.rows + r];
        f = fl_first(v);
        l = fl_last(v);
    }
    if (!(live && l > f)) f = l = 0;  // no cell of this lane is added
    int lo = l > f ? f : INT_MAX, hi = l > f ? l : INT_MIN;
    // [fmax, lmin): inside every lane's range (empty when some lane has none)
    int fmax = l > f ? f : lane == 0 ? INT_MIN : INT_MAX, lmin = l > f ? l : lane == 0 ? INT_MAX : INT_MIN;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        lo = min(lo, __shfl_xor(lo, off, 64));
        hi = max(hi, __shfl_xor(hi, off, 64));
        fmax = max(fmax, __shfl_xor(fmax, off, 64));
        lmin = min(lmin, __shfl_xor(lmin, off, 64));
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    fmax = __builtin_amdgcn_readfirstlane(fmax);
    lmin = __builtin_amdgcn_readfirstlane(lmin);
    // Both taps of a row r in the image: r - dim_o < t_j < r.  Column j is in the
    // range of row x only if x - dim_o <= t_j <= x, so the columns from the row
    // after the wave's last on, and up to the row before its first, have that.
    int ia = hi, ib = hi;
    if (r0 > 0 && r0 + kRowsumRows < sd.H && lo < hi) {
        ia = max(fmax, __builtin_amdgcn_readfirstlane((int)fl_first(fl[sd.rows + r0 + kRowsumRows])));
        ib = min(lmin, __builtin_amdgcn_readfirstlane((int)fl_last(fl[sd.rows + r0 - 1])));
    }
    const int dim_o = sd.dim_o, dim_i = sd.dim_i, type = sd.type;
    const int partner = type == 0 ? 2 : type == 1 ? 3 : type == 2 ? 0 : 2;
    // the partner copy as a raw buffer of N floats: a tap outside it (a row
    // index outside the image, whose cell is masked anyway) reads zero
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(in4 + sd.img + (size_t)partner * sd.N), 0, sd.N * 4, kBufferRsrcWord3);
    const int* const tt = target + sd.tab;
    const float* const ww = weight + sd.tab;
    // byte offset of tap r - t of column j, row r: A + B j + C t + D r
    //   type 0: partner row j, position dim_o-1-(r-t)     type 3: partner row dim_i-1-j, the same position
    //   types 1, 2: partner row dim_i-1-j, position r-t
    const int D = type == 0 || type == 3 ? -4 : 4;
    const int A = 4 * ((type == 0 ? 0 : (dim_i - 1) * dim_o) + (D < 0 ? dim_o - 1 : 0));
    const double acc = rowsum_cols_walk(tt, ww, src, A, type == 0 ? 4 * dim_o : -4 * dim_o, -D, D * r, r, dim_o, f, l,
                                        lo, hi, ia, ib);
    if (live) P[sd.q + r] = acc;
}

hipError_t launch_radn_rowsum(const DevPlan& p, const float* in4, const float* Sbuf, double* P, hipStream_t s) {
    if (!Sbuf) {  // writes every row r < H of every sector (rows without cells: 0)
        if (p.nsec == 0 || p.maxH <= 0) return hipSuccess;
        const int nblk = (p.maxH + kRowsumRows * kRowsumWaves - 1) / (kRowsumRows * kRowsumWaves);
        const int rounds = (p.nsec + 8 * kXcdSectors - 1) / (8 * kXcdSectors), run = (p.nsec + 8 * rounds - 1) / (8 * rounds);
        hipLaunchKernelGGL(k_radn_rowsum_cols, dim3(8u * run * rounds * nblk), dim3(64 * kRowsumWaves), 0, s, p.secs,
                           in4, p.target, p.weight, p.fl, P, p.nsec, nblk, run);
        return hipGetLastError();
    }
    if (p.nwork == 0) return hipSuccess;  // writes the rows of the work list only: P zeroed by the caller
    hipLaunchKernelGGL(k_radn_rowsum, dim3((p.nwork + 3) / 4), dim3(256), 0, s, p.secs, p.work, p.nwork, p.fl, Sbuf, P);
    return hipGetLastError();
}

// The DIF stages of a transform over re/im in LDS (src/helper.h:65-82), two a
// pass: a thread takes the four points l, l + n/4, l + n/2, l + 3n/4 of a block
// of n through the stages n and n/2 in registers (the same butterflies and
// twiddles, half the LDS passes and barriers).  The result stands in
// bit-reversed order; the caller reads it there.  kPad: one double of padding
// per 16, which spreads the power-of-two strides over the banks.
template <bool kPad>
__device__ __forceinline__ int fft_at(int i) { return kPad ? i + (i >> 4) : i; }

struct Cplx {
    double r, i;
};
__device__ __forceinline__ void dif_butterfly(Cplx& a, Cplx& b, double2 t) {
    const double tr = a.r - b.r, ti = a.i - b.i;
    a.r = a.r + b.r;
    a.i = a.i + b.i;
    b.r = tr * t.x - ti * t.y;
    b.i = tr * t.y + ti * t.x;
}

template <bool kPad>
__device__ void lds_fft(double* re, double* im, int N, const double2* __restrict__ tw) {
    int n = N;
    for (; n > 2; n >>= 2) {
        const int k = n >> 2, sh = __ffs(k) - 1;
        const double2* T = tw + (N - n);             // stage n: entries 0 .. n/2 - 1
        const double2* T2 = tw + (N - (n >> 1));     // stage n/2
        for (int beta = threadIdx.x; beta < (N >> 2); beta += blockDim.x) {
            const int l = beta & (k - 1);
            const int a = ((beta >> sh) << (sh + 2)) + l;
            const int p0 = fft_at<kPad>(a), p1 = fft_at<kPad>(a + k), p2 = fft_at<kPad>(a + 2 * k),
                      p3 = fft_at<kPad>(a + 3 * k);
            Cplx x0{re[p0], im[p0]}, x1{re[p1], im[p1]}, x2{re[p2], im[p2]}, x3{re[p3], im[p3]};
            const double2 ta = T[l], tb = T[l + k], tc = T2[l];
            dif_butterfly(x0, x2, ta);
            dif_butterfly(x1, x3, tb);
            dif_butterfly(x0, x1, tc);
            dif_butterfly(x2, x3, tc);
            re[p0] = x0.r, im[p0] = x0.i;
            re[p1] = x1.r, im[p1] = x1.i;
            re[p2] = x2.r, im[p2] = x2.i;
            re[p3] = x3.r, im[p3] = x3.i;
        }
        __syncthreads();
    }
    if (n == 2) {
        const double2 t = tw[N - 2];
        for (int beta = threadIdx.x; beta < (N >> 1); beta += blockDim.x) {
            const int p0 = fft_at<kPad>(2 * beta), p1 = fft_at<kPad>(2 * beta + 1);
            Cplx x0{re[p0], im[p0]}, x1{re[p1], im[p1]};
            dif_butterfly(x0, x1, t);
            re[p0] = x0.r, im[p0] = x0.i;
            re[p1] = x1.r, im[p1] = x1.i;
        }
        __syncthreads();
    }
}

// Between the transforms the ramp reads the spectrum from its bit-reversed
// places, into registers (16 values a thread at most: H2 <= 4096), and writes
// it in order for the second transform; the result is read bit-reversed too.
// Bound by LDS passes and their barriers (two radix-2 stages a pass, no
// permutation passes: 2,880 sectors of 512^2 slices 68 -> 36 us).
template <bool kPad>
__global__ __launch_bounds__(256) void k_radn_filter(const SecDesc* __restrict__ secs, const double* __restrict__ P,
                                                     float* __restrict__ q, const double2* __restrict__ tw,
                                                     const int* __restrict__ tw_off, int maxH2) {
    extern __shared__ double buf[];
    const SecDesc& sd = secs[blockIdx.x];
    const int H = sd.H;
    const int m = (H <= 1) ? 0 : 32 - __clz(H - 1);  // H2 = 2^ceil(log2 H)
    const int H2 = 1 << m;
    double* re = buf;
    double* im = buf + fft_at<kPad>(maxH2);
    for (int i = threadIdx.x; i < H2; i += blockDim.x) {
        re[fft_at<kPad>(i)] = (i < H) ? P[sd.q + i] : 0.0;
        im[fft_at<kPad>(i)] = 0.0;
    }
    __syncthreads();
    const double2* T = tw + tw_off[m];
    auto rev = [&](int i) { return fft_at<kPad>(m ? (int)(__brev((unsigned)i) >> (32 - m)) : 0); };
    if (H2 > 1) lds_fft<kPad>(re, im, H2, T);
    // ramp: zero above H/2, gain (double)i/H below (kernelRADN.h:247);
    // then the conj of ifft's first step.
    constexpr int kPer = (1 << 12) / 256;
    Cplx x[kPer];
#pragma unroll
    for (int e = 0; e < kPer; e++) {
        const int i = threadIdx.x + 256 * e;
        x[e] = Cplx{0.0, -0.0};
        if (i < H2 && i <= H / 2) {
            const double g = (double)i / H;
            x[e].r = g * re[rev(i)];
            x[e].i = -(g * im[rev(i)]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPer; e++) {
        const int i = threadIdx.x + 256 * e;
        if (i < H2) {
            re[fft_at<kPad>(i)] = x[e].r;
            im[fft_at<kPad>(i)] = x[e].i;
        }
    }
    __syncthreads();
    if (H2 > 1) lds_fft<kPad>(re, im, H2, T);
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
        const double v = re[rev(i)] / H2;
        q[sd.q + i] = (float)(0.0 + v);  // skewOutput (zero) += Re
    }
}

hipError_t launch_radn_filter(const DevPlan& p, const double* P, float* q, const double* tw, const int* tw_off,
                              int maxH2, hipStream_t s) {
    if (p.nsec == 0) return hipSuccess;
    // padded up to 2048 points (35 KB); 4096 points take 64 KB unpadded
    if (maxH2 <= 2048) {
        const size_t lds = sizeof(double) * 2 * (size_t)(maxH2 + maxH2 / 16 + 1);
        hipLaunchKernelGGL(k_radn_filter<true>, dim3(p.nsec), dim3(256), lds, s, p.secs, P, q,
                           reinterpret_cast<const double2*>(tw), tw_off, maxH2);
    } else {
        const size_t lds = sizeof(double) * 2 * (size_t)maxH2;
        hipLaunchKernelGGL(k_radn_filter<false>, dim3(p.nsec), dim3(256), lds, s, p.secs, P, q,
                           reinterpret_cast<const double2*>(tw), tw_off, maxH2);
    }
    return hipGetLastError();
}

// Smear the filtered projection back along each row (kernelRADN.h:252-257)
// into a materialised skewOutput (the per-sector engine API).
__global__ __launch_bounds__(256) void k_radn_smear(const SecDesc* __restrict__ secs, const RowWork* __restrict__ work,
                                                    int nwork, const uint32_t* __restrict__ fl,
                                                    const float* __restrict__ q, float* __restrict__ SO) {
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= nwork) return;
    const int lane = threadIdx.x & 63;
    const RowWork w = work[item];
    const SecDesc sd = secs[w.sec];
    const uint32_t v = fl[sd.rows + w.row];
    const float x = q[sd.q + w.row];
    for (int j = fl_first(v) + lane; j < fl_last(v); j += 64) SO[sd.so + (size_t)w.row * sd.dim_i + j] = x;
}

hipError_t launch_radn_smear(const DevPlan& p, const float* q, float* SO, hipStream_t s) {
    if (p.nwork == 0) return hipSuccess;
    hipLaunchKernelGGL(k_radn_smear, dim3((p.nwork + 3) / 4), dim3(256), 0, s, p.secs, p.work, p.nwork, p.fl, q, SO);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Local Radon transform (LRT=true).  For skewed cell (i, j) the reference
// (pointRadon, kernelRADN.h:114-182) forms 64 samples
//   x_kk = g_kk * sum_{l=j-32}^{j+32} S(k, l) [first_k <= l < last_k],
//   k = i - 32 + kk (zero for k outside [0, H)),
// g_kk = exp(-(kk-32)^2 / (2 sigma^2)), sigma = (64/5)/scale, then
//   X = FFT64(x)/8,  y_f = sin(f/24.6 * pi/2) Re X_f for f <= 25, 0 above,
//   Y = FFT64(y)/8,  out = |Y_{m-1}|^2 at the first m in [5, 32) with
//   |Y_m|^2 > |Y_{m-1}|^2 (0 if none; getParameter :96-108).
// Here in two passes:
//   lrt_rowsum: one wave per skewed row forms every column's 65-wide window
//     sum in double -> W, all rows and columns of the sector.
//   op_lrt: a workgroup stages the 95 rows of window sums that a tile of 64
//     columns x 32 rows reaches in LDS; each cell then takes its 64 window
//     sums from there and evaluates the 26 needed real parts of X and
//     |Y_m|^2 for m = 4, 5, ... as cosine/sine sums (FP64), stopping at the
//     first rise.  The sums differ from the reference's radix-2 FFT only by
//     FP64 rounding.
// ---------------------------------------------------------------------------

// Blocks of a launch over all sectors of a plan: blockIdx.x the block within
// the sector, the sector split over y and z (a grid's y and z end at 65535).
constexpr int kSecY = 32768;
inline dim3 sector_grid(unsigned per_sector, int nsec) {
    return dim3(per_sector, (unsigned)(nsec < kSecY ? nsec : kSecY), (unsigned)((nsec + kSecY - 1) / kSecY));
}
__device__ __forceinline__ int sector_index() { return (int)(blockIdx.z * kSecY + blockIdx.y); }

// Inclusive sums over the 64 lanes, from lane 0 up (kUp) or from lane 63
// down: four DPP steps inside the rows of 16 lanes, then the totals of the
// rows before (after) this lane's, read as scalars.  Additions only, so a run
// of zeros stays exactly zero.
template <int kCtrl>
__device__ __forceinline__ double dpp_add(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, 0xf, 0xf, false);
    return x + __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double lane_value(double x, int lane) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <bool kUp>
__device__ __forceinline__ double wave_scan(double x, int lane) {
    constexpr int kShift = kUp ? 0x110 : 0x100;  // row_shr / row_shl
    x = dpp_add<kShift + 1>(x);
    x = dpp_add<kShift + 2>(x);
    x = dpp_add<kShift + 4>(x);
    x = dpp_add<kShift + 8>(x);
    const int row = kUp ? lane >> 4 : 3 - (lane >> 4);  // rows already passed
    const double t0 = lane_value(x, kUp ? 15 : 48), t1 = lane_value(x, kUp ? 31 : 32),
                 t2 = lane_value(x, kUp ? 47 : 16);
    const double t01 = t0 + t1, t012 = t01 + t2;
    return x + (row == 0 ? 0.0 : row == 1 ? t0 : row == 2 ? t01 : t012);
}

// Window sums W(r, j) = sum_{l=j-32}^{j+32} S(r, l) [first <= l < last].  With
// the row cut in blocks of 64 cells, the window of column 64 t - 32 + s is the
// tail of block t - 1 from its cell s and the head of block t up to its cell
// s, so two scans of a block's 64 cells serve 64 windows.  65 additions a cell and a
// zero fill before: 482 + 66 us for the 180 sectors of a 512^2 slice; now 206
// us, of which the 543 MB it writes take 112.  Every column of every row of the
// sector is written, rows without cells as zeros.
__global__ __launch_bounds__(256) void k_lrt_rowsum(const SecDesc* __restrict__ secs, int nsec,
                                                    const float* __restrict__ in4,
                                                    const int* __restrict__ target, const float* __restrict__ weight,
                                                    const uint32_t* __restrict__ fl, const float* __restrict__ Sbuf,
                                                    double* __restrict__ W) {
    const int si = sector_index();
    if (si >= nsec) return;
    const SecDesc& sd = secs[si];
    const int r = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (r >= sd.H) return;  // wave-uniform
    const int lane = threadIdx.x & 63;
    const uint32_t v = fl[sd.rows + r];
    const int f = fl_first(v), l = fl_last(v);
    const int dim_i = sd.dim_i, dim_o = sd.dim_o;
    const float* src = in4 + sd.img + (size_t)sd.type * sd.N;
    const int* tt = target + sd.tab;
    const float* ww = weight + sd.tab;
    double* out = W + sd.so + (size_t)r * dim_i;
    auto cell = [&](int j) -> float {
        if (j < f || j >= l) return 0.0f;
        return Sbuf ? Sbuf[(size_t)r * dim_i + j] : skew_cell_sel(src, tt[j], ww[j], r, j, dim_i, dim_o);
    };
    double tail = 0.0;
    float next = cell(lane);
    for (int c = 0; c - 32 < dim_i; c += 64) {
        const double x = (double)next;
        next = cell(c + 64 + lane);
        const bool some = c < l && c + 64 > f;  // uniform
        const double head = some ? wave_scan<true>(x, lane) : 0.0;
        const int j = c - 32 + lane;
        if (j >= 0 && j < dim_i) out[j] = tail + head;
        tail = some ? wave_scan<false>(x, lane) : 0.0;
    }
}

// The transform.  x_kk (times 1/8) is folded before the first cosine sum:
// cos(pi q kk/32) is even about kk = 32 and even or odd about 16 and 8 with
// the parity of q and q/2, so the 64 samples fall into nine groups ("orbits"
// k = 0..8 of kk -> 64 - kk, 32 - kk, 16 - kk) of which q = 0, 4, .. needs 9,
// q = 2, 6, .. 8 and odd q 16 values: 319 products instead of 64 x 26.  The
// coefficients (with the sine ramp and both factors 1/8, exact powers of two,
// already in them) come in wave-uniform rows: scalar loads.
// A cell whose 26 values are all zero (no image in its windows) is 0 by the
// peak rule and leaves the search for the first rise at once; otherwise 97% of
// cells stop at m <= 9.
// Bound by FP64 VALU issue: 64 columns x 32 rows a workgroup, a wave per row
// at a time, three window-sum reads of 8 B per cell from memory and 64 from LDS
// (conflict-free).  512^2, 180 sectors: 5.28 -> 1.42 ms.
constexpr int kLrtRows = 32, kLrtWin = kLrtRows + 63;
__global__ __launch_bounds__(512) void k_op_lrt(const SecDesc* __restrict__ secs, int nsec, int coltiles,
                                                const uint32_t* __restrict__ fl, const double* __restrict__ W,
                                                const double* __restrict__ tab, const double* __restrict__ gauss,
                                                float* __restrict__ arena) {
    __shared__ double win[kLrtWin * 64];
    const int si = sector_index();
    if (si >= nsec) return;  // uniform
    const SecDesc& sd = secs[si];
    const int H = sd.H, dim_i = sd.dim_i;
    const int rt = (int)blockIdx.x / coltiles;
    const int i0 = rt * kLrtRows, j0 = ((int)blockIdx.x - rt * coltiles) * 64;
    if (i0 >= H || j0 >= dim_i) return;  // uniform
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    {   // leave when no row of the tile has a cell in these columns (every wave finds the same)
        bool some = false;
        if (lane < kLrtRows && i0 + lane < H) {
            const uint32_t v = fl[sd.rows + i0 + lane];
            some = fl_first(v) < j0 + 64 && fl_last(v) > j0 && fl_first(v) < fl_last(v);
        }
        if (__builtin_amdgcn_ballot_w64(some) == 0) return;
    }
    const double* Wb = W + sd.so;
    const int j = j0 + lane;
    for (int y = wave; y < kLrtWin; y += 8) {
        const int k = i0 - 32 + y;
        win[y * 64 + lane] = (k >= 0 && k < H && j < dim_i) ? Wb[(size_t)k * dim_i + j] : 0.0;
    }
    __syncthreads();
    const double* g = gauss + 64 * sd.newAngle;
    for (int y = wave; y < kLrtRows; y += 8) {
        const int i = i0 + y;
        if (i >= H) break;  // uniform
        const uint32_t v = fl[sd.rows + i];
        const bool in = j >= fl_first(v) && j < fl_last(v);
        if (__builtin_amdgcn_ballot_w64(in) == 0) continue;
        const double* w = win + y * 64 + lane;  // sample kk at w[64 kk]
        double re[26];  // q = 0, 4, .., 24; q = 2, 6, .., 22; q = 1, 3, .., 25
        {
            const double u0 = g[0] * w[0], u32 = g[32] * w[64 * 32], u16 = g[16] * (w[64 * 16] + w[64 * 48]);
            const double v0 = u0 + u32, e = v0 + u16, o = v0 - u16, d = u0 - u32;
            const double* C = tab + kLrtC;
#pragma unroll
            for (int q = 0; q < 7; ++q) re[q] = e * C[q];
#pragma unroll
            for (int q = 0; q < 6; ++q) re[7 + q] = o * C[7 + q];
#pragma unroll
            for (int q = 0; q < 13; ++q) re[13 + q] = d * C[13 + q];
        }
        {
            const double u8 = g[8] * (w[64 * 8] + w[64 * 56]), u24 = g[24] * (w[64 * 24] + w[64 * 40]);
            const double e = u8 + u24, d = u8 - u24;
            const double* C = tab + kLrtC + 40 * 8;
#pragma unroll
            for (int q = 0; q < 7; ++q) re[q] = __builtin_fma(e, C[q], re[q]);
#pragma unroll
            for (int q = 0; q < 13; ++q) re[13 + q] = __builtin_fma(d, C[13 + q], re[13 + q]);
        }
#pragma unroll 1
        for (int k = 1; k < 8; ++k) {
            const double* wp = w + 64 * k;
            const double* wm = w - 64 * k;
            const double ua = g[k] * (wp[0] + wm[64 * 64]), ub = g[16 - k] * (wm[64 * 16] + wp[64 * 48]);
            const double uc = g[16 + k] * (wp[64 * 16] + wm[64 * 48]), ud = g[32 - k] * (wm[64 * 32] + wp[64 * 32]);
            const double va = ua + ud, vb = ub + uc;
            const double e = va + vb, o = va - vb, da = ua - ud, db = ub - uc;
            const double* C = tab + kLrtC + 40 * k;
#pragma unroll
            for (int q = 0; q < 7; ++q) re[q] = __builtin_fma(e, C[q], re[q]);
#pragma unroll
            for (int q = 0; q < 6; ++q) re[7 + q] = __builtin_fma(o, C[7 + q], re[7 + q]);
#pragma unroll
            for (int q = 0; q < 13; ++q)
                re[13 + q] = __builtin_fma(db, C[26 + q], __builtin_fma(da, C[13 + q], re[13 + q]));
        }
        uint32_t some = 0;
#pragma unroll
        for (int q = 0; q < 26; ++q) some |= (uint32_t)(__builtin_bit_cast(uint64_t, re[q]) >> 32);
        bool search = in && (some << 1) != 0;
        double prev = 0.0, val = 0.0;
        for (int m = 4; m < 32 && __builtin_amdgcn_ballot_w64(search) != 0; ++m) {
            const double* Y = tab + kLrtY + 64 * m;  // the 26 cosines, then the sines, in the order of re
            double yr[2] = {0.0, 0.0}, yi[2] = {0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 26; ++q) {
                yr[q & 1] = __builtin_fma(re[q], Y[2 * q], yr[q & 1]);
                yi[q & 1] = __builtin_fma(re[q], Y[2 * q + 1], yi[q & 1]);
            }
            const double r = yr[0] + yr[1], s = yi[0] + yi[1];
            const double cur = r * r + s * s;
            if (m > 4 && search && cur > prev) {
                val = prev;
                search = false;
            }
            prev = cur;
        }
        if (in) arena[sd.so + (size_t)i * dim_i + j] = (float)val;
    }
}

// The vectors the reference records at a sample point (pointRadon,
// kernelRADN.h:117-170, for the cells of samplePoints): x = the 64 windowed
// sums (from W) times the Gaussian, the Gaussian-weighted row through the
// cell (column j - 32 + kk of row i, inside the extents of row k = i - 32 + kk
// as the reference reads them; 0 for k outside [0, H)), y = the filtered
// real spectrum and Re FFT64(y)/8.  One 64-lane wave per request; direct
// sums in FP64 (cos/sin(2 pi t/64) from tab).
__global__ __launch_bounds__(64) void k_lrt_samples(const SecDesc* __restrict__ secs,
                                                    const SampleReq* __restrict__ req,
                                                    const uint32_t* __restrict__ fl, const double* __restrict__ W,
                                                    const float* __restrict__ in4, const int* __restrict__ target,
                                                    const float* __restrict__ weight, const double* __restrict__ tab,
                                                    const double* __restrict__ gauss, float* __restrict__ out) {
    __shared__ double xs[64], ys[64];
    const SampleReq r = req[blockIdx.x];
    const SecDesc sd = secs[r.sec];
    const int kk = threadIdx.x;
    const double g = gauss[64 * sd.newAngle + kk];
    const int k = r.i - 32 + kk;
    double win = 0.0, axis = 0.0;
    if (k >= 0 && k < sd.H) {
        win = W[sd.so + (size_t)k * sd.dim_i + r.j];
        const uint32_t v = fl[sd.rows + k];
        const int c = r.j - 32 + kk;
        if (c >= fl_first(v) && c < fl_last(v)) {
            const float* src = in4 + sd.img + (size_t)sd.type * sd.N;
            axis = g * (double)skew_cell(src, target[sd.tab + c], weight[sd.tab + c], r.i, c, sd.dim_i, sd.dim_o);
        }
    }
    const double x = win * g;
    xs[kk] = x;
    __syncthreads();
    double re = 0.0;
    for (int m = 0; m < 64; ++m) re = __builtin_fma(xs[m], tab[2 * ((kk * m) & 63)], re);
    const double y = kk <= 25 ? tab[160 + kk] * (re * 0.125) : 0.0;  // cutoff 0.4 * 64, sine ramp
    ys[kk] = y;
    __syncthreads();
    double yr = 0.0;
    for (int m = 0; m < 64; ++m) yr = __builtin_fma(ys[m], tab[2 * ((kk * m) & 63)], yr);
    float* o = out + (size_t)r.slot * 256;
    o[kk] = (float)x;
    o[64 + kk] = (float)axis;
    o[128 + kk] = (float)y;
    o[192 + kk] = (float)(yr * 0.125);
}

hipError_t launch_lrt_samples(const DevPlan& p, const SampleReq* req, int nreq, const float* in4, const double* W,
                              const double* tab, const double* gauss, float* out, hipStream_t s) {
    if (nreq == 0) return hipSuccess;
    hipLaunchKernelGGL(k_lrt_samples, dim3(nreq), dim3(64), 0, s, p.secs, req, p.fl, W, in4, p.target, p.weight, tab,
                       gauss, out);
    return hipGetLastError();
}

hipError_t launch_lrt(const DevPlan& p, const float* in4, const float* Sbuf, double* W, float* arena,
                      const double* tab, const double* gauss, hipStream_t s) {
    if (p.nsec == 0 || p.maxH <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_lrt_rowsum, sector_grid((unsigned)(p.maxH + 3) / 4, p.nsec), dim3(256), 0, s, p.secs, p.nsec,
                       in4, p.target, p.weight, p.fl, Sbuf, W);
    const unsigned ct = (unsigned)(p.maxI + 63) / 64, rt = (unsigned)(p.maxH + kLrtRows - 1) / kLrtRows;
    hipLaunchKernelGGL(k_op_lrt, sector_grid(ct * rt, p.nsec), dim3(512), 0, s, p.secs, p.nsec, (int)ct, p.fl, W, tab,
                       gauss, arena);
    return hipGetLastError();
}

}  // namespace ske
