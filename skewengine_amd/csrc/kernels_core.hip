// kernels_core.hip -- orientation copies, skew, identity operator, deskew and
// reduce on gfx950 (wave64).  Float arithmetic follows the reference CPU
// path operation by operation (built with -ffp-contract=off), so the
// per-sector and accumulated results are bit-identical to a one-thread run
// of the reference.
#include "device_common.h"
#include "launch.h"

namespace ske {

// ---------------------------------------------------------------------------
// prepare (src/skewEngine.cuh:962-987).  32x32 tiles through LDS so that the
// two transposed copies are written coalesced.  *odd, if not null, becomes 1
// when a value is not finite or above 1e30.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_prepare(const float* __restrict__ in0, float* __restrict__ in1,
                                                 float* __restrict__ in2, float* __restrict__ in3,
                                                 int dimx, int dimy, int* __restrict__ odd) {
    __shared__ float tile[32][33];
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
    for (int k = ty; k < 32; k += 8) {
        const int i = y0 + k, j = x0 + tx;
        if (i < dimy && j < dimx) {
            const float v = in0[(size_t)i * dimx + j];
            tile[k][tx] = v;
            if (odd && !(fabsf(v) <= 1e30f)) *odd = 1;
            in3[(size_t)i * dimx + (dimx - 1 - j)] = v;  // in3[dimx*i + cj]
        }
    }
    __syncthreads();
    // in1[dimy*cj + ci] and in2[dimy*j + ci]: output row indexed by x, column by y
    for (int k = ty; k < 32; k += 8) {
        const int j = x0 + k;       // source column -> output row
        const int i = y0 + tx;      // source row -> output column
        if (i < dimy && j < dimx) {
            const float v = tile[tx][k];
            const int ci = dimy - 1 - i, cj = dimx - 1 - j;
            in1[(size_t)dimy * cj + ci] = v;
            in2[(size_t)dimy * j + ci] = v;
        }
    }
}

__global__ __launch_bounds__(256) void k_fill_f32(float* __restrict__ p, size_t n, float v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

static unsigned fill_blocks(size_t n) {
    const size_t b = (n + 255) / 256;
    return (unsigned)(b < 65536 ? (b ? b : 1) : 65536);
}

hipError_t launch_fill_f32(float* p, size_t n, float v, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_f32, dim3(fill_blocks(n)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t launch_prepare(const float* in0, float* in1, float* in2, float* in3, int dimx, int dimy, int* odd,
                          hipStream_t s) {
    dim3 grid((dimx + 31) / 32, (dimy + 31) / 32);
    hipLaunchKernelGGL(k_prepare, grid, dim3(256), 0, s, in0, in1, in2, in3, dimx, dimy, odd);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// skew, materialised: every cell of the H x dim_i skewed block; the output
// buffer's block is zeroed (resetSkew).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_skew_full(const SecDesc* __restrict__ secs,
                                                   const float* __restrict__ in4,
                                                   const int* __restrict__ target,
                                                   const float* __restrict__ weight,
                                                   float* __restrict__ S, float* __restrict__ SO) {
    const SecDesc& sd = secs[0];
    const int r = blockIdx.y;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= sd.dim_i) return;
    const float* src = in4 + sd.img + (size_t)sd.type * sd.N;
    const size_t at = (size_t)r * sd.dim_i + j;
    SO[at] = 0.0f;
    S[at] = skew_cell_sel(src, target[sd.tab + j], weight[sd.tab + j], r, j, sd.dim_i, sd.dim_o);
}

hipError_t launch_skew_full(const DevPlan& p, const SecDesc& h, const float* in4, float* S, float* SO, hipStream_t s) {
    dim3 grid((h.dim_i + 255) / 256, h.H);
    hipLaunchKernelGGL(k_skew_full, grid, dim3(256), 0, s, p.secs, in4, p.target, p.weight, S, SO);
    return hipGetLastError();
}

// n 16-byte words, from pinned host memory to the device.
__global__ __launch_bounds__(256) void k_copy16(uint4* __restrict__ dst, const uint4* __restrict__ src, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

hipError_t launch_copy16(void* dst, const void* src, int n, hipStream_t s) {
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)(n + 255) / 256), dim3(256), 0, s, reinterpret_cast<uint4*>(dst),
                       reinterpret_cast<const uint4*>(src), n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// identity operator (src/kernelUNIT.h:16-23): SO = S on [first, last).
// One wave per row work item, four rows per block.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_op_unit(const SecDesc* __restrict__ secs, const RowWork* __restrict__ work,
                                                 int nwork, const float* __restrict__ in4,
                                                 const int* __restrict__ target, const float* __restrict__ weight,
                                                 const uint32_t* __restrict__ fl, const float* __restrict__ Sbuf,
                                                 float* __restrict__ arena) {
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= nwork) return;
    const int lane = threadIdx.x & 63;
    const RowWork w = work[item];
    const SecDesc sd = secs[w.sec];
    const uint32_t v = fl[sd.rows + w.row];
    const int f = fl_first(v), l = fl_last(v);
    const float* src = in4 + sd.img + (size_t)sd.type * sd.N;
    float* so = arena + sd.so + (size_t)w.row * sd.dim_i;
    for (int j = f + lane; j < l; j += 64) {
        float x;
        if (Sbuf)
            x = Sbuf[(size_t)w.row * sd.dim_i + j];
        else
            x = skew_cell(src, target[sd.tab + j], weight[sd.tab + j], w.row, j, sd.dim_i, sd.dim_o);
        so[j] = x;
    }
}

hipError_t launch_op_unit(const DevPlan& p, const float* in4, const float* Sbuf, float* arena, hipStream_t s) {
    if (p.nwork == 0) return hipSuccess;
    hipLaunchKernelGGL(k_op_unit, dim3((p.nwork + 3) / 4), dim3(256), 0, s, p.secs, p.work, p.nwork, in4,
                       p.target, p.weight, p.fl, Sbuf, arena);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// deskew (src/skewEngine.cuh:755-793) of all sectors of a plan, one thread per
// column of a few oriented output rows, sectors in ascending order per
// orientation.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float stdmaxf(float a, float b) { return (a < b) ? b : a; }

// skewOutput cell (r, j) of sector index si as the deskew gather sees it.
template <int kSource>
__device__ __forceinline__ float so_cell(const SecDesc* __restrict__ secs, int si, const SecDesc& sd,
                                         const uint32_t* __restrict__ fl, const float* __restrict__ src,
                                         int r, int j) {
    if (kSource == kDeskewDense) return src[(size_t)r * sd.dim_i + j];  // single reused buffer
    if (r < sd.H) {
        const uint32_t v = fl[sd.rows + r];
        return j < fl_first(v) || j >= fl_last(v) ? 0.0f : src[sd.so + (size_t)r * sd.dim_i + j];
    }
    // r == H happens only when newAngle == 0 (weight 0).  The reference reads
    // the row the previously processed sector left in its reused buffer.
    if (sd.stale >= 0) {
        const SecDesc pv = secs[sd.stale];
        if (r < pv.H && pv.dim_i == sd.dim_i) {
            const uint32_t v = fl[pv.rows + r];
            if (j >= fl_first(v) && j < fl_last(v)) return src[pv.so + (size_t)r * sd.dim_i + j];
        }
    }
    return 0.0f;
}

template <int kMax>
__device__ __forceinline__ float deskew_acc(float O, float a, float b, float wj, int angle) {
    if (kMax) {
        O = stdmaxf(O, stdmaxf(a, b));
        return (float)(angle + 1000 * (int)(O / 1000));
    }
    return O + ((1.0f - wj) * a + wj * b);
}

// Which taps need a look at first/last.  Output cell (i, j) reads the skewed
// rows t_j + i and t_j + i + 1, i.e. t_j + e with 0 <= e <= n (n = dim_o).  In
// a sector's maps j lies in [first, last) of the rows t_j + 1 .. t_j + n always
// (t rises by 0 or 1 per column; first is exact, last at most one short, and
// one short only for the column whose t is the row itself), so only e = 0 may
// fall outside, and e = n where the sector has no such row (newAngle 0).
// Checked over all sectors of many sides on the CPU: tests/test_deskew_taps.py.

// Taps e = i0 .. i0 + kRows of column j in the first or the last block of rows:
// taps past e = n are not used, e = 0 is tested by the caller.
template <int kSource, int kRows>
__device__ __forceinline__ void deskew_edge_taps(const SecDesc* __restrict__ secs, int si, const SecDesc& sd,
                                                 const uint32_t* __restrict__ fl, const float* __restrict__ src, int i0,
                                                 int tj, int j, int dim_o, float (&v)[kRows + 1]) {
    const float* p = src + (kSource == kDeskewArena ? sd.so : 0);
#pragma unroll
    for (int m = 0; m <= kRows; ++m) v[m] = p[(size_t)min(tj + min(i0 + m, dim_o), sd.H - 1) * sd.dim_i + j];
    if (i0 + kRows >= dim_o && sd.newAngle == 0) {  // uniform
        const float x = so_cell<kSource>(secs, si, sd, fl, src, tj + dim_o, j);
#pragma unroll
        for (int m = 0; m <= kRows; ++m)
            if (i0 + m == dim_o) v[m] = x;
    }
}

// The same taps in an inner block (0 < i0, i0 + kRows < n), which need no look.
// Lane j's taps are the rows i0 + t_j .. i0 + t_j + kRows of its column: taken
// in that order, the 64 lanes of a steep sector read 64 rows at once, and a
// line comes from L2 again for every lane that shares it.  Each lane starts
// (t_j - t_0) mod (kRows + 1) rows further up instead and wraps, so that at
// every load the lanes of a band of kRows + 1 rows read one row; a pass through
// the wave's own LDS puts the taps back in order.  The row blocks start at
// different rows of the band: with a side of 1024 they would otherwise all
// read rows a multiple of 64 KB apart, and so few memory channels, at a time.
template <int kRows>
__device__ __forceinline__ int deskew_shift(int tj, unsigned by) {
    return (int)((unsigned)(tj - __builtin_amdgcn_readfirstlane(tj)) + 5u * by) % (kRows + 1);
}
template <int kSource, int kRows>
__device__ __forceinline__ void deskew_inner_taps(const SecDesc& sd, const float* __restrict__ src, int i0, int tj,
                                                  int shift, int j, float (&v)[kRows + 1]) {
    const float* p = src + (kSource == kDeskewArena ? sd.so : 0);
    // loads k < shift are the last taps, k >= shift the first
    const unsigned lo = (unsigned)(i0 + tj - shift) * (unsigned)sd.dim_i + (unsigned)j;
    const unsigned hi = lo + (unsigned)((kRows + 1) * sd.dim_i);
#pragma unroll
    for (int k = 0; k <= kRows; ++k) v[k] = (p + (size_t)k * sd.dim_i)[k < shift ? hi : lo];
}
// `lds`: this lane's column of (kRows + 1) x 64, with kRows x 64 in front.
template <int kRows>
__device__ __forceinline__ void deskew_order(float* lds, int shift, float (&v)[kRows + 1]) {
    float* const lo = lds - 64 * shift;
    float* const hi = lo + 64 * (kRows + 1);
#pragma unroll
    for (int k = 0; k <= kRows; ++k) (k < shift ? hi : lo)[64 * k] = v[k];
#pragma unroll
    for (int m = 0; m <= kRows; ++m) v[m] = lds[64 * m];
}

// kRows consecutive output rows per thread: the kRows + 1 taps of a sector are
// shared by neighbouring rows; each row accumulates in ascending sector order.
// While a sector is added, the taps of the next and the table entries of the
// one after are on their way.
template <int kSource, int kMax, int kRows, bool kEdge>
__device__ __forceinline__ void deskew_rows(const SecDesc* __restrict__ secs, const int* __restrict__ target,
                                            const float* __restrict__ weight, const uint32_t* __restrict__ fl,
                                            const float* __restrict__ src, int sb, int se, int i0, int j, int dim_o,
                                            unsigned by, float* own, float (&O)[kRows]) {
    float v[kRows + 1], vn[kRows + 1];
    uint32_t f = 0, fn = 0;  // the row range of e = 0
    auto load = [&](int si, int t, int shift, uint32_t& fx, float (&x)[kRows + 1]) {
        if constexpr (kEdge) {
            if (kSource != kDeskewDense && i0 == 0) fx = fl[secs[si].rows + t];
            deskew_edge_taps<kSource, kRows>(secs, si, secs[si], fl, src, i0, t, j, dim_o, x);
        } else {
            deskew_inner_taps<kSource, kRows>(secs[si], src, i0, t, shift, j, x);
        }
    };
    int tn = target[secs[sb].tab + j], shift = deskew_shift<kRows>(tn, by), shift_n = 0;
    float w = weight[secs[sb].tab + j], wn = 0.0f;
    load(sb, tn, shift, f, v);
    if (sb + 1 < se) {
        tn = target[secs[sb + 1].tab + j];
        wn = weight[secs[sb + 1].tab + j];
    }
    for (int si = sb; si < se; ++si) {
        int t2 = 0;
        float w2 = 0.0f;
        if (si + 2 < se) {
            t2 = target[secs[si + 2].tab + j];
            w2 = weight[secs[si + 2].tab + j];
        }
        if (si + 1 < se) {
            shift_n = deskew_shift<kRows>(tn, by);
            load(si + 1, tn, shift_n, fn, vn);
        }
        if constexpr (kEdge) {
            if (kSource != kDeskewDense && i0 == 0 && (j < fl_first(f) || j >= fl_last(f))) v[0] = 0.0f;
        } else {
            deskew_order<kRows>(own, shift, v);
        }
        const int angle = secs[si].angle;
#pragma unroll
        for (int k = 0; k < kRows; ++k) O[k] = deskew_acc<kMax>(O[k], v[k], v[k + 1], w, angle);
#pragma unroll
        for (int m = 0; m <= kRows; ++m) v[m] = vn[m];
        f = fn;
        w = wn;
        wn = w2;
        tn = t2;
        shift = shift_n;
    }
}

// Orientation t of one image: sectors [sb, se), accumulators acc (four
// dimx*dimy buffers), started from zero with `init`.
template <int kSource, int kMax, int kRows>
__device__ __forceinline__ void deskew_body(const SecDesc* __restrict__ secs, const int* __restrict__ target,
                                            const float* __restrict__ weight, const uint32_t* __restrict__ fl,
                                            const float* __restrict__ src, int t, int sb, int se, bool init,
                                            float* __restrict__ acc, int dimx, int dimy) {
    __shared__ float lds[64 * (kRows + 4 * (kRows + 1))];
    if (sb >= se) return;
    const bool tr = (t == 1 || t == 2);
    const int dim_i = tr ? dimy : dimx, dim_o = tr ? dimx : dimy;
    // Workgroups go to the eight XCDs in turn: each XCD takes a run of blocks, so
    // that a line which two neighbouring row blocks share comes to one L2 once.
    const unsigned total = gridDim.x * gridDim.y, lin = blockIdx.x + gridDim.x * blockIdx.y, xcd = lin & 7;
    const unsigned at = xcd * (total >> 3) + min(xcd, total & 7) + (lin >> 3);
    const unsigned by = at / gridDim.x, bx = at - by * gridDim.x;
    const int i0 = (int)by * kRows;
    const int j = (int)(bx * blockDim.x + threadIdx.x);
    if (i0 >= dim_o || j >= dim_i) return;
    const size_t N = (size_t)dimx * dimy;
    float* o = acc + (size_t)t * N + (size_t)i0 * dim_i + j;
    const int nrow = min(kRows, dim_o - i0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* const own = lds + 64 * (kRows + wave * (kRows + 1)) + lane;
    float O[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k) O[k] = (!init && k < nrow) ? o[(size_t)k * dim_i] : 0.0f;
    if (i0 == 0 || i0 + kRows >= dim_o)  // uniform
        deskew_rows<kSource, kMax, kRows, true>(secs, target, weight, fl, src, sb, se, i0, j, dim_o, by, own, O);
    else
        deskew_rows<kSource, kMax, kRows, false>(secs, target, weight, fl, src, sb, se, i0, j, dim_o, by, own, O);
#pragma unroll
    for (int k = 0; k < kRows; ++k)
        if (k < nrow) o[(size_t)k * dim_i] = O[k];
}

// Bound by the reads of the arena (each cell once: 500^2 moves 190 MB, 2048^2 3
// GB).  All sectors with every tap tested, taken straight down the columns, one
// sector at a time and the last rows of an odd side one by one -> now: 250^2
// 536 -> 56 us, 500^2 263 -> 68, 1024^2 260 -> 250 (maximum: 368 -> 253), 1501^2
// 1,444 -> 435, 2048^2 991 -> 739 us (4.1 TB/s).  Without the rotated order
// 1501^2 takes 866 us, without the runs of blocks per XCD about 500; 8 rows a
// thread instead of 16: 500^2 130 -> 158 us, 2048^2 852 -> 1,240.
// The Radon source below 1024 workgroups: 4 rows 40 us (one 512^2 image; 49
// with the taps gathered, 16 rows a thread).
constexpr int kDeskewRows = 16;      // output rows per thread
constexpr int kDeskewRadonRows = 4;  // of the Radon source below 1024 workgroups

__device__ __forceinline__ int range_begin(int t, int4 lo, int4 hi) {
    return (t == 0) ? lo.x : (t == 1) ? lo.z : (t == 2) ? hi.x : hi.z;
}
__device__ __forceinline__ int range_end(int t, int4 lo, int4 hi) {
    return (t == 0) ? lo.y : (t == 1) ? lo.w : (t == 2) ? hi.y : hi.w;
}

// One image: blockIdx.z = orientation; bit t of `init`: orientation t starts
// from zero.
template <int kSource, int kMax, int kRows>
__global__ __launch_bounds__(256) void k_deskew(const SecDesc* __restrict__ secs, const int* __restrict__ target,
                                                const float* __restrict__ weight, const uint32_t* __restrict__ fl,
                                                const float* __restrict__ src, int4 rlo, int4 rhi, int init,
                                                float* __restrict__ acc, int dimx, int dimy) {
    const int t = blockIdx.z;
    deskew_body<kSource, kMax, kRows>(secs, target, weight, fl, src, t, range_begin(t, rlo, rhi),
                                      range_end(t, rlo, rhi), (init >> t) & 1, acc, dimx, dimy);
}

// The Radon deskew with the taps staged in LDS.  A Radon skewOutput row r
// holds q[r] on [first_r, last_r), so a sector's taps for a workgroup's 256
// columns j0 .. j0+255 and rows i0 .. i0+15 are q of the rows i0 + t_j ..
// i0 + t_j + 16: since t is nondecreasing with steps of 0 or 1, the rows
// i0 + t_{j0} .. i0 + t_{j0} + 271, at most.  A pass stages them for kRadonU
// sectors (zeros past H), two sectors a wave; the next pass's rows and table
// entries are loaded into registers while this one's are added.  Then every
// thread reads its 17 taps per sector from LDS: the values so_cell gives
// (first/last matter for the tap of row t_j alone, see above), added in
// ascending sector order, so the result is the k_deskew one bit for bit.
// Bound by VALU and LDS issue at four workgroups per CU: 16 x 512^2 189 us (260
// with the row ranges staged and tested too and no loads in flight meanwhile).
constexpr int kRadonU = 8, kRadonStage = 288;  // 9 KB of LDS: eight sectors per pass
template <int kRows>
__device__ __forceinline__ void deskew_radon_body(const SecDesc* __restrict__ secs, const int* __restrict__ target,
                                                  const float* __restrict__ weight,
                                                  const uint32_t* __restrict__ fl, const float* __restrict__ q,
                                                  int t, int sb, int se, bool init, float* __restrict__ acc, int dimx,
                                                  int dimy) {
    constexpr int kPer = kRadonU / 4, kLoads = (kRadonStage + 63) / 64;
    __shared__ float sq[kRadonU * kRadonStage];
    if (sb >= se) return;  // uniform
    const bool tr = (t == 1 || t == 2);
    const int dim_i = tr ? dimy : dimx, dim_o = tr ? dimx : dimy;
    const int i0 = blockIdx.y * kRows;
    const int j0 = blockIdx.x * blockDim.x;
    if (i0 >= dim_o || j0 >= dim_i) return;  // uniform
    const int j = min(j0 + (int)threadIdx.x, dim_i - 1);
    const bool col = j0 + (int)threadIdx.x < dim_i;
    const size_t N = (size_t)dimx * dimy;
    float* o = acc + (size_t)t * N + (size_t)i0 * dim_i + j;
    const int nrow = min(kRows, dim_o - i0);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    float O[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k) O[k] = (!init && col && k < nrow) ? o[(size_t)k * dim_i] : 0.0f;
    // sector si + u: this thread's table entries (d: its row past the stage's first), the wave's stage rows
    int dn[kRadonU];
    float wn[kRadonU], sn[kPer][kLoads];
    auto load = [&](int si) {
#pragma unroll
        for (int u = 0; u < kRadonU; ++u) {
            const int tab = secs[min(si + u, se - 1)].tab;
            dn[u] = target[tab + j] - target[tab + j0];
            wn[u] = weight[tab + j];
        }
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            const SecDesc& sd = secs[min(si + kPer * wave + c, se - 1)];
            const int r0 = i0 + target[sd.tab + j0];
#pragma unroll
            for (int e = 0; e < kLoads; ++e) {
                const int r = r0 + 64 * e + lane;
                sn[c][e] = r < sd.H ? q[sd.q + r] : 0.0f;
            }
        }
    };
    load(sb);
    for (int si = sb; si < se; si += kRadonU) {
        const int nu = min(kRadonU, se - si);
        int d[kRadonU];
        float w[kRadonU];
        __syncthreads();  // the previous pass's reads are done
#pragma unroll
        for (int c = 0; c < kPer; ++c)
#pragma unroll
            for (int e = 0; e < kLoads; ++e)
                if (64 * e + lane < kRadonStage) sq[(kPer * wave + c) * kRadonStage + 64 * e + lane] = sn[c][e];
#pragma unroll
        for (int u = 0; u < kRadonU; ++u) {
            d[u] = dn[u];
            w[u] = wn[u];
        }
        __syncthreads();
        if (si + kRadonU < se) load(si + kRadonU);
#pragma unroll
        for (int u = 0; u < kRadonU; ++u) {
            if (u >= nu) break;  // uniform
            // stage index of row i0 + t_j (t_j - t_{j0} <= j - j0 <= 255; the clamp only guards the stage's bounds)
            const float* p = sq + u * kRadonStage + min(d[u], kRadonStage - kRows - 1);
            float v[kRows + 1];
#pragma unroll
            for (int m = 0; m <= kRows; ++m) v[m] = p[m];
            if (i0 == 0) {  // uniform: the tap of row t_j
                const SecDesc& sd = secs[si + u];
                if (j >= fl_last(fl[sd.rows + target[sd.tab + j]])) v[0] = 0.0f;
            }
#pragma unroll
            for (int k = 0; k < kRows; ++k) O[k] = deskew_acc<0>(O[k], v[k], v[k + 1], w[u], 0);
        }
    }
    if (col) {
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (k < nrow) o[(size_t)k * dim_i] = O[k];
    }
}

template <int kRows>
__global__ __launch_bounds__(256) void k_deskew_radon(const SecDesc* __restrict__ secs,
                                                      const int* __restrict__ target,
                                                      const float* __restrict__ weight,
                                                      const uint32_t* __restrict__ fl, const float* __restrict__ q,
                                                      int4 rlo, int4 rhi, int init, float* __restrict__ acc, int dimx,
                                                      int dimy) {
    const int t = blockIdx.z;
    deskew_radon_body<kRows>(secs, target, weight, fl, q, t, range_begin(t, rlo, rhi), range_end(t, rlo, rhi),
                      (init >> t) & 1, acc, dimx, dimy);
}

template <int kRows>
__global__ __launch_bounds__(256) void k_deskew_radon_parts(const SecDesc* __restrict__ secs,
                                                            const int* __restrict__ target,
                                                            const float* __restrict__ weight,
                                                            const uint32_t* __restrict__ fl,
                                                            const float* __restrict__ q,
                                                            const DeskewPart* __restrict__ parts,
                                                            float* __restrict__ acc) {
    const DeskewPart& P = parts[blockIdx.z >> 2];
    const int t = blockIdx.z & 3;
    deskew_radon_body<kRows>(secs, target, weight, fl, q, t, P.range[2 * t], P.range[2 * t + 1], (P.init >> t) & 1,
                      acc + P.acc_off, P.dimx, P.dimy);
}

hipError_t launch_deskew(const DevPlan& p, const int range[8], const float* src, int source, int is_max, int init,
                         float* acc, int dimx, int dimy, long long img_acc, hipStream_t s) {
    const int dl = dimx > dimy ? dimx : dimy;
    int4 lo = make_int4(range[0], range[1], range[2], range[3]);
    int4 hi = make_int4(range[4], range[5], range[6], range[7]);
    float* a = acc + img_acc;
    const unsigned gx = (unsigned)(dl + 255) / 256;
#define SKE_DESKEW(SRC, MX, ROWS)                                                                                    \
    hipLaunchKernelGGL((k_deskew<SRC, MX, ROWS>), dim3(gx, (unsigned)(dl + ROWS - 1) / ROWS, 4), dim3(256), 0, s,    \
                       p.secs, p.target, p.weight, p.fl, src, lo, hi, init, a, dimx, dimy)
#define SKE_DESKEW_RADON(ROWS)                                                                                         \
    hipLaunchKernelGGL((k_deskew_radon<ROWS>), dim3(gx, (unsigned)(dl + ROWS - 1) / ROWS, 4), dim3(256), 0, s, p.secs, \
                       p.target, p.weight, p.fl, src, lo, hi, init, a, dimx, dimy)
    if (source == kDeskewDense) {
        if (is_max) SKE_DESKEW(kDeskewDense, 1, kDeskewRows); else SKE_DESKEW(kDeskewDense, 0, kDeskewRows);
    } else if (source == kDeskewArena) {
        if (is_max) SKE_DESKEW(kDeskewArena, 1, kDeskewRows); else SKE_DESKEW(kDeskewArena, 0, kDeskewRows);
    } else if ((size_t)gx * ((dl + kDeskewRows - 1) / kDeskewRows) * 4 >= 1024) {
        SKE_DESKEW_RADON(kDeskewRows);
    } else {
        SKE_DESKEW_RADON(kDeskewRadonRows);
    }
#undef SKE_DESKEW
#undef SKE_DESKEW_RADON
    return hipGetLastError();
}

hipError_t launch_deskew_parts(const DevPlan& p, const DeskewPart* parts, int nparts, int max_dim, const float* q,
                               float* acc, hipStream_t s) {
    if (nparts <= 0) return hipSuccess;
    if (nparts > 16383) return hipErrorInvalidValue;
    const unsigned gx = (unsigned)(max_dim + 255) / 256, gz = 4u * (unsigned)nparts;
#define SKE_DESKEW_P(ROWS)                                                                                             \
    hipLaunchKernelGGL((k_deskew_radon_parts<ROWS>), dim3(gx, (unsigned)(max_dim + ROWS - 1) / ROWS, gz), dim3(256),   \
                       0, s, p.secs, p.target, p.weight, p.fl, q, parts, acc)
    if ((size_t)gx * gz * ((max_dim + kDeskewRows - 1) / kDeskewRows) >= 1024)
        SKE_DESKEW_P(kDeskewRows);
    else
        SKE_DESKEW_P(kDeskewRadonRows);
#undef SKE_DESKEW_P
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// reduce (src/skewEngine.cuh:885-912).  out[i,j] (+)= o0[i,j], o1[cj,ci],
// o2[j,ci], o3[i,cj] in that order.  o1/o2 are read through an LDS tile so
// that their transposed accesses stay coalesced.  kInit: out starts from zero
// (it is written, not read).
// ---------------------------------------------------------------------------
template <int kMax, bool kInit>
__device__ __forceinline__ void reduce_body(const float* __restrict__ acc, int4 present, float* __restrict__ out,
                                            int dimx, int dimy) {
    __shared__ float t1[32][33];
    __shared__ float t2[32][33];
    const size_t N = (size_t)dimx * dimy;
    const float* o0 = acc;
    const float* o1 = acc + N;
    const float* o2 = acc + 2 * N;
    const float* o3 = acc + 3 * N;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    if (x0 >= dimx || y0 >= dimy) return;  // uniform: a smaller image of a batch
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    // o1 rows cj = dimx-1-j (j in [x0, x0+32)), columns ci = dimy-1-i;
    // o2 rows j, columns ci.  Load both tiles with ci along threadIdx.x.
#pragma unroll
    for (int k = ty; k < 32; k += 8) {
        const int j = x0 + k;
        const int i = y0 + 31 - tx;  // ci = dimy-1-i runs forward with tx
        if (j < dimx && i >= 0 && i < dimy) {
            const int ci = dimy - 1 - i, cj = dimx - 1 - j;
            if (present.y) t1[k][31 - tx] = o1[(size_t)cj * dimy + ci];
            if (present.z) t2[k][31 - tx] = o2[(size_t)j * dimy + ci];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = ty; k < 32; k += 8) {
        const int i = y0 + k, j = x0 + tx;
        if (i >= dimy || j >= dimx) continue;
        const size_t oi = (size_t)i * dimx + j;
        float v = kInit ? 0.0f : out[oi];
        const int cj = dimx - 1 - j;
        if (kMax) {
            if (present.x) { const float u = o0[oi]; v = (v > u) ? v : u; }
            if (present.y) { const float u = t1[tx][k]; v = (v > u) ? v : u; }
            if (present.z) { const float u = t2[tx][k]; v = (v > u) ? v : u; }
            if (present.w) { const float u = o3[(size_t)i * dimx + cj]; v = (v > u) ? v : u; }
        } else {
            if (present.x) v += o0[oi];
            if (present.y) v += t1[tx][k];
            if (present.z) v += t2[tx][k];
            if (present.w) v += o3[(size_t)i * dimx + cj];
        }
        out[oi] = v;
    }
}

template <int kMax>
__global__ __launch_bounds__(256) void k_reduce(const float* __restrict__ acc, int4 present,
                                                float* __restrict__ out, int dimx, int dimy) {
    reduce_body<kMax, false>(acc, present, out, dimx, dimy);
}

// Up to kReduceImages images of an engine or batch in one launch (blockIdx.z),
// written from zero: 16 maps of 512^2 in 16 us (16 launches of 7 us and a fill
// of 10 us before).
constexpr int kReduceImages = 64;
struct ReduceGroup {
    ReduceImage im[kReduceImages];  // 1.5 KB of kernel arguments
};
template <int kMax>
__global__ __launch_bounds__(256) void k_reduce_images(const float* __restrict__ acc, int4 present,
                                                       float* __restrict__ out, ReduceGroup g) {
    const ReduceImage im = g.im[blockIdx.z];
    reduce_body<kMax, true>(acc + im.acc_off, present, out + im.out_off, im.n, im.n);
}

hipError_t launch_reduce(const float* acc, const int present[4], float* out, int dimx, int dimy, int is_max,
                         hipStream_t s) {
    dim3 grid((dimx + 31) / 32, (dimy + 31) / 32);
    int4 pr = make_int4(present[0], present[1], present[2], present[3]);
    if (is_max)
        hipLaunchKernelGGL(k_reduce<1>, grid, dim3(256), 0, s, acc, pr, out, dimx, dimy);
    else
        hipLaunchKernelGGL(k_reduce<0>, grid, dim3(256), 0, s, acc, pr, out, dimx, dimy);
    return hipGetLastError();
}

hipError_t launch_reduce_images(const float* acc, const int present[4], float* out, const ReduceImage* imgs, int count,
                                int is_max, hipStream_t s) {
    const int4 pr = make_int4(present[0], present[1], present[2], present[3]);
    for (int first = 0; first < count; first += kReduceImages) {
        ReduceGroup g{};
        const int m = count - first < kReduceImages ? count - first : kReduceImages;
        int side = 1;
        for (int i = 0; i < m; ++i) {
            g.im[i] = imgs[first + i];
            side = g.im[i].n > side ? g.im[i].n : side;
        }
        const dim3 grid((unsigned)(side + 31) / 32, (unsigned)(side + 31) / 32, (unsigned)m);
        if (is_max)
            hipLaunchKernelGGL(k_reduce_images<1>, grid, dim3(256), 0, s, acc, pr, out, g);
        else
            hipLaunchKernelGGL(k_reduce_images<0>, grid, dim3(256), 0, s, acc, pr, out, g);
    }
    return hipGetLastError();
}

}  // namespace ske
