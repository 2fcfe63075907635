// kernels_sdem.hip -- total-viewshed operator (src/kernelSDEM.h:168-222) on
// gfx950.
//
// Layout: one workgroup (2 to 8 waves) per skewed row.  The row is staged once
// in LDS.  Per-step and one-chunk kernels: each wave takes 64 consecutive
// observers and runs their right scans then their left scans with a
// wave-uniform step d = 1, 2, ... (the default kernels take pools of up to four
// such chunks and skip blocks of steps that cannot be visible: below).  As d is
// uniform, 1/d and d*d come from a scalar table and every lane reads
// row[j +/- d] from consecutive LDS words (no bank conflicts).  Each lane
// keeps the reference's per-observer state (max angle, visible flag, opening
// distance) and accumulates cv in the reference's order, so cv and every
// visibility decision are bit-identical to the CPU path.
//
// Division.  The reference computes cAngle = (S[k]-h)/d with an IEEE divide.
// Variant 1 does exactly that.  Variant 0 uses q = fma(a, yh, a*yl) with
// yh = RN(1/d), yl = RN(1/d - yh): |q_exact - a/d| < 2^-47 |a/d| before the
// final rounding, while for d < 2^22 the quotient a/d of a float a is never
// closer than 2^-13 ulp to a rounding midpoint (a is a multiple of ulp(a/d)
// and a midpoint times d is an odd multiple of half an ulp with at least
// 25 significant bits, so it is never a float).  Hence fma(a, yh, a*yl)
// rounds to exactly RN(a/d): two VALU operations instead of the ~10 of the
// IEEE divide sequence.  The tests check both variants against each other
// and against the oracle.
#include <float.h>

#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "launch.h"

namespace ske {

template <int kVariant>
__device__ __forceinline__ void sdem_step(float sk, float h, const float4 t, float& M, float& od2, bool& vis,
                                          float& cv) {
    const float a = sk - h;
    float q;
    if (kVariant == 0) {
        q = __builtin_fmaf(a, t.x, a * t.y);
        q = __builtin_isinf(a) ? a : q;  // the products would give inf * 0
    } else {
        q = a / t.z;
    }
    const bool above = q > M;
    M = q < M ? M : q;  // std::max(cAngle, max_angle): a quotient that is no number stays
    const bool opening = above && !vis;
    const bool closing = !above && vis;
    vis = above;
    od2 = opening ? t.w : od2;               // open_delta_d^2 (exact: integers < 2^24)
    cv = closing ? cv + (t.w - od2) : cv;    // cv += d*d - od*od
}

// Chunk c of 64 observers: every step of both scans.
template <int kVariant>
__device__ __forceinline__ void sdem_steps_chunk(const float* row, int L, int c, float povh,
                                                 const float4* __restrict__ rtab, float* __restrict__ so, float R) {
    const int lane = threadIdx.x & 63;
    const int j0 = c << 6;
    const int jj = j0 + lane;
    const bool valid = jj < L;
    const float h = row[jj] + povh;
    float cv = 0.0f;
    {   // right scan: k = j+1 .. last-1
        float M = -2000.0f, od2 = 0.0f;
        bool vis = true;
        const int myR = valid ? (L - 1 - jj) : 0;
        const int dall = L - 1 - (j0 + 63);  // every lane active up to here
        const int dmax = L - 1 - j0;
        int d = 1;
        for (; d <= dall; ++d) sdem_step<kVariant>(row[jj + d], h, rtab[d], M, od2, vis, cv);
        for (; d <= dmax; ++d) {
            const float4 t = rtab[d];
            const float sk = row[jj + d];
            if (d <= myR) sdem_step<kVariant>(sk, h, t, M, od2, vis, cv);
        }
    }
    {   // left scan: k = j-1 .. first
        float M = -2000.0f, od2 = 0.0f;
        bool vis = true;
        const int myL = valid ? jj : 0;
        const int dall = (j0 + 63 < L) ? j0 : -1;
        const int dmax = (j0 + 63 < L) ? (j0 + 63) : (L - 1);
        int d = 1;
        for (; d <= dall; ++d) sdem_step<kVariant>(row[jj - d], h, rtab[d], M, od2, vis, cv);
        for (; d <= dmax; ++d) {
            const float4 t = rtab[d];
            const float sk = row[jj - d];
            if (d <= myL) sdem_step<kVariant>(sk, h, t, M, od2, vis, cv);
        }
    }
    if (valid) so[jj] = cv * R;
}

template <int kVariant>
__global__ __launch_bounds__(256) void k_op_sdem(const SecDesc* __restrict__ secs,
                                                 const RowWork* __restrict__ work,
                                                 const float* __restrict__ in4,
                                                 const int* __restrict__ target,
                                                 const float* __restrict__ weight,
                                                 const uint32_t* __restrict__ fl,
                                                 const float* __restrict__ Sbuf,
                                                 const float4* __restrict__ rtab, float povh,
                                                 float* __restrict__ arena) {
    extern __shared__ float lds[];
    float* row = lds + kPad;
    const RowWork w = work[blockIdx.x];
    const SecDesc sd = secs[w.sec];
    const int r = w.row;
    const uint32_t v = fl[sd.rows + r];
    const int f = fl_first(v);
    const int L = fl_last(v) - f;
    if (L <= 0) return;
    stage_row(row, sd, r, f, L, in4, target, weight, Sbuf);
    __syncthreads();

    const int nchunk = (L + 63) >> 6;
    float* so = arena + sd.so + (size_t)r * sd.dim_i + f;
    for (int c = threadIdx.x >> 6; c < nchunk; c += 4) sdem_steps_chunk<kVariant>(row, L, c, povh, rtab, so, sd.R);
}

// ---------------------------------------------------------------------------
// Bit-block variant.  One scan direction of one observer sees visibility
// flags V_1..V_D (V_0 = 1: the observer's own cell).  The reference adds
// d_c^2 - d_o^2 for every visible run (d_o, d_c] that closes before the row
// end; since d_c^2 - d_o^2 = sum_{k=d_o}^{d_c-1} (2k+1), that total is
//     cv = sum_{k=0..D} V_k (2k+1)  -  sum over the trailing run of (2k+1)
//        = A - ((D+1)^2 - s^2),  s = 1 + last step with V = 0 (0 if none).
// Steps past a lane's own scan length are recorded as visible: they extend
// the trailing run and cancel exactly, so every lane runs the same
// wave-uniform D (a multiple of 32).  Per step a lane only computes the
// quotient, one compare, one max and appends the flag to a 32-bit word;
// every 32 steps popcounts of the word update A and s:
//     sum_{V=1} (2k+1) = (2 d0 + 65) popc(w) - 2 sum_p p w_p,
//     sum_p p w_p = sum_i 2^i popc(w & M_i),   k = d0 + 32 - p.
// All quantities are integers below 2^24 for rows of at most 4096 cells, so
// the float cv of the reference (whose partial sums are exact integers
// there) is reproduced bit for bit.
// ---------------------------------------------------------------------------
// Guard band on each side of a staged row: the one-chunk scans of a chunk
// run to its first lane's row end, up to 95 cells past the row (128); with
// pools a block only runs while some lane's row continues, so every read
// stays within 32 cells of the row (and of the safe positions), and of the
// per-step scans within kPad.
template <int kG>
constexpr int pad_bits() { return kG > 1 ? kPad : 128; }
// 32-cell chunks of a row of <= 4096 cells, and of the longest (16,000 cells).
constexpr int kChunksMax = 128, kChunksLong = 512;
// Chunk-maximum tables of a staged row: eight words per chunk c in [-kTabLo,
// nch + kTabHi), nch the row's chunks: level 0 max row[32c .. 32c+31], levels
// 1..3 the maxima of 2, 4 and 8 consecutive chunks starting at c, then suffix
// and prefix maxima (two words are free: 32 bytes a chunk, so a position's byte
// offset is itself rounded down to 32).  Chunks outside the row hold -inf (the
// prefix maximum repeats the row's past the end).
constexpr int kTabLo = 16, kTabHi = 16, kTabWords = 8;
enum { kTabL0 = 0, kTabL1 = 1, kTabL2 = 2, kTabL3 = 3, kTabSuf = 4, kTabPre = 5 };
__host__ __device__ inline int tab_words(int L) { return kTabWords * (kTabLo + ((L + 31) >> 5) + kTabHi); }
// The words of the chunk of position p (may lie outside the row).
__device__ __forceinline__ const float* tab_at(const float* tab, int p) {
    return tab + kTabLo * kTabWords + ((p & ~31) >> 2);
}

__device__ __forceinline__ int lshl1_add(int a, int b) {
    int r;
    asm("v_lshl_add_u32 %0, %1, 1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ void flush_block(uint32_t w, int d0, int& A, int& s) {
    const int pc = __popc(w);
    // sp in Horner form, one v_lshl_add per level (the compiler would
    // otherwise expand it into separate shifts and adds)
    int sp = __popc(w & 0xFFFF0000u);
    sp = lshl1_add(sp, __popc(w & 0xFF00FF00u));
    sp = lshl1_add(sp, __popc(w & 0xF0F0F0F0u));
    sp = lshl1_add(sp, __popc(w & 0xCCCCCCCCu));
    sp = lshl1_add(sp, __popc(w & 0xAAAAAAAAu));
    A += (int)__umul24(2 * d0 + 65, pc) - 2 * sp;  // operands < 2^13
    // s = d0 + 33 - ctz(~w) when the block has an invisible step: such a value
    // exceeds every earlier s (<= d0 + 1).  v_ffbl gives ~0u for ~w == 0, which
    // the saturating subtraction turns into 0, so the max keeps s.
    uint32_t f;
    asm("v_ffbl_b32 %0, %1" : "=v"(f) : "v"(~w));
    s = max(s, (int)__builtin_elementwise_sub_sat((uint32_t)(d0 + 33), f));
}

// Rows past 4096 cells: the sums pass 2^24, so the float additions round and
// their order counts.  cv then takes the closed runs of a block one by one, as
// the reference does (a few per lane and block; none in most blocks).  cv holds
// the sum; s the open run's d_o^2 with the flag of the last step as its sign.
// A run in progress at the end of the row adds nothing; steps past the row end
// are recorded as visible and close none.
__device__ __forceinline__ float square(int d) {
#pragma clang fp contract(off)
    return (float)d * (float)d;
}
__device__ __forceinline__ float add_run(float cv, int dc, float od2) {
#pragma clang fp contract(off)
    return cv + (square(dc) - od2);  // cv += d*d - od*od
}
__device__ __forceinline__ void flush_runs(uint32_t w, int d0, bool live, int& A, int& s) {
    const uint32_t prev = (w >> 1) | ((uint32_t)s & 0x80000000u);  // each step's predecessor
    const uint32_t open = w & ~prev;
    uint32_t close = live ? prev & ~w : 0u;
    float cv = __int_as_float(A), od2 = __int_as_float(s & 0x7FFFFFFF);
    while (close) {
        const int p = __clz(close);  // step d0 + 1 + p
        const uint32_t before = open & ~(0xFFFFFFFFu >> p);
        if (before) od2 = square(d0 + 33 - __ffs(before));
        cv = add_run(cv, d0 + 1 + p, od2);
        close &= ~(0x80000000u >> p);
    }
    if (open) od2 = square(d0 + 33 - __ffs(open));
    A = __float_as_int(cv);
    s = (int)(__float_as_uint(od2) | (w << 31));
}

// The visibility flag is the sign of t = M - q: rounding preserves the sign
// of the exact difference and M == q gives +0, so sign(t) = (q > M).
// alignbit(w, t, 31) = (w << 1) | (t >> 31) appends it in one operation.
// The 32 reciprocal pairs of a block are loaded up front (wave-uniform:
// scalar loads, one wait), so the steps themselves wait only on LDS.
template <int kDir, bool kTail>
__device__ __forceinline__ uint32_t scan_block(const float* rowj, float h, const float4* __restrict__ rtab, int d0,
                                               int myLen, float& M) {
    const float2* __restrict__ ytab = reinterpret_cast<const float2*>(rtab + kMaxDim + 1);
    float2 y[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) y[u] = ytab[d0 + 1 + u];
    uint32_t w = 0;
#pragma unroll
    for (int u = 1; u <= 32; ++u) {
        const int d = d0 + u;
        const float a = rowj[kDir * d] - h;
        const float q = __builtin_fmaf(a, y[u - 1].x, a * y[u - 1].y);
        float t = M - q;
        if (kTail) t = (d > myLen) ? -1.0f : t;  // past this lane's row end: record visible
        M = fmaxf(M, q);
        w = __builtin_amdgcn_alignbit(w, __float_as_uint(t), 31);
    }
    return w;
}

// 16 steps d0 + u0 + 1 .. d0 + u0 + 16 of a block (no tail handling),
// appended to w: the pools run a block as two halves, so only 16
// reciprocal pairs are live in scalar registers at a time.
template <int kDir>
__device__ __forceinline__ uint32_t scan_half(const float* rowj, float h, const float2* __restrict__ ytab, int d0,
                                              int u0, float& M, uint32_t w) {
#pragma unroll
    for (int u = 1; u <= 16; ++u) {
        const int d = d0 + u0 + u;
        const float2 y = ytab[d];
        const float a = rowj[kDir * d] - h;
        const float q = __builtin_fmaf(a, y.x, a * y.y);
        const float t = M - q;
        M = fmaxf(M, q);
        w = __builtin_amdgcn_alignbit(w, __float_as_uint(t), 31);
    }
    return w;
}

// Early exit.  After the steps up to db, no later target of a lane can be
// visible once an upper bound of its quotient is <= M.  The remaining
// targets (distances e = db+1 .. myLen) are split into four segments that
// start at distances e, e+32, e+96 and e+224 (the last runs to the row end);
// with a_i = (largest height of segment i) - h, every later a_k is <= the
// a_i of its segment by monotone rounding, so every later quotient is
//     <= max( max_i a_i / e_i ,  (max_i a_i) / L ).
// (The second term covers a_i < 0, where a farther target has the larger
// quotient; L exceeds every distance.  When some a_i >= 0 it is dominated by
// the first term.)  Segment maxima come from the chunk tables over a
// superset of each segment's cells: extra cells only raise the bound.  The
// products use RN(1/e) and are rounded once, so the bound is raised by
// 2^-20 of its magnitude to stay above the rounded quotients.  When every
// lane of the wave is past its row end or bounded by its running maximum
// M, the scan stops: a lane with steps left has only invisible steps ahead,
// so its trailing visible run closes and counts (cv = A); a lane whose row
// ended keeps the usual correction of the padded steps.
// kClamp: clamp the nearest-target position into the row (callers whose
// lanes may lie far past their row end); without it p must lie in
// [-32, L + 31], which the chunk tables' padding covers.
// kCh > kChunksMax: distances are cut to L in the reciprocal table, which ends
// 32 entries past the longest row; a segment that starts past L holds no target.
template <int kDir, bool kClamp = true, int kCh = kChunksMax>
__device__ __forceinline__ float exit_bound(const float* __restrict__ tab, int jj, int L, float h, int db,
                                            const float2* __restrict__ ytab, float invL) {
    const int e = db + 1;
    int p = jj + kDir * e;  // nearest remaining target
    if (kClamp) p = p < 0 ? 0 : (p > L - 1 ? L - 1 : p);
    const float* t = tab_at(tab, p);
    float s1, s2, s3, s4;
    if (kDir > 0) {  // cells [p, p+32), [p+32, p+96), [p+96, p+224), [p+224, end)
        s1 = t[kTabL1];
        s2 = t[kTabL2 + kTabWords];
        s3 = t[kTabL3 + 3 * kTabWords];
        s4 = t[kTabSuf + 7 * kTabWords];
    } else {         // cells (p-32, p], (p-96, p-32], (p-224, p-96], [0, p-224]
        s1 = t[kTabL1 - kTabWords];
        s2 = t[kTabL2 - 4 * kTabWords];
        s3 = t[kTabL3 - 10 * kTabWords];
        s4 = t[kTabPre - 7 * kTabWords];
    }
    const float a1 = s1 - h, a2 = s2 - h, a3 = s3 - h, a4 = s4 - h;
    const float amax = fmaxf(fmaxf(a1, a2), fmaxf(a3, a4));
    auto y = [&](int d) { return ytab[kCh > kChunksMax ? min(d, L) : d].x; };
    float b = fmaxf(fmaxf(a1 * y(e), a2 * y(e + 32)), fmaxf(a3 * y(e + 96), a4 * y(e + 224)));
    b = fmaxf(b, amax * invL);
    return __builtin_fmaf(fabsf(b), 9.5367431640625e-7f, b);  // b + |b| 2^-20
}

template <int kDir>
__device__ __forceinline__ bool scan_done(const float* __restrict__ tab, int jj, int L, float h, float invL,
                                          const float2* __restrict__ ytab, int myLen, int db, float M) {
    const bool done = (myLen <= db) | (exit_bound<kDir>(tab, jj, L, h, db, ytab, invL) <= M);
    // every lane of the wave is active here; a ballot keeps the exit uniform
    return __builtin_amdgcn_readfirstlane((int)(__builtin_amdgcn_ballot_w64(!done) != 0)) == 0;
}

template <int kDir>
__device__ __forceinline__ int scan_dir(const float* rowj, float h, const float4* __restrict__ rtab, int myLen,
                                        int dfull, int D, const float* __restrict__ tab, int jj, int L,
                                        int& nblk) {
    const float2* __restrict__ ytab = reinterpret_cast<const float2*>(rtab + kMaxDim + 1);
    const float invL = ytab[L].x;
    float M = -2000.0f;
    int A = 1, s = 0;
    int d0 = 0;
    int e1 = dfull, e2 = D;  // loop ends, lowered to the current step when the scan stops
    for (; d0 + 32 <= e1; d0 += 32) {
        flush_block(scan_block<kDir, false>(rowj, h, rtab, d0, myLen, M), d0, A, s);
        if (scan_done<kDir>(tab, jj, L, h, invL, ytab, myLen, d0 + 32, M)) e1 = e2 = d0 + 32;
    }
    for (; d0 < e2; d0 += 32) {
        flush_block(scan_block<kDir, true>(rowj, h, rtab, d0, myLen, M), d0, A, s);
        if (scan_done<kDir>(tab, jj, L, h, invL, ytab, myLen, d0 + 32, M)) e2 = d0 + 32;
    }
    nblk += d0 >> 5;
    return myLen > d0 ? A : A - ((d0 + 1) * (d0 + 1) - s * s);
}

// Build the chunk tables of a staged row of L <= 32 kCh cells.  Ends with a
// barrier.  kCheck: returns whether every height lies in [-FLT_MAX, 1e30].
template <int kWaves, int kCh, bool kCheck>
__device__ __forceinline__ bool row_tables(const float* row, int L, float* tab) {
    constexpr int kPer = kCh / 64;
    const int nch = (L + 31) >> 5, total = kTabLo + nch + kTabHi;
    float* t0 = tab + kTabLo * kTabWords;
    for (int i = threadIdx.x; i < kTabWords * total; i += 64 * kWaves) tab[i] = -INFINITY;
    __syncthreads();
    bool plain = true;
    for (int t0i = 0; t0i < nch * 32; t0i += 64 * kWaves) {
        const int t = t0i + (int)threadIdx.x;
        float v = t < L ? row[t] : -INFINITY;
        if (kCheck) plain &= t >= L || (v >= -FLT_MAX && v <= 1e30f);
#pragma unroll
        for (int o = 16; o; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
        if ((t & 31) == 0 && t < nch * 32) t0[kTabL0 + kTabWords * (t >> 5)] = v;
    }
    if (kCheck)
        plain = __syncthreads_and(plain);
    else
        __syncthreads();
    if (threadIdx.x < 64) {  // one wave: suffix and prefix maxima, kPer chunks per lane
        const int l = threadIdx.x;
        float x[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) x[i] = kPer * l + i < nch ? t0[kTabL0 + kTabWords * (kPer * l + i)] : -INFINITY;
        float vs = x[0];
#pragma unroll
        for (int i = 1; i < kPer; ++i) vs = fmaxf(vs, x[i]);
        float vp = vs;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float us = __shfl_down(vs, o), up = __shfl_up(vp, o);  // own value when out of range
            vs = fmaxf(vs, us);
            vp = fmaxf(vp, up);
        }
        float ns = __shfl_down(vs, 1), np = __shfl_up(vp, 1);
        if (l == 63) ns = -INFINITY;
        if (l == 0) np = -INFINITY;
#pragma unroll
        for (int i = kPer - 1; i >= 0; --i) {
            ns = fmaxf(x[i], ns);
            if (kPer * l + i < nch) t0[kTabSuf + kTabWords * (kPer * l + i)] = ns;
        }
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            np = fmaxf(x[i], np);
            if (kPer * l + i < nch) t0[kTabPre + kTabWords * (kPer * l + i)] = np;
        }
        const float top = __shfl(np, 63);  // whole-row maximum
        if (l < kTabHi) t0[kTabPre + kTabWords * (nch + l)] = top;
    }
    for (int lev = 1; lev <= 3; ++lev) {  // level lev from level lev-1: max of two runs 2^(lev-1) apart
        const int off = 1 << (lev - 1);
        for (int i = threadIdx.x; i < total - off; i += 64 * kWaves)
            tab[lev + kTabWords * i] = fmaxf(tab[lev - 1 + kTabWords * i], tab[lev - 1 + kTabWords * (i + off)]);
        __syncthreads();
    }
    return plain;
}

// ---------------------------------------------------------------------------
// Pools.  With the early exit a wave still runs until its longest scan stops,
// while most of its lanes are done, and most blocks of a scan that goes on hold
// no visible step: its running maximum bounds them from their chunk maximum
// alone.  A wave therefore takes a pool of up to kPoolChunks chunks (64 scans
// of one direction each, all starting at d = 1) and steps them in rounds of one
// 32-step block with the same uniform d.  A round first tests every live scan:
//   - over: nothing beyond can be visible (exit_bound, every other round); it
//     stores its cv and leaves;
//   - nothing visible in this block: it stays as it is;
//   - otherwise it goes on the round's list.
// Then the listed scans run the block, 64 at a time.  State (running maximum,
// sums) stays at the scan's place in the wave's own LDS; two lists of places
// are kept in order, the live one rewritten in place (a place is never written
// past the ones still to be read).
// A block left out counts as 32 invisible steps: a trailing visible run ends
// with the last block run, so the sums of the steps with V = 1 and that block's
// end say everything.
// A lane's steps past its row end are recorded as visible by or-ing the low
// bits of its block word; empty lanes read from a position whose remaining
// steps stay inside the staged row and guard bands.  The right-scan pass stores
// cv as an integer in the output cell; the left-scan pass of the same pool
// (same wave, later) adds its cv and stores the float (float)(cvR + cvL) * R,
// the same value as the one-chunk path.
//
// Bound by VALU issue (1.24 wave instructions a clock and CU; the steps' mix
// reaches 1.5) and LDS gathers of the thinned lists (2.3 clocks a wave and cell
// in a row, 6 scattered).  Against groups of four chunks packed in registers,
// every block of a live scan run: all sectors of 1000^2 11.5 -> 9.9 ms, 1501^2
// 30.2 -> 29.2, 30 of 3000^2 28.6 -> 25.0, 20 of 4000^2 34.5 -> 30.7; 12 of
// 4600^2 (long rows) 43 -> 36.  Pools of 3 chunks run too many part-filled
// batches (1000^2 10.4 ms), of 6 leave too few waves per CU (3000^2 27.0).  Two
// batches at a time hide the LDS latency (one: 34.5 ms at 1501^2); four need
// 129 registers (45 ms).  One pool for all waves of a row with two barriers a
// round: 38.7.
// ---------------------------------------------------------------------------
constexpr int kPoolChunks = 4, kPoolChunksLong = 4;
// LDS bytes of a pool per scan: M, A | last block run << 24, the trailing run's
// start s and two places of two bytes; long rows M, cv, d_o^2 with the flag,
// the last block and the places.
template <bool kLong>
__host__ __device__ constexpr int pool_bytes() { return kLong ? 18 : 14; }
// Chunks of a pool of a row of nchunk chunks: every wave as many pools, of at
// most `cap` chunks.
__host__ __device__ inline int pool_chunks(int nchunk, int waves, int cap) {
    const int turns = (nchunk + waves * cap - 1) / (waves * cap);
    return (nchunk + waves * turns - 1) / (waves * turns);
}
// The cap of a launch: the pools of its longest row.
template <bool kLong>
__host__ __device__ inline int pool_cap(int maxL, int waves) {
    return pool_chunks((maxL + 63) / 64, waves, kLong ? kPoolChunksLong : kPoolChunks);
}

__device__ __forceinline__ int lanes_below(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Chunks [c0, c0 + nck) of a row; st: pool_bytes x stride of this wave's LDS
// (4-byte aligned), stride >= 64 nck.
template <int kDir, bool kLong>
__device__ __forceinline__ void scan_pool(const float* row, int L, float povh, int c0, int nck,
                                          const float* __restrict__ tab, const float4* __restrict__ rtab,
                                          float* __restrict__ so, float R, char* st, int stride, int& nblk) {
    const float2* __restrict__ ytab = reinterpret_cast<const float2*>(rtab + kMaxDim + 1);
    constexpr int kCh = kLong ? kChunksLong : kChunksMax;
    const float invL = ytab[L].x;
    const int lane = threadIdx.x & 63;
    const int safe = kDir > 0 ? 0 : L - 1;  // reads row[safe + kDir*d], d <= L + 31: inside the guard bands
    float* const smax = reinterpret_cast<float*>(st);
    int* const sums = reinterpret_cast<int*>(st + 4 * stride);  // A < 2^24 while steps are left; long rows cv
    uint32_t* const open = reinterpret_cast<uint32_t*>(st + 8 * stride);  // long rows
    uint16_t* const tail = reinterpret_cast<uint16_t*>(st + (kLong ? 12 : 8) * stride);  // s; long rows: the last block
    uint16_t* const live = tail + stride;
    uint16_t* const todo = live + stride;
    const int jb = 64 * c0;
    // the right scan's cv as an integer in the output cell (a float's bits: every access is of the one type)
    auto put = [&](int j, int cv) { so[j] = __int_as_float(cv); };
    auto right = [&](int j) { return __float_as_int(so[j]); };

    // cv of a scan with steps left, all invisible
    auto over = [&](int id, int j) {
        if (kLong) {
            float cv = __int_as_float(sums[id]);
            const uint32_t o = open[id];  // its open run closes after the last block run
            if (o >> 31) cv = add_run(cv, 32 * tail[id] + 1, __uint_as_float(o & 0x7FFFFFFFu));
            so[j] = kDir > 0 ? cv : cv * R;
        } else {
            const int cv = sums[id] & 0xFFFFFF;
            if (kDir > 0)
                put(j, cv);
            else
                so[j] = (float)(cv + right(j)) * R;
        }
    };
    // Block d0 of kN batches of scans (places id of the pool, positions j; a:
    // lane in use).  M, A, s: state before it, s the trailing run's start (long
    // rows: d_o^2 and flag).  Stores the state, or cv where the row ends; on:
    // the lanes that go on.
    auto block = [&](auto kn, const bool* a, const int* id, const int* j, int d0, const float* M0, const int* A0,
                     const int* s0, bool* on) {
        constexpr int kN = decltype(kn)::value;
        const int db = d0 + 32;
        float h[kN], M[kN];
        int A[kN], s[kN];
        uint32_t w[kN];
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            h[i] = row[j[i]] + povh;
            M[i] = M0[i];
            A[i] = A0[i];
            s[i] = s0[i];
        }
#pragma unroll
        for (int i = 0; i < kN; ++i) w[i] = scan_half<kDir>(row + j[i], h[i], ytab, d0, 0, M[i], 0u);
#pragma unroll
        for (int i = 0; i < kN; ++i) w[i] = scan_half<kDir>(row + j[i], h[i], ytab, d0, 16, M[i], w[i]);
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            const int myLen = kDir > 0 ? L - 1 - j[i] : j[i];
            // steps past the row end (the last e of the block) are recorded as
            // visible; skipped when no lane's row ends in this block
            if (__builtin_amdgcn_ballot_w64(myLen < db) != 0) {
                const int e = min(max(db - myLen, 0), 31);
                w[i] |= (1u << e) - 1u;
            }
            if (kLong)
                flush_runs(w[i], d0, a[i], A[i], s[i]);
            else
                flush_block(w[i], d0, A[i], s[i]);
            on[i] = a[i] && myLen > db;
            if (on[i]) {
                smax[id[i]] = M[i];
                if (kLong) {
                    sums[id[i]] = A[i];
                    open[id[i]] = (uint32_t)s[i];
                    tail[id[i]] = (uint16_t)(db >> 5);
                } else {
                    sums[id[i]] = A[i] | (db >> 5) << 24;  // db < L: A <= (db + 1)^2 < 2^24
                    tail[id[i]] = (uint16_t)s[i];
                }
            } else if (a[i]) {
                if (kLong) {
                    const float cv = __int_as_float(A[i]);
                    so[j[i]] = kDir > 0 ? cv : cv * R;
                } else {
                    const int cv = A[i] - ((db + 1) * (db + 1) - s[i] * s[i]);
                    if (kDir > 0)
                        put(j[i], cv);
                    else
                        so[j[i]] = (float)(cv + right(j[i])) * R;
                }
            }
        }
        nblk += kN;
    };
    // kN batches of the first block: chunks k, k + 1, ..; the live list so far.
    int n = 0;  // live scans (wave-uniform)
    auto first = [&](auto kn, int k) {
        constexpr int kN = decltype(kn)::value;
        bool a[kN], on[kN];
        int id[kN], j[kN], A[kN], s[kN];
        float M[kN];
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            id[i] = 64 * (k + i) + lane;
            j[i] = jb + id[i];
            const int myLen = kDir > 0 ? L - 1 - j[i] : j[i];
            const bool in = j[i] < L;
            a[i] = in && myLen > 0;
            if (in && !a[i]) {  // no targets in this direction: cv = 0
                if (kDir > 0)
                    put(j[i], 0);  // long rows: +0
                else
                    so[j[i]] = (kLong ? so[j[i]] : (float)right(j[i])) * R;
            }
            // A counts the observer's own cell; long rows go on with the right
            // scan's sum, visible from d = 0
            A[i] = kLong ? (kDir < 0 && a[i] ? __float_as_int(so[j[i]]) : 0) : 1;
            s[i] = kLong ? (int)0x80000000 : 0;
            if (!a[i]) j[i] = safe;
            M[i] = -2000.0f;
        }
        block(kn, a, id, j, 0, M, A, s, on);
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            const uint64_t m = __builtin_amdgcn_ballot_w64(on[i]);
            if (on[i]) live[n + lanes_below(m)] = (uint16_t)id[i];
            n += (int)__popcll(m);
        }
    };
    {
        int k = 0;
        for (; k + 2 <= nck; k += 2) first(std::integral_constant<int, 2>{}, k);
        if (k < nck) first(std::integral_constant<int, 1>{}, k);
    }
    for (int d0 = 32; n > 0; d0 += 32) {
        const int db = d0 + 32, e = d0 + 1;
        const bool far = ((d0 >> 5) & 1) != 0;  // rounds that test the exit
        const float y1 = ytab[e].x, y32 = ytab[e + 31].x;
        int nn = 0, nt = 0;
        auto test = [&](auto kn, int b) {
            constexpr int kN = decltype(kn)::value;
            bool a[kN], need[kN], done[kN];
            int id[kN], j[kN];
            float M[kN], h[kN];
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                a[i] = b + 64 * i + lane < n;
                id[i] = live[b + 64 * i + lane];
            }
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                id[i] = a[i] ? id[i] : 0;
                j[i] = a[i] ? jb + id[i] : safe;
                M[i] = smax[id[i]];
                h[i] = row[j[i]] + povh;
                // the block's cells lie in two chunks at most
                const float a1 = tab_at(tab, j[i] + kDir * e)[kDir > 0 ? kTabL1 : kTabL1 - kTabWords] - h[i];
                float bnd = fmaxf(a1 * y1, a1 * y32);
                bnd = __builtin_fmaf(fabsf(bnd), 9.5367431640625e-7f, bnd);
                need[i] = a[i] && bnd > M[i];
                done[i] = false;
            }
            if (far) {
#pragma unroll
                for (int i = 0; i < kN; ++i)
                    done[i] = exit_bound<kDir, false, kCh>(tab, j[i], L, h[i], d0, ytab, invL) <= M[i];
            }
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                const int myLen = kDir > 0 ? L - 1 - j[i] : j[i];
                const bool run = need[i] && !done[i];
                if (a[i] && !run && (done[i] || myLen <= db)) over(id[i], j[i]);
                const uint64_t mr = __builtin_amdgcn_ballot_w64(run);
                if (run) todo[nt + lanes_below(mr)] = (uint16_t)id[i];
                nt += (int)__popcll(mr);
                const bool on = a[i] && !done[i] && myLen > db;
                const uint64_t ml = __builtin_amdgcn_ballot_w64(on);
                if (on) live[nn + lanes_below(ml)] = (uint16_t)id[i];
                nn += (int)__popcll(ml);
            }
        };
        auto run = [&](auto kn, int b) {
            constexpr int kN = decltype(kn)::value;
            bool a[kN], on[kN];
            int id[kN], j[kN], A[kN], s[kN];
            float M[kN];
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                a[i] = b + 64 * i + lane < nt;
                id[i] = todo[b + 64 * i + lane];
            }
#pragma unroll
            for (int i = 0; i < kN; ++i) {
                id[i] = a[i] ? id[i] : 0;
                j[i] = a[i] ? jb + id[i] : safe;
                M[i] = smax[id[i]];
                A[i] = sums[id[i]];
                if (kLong) {
                    s[i] = (int)open[id[i]];
                    const int last = 32 * tail[id[i]];
                    if (a[i] && s[i] < 0 && last != d0) {  // blocks left out since: the open run closed after `last`
                        A[i] = __float_as_int(
                            add_run(__int_as_float(A[i]), last + 1, __int_as_float(s[i] & 0x7FFFFFFF)));
                        s[i] &= 0x7FFFFFFF;
                    }
                } else {
                    s[i] = 32 * (A[i] >> 24) == d0 ? (int)tail[id[i]] : d0 + 1;
                    A[i] &= 0xFFFFFF;
                }
            }
            block(kn, a, id, j, d0, M, A, s, on);
        };
        int b = 0;
        for (; b + 64 < n; b += 128) test(std::integral_constant<int, 2>{}, b);
        if (b < n) test(std::integral_constant<int, 1>{}, b);
        b = 0;
        for (; b + 64 < nt; b += 128) run(std::integral_constant<int, 2>{}, b);
        if (b < nt) run(std::integral_constant<int, 1>{}, b);
        n = __builtin_amdgcn_readfirstlane(nn);
    }
}

// LDS of the bit-block kernels: the waves' pools, guard band, row, guard band,
// chunk tables.
template <bool kLong>
__host__ __device__ inline int sdem_pools(int maxL, int group, int waves) {
    return group > 1 ? waves * 64 * pool_cap<kLong>(maxL, waves) * pool_bytes<kLong>() : 0;
}
inline size_t sdem_bits_lds(int maxL, int group, int waves) {
    return sdem_pools<false>(maxL, group, waves) +
           sizeof(float) * ((size_t)maxL + 2 * (group > 1 ? pad_bits<4>() : pad_bits<1>()) + tab_words(maxL));
}
inline size_t sdem_long_lds(int maxL, int waves) {
    return sdem_pools<true>(maxL, 4, waves) +
           sizeof(float) * ((size_t)maxL + 2 * pad_bits<4>() + tab_words(maxL));
}

// One skewed row: stage it, then every wave of the workgroup takes chunks
// of 64 observers (kG = 1), or pools of chunks, handed out by an LDS counter.  Ends with a barrier so the caller may
// restage LDS.
template <int kWaves, int kG, bool kCheck, bool kLong = false>
__device__ __forceinline__ void sdem_bits_row(const RowWork w, const SecDesc* __restrict__ secs,
                                              const float* __restrict__ in4, const int* __restrict__ target,
                                              const float* __restrict__ weight, const uint32_t* __restrict__ fl,
                                              const float* __restrict__ Sbuf, const float4* __restrict__ rtab,
                                              float povh, float* __restrict__ arena, char* pools, int pools_bytes,
                                              unsigned long long* __restrict__ steps, int* gnext) {
    float* const row = reinterpret_cast<float*>(pools + pools_bytes) + pad_bits<kG>();
    const SecDesc sd = secs[w.sec];
    const int r = w.row;
    const uint32_t v = fl[sd.rows + r];
    const int f = fl_first(v);
    const int L = fl_last(v) - f;
    if (L <= 0) return;  // uniform; the work list holds only rows with L > 0
    stage_row(row, sd, r, f, L, in4, target, weight, Sbuf, pad_bits<kG>());
    if (kG > 1 && threadIdx.x == 0) *gnext = kWaves;
    __syncthreads();
    const int nchunk = (L + 63) >> 6;
    float* so = arena + sd.so + (size_t)r * sd.dim_i + f;
    float* tab = row + L + pad_bits<kG>();  // past the right guard band
    const bool plain = row_tables<kWaves, kLong ? kChunksLong : kChunksMax, kCheck>(row, L, tab);
    if (kCheck && !(plain && fabsf(povh) <= 1e30f)) {
        // The bit of a step is the sign of M - q, which is not q > M once a
        // difference is infinite or no number.  Heights in [-FLT_MAX, 1e30]
        // keep every one finite (1e30 is below half an ulp of FLT_MAX); a row
        // with any other takes the per-step scans, which compare as the
        // reference does.
        for (int c = threadIdx.x >> 6; c < nchunk; c += kWaves)
            sdem_steps_chunk<0>(row, L, c, povh, rtab, so, sd.R);
        __syncthreads();
        return;
    }

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int nblk = 0;  // 32-step blocks this wave ran (both directions)
    if (kG > 1) {
        const int cap = pools_bytes / (64 * kWaves * pool_bytes<kLong>());
        const int per = pool_chunks(nchunk, kWaves, cap), stride = 64 * per;
        const int npools = (nchunk + per - 1) / per;
        for (int g = wave; g < npools;) {
            const int c0 = g * per;
            const int nck = min(per, nchunk - c0);
            char* st = pools + wave * pool_bytes<kLong>() * stride;
            scan_pool<+1, kLong>(row, L, povh, c0, nck, tab, rtab, so, sd.R, st, stride, nblk);
            scan_pool<-1, kLong>(row, L, povh, c0, nck, tab, rtab, so, sd.R, st, stride, nblk);
            int ng = 0;
            if (lane == 0) ng = atomicAdd(gnext, 1);
            g = __builtin_amdgcn_readfirstlane(ng);
        }
    }
    for (int c = wave; kG == 1 && c < nchunk; c += kWaves) {
        const int j0 = c << 6;
        const int jj = j0 + lane;
        const bool valid = jj < L;
        const bool full = j0 + 63 < L;  // all 64 observers of the chunk exist
        const float h = row[jj] + povh;
        // right scan: k = j+1 .. last-1
        const int dmaxR = L - 1 - j0;
        const int cvR = scan_dir<+1>(row + jj, h, rtab, valid ? L - 1 - jj : 0, full ? L - 1 - (j0 + 63) : 0,
                                     (dmaxR + 31) & ~31, tab, jj, L, nblk);
        // left scan: k = j-1 .. first
        const int dmaxL = full ? j0 + 63 : L - 1;
        const int cvL = scan_dir<-1>(row + jj, h, rtab, valid ? jj : 0, full ? j0 : 0, (dmaxL + 31) & ~31, tab,
                                     jj, L, nblk);
        if (valid) so[jj] = (float)(cvR + cvL) * sd.R;
    }
    if (steps && lane == 0 && nblk) atomicAdd(steps, 2048ull * (unsigned long long)nblk);  // 32 steps x 64 lanes
    __syncthreads();
}

// One workgroup per row of the work list.
template <int kWaves, int kG, bool kCheck>
__global__ __launch_bounds__(64 * kWaves) void k_op_sdem_bits(const SecDesc* __restrict__ secs,
                                                              const RowWork* __restrict__ work,
                                                              const float* __restrict__ in4,
                                                              const int* __restrict__ target,
                                                              const float* __restrict__ weight,
                                                              const uint32_t* __restrict__ fl,
                                                              const float* __restrict__ Sbuf,
                                                              const float4* __restrict__ rtab, float povh,
                                                              float* __restrict__ arena, int pools,
                                                              unsigned long long* __restrict__ steps) {
    extern __shared__ double lds8[];
    __shared__ int gnext;
    sdem_bits_row<kWaves, kG, kCheck>(work[blockIdx.x], secs, in4, target, weight, fl, Sbuf, rtab, povh, arena,
                              reinterpret_cast<char*>(lds8), pools, steps, &gnext);
}

// Rows past 4096 cells (see flush_runs), one workgroup per row.  Bound by VALU,
// like the shorter rows.  Eight waves share a staged row and its tables (18 KB
// and 6 KB at 4600 cells, 64 and 17 KB at the longest).  Twelve sectors
// of a 4600^2 DEM: 256 ms with every step of every scan (k_op_sdem), 32 ms
// here.
constexpr int kLongWaves = 8;
__global__ __launch_bounds__(64 * kLongWaves) void k_op_sdem_long(
    const SecDesc* __restrict__ secs, const RowWork* __restrict__ work, const float* __restrict__ in4,
    const int* __restrict__ target, const float* __restrict__ weight, const uint32_t* __restrict__ fl,
    const float* __restrict__ Sbuf, const float4* __restrict__ rtab, float povh, float* __restrict__ arena,
    int pools, unsigned long long* __restrict__ steps) {
    extern __shared__ double lds8[];
    __shared__ int gnext;
    sdem_bits_row<kLongWaves, 4, true, true>(work[blockIdx.x], secs, in4, target, weight, fl, Sbuf, rtab, povh, arena,
                                       reinterpret_cast<char*>(lds8), pools, steps, &gnext);
}

static hipError_t launch_op_sdem_long(const DevPlan& p, const float* in4, const float* Sbuf, float* arena,
                                      const float4* rtab, float povh, unsigned long long* steps, hipStream_t s) {
    hipLaunchKernelGGL(k_op_sdem_long, dim3(p.nwork), dim3(64 * kLongWaves), sdem_long_lds(p.maxL, kLongWaves), s, p.secs, p.work,
                       in4, p.target, p.weight, p.fl, Sbuf, rtab, povh, arena, sdem_pools<true>(p.maxL, 4, kLongWaves), steps);
    return hipGetLastError();
}

// Persistent: a fixed grid pulls rows off the (cost-sorted) work list with
// an atomic counter until the list is exhausted; every workgroup exits once
// the counter passes nwork.  The counter is cleared by the launcher.
// kOcc > 1 asks the compiler for at least kOcc waves per SIMD (fewer VGPRs,
// less software pipelining of the LDS loads, more waves to hide latency).
template <int kWaves, int kOcc, int kG>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kOcc, 8))) void k_op_sdem_bits_persistent(
    const SecDesc* __restrict__ secs, const RowWork* __restrict__ work, int nwork, int* __restrict__ counter,
    const float* __restrict__ in4, const int* __restrict__ target, const float* __restrict__ weight,
    const uint32_t* __restrict__ fl, const float* __restrict__ Sbuf, const float4* __restrict__ rtab, float povh,
    float* __restrict__ arena, int pools, unsigned long long* __restrict__ steps) {
    extern __shared__ double lds8[];
    __shared__ int item, gnext;
    for (;;) {
        if (threadIdx.x == 0) item = atomicAdd(counter, 1);
        __syncthreads();
        const int it = __builtin_amdgcn_readfirstlane(item);  // the same value in every lane
        __syncthreads();  // every lane has read `item` before thread 0 overwrites it
        if (it >= nwork) break;
        sdem_bits_row<kWaves, kG, false>(work[it], secs, in4, target, weight, fl, Sbuf, rtab, povh, arena,
                                  reinterpret_cast<char*>(lds8), pools, steps, &gnext);
    }
}

__global__ void k_zero_int(int* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

hipError_t launch_op_sdem_tuned(const DevPlan& p, const float* in4, const float* Sbuf, float* arena,
                                const float4* rtab, float povh, const SdemTuning& t, int* counter,
                                unsigned long long* steps, hipStream_t s) {
    if (p.nwork == 0) return hipSuccess;
    if (p.maxL > 32 * kChunksMax) return launch_op_sdem_long(p, in4, Sbuf, arena, rtab, povh, steps, s);
    const int G = t.group > 1 ? 4 : 1;
    const int W = t.waves == 2 || t.waves == 8 ? t.waves : 4;
    const size_t lds = sdem_bits_lds(p.maxL, G, W);
    const int pools = sdem_pools<false>(p.maxL, G, W);
    if (t.persistent_wgs_per_cu > 0 && counter && !t.check) {
        int dev = 0, ncu = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, s, counter, 1);
        const int grid = std::min(p.nwork, ncu * t.persistent_wgs_per_cu);
#define SKE_PERS(W, O, G)                                                                                        \
    hipLaunchKernelGGL((k_op_sdem_bits_persistent<W, O, G>), dim3(grid), dim3(64 * W), lds, s, p.secs, p.work,    \
                       p.nwork, counter, in4, p.target, p.weight, p.fl, Sbuf, rtab, povh, arena, pools, steps)
#define SKE_PERS_W(O, G)                                                                                         \
    if (t.waves == 2) SKE_PERS(2, O, G); else if (t.waves == 8) SKE_PERS(8, O, G); else SKE_PERS(4, O, G)
#define SKE_PERS_G(O)                                                                                            \
    if (G == 4) { SKE_PERS_W(O, 4); } else { SKE_PERS_W(O, 1); }
        if (t.occupancy >= 8) {
            SKE_PERS_G(8);
        } else if (t.occupancy >= 6) {
            SKE_PERS_G(6);
        } else {
            SKE_PERS_G(1);
        }
#undef SKE_PERS_G
#undef SKE_PERS_W
#undef SKE_PERS
        return hipGetLastError();
    }
#define SKE_GRID(W, G, C)                                                                                         \
    hipLaunchKernelGGL((k_op_sdem_bits<W, G, C>), dim3(p.nwork), dim3(64 * W), lds, s, p.secs, p.work, in4, p.target, \
                       p.weight, p.fl, Sbuf, rtab, povh, arena, pools, steps)
#define SKE_GRID_W(G, C)                                                                                          \
    if (t.waves == 2) SKE_GRID(2, G, C); else if (t.waves == 8) SKE_GRID(8, G, C); else SKE_GRID(4, G, C)
    if (G == 4) {
        if (t.check) { SKE_GRID_W(4, true); } else { SKE_GRID_W(4, false); }
    } else {
        if (t.check) { SKE_GRID_W(1, true); } else { SKE_GRID_W(1, false); }
    }
#undef SKE_GRID_W
#undef SKE_GRID
    return hipGetLastError();
}

hipError_t launch_op_sdem(const DevPlan& p, const float* in4, const float* Sbuf, float* arena,
                          const float4* rtab, float povh, int variant, bool check, hipStream_t s) {
    if (variant == 0) {
        SdemTuning t;
        t.group = 1;
        t.check = check;
        return launch_op_sdem_tuned(p, in4, Sbuf, arena, rtab, povh, t, nullptr, nullptr, s);
    }
    if (p.nwork == 0) return hipSuccess;
    const size_t lds = sizeof(float) * (size_t)(p.maxL + 2 * kPad);
    if (variant == 1)
        hipLaunchKernelGGL(k_op_sdem<1>, dim3(p.nwork), dim3(256), lds, s, p.secs, p.work, in4, p.target,
                           p.weight, p.fl, Sbuf, rtab, povh, arena);
    else
        hipLaunchKernelGGL(k_op_sdem<0>, dim3(p.nwork), dim3(256), lds, s, p.secs, p.work, in4, p.target,
                           p.weight, p.fl, Sbuf, rtab, povh, arena);
    return hipGetLastError();
}

}  // namespace ske
