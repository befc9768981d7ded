// DIA x DIA SpGEMM numeric phase for contiguous bands: A holds every offset
// a0 .. a0 + nA - 1 and B every offset b0 .. b0 + nB - 1, both in ascending
// order (make_banded of spmspm/bench_spmspm.cu:89-106, gemm_diag's defaults
// of gemm_diag/gemm_diag.cu:467-486), so C holds c0 = a0 + b0 .. c0 + nA +
// nB - 2 and its k-th diagonal is
//
//   C(i, i + c0 + k) = sum over p of A(i, i + a0 + p) * B(m, m + b0 + k - p),
//   m = i + a0 + p,  0 <= p < nA,  0 <= k - p < nB
//
// The general kernels read one A and one B value from LDS or memory for
// every multiply-add.  Here the plan's structure is known, so a lane holds a
// register tile of C: RR consecutive rows by KT consecutive diagonals.  For
// the RR rows m = base + RR g + t (t = 0 .. RR - 1) of B, the RR rows and KT
// diagonals of the tile need KT + 2 RR - 2 diagonals of B (one RR-wide LDS
// read each) and 2 RR - 1 diagonals of A, for RR RR KT multiply-adds.
//
// A workgroup stages a block of 64 RR rows: A's rows and, for every B
// diagonal, the window of rows that A's offsets reach, with direct
// global-to-LDS loads, and one row of zeros behind each operand.  Wave w then
// computes the k-tile w of every row of the block.  The p of each C value run
// downwards, which is the plan's order (B ascending), one fused multiply-add
// each: the bits of the gather kernel, but for the sign of a zero that
// underflow makes (below).  At the ends of a tile's p range some
// of a group's p or q lie outside [0, nA) or [0, nB): those read the row of
// zeros, and A elements that do not exist (rows m outside [0, n)) are staged
// as zeros, so every group runs the same straight-line code; a product with
// a zero leaves its sum as it is unless the other factor is infinite or NaN,
// which is found afterwards and formed again term by term, or the sum is -0.
// Sums start at +0, and only a negative product below half the smallest
// denormal makes one -0; a product that is +0 then makes it +0, where the
// gather, which has no such product, keeps -0.  No other value depends on it.
// (With the ends' terms behind uniform branches the kernel took 34 us instead
// of 19 on the first shape below.)
//
// What bounds it: at 33 x 33 diagonals and n = 100000 LDS reads (21 of 16
// bytes for 128 multiply-adds per lane at RR = 4, KT = 8) and the one round
// of staging, evaluation and stores that so few rows give; on long bands of
// 15 x 15 and less the memory rate.  Measured (us, rotated sets, the general
// kernels -> this one):
//   fp32  33 x 33: n = 100003 24.0 -> 15.6, 2^20 245 -> 130;  49 x 49: 2^20
//         465 -> 223;  21 x 21: 4096 6.3 -> 4.8, 100003 14.1 -> 11.9, 2^20
//         99 -> 84;  15 x 15: 300007 19.7 -> 18.0
//   complex  33 x 33: n = 100003 71 -> 37;  25 x 25: 10^6 404 -> 178;  7 x 7:
//         10^6 56 -> 43
// Two k-tiles per wave (half the waves) lost 5 to 25 % everywhere.
#include <climits>

#include "common.hpp"
#include "elem.hpp"

namespace diagpu {
namespace {

constexpr size_t kLdsMax = 160 * 1024;

// m + 0 * v: NaN from the first v that is not finite on
__device__ __forceinline__ float mark_(float v, float z, float m) { return fma_(v, z, m); }
__device__ __forceinline__ float mark_(cf32 v, float z, float m) { return fma_(v.im, z, fma_(v.re, z, m)); }

template <typename T, int RR> struct alignas(RR * sizeof(T)) Rows { T v[RR]; };

// Rows of a B window: the block's rows, plus what A's nA offsets and the
// last lane's RR-wide read reach (nA <= kMaxA).  A constant, so that every
// B read of a group is one base and an immediate offset.
constexpr int kReach = 68;
template <int RR> struct Full {
    static constexpr int kRB = 64 * RR;
    static constexpr int kWB = kRB + kReach;
    static constexpr int kMaxA = kReach - RR + 2;
    static constexpr size_t lds(int nA, int nB, size_t size)
    {
        return ((size_t)(nA + 1) * kRB + (size_t)(nB + 1) * kWB) * size;
    }
};

// One diagonal's window rows [w0, w0 + rows), rows <= MAXR, into dst: dword f
// of the window by lane f mod 64; positions clamped into the diagonal (an
// always valid address).
template <typename T, int MAXR>
__device__ __forceinline__ void stage_diag(const T* __restrict__ vals, int64_t start, int off, int n,
                                           int w0, int rows, T* dst, int lane)
{
    constexpr int kWords = (int)(sizeof(T) / 4);
    const int top = n - 1 - (off < 0 ? -off : off), lo = w0 + (off < 0 ? off : 0);
    const float* src = reinterpret_cast<const float*>(vals + start);
    float* d = reinterpret_cast<float*>(dst);
#pragma unroll
    for (int f0 = 0; f0 < MAXR * kWords; f0 += 64) {
        if (f0 >= rows * kWords) break;
        const int f = f0 + lane;
        if (f < rows * kWords) {
            const uint32_t pos = (uint32_t)min(max(lo + f / kWords, 0), top);
            __builtin_amdgcn_global_load_lds(src + (uint64_t)pos * kWords + f % kWords, d + f0, 4, 0,
                                             0);
        }
    }
}

template <typename T, int RR, int KT>
__global__ __launch_bounds__(1024) void k_full(
    int32_t n, int32_t a0, int32_t nA, const int64_t* __restrict__ A_starts,
    const T* __restrict__ Av, int32_t b0, int32_t nB, const int64_t* __restrict__ B_starts,
    const T* __restrict__ Bv, const int64_t* __restrict__ C_starts, T* __restrict__ Cv,
    int32_t blocks, int32_t groups, int32_t per_xcd, int32_t tiles)
{
    typedef Full<RR> F;
    typedef Rows<T, RR> V;
    constexpr int kRB = F::kRB, kWB = F::kWB;
    extern __shared__ __align__(16) char lds_raw[];
    T* A_l = reinterpret_cast<T*>(lds_raw);          // [nA + 1][kRB], the last row zero
    T* B_l = A_l + (int64_t)(nA + 1) * kRB;          // [nB + 1][kWB], window rows from i0 + a0
    // each XCD owns a contiguous range of blocks: neighbours share its L2
    const int unit = (int)(blockIdx.x % kNumXcd) * per_xcd + (int)(blockIdx.x / kNumXcd);
    if (unit >= blocks * groups) return;
    const int blk = unit / groups, grp = unit % groups;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nw = (int)(blockDim.x >> 6);
    const int i0 = blk * kRB;

    // stage A and B, kS diagonals' starts (scalar loads) ahead of their rows
    constexpr int kS = 4;
    const int wrows = kRB + nA + RR - 2;
    for (int d0 = wave * kS; d0 < nA + nB; d0 += nw * kS) {
        int64_t st[kS];
#pragma unroll
        for (int u = 0; u < kS; ++u) {
            const int d = min(d0 + u, nA + nB - 1);
            st[u] = d < nA ? at_byte(A_starts, (uint32_t)d << 3)
                           : at_byte(B_starts, (uint32_t)(d - nA) << 3);
        }
#pragma unroll
        for (int u = 0; u < kS; ++u) {
            const int d = d0 + u;
            if (d < nA)
                stage_diag<T, kRB>(Av, st[u], a0 + d, n, i0, kRB, A_l + d * kRB, lane);
            else if (d < nA + nB)
                stage_diag<T, kWB>(Bv, st[u], b0 + d - nA, n, i0 + a0, wrows,
                                   B_l + (d - nA) * kWB, lane);
        }
    }
    for (int f = (int)threadIdx.x; f < kRB; f += 64 * nw) A_l[nA * kRB + f] = zero_of<T>();
    for (int f = (int)threadIdx.x; f < kWB; f += 64 * nw) B_l[nB * kWB + f] = zero_of<T>();
    __builtin_amdgcn_s_waitcnt(0);   // this wave's direct loads have landed in LDS
    __syncthreads();
    // Rows i whose A element (i, i + da) does not exist: zero.
    const bool inside = i0 + a0 >= 0 && i0 + kRB - 1 + a0 + nA - 1 < n;
    if (!inside) {
        for (int e = (int)threadIdx.x; e < nA * kRB; e += 64 * nw) {
            const int m = i0 + a0 + e / kRB + e % kRB;
            if (m < 0 || m >= n) A_l[e] = zero_of<T>();
        }
        __syncthreads();
    }

    const int tile = grp * nw + wave;
    if (tile >= tiles) return;
    const int nC = nA + nB - 1, k0 = tile * KT;
    int64_t cst[KT];   // C starts (scalar loads), wanted at the end
#pragma unroll
    for (int k = 0; k < KT; ++k) cst[k] = at_byte(C_starts, (uint32_t)min(k0 + k, nC - 1) << 3);
    T acc[RR][KT];
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
        for (int k = 0; k < KT; ++k) acc[r][k] = zero_of<T>();

    // p of the tile's terms: [plo, phi]; group g covers p in [RR g - (RR - 1),
    // RR g + RR - 1], so both ends' groups cover them all
    const int plo = max(0, k0 - (nB - 1)), phi = min(nA - 1, k0 + KT - 1);
    const int ghi = (phi + RR - 1) / RR, glo = plo / RR;
    constexpr int NJ = KT + 2 * RR - 2, NU = 2 * RR - 1;
    auto fmas = [&](const V (&av)[NU], const V (&bv)[NJ]) {
        // j ascending visits, for each (row, diagonal) of the tile, t and so
        // p downwards
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int t = RR - 1; t >= 0; --t)
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    const int k = j + t - r - (RR - 1);
                    if (k >= 0 && k < KT)
                        acc[r][k] = mad(acc[r][k], av[t - r + RR - 1].v[r], bv[j].v[t]);
                }
    };
    const T* A_r = A_l + RR * lane;
    const T* B_r = B_l + RR * lane;
    auto padded = [&](int g) {
        V av[NU], bv[NJ];
        const int p0 = RR * g - (RR - 1), q0 = k0 - RR * g - (RR - 1);
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int p = (uint32_t)(p0 + u) < (uint32_t)nA ? p0 + u : nA;
            av[u] = *reinterpret_cast<const V*>(A_r + p * kRB);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int q = (uint32_t)(q0 + j) < (uint32_t)nB ? q0 + j : nB;
            bv[j] = *reinterpret_cast<const V*>(B_r + q * kWB + RR * g);
        }
        fmas(av, bv);
    };
    int g = ghi;
    // whole groups: every p in [0, nA), every q in [0, nB)
    const int g1 = min(min((nA - RR) / RR, (k0 - (RR - 1)) / RR), ghi);
    const int g0 = max(max(1, (k0 + KT - 1 + RR - 1 - (nB - 1) + RR - 1) / RR), glo);
    if (k0 - (RR - 1) < 0 || nA < RR || g0 > g1) {
        for (; g >= glo; --g) padded(g);
    } else {
        for (; g > g1; --g) padded(g);
        const T* ap = A_r + (RR * g - (RR - 1)) * kRB;
        const T* bp = B_r + (k0 - RR * g - (RR - 1)) * kWB + RR * g;
        for (; g >= g0; --g) {
            V av[NU], bv[NJ];
#pragma unroll
            for (int u = 0; u < NU; ++u) av[u] = *reinterpret_cast<const V*>(ap + u * kRB);
#pragma unroll
            for (int j = 0; j < NJ; ++j) bv[j] = *reinterpret_cast<const V*>(bp + j * kWB);
            fmas(av, bv);
            ap -= RR * kRB;
            bp += RR * kWB - RR;
        }
        for (; g >= glo; --g) padded(g);
    }

    // The padding's products are 0 times a staged value.  Where that value is
    // infinite or NaN the sum turns NaN; a sum that stayed finite met none.  A
    // wave with a sum that is not finite forms its tile again term by term.
    // (One fused multiply-add per sum; per-sum classes cost 23 more registers
    // at RR = 4 and 15.6 -> 19 us on 33 x 33, n = 100000.)
    float zero = 0.f;
    asm volatile("" : "+v"(zero));   // not a constant to fold
    float mark = 0.f;
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
        for (int k = 0; k < KT; ++k) mark = mark_(acc[r][k], zero, mark);
    const bool finite = mark == 0.f;
    const int c0 = a0 + b0;
    if (__builtin_expect(__ballot(!finite) != 0, 0)) {
        for (int k = k0; k < min(k0 + KT, nC); ++k) {
            const int dc = c0 + k;
            T* cp = Cv + at_byte(C_starts, (uint32_t)k << 3) + (dc < 0 ? dc : 0);
            for (int row = lane; row < kRB; row += 64) {
                const int i = i0 + row;
                if (i >= n || i + dc < 0 || i + dc >= n) continue;
                T sum = zero_of<T>();
                for (int p = min(nA - 1, k); p >= max(0, k - (nB - 1)); --p) {
                    const int m = i + a0 + p;
                    if (m >= 0 && m < n)
                        sum = mad(sum, A_l[p * kRB + row], B_l[(k - p) * kWB + row + p]);
                }
                cp[i] = sum;
            }
        }
        return;
    }

    // C: RR consecutive values per lane and diagonal
    const int i = i0 + RR * lane;
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        if (k0 + k >= nC) break;
        const int dc = c0 + k0 + k;
        T* cp = Cv + cst[k] + (dc < 0 ? dc : 0);
        if (i0 + kRB <= n && i0 + dc >= 0 && i0 + kRB + dc <= n) {
            typedef float vec __attribute__((ext_vector_type(RR * (int)sizeof(T) / 4), aligned(4)));
            vec q;
            T row[RR];
#pragma unroll
            for (int r = 0; r < RR; ++r) row[r] = acc[r][k];
            __builtin_memcpy(&q, row, sizeof(q));
            __builtin_nontemporal_store(q, reinterpret_cast<vec*>(cp + i));
        } else {
#pragma unroll
            for (int r = 0; r < RR; ++r)
                if (i + r < n && i + r + dc >= 0 && i + r + dc < n) cp[i + r] = acc[r][k];
        }
    }
}

// Rows per lane and diagonals per tile of a launch.
enum FullKind : int { kNone = 0, k1x4, k2x4, k2x6, k2x8, k4x8 };

bool fits(FullKind kind, int nA, int nB, size_t size)
{
    switch (kind) {
    case k1x4: return nA <= Full<1>::kMaxA && Full<1>::lds(nA, nB, size) <= kLdsMax;
    case k2x4:
    case k2x6:
    case k2x8: return nA <= Full<2>::kMaxA && Full<2>::lds(nA, nB, size) <= kLdsMax;
    case k4x8: return nA <= Full<4>::kMaxA && Full<4>::lds(nA, nB, size) <= kLdsMax;
    default: return false;
    }
}

// The form a launch takes (kNone: the operands do not fit in LDS).  Few rows:
// small blocks, so that more workgroups share the work (21 x 21, n = 4096:
// 4.8 us at 1 x 4, 6.8 at 2 x 8, 9.0 at 4 x 8), as long as every CU gets at
// most one workgroup, 256 blocks of 64 rows, or two of few waves (fp32 33 x
// 33 at n = 16000: 8.1 us at 1 x 4, 8.5 at 2 x 8, at 17000 10.2 and 8.5, 33 x
// 19 at 17000 7.7 and 8.2; complex 15 x 15 at 18000 6.3 at 1 x 4 and at 2 x 4,
// 21 x 21 8.0 and 7.4, 11 x 11 5.4 and 5.8, at 26000 5.7 and 5.8, 21 x 11 at
// 26000 6.9 and 6.7, 9 x 9 at 40000 5.9 and 6.5, at 55000 7.0 and 6.5).
// fp32 above: 2 x 8, and 4 x 8 where the LDS reads bound it (about 14 entries
// per C diagonal) and two workgroups still fit a CU (33 x 33, n = 100003: 17.6
// against 15.6; 17 x 17, n = 200003: 15.6 against 17.0).  Complex values: 2 x
// 4 for short tiles (11 x 11, n = 300007: 19.9 us, 23.0 at 2 x 6) and, up to
// 32768 rows, where one workgroup holds all tiles (64 C diagonals; 29 x 11 at
// 26000 7.2 us, 8.3 at 2 x 6, 33 x 33 at 24000 16.3 and 10.6), 2 x 6 above
// (33 x 33, n = 100003: 50.8 at 2 x 4, 37.4 at 2 x 6, 42.5 at 2 x 8).
FullKind full_kind(int32_t n, int nA, int nB, bool cplx)
{
    const size_t size = cplx ? sizeof(cf32) : sizeof(float);
    const int64_t pairs = (int64_t)nA * nB, nC = nA + nB - 1;
    FullKind kind;
    if (n <= 16384 || (n < 20000 && nC <= (cplx ? 32 : 52)) || (cplx && n <= 32768 && nC <= 24))
        kind = k1x4;
    else if (cplx)
        kind = pairs < 6 * nC || (n <= 32768 && nC <= 64) ? k2x4 : k2x6;
    else
        kind = n >= 65536 && pairs >= 14 * nC && Full<4>::lds(nA, nB, size) <= 80 * 1024 ? k4x8 : k2x8;
    if (!fits(kind, nA, nB, size)) kind = k1x4;
    return fits(kind, nA, nB, size) ? kind : kNone;
}

// Tenths of an entry per C diagonal from which this kernel is the faster one
// (us, the general kernels against this one; -1: never).
int full_tenths(int32_t n, int nA, int nB, bool cplx)
{
    const int nC = nA + nB - 1;
    // the gather: fp32 5 x 5 (2.8) at n = 2000 5.8 / 3.3, complex 3 x 37 (2.9)
    // 5.4 / 4.4 (the exceptions are complex 5 x 49, 37 x 5 and 49 x 5, 0.89 to
    // 0.96 of the general kernel's rate)
    if (n < 4096) return 25;
    if (cplx) {
        // 5 x 5 (2.8) at n = 5000 4.2 / 3.7; 3 x 49 (2.9) 4.7 / 5.0
        if (n <= 10000) return 25;
        // Each wave of the A-stationary kernel takes one C diagonal, and its
        // blocks of 256 rows (with 32 before them) are one round of
        // workgroups: 7 x 7 (3.8) at n = 33000 4.9 / 5.4, 55000 5.1 / 5.6, 9 x
        // 7 (4.2) 5.6 / 6.0; past one of the two 9 x 9 (4.8) at 55000 9.0 /
        // 6.5, 7 x 7 at 65535 6.8 / 5.7
        if (nC <= 16 && n > 32768 && n <= 65536 - 32) return -1;
        // 5 x 5 (2.8) at n = 100003 5.1 / 5.6; 7 x 7 (3.8) 7.0 / 6.9, 24000
        // 4.9 / 4.4, 10^6 56 / 43; 5 x 21 (4.2) at 18000 5.6 / 5.4 (5 x 37, 4.5,
        // loses up to 40000: 5.9 / 6.3 at 18000, 8.4 / 9.0 at 40000)
        return 35;
    }
    // 7 x 7 (3.8) at 100003 4.4 / 6.4; 11 x 11 (5.8) at 300007 13.6 / 14.8; 33 x
    // 9 (7.2) at 491830 36.0 / 37.8; 21 x 11 (7.5) at 94475 9.1 / 9.5; 15 x 15
    // (7.8) at 300007 19.7 / 18.0, 100003 10.7 / 9.5
    if (n >= 65536) return 76;
    // more than 64 C diagonals are two workgroups per 64 rows, from 8192 rows
    // on more than one per CU: 21 x 49 (14.9) at n = 9999 7.6 / 8.0, 17 x 49
    // (12.8) at 12500 6.8 / 7.5, 33 x 33 (16.8) 9.3 / 8.0; at 15000, where the
    // A-stationary kernel takes a second round, 21 x 49 9.0 / 8.3
    if (nC > 64 && n > 8192 && n < 15000) return 150;
    // 21 x 21 (10.8) at n = 20000 6.2 / 7.0; 17 x 39 (12.1) 8.7 / 7.7; 33 x 25
    // (14.5) at 30011 11.5 / 8.5
    if (n > 10000) return 120;
    // latency: a launch's waves grow with the C diagonals, the general
    // kernels' time with the entries.  At n = 4200: 5 x 5 (2.8) 3.4 / 3.3, 7 x 5
    // (3.2) 3.3 / 3.5, 3 x 29 (2.8) 3.5 / 3.7, 7 x 7 (3.8) 3.6 / 3.5, 5 x 29
    // (4.4) 3.9 / 3.8; 5 x 37 (4.5) 3.9 / 4.3, 3 x 49 (2.9) 3.5 / 4.7, 7 x 37
    // (6.0) 4.3 / 4.5, 37 x 7 4.9 / 4.8, 9 x 37 (7.4) 4.8 / 4.5
    return nC <= 9 ? 25 : nC <= 36 ? 33 : nB > nA ? 70 : 60;
}

template <typename T, int RR, int KT>
int launch(const char* fn, int32_t n, int32_t a0, int32_t nA, const int64_t* A_starts,
           const T* A_vals, int32_t b0, int32_t nB, const int64_t* B_starts, const T* B_vals,
           const int64_t* C_starts, T* C_vals, void* stream)
{
    typedef Full<RR> F;
    const int tiles = ceil_div(nA + nB - 1, KT);
    const int blocks = (int)ceil_div<int64_t>(n, F::kRB);
    const int groups = ceil_div(tiles, 16);      // workgroups of at most 16 waves
    const int W = ceil_div(tiles, groups);
    const int64_t per_xcd = ceil_div<int64_t>((int64_t)blocks * groups, kNumXcd);
    if (per_xcd * kNumXcd > INT_MAX)
        return fail(DIAGPU_ERR_CAPACITY, "%s: %lld workgroups", fn, (long long)(per_xcd * kNumXcd));
    // more than 64 KiB of dynamic LDS must be allowed explicitly
    const int st = check_hip(hipFuncSetAttribute((const void*)k_full<T, RR, KT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)kLdsMax), fn);
    if (st) return st;
    hipLaunchKernelGGL((k_full<T, RR, KT>), dim3((unsigned)(per_xcd * kNumXcd)), dim3(64 * W),
                       F::lds(nA, nB, sizeof(T)), as_stream(stream), n, a0, nA, A_starts, A_vals,
                       b0, nB, B_starts, B_vals, C_starts, C_vals, blocks, groups, (int32_t)per_xcd,
                       tiles);
    return check_launch(fn);
}

// Whether offsets d0 .. d0 + cnt - 1 lie inside (-n, n).
bool inside_n(int32_t n, int64_t d0, int64_t cnt)
{
    return d0 > -(int64_t)n && d0 + cnt - 1 < n;
}

template <typename T>
int run_full(const char* fn, int32_t n, int32_t a0, int32_t nA, const int64_t* A_starts,
             const T* A_vals, int32_t b0, int32_t nB, const int64_t* B_starts, const T* B_vals,
             const int64_t* C_starts, int64_t c_ndiag, T* C_vals, void* stream)
{
    if (n < 1 || n > (1 << 30) || nA < 1 || nB < 1)
        return fail(DIAGPU_ERR_ARG, "%s: need 1 <= n <= 2^30 and nA, nB >= 1", fn);
    if (!inside_n(n, a0, nA) || !inside_n(n, b0, nB) ||
        !inside_n(n, (int64_t)a0 + b0, (int64_t)nA + nB - 1) || c_ndiag != (int64_t)nA + nB - 1)
        return fail(DIAGPU_ERR_ARG,
                    "%s: offsets outside (-n, n), or c_ndiag is not nA + nB - 1", fn);
    if (!A_starts || !A_vals || !B_starts || !B_vals || !C_starts || !C_vals)
        return fail(DIAGPU_ERR_ARG, "%s: a pointer is NULL", fn);
#define DIAGPU_FULL(RR, KT)                                                                     \
    return launch<T, RR, KT>(fn, n, a0, nA, A_starts, A_vals, b0, nB, B_starts, B_vals, C_starts, \
                             C_vals, stream)
    const FullKind kind = full_kind(n, nA, nB, sizeof(T) == sizeof(cf32));
    if (kind == k1x4) DIAGPU_FULL(1, 4);
    if constexpr (sizeof(T) == sizeof(cf32)) {
        if (kind == k2x4) DIAGPU_FULL(2, 4);
        if (kind == k2x6) DIAGPU_FULL(2, 6);
    } else {
        if (kind == k2x8) DIAGPU_FULL(2, 8);
        if (kind == k4x8) DIAGPU_FULL(4, 8);
    }
#undef DIAGPU_FULL
    return fail(DIAGPU_ERR_CAPACITY, "%s: %d x %d diagonals do not fit in LDS", fn, nA, nB);
}

}  // namespace
}  // namespace diagpu

extern "C" {

DIAGPU_API int diagpu_spgemm_full_choice(int32_t n, int32_t nA, int32_t nB, int64_t c_ndiag,
                                         int64_t n_pairs, const diagpu_spgemm_shape* shape,
                                         int32_t complex_values)
{
    using namespace diagpu;
    if (!shape || !shape->contiguous || n < 1 || nA < 1 || nB < 1 || nA > 4096 || nB > 4096)
        return 0;
    const int64_t nC = (int64_t)nA + nB - 1, pairs = (int64_t)nA * nB;
    // every sum of offsets inside (-n, n)
    if (c_ndiag != nC || n_pairs != pairs || !inside_n(n, shape->a_off_min, nA) ||
        !inside_n(n, shape->b_off_min, nB) ||
        !inside_n(n, (int64_t)shape->a_off_min + shape->b_off_min, nC))
        return 0;
    if (full_kind(n, nA, nB, complex_values != 0) == kNone) return 0;
    const int tenths = full_tenths(n, nA, nB, complex_values != 0);
    return tenths >= 0 && 10 * pairs >= tenths * nC ? 1 : 0;
}

DIAGPU_API int diagpu_spgemm_numeric_full_f32(int32_t n, int32_t a_off_min, int32_t nA,
                                              const int64_t* A_starts, const float* A_vals,
                                              int32_t b_off_min, int32_t nB,
                                              const int64_t* B_starts, const float* B_vals,
                                              const int64_t* C_starts, int64_t c_ndiag,
                                              float* C_vals, void* stream)
{
    return diagpu::run_full<float>("diagpu_spgemm_numeric_full_f32", n, a_off_min, nA, A_starts,
                                   A_vals, b_off_min, nB, B_starts, B_vals, C_starts, c_ndiag,
                                   C_vals, stream);
}

DIAGPU_API int diagpu_spgemm_numeric_full_c64(int32_t n, int32_t a_off_min, int32_t nA,
                                              const int64_t* A_starts,
                                              const diagpu_complex64* A_vals, int32_t b_off_min,
                                              int32_t nB, const int64_t* B_starts,
                                              const diagpu_complex64* B_vals,
                                              const int64_t* C_starts, int64_t c_ndiag,
                                              diagpu_complex64* C_vals, void* stream)
{
    using diagpu::cf32;
    return diagpu::run_full<cf32>("diagpu_spgemm_numeric_full_c64", n, a_off_min, nA, A_starts,
                                  reinterpret_cast<const cf32*>(A_vals), b_off_min, nB, B_starts,
                                  reinterpret_cast<const cf32*>(B_vals), C_starts, c_ndiag,
                                  reinterpret_cast<cf32*>(C_vals), stream);
}

}  // extern "C"
