// DIA SpMV on the column-indexed Recon layout, gfx950.
//
//   y[r] = sum_k [0 <= r + d_k < lim] Recon[k][r + d_k] * x[r + d_k],
//   lim = min(cols, x_size)
//
// (spmv/src/dia_reconstruct.cuh:22, bounds as in
// spmv/src/tc_spmv_regdirect_kernel.cu:85-104).  The reference lifts the band
// to a TF32 MMA and keeps 1/16 of the product; here the sum is what it is, an
// HBM stream: every useful value is read once and fused into its row's
// accumulator.
//
// Element types.  One kernel family serves real fp32 and fp64, complex64
// matrices with complex64 vectors, and real fp32 matrices with complex64
// vectors (a real Hamiltonian applied to a complex state: the matrix is read
// once for both parts of x).  A lane owns R rows, R times the wider of the
// two elements being 16 bytes: its x and y runs are 16 bytes, its value run
// 16 bytes (8 for a real matrix with complex vectors, where 32-byte x runs
// would leave every 16-byte x load half coalesced).
//
// Mapping.  A workgroup of 256 lanes owns a tile of 256 x R consecutive rows.
// For diagonal k the lane needs Recon[k][r+d_k ..] and x[r+d_k ..]: runs at
// the same column, loaded as 16-byte vectors (dword aligned: gfx950 serves
// unaligned global loads); the 64 lanes of a wave cover 1 KiB of each
// stream.  Value loads and the y store are non-temporal: each value is used
// once, while x stays in L2 for the tiles that re-read it.
//
// Memory-level parallelism.  What bounds this kernel is how many HBM bytes
// each CU keeps in flight, not the x re-reads or the misalignment (measured:
// a 64-stream read with the same offsets and no x runs at 80% of 8 TB/s, and
// adding the x loads costs 3 points).  So loads are never drained in chunks:
// the ring kernel keeps W diagonals' loads in flight per lane at all times --
// step j consumes slot j and refills it with the diagonal W ahead, and
// sched_barrier pins that order so the compiler emits a steady vmcnt window
// instead of hoisting or sinking the loads.  Offsets come through the scalar
// cache (the compiler batches them into s_load_dwordx4/x2), which does not
// queue behind the HBM stream, so one ring runs over all K diagonals with no
// drain anywhere (measured against 64 offsets per VGPR broadcast by
// readlane, with a refill of that VGPR every 64 diagonals: 1.7 points of
// 8 TB/s on config 3's 64 diagonals, about 1 point at 85 and 377).  For
// K <= 16 the short kernel issues all 2K loads straight-line.  Where the rows
// are too few to fill the chip with waves, several waves share a tile and
// split its diagonals (spmv_split_kernel).
//
// Edge tiles.  A tile whose rows or columns leave the matrix for some
// diagonal runs the same ring, still with 16-byte runs, each loaded at its
// start column clamped into [0, lim - R] (always a valid run), and masked
// accumulation: no branch around a load, so the loads pipeline like the
// interior ones.  A lane whose run straddles column 0 or lim finds its
// in-range elements inside the clamped run, shifted by (start - clamped
// start), and picks them out with selects; lanes wholly out of range all load
// the same clamped run (one cache line per wave) and mask every term.  This
// keeps an edge tile about as fast as an interior one, which matters when
// the offset spread is a sizeable part of n (a propagator with hundreds of
// diagonals spread over +-10^5 rows has a fifth of its tiles at the edges,
// all on the XCDs that own the first and last rows).  Only a matrix
// narrower than one run (lim < R) falls back to per-element loads at
// clamped columns.  An edge tile is also dispatched early (odd XCDs walk
// their row range from the end).
//
// XCD awareness: workgroup b runs on XCD b mod 8; tiles are remapped so each
// XCD owns one contiguous eighth of the rows.  x[c] is used by rows c - d_k
// of every diagonal, i.e. by this tile and by tiles up to max|d_k| rows away,
// which then sit on the same XCD and find x in its L2.
//
// Dot epilogue (Krylov drivers).  With DOT, each workgroup also forms
// sum_r Re(conj(x[r]) * y[r]) over its rows in fp64 and stores it as one
// partial; a one-workgroup kernel launched next adds the partials in tile
// order (a deterministic result).
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "elem.hpp"
#include "reduce.hpp"
#include "spmv_internal.hpp"

namespace diagpu {
namespace {

constexpr int kBlock = 256;
constexpr int kShortMax = 16;   // K <= kShortMax: straight-line kernel
constexpr int kSplitChunk = 8;   // split kernel: diagonals whose loads a wave issues at once

// Per (matrix element, vector element) pair: rows per lane and ring depths,
// chosen so the kernels stay within 64 VGPRs (8 waves per SIMD).
template <typename TV, typename TX> struct Shape {
    // 16 bytes of the wider of the two elements: a real matrix applied to a
    // complex vector takes 2 rows per lane (8-byte value runs), so that every
    // x load and y store is a fully coalesced 16-byte run.
    static constexpr int R = (int)(16 / (sizeof(TV) > sizeof(TX) ? sizeof(TV) : sizeof(TX)));
    static constexpr int W = 6;    // interior ring
    static constexpr int WR = 4;   // edge ring
    static constexpr int TILE = kBlock * R;
};

// ---------------------------------------------------------------------------
// Shared pieces
// ---------------------------------------------------------------------------

// Tile index of workgroup b: XCD x = b mod 8 owns tiles [x*per_xcd,
// (x+1)*per_xcd); even XCDs walk their range upwards, odd ones downwards, so
// the last tile of the matrix (an edge tile) is among the first dispatched.
inline __device__ int tile_of_block(int per_xcd)
{
    const int x = (int)(blockIdx.x % kNumXcd);
    const int l = (int)(blockIdx.x / kNumXcd);
    return x * per_xcd + ((x & 1) ? per_xcd - 1 - l : l);
}

// min and max of a group of offsets held one per lane (lanes >= gn hold a
// copy of a valid offset), uniform across the wave.
inline __device__ void wave_minmax(int v, int& lo, int& hi)
{
    int a = v, b = v;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const int oa = __shfl_xor(a, s);
        const int ob = __shfl_xor(b, s);
        a = oa < a ? oa : a;
        b = ob > b ? ob : b;
    }
    lo = __builtin_amdgcn_readfirstlane(a);
    hi = __builtin_amdgcn_readfirstlane(b);
}

// How a group's loads treat columns outside [0, lim).
enum EdgeMode {
    kInterior = 0,   // the whole tile is in range: plain 16-byte runs
    kEdgeRun = 1,    // 16-byte runs at clamped starts, shifted and masked
};

// The gn diagonals with offsets `offs` (read with uniform indices: scalar
// loads) and values `vg` (Recon rows) accumulated into `acc` for the lane's R
// rows starting at row `r`.  W diagonals' loads in flight; every index is
// clamped to [0, gn) so all loads are valid, and the slots past the end are
// masked.  kEdgeRun needs lim >= R and masks every term whose column is
// outside [0, lim).
// With LG > 0 the diagonals [gn w / S, gn (w + 1) / S), S = 2^LG, make one sum
// each, and these are added in order of w: the split kernel's sums, bit for
// bit (the first is added to -0, which leaves it as it is).
template <typename TV, typename TX, int W, int MODE, int LG = 0>
__device__ __forceinline__ void ring_group(int64_t r, int64_t cols, int64_t lim, int gn,
                                           const int32_t* __restrict__ offs,
                                           const TV* __restrict__ vg, const TX* __restrict__ x,
                                           Run<TX, Shape<TV, TX>::R>& acc)
{
    constexpr int R = Shape<TV, TX>::R;
    Run<TX, R> sum;
    int w = 1, next = gn >> LG;   // next: sum w's first diagonal
    if constexpr (LG > 0) {
#pragma unroll
        for (int e = 0; e < R; ++e) sum.v[e] = neg_zero_of<TX>();
    }
    Run<TV, R> a[W];
    Run<TX, R> b[W];
    // a run start clamped to a valid run, [0, lim - R] (kEdgeRun)
    auto clamp_run = [&](int64_t c) -> int64_t {
        const int64_t hi = lim - R;
        return c < 0 ? 0 : (c > hi ? hi : c);
    };
    auto issue = [&](int j, int k) {
        const int d = offs[k];
        const TV* vk = vg + (int64_t)k * cols;
        if constexpr (MODE == kInterior) {
            a[j] = load_run<TV, R, true>(vk + r + d);
            b[j] = load_run<TX, R, false>(x + r + d);
        } else {
            const uint32_t cc = (uint32_t)clamp_run(r + d);
            a[j] = load_run<TV, R, true>(vk + cc);
            b[j] = load_run<TX, R, false>(x + cc);
        }
    };
    // slot j holds diagonal k (k uniform); `on` = the slot is part of the group
    auto consume = [&](int j, int k, bool on) {
        if constexpr (LG > 0) {
            const bool ends = on && k == next;   // sum w - 1 is complete
#pragma unroll
            for (int e = 0; e < R; ++e) {
                sum.v[e] = sel(ends, add_(sum.v[e], acc.v[e]), sum.v[e]);
                acc.v[e] = sel(ends, zero_of<TX>(), acc.v[e]);
            }
            w += ends;
            next = (int)((int64_t)gn * w >> LG);
        }
        if constexpr (MODE == kInterior) {
#pragma unroll
            for (int e = 0; e < R; ++e)
                acc.v[e] = sel(on, mad(acc.v[e], a[j].v[e], b[j].v[e]), acc.v[e]);
        } else {
            const int64_t c = r + offs[k];
            // element e of the run sits at index e + s of what was loaded
            const int s = (int)(c - clamp_run(c));
#pragma unroll
            for (int e = 0; e < R; ++e) {
                const bool ok = on && (uint64_t)(c + e) < (uint64_t)lim;
                TV av = a[j].v[0];
                TX bv = b[j].v[0];
#pragma unroll
                for (int i = 1; i < R; ++i) {
                    const bool m = e + s == i;
                    av = sel(m, a[j].v[i], av);
                    bv = sel(m, b[j].v[i], bv);
                }
                acc.v[e] = sel(ok, mad(acc.v[e], av, bv), acc.v[e]);
            }
        }
    };

#pragma unroll
    for (int j = 0; j < W; ++j) issue(j, j < gn ? j : gn - 1);
    __builtin_amdgcn_sched_barrier(0);
    int k0 = 0;
    while (k0 + 2 * W <= gn) {   // every refill of this round is in range
#pragma unroll
        for (int j = 0; j < W; ++j) {
            consume(j, k0 + j, true);
            __builtin_amdgcn_sched_barrier(0);
            issue(j, k0 + W + j);
            __builtin_amdgcn_sched_barrier(0);
        }
        k0 += W;
    }
    // Last two rounds: slots hold k0 .. k0+W-1 (those >= gn are clamped
    // copies); refills are clamped the same way.
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const int kc = k0 + j;
        consume(j, kc < gn ? kc : gn - 1, kc < gn);
        __builtin_amdgcn_sched_barrier(0);
        const int kn = k0 + W + j;
        issue(j, kn < gn ? kn : gn - 1);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < W - 1; ++j) {
        const int kc = k0 + W + j;
        consume(j, kc < gn ? kc : gn - 1, kc < gn);
    }
    if constexpr (LG > 0) {
#pragma unroll
        for (int e = 0; e < R; ++e) acc.v[e] = add_(sum.v[e], acc.v[e]);
    }
}

// A non-interior tile (lim >= R: the host sends narrower matrices to
// spmv_narrow_kernel).
template <typename TV, typename TX, int LG = 0>
__device__ __forceinline__ void edge_group(int64_t r, int64_t cols, int64_t lim, int gn,
                                           const int32_t* __restrict__ offs,
                                           const TV* __restrict__ vg, const TX* __restrict__ x,
                                           Run<TX, Shape<TV, TX>::R>& acc)
{
    ring_group<TV, TX, Shape<TV, TX>::WR, kEdgeRun, LG>(r, cols, lim, gn, offs, vg, x, acc);
}

template <typename TX, int R>
__device__ __forceinline__ void store_rows(TX* __restrict__ y, int64_t r, int64_t rows,
                                           const Run<TX, R>& acc, bool full)
{
    if (full) {
        store_run_nt<TX, R>(y + r, acc);
    } else {
#pragma unroll
        for (int e = 0; e < R; ++e)
            if (r + e < rows) y[r + e] = acc.v[e];
    }
}

// DOT epilogue: see the file comment.  x must hold the lane's rows
// (x_size >= rows, checked by the host).
template <typename TX, int R>
__device__ __forceinline__ void dot_epilogue(const Run<TX, R>& acc, const TX* __restrict__ x,
                                             int64_t r, int64_t rows, bool full, int tile,
                                             int tiles, const DotArgs& da)
{
    double s = 0.0;
    if (full) {
        const Run<TX, R> u = load_run<TX, R, false>(x + r);
#pragma unroll
        for (int e = 0; e < R; ++e) s += dotpart(u.v[e], acc.v[e]);
    } else {
#pragma unroll
        for (int e = 0; e < R; ++e)
            if (r + e < rows) s += dotpart(x[r + e], acc.v[e]);
    }
    store_partial<kBlock>(s, tile, da.partials);
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// K > kShortMax: one ring over all K diagonals (LG: ring_group).
template <typename TV, typename TX, bool DOT, int LG = 0>
__global__ __launch_bounds__(kBlock) void spmv_ring_kernel(
    int32_t rows, int32_t cols, int64_t lim, int32_t K, const int32_t* __restrict__ offs,
    const TV* __restrict__ vals, const TX* __restrict__ x, TX* __restrict__ y, int32_t tiles,
    int32_t per_xcd, DotArgs da)
{
    typedef Shape<TV, TX> S;
    constexpr int R = S::R;
    const int tile = tile_of_block(per_xcd);
    if (tile >= tiles) return;
    const int lane = (int)threadIdx.x & 63;
    const int64_t r0 = (int64_t)tile * S::TILE;
    const int64_t r = r0 + (int64_t)threadIdx.x * R;

    // offset range (one vector load per 64 offsets, reduced across the wave)
    int dmin = INT_MAX, dmax = INT_MIN;
    for (int g0 = 0; g0 < K; g0 += 64) {
        const int gn = (K - g0) < 64 ? (K - g0) : 64;
        int lo, hi;
        wave_minmax(offs[g0 + (lane < gn ? lane : gn - 1)], lo, hi);
        dmin = lo < dmin ? lo : dmin;
        dmax = hi > dmax ? hi : dmax;
    }
    const bool interior =
        r0 + S::TILE <= rows && r0 + dmin >= 0 && r0 + S::TILE + (int64_t)dmax <= lim;

    Run<TX, R> acc;
#pragma unroll
    for (int e = 0; e < R; ++e) acc.v[e] = zero_of<TX>();
    if (interior)
        ring_group<TV, TX, S::W, kInterior, LG>(r, cols, lim, K, offs, vals, x, acc);
    else
        edge_group<TV, TX, LG>(r, cols, lim, K, offs, vals, x, acc);
    store_rows<TX, R>(y, r, rows, acc, interior);
    if constexpr (DOT) dot_epilogue<TX, R>(acc, x, r, rows, interior, tile, tiles, da);
}

// K == KF <= kShortMax: offsets by scalar loads, all 2K loads straight-line.
template <typename TV, typename TX, int KF, bool DOT>
__global__ __launch_bounds__(kBlock) void spmv_short_kernel(
    int32_t rows, int32_t cols, int64_t lim, int32_t K, const int32_t* __restrict__ offs,
    const TV* __restrict__ vals, const TX* __restrict__ x, TX* __restrict__ y, int32_t tiles,
    int32_t per_xcd, DotArgs da)
{
    typedef Shape<TV, TX> S;
    constexpr int R = S::R;
    const int tile = tile_of_block(per_xcd);
    if (tile >= tiles) return;
    const int64_t r0 = (int64_t)tile * S::TILE;
    const int64_t r = r0 + (int64_t)threadIdx.x * R;
    (void)K;

    int d[KF > 0 ? KF : 1];
    int dmin = INT_MAX, dmax = INT_MIN;
#pragma unroll
    for (int k = 0; k < KF; ++k) {
        d[k] = offs[k];
        dmin = d[k] < dmin ? d[k] : dmin;
        dmax = d[k] > dmax ? d[k] : dmax;
    }
    const bool interior = r0 + S::TILE <= rows &&
                          (KF == 0 || (r0 + dmin >= 0 && r0 + S::TILE + (int64_t)dmax <= lim));

    Run<TX, R> acc;
#pragma unroll
    for (int e = 0; e < R; ++e) acc.v[e] = zero_of<TX>();
    if constexpr (KF > 0) {
        if (interior) {
            Run<TV, R> a[KF];
            Run<TX, R> b[KF];
#pragma unroll
            for (int k = 0; k < KF; ++k) {
                a[k] = load_run<TV, R, true>(vals + (int64_t)k * cols + r + d[k]);
                b[k] = load_run<TX, R, false>(x + r + d[k]);
            }
#pragma unroll
            for (int k = 0; k < KF; ++k)
#pragma unroll
                for (int e = 0; e < R; ++e) acc.v[e] = mad(acc.v[e], a[k].v[e], b[k].v[e]);
        } else {
            edge_group<TV, TX>(r, cols, lim, KF, offs, vals, x, acc);
        }
    }
    store_rows<TX, R>(y, r, rows, acc, interior);
    if constexpr (DOT) dot_epilogue<TX, R>(acc, x, r, rows, interior, tile, tiles, da);
}

// lim < R (fewer than R columns of x in range): no 16-byte run fits, so
// every term is a per-element load behind its bounds check.  Same tiles and
// epilogues as the other kernels.
template <typename TV, typename TX, bool DOT>
__global__ __launch_bounds__(kBlock) void spmv_narrow_kernel(
    int32_t rows, int32_t cols, int64_t lim, int32_t K, const int32_t* __restrict__ offs,
    const TV* __restrict__ vals, const TX* __restrict__ x, TX* __restrict__ y, int32_t tiles,
    int32_t per_xcd, DotArgs da)
{
    typedef Shape<TV, TX> S;
    constexpr int R = S::R;
    const int tile = tile_of_block(per_xcd);
    if (tile >= tiles) return;
    const int64_t r = (int64_t)tile * S::TILE + (int64_t)threadIdx.x * R;
    Run<TX, R> acc;
#pragma unroll
    for (int e = 0; e < R; ++e) acc.v[e] = zero_of<TX>();
    for (int k = 0; k < K; ++k) {
        const int64_t c = r + offs[k];
        const TV* vk = vals + (int64_t)k * cols;
#pragma unroll
        for (int e = 0; e < R; ++e)
            if ((uint64_t)(c + e) < (uint64_t)lim) acc.v[e] = mad(acc.v[e], vk[c + e], x[c + e]);
    }
    store_rows<TX, R>(y, r, rows, acc, false);
    if constexpr (DOT) dot_epilogue<TX, R>(acc, x, r, rows, false, tile, tiles, da);
}

// m diagonals (1 <= m <= N) of an interior tile: all 2 N loads at once, the
// slots past m a copy of the last diagonal's whose terms are dropped.
template <typename TV, typename TX, int N>
__device__ __forceinline__ void straight_chunk(int64_t r, int64_t cols, int m,
                                               const int32_t* __restrict__ offs,
                                               const TV* __restrict__ vg,
                                               const TX* __restrict__ x,
                                               Run<TX, Shape<TV, TX>::R>& acc)
{
    constexpr int R = Shape<TV, TX>::R;
    Run<TV, R> a[N];
    Run<TX, R> b[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int k = j < m ? j : m - 1;
        const int64_t c = r + offs[k];
        a[j] = load_run<TV, R, true>(vg + (int64_t)k * cols + c);
        b[j] = load_run<TX, R, false>(x + c);
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int e = 0; e < R; ++e)
            acc.v[e] = sel(j < m, mad(acc.v[e], a[j].v[e], b[j].v[e]), acc.v[e]);
}

// Few rows, many diagonals (split_waves): S waves share one tile of 64 R
// rows, wave w accumulating the diagonals [K w / S, K (w + 1) / S), and the
// S sums of each row are added in wave order through LDS (a fixed order:
// deterministic).  The shorter sums round less: fp64, n = 100003, K = 64
// against an 80-bit sum 2.7e-16 in one sum, 1.45e-16 in eight.
//
// What bounds such a call is the chain of load latencies of one wave over
// its K diagonals, with too few waves to hide it (fp64, n = 100003, K = 64:
// 200 workgroups of the ring kernel on 256 CUs).  S waves per row cut the
// chain to K / S diagonals, taken in chunks of at most kSplitChunk whose
// loads are all in flight at once (exact chunk sizes 2, 4, 6, 8: padding
// slots would be real loads), and put S times as many waves on the chip.
template <typename TV, typename TX, int S>
__global__ __launch_bounds__(64 * S) void spmv_split_kernel(
    int32_t rows, int32_t cols, int64_t lim, int32_t K, const int32_t* __restrict__ offs,
    const TV* __restrict__ vals, const TX* __restrict__ x, TX* __restrict__ y, int32_t tiles,
    int32_t per_xcd)
{
    constexpr int R = Shape<TV, TX>::R;
    constexpr int kRows = 64 * R;
    __shared__ Run<TX, R> part[S * 64];
    const int tile = tile_of_block(per_xcd);
    if (tile >= tiles) return;   // uniform over the workgroup
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int64_t r0 = (int64_t)tile * kRows;
    const int64_t r = r0 + (int64_t)lane * R;
    // K >= S (split_waves): every wave has a diagonal
    const int k0 = (int)((int64_t)K * wave / S);
    const int gn = (int)((int64_t)K * (wave + 1) / S) - k0;
    const int32_t* od = offs + k0;
    const TV* vg = vals + (int64_t)k0 * cols;

    int dmin = INT_MAX, dmax = INT_MIN;
    for (int g0 = 0; g0 < gn; g0 += 64) {
        const int gm = (gn - g0) < 64 ? (gn - g0) : 64;
        int lo, hi;
        wave_minmax(od[g0 + (lane < gm ? lane : gm - 1)], lo, hi);
        dmin = lo < dmin ? lo : dmin;
        dmax = hi > dmax ? hi : dmax;
    }
    const bool interior =
        r0 + kRows <= rows && r0 + dmin >= 0 && r0 + kRows + (int64_t)dmax <= lim;

    Run<TX, R> acc;
#pragma unroll
    for (int e = 0; e < R; ++e) acc.v[e] = zero_of<TX>();
    if (!interior) {
        edge_group<TV, TX>(r, cols, lim, gn, od, vg, x, acc);
    } else {
        // equal chunks of at most kSplitChunk diagonals, each chunk's loads
        // straight-line
        const int chunks = (gn + kSplitChunk - 1) / kSplitChunk;
        for (int c = 0; c < chunks; ++c) {
            const int a0 = (int)((int64_t)gn * c / chunks);
            const int m = (int)((int64_t)gn * (c + 1) / chunks) - a0;
            const TV* vc = vg + (int64_t)a0 * cols;
            if (m > 6)
                straight_chunk<TV, TX, 8>(r, cols, m, od + a0, vc, x, acc);
            else if (m > 4)
                straight_chunk<TV, TX, 6>(r, cols, m, od + a0, vc, x, acc);
            else if (m > 2)
                straight_chunk<TV, TX, 4>(r, cols, m, od + a0, vc, x, acc);
            else
                straight_chunk<TV, TX, 2>(r, cols, m, od + a0, vc, x, acc);
        }
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    // row i of the tile: lane i / R's element i % R of every wave
    const TX* p = reinterpret_cast<const TX*>(part);
    for (int i = (int)threadIdx.x; i < kRows; i += 64 * S) {
        TX sum = p[i];
#pragma unroll
        for (int w = 1; w < S; ++w) sum = add_(sum, p[w * kRows + i]);
        if (r0 + i < rows) y[r0 + i] = sum;
    }
}

// Waves per tile of the split kernel, or 1 for the other kernels: a rule on
// the matrix type, rows and diagonals alone, so that a real matrix takes the
// same order of sums with real and with complex vectors.  About 8 diagonals
// per wave (4 at K <= 16, where the short kernel already issues every load at
// once).  Measured (us, 3 rotated sets, ring or short kernel -> split):
//   fp32, K 64:  n = 1000 18.1 -> 5.4, 100003 17.5 -> 6.8, 250000 17.9 -> 13.2,
//                399999 24.1 -> 20.7, 600011 30.9 -> 26.8, 10^6 43.9 -> 43.7
//   fp64, K 64:  n = 130000 15.1 -> 14.4, 160000 20.9 -> 16.9, 210000 22.3 ->
//                21.5, 250000 23.4 -> 25.0, 275000 30.4 -> 27.3, 350000 33.5 ->
//                33.5, 399999 41.3 -> 39.3, 10^6 88.6 -> 92.3;  K 17: 90000 5.5
//                -> 4.9, 130000 5.6 -> 5.7;  complex, K 85: 250000 29.9 -> 34.8,
//                300000 41.8 -> 42.1
//   fp32 matrix, complex vector: K 64, n = 250000 16.6 -> 18.3, 275000 21.2 ->
//                19.8, 600011 35.8 -> 37.6
//   fp32, K 16:  n = 50000 5.3 -> 4.0, 100003 5.3 -> 4.1;  fp64 50000 4.6 ->
//                3.9, 80000 0.97 of the rate, 99999 0.88;  K 12: fp32 50000 4.6
//                -> 4.0;  K 10: n = 1000 fp32 3.59 -> 3.71, complex vector 2.78 ->
//                3.09, 5000 1.00 to 1.04 of the rate, 15000 1.03 to 1.08
// So it starts at K = 10, from 4096 rows (K = 12 below: K 12, n = 1000 1.06 to
// 1.16), and ends at 400000 rows, and 100000 (8-byte values 65536) for K <= 16.
// With 8-byte values between, the ring kernel has one workgroup per 512 rows
// and is the faster one where its last round of workgroups is well filled:
// above 60 % of the 256 CUs.  (The fp32 matrix with a complex vector, which
// shares the real vector's order of sums, then forms them in the ring kernel:
// ring_sums.)  It is the
// faster one above 100000 rows, too, where a wave has 5 diagonals, which are
// padded to 6 (fp64, K 40: 130000 0.91 of its rate, 300000 21.4 -> 23.9).
template <typename TV, typename TX> int split_waves(int32_t rows, int K)
{
    constexpr bool kWide = sizeof(TV) == 8;
    if (K < 10 || (K < 12 && rows < 4096)) return 1;
    if (K <= kShortMax) return rows <= (kWide ? 65536 : 100000) ? (K < 13 ? 2 : 4) : 1;
    if (rows > 400000) return 1;
    if (kWide) {
        const int wgs = ceil_div<int>(rows, kBlock * Shape<TV, TX>::R), last = wgs % 256;
        if (wgs <= 256 ? K < 20 && wgs > 195 : last == 0 || last > 154) return 1;
        if (wgs > 195 && K >= 40 && K < 44) return 1;
    }
    return K < 20 ? 2 : (K < 40 ? 4 : 8);
}

// A real matrix with a complex vector takes twice the workgroups of a real
// vector for the same rows, so the ring kernel fills the chip sooner: where
// its last round of 256 workgroups is well filled it forms the split kernel's
// sums (the real vector's order, for which the split kernel stays the faster)
// at 0.95 to 1.0 of its rate with one sum.  Where a wave of the split kernel
// would have 5 or 7 diagonals, padded to 6 or 8, it is the faster one earlier.
// Rate against the split kernel (fp32 matrix): n = 262144 (2 full rounds) K =
// 24 1.06, 28 1.23, 40 1.26, 64 1.11, 78 1.10, 96 0.97; 225000 (1.7 rounds) K =
// 40 1.14, 64 0.99, 96 0.87; 150000 (1.1) 0.67 to 0.93; 392000 (3.0) K = 24
// 1.02, 40 1.31, 78 1.09; 290000 (2.2) K = 28 1.02, 40 1.11, 78 0.89.
template <typename TV, typename TX> bool ring_sums(int32_t rows, int K, int S)
{
    const int wgs = ceil_div<int>(rows, Shape<TV, TX>::TILE);
    if (K <= kShortMax || wgs <= 256) return false;
    const int last = (wgs - 1) % 256 + 1, per = K / S;
    if (per == 5 || per == 7) return wgs > 512 || last > 128;
    return last > (wgs > 512 ? 128 : 180);
}

template <typename TV, typename TX>
using SpmvKernel = void (*)(int32_t, int32_t, int64_t, int32_t, const int32_t*, const TV*,
                            const TX*, TX*, int32_t, int32_t, DotArgs);

template <typename TV, typename TX, bool DOT>
SpmvKernel<TV, TX> pick_kernel(int K, int64_t lim)
{
    if (K > 0 && lim < Shape<TV, TX>::R) return spmv_narrow_kernel<TV, TX, DOT>;
    switch (K) {
    case 0: return spmv_short_kernel<TV, TX, 0, DOT>;
    case 1: return spmv_short_kernel<TV, TX, 1, DOT>;
    case 2: return spmv_short_kernel<TV, TX, 2, DOT>;
    case 3: return spmv_short_kernel<TV, TX, 3, DOT>;
    case 4: return spmv_short_kernel<TV, TX, 4, DOT>;
    case 5: return spmv_short_kernel<TV, TX, 5, DOT>;
    case 6: return spmv_short_kernel<TV, TX, 6, DOT>;
    case 7: return spmv_short_kernel<TV, TX, 7, DOT>;
    case 8: return spmv_short_kernel<TV, TX, 8, DOT>;
    case 9: return spmv_short_kernel<TV, TX, 9, DOT>;
    case 10: return spmv_short_kernel<TV, TX, 10, DOT>;
    case 11: return spmv_short_kernel<TV, TX, 11, DOT>;
    case 12: return spmv_short_kernel<TV, TX, 12, DOT>;
    case 13: return spmv_short_kernel<TV, TX, 13, DOT>;
    case 14: return spmv_short_kernel<TV, TX, 14, DOT>;
    case 15: return spmv_short_kernel<TV, TX, 15, DOT>;
    case 16: return spmv_short_kernel<TV, TX, 16, DOT>;
    default: return spmv_ring_kernel<TV, TX, DOT>;
    }
}
static_assert(kShortMax == 16, "pick_kernel covers K = 0..16");

}  // namespace

template <typename TV, typename TX>
int32_t spmv_tiles(int32_t rows)
{
    return (int32_t)ceil_div<int64_t>(rows, Shape<TV, TX>::TILE);
}

template <typename TV, typename TX>
int spmv_run(int32_t rows, int32_t cols, int32_t num_diags, const int32_t* offs, const TV* vals,
             const TX* x, int64_t x_size, TX* y, const DotArgs* dot, void* stream,
             const char* name)
{
    if (rows < 0 || cols < 0 || num_diags < 0)
        return fail(DIAGPU_ERR_ARG, "%s: negative size (rows=%d cols=%d num_diags=%d)", name,
                    rows, cols, num_diags);
    if (x_size < 0) return fail(DIAGPU_ERR_ARG, "%s: negative x_size %lld", name, (long long)x_size);
    if (rows == 0) return DIAGPU_OK;
    if (!y) return fail(DIAGPU_ERR_ARG, "%s: y is NULL", name);
    const int64_t lim = x_size < cols ? x_size : (int64_t)cols;
    int K = num_diags;
    if (K > 0) {
        if (!offs) return fail(DIAGPU_ERR_ARG, "%s: diag_offsets is NULL", name);
        if (cols > 0 && !vals) return fail(DIAGPU_ERR_ARG, "%s: values is NULL", name);
        if (lim > 0 && !x) return fail(DIAGPU_ERR_ARG, "%s: x is NULL", name);
    }
    if (dot && (x_size < rows || !x || !dot->partials))
        return fail(DIAGPU_ERR_ARG, "%s: the dot epilogue needs x_size >= rows and its buffers",
                    name);
    if (lim == 0) K = 0;   // no column in range: y = 0 without touching values or x
    const int S = dot || lim < Shape<TV, TX>::R ? 1 : split_waves<TV, TX>(rows, K);
    const int32_t tiles = spmv_tiles<TV, TX>(rows);
    const int32_t per_xcd = ceil_div<int32_t>(tiles, kNumXcd);
    if constexpr (sizeof(TV) < sizeof(TX)) {
        if (S > 1 && ring_sums<TV, TX>(rows, K, S)) {
            hipLaunchKernelGGL((S == 2   ? spmv_ring_kernel<TV, TX, false, 1>
                                : S == 4 ? spmv_ring_kernel<TV, TX, false, 2>
                                         : spmv_ring_kernel<TV, TX, false, 3>),
                               dim3(per_xcd * kNumXcd), dim3(kBlock), 0, as_stream(stream), rows,
                               cols, lim, K, offs, vals, x, y, tiles, per_xcd,
                               DotArgs{nullptr, nullptr});
            return check_launch(name);
        }
    }
    if (S > 1) {
        const int32_t st = (int32_t)ceil_div<int64_t>(rows, 64 * Shape<TV, TX>::R);
        const int32_t sx = ceil_div<int32_t>(st, kNumXcd);
        hipLaunchKernelGGL((S == 2   ? spmv_split_kernel<TV, TX, 2>
                            : S == 4 ? spmv_split_kernel<TV, TX, 4>
                                     : spmv_split_kernel<TV, TX, 8>),
                           dim3(sx * kNumXcd), dim3(64 * S), 0, as_stream(stream), rows, cols, lim,
                           K, offs, vals, x, y, st, sx);
        return check_launch(name);
    }
    const DotArgs da = dot ? *dot : DotArgs{nullptr, nullptr};
    hipLaunchKernelGGL((dot ? pick_kernel<TV, TX, true>(K, lim) : pick_kernel<TV, TX, false>(K, lim)),
                       dim3(per_xcd * kNumXcd), dim3(kBlock), 0, as_stream(stream), rows, cols,
                       lim, K, offs, vals, x, y, tiles, per_xcd, da);
    const int st = check_launch(name);
    if (st || !dot || !dot->out) return st;
    return sum_partials(dot->partials, tiles, dot->out, stream);
}

namespace {
constexpr int kSumBlock = 1024;
constexpr int kSumUnroll = 8;

struct SumJob {
    const double* partials;
    int32_t n;
    double* out;
};

// Workgroup b sums job b.  Lane l adds partials l, l + 1024, l + 2048, ... in
// that order (loads of a batch of 8 issued before their adds), then a fixed
// tree: deterministic, and up to 8192 partials cost one memory round trip.
__global__ __launch_bounds__(kSumBlock) void k_sum_partials(SumJob j0, SumJob j1)
{
    const SumJob job = blockIdx.x == 0 ? j0 : j1;
    const double* __restrict__ partials = job.partials;
    const int32_t n = job.n;
    double t = 0.0;
    int i = (int)threadIdx.x;
    for (; i + (kSumUnroll - 1) * kSumBlock < n; i += kSumUnroll * kSumBlock) {
        double v[kSumUnroll];
#pragma unroll
        for (int u = 0; u < kSumUnroll; ++u) v[u] = partials[i + u * kSumBlock];
#pragma unroll
        for (int u = 0; u < kSumUnroll; ++u) t += v[u];
    }
    for (; i < n; i += kSumBlock) t += partials[i];
    t = block_sum<kSumBlock>(t);
    if (threadIdx.x == 0) *job.out = t;
}
}  // namespace

int sum_partials(const double* partials, int32_t n, double* out, void* stream)
{
    const SumJob j0{partials, n, out};
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kSumBlock), 0, as_stream(stream), j0, j0);
    return check_launch("sum_partials");
}

int sum_partials2(const double* p0, int32_t n0, double* out0, const double* p1, int32_t n1,
                  double* out1, void* stream)
{
    hipLaunchKernelGGL(k_sum_partials, dim3(2), dim3(kSumBlock), 0, as_stream(stream),
                       SumJob{p0, n0, out0}, SumJob{p1, n1, out1});
    return check_launch("sum_partials2");
}

#define DIAGPU_SPMV_INSTANCE(TV, TX)                                                          \
    template int32_t spmv_tiles<TV, TX>(int32_t);                                             \
    template int spmv_run<TV, TX>(int32_t, int32_t, int32_t, const int32_t*, const TV*,       \
                                  const TX*, int64_t, TX*, const DotArgs*, void*, const char*);
DIAGPU_SPMV_INSTANCE(float, float)
DIAGPU_SPMV_INSTANCE(double, double)
DIAGPU_SPMV_INSTANCE(cf32, cf32)
DIAGPU_SPMV_INSTANCE(float, cf32)
#undef DIAGPU_SPMV_INSTANCE

}  // namespace diagpu

extern "C" {

DIAGPU_API int diagpu_spmv_recon_f32(const diagpu_recon_view_f32* R, const float* x,
                                     int64_t x_size, float* y, void* stream)
{
    const char* fn = "diagpu_spmv_recon_f32";
    if (!R) return diagpu::fail(DIAGPU_ERR_ARG, "%s: R is NULL", fn);
    return diagpu::spmv_run<float, float>(R->rows, R->cols, R->num_diags, R->diag_offsets,
                                          R->values, x, x_size, y, nullptr, stream, fn);
}

DIAGPU_API int diagpu_spmv_recon_f64(const diagpu_recon_view_f64* R, const double* x,
                                     int64_t x_size, double* y, void* stream)
{
    const char* fn = "diagpu_spmv_recon_f64";
    if (!R) return diagpu::fail(DIAGPU_ERR_ARG, "%s: R is NULL", fn);
    return diagpu::spmv_run<double, double>(R->rows, R->cols, R->num_diags, R->diag_offsets,
                                            R->values, x, x_size, y, nullptr, stream, fn);
}

DIAGPU_API int diagpu_spmv_recon_c64(const diagpu_recon_view_c64* R, const diagpu_complex64* x,
                                     int64_t x_size, diagpu_complex64* y, void* stream)
{
    using diagpu::cf32;
    const char* fn = "diagpu_spmv_recon_c64";
    if (!R) return diagpu::fail(DIAGPU_ERR_ARG, "%s: R is NULL", fn);
    return diagpu::spmv_run<cf32, cf32>(R->rows, R->cols, R->num_diags, R->diag_offsets,
                                        reinterpret_cast<const cf32*>(R->values),
                                        reinterpret_cast<const cf32*>(x), x_size,
                                        reinterpret_cast<cf32*>(y), nullptr, stream, fn);
}

DIAGPU_API int diagpu_spmv_recon_f32_c64(const diagpu_recon_view_f32* R,
                                         const diagpu_complex64* x, int64_t x_size,
                                         diagpu_complex64* y, void* stream)
{
    using diagpu::cf32;
    const char* fn = "diagpu_spmv_recon_f32_c64";
    if (!R) return diagpu::fail(DIAGPU_ERR_ARG, "%s: R is NULL", fn);
    return diagpu::spmv_run<float, cf32>(R->rows, R->cols, R->num_diags, R->diag_offsets,
                                         R->values, reinterpret_cast<const cf32*>(x), x_size,
                                         reinterpret_cast<cf32*>(y), nullptr, stream, fn);
}

}  // extern "C"
