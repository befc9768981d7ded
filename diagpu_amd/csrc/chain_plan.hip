// Plans of a matrix-power or Taylor chain on the host: C_t = H C_{t-1} for t
// = 1 .. steps, C_0 = S, from the offsets alone.
//
// A plan on the device costs its caller a launch, a kernel of 12 to 45 us and
// a read-back of the counts before the product can be launched, and every
// next plan needs the one before it: four plans held a propagator whose
// products take 200 us at 500 us.  The offsets of a chain's operands are known
// on the host, its plans are a few thousand integers, and all of them are
// formed here in one call (order 6 of the 7-point stencil: 3185 entries), to be
// copied to the device together.
//
// The arrays are those of the symbolic phase for the operands H and C_{t-1}
// (C_0 in the standard layout: diagonals in offset order, each after the one
// before): the C structure, pair_ptr, and the A-stationary kernel's records
// with the four ints after them.  Entries are in plan order: per C diagonal,
// the B diagonals in B's order.
#include <algorithm>
#include <climits>
#include <new>
#include <vector>

#include "common.hpp"

namespace diagpu {
namespace {

// Plan entries of all steps together up to which the host forms them (10 ns
// an entry; callers that want the faster planner stop earlier).
constexpr int64_t kMaxEntries = 32768;
// Words of 64 offsets that a bit per offset may take (512 KiB); sums over a
// wider span are sorted.
constexpr int64_t kSpanWords = 1 << 16;

int64_t absl(int64_t x) { return x < 0 ? -x : x; }
int64_t min0(int64_t x) { return x < 0 ? x : 0; }

bool ascending_inside(int32_t n, const int32_t* off, int32_t cnt)
{
    for (int32_t i = 0; i < cnt; ++i)
        if (off[i] <= -n || off[i] >= n || (i && off[i] <= off[i - 1])) return false;
    return true;
}

// Bytes of the step's arrays, 16-byte aligned parts, at their offsets from
// `at` on.
size_t place(diagpu_chain_step& s, size_t at)
{
    auto part = [&](int64_t bytes) {
        const size_t o = at;
        at += ((size_t)bytes + 15) & ~(size_t)15;
        return (int64_t)o;
    };
    s.c_starts = part(8 * s.c_ndiag);
    s.pair_ptr = part(8 * (s.c_ndiag + 1));
    s.records = part(16 * s.n_pairs + 16);
    s.c_off = part(4 * s.c_ndiag);
    s.c_len = part(4 * s.c_ndiag);
    return at;
}

int chain_plans(const char* fn, int32_t n, int32_t nh, const int32_t* h, int32_t ns,
                const int32_t* s0, int32_t steps, char* out, size_t capacity, size_t* needed,
                diagpu_chain_step* info)
{
    std::vector<std::vector<int32_t>> lists((size_t)steps + 1);   // C_t's offsets
    std::vector<uint64_t> bits;
    std::vector<int32_t> before, rank;
    std::vector<int64_t> bstart, count;
    // The sums of step t lie in [low(t), high(t)], inside (-n, n).
    auto low = [&](int32_t t) {
        const auto& b = lists[(size_t)t];
        return b.empty() ? 0 : std::max<int64_t>((int64_t)h[0] + b.front(), 1 - (int64_t)n);
    };
    auto high = [&](int32_t t) {
        const auto& b = lists[(size_t)t];
        return b.empty() ? -1
                         : std::min<int64_t>((int64_t)h[nh - 1] + b.back(), (int64_t)n - 1);
    };
    // All offsets first (a bit per offset of the span, 1 to 2 ns a sum), so
    // that a chain that is refused costs little.
    lists[0].assign(s0, s0 + ns);
    int64_t entries = 0;
    for (int32_t t = 0; t < steps; ++t) {
        const std::vector<int32_t>& b = lists[(size_t)t];
        std::vector<int32_t>& c = lists[(size_t)t + 1];
        entries += (int64_t)nh * (int64_t)b.size();
        if (entries > kMaxEntries)
            return fail(DIAGPU_ERR_OVERFLOW, "%s: more than %lld entries by step %d", fn,
                        (long long)kMaxEntries, t + 1);
        const int64_t lo = low(t), span = high(t) - lo + 1;
        const int64_t words = span <= 0 ? 0 : (span + 63) / 64;
        if (words > kSpanWords) {
            for (int32_t a = 0; a < nh; ++a)
                for (const int32_t db : b) {
                    const int64_t q = (int64_t)h[a] + db - lo;
                    if (q >= 0 && q < span) c.push_back((int32_t)(q + lo));
                }
            std::sort(c.begin(), c.end());
            c.erase(std::unique(c.begin(), c.end()), c.end());
            continue;
        }
        bits.assign((size_t)words, 0);
        for (int32_t a = 0; a < nh; ++a)
            for (const int32_t db : b) {
                const int64_t q = (int64_t)h[a] + db - lo;
                if (q >= 0 && q < span) bits[(size_t)(q >> 6)] |= 1ull << (q & 63);
            }
        for (int64_t w = 0; w < words; ++w)
            for (uint64_t m = bits[(size_t)w]; m; m &= m - 1)
                c.push_back((int32_t)(lo + 64 * w + __builtin_ctzll(m)));
    }
    size_t at = 0;
    for (int32_t t = 0; t < steps; ++t) {
        const std::vector<int32_t>&b = lists[(size_t)t], &c = lists[(size_t)t + 1];
        const int32_t nb = (int32_t)b.size();
        bstart.resize((size_t)nb);
        int64_t bnnz = 0;
        for (int32_t i = 0; i < nb; ++i) {
            bstart[i] = bnnz;
            bnnz += n - absl(b[i]);
        }
        // C's bits again, and the offsets before each word
        const int64_t lo = low(t), span = high(t) - lo + 1;
        const bool marked = span <= 64 * kSpanWords;
        const size_t words = span <= 0 || !marked ? 0 : (size_t)((span + 63) / 64);
        bits.assign(words, 0);
        if (marked)
            for (const int32_t dc : c) bits[(size_t)((dc - lo) >> 6)] |= 1ull << ((dc - lo) & 63);
        before.resize(words);
        int32_t seen = 0;
        for (size_t w = 0; w < words; ++w) {
            before[w] = seen;
            seen += __builtin_popcountll(bits[w]);
        }
        diagpu_chain_step& s = info[t];
        s = diagpu_chain_step{};
        s.c_ndiag = (int64_t)c.size();
        s.b_extent = bnnz;
        // each sum's C diagonal, in B order, and the entries per C diagonal
        count.assign(c.size() + 1, 0);
        rank.resize((size_t)nh * nb);
        for (int32_t i = 0; i < nb; ++i)
            for (int32_t a = 0; a < nh; ++a) {
                const int64_t q = (int64_t)h[a] + b[i] - lo;
                int32_t k = -1;
                if (q >= 0 && q < span) {
                    const size_t w = (size_t)(q >> 6);
                    k = marked ? before[w] + __builtin_popcountll(bits[w] & ((1ull << (q & 63)) - 1))
                               : (int32_t)(std::lower_bound(c.begin(), c.end(), q + lo) - c.begin());
                    ++count[(size_t)k + 1];
                }
                rank[(size_t)i * nh + a] = k;
            }
        for (size_t k = 0; k < c.size(); ++k) {
            s.c_nnz += n - absl(c[k]);
            s.max_pairs = std::max(s.max_pairs, count[k + 1]);
            s.n_pairs += count[k + 1];
            s.has_main |= c[k] == 0;
        }
        s.b_in_range = 1;
        const size_t end = place(s, at);
        if (end <= capacity) {
            int64_t* starts = reinterpret_cast<int64_t*>(out + s.c_starts);
            int64_t* ptr = reinterpret_cast<int64_t*>(out + s.pair_ptr);
            int32_t* rec = reinterpret_cast<int32_t*>(out + s.records);
            int32_t* coff = reinterpret_cast<int32_t*>(out + s.c_off);
            int32_t* clen = reinterpret_cast<int32_t*>(out + s.c_len);
            int64_t pos = 0, g = 0;
            for (size_t k = 0; k < c.size(); ++k) {
                coff[k] = c[k];
                clen[k] = (int32_t)(n - absl(c[k]));
                starts[k] = pos;
                pos += clen[k];
                ptr[k] = g;
                g += count[k + 1];
                count[k + 1] = ptr[k];   // the diagonal's next free entry
            }
            ptr[c.size()] = g;
            for (int32_t i = 0; i < nb; ++i)   // B order within a C diagonal
                for (int32_t a = 0; a < nh; ++a) {
                    const int32_t k = rank[(size_t)i * nh + a];
                    if (k < 0) continue;
                    const int64_t da = h[a], db = b[i], dc = da + db;
                    // GPair {A start, B start, ash, bsh, al, bl} as a record
                    const int64_t ash = min0(da) - min0(dc), bsh = da + min0(db) - min0(dc);
                    const int64_t lo = std::max<int64_t>(0, std::max(-ash, -bsh));
                    const int64_t hi = std::min(n - absl(da) - ash, n - absl(db) - bsh);
                    const int64_t bq = bstart[i] + bsh;
                    int32_t* r = rec + 4 * count[k + 1]++;
                    const bool none = lo >= hi;
                    if (!none && (bq < INT_MIN || bq + hi > ((int64_t)1 << 30))) s.b_in_range = 0;
                    r[0] = a;
                    r[1] = none ? 1 : (int32_t)lo;
                    r[2] = none ? 1 : (int32_t)hi;
                    r[3] = none || !s.b_in_range ? 0 : (int32_t)bq;
                }
            int32_t* tail = rec + 4 * g;
            tail[0] = tail[1] = 0;
            tail[2] = h[0];
            tail[3] = h[nh - 1];
        }
        at = end;
    }
    *needed = at;
    if (at > capacity)
        return fail(DIAGPU_ERR_CAPACITY, "%s: the plans take %zu bytes, the buffer has %zu", fn, at,
                    capacity);
    return DIAGPU_OK;
}

}  // namespace
}  // namespace diagpu

extern "C" DIAGPU_API int diagpu_chain_plans(int32_t n, int32_t h_ndiag, const int32_t* h_offsets,
                                             int32_t s_ndiag, const int32_t* s_offsets, int32_t steps,
                                             void* out, size_t capacity, size_t* needed,
                                             diagpu_chain_step* info)
{
    using namespace diagpu;
    const char* fn = "diagpu_chain_plans";
    if (n < 1 || n > (1 << 30) || h_ndiag < 1 || s_ndiag < 1 || steps < 1)
        return fail(DIAGPU_ERR_ARG, "%s: need 1 <= n <= 2^30 and at least one diagonal and step", fn);
    if (!h_offsets || !s_offsets || !needed || !info || (capacity > 0 && !out))
        return fail(DIAGPU_ERR_ARG, "%s: a pointer is NULL", fn);
    if (!ascending_inside(n, h_offsets, h_ndiag) || !ascending_inside(n, s_offsets, s_ndiag))
        return fail(DIAGPU_ERR_OFFSET, "%s: offsets must be ascending, distinct and inside (-n, n)",
                    fn);
    try {
        return chain_plans(fn, n, h_ndiag, h_offsets, s_ndiag, s_offsets, steps,
                           static_cast<char*>(out), capacity, needed, info);
    } catch (const std::bad_alloc&) {
        return fail(DIAGPU_ERR_CAPACITY, "%s: out of host memory", fn);
    } catch (const std::exception& e) {
        return fail(DIAGPU_ERR_CAPACITY, "%s: %s", fn, e.what());
    }
}
