// Row kernels of the sparse multi-tau path: a group of lanes per pixel row
// (Corr::multiTau2, src/xpcs/corr.cpp:315-431), exact in integers.
//
// A wave holds 64 / G rows of at most 16 G events, G lanes to a row, so what a
// row costs beside its events (offsets, boundary sums, level loops, output) is
// shared by up to 16 rows instead of taking a wave each.
//
// Narrow rows (k_mt_rows): events packed as frame << 16 | count and a row total
// of at most 65535.  Then every binned value fits 16 bits, every lag sum (at
// most total^2) fits 32 bits and a product is one 24-bit multiply.  Rows with a
// larger total are flagged for the wide form of the same steps
// (k_mt_rows_wide).
//
// Levels below ldeep: the lag sums are bilinear in the events, so no level is
// binned.  Two events at distance D = f_j - f_i >= 1 meet at level L with lag
// d = (f_j >> L) - (f_i >> L), and at most one level has that lag in its
// schedule (lags 1 .. 2 dpl at level 0, dpl + 1 .. 2 dpl above): with L the
// largest level whose dpl 2^L is below D, either d > dpl at L, or d == dpl
// there and the pair counts one level down exactly when its lag is 2 dpl.  One
// walk over the event pairs closer than (2 dpl + 1) 2^(ldeep-1) frames
// therefore serves all those levels.
//
// Measured against one wave per row (k_mt_reg, k_mt_reg2, k_mt_sparse and
// k_mt_deep in k_multitau.hip): the rows of the 1024 x 1024 x 10,000-frame job
// (41 M events, dpl 8) 1.42 -> 0.69 ms, of the 600 x 600 x 12,000-frame job
// (100 M events in rows of 129..512, dpl 4) 3.73 -> 1.10 ms.  What bounds it
// is vector issue (the <= 64-event rows: 3560 instructions per wave of 8 rows,
// nearly half of them the pair walk, a third the series) with half of each
// wave's time in waits on LDS.  Eight lanes of 8 events to such a row measured
// better than four of 16 (0.61 against 0.77 ms: twice the waves fit the LDS);
// for 129..512 events 32 lanes of 16 better than 64 of 8 (1.27 against 1.42 ms).
//
// Levels from ldeep on: the binned series as 16-bit pairs in LDS, the group's
// lanes over time, lag sums by two-element dot products against a register
// window, binning by adding a word's halves.  From level 0 on where the frames
// are few for the row's events: with several events a frame, as averaging frames
// leaves them, the pairs would be many times the series (256 x 256, dpl 8, whole
// passes with the walk on level 0, with the series, and with a wave per row: 60
// frames of 16 averaged, 480 events a row, 5.7, 0.69 and 1.29 ms; 200 of 4, 400
// events, 1.98, 0.67 and 1.09 ms).
#include <algorithm>
#include <type_traits>

#include "device_util.h"
#include "internal.h"

namespace xpcs {

namespace {

constexpr int kRowsWaves = 2;     // waves per workgroup
constexpr int kRowsSeries = 3;    // the series form starts at the first level of at most 3 N frames (level 0: half that), N the class's events
static_assert(kRowSlack >= 64 * 16, "a row kernel reads up to its capacity past a row's first event");

// One length class: its rows and how a wave lays them out.
struct RowsClass {
    const int32_t* list;          // rows (list[r * step]), or NULL: rows 0 .. P-1 in place
    int32_t step;
    const uint32_t* count;        // rows listed (with list)
    int32_t ldeep;
    int32_t aw, bw;               // LDS words per row: boundary slots / lag sums, events / series
    uint8_t* wide;                // per wave of rows: bit g set, its row g is wide
    int32_t flags;                // bytes of `wide` that a wave of k_mt_rows_wide takes at a time (1, 2, 4, 8)
};

struct RowsArgs {
    const uint64_t* ev;
    const int64_t* off;
    const int32_t* rowmap;
    int32_t P, T, F, nb, nlev;
    const int4* tau_bnd;
    const uint16_t* frame_rank;
    int64_t* G2;
    int64_t* IP;
    int64_t* IF;
    uint64_t* pix_total;
    int32_t* big_list;            // rows with a count above 65535 (pixel-major rows only)
    uint32_t* big_count;
    uint32_t* any_wide;           // set by any wave that meets a wide row
    bool w32;
};

// Sum over the group's G lanes; the group's last lane holds it.
template <int G>
__device__ __forceinline__ uint32_t group_sum(uint32_t x)
{
    x += dpp_u32<kDppQuadXor1>(0u, x);
    x += dpp_u32<kDppQuadXor2>(0u, x);
    if constexpr (G >= 8) x += dpp_u32<0x141>(0u, x);    // row_half_mirror
    if constexpr (G >= 16) x += dpp_u32<0x140>(0u, x);   // row_mirror
    if constexpr (G >= 32) x += dpp_u32<kDppBcast15, 0xA>(0u, x);
    if constexpr (G >= 64) x += dpp_u32<kDppBcast31, 0xC>(0u, x);
    return x;
}

// Exclusive prefix sum over the group's lanes.
template <int G>
__device__ __forceinline__ uint32_t group_excl_scan(uint32_t x, int h)
{
    uint32_t s = x;
    uint32_t t;
    t = dpp_u32<kDppRowShr + 1, 0xF, true>(0u, s); s += h >= 1 ? t : 0u;
    t = dpp_u32<kDppRowShr + 2, 0xF, true>(0u, s); s += h >= 2 ? t : 0u;
    if constexpr (G >= 8) { t = dpp_u32<kDppRowShr + 4, 0xF, true>(0u, s); s += h >= 4 ? t : 0u; }
    if constexpr (G >= 16) { t = dpp_u32<kDppRowShr + 8, 0xF, true>(0u, s); s += h >= 8 ? t : 0u; }
    if constexpr (G >= 32) s += dpp_u32<kDppBcast15, 0xA>(0u, s);
    if constexpr (G >= 64) s += dpp_u32<kDppBcast31, 0xC>(0u, s);
    return s - x;
}

__device__ __forceinline__ void order2(uint32_t& a, uint32_t& b)
{
    const uint32_t lo = min(a, b);
    b = max(a, b);
    a = lo;
}

// Ascending sort of E registers (odd-even merge network).
template <int E>
__device__ __forceinline__ void sort_regs(uint32_t (&e)[E])
{
#pragma unroll
    for (int p = 1; p < E; p <<= 1)
#pragma unroll
        for (int k = p; k >= 1; k >>= 1)
#pragma unroll
            for (int j = k % p; j + k < E; j += 2 * k)
#pragma unroll
                for (int i = 0; i < k; i++)
                    if (i + j + k < E && (i + j) / (2 * p) == (i + j + k) / (2 * p)) order2(e[i + j], e[i + j + k]);
}

constexpr uint32_t kPad = 0xFFFF0000u;   // frame key 65535, no count

// Row events in LDS: blocks of E consecutive events, one per lane of the
// group, with a filler word after each block, so that lanes reading their
// blocks word by word meet no bank twice (an unpadded block stride of 16 words
// put 16 lanes on a bank: sorting the rows of the 600 x 600 x 12,000-frame job
// took 0.7 ms).
template <int E>
__device__ __forceinline__ int slot_of(int i) { return i + i / E; }

// The row's events into ascending order; on return e holds the lane's block.
// The transpose leaves a row in frame order up to short shuffles, so blocks of
// E sorted at offsets 0 and E / 2 in turn finish in a round or two; the rounds
// repeat until the wave's rows are all sorted (odd-even transposition of half
// blocks).  A filler word repeats the next block's first key without a count,
// so the pair walk may run over it.
template <int G, int E>
__device__ __forceinline__ void sort_rows(uint32_t* B, int h, uint32_t (&e)[E])
{
    constexpr int N = E * G;
    uint32_t* blk = B + h * (E + 1);
    uint32_t nx = 0u;
    for (int r = 0; r <= 2 * N / E; r++) {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < E; i++) e[i] = blk[i];
#pragma unroll
        for (int i = 0; i + 1 < E; i++) bad |= e[i] > e[i + 1];
        nx = dpp_u32<kDppWaveShl1>(kPad, e[0]);
        if (h == G - 1) nx = kPad;
        bad |= e[E - 1] > nx;
        if (__ballot(bad) == 0ull) break;
        sort_regs(e);
        wave_sync();
#pragma unroll
        for (int i = 0; i < E; i++) blk[i] = e[i];
        wave_sync();
        // blocks at offset E / 2 (the last lane's has E / 2 entries)
#pragma unroll
        for (int i = 0; i < E; i++) e[i] = i < E / 2 ? blk[E / 2 + i] : (h < G - 1 ? blk[E / 2 + i + 1] : 0xFFFFFFFFu);
        sort_regs(e);
        wave_sync();
#pragma unroll
        for (int i = 0; i < E; i++)
            if (i < E / 2) blk[E / 2 + i] = e[i];
            else if (h < G - 1) blk[E / 2 + i + 1] = e[i];
        wave_sync();
    }
    blk[E] = nx & 0xFFFF0000u;
}

// Words of zeros kept before and after a series (the window of a stretch's
// first block, the tail of its last).
constexpr int kSeriesPad = 8;

using u16x2 = __attribute__((ext_vector_type(2))) unsigned short;
__device__ __forceinline__ uint32_t dot2(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_udot2(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b), c, false);
}

// Lag sums of one level's series (x: nw words of two 16-bit values between
// kSeriesPad words of zeros, 16-byte aligned) for lags LO .. LO + DPL - 1.  The
// group's lanes take consecutive stretches of whole 8-word blocks (two 16-byte
// reads each) with the 8 words before a stretch in registers (win: words, sh:
// the same one frame earlier); the group's last lane stores the sums.
template <int G, int DPL, int LO>
__device__ __forceinline__ void series_lags(const uint32_t* x, int nw, int h, uint32_t* out)
{
    constexpr int U = 8;
    const int nblk = (nw + U * G - 1) / (U * G);
    const int k0 = h * nblk * U;
    uint32_t win[U], sh[U], acc[DPL];
#pragma unroll
    for (int l = 0; l < DPL; l++) acc[l] = 0u;
    if (k0 < nw) {
        const uint4* xs = reinterpret_cast<const uint4*>(x + k0);
        auto load8 = [](const uint4* q, uint32_t (&d)[U]) {
            const uint4 a = q[0], b = q[1];
            d[0] = a.x; d[1] = a.y; d[2] = a.z; d[3] = a.w;
            d[4] = b.x; d[5] = b.y; d[6] = b.z; d[7] = b.w;
        };
        // slot u: word k0 - 8 + u (the ring advances one slot per word)
        load8(xs - 2, win);
        sh[0] = 0u;   // one frame before the window: in no lag
#pragma unroll
        for (int u = 1; u < U; u++) sh[u] = __builtin_amdgcn_alignbit(win[u], win[u - 1], 16);
        const int nb = min(nblk, (nw - k0 + U - 1) / U);
        for (int b = 0; b < nb; b++, xs += 2) {
            uint32_t cur[U];
            load8(xs, cur);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t prev = u > 0 ? cur[u > 0 ? u - 1 : 0] : win[U - 1];
                const uint32_t here = __builtin_amdgcn_alignbit(cur[u], prev, 16);
                if constexpr (LO == 1) sh[u] = here;   // lag 1's
#pragma unroll
                for (int l = 0; l < DPL; l++) {
                    const int lag = LO + l;
                    const int m = lag / 2;   // even lag 2 m: word k - m; odd lag 2 m + 1: sh of word k - m
                    acc[l] = dot2(cur[u], (lag & 1) ? sh[(u + U - m) % U] : win[(u + U - m) % U], acc[l]);
                }
                sh[u] = here;
                win[u] = cur[u];
            }
        }
    }
#pragma unroll
    for (int l = 0; l < DPL; l++) {
        const uint32_t s = group_sum<G>(acc[l]);
        if (h == G - 1) out[l] = s;
    }
}

// The next level's series in place: nx values from the words of this one.  A
// wave's LDS accesses are in order and output word m comes from words 2 m and
// 2 m + 1, so each step reads at or past what it overwrites.
template <int G>
__device__ __forceinline__ void series_bin(uint32_t* x, int nx, int h)
{
    const int nw = (nx + 1) / 2;
    for (int m0 = 0; m0 < nw + kSeriesPad; m0 += G) {
        const int m = m0 + h;
        uint32_t v = 0u;
        if (m < nw) {
            const uint2 q = *reinterpret_cast<const uint2*>(x + 2 * m);
            const uint32_t lo = dot2(q.x, 0x00010001u, 0u);
            const uint32_t hi = dot2(q.y, 0x00010001u, 0u);
            v = lo | (2 * m + 1 < nx ? hi << 16 : 0u);
        }
        wave_sync();
        if (m < nw + kSeriesPad) x[m] = v;
        wave_sync();
    }
}

// Sum of 64-bit values over the group's G lanes; the group's last lane holds it.
template <int G>
__device__ __forceinline__ uint64_t group_sum64(uint64_t x)
{
    auto half = [&](auto step) {
        const uint32_t lo = step((uint32_t)x), hi = step((uint32_t)(x >> 32));
        x += ((uint64_t)hi << 32) | lo;
    };
    half([](uint32_t v) { return dpp_u32<kDppQuadXor1>(0u, v); });
    half([](uint32_t v) { return dpp_u32<kDppQuadXor2>(0u, v); });
    if constexpr (G >= 8) half([](uint32_t v) { return dpp_u32<0x141>(0u, v); });    // row_half_mirror
    if constexpr (G >= 16) half([](uint32_t v) { return dpp_u32<0x140>(0u, v); });   // row_mirror
    if constexpr (G >= 32) half([](uint32_t v) { return dpp_u32<kDppBcast15, 0xA>(0u, v); });
    if constexpr (G >= 64) half([](uint32_t v) { return dpp_u32<kDppBcast31, 0xC>(0u, v); });
    return x;
}

// Words of zeros kept before and after the series of a wide row.
constexpr int kWidePad = 16;

// series_lags for a wide row: a word per value (x: nw words between kWidePad
// words of zeros).  Values are at most 1024 x 65535, so products and sums
// (at most total^2) are whole numbers below 2^53, exact in FP64.
template <int G, int DPL, int LO>
__device__ __forceinline__ void wide_series_lags(const uint32_t* x, int nw, int h, unsigned long long* out)
{
    constexpr int U = 8, W = 2 * DPL;
    const int nblk = (nw + U * G - 1) / (U * G);
    const int k0 = h * nblk * U;
    double win[W], acc[DPL];   // win[W - j]: value j back
#pragma unroll
    for (int l = 0; l < DPL; l++) acc[l] = 0.0;
    if (k0 < nw) {
        const uint4* xs = reinterpret_cast<const uint4*>(x + k0);
#pragma unroll
        for (int i = 0; i < W / 4; i++) {
            const uint4 q = xs[i - W / 4];
            win[4 * i] = (double)q.x; win[4 * i + 1] = (double)q.y;
            win[4 * i + 2] = (double)q.z; win[4 * i + 3] = (double)q.w;
        }
        const int nb = min(nblk, (nw - k0 + U - 1) / U);
        for (int b = 0; b < nb; b++, xs += 2) {
            const uint4 qa = xs[0], qb = xs[1];
            const double cur[U] = {(double)qa.x, (double)qa.y, (double)qa.z, (double)qa.w,
                                   (double)qb.x, (double)qb.y, (double)qb.z, (double)qb.w};
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int l = 0; l < DPL; l++) {
                    const int lag = LO + l;
                    acc[l] = fma(cur[u], u >= lag ? cur[u >= lag ? u - lag : 0] : win[u >= lag ? 0 : W + u - lag], acc[l]);
                }
#pragma unroll
            for (int i = 0; i < W; i++) win[i] = i + U < W ? win[i + U < W ? i + U : 0] : cur[i + U < W ? 0 : i + U - W];
        }
    }
#pragma unroll
    for (int l = 0; l < DPL; l++) {
        const uint64_t s = group_sum64<G>((uint64_t)acc[l]);
        if (h == G - 1) out[l] = s;
    }
}

// series_bin for a wide row.
template <int G>
__device__ __forceinline__ void wide_series_bin(uint32_t* x, int nx, int h)
{
    for (int m0 = 0; m0 < nx + kWidePad; m0 += G) {
        const int m = m0 + h;
        uint32_t v = 0u;
        if (m < nx) {
            const uint2 q = *reinterpret_cast<const uint2*>(x + 2 * m);
            v = q.x + q.y;
        }
        wave_sync();
        if (m < nx + kWidePad) x[m] = v;
        wave_sync();
    }
}

// A wave's rows: lane group g has row p (-1: none), n events from `base` on.
// A0, B0: the wave's LDS.  Narrow forms: store the mask of the wave's rows that
// are wide (bit g), if any, to *flag and leave their sums; one for the series from a level
// above 0 on, one for all levels (together in one kernel they cost it 1 to 2 %
// in spilled scalar registers).  Wide form: counts of 16 bits and any total,
// boundary slots and series of 32, lag sums of 64 bits.
enum RowsForm { kRowsNarrow, kRowsNarrowSeries, kRowsWide };

template <int G, int E, int DPL, RowsForm FORM>
__device__ __forceinline__ void mt_rows(const RowsArgs& a, const RowsClass& k, uint32_t* A0, uint32_t* B0, int32_t p,
                                        int64_t base, int n, uint8_t* flag)
{
    constexpr bool WIDE = FORM == kRowsWide;
    constexpr int R = kWave / G;
    constexpr int N = E * G;
    using Acc = std::conditional_t<WIDE, unsigned long long, uint32_t>;
    const int lane = lane_id();
    const int g = lane / G, h = lane % G;
    const int T = a.T, aw = k.aw, bw = k.bw;
    const int ldeep = FORM == kRowsNarrowSeries ? 0 : k.ldeep;
    uint32_t* A = A0 + g * aw;
    uint32_t* B = B0 + g * bw;
    const int nbw = WIDE ? a.nb + 1 : a.nb / 2 + 1;   // words of the boundary slots 0 .. nb
    // ---- events to LDS, boundary slots
    uint32_t e[E];
    uint32_t tot = 0u;
    bool big = false;
    {
        // reads past the row's end stay inside the event buffer (kRowSlack)
        uint64_t q[E];
        const uint64_t* ev = a.ev + base + h;
#pragma unroll
        for (int i = 0; i < E; i++) q[i] = ev[i * G];
        for (int i = h; i < nbw; i += G) A[i] = 0u;
#pragma unroll
        for (int i = 0; i < E; i++) {
            const bool in = i * G + h < n;
            const uint32_t c = in ? (uint32_t)q[i] : 0u;
            tot += min(c, 65536u);
            if constexpr (WIDE) big |= c > 65535u;
            e[i] = in ? ((uint32_t)(q[i] >> 32) << 16) | (c & 0xFFFFu) : kPad;
        }
    }
    tot = group_sum<G>(tot);
    bool leave;            // another kernel's row
    if constexpr (WIDE) {
        const uint64_t bm = __ballot(big);
        leave = ((bm >> (g * G)) & (~0ull >> (64 - G))) != 0ull;
        if (h == G - 1 && p >= 0) {
            if (leave) {
                if (a.big_list) a.big_list[atomicAdd(a.big_count, 1u)] = p;
            } else {
                a.pix_total[p] = tot;
            }
        }
    } else {
        if (h == G - 1 && p >= 0 && tot <= 65535u) a.pix_total[p] = tot;
        tot = (uint32_t)__shfl((int)tot, lane | (G - 1), kWave);
        leave = tot > 65535u;
        const uint64_t wm = __ballot(leave && p >= 0);
        if (wm != 0ull) {
            uint32_t wide_mask = 0u;
            // the next launch reads it: a store that stays in the L2 (one at
            // device scope went to memory, 30 ns each, 4 ms on a million rows)
            if (lane == 0) __hip_atomic_store(a.any_wide, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
            for (int r = 0; r < R; r++) wide_mask |= (uint32_t)((wm >> (r * G)) & 1ull) << r;
            if (lane == 0) *flag = (uint8_t)wide_mask;
        }
    }
    if (leave) p = -1;
    const uint64_t ok = __ballot(p >= 0);
    if (ok == 0ull) return;
    wave_sync();
#pragma unroll
    for (int i = 0; i < E; i++) B[slot_of<E>(i * G + h)] = leave ? kPad : e[i];
    wave_sync();
    sort_rows<G, E>(B, h, e);
    // The values of a lane's consecutive events go to their boundary slots
    // one run of equal slots at a time: between boundaries whole rows share
    // a slot, and one LDS atomic per event to one address took 0.2 ms of
    // the 600 x 600 x 12,000-frame job.  Padding adds 0 to the last
    // frame's slot.
    {
        uint32_t rank[E];
#pragma unroll
        for (int i = 0; i < E; i++) rank[i] = a.frame_rank[min(e[i] >> 16, (uint32_t)a.F - 1u)];
        auto add = [&](uint32_t slot, uint32_t sum) {
            if constexpr (WIDE) atomicAdd(&A[slot], sum);
            else atomicAdd(&A[slot >> 1], sum << (16u * (slot & 1u)));
        };
        uint32_t sum = e[0] & 0xFFFFu;
#pragma unroll
        for (int i = 1; i < E; i++) {
            if (rank[i] != rank[i - 1]) {
                add(rank[i - 1], sum);
                sum = 0u;
            }
            sum += e[i] & 0xFFFFu;
        }
        add(rank[E - 1], sum);
    }
    wave_sync();
    // prefix sums over the slots: slot j = sum of the values of the frames
    // below boundary j
    {
        const int per = (nbw + G - 1) / G;
        const int b0 = min(h * per, nbw), b1 = min(b0 + per, nbw);
        uint32_t s = 0u;
        if constexpr (WIDE) {
            for (int i = b0; i < b1; i++) s += A[i];
            uint32_t run = group_excl_scan<G>(s, h);
            for (int i = b0; i < b1; i++) {
                run += A[i];
                A[i] = run;
            }
        } else {
            for (int i = b0; i < b1; i++) s = dot2(A[i], 0x00010001u, s);
            uint32_t run = group_excl_scan<G>(s, h) * 0x00010001u;   // in both halves
            for (int i = b0; i < b1; i++) {
                const uint32_t x = A[i];
                const uint32_t y = run + x + (x << 16);
                run = __builtin_amdgcn_perm(y, y, 0x03020302u);
                A[i] = y;
            }
        }
    }
    wave_sync();
    // IP = S(B_ip), IF = S(B_end) - S(B_head) of every tau
    for (int t0 = 0; t0 < T; t0 += kWave) {
        const int t = t0 + lane;
        if (t < T) {
            const int4 b = a.tau_bnd[t];
            using M = std::conditional_t<WIDE, uint32_t, uint16_t>;
            constexpr int kPer = sizeof(uint32_t) / sizeof(M);
            const M* m = reinterpret_cast<const M*>(A0);
#pragma unroll 4
            for (int rr = 0; rr < R; rr++) {
                const uint32_t ip = m[kPer * rr * aw + b.x];
                const uint32_t jf = (uint32_t)m[kPer * rr * aw + b.z] - (uint32_t)m[kPer * rr * aw + b.y];
                if ((ok >> (rr * G)) & 1ull) {
                    const uint64_t row0 = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(p, rr * G) * (uint32_t)T;
                    if (a.w32) {
                        (reinterpret_cast<uint32_t*>(a.IP) + row0)[t] = ip;
                        (reinterpret_cast<uint32_t*>(a.IF) + row0)[t] = jf;
                    } else {
                        (a.IP + row0)[t] = (int64_t)ip;
                        (a.IF + row0)[t] = (int64_t)jf;
                    }
                }
            }
        }
    }
    wave_sync();
    for (int i = h; i < aw; i += G) A[i] = 0u;
    wave_sync();
    // ---- event pairs of the levels below ldeep: the lanes step over the
    // wave's events, a lane's row changing with every step, so that rows
    // with many pairs spread over the wave
    if (FORM == kRowsNarrow || ldeep > 0) {
        const uint32_t dlim = (uint32_t)(2 * DPL + 1) << (ldeep - 1);
        const uint32_t fc = ((uint32_t)a.F >> (ldeep - 1)) << (ldeep - 1);   // whole frames of every level
        // events to visit: the longest row's, in steps of G
        int nmax = n;
#pragma unroll
        for (int d = G; d < kWave; d <<= 1) nmax = max(nmax, __shfl_xor(nmax, d, kWave));
        int rr = lane % R, i = lane / R;
        const uint32_t* pj = B0 + rr * bw + slot_of<E>(i);
        Acc* acc = reinterpret_cast<Acc*>(A0 + rr * aw) - 1;
        uint32_t ei = *pj;
        uint32_t ki = ei >> 16, vi = ei & 0xFFFFu;
        if (ki == 0xFFFFu) ki = 0u;       // padding: its first partner is out of reach
        while (i < nmax) {
            const uint32_t ej = *++pj;
            const uint32_t kj = ej >> 16;
            const uint32_t D = kj - ki;
            if (D < dlim) {
                if (D != 0u) {
                    const uint32_t L = 31u - (uint32_t)__builtin_clz(((D - 1u) / DPL) | 1u);
                    const uint32_t d = (kj >> L) - (ki >> L);
                    // lag dpl at level L >= 1 stands for lag 2 dpl one
                    // level down (the same slot), where it needs equal low bits
                    bool in = !(d == (uint32_t)DPL && ((((kj ^ ki) << 1) >> L) & 1u));
                    if (kj >= fc) {
                        const uint32_t Lc = L - (uint32_t)(L > 0u && d == (uint32_t)DPL);
                        in = in && (kj >> Lc) < ((uint32_t)a.F >> Lc);
                    }
                    if (in) atomicAdd(acc + (L * DPL + d), (Acc)(uint32_t)__umul24(vi, ej & 0xFFFFu));
                }
            } else {
                i += G;
                rr = (rr + (R > 1 ? R / 2 - 1 : 0)) % R;
                pj = B0 + rr * bw + slot_of<E>(min(i, N - 1));
                acc = reinterpret_cast<Acc*>(A0 + rr * aw) - 1;
                ei = *pj;
                ki = ei >> 16;
                vi = ei & 0xFFFFu;
                if (ki == 0xFFFFu) ki = 0u;
            }
        }
        wave_sync();
    }
    // ---- binned series of the levels from ldeep on
    if (ldeep < a.nlev) {
        int lf = a.F >> ldeep;
        const int nz = WIDE ? lf + 2 * kWidePad : (lf + 1) / 2 + 2 * kSeriesPad;
        for (int i = h; i < nz; i += G) B[i] = 0u;
        wave_sync();
        uint32_t* X = B + (WIDE ? kWidePad : kSeriesPad);
#pragma unroll
        for (int i = 0; i < E; i++) {
            const uint32_t f = (e[i] >> 16) >> ldeep;
            if (f < (uint32_t)lf) {
                if constexpr (WIDE) atomicAdd(&X[f], e[i] & 0xFFFFu);
                else atomicAdd(&X[f >> 1], (e[i] & 0xFFFFu) << (16u * (f & 1u)));
            }
        }
        wave_sync();
        for (int L = ldeep; L < a.nlev; L++) {
            Acc* out = reinterpret_cast<Acc*>(A) + (L + 1) * DPL;
            if (FORM != kRowsNarrow && L == 0) {   // lags 1 .. dpl as well
                if constexpr (WIDE) wide_series_lags<G, DPL, 1>(X, lf, h, out - DPL);
                else series_lags<G, DPL, 1>(X, (lf + 1) / 2, h, out - DPL);
            }
            if constexpr (WIDE) wide_series_lags<G, DPL, DPL + 1>(X, lf, h, out);
            else series_lags<G, DPL, DPL + 1>(X, (lf + 1) / 2, h, out);
            lf >>= 1;
            wave_sync();
            if (L + 1 < a.nlev) {
                if constexpr (WIDE) wide_series_bin<G>(X, lf, h);
                else series_bin<G>(X, lf, h);
            }
        }
        wave_sync();
    }
    // ---- lag sums out
    for (int t0 = 0; t0 < T; t0 += kWave) {
        const int t = t0 + lane;
        if (t < T) {
#pragma unroll 4
            for (int rr = 0; rr < R; rr++) {
                const uint64_t v = reinterpret_cast<const Acc*>(A0 + rr * aw)[t];
                if ((ok >> (rr * G)) & 1ull) {
                    const uint64_t row0 = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(p, rr * G) * (uint32_t)T;
                    (a.G2 + row0)[t] = (int64_t)v;
                }
            }
        }
    }
    wave_sync();
}

// Row r of a class, for the lane's group: its pixel, first event and length (n
// is 0 and p -1 where there is none or the length is another class's).
template <int N>
__device__ __forceinline__ void class_row(const RowsArgs& a, const RowsClass& k, int64_t r, bool in, int32_t& p,
                                          int64_t& base, int& n)
{
    p = -1;
    n = 0;
    base = 0;
    if (!in) return;
    p = k.list ? k.list[r * k.step] : (int32_t)r;
    const int64_t row = a.rowmap ? (int64_t)a.rowmap[p] : (int64_t)p;
    base = a.off[row];
    const int64_t len = a.off[row + 1] - base;
    if (len > N) p = -1;           // another kernel's row
    else n = (int)len;
}

template <int G, int E, int DPL, RowsForm FORM>
__global__ void __launch_bounds__(kWave * kRowsWaves)
k_mt_rows(const RowsArgs a, const RowsClass k)
{
    constexpr int R = kWave / G;
    extern __shared__ __align__(16) uint32_t s_rows[];
    const int lane = lane_id();
    const int w = wave_id();
    uint32_t* A0 = s_rows + w * R * (k.aw + k.bw);
    uint32_t* B0 = A0 + R * k.aw;
    const int64_t nrows = k.list ? (int64_t)*k.count : (int64_t)a.P;
    const int64_t nwaves = (int64_t)gridDim.x * kRowsWaves;
    for (int64_t r0 = ((int64_t)blockIdx.x * kRowsWaves + w) * R; r0 < nrows; r0 += nwaves * R) {
        const int64_t r = r0 + lane / G;
        int32_t p;
        int64_t base;
        int n;
        class_row<E * G>(a, k, r, r < nrows, p, base, n);
        uint8_t* const flag = k.wide + r0 / R;
        if (__ballot(p >= 0) != 0ull) mt_rows<G, E, DPL, FORM>(a, k, A0, B0, p, base, n, flag);
    }
}

// ---- wide rows ------------------------------------------------------------------
// The rows that k_mt_rows left, from its flags: a wave takes up to 8 flag bytes
// (64 rows), packs the flagged ones and runs them R at a time.
//
// One launch for all classes, which most jobs have no use for: then each wave
// reads one word.  64-bit lag sums halve the rows that a CU's LDS holds, and
// 143 registers allow three waves per SIMD.  Measured on jobs whose rows are
// all wide, the whole pass, against a wave per row (the register and LDS
// kernels of k_multitau.hip): 1024 x 1024 x 10,000 frames, 50 events a row,
// dpl 8: 2.56 -> 2.36 ms (this kernel 1.2); 600 x 600 x 12,000, 293 a row,
// dpl 4: 5.7 -> 3.4 ms; 512 x 384 x 6000, 690 a row: 9.8 -> 7.2 ms; 256 x 256 x
// 1000, 91 a row: 0.47 -> 0.39 ms.  (Listed one by one, with an atomic each, for
// k_mt_sparse<1024>, these rows took 18.7, 14.3, 20.4 and 1.4 ms.)
constexpr int kWideFlags = 8;
// A wave takes fewer flags where there are not that many pieces: with 16 a
// wave, and so 128 waves for a 128 x 128 detector, a job of 2000 frames took
// 460 us, with at least this many waves 234 (256 x 256: 600 and 393 us, 1024 x
// 1024: 2516 and 2324).
constexpr int kWideChunks = 8192;
struct WideArgs {
    RowsArgs a;
    RowsClass k[4];
};

template <int G, int E, int DPL>
__device__ __forceinline__ void wide_class(const RowsArgs& a, const RowsClass& k, int64_t nrows, uint32_t* lds,
                                           uint8_t* pick, int64_t wave, int64_t nwaves, int64_t& used)
{
    constexpr int R = kWave / G;
    const int lane = lane_id();
    uint32_t* A0 = lds;
    uint32_t* B0 = A0 + R * k.aw;
    const int64_t nflags = (nrows + R - 1) / R;
    const int64_t nchunks = (nflags + k.flags - 1) / k.flags;
    // each class begins where the one before it ended, so that short lists
    // spread over the waves
    int64_t c = wave - used;
    if (c < 0) c += nwaves;
    used = (used + nchunks) % nwaves;
    for (; c < nchunks; c += nwaves) {
        const int64_t f0 = c * k.flags;
        uint64_t m = reinterpret_cast<const uint64_t*>(k.wide)[f0 / 8] >> (8 * (f0 % 8));
        const int64_t nf = min(nflags - f0, (int64_t)k.flags);
        if (nf < 8) m &= ~(~0ull << (8 * nf));
        if (m == 0ull) continue;
        const int total = __popcll(m);
        if ((m >> lane) & 1ull) pick[mask_rank(m)] = (uint8_t)lane;
        wave_sync();
        for (int i0 = 0; i0 < total; i0 += R) {
            const int i = i0 + lane / G;
            const bool in = i < total;
            const int b = in ? pick[i] : 0;
            int32_t p;
            int64_t base;
            int n;
            class_row<E * G>(a, k, (f0 + (b >> 3)) * R + (b & 7), in, p, base, n);
            if (__ballot(p >= 0) != 0ull) mt_rows<G, E, DPL, kRowsWide>(a, k, A0, B0, p, base, n, nullptr);
        }
        wave_sync();
    }
}

template <int DPL>
__global__ void __launch_bounds__(kWave * kRowsWaves)
k_mt_rows_wide(const WideArgs a, int32_t lds_words)
{
    if (*a.a.any_wide == 0u) return;
    extern __shared__ __align__(16) uint32_t s_rows[];
    __shared__ uint8_t s_pick[kRowsWaves][8 * kWideFlags];
    const int w = wave_id();
    const int64_t wave = (int64_t)blockIdx.x * kRowsWaves + w, nwaves = (int64_t)gridDim.x * kRowsWaves;
    uint32_t* lds = s_rows + w * lds_words;
    const int64_t n1 = *a.k[1].count, n2 = *a.k[2].count, n3 = *a.k[3].count;
    int64_t used = 0;
    wide_class<8, 8, DPL>(a.a, a.k[0], a.a.P, lds, s_pick[w], wave, nwaves, used);
    wide_class<16, 8, DPL>(a.a, a.k[1], n1, lds, s_pick[w], wave, nwaves, used);
    wide_class<32, 16, DPL>(a.a, a.k[2], n2, lds, s_pick[w], wave, nwaves, used);
    wide_class<64, 16, DPL>(a.a, a.k[3], n3, lds, s_pick[w], wave, nwaves, used);
}

}  // namespace

// First level of the series form for rows of at most N events: the first
// level of at most 3 N binned frames, where a full row has an event in
// every third frame and the series costs about what its event pairs do (2 N
// and 6 N: 0.69 and 0.71 against 0.61 ms for the <= 64-event rows of the
// 1 Mpx job, 1.46 and 1.64 against 1.42 ms for the 129..512-event rows of the
// 600 x 600 x 12,000-frame job), or of at most deep_frames (tuning; negative:
// none, the level count).  Level 0 has twice the lags, so it begins there with
// at most 3 N / 2 frames (with 3 N, rows of 129 events in 1536 frames would sum
// a series of three times their pairs' work).
int rows_series_level(const xpcs_mt_plan* p, int N)
{
    const HostTables& h = p->h;
    const int nlev = (int)h.levels.size();
    if (p->tune.deep_frames < 0) return nlev;
    const int lim = p->tune.deep_frames > 0 ? p->tune.deep_frames : kRowsSeries * N;
    if (h.levels[0].lf <= (p->tune.deep_frames > 0 ? lim : lim / 2)) return 0;
    for (int L = 1; L < nlev; L++)
        if (h.levels[(size_t)L].lf <= lim) return L;
    return nlev;
}

bool rows_with_big_counts(const xpcs_mt_plan* p) { return p->mode == 3 && p->big_rows > 0; }

// The schedules and frame counts the row kernels take: 4 or 8 delays per
// level, every level's lags where the pair walk expects them, and frames that
// leave the padding key (65535) out of reach of every row's last event: with
// automatic tuning 63,231 frames at dpl 4 and 61,183 at dpl 8.
// Pixel-major rows with counts above 65535: up to one row in 32 these go to the
// LDS kernel, which takes 16 ns a row; with more the kernels in k_multitau.hip
// take all rows, 1.4 against 0.7 ms for the million rows of the 1 Mpx job.
bool rows_supported(const xpcs_mt_plan* p)
{
    const HostTables& h = p->h;
    if (rows_with_big_counts(p) && p->big_rows > h.P / 32) return false;
    if (p->fsnorm || (h.dpl != 4 && h.dpl != 8) || h.levels.empty()) return false;
    const int nlev = (int)h.levels.size();
    for (int L = 0; L < nlev; L++) {
        const LevelParam& lp = h.levels[(size_t)L];
        if (L == 0 ? (lp.lo != 1 || lp.first != 0 || lp.count > 2 * h.dpl)
                   : (lp.lo != h.dpl + 1 || lp.first != (L + 1) * h.dpl || lp.count > h.dpl))
            return false;
    }
    const int L = rows_series_level(p, kWave);
    const int64_t dlim = L > 0 ? (int64_t)(2 * h.dpl + 1) << (L - 1) : 0;
    return (int64_t)h.F + dlim <= 65535;
}

static RowsArgs rows_args(xpcs_mt_plan* p)
{
    const HostTables& h = p->h;
    RowsArgs a{};
    a.ev = p->d_ev;
    a.off = p->d_off;
    a.rowmap = p->d_rowmap;
    a.P = h.P;
    a.T = h.T;
    a.F = h.F;
    a.nb = p->nrank;
    a.nlev = (int)h.levels.size();
    a.tau_bnd = p->d_tau_bnd;
    a.frame_rank = p->d_frame_rank;
    a.G2 = p->d_G2;
    a.IP = p->d_IP;
    a.IF = p->d_IF;
    a.pix_total = p->d_pix_total;
    a.big_list = rows_with_big_counts(p) ? p->d_wide_list : nullptr;
    a.big_count = p->d_counters + 6;
    a.any_wide = p->d_counters + 7;
    a.w32 = p->ipif32;
    return a;
}

// Flag bytes of a class of R rows to a wave, in whole 64-bit words.
static size_t wide_flag_bytes(int32_t P, int R)
{
    return ((size_t)(P + R - 1) / R + kWideFlags - 1) / kWideFlags * kWideFlags;
}
size_t rows_wide_flags(const xpcs_mt_plan* p)
{
    size_t n = 0;
    for (int R : {8, 4, 2, 1}) n += wide_flag_bytes(p->h.P, R);
    return (n + 15) / 16 * 16;
}

// Layout of the class of at most N events, G lanes to a row.
static RowsClass rows_class(const xpcs_mt_plan* p, int G, int N, bool wide)
{
    const int R = kWave / G;
    const HostTables& h = p->h;
    const int nlev = (int)h.levels.size();
    RowsClass k{};
    const int c = G == 8 ? 0 : G == 16 ? 1 : G == 32 ? 2 : 3;
    k.list = c == 0 ? nullptr : c == 1 ? p->d_mid_list : c == 2 ? p->d_mid_list + (h.P - 1) : p->d_long_list;
    k.step = c == 2 ? -1 : 1;
    k.count = p->d_counters + (c == 1 ? 2 : c == 2 ? 4 : 5);
    k.ldeep = rows_series_level(p, N);
    k.wide = p->d_wide_flags;
    for (int i = 0; i < c; i++) k.wide += wide_flag_bytes(h.P, 8 >> i);
    for (k.flags = kWideFlags; k.flags > 1 && (int64_t)h.P / R / k.flags < kWideChunks;) k.flags /= 2;
    const int lf = k.ldeep < nlev ? h.levels[(size_t)k.ldeep].lf : 0;
    const int series = k.ldeep == nlev ? 0 : wide ? lf + 2 * kWidePad : (lf + 1) / 2 + 2 * kSeriesPad;
    const int slots = wide ? p->nrank + 1 : p->nrank / 2 + 1;
    const int sums = std::max(h.T, (nlev + 1) * h.dpl + 1) * (wide ? 2 : 1);
    // pitches of 4 mod 8 words: rows aligned to 16 bytes, 16 of them on distinct banks
    auto pitch = [](int words) { return (words + 3) / 8 * 8 + 4; };
    k.aw = pitch(std::max(slots, sums));
    k.bw = pitch(std::max(N + G, series));
    return k;
}

template <int G, int E, int DPL>
static void launch_rows_class(xpcs_mt_plan* p, hipStream_t s, int max_blocks)
{
    constexpr int R = kWave / G;
    const RowsClass k = rows_class(p, G, E * G, false);
    const size_t lds = sizeof(uint32_t) * (size_t)(kRowsWaves * R * (k.aw + k.bw));
    const int64_t need = ((int64_t)p->h.P + R * kRowsWaves - 1) / (R * kRowsWaves);
    const unsigned nb = (unsigned)std::max<int64_t>(1, std::min<int64_t>(need, max_blocks));
    if (k.ldeep == 0) k_mt_rows<G, E, DPL, kRowsNarrowSeries><<<nb, kWave * kRowsWaves, lds, s>>>(rows_args(p), k);
    else k_mt_rows<G, E, DPL, kRowsNarrow><<<nb, kWave * kRowsWaves, lds, s>>>(rows_args(p), k);
}

template <int DPL>
static void launch_rows_wide(xpcs_mt_plan* p, hipStream_t s)
{
    WideArgs w{};
    w.a = rows_args(p);
    int words = 0;
    for (int c = 0; c < 4; c++) {
        const int G = 8 << c;
        w.k[c] = rows_class(p, G, G * (c < 2 ? 8 : 16), true);
        words = std::max(words, kWave / G * (w.k[c].aw + w.k[c].bw));
    }
    const int64_t need = ((int64_t)p->h.P + 8 * kRowsWaves - 1) / (8 * kRowsWaves);
    const size_t lds = sizeof(uint32_t) * (size_t)(kRowsWaves * words);
    // what the chip holds at once (six workgroups a CU by registers); four such rounds balance whole waves of
    // long rows better (690 events a row: 6.9 against 7.2 ms), but cost every job without wide rows 4 us
    const int64_t fit = 256 * std::min<int64_t>(6, (int64_t)((160 << 10) / lds));
    const unsigned nb = (unsigned)std::max<int64_t>(1, std::min(need, fit));
    k_mt_rows_wide<DPL><<<nb, kWave * kRowsWaves, lds, s>>>(w, words);
}

// Rows of at most 64 events in place, the listed rows of 65 .. 1024 events,
// then the wide rows among them.
void launch_mt_rows(xpcs_mt_plan* p, hipStream_t s)
{
    const HostTables& h = p->h;
    const int bp = p->tune.reg_blocks > 0 ? p->tune.reg_blocks : 1 << 20;
    const int bl = p->tune.lds_blocks > 0 ? p->tune.lds_blocks : 4096;
    auto run = [&](auto dpl) {
        constexpr int D = decltype(dpl)::value;
        timer_begin(p, s, "k_mt_reg");
        launch_rows_class<8, 8, D>(p, s, bp);
        timer_end(p, s);
        timer_begin(p, s, "k_mt_lds");
        launch_rows_class<16, 8, D>(p, s, bl);
        launch_rows_class<32, 16, D>(p, s, bl);
        launch_rows_class<64, 16, D>(p, s, bl);
        launch_rows_wide<D>(p, s);
        timer_end(p, s);
    };
    if (h.dpl == 4) run(std::integral_constant<int, 4>{});
    else run(std::integral_constant<int, 8>{});
}

}  // namespace xpcs
