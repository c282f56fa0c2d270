// Dense path (DenseFilter, src/xpcs/filter/dense_filter.cpp:121-210, followed by
// Corr::multiTau2, src/xpcs/corr.cpp:315-431): thread-per-pixel streaming
// multi-tau over frame-major data.
//
// One thread owns one detector pixel and walks the frames in order.  A wave's
// loads of a frame are 64 consecutive pixels, so the raw IMM frames are read
// once, fully coalesced, with no transposed copy.  Frames are taken 16 at a
// time; within such a group the pairing of every level up to 2^4 is fixed at
// compile time, so levels 0..4 are fully unrolled (no shift-register moves,
// no branches) and only the levels above follow the group index (a
// wave-uniform branch).  Each level keeps its last 2*dpl values; a new level-L
// value x at index k adds x * x_L[k-d] to the lag-d sum for every lag d of the
// level.
//
// Lag sums are accumulated with FP64 fused multiply-adds, which is exact here:
// every value is a non-negative integer, and every product and partial sum of
// a pixel is at most S^2, S = the pixel's total count, so while S^2 < 2^53 no
// result is ever rounded.  A pixel with a larger total is listed by the first
// pass and recomputed with 64-bit integer sums by k_mt_dense_exact.
//
// IP and IF come from level-0 prefix sums captured at the schedule's frame
// boundaries (IP = S0(2^L (lf - tau')), IF = S0(2^L lf) - S0(2^L tau')); the
// boundary list is sorted on the host and walked with a wave-uniform index.
//
// Levels are processed K at a time (register budget).  The first pass reads the
// raw frames (dark subtraction, threshold and mask fused) and, when more
// levels remain, writes the level-K series frame-major ([lf_K][W*H], the
// column of a pixel is its raster index); each further pass reads the
// previous series with the same coalesced pattern.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "device_util.h"
#include "internal.h"

namespace xpcs {

// Largest pixel total S with S^2 < 2^53 (every lag sum exact in FP64).
constexpr uint32_t kExactF64Total = 94906265u;
constexpr int kGroup = 16;

// Levels per pass (register budget): dpl 4 at 4 levels keeps two waves per
// SIMD; dpl 8 at 3 levels runs one wave per SIMD and is as fast as 2 levels at
// two waves, with fewer passes over the coarsened series.
template <int DPL>
constexpr int dense_levels_per_pass()
{
    return DPL == 4 ? 4 : 3;
}

template <int DPL, bool FIRST, int l>
constexpr int lag_lo()
{
    // level 0 of the schedule has lags 1..2*dpl, every other level dpl+1..2*dpl
    return (FIRST && l == 0) ? 1 : DPL + 1;
}

template <int DPL, int K>
struct FState {
    double win[K][2 * DPL];   // win[l][j] = value j+1 steps back at level L0+l
    double acc[K][2 * DPL];   // lag sums, acc[l][d-1] for lag d
    double pend[K];           // first value of an incomplete pair (levels above the group)
};

// ST: uint32_t for counts, double for frame-weighted values (normalize_by_framesum)
template <typename ST>
struct SeriesOut {
    ST* col;                  // element k of the output series at col[k * stride]
    int64_t stride;
    uint32_t lf;              // values of the output level
};

// One value of level l (index k, wave-uniform): lag products, window shift,
// and pairing into level l+1 by the parity of k.
template <int DPL, int K, bool FIRST, int l, typename ST>
__device__ __forceinline__ void push_one(FState<DPL, K>& s, double v, uint32_t k, const SeriesOut<ST>& o)
{
    if constexpr (l < K) {
        constexpr int dlo = lag_lo<DPL, FIRST, l>();
#pragma unroll
        for (int d = dlo; d <= 2 * DPL; d++) s.acc[l][d - 1] = __builtin_fma(v, s.win[l][d - 1], s.acc[l][d - 1]);
#pragma unroll
        for (int j = 2 * DPL - 1; j > 0; j--) s.win[l][j] = s.win[l][j - 1];
        s.win[l][0] = v;
        if (k & 1u) push_one<DPL, K, FIRST, l + 1>(s, s.pend[l] + v, k >> 1, o);
        else s.pend[l] = v;
    } else {
        if (o.col && k < o.lf) o.col[(int64_t)k * o.stride] = (ST)v;
    }
}

// N consecutive values of level l, the first with index kb (N = 16 >> l).
// TAIL: the last, partial group; values with index >= lf of their level are
// zeroed (they do not exist in the series) and nothing reaches the levels
// above the group.
template <int DPL, int K, bool FIRST, bool TAIL, int l, int N, typename ST>
__device__ __forceinline__ void push_block(FState<DPL, K>& s, double (&v)[N], uint32_t kb, uint32_t n_in,
                                           const SeriesOut<ST>& o)
{
    if constexpr (TAIL) {
        const uint32_t lim = n_in >> l;
#pragma unroll
        for (int j = 0; j < N; j++)
            if (kb + j >= lim) v[j] = 0.0;
    }
    if constexpr (l < K) {
        constexpr int dlo = lag_lo<DPL, FIRST, l>();
#pragma unroll
        for (int j = 0; j < N; j++) {
#pragma unroll
            for (int d = dlo; d <= 2 * DPL; d++) {
                const double w = (j >= d) ? v[j >= d ? j - d : 0] : s.win[l][j >= d ? 0 : d - j - 1];
                s.acc[l][d - 1] = __builtin_fma(v[j], w, s.acc[l][d - 1]);
            }
        }
        double nw[2 * DPL];
#pragma unroll
        for (int i = 0; i < 2 * DPL; i++) nw[i] = (i < N) ? v[i < N ? N - 1 - i : 0] : s.win[l][i < N ? 0 : i - N];
#pragma unroll
        for (int i = 0; i < 2 * DPL; i++) s.win[l][i] = nw[i];
        if constexpr (N >= 2) {
            double u[N / 2];
#pragma unroll
            for (int j = 0; j < N / 2; j++) u[j] = v[2 * j] + v[2 * j + 1];
            push_block<DPL, K, FIRST, TAIL, l + 1, N / 2>(s, u, kb >> 1, n_in, o);
        } else if constexpr (!TAIL) {
            if (kb & 1u) push_one<DPL, K, FIRST, l + 1>(s, s.pend[l] + v[0], kb >> 1, o);
            else s.pend[l] = v[0];
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; j++)
            if (o.col && kb + j < o.lf) o.col[(int64_t)(kb + j) * o.stride] = (ST)v[j];
    }
}

// Dark subtraction and threshold of one raw value (n-scaled integers: kept iff
// n*raw - sum(dark) > max(floor(n*threshold), 0)).
__device__ __forceinline__ uint32_t dense_value(uint32_t raw, int32_t nscale, int32_t nds, int32_t th)
{
    const int32_t y = __mul24((int32_t)raw, nscale) + nds;
    return y > th ? (uint32_t)y : 0u;
}

// Input of a pass: the level-K series of the previous pass, the raw frames
// one 2-byte load per lane and frame, or the raw frames staged through LDS
// (evenly spaced frames, avg 1): a wave fetches a 16-frame x 64-pixel tile
// with two 16-byte loads per lane, DEPTH tiles ahead of use.
enum DenseInput { kSeries = 0, kRawLanes = 1, kRawTiles = 2 };
constexpr int kTileDepth = 3;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// FP (normalize_by_framesum, main.cpp:313-336): level-0 values are the counts
// times fw[frame], the series between passes are FP64, and G2/IP/IF are FP64
// sums stored as bit patterns (no exactness bound, no integer redo);
// pix_total stays the raw count total.
template <int DPL, int K, int MODE, bool FP>
__global__ void __launch_bounds__(256)
k_mt_dense_f64(const uint8_t* __restrict__ imm, const int64_t* __restrict__ sel_off, int64_t tile_off0,
               int64_t tile_step, int avg, const int32_t* __restrict__ pix2c, uint32_t npix,
               const int64_t* __restrict__ dark_sum, const int64_t* __restrict__ thr, int32_t nscale,
               const std::conditional_t<FP, double, uint32_t>* __restrict__ series_in, uint32_t n_in,
               const LevelParam* __restrict__ levels, int32_t L0, int32_t nlev_pass, const int4* __restrict__ bnd,
               int32_t nbnd, int32_t T, int64_t* __restrict__ G2, int64_t* __restrict__ IP,
               int64_t* __restrict__ IF, uint64_t* __restrict__ pix_total,
               std::conditional_t<FP, double, uint32_t>* __restrict__ series_out, uint32_t lf_out,
               uint32_t* __restrict__ redo_count, int32_t* __restrict__ redo_list, const double* __restrict__ fw,
               bool w32, const uint32_t* __restrict__ only)
{
    using ST = std::conditional_t<FP, double, uint32_t>;   // series element
    constexpr bool RAW = MODE != kSeries;
    // only: a flag per 64 pixels; waves without it have nothing to do
    if (RAW && only && only[(blockIdx.x * blockDim.x + threadIdx.x) >> 6] == 0u) return;
    // values of a group: integers from the raw frames, or the input series
    using XT = std::conditional_t<FP && !RAW, double, uint32_t>;
    constexpr bool TILES = MODE == kRawTiles;
    __shared__ u32x4 s_tile[TILES ? 4 : 1][2][64];

    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int32_t c = gid < npix ? pix2c[gid] : -1;
    const bool active = c >= 0;
    if constexpr (TILES) {
        // every lane of a wave takes part in the tile loads; a wave without a
        // mapped pixel has nothing to do
        if (__ballot(active) == 0ull) return;
    } else {
        if (!active) return;
    }
    FState<DPL, K> s;
#pragma unroll
    for (int l = 0; l < K; l++) {
        s.pend[l] = 0.0;
#pragma unroll
        for (int j = 0; j < 2 * DPL; j++) {
            s.win[l][j] = 0.0;
            s.acc[l][j] = 0.0;
        }
    }
    const SeriesOut<ST> o{(active && series_out && nlev_pass == K) ? series_out + gid : nullptr, (int64_t)npix,
                          lf_out};
    int32_t nds = 0, th = 0;
    if constexpr (RAW) {
        if (active) {
            nds = dark_sum ? -(int32_t)dark_sum[c] : 0;
            const int64_t t = thr ? thr[c] : 0;
            th = t < 0 ? 0 : (t > INT32_MAX ? INT32_MAX : (int32_t)t);
        }
    }
    const int64_t rowT = (int64_t)(active ? c : 0) * T;
    uint32_t S = 0;
    double Sd = 0.0;   // FP: running sum of the weighted values
    int bi = 0;
    if constexpr (RAW) {
        while (bi < nbnd && bnd[bi].x == 0) bi++;
    }
    int nextb = (RAW && bi < nbnd) ? bnd[bi].x : INT_MAX;

    // boundary captures inside group t0 (wave-uniform test), then the running sums
    auto captures = [&](const XT (&x)[kGroup], const double (&v)[kGroup], uint32_t t0) {
        if constexpr (RAW) {
            while (nextb <= (int)(t0 + kGroup)) {
                const int4 b = bnd[bi];
                const int n = b.x - (int)t0;
                if constexpr (FP) {
                    double part = Sd;
#pragma unroll
                    for (int u = 0; u < kGroup; u++) part += (u < n) ? v[u] : 0.0;
                    if (active) {
                        if (b.y == 0) IP[rowT + b.z] = (int64_t)__double_as_longlong(part);
                        else if (b.y == 1) IF[rowT + b.z] = (int64_t)__double_as_longlong(part);
                        else
                            IF[rowT + b.z] =
                                (int64_t)__double_as_longlong(part - __longlong_as_double((long long)IF[rowT + b.z]));
                    }
                } else {
                    uint32_t part = S;
#pragma unroll
                    for (int u = 0; u < kGroup; u++) part += (u < n) ? x[u] : 0u;
                    if (active) {
                        if (b.y == 0) put_sum(IP, rowT + b.z, (int64_t)part, w32);
                        else if (b.y == 1) put_sum(IF, rowT + b.z, (int64_t)part, w32);
                        else put_sum(IF, rowT + b.z, (int64_t)part - get_sum(IF, rowT + b.z, w32), w32);
                    }
                }
                bi++;
                nextb = bi < nbnd ? bnd[bi].x : INT_MAX;
            }
#pragma unroll
            for (int u = 0; u < kGroup; u++) S += (uint32_t)x[u];
            if constexpr (FP) {
#pragma unroll
                for (int u = 0; u < kGroup; u++) Sd += v[u];
            }
        }
    };
    // the group's values (counts x fw[frame] for FP raw input)
    auto weigh = [&](const XT (&x)[kGroup], double (&v)[kGroup], uint32_t t0) {
#pragma unroll
        for (int u = 0; u < kGroup; u++) {
            v[u] = (double)x[u];
            if constexpr (FP && RAW) v[u] *= fw[min(t0 + (uint32_t)u, n_in - 1)];
        }
    };
    auto group = [&](XT (&x)[kGroup], uint32_t t0) {
        double v[kGroup];
        if constexpr (FP) {
            weigh(x, v, t0);
            captures(x, v, t0);
        } else {   // counts: captures read x only
            captures(x, v, t0);
            weigh(x, v, t0);
        }
        push_block<DPL, K, RAW, false, 0, kGroup>(s, v, t0, n_in, o);
    };
    auto tail_group = [&](XT (&x)[kGroup], uint32_t t0) {
#pragma unroll
        for (int u = 0; u < kGroup; u++)
            if (t0 + (uint32_t)u >= n_in) x[u] = XT(0);
        double v[kGroup];
        if constexpr (FP) {
            weigh(x, v, t0);
            captures(x, v, t0);
        } else {
            captures(x, v, t0);
            weigh(x, v, t0);
        }
        push_block<DPL, K, RAW, true, 0, kGroup>(s, v, t0, n_in, o);
    };
    const uint32_t nfull = n_in / kGroup * kGroup;

    if constexpr (TILES) {
        // lane = 8 * f + j loads frame t0 + 8 * i + f, pixels 8 j .. 8 j + 7 of
        // the wave, for i = 0, 1; in LDS the tile is [16 frames][64 pixels]
        const uint32_t lane = threadIdx.x & 63u;
        const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const uint8_t* wsrc = imm + tile_off0 + 2 * (int64_t)(gid - lane) + 16 * (lane & 7u);
        auto issue = [&](u32x4 (&r)[2], uint32_t t0) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t t = min(t0 + 8u * i + (lane >> 3), n_in - 1);
                r[i] = *reinterpret_cast<const u32x4*>(wsrc + (int64_t)t * tile_step);
            }
        };
        auto stage = [&](const u32x4 (&r)[2], uint32_t (&x)[kGroup]) {
            s_tile[w][0][lane] = r[0];
            s_tile[w][1][lane] = r[1];
            wave_sync();
            const uint16_t* t16 = reinterpret_cast<const uint16_t*>(&s_tile[w][0][0]);
#pragma unroll
            for (int u = 0; u < kGroup; u++) x[u] = dense_value(t16[u * 64 + lane], nscale, nds, th);
            wave_sync();
        };
        u32x4 ring[kTileDepth][2];
#pragma unroll
        for (int d = 0; d < kTileDepth; d++) issue(ring[d], (uint32_t)(d * kGroup));
        for (uint32_t g0 = 0; g0 < nfull; g0 += kTileDepth * kGroup) {
#pragma unroll
            for (int d = 0; d < kTileDepth; d++) {
                const uint32_t t0 = g0 + (uint32_t)(d * kGroup);
                if (t0 < nfull) {
                    uint32_t x[kGroup];
                    stage(ring[d], x);
                    issue(ring[d], t0 + kTileDepth * kGroup);
                    group(x, t0);
                }
            }
        }
        if (nfull < n_in) {
            u32x4 r[2];
            issue(r, nfull);
            uint32_t x[kGroup];
            stage(r, x);
            tail_group(x, nfull);
        }
    } else {
        const uint16_t* col16 = reinterpret_cast<const uint16_t*>(imm) + gid;
        const ST* col32 = RAW ? nullptr : series_in + gid;
        // loads of group t0 (frame indices clamped into range; the tail zeroes them)
        auto load = [&](XT (&r)[kGroup], uint32_t t0) {
#pragma unroll
            for (int u = 0; u < kGroup; u++) {
                const uint32_t t = min(t0 + (uint32_t)u, n_in - 1);
                if constexpr (RAW) r[u] = *reinterpret_cast<const uint16_t*>(
                                              reinterpret_cast<const uint8_t*>(col16) + sel_off[t]);
                else r[u] = col32[(int64_t)t * npix];
            }
        };
        auto values = [&](XT (&x)[kGroup], const XT (&r)[kGroup], uint32_t t0) {
            if constexpr (RAW) {
                if (avg == 1) {
#pragma unroll
                    for (int u = 0; u < kGroup; u++) x[u] = dense_value(r[u], nscale, nds, th);
                } else {
#pragma unroll
                    for (int u = 0; u < kGroup; u++) {
                        const uint32_t t = min(t0 + (uint32_t)u, n_in - 1);
                        uint32_t a_sum = 0;
                        for (int a = 0; a < avg; a++) {
                            const uint32_t raw = *reinterpret_cast<const uint16_t*>(
                                reinterpret_cast<const uint8_t*>(col16) + sel_off[(int64_t)t * avg + a]);
                            a_sum += dense_value(raw, nscale, nds, th);
                        }
                        x[u] = a_sum;
                    }
                }
            } else {
#pragma unroll
                for (int u = 0; u < kGroup; u++) x[u] = r[u];
            }
        };
        XT rcur[kGroup];
        if (RAW && avg != 1) {
#pragma unroll
            for (int u = 0; u < kGroup; u++) rcur[u] = XT(0);
        } else {
            load(rcur, 0);
        }
        for (uint32_t t0 = 0; t0 < nfull; t0 += kGroup) {
            // next group's loads are issued before this group is processed
            XT rnext[kGroup];
            if (RAW && avg != 1) {
#pragma unroll
                for (int u = 0; u < kGroup; u++) rnext[u] = XT(0);
            } else {
                load(rnext, t0 + kGroup);
            }
            XT x[kGroup];
            values(x, rcur, t0);
            group(x, t0);
#pragma unroll
            for (int u = 0; u < kGroup; u++) rcur[u] = rnext[u];
        }
        if (nfull < n_in) {
            XT x[kGroup];
            values(x, rcur, nfull);
            tail_group(x, nfull);
        }
    }
    if (!active) return;
    if constexpr (RAW) {
        pix_total[c] = S;
        // boundaries at frame 0 cover no frames
        for (int i = 0; i < nbnd; i++) {
            const int4 b = bnd[i];
            if (b.x != 0) break;
            if (b.y == 0) put_sum(IP, rowT + b.z, 0, !FP && w32);
            else if (b.y == 1) put_sum(IF, rowT + b.z, 0, !FP && w32);
        }
        if (!FP && S > kExactF64Total) redo_list[atomicAdd(redo_count, 1u)] = (int32_t)gid;
    }
#pragma unroll
    for (int l = 0; l < K; l++) {
        if (l < nlev_pass) {
            const LevelParam lp = levels[L0 + l];
            const int dlo = (RAW && l == 0) ? 1 : DPL + 1;
#pragma unroll
            for (int d = 1; d <= 2 * DPL; d++) {
                const int rel = d - lp.lo;
                if (d >= dlo && rel >= 0 && rel < lp.count)
                    G2[rowT + lp.first + rel] =
                        FP ? (int64_t)__double_as_longlong(s.acc[l][d - 1]) : (int64_t)s.acc[l][d - 1];
            }
        }
    }
}

// ---- raw pass over counts: two-element dot products --------------------------
// The same streaming pass (thread per pixel, 16-frame groups, K levels) with
// the values of two consecutive frames in one register: a lag sum takes one
// two-element integer dot product per two frames (even lags against earlier
// words, odd lags against words one frame off) instead of two FP64
// multiply-adds, the pair sums and the running total are dot products with
// (1, 1), and dark subtraction and threshold work on both halves at once.
//
// Lag sums run in 32 bits and are added to 64-bit totals (flush) before they
// could overflow: between flushes a pixel counts at most `chunk` (kDotChunk, or
// half of it), each of those counts meets one value per lag, and values have 16
// bits, so a lag sum is at most kDotChunk 65535 < 2^32.  That also keeps every
// value of a group's levels in 16 bits.  A wave that meets a 16-frame group
// beyond `chunk` in any pixel flags its 64 pixels and stops; the FP64 kernel
// then takes exactly those.
//
// The FP64 form was bound by vector issue (20 instructions per frame and
// wave, two waves per SIMD); measured on the 512 x 512 x 20,000-frame job
// (dpl 4, two darks): 3.45 -> 2.58 ms (11 GB of HBM traffic, 4.3 TB/s: memory
// now bounds it), on 333 x 251 x 3001 frames (dpl 8) 1.04 -> 0.36 ms.
constexpr uint32_t kDotChunk = 64500u;
using i16x2 = __attribute__((ext_vector_type(2))) short;
using u16x2 = __attribute__((ext_vector_type(2))) unsigned short;

__device__ __forceinline__ uint32_t dot2_u16(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_udot2(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b), c, false);
}

template <int DPL, int K>
struct DState {
    uint32_t win[K][DPL];       // win[l][j]: word j + 1 back at level l
    uint32_t sh[K][DPL];        // the same one frame earlier: (last of word j + 2 back, first of word j + 1 back)
    uint32_t acc[K][2 * DPL];   // lag sums since the last flush
};

// Lags of the first K levels, and the slot of lag d at level l among them.
template <int DPL, int K>
constexpr int dot_lags() { return 2 * DPL + (K - 1) * DPL; }
template <int DPL>
constexpr int dot_slot(int l, int d) { return l * DPL + d - 1; }

// Lag sums of the NW words of level l.
template <int DPL, int K, int l, int NW>
__device__ __forceinline__ void dot_level(DState<DPL, K>& s, const uint32_t (&cur)[NW])
{
    constexpr int lo = lag_lo<DPL, true, l>();
    uint32_t sc[NW];
#pragma unroll
    for (int i = 0; i < NW; i++) {
        const uint32_t prev = i > 0 ? cur[i > 0 ? i - 1 : 0] : s.win[l][0];
        sc[i] = __builtin_amdgcn_alignbit(cur[i], prev, 16);
#pragma unroll
        for (int lag = lo; lag <= 2 * DPL; lag++) {
            const int m = lag / 2;
            uint32_t w;
            if (lag & 1) w = m <= i ? sc[m <= i ? i - m : 0] : s.sh[l][m <= i ? 0 : m - i - 1];
            else w = m <= i ? cur[m <= i ? i - m : 0] : s.win[l][m <= i ? 0 : m - i - 1];
            s.acc[l][lag - 1] = dot2_u16(cur[i], w, s.acc[l][lag - 1]);
        }
    }
    uint32_t nw[DPL], ns[DPL];
#pragma unroll
    for (int j = 0; j < DPL; j++) {
        nw[j] = j < NW ? cur[j < NW ? NW - 1 - j : 0] : s.win[l][j < NW ? 0 : j - NW];
        ns[j] = j < NW ? sc[j < NW ? NW - 1 - j : 0] : s.sh[l][j < NW ? 0 : j - NW];
    }
#pragma unroll
    for (int j = 0; j < DPL; j++) {
        s.win[l][j] = nw[j];
        s.sh[l][j] = ns[j];
    }
}

// The lag sums into the lane's 64-bit totals, tot[slot][lane].
template <int DPL, int K>
__device__ __forceinline__ void dot_flush(DState<DPL, K>& s, unsigned long long* tot)
{
#pragma unroll
    for (int l = 0; l < K; l++)
#pragma unroll
        for (int d = (l == 0 ? 1 : DPL + 1); d <= 2 * DPL; d++) {
            atomicAdd(tot + dot_slot<DPL>(l, d) * 64, (unsigned long long)s.acc[l][d - 1]);
            s.acc[l][d - 1] = 0u;
        }
}

__device__ __forceinline__ u16x2 as_pair(uint32_t w) { return __builtin_bit_cast(u16x2, w); }
__device__ __forceinline__ uint32_t as_word(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// The next level's word from two words of a level: (a.lo + a.hi, b.lo + b.hi),
// saturated.  (Dot products with (1, 1) would need wait states before every
// use.)
__device__ __forceinline__ uint32_t pair_up(uint32_t a, uint32_t b)
{
    const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05040100u), hi = __builtin_amdgcn_perm(b, a, 0x07060302u);
    return as_word(__builtin_elementwise_add_sat(as_pair(lo), as_pair(hi)));
}

struct DotArgs {
    const uint8_t* src;           // payload of frame t at src + t * step
    int64_t step;
    const int32_t* pix2c;
    uint32_t npix, n_in, chunk;
    const int64_t* dark_sum;
    const int64_t* thr;
    int32_t nscale;
    const LevelParam* levels;
    int32_t nlev_pass;
    const int32_t* cap;           // distinct frame boundaries, sorted, and an entry beyond every frame
    int32_t ncap, T;
    const int4* tau_bnd;          // per tau: boundary of IP, of the IF head, of the level's end
    uint32_t* cap_sums;           // [boundary][npix] sums below the boundary
    int64_t* G2;
    int64_t* IP;
    int64_t* IF;
    uint64_t* pix_total;
    uint32_t* series_out;
    uint32_t lf_out;
    uint32_t* redo_count;
    int32_t* redo_list;
    uint32_t* wave_flags;         // per 64 pixels: left to the FP64 kernel
    const uint32_t* bright;       // waves that k_dense_look flagged; NULL: it has not run
    uint32_t most;                // beyond so many of them all are left to the FP64 kernel
    bool w32;
};

// A look at groups across the run before the dot kernel: a wave with one above
// two thirds of the chunk is likely to pass it somewhere, and would then have
// walked its frames for nothing.  Flags such waves and counts them.  Speckle
// frames of a mean of 300 (900) counts, 333 x 251 x 3001, dpl 8: 1.54 (1.34) ->
// 1.24 (1.25) ms, the FP64 kernel's own time, where the dot kernel alone had
// taken waves to their first group beyond 26000; of 300 scaled counts, 512 x
// 512 x 6000 with two darks, dpl 4: 2.0 -> 1.65 ms; of 600: 1.74 -> 1.42 ms.  The
// look takes 7 to 10 us.
constexpr uint32_t kDotLookFrames = 1024u;   // shorter runs: not worth a launch
constexpr int kLookGroups = 4;

__global__ void __launch_bounds__(256)
k_dense_look(const uint8_t* __restrict__ src, int64_t step, const int32_t* __restrict__ pix2c, uint32_t npix,
             uint32_t n_in, const int64_t* __restrict__ dark_sum, const int64_t* __restrict__ thr, int32_t nscale,
             uint32_t limit, uint32_t* __restrict__ wave_flags, uint32_t* __restrict__ bright)
{
    const uint32_t gid = blockIdx.x * 256u + threadIdx.x;
    const int32_t c = gid < npix ? pix2c[gid] : -1;
    bool hit = false;
    if (c >= 0) {
        const int32_t nds = -(int32_t)dark_sum[c];
        const int64_t t = thr[c];
        const int32_t th = t < 0 ? 0 : (t > INT32_MAX ? INT32_MAX : (int32_t)t);
        const uint8_t* col = src + 2 * (int64_t)gid;
#pragma unroll
        for (int g = 0; g < kLookGroups; g++) {
            const uint32_t t0 = n_in / kGroup * (2u * (uint32_t)g + 1u) / (2u * kLookGroups) * kGroup;
            uint32_t sum = 0u;
#pragma unroll
            for (int u = 0; u < kGroup; u++)
                sum += dense_value(*reinterpret_cast<const uint16_t*>(col + (int64_t)(t0 + (uint32_t)u) * step), nscale, nds, th);
            hit |= sum > limit;
        }
    }
    const uint64_t m = __ballot(hit);
    if ((threadIdx.x & 63u) == 0u && gid < npix) {
        wave_flags[gid >> 6] = m != 0ull;
        if (m != 0ull) atomicAdd(bright, 1u);
    }
}


struct __attribute__((packed, aligned(2))) Raw8 {
    uint32_t w[4];
};

// DARK: n-scaled values y = n raw - sum(dark), kept iff y > max(threshold, 0):
// with m = floor((max(threshold, 0) + sum(dark)) / n) and t = max(raw - m, 0)
// that is t > 0 and y = n t + (n m - sum(dark)).  t is limited so that y fits
// 16 bits (a limited value is above 65535 - n, n at most 1024) and t 15: with
// n >= 2 that limits no further, with n = 1 to 32767, and `chunk` is below that.
// So a limited value alone passes `chunk`.
//
// W neighbouring waves to a workgroup and two waves per SIMD: more waves in
// flight scatter the frame reads (512 x 512 x 20,000 frames, dpl 4: 2.58 ms
// with 8 waves a workgroup, 2.65 with 4, 2.9 with 1; 3.2 and 3.6 ms at three
// and four waves per SIMD).  Four tiles in flight: 2.58 against 2.66 ms with
// three.
template <int DPL, int K, bool DARK, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_mt_dense_dot(const DotArgs a)
{
    constexpr int kDepth = 4;   // 16-frame tiles in flight
    __shared__ u32x4 s_tile_[W][2 * 64];
    __shared__ unsigned long long s_tot[W][dot_lags<DPL, K>()][64];
    const uint32_t lane = threadIdx.x & 63u;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    u32x4* s_tile = s_tile_[w];
    // consecutive workgroups go to the eight XCDs in turn: each takes a
    // contiguous eighth of the detector
    const uint32_t blk = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t gid = blk * (64u * W) + threadIdx.x;
    unsigned long long* tot = &s_tot[w][0][lane];
    const uint32_t n_in = a.n_in;
    const int32_t c = gid < a.npix ? a.pix2c[gid] : -1;
    const bool active = c >= 0;
    if (__ballot(active) == 0ull) return;
    const bool left = a.bright && (*a.bright > a.most || a.wave_flags[gid >> 6] != 0u);
    if (lane == 0) a.wave_flags[gid >> 6] = left;
    if (left) return;
    uint32_t rm = 0u, c0 = 0u, tlim = 0u, nsc = 0u;   // in both halves
    if constexpr (DARK) {
        const int64_t n = a.nscale;
        const int64_t ds = active ? a.dark_sum[c] : 0;
        const int64_t th = active ? a.thr[c] : 0;
        const int64_t m = min(((th < 0 ? 0 : th) + ds) / n, (int64_t)65535);
        int64_t k0 = n * m - ds, tl = min((int64_t)32767, (65535 - k0) / n), sc = n;
        if (tl < 1) {
            // the smallest kept value passes 16 bits: any kept value ends the wave
            k0 = 65535;
            tl = 1;
            sc = 0;
        }
        rm = (uint32_t)m * 0x00010001u;
        c0 = ((uint32_t)k0 & 0xFFFFu) * 0x00010001u;
        tlim = (uint32_t)tl * 0x00010001u;
        nsc = (uint32_t)sc * 0x00010001u;
    }
    DState<DPL, K> s;
#pragma unroll
    for (int l = 0; l < K; l++) {
#pragma unroll
        for (int j = 0; j < DPL; j++) s.win[l][j] = s.sh[l][j] = 0u;
#pragma unroll
        for (int j = 0; j < 2 * DPL; j++) {
            s.acc[l][j] = 0u;
        }
    }
#pragma unroll
    for (int j = 0; j < dot_lags<DPL, K>(); j++) tot[j * 64] = 0ull;
    const int64_t rowT = (int64_t)(active ? c : 0) * a.T;
    uint32_t S = 0u, S0 = 0u;      // running total, total at the last flush
    // Boundaries, two ahead in scalar registers.  Their sums leave frame-major,
    // a full line per wave: written to the pixels' rows as they came (4 bytes
    // per pixel, each line revisited ~100 times over the job) they made 18 M
    // partial HBM writes on the 512 x 512 x 20,000-frame job.
    using Cap = const __attribute__((address_space(4))) int32_t*;
    const Cap cap = (Cap)(uintptr_t)a.cap;
    auto boundary = [&](int i) { return cap[__builtin_amdgcn_readfirstlane(min(i, a.ncap))]; };
    int bi = 0, cur = boundary(0), nxt = boundary(1);
    auto capture = [&](uint32_t part) {
        if (active) a.cap_sums[(int64_t)bi * a.npix + gid] = part;
        cur = nxt;
        bi++;
        nxt = boundary(bi + 1);
    };
    while (cur == 0) capture(0u);   // a boundary at frame 0 covers no frames

    // one group; `over` once a pixel of the wave has passed the chunk (what the
    // group then adds is not used)
    bool over = false;
    auto group = [&](const uint32_t (&raw)[8], uint32_t t0, auto tail) {
        constexpr bool TAIL = decltype(tail)::value;
        uint32_t x0[8], x1[4], x2[2], x3[1];   // words of levels 0 .. 3
#pragma unroll
        for (int i = 0; i < 8; i++) {
            uint32_t x = raw[i];
            if constexpr (DARK) {
                u16x2 t = __builtin_elementwise_sub_sat(as_pair(x), as_pair(rm));
                t = __builtin_elementwise_min(t, as_pair(tlim));
                // all ones where t > 0 (t is below 2^15)
                const i16x2 kept = (i16x2{0, 0} - __builtin_bit_cast(i16x2, t)) >> 15;
                const uint32_t add = as_word(__builtin_bit_cast(u16x2, kept)) & c0;
                x = as_word(t * as_pair(nsc) + as_pair(add));
            }
            if constexpr (TAIL) {
                const uint32_t t = t0 + 2u * (uint32_t)i;
                x = t + 1 < n_in ? x : t < n_in ? x & 0xFFFFu : 0u;
            }
            x0[i] = x;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) x1[i] = pair_up(x0[2 * i], x0[2 * i + 1]);
#pragma unroll
        for (int i = 0; i < 2; i++) x2[i] = pair_up(x1[2 * i], x1[2 * i + 1]);
        x3[0] = pair_up(x2[0], x2[1]);
        // the group's sum (saturated halves pass the chunk)
        const uint32_t gs = (x3[0] & 0xFFFFu) + (x3[0] >> 16);
        if constexpr (TAIL) {
            // values past the end of their level do not exist in its series
            auto cut = [&](uint32_t* w, int nw, int l) {
                for (int i = 0; i < nw; i++) {
                    const uint32_t k = (t0 >> l) + 2u * (uint32_t)i, lim = n_in >> l;
                    w[i] = k + 1 < lim ? w[i] : k < lim ? w[i] & 0xFFFFu : 0u;
                }
            };
            cut(x1, 4, 1);
            x2[0] = pair_up(x1[0], x1[1]);
            x2[1] = pair_up(x1[2], x1[3]);
            cut(x2, 2, 2);
            x3[0] = pair_up(x2[0], x2[1]);
            cut(x3, 1, 3);
        }
        if (__ballot(active && S + gs - S0 > a.chunk) != 0ull) {
            over = over || __ballot(active && gs > a.chunk) != 0ull;
            dot_flush<DPL, K>(s, tot);
            S0 = S;
        }
        // boundary captures (wave-uniform), then the running total
        while (cur <= (int)(t0 + kGroup)) {
            const int n = cur - (int)t0;
            uint32_t part = S;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t ones = n > 2 * i + 1 ? 0x00010001u : n > 2 * i ? 1u : 0u;
                part = dot2_u16(x0[i], ones, part);
            }
            capture(part);
        }
        S += gs;
        dot_level<DPL, K, 0, 8>(s, x0);
        if constexpr (K > 1) dot_level<DPL, K, 1, 4>(s, x1);
        if constexpr (K > 2) dot_level<DPL, K, 2, 2>(s, x2);
        if constexpr (K > 3) dot_level<DPL, K, 3, 1>(s, x3);
        if (a.lf_out && active) {
            // level K's values: the sum of 16 frames, or halves of words
            const uint32_t kb = t0 >> K;
            uint32_t* o = a.series_out + (int64_t)kb * a.npix + gid;
#pragma unroll
            for (int i = 0; i < (16 >> K); i++) {
                uint32_t v;
                if constexpr (K == 4) {
                    v = TAIL ? (kb < a.lf_out ? gs : 0u) : gs;
                } else {
                    const uint32_t word = K == 3 ? x3[0] : x2[i >> 1];
                    v = (i & 1) ? word >> 16 : word & 0xFFFFu;
                }
                if (!TAIL || kb + (uint32_t)i < a.lf_out) o[(int64_t)i * a.npix] = v;
            }
        }
    };

    // lane = 8 f + j loads frames t0 + 2 f and t0 + 2 f + 1, pixels 8 j .. 8 j + 7
    // of the wave; in LDS the tile is [8 frame pairs][64 pixels]
    uint32_t px = (gid - lane) + 8u * (lane & 7u);
    const uint32_t back = px + 8u > a.npix ? px + 8u - a.npix : 0u;   // 1..7 for the last pixels' lane
    px -= back;
    const bool partial = __builtin_amdgcn_readfirstlane((int)((gid - lane) + 64u > a.npix)) != 0;
    const uint8_t* src = a.src + 2 * (int64_t)px;
    auto issue = [&](Raw8 (&r)[2], uint32_t t0) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t t = min(t0 + 2u * (lane >> 3) + (uint32_t)i, n_in - 1);
            const uint8_t* q = src + (int64_t)t * a.step;
            r[i] = *reinterpret_cast<const Raw8*>(q);
        }
    };
    auto stage = [&](Raw8 (&r)[2], uint32_t (&x)[8]) {
        if (partial) {
            // the detector's last pixels, read from its last 8: move them down
            // (lanes past the detector keep what they read)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                if (back & 1u) {
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        r[i].w[k] = (r[i].w[k] >> 16) | (k < 3 ? r[i].w[k < 3 ? k + 1 : 3] << 16 : 0u);
                }
                if (back & 2u) {
                    r[i].w[0] = r[i].w[1];
                    r[i].w[1] = r[i].w[2];
                    r[i].w[2] = r[i].w[3];
                }
                if (back & 4u) {
                    r[i].w[0] = r[i].w[2];
                    r[i].w[1] = r[i].w[3];
                }
            }
        }
        uint32_t q[8];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            q[2 * k] = __builtin_amdgcn_perm(r[1].w[k], r[0].w[k], 0x05040100u);
            q[2 * k + 1] = __builtin_amdgcn_perm(r[1].w[k], r[0].w[k], 0x07060302u);
        }
        s_tile[2 * lane] = u32x4{q[0], q[1], q[2], q[3]};
        s_tile[2 * lane + 1] = u32x4{q[4], q[5], q[6], q[7]};
        wave_sync();
        const uint32_t* t32 = reinterpret_cast<const uint32_t*>(&s_tile[0]);
#pragma unroll
        for (int f = 0; f < 8; f++) x[f] = t32[f * 64 + lane];
        wave_sync();
    };
    const uint32_t nfull = n_in / kGroup * kGroup;
    Raw8 ring[kDepth][2];
#pragma unroll
    for (int d = 0; d < kDepth; d++) issue(ring[d], (uint32_t)(d * kGroup));
    // whole rounds of the ring without a test per tile: a tile skipped on some
    // path would make every wait drain the loads in flight
    uint32_t g0 = 0;
    for (; g0 + kDepth * kGroup <= nfull; g0 += kDepth * kGroup) {
        if (over) break;
#pragma unroll
        for (int d = 0; d < kDepth; d++) {
            const uint32_t t0 = g0 + (uint32_t)(d * kGroup);
            uint32_t x[8];
            stage(ring[d], x);
            issue(ring[d], t0 + kDepth * kGroup);
            group(x, t0, std::false_type{});
        }
    }
    for (; g0 < nfull && !over; g0 += kGroup) {
        uint32_t x[8];
        stage(ring[0], x);
#pragma unroll
        for (int d = 0; d + 1 < kDepth; d++) {
            ring[d][0] = ring[d + 1][0];
            ring[d][1] = ring[d + 1][1];
        }
        group(x, g0, std::false_type{});
    }
    if (!over && nfull < n_in) {
        Raw8 r[2];
        issue(r, nfull);
        uint32_t x[8];
        stage(r, x);
        group(x, nfull, std::true_type{});
    }
    if (over) {
        if (lane == 0) a.wave_flags[gid >> 6] = 1u;
        return;
    }
    dot_flush<DPL, K>(s, tot);
    if (!active) return;
    a.pix_total[c] = S;
    // IP = S(B_ip), IF = S(B_end) - S(B_head)
#pragma unroll 4
    for (int t = 0; t < a.T; t++) {
        const int4 b = a.tau_bnd[t];
        const uint32_t ip = a.cap_sums[(int64_t)b.x * a.npix + gid];
        const uint32_t head = a.cap_sums[(int64_t)b.y * a.npix + gid], end = a.cap_sums[(int64_t)b.z * a.npix + gid];
        put_sum(a.IP, rowT + t, (int64_t)ip, a.w32);
        put_sum(a.IF, rowT + t, (int64_t)end - (int64_t)head, a.w32);
    }
    if (S > kExactF64Total) a.redo_list[atomicAdd(a.redo_count, 1u)] = (int32_t)gid;
#pragma unroll
    for (int l = 0; l < K; l++) {
        if (l < a.nlev_pass) {
            const LevelParam lp = a.levels[l];
            const int dlo = l == 0 ? 1 : DPL + 1;
#pragma unroll
            for (int d = 1; d <= 2 * DPL; d++) {
                const int rel = d - lp.lo;
                if (d >= dlo && rel >= 0 && rel < lp.count)
                    a.G2[rowT + lp.first + rel] = (int64_t)tot[dot_slot<DPL>(l, d) * 64];
            }
        }
    }
}

// ---- exact 64-bit integer variant for the listed pixels ---------------------

template <int DPL, int K>
struct XState {
    uint32_t win[K][2 * DPL];
    uint32_t pend[K];
    uint64_t acc[K][2 * DPL];
};

template <int DPL, int K, bool FIRST, int l>
__device__ __forceinline__ void push_exact(XState<DPL, K>& s, uint32_t x, uint32_t (&cnt)[K])
{
    if constexpr (l < K) {
        constexpr int dlo = lag_lo<DPL, FIRST, l>();
#pragma unroll
        for (int d = dlo; d <= 2 * DPL; d++) s.acc[l][d - 1] += (uint64_t)x * (uint64_t)s.win[l][d - 1];
#pragma unroll
        for (int j = 2 * DPL - 1; j > 0; j--) s.win[l][j] = s.win[l][j - 1];
        s.win[l][0] = x;
        const uint32_t k = cnt[l]++;
        if (k & 1u) push_exact<DPL, K, FIRST, l + 1>(s, s.pend[l] + x, cnt);
        else s.pend[l] = x;
    }
}

// Lag sums of the pixels listed by k_mt_dense_f64 (totals too large for exact
// FP64), one thread per listed pixel, 64-bit integer accumulation.  Only G2
// is rewritten: IP, IF and the series are integer results of the FP64 pass.
template <int DPL, int K, bool RAW>
__global__ void __launch_bounds__(256)
k_mt_dense_exact(const uint8_t* __restrict__ imm, const int64_t* __restrict__ sel_off, int avg,
                 const int32_t* __restrict__ pix2c, uint32_t npix, const int64_t* __restrict__ dark_sum,
                 const int64_t* __restrict__ thr, int32_t nscale, const uint32_t* __restrict__ series_in,
                 uint32_t n_in, const LevelParam* __restrict__ levels, int32_t L0, int32_t nlev_pass, int32_t T,
                 int64_t* __restrict__ G2, const uint32_t* __restrict__ redo_count,
                 const int32_t* __restrict__ redo_list)
{
    const uint32_t n = *redo_count;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t gid = (uint32_t)redo_list[i];
        const int32_t c = pix2c[gid];
        XState<DPL, K> s;
        uint32_t cnt[K];
#pragma unroll
        for (int l = 0; l < K; l++) {
            s.pend[l] = 0u;
            cnt[l] = 0u;
#pragma unroll
            for (int j = 0; j < 2 * DPL; j++) {
                s.win[l][j] = 0u;
                s.acc[l][j] = 0ull;
            }
        }
        int32_t nds = 0, th = 0;
        if constexpr (RAW) {
            nds = dark_sum ? -(int32_t)dark_sum[c] : 0;
            const int64_t t = thr ? thr[c] : 0;
            th = t < 0 ? 0 : (t > INT32_MAX ? INT32_MAX : (int32_t)t);
        }
        for (uint32_t t = 0; t < n_in; t++) {
            uint32_t x;
            if constexpr (RAW) {
                x = 0;
                for (int a = 0; a < avg; a++) {
                    const uint32_t raw = reinterpret_cast<const uint16_t*>(imm + sel_off[(int64_t)t * avg + a])[gid];
                    x += dense_value(raw, nscale, nds, th);
                }
            } else {
                x = series_in[(int64_t)t * npix + gid];
            }
            push_exact<DPL, K, RAW, 0>(s, x, cnt);
        }
        const int64_t rowT = (int64_t)c * T;
#pragma unroll
        for (int l = 0; l < K; l++) {
            if (l < nlev_pass) {
                const LevelParam lp = levels[L0 + l];
                const int dlo = (RAW && l == 0) ? 1 : DPL + 1;
#pragma unroll
                for (int d = 1; d <= 2 * DPL; d++) {
                    const int rel = d - lp.lo;
                    if (d >= dlo && rel >= 0 && rel < lp.count)
                        G2[rowT + lp.first + rel] = (int64_t)s.acc[l][d - 1];
                }
            }
        }
    }
}

// Side statistics of the dense path straight from the raw frames: per
// (output frame, static bin) sums of the thresholded, flat-field weighted
// values (the per-frame partition sums of dense_filter.cpp / sparse_filter.cpp
// :134-191). A lane owns 8 consecutive detector pixels (one 16-byte load per
// raw frame when VEC) and keeps their bin, dark, threshold and weight in
// registers for a chunk of FC frames. Pixels of equal bin are summed inside the
// lane (the runs before the lane's last bin change go to LDS directly), the
// last runs across lanes by a segmented scan whose segments (equal bins of
// neighbouring lanes) are fixed for the whole kernel; segment tails add into
// the block's LDS table [FC][S], which goes to fs with one global atomic per
// nonzero entry. Values in 32-bit arithmetic: the caller guarantees
// 65535 * nscale < 2^31. INT (no flat field, F >= 512): the sums stay u32 up to
// the LDS atomic -- one value is below 2^32 / F (F * 65535 * nscale * avg <
// 2^32), so a wave segment of at most 512 pixels sums below 2^32.
constexpr int kSidePix = 8;
constexpr int kSideLdsDoubles = 4096;   // LDS table of one block (32 KB)
constexpr int kSideRing = 3;            // raw frames loaded ahead (VEC, avg 1)

template <bool VEC, bool INT>
__global__ void __launch_bounds__(256)
k_side_dense_raw(const uint8_t* __restrict__ imm, const int64_t* __restrict__ sel_off, int avg, int32_t F,
                 const int32_t* __restrict__ pix2c, uint32_t npix_det, const int64_t* __restrict__ dark_sum,
                 const int64_t* __restrict__ thr, int32_t nscale, const int32_t* __restrict__ sbin_of_c,
                 const double* __restrict__ weight, int32_t S, int32_t FC, double* __restrict__ fs)
{
    extern __shared__ double s_acc[];   // [FC][S]
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    const uint32_t j0 = g * kSidePix;
    const bool live = j0 < npix_det;    // VEC: npix_det % 8 == 0
    int32_t bin[kSidePix], nds[kSidePix], th[kSidePix];
    double w[kSidePix];
#pragma unroll
    for (int k = 0; k < kSidePix; k++) {
        const uint32_t j = j0 + (uint32_t)k;
        const int32_t c = j < npix_det ? pix2c[j] : -1;
        if (c >= 0) {
            bin[k] = sbin_of_c[c] - 1;
            nds[k] = dark_sum ? -(int32_t)dark_sum[c] : 0;
            const int64_t t = thr ? thr[c] : 0;
            th[k] = t < 0 ? 0 : (t > INT32_MAX ? INT32_MAX : (int32_t)t);
            w[k] = weight ? weight[c] : 1.0;
        } else {
            bin[k] = -1;
            nds[k] = 0;
            th[k] = INT32_MAX;   // no value passes
            w[k] = 0.0;
        }
    }
    uint32_t brk = 0;   // bit k: pixel k starts a new run inside the lane
#pragma unroll
    for (int k = 1; k < kSidePix; k++)
        if (bin[k] != bin[k - 1]) brk |= 1u << k;
    // segments of equal last-run bins across the lanes
    const int32_t lb = bin[kSidePix - 1];
    const int32_t lb_prev = (int32_t)prev_lane_u32((uint32_t)lb, 0xFFFFFFFEu);
    const int32_t lb_next = (int32_t)next_lane_u32((uint32_t)lb, 0xFFFFFFFEu);
    const uint32_t start = wave_incl_max_u32(lane == 0 || lb != lb_prev ? lane : 0u);
    const bool tail = lane == 63 || lb != lb_next;

    const int32_t nchunks = (F + FC - 1) / FC;
    for (int32_t ch = blockIdx.y; ch < nchunks; ch += gridDim.y) {
        const int32_t f0 = ch * FC;
        const int32_t nf = min(FC, F - f0);
        for (int i = threadIdx.x; i < FC * S; i += 256) s_acc[i] = 0.0;
        __syncthreads();
        auto frame = [&](const uint32_t (&x)[kSidePix], int32_t fl) {
            double* row = s_acc + (int64_t)fl * S;
            if constexpr (INT) {
                uint32_t run = 0u;
#pragma unroll
                for (int k = 0; k < kSidePix; k++) {
                    if (k > 0 && ((brk >> k) & 1u)) {
                        if (bin[k - 1] >= 0 && run) atomicAdd(&row[bin[k - 1]], (double)run);
                        run = 0u;
                    }
                    run += x[k];
                }
                run = wave_seg_scan_u32(run, start);
                if (tail && lb >= 0 && run) atomicAdd(&row[lb], (double)run);
                return;
            }
            double run = 0.0;
#pragma unroll
            for (int k = 0; k < kSidePix; k++) {
                if (k > 0 && ((brk >> k) & 1u)) {
                    if (bin[k - 1] >= 0 && run != 0.0) atomicAdd(&row[bin[k - 1]], run);
                    run = 0.0;
                }
                run += (double)x[k] * w[k];
            }
            run = wave_seg_scan_f64(run, start);
            if (tail && lb >= 0 && run != 0.0) atomicAdd(&row[lb], run);
        };
        auto decode = [&](const u32x4& r, uint32_t (&x)[kSidePix]) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                x[2 * q] = dense_value(r[q] & 0xFFFFu, nscale, nds[2 * q], th[2 * q]);
                x[2 * q + 1] = dense_value(r[q] >> 16, nscale, nds[2 * q + 1], th[2 * q + 1]);
            }
        };
        if constexpr (VEC) {
            if (avg == 1) {
                auto issue = [&](u32x4& r, int32_t fl) {
                    const int32_t f = f0 + min(fl, nf - 1);
                    // each frame is streamed once: nontemporal (about 1 % faster)
                    r = live ? __builtin_nontemporal_load(
                                   reinterpret_cast<const u32x4*>(imm + sel_off[f] + 2 * (int64_t)j0))
                             : u32x4{0, 0, 0, 0};
                };
                u32x4 ring[kSideRing];
#pragma unroll
                for (int d = 0; d < kSideRing; d++) issue(ring[d], d);
                for (int32_t fb = 0; fb < nf; fb += kSideRing) {
#pragma unroll
                    for (int d = 0; d < kSideRing; d++) {
                        if (fb + d < nf) {
                            uint32_t x[kSidePix];
                            decode(ring[d], x);
                            issue(ring[d], fb + d + kSideRing);
                            frame(x, fb + d);
                        }
                    }
                }
            } else {
                for (int32_t fl = 0; fl < nf; fl++) {
                    uint32_t x[kSidePix] = {};
                    for (int a = 0; a < avg; a++) {
                        const u32x4 r = live ? *reinterpret_cast<const u32x4*>(
                                                   imm + sel_off[(int64_t)(f0 + fl) * avg + a] + 2 * (int64_t)j0)
                                             : u32x4{0, 0, 0, 0};
                        uint32_t y[kSidePix];
                        decode(r, y);
#pragma unroll
                        for (int k = 0; k < kSidePix; k++) x[k] += y[k];
                    }
                    frame(x, fl);
                }
            }
        } else {
            for (int32_t fl = 0; fl < nf; fl++) {
                uint32_t x[kSidePix] = {};
                for (int a = 0; a < avg; a++) {
                    const uint16_t* fr =
                        reinterpret_cast<const uint16_t*>(imm + sel_off[(int64_t)(f0 + fl) * avg + a]);
#pragma unroll
                    for (int k = 0; k < kSidePix; k++)
                        if (j0 + (uint32_t)k < npix_det) x[k] += dense_value(fr[j0 + k], nscale, nds[k], th[k]);
                }
                frame(x, fl);
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nf * S; i += 256)
            if (s_acc[i] != 0.0) atomicAdd(&fs[(int64_t)f0 * S + i], s_acc[i]);
        __syncthreads();
    }
}

// ---- dark image ------------------------------------------------------------------

constexpr int kDarkPer = 64;
struct DarkFrames {
    int64_t off[kDarkPer];
    int32_t n, first;        // frames of this launch, index of the first
};

// Dark image of the leading frames (DarkImage::Compute,
// src/xpcs/data_structure/dark_image.cpp:81-106: Welford in double, in frame
// order, no fused operations), the exact integer sums, and after the last
// frame the n-scaled threshold floor(n (lld + sigma std)) per compact pixel.
// Dark values are uint16 like every count (the reference reads int16,
// src/xpcs/io/imm.cpp:87; equal below 32768).  On the host, with the frames
// copied back and the results copied up, this took 1.5 of the 5.4 ms of a
// 512 x 512 x 20,000-frame pass with two darks.
__global__ void __launch_bounds__(256)
k_dark_image(const uint8_t* __restrict__ base, const DarkFrames d, int32_t darks, uint32_t npix, float lld, float sigma,
             const int32_t* __restrict__ pix2c, double* __restrict__ avg, double* __restrict__ dev,
             int64_t* __restrict__ isum, int64_t* __restrict__ dark_sum, int64_t* __restrict__ thr)
{
#pragma clang fp contract(off)
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= npix) return;
    double m = 0.0, q = 0.0;
    int64_t s = 0;
    if (d.first > 0) {
        m = avg[j];
        q = dev[j];
        s = isum[j];
    }
    for (int i = 0; i < d.n; i++) {
        const uint16_t raw = reinterpret_cast<const uint16_t*>(base + d.off[i])[j];
        const double x = (double)raw;
        const double prev = m;
        m = m + (x - m) / (double)(d.first + i + 1);
        q = q + (x - prev) * (x - m);
        s += raw;
    }
    const bool last = d.first + d.n == darks;
    if (last) q = sqrt(q / (double)darks);
    avg[j] = m;
    dev[j] = q;
    isum[j] = s;
    const int32_t c = pix2c[j];
    if (last && c >= 0) {
        const float t = (float)((double)lld + (double)sigma * q);
        const double f = floor((double)darks * (double)t);
        dark_sum[c] = s;
        // out of range or NaN: as the host conversion gives
        thr[c] = f >= -9.2e18 && f <= 9.2e18 ? (int64_t)f : INT64_MIN;
    }
}

void launch_dark_image(xpcs_mt_plan* p, const uint8_t* base, const std::vector<int64_t>& off, hipStream_t s)
{
    const HostTables& h = p->h;
    const uint32_t npd = (uint32_t)(h.W * h.H);
    for (size_t k = 0; k < off.size(); k += kDarkPer) {
        DarkFrames d{};
        d.first = (int32_t)k;
        d.n = (int32_t)std::min((size_t)kDarkPer, off.size() - k);
        for (int i = 0; i < d.n; i++) d.off[i] = off[k + (size_t)i];
        k_dark_image<<<(npd + 255) / 256, 256, 0, s>>>(base, d, (int32_t)off.size(), npd, h.lld, h.sigma, p->d_pix2c,
                                                       p->d_dark_avg, p->d_dark_std, p->d_dark_isum, p->d_dark_sum,
                                                       p->d_thr);
    }
}

// ---- host side --------------------------------------------------------------------

bool dense_stream_supported(const HostTables& h)
{
    return h.dpl == 4 || h.dpl == 8;
}

bool dense_levels_allowed(int dpl, int k)
{
    return dpl == 4 ? (k >= 3 && k <= 5) : (dpl == 8 && (k == 2 || k == 3));
}

int dense_levels(const xpcs_mt_plan* p)
{
    const int k = p->tune.dense_levels;
    if (k > 0 && dense_levels_allowed(p->h.dpl, k)) return k;
    return p->h.dpl == 4 ? dense_levels_per_pass<4>() : dense_levels_per_pass<8>();
}

// The dot-product raw pass: counts, one raw frame per output frame, evenly
// spaced frames of any 2-byte alignment, value scales of 16 bits.
static bool dense_dot_ok(const xpcs_mt_plan* p)
{
    return !p->fsnorm && p->even_off0 >= 0 && p->h.avg == 1 && (int64_t)p->h.W * p->h.H >= 8 && p->nscale <= 1024 && p->d_wave_flags;
}

// 32-bit words of the two series buffers: the first pass writes the first one,
// the next the second, and so on; level values as u32, or frame-weighted as
// FP64 (2 words).  The first pass also keeps its boundary sums in the second.
size_t dense_series_elems(const xpcs_mt_plan* p, int which)
{
    const HostTables& h = p->h;
    const size_t npd = (size_t)h.W * (size_t)h.H;
    const size_t L = (size_t)dense_levels(p) * (size_t)(which + 1);   // first level that the buffer holds
    const size_t words = p->fsnorm ? 2 : 1;
    const size_t series = h.levels.size() > L ? words * (size_t)h.levels[L].lf * npd : 1;
    return std::max(series, which == 1 && dense_dot_ok(p) ? (size_t)p->nrank * npd : (size_t)1);
}

template <int DPL, int K>
static void launch_dense_dot(xpcs_mt_plan* p, hipStream_t s, int nlev_pass, uint32_t* out, uint32_t lf_out,
                             uint32_t* redo_count)
{
    const HostTables& h = p->h;
    DotArgs a{};
    a.src = p->d_imm + p->even_off0;
    a.step = p->even_step;
    a.pix2c = p->d_pix2c;
    a.npix = (uint32_t)(h.W * h.H);
    a.n_in = (uint32_t)h.F;
    a.chunk = h.darks == 1 ? kDotChunk / 2 : kDotChunk;
    a.dark_sum = p->d_dark_sum;
    a.thr = p->d_thr;
    a.nscale = (int32_t)p->nscale;
    a.levels = p->d_levels;
    a.nlev_pass = nlev_pass;
    a.cap = p->d_cap;
    a.ncap = p->nrank;
    a.T = h.T;
    a.tau_bnd = p->d_tau_bnd;
    a.cap_sums = p->d_series_b;   // free during the first pass
    a.G2 = p->d_G2;
    a.IP = p->d_IP;
    a.IF = p->d_IF;
    a.pix_total = p->d_pix_total;
    a.series_out = out;
    a.lf_out = (out && nlev_pass == K) ? lf_out : 0u;
    a.redo_count = redo_count;
    a.redo_list = p->d_long_list;
    a.wave_flags = p->d_wave_flags;
    if (a.n_in >= kDotLookFrames) {
        uint32_t* const bright = p->d_counters + 7;
        k_dense_look<<<(a.npix + 255) / 256, 256, 0, s>>>(a.src, a.step, a.pix2c, a.npix, a.n_in, a.dark_sum, a.thr,
                                                          a.nscale, a.chunk / 3 * 2, a.wave_flags, bright);
        a.bright = bright;
        // this kernel takes 0.7 (dpl 4) or 0.36 (dpl 8) of the FP64 kernel's
        // time, so with that share of the waves left to it one pass of both is
        // slower; a detector of at most two waves per SIMD takes either
        // kernel's time as soon as one wave runs it
        const uint32_t waves = (a.npix + 63) / 64;
        a.most = waves <= 2048 ? 0 : DPL == 4 ? waves / 4 : waves / 8 * 5;
    }
    a.w32 = p->ipif32;
    auto go = [&](auto waves) {
        constexpr int W = decltype(waves)::value;
        const unsigned grid = ((a.npix + 64 * W - 1) / (64 * W) + 7) / 8 * 8;
        if (h.darks > 0) k_mt_dense_dot<DPL, K, true, W><<<grid, 64 * W, 0, s>>>(a);
        else k_mt_dense_dot<DPL, K, false, W><<<grid, 64 * W, 0, s>>>(a);
    };
    // detectors of at most two waves per CU: single waves spread over the chip
    if (a.npix <= 2 * 256 * 64) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, DPL == 4 ? 8 : 4>{});
}

template <int DPL, int K, bool FP>
static void run_passes(xpcs_mt_plan* p, hipStream_t s)
{
    using ST = std::conditional_t<FP, double, uint32_t>;
    const HostTables& h = p->h;
    const int nlev = (int)h.levels.size();
    const uint32_t npd = (uint32_t)(h.W * h.H);
    const unsigned grid = (npd + 255) / 256;
    uint32_t* redo_count = p->d_counters + 3;
    ST* const sa = reinterpret_cast<ST*>(p->d_series_a);
    ST* const sb = reinterpret_cast<ST*>(p->d_series_b);
    const double* fw = FP ? p->d_fw : nullptr;
    int L0 = 0;
    uint32_t n_in = (uint32_t)h.F;
    int pass = 0;
    while (L0 < nlev) {
        const int k = std::min(K, nlev - L0);
        const bool more = L0 + k < nlev;
        const uint32_t lf_out = more ? (uint32_t)h.levels[L0 + k].lf : 0u;
        ST* out = more ? (pass % 2 == 0 ? sa : sb) : nullptr;
        const ST* in = pass == 0 ? nullptr : (pass % 2 == 1 ? sa : sb);
        if (pass == 0) {
            timer_begin(p, s, FP ? "k_mt_dense_raw_f64" : "k_mt_dense_raw");
            // counts of evenly spaced frames: the dot-product kernel, then the
            // FP64 one for the pixels it left
            const uint32_t* only = nullptr;
            if constexpr (!FP && (8 >> (K - 1)) >= 1) {
                if (dense_dot_ok(p)) {
                    launch_dense_dot<DPL, K>(p, s, k, out, lf_out, redo_count);
                    only = p->d_wave_flags;
                }
            }
            if (p->tile_off0 >= 0)
                k_mt_dense_f64<DPL, K, kRawTiles, FP><<<grid, 256, 0, s>>>(
                    p->d_imm, p->d_sel_off, p->tile_off0, p->tile_step, h.avg, p->d_pix2c, npd, p->d_dark_sum,
                    p->d_thr, (int32_t)p->nscale, nullptr, n_in, p->d_levels, L0, k, p->d_bnd, p->nbnd, h.T,
                    p->d_G2, p->d_IP, p->d_IF, p->d_pix_total, out, lf_out, redo_count, p->d_long_list, fw, !FP && p->ipif32, only);
            else
                k_mt_dense_f64<DPL, K, kRawLanes, FP><<<grid, 256, 0, s>>>(
                    p->d_imm, p->d_sel_off, 0, 0, h.avg, p->d_pix2c, npd, p->d_dark_sum, p->d_thr,
                    (int32_t)p->nscale, nullptr, n_in, p->d_levels, L0, k, p->d_bnd, p->nbnd, h.T, p->d_G2,
                    p->d_IP, p->d_IF, p->d_pix_total, out, lf_out, redo_count, p->d_long_list, fw, !FP && p->ipif32, only);
            timer_end(p, s);
            if constexpr (!FP) {
                timer_begin(p, s, "k_mt_dense_exact");
                k_mt_dense_exact<DPL, K, true><<<256, 256, 0, s>>>(
                    p->d_imm, p->d_sel_off, h.avg, p->d_pix2c, npd, p->d_dark_sum, p->d_thr, (int32_t)p->nscale,
                    nullptr, n_in, p->d_levels, L0, k, h.T, p->d_G2, redo_count, p->d_long_list);
                timer_end(p, s);
            }
        } else {
            timer_begin(p, s, FP ? "k_mt_dense_series_f64" : "k_mt_dense_series");
            k_mt_dense_f64<DPL, K, kSeries, FP><<<grid, 256, 0, s>>>(
                nullptr, nullptr, 0, 0, 1, p->d_pix2c, npd, nullptr, nullptr, 1, in, n_in, p->d_levels, L0, k,
                nullptr, 0, h.T, p->d_G2, p->d_IP, p->d_IF, p->d_pix_total, out, lf_out, nullptr, nullptr, fw,
                !FP && p->ipif32, nullptr);
            timer_end(p, s);
            if constexpr (!FP) {
                timer_begin(p, s, "k_mt_dense_exact");
                k_mt_dense_exact<DPL, K, false><<<256, 256, 0, s>>>(
                    nullptr, nullptr, 1, p->d_pix2c, npd, nullptr, nullptr, 1, in, n_in, p->d_levels, L0, k, h.T,
                    p->d_G2, redo_count, p->d_long_list);
                timer_end(p, s);
            }
        }
        n_in = lf_out;
        L0 += k;
        pass++;
    }
}

template <bool FP>
static void launch_dense_passes(xpcs_mt_plan* p, hipStream_t s)
{
    const int k = dense_levels(p);
    if (p->h.dpl == 4) {
        if (k == 3) run_passes<4, 3, FP>(p, s);
        else if (k == 5) run_passes<4, 5, FP>(p, s);
        else run_passes<4, 4, FP>(p, s);
    } else {
        if (k == 2) run_passes<8, 2, FP>(p, s);
        else run_passes<8, 3, FP>(p, s);
    }
}

void launch_mt_dense(xpcs_mt_plan* p, hipStream_t s, bool fsnorm)
{
    if (fsnorm) launch_dense_passes<true>(p, s);
    else launch_dense_passes<false>(p, s);
}

void launch_side_dense_raw(xpcs_mt_plan* p, hipStream_t s)
{
    const HostTables& h = p->h;
    const uint32_t npd = (uint32_t)(h.W * h.H);
    const uint32_t groups = (npd + kSidePix - 1) / kSidePix;
    const int32_t fc = std::max(1, std::min(64, kSideLdsDoubles / std::max(h.ns, 1)));
    const int32_t nchunks = (h.F + fc - 1) / fc;
    const dim3 grid((groups + 255) / 256, (unsigned)std::min(nchunks, 65535));
    const size_t lds = (size_t)fc * (size_t)h.ns * sizeof(double);
    timer_begin(p, s, "k_side");
    auto go = [&](auto vec, auto integer) {
        k_side_dense_raw<decltype(vec)::value, decltype(integer)::value><<<grid, 256, lds, s>>>(
            p->d_imm, p->d_sel_off, h.avg, h.F, p->d_pix2c, npd, p->d_dark_sum, p->d_thr, (int32_t)p->nscale,
            p->d_sbin_of_c, p->d_weight, h.ns, fc, p->d_fs);
    };
    const bool integer = !p->d_weight && h.F >= 512;
    if (p->side_vec) {
        if (integer) go(std::true_type{}, std::true_type{});
        else go(std::true_type{}, std::false_type{});
    } else {
        if (integer) go(std::false_type{}, std::true_type{});
        else go(std::false_type{}, std::false_type{});
    }
    timer_end(p, s);
}

}  // namespace xpcs
