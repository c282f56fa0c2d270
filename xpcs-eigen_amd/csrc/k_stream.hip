// Online multi-tau for streams of sparse frames (no reference counterpart: the
// reference correlates a finished file, Corr::multiTau2, src/xpcs/corr.cpp:315-431).
//
// Per stream and masked pixel the state lives in HBM, level-major with the
// pixel index fastest (every access coalesced):
//   win [L][D2][P] u32  the last D2 = 2*dpl values of level L: value k in slot
//                       k mod D2, zero before the first D2 values
//   head[L][D2][P] u32  the first D2 values of level L
//   acc [L][D2][P] u64  lag sums  sum_t x_L[t-d] x_L[t]  for the level's lags,
//                       d = 1..D2 at level 0, d = dpl+1..D2 above it
//   pend[L][P]     u32  the last level-L value while its pair is incomplete
//   total[P]       u64  sum of all level-0 values
// After n frames, level L holds lf_L = floor(n / 2^L) values, and for a lag
// tau' of level L
//   G2 = acc[L][tau'],  IP = T_L - sum of the last tau' values,
//   IF = T_L - sum_{k<tau'} head[L][k],  T_L = sum_k x_L[k]
//      = total - sum_{l<L, lf_l odd} pend[l],
// which are exactly the batch sums for F = n: a lag product is added when its
// later value arrives, and the schedule for n frames is a prefix of the
// schedule for the stream's maximum length.
#include <algorithm>

#include "device_util.h"
#include "internal.h"

namespace xpcs {

// Frames of a push: events into a dense [nb][P] value tile (summed per pixel).
// A block per frame; its threads hold a frame of few photons in one round, since
// a round is three dependent accesses to memory (655 photons: 4.2 us, with 256
// threads 4.8).
constexpr int kScatterThreads = 1024;

__global__ void __launch_bounds__(kScatterThreads)
k_stream_scatter(const uint8_t* __restrict__ imm, const StreamFrames fr, int32_t nb,
                 const int32_t* __restrict__ pix2c, uint32_t npix_det, int32_t P, uint32_t* __restrict__ tile,
                 uint32_t* __restrict__ counters)
{
    for (int f = blockIdx.x; f < nb; f += gridDim.x) {
        const uint8_t* base = imm + fr.off[f];
        const uint32_t n = fr.dlen[f];
        for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) {
            const uint32_t idx = load_u32_a2(base + 4 * (size_t)j);
            const uint32_t v = reinterpret_cast<const uint16_t*>(base + 4 * (size_t)n)[j];
            if (idx >= npix_det) {
                atomicOr(&counters[1], 1u);
                continue;
            }
            const int32_t c = pix2c[idx];
            if (c >= 0 && v) atomicAdd(&tile[(int64_t)f * P + c], v);
        }
    }
}

// One chunk of nb frames through the levels that gain a value: a block holds 64
// pixels, a wave per level, a lane per pixel.  A stream's state is larger than
// the L2 and a launch is short, so what bounds it is the state that it moves
// and the length of a thread's chain of memory accesses:
//  - a level's new values are sums of the chunk's frames (the first one begins
//    with what is pending below it), so that no level waits for the one before;
//  - the windows are rings: a chunk stores the values that it adds, not the
//    whole window;
//  - the chunk's part of a lag sum starts at zero and is added to the state
//    only where it is not zero, by an atomic that returns nothing.  One thread
//    owns each sum; the atomic saves the read and its wait.  With few photons
//    hardly any sum changes in a chunk.
// A push of 16 frames of 256 x 256 at 0.01 photons: 8.8 us, against 19.8 with a
// thread per pixel walking the levels one after the other (36 MB of windows and
// sums moved, 15.3 still without the moves).
constexpr int kStreamLanes = 64;    // pixels of a block
constexpr int kStreamWaves = 16;    // levels of a block at a time

// The D2 values before value k, newest first (zero before value 0).
template <int D2>
__device__ inline void stream_window(const uint32_t* __restrict__ win, int L, int64_t P, int64_t c, uint32_t k,
                                     uint32_t (&w)[D2])
{
#pragma unroll
    for (int j = 0; j < D2; j++)
        w[j] = win[((int64_t)L * D2 + ((k - 1u - (uint32_t)j) & (uint32_t)(D2 - 1))) * P + c];
}

// Level L of a chunk: its window w holds the values before the chunk, run the
// frames before the chunk that belong to the first new value; lags D0+1..D2.
template <int D2, int D0>
__device__ inline void stream_level(const uint32_t* __restrict__ vals, int nb, uint32_t n0, int L, int64_t P,
                                    int64_t c, uint32_t run, uint32_t (&w)[D2], uint32_t* __restrict__ win,
                                    uint32_t* __restrict__ head, uint64_t* __restrict__ acc,
                                    uint32_t* __restrict__ pend)
{
    const int64_t lb = (int64_t)L * D2 * P + c;
    const uint32_t last = (1u << L) - 1u;   // phase of a value's last frame
    uint64_t a[D2];
#pragma unroll
    for (int d = D0; d < D2; d++) a[d] = 0;
    uint32_t k = n0 >> L;
    uint32_t x = vals[0];
    for (int i = 0; i < nb; i++) {
        run += x;
        x = i + 1 < nb ? vals[(i + 1) * kStreamLanes] : 0u;
        if (((n0 + (uint32_t)i) & last) != last) continue;
        if (run) {
#pragma unroll
            for (int d = D0; d < D2; d++) a[d] += (uint64_t)run * (uint64_t)w[d];
        }
#pragma unroll
        for (int j = D2 - 1; j > 0; j--) w[j] = w[j - 1];
        w[0] = run;
        if (k < (uint32_t)D2) head[lb + (int64_t)k * P] = run;
        k++;
        run = 0;
    }
    const uint32_t m = k - (n0 >> L);
#pragma unroll
    for (int j = 0; j < D2; j++)
        if ((uint32_t)j < m) win[lb + (int64_t)((k - 1u - (uint32_t)j) & (uint32_t)(D2 - 1)) * P] = w[j];
    if (k & 1u) pend[(int64_t)L * P + c] = w[0];
#pragma unroll
    for (int d = D0; d < D2; d++)
        if (a[d]) atomicAdd(reinterpret_cast<unsigned long long*>(&acc[lb + (int64_t)d * P]), a[d]);
}

// nlev: the levels that gain a value (at most 2 * kStreamWaves).
template <int D2>
__global__ void __launch_bounds__(kStreamLanes* kStreamWaves)
k_stream_update(uint32_t* __restrict__ tile, int32_t nb, int32_t P, int32_t n0, int32_t nlev,
                uint32_t* __restrict__ win, uint32_t* __restrict__ head, uint64_t* __restrict__ acc,
                uint32_t* __restrict__ pend, uint64_t* __restrict__ total)
{
    extern __shared__ uint32_t s_vals[];   // [nb][kStreamLanes]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6;
    const int64_t c = (int64_t)blockIdx.x * kStreamLanes + lane;
    const bool active = c < P;
    uint32_t w[D2] = {};
    uint32_t run0 = 0, run1 = 0;   // this wave's levels: wave and wave + nw
    if (active) {
        if (wave < nlev) stream_window<D2>(win, wave, P, c, (uint32_t)n0 >> wave, w);
        for (int l = 0; l < wave; l++)
            if ((n0 >> l) & 1) run0 += pend[(int64_t)l * P + c];
        if (wave + nw < nlev) {
            run1 = run0;
            for (int l = wave; l < wave + nw; l++)
                if ((n0 >> l) & 1) run1 += pend[(int64_t)l * P + c];
        }
    }
    for (int i0 = wave; i0 < nb; i0 += 4 * nw) {
        uint32_t v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = i0 + j * nw;
            v[j] = active && i < nb ? tile[(int64_t)i * P + c] : 0u;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = i0 + j * nw;
            if (i >= nb) break;
            // read entries go back to zero, ready for the next push's scatter
            if (v[j]) tile[(int64_t)i * P + c] = 0u;
            s_vals[i * kStreamLanes + lane] = v[j];
        }
    }
    // every pending value has been read: the levels may store theirs
    __syncthreads();
    if (!active) return;
    const uint32_t* const vals = s_vals + lane;
    if (wave == nw - 1) {
        uint64_t add = 0;
        for (int i = 0; i < nb; i++) add += vals[i * kStreamLanes];
        if (add) total[c] += add;
    }
    if (wave < nlev) {
        if (wave == 0)
            stream_level<D2, 0>(vals, nb, (uint32_t)n0, 0, P, c, 0u, w, win, head, acc, pend);
        else
            stream_level<D2, D2 / 2>(vals, nb, (uint32_t)n0, wave, P, c, run0, w, win, head, acc, pend);
    }
    if (wave + nw < nlev) {
        stream_window<D2>(win, wave + nw, P, c, (uint32_t)n0 >> (wave + nw), w);
        stream_level<D2, D2 / 2>(vals, nb, (uint32_t)n0, wave + nw, P, c, run1, w, win, head, acc, pend);
    }
}

// Sums for the schedule of n frames, taus [t0, t1) of it, into rows of stride
// S ([P][S]), and those taus' table entries (lf, N for n frames) that the
// normalisation reads.  Only the levels holding those taus are read: a block
// holds 64 pixels, a wave per level l0 + wave, a lane per pixel, so that no
// level waits for the one before.  A pixel's taus of one level are 8 B each in
// rows that lie S words apart; they are put together in LDS and stored as rows.
// 256 x 256, 32 of 36 taus: 14.7 us, against 56 with a thread per pixel storing
// its taus one by one, and 37 with a grid row per level that does.
template <int D2>
__global__ void __launch_bounds__(kStreamLanes* kStreamWaves)
k_stream_snapshot(const uint32_t* __restrict__ win, const uint32_t* __restrict__ head,
                  const uint64_t* __restrict__ acc, const uint32_t* __restrict__ pend,
                  const uint64_t* __restrict__ total, int32_t P, int32_t n, int32_t l0,
                  const LevelParam* __restrict__ levels, const TauParam* __restrict__ taus_max, int32_t t0,
                  int32_t t1, int32_t S, TauParam* __restrict__ taus, int64_t* __restrict__ G2,
                  int64_t* __restrict__ IP, int64_t* __restrict__ IF)
{
    extern __shared__ int64_t s_rows[];   // [kStreamLanes][(t1 - t0) | 1]
    if (blockIdx.x == 0) {
        for (int i = t0 + (int)threadIdx.x; i < t1; i += blockDim.x) {
            TauParam t = taus_max[i];
            t.lf = n >> t.level;
            t.N = t.lf - t.tp;
            taus[i] = t;
        }
    }
    const int lane = threadIdx.x & 63;
    const int L = l0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c0 = (int64_t)blockIdx.x * kStreamLanes;
    const int64_t c = c0 + lane;
    const int np = (int)min((int64_t)kStreamLanes, P - c0);
    const LevelParam lp = levels[L];
    const int nt = t1 - t0, pitch = nt | 1;
    uint32_t w[D2] = {}, h[D2] = {};
    uint64_t g[D2] = {};
    uint64_t TL = 0;
    if (lane < np) {
        const int64_t lb = (int64_t)L * D2 * P + c;
        TL = total[c];
        stream_window<D2>(win, L, P, c, (uint32_t)n >> L, w);
#pragma unroll
        for (int j = 0; j < D2; j++) {
            h[j] = head[lb + (int64_t)j * P];
            g[j] = j + 1 >= lp.lo ? acc[lb + (int64_t)j * P] : 0ull;   // lags below belong to the level before
        }
        for (int l = 0; l < L; l++)
            if ((n >> l) & 1) TL -= pend[(int64_t)l * P + c];
    }
    int64_t* const row = s_rows + lane * pitch + lp.first - lp.lo - t0;   // row[d]: lag d of this level
    const int da = max(lp.lo, lp.lo + t0 - lp.first);                     // this level's lags in range: [da, db)
    const int db = min(lp.lo + lp.count, lp.lo + t1 - lp.first);
    // the block's rows, in the order of memory: element threadIdx.x first,
    // then blockDim.x further each time
    const int r_step = blockDim.x / nt, k_step = blockDim.x % nt;
    const int r_first = threadIdx.x / nt, k_first = threadIdx.x % nt;
#pragma unroll
    for (int which = 0; which < 3; which++) {
        if (which == 0) {
#pragma unroll
            for (int d = 1; d <= D2; d++)
                if (d >= da && d < db) row[d] = (int64_t)g[d - 1];
        } else {
            uint64_t s = TL;   // less the newest / oldest d values
#pragma unroll
            for (int d = 1; d <= D2; d++) {
                s -= which == 1 ? w[d - 1] : h[d - 1];
                if (d >= da && d < db) row[d] = (int64_t)s;
            }
        }
        __syncthreads();
        int64_t* const out = which == 0 ? G2 : which == 1 ? IP : IF;
        for (int r = r_first, k = k_first; r < np;) {
            out[(c0 + r) * S + t0 + k] = s_rows[r * pitch + k];
            r += r_step;
            k += k_step;
            if (k >= nt) {
                k -= nt;
                r++;
            }
        }
        if (which < 2) __syncthreads();
    }
}

void launch_stream_update(const StreamLaunch& a, hipStream_t s)
{
    // the tile is zero here: cleared when the stream opens, and every entry a
    // scatter sets is cleared again by the update that reads it
    k_stream_scatter<<<a.nb, kScatterThreads, 0, s>>>(a.imm, a.fr, a.nb, a.pix2c, a.npix_det, a.P, a.tile, a.counters);
    // level L gains a value when n >> L changes
    const uint32_t x = (uint32_t)a.n0 ^ (uint32_t)(a.n0 + a.nb);
    const int nlev = std::min<int>(a.nlev, 32 - __builtin_clz(x));
    const unsigned gp = (unsigned)((a.P + kStreamLanes - 1) / kStreamLanes);
    const unsigned threads = (unsigned)(std::max(1, std::min(nlev, kStreamWaves)) * 64);
    const size_t lds = (size_t)a.nb * kStreamLanes * sizeof(uint32_t);
    if (a.d2 == 8)
        k_stream_update<8><<<gp, threads, lds, s>>>(a.tile, a.nb, a.P, a.n0, nlev, a.win, a.head, a.acc, a.pend,
                                                    a.total);
    else
        k_stream_update<16><<<gp, threads, lds, s>>>(a.tile, a.nb, a.P, a.n0, nlev, a.win, a.head, a.acc, a.pend,
                                                     a.total);
}

// taus_host: the levels of the taus (ascending), for the split into launches
// whose levels fit a block and whose rows fit 64 KiB of LDS.
void launch_stream_snapshot(const StreamLaunch& a, int32_t n, const LevelParam* levels, const TauParam* taus_host,
                            const TauParam* taus_max, int32_t t0, int32_t t1, int32_t S, TauParam* taus,
                            int64_t* G2, int64_t* IP, int64_t* IF, hipStream_t s)
{
    const unsigned gp = (unsigned)((a.P + kStreamLanes - 1) / kStreamLanes);
    constexpr int kMaxRow = 65536 / (8 * kStreamLanes) - 1;   // an odd pitch of at most this fits
    for (int32_t b = t0, e; b < t1; b = e) {
        const int32_t l0 = taus_host[b].level;
        for (e = b + 1; e < t1 && e - b < kMaxRow && taus_host[e].level < l0 + kStreamWaves;) e++;
        const unsigned threads = (unsigned)(taus_host[e - 1].level - l0 + 1) * 64;
        const size_t lds = (size_t)kStreamLanes * (size_t)((e - b) | 1) * sizeof(int64_t);
        if (a.d2 == 8)
            k_stream_snapshot<8><<<gp, threads, lds, s>>>(a.win, a.head, a.acc, a.pend, a.total, a.P, n, l0, levels,
                                                          taus_max, b, e, S, taus, G2, IP, IF);
        else
            k_stream_snapshot<16><<<gp, threads, lds, s>>>(a.win, a.head, a.acc, a.pend, a.total, a.P, n, l0, levels,
                                                           taus_max, b, e, S, taus, G2, IP, IF);
    }
}

}  // namespace xpcs
