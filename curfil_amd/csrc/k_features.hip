// Per-(tree, level) random feature generation on the device, with the exact
// semantics of the reference CPU generator:
//   ImageFeatureEvaluation::generateRandomFeatures  random_tree_image.cpp:577-646
//   ImageFeatureEvaluation::sampleFeature           random_tree_image.cpp:648-700
//   sortFeatures (stable sort by getSortKey)        random_tree_image.cpp:504-566,
//                                                   random_tree_image.h:444-452
//
// RandomSource(seed) hands seed to the sample-index sampler and seeds
// seed+1+4k .. seed+4+4k to candidate k's four samplers (type, offset,
// region, channel).  Candidates are therefore independent and are drawn in
// parallel, and so is the stream of sample-index draws (k_fg_draws,
// k_fg_records).  Thresholds consume that one stream in order, and
// how many draws a candidate consumes depends on which responses are NaN, so a
// candidate's first draw is known only after its predecessor's last.  That
// chain is taken in rounds of two launches:
//   k_fg_round    a workgroup per candidate evaluates it on a band of draws
//                 around its expected first draw and, from the finite bits,
//                 tabulates for every start in the band where in the next
//                 candidate's band that one would start, and whether the
//                 candidate would be accepted;
//   k_fg_advance  a workgroup per tree follows the chain through the tables
//                 (one LDS read per eight candidates, whose tables it has
//                 composed) and writes the accepted candidates' thresholds.
// The bands only decide how far a round gets, never which draws a candidate
// uses.  Per level of 5 trees with F = 4000, T = 32 on 50 frames of 640x480 the
// walk takes 1.1 ms (about 40 rounds of 112 candidates: 15 us + 11 us each);
// one workgroup per tree that evaluated 16 candidates a round on its own CU
// took 15.2 ms, bound by that CU's gathers.
#include <algorithm>
#include <cstring>

#include "cf_internal.h"
#include "cf_rng.h"

namespace cf {

constexpr int kPrefixDraws = 24;   // engine outputs available to one feature sampler

// Candidates [first, first + count) of every job.  A lane per (candidate, sampler) runs the chain of 420
// seeding steps that a sampler's first outputs need (the bound: with the four samplers one after another in
// one lane, and the outputs indexed in scratch memory, 71 us a launch), then a lane per candidate draws from
// the outputs in LDS.
//
// g++ on x86-64 evaluates the two getNext() calls of `Offset(rgen.getNext(),
// rgen.getNext())` right to left, so the second coordinate is drawn first
// (pinned by the reference's golden feature hash).
constexpr int kCandBlock = 64;   // candidates of a workgroup (its first 256 lanes)
__device__ __forceinline__ void drawCandidates(const FeatGenJob* __restrict__ jobs, int job, int block, int numCand,
        int first, int count, int boxRadius, int regionSize, int useDepth, FeatRec* __restrict__ cand,
        int* __restrict__ err) {
    constexpr int kStride = kPrefixDraws + 1;
    __shared__ uint32_t outputs[4 * kCandBlock * kStride];
    if (threadIdx.x >= 4 * kCandBlock) return;
    {
        const int k = first + block * kCandBlock + static_cast<int>(threadIdx.x >> 2);
        uint32_t out[kPrefixDraws];
        mtPrefix<kPrefixDraws>(static_cast<uint32_t>(jobs[job].seed + 1 + 4 * k + static_cast<int>(threadIdx.x & 3)), out);
#pragma unroll
        for (int i = 0; i < kPrefixDraws; i++) outputs[threadIdx.x * kStride + i] = out[i];
    }
    __syncthreads();
    const int k = first + block * kCandBlock + threadIdx.x;
    if (threadIdx.x >= kCandBlock || k >= first + count) return;
    const uint32_t* mine = outputs + threadIdx.x * 4 * kStride;   // samplers: type, offset, region, channel
    FeatRec f;
#pragma unroll
    for (int i = 0; i < 16; i++) f.p[i] = 0;
    bool ok = true;
    int a, b;
    {
        DevPrefixSampler<kPrefixDraws> xy;
        xy.init(mine + kStride, -boxRadius, boxRadius);
        int o1x = 0, o1y = 0, o2x = 0, o2y = 0;
        ok &= xy.next(b);
        ok &= xy.next(a);
        o1x = a;
        o1y = b;
        do {
            ok &= xy.next(b);
            ok &= xy.next(a);
            o2x = a;
            o2y = b;
        } while (ok && o1x == o2x && o1y == o2y);
        f.p[P_O1X] = static_cast<int8_t>(o1x);
        f.p[P_O1Y] = static_cast<int8_t>(o1y);
        f.p[P_O2X] = static_cast<int8_t>(o2x);
        f.p[P_O2Y] = static_cast<int8_t>(o2y);
    }
    {
        DevPrefixSampler<kPrefixDraws> rg;
        rg.init(mine + 2 * kStride, 1, regionSize);
        ok &= rg.next(b);
        ok &= rg.next(a);
        f.p[P_R1X] = static_cast<int8_t>(a);
        f.p[P_R1Y] = static_cast<int8_t>(b);
        ok &= rg.next(b);
        ok &= rg.next(a);
        f.p[P_R2X] = static_cast<int8_t>(a);
        f.p[P_R2Y] = static_cast<int8_t>(b);
    }
    int type = T_COLOR;
    if (useDepth) {
        DevPrefixSampler<kPrefixDraws> ft;
        ft.init(mine, 0, 1);
        int v = 0;
        ok &= ft.next(v);
        type = (v == 0) ? T_DEPTH : T_COLOR;
    }
    f.p[P_TYPE] = static_cast<int8_t>(type);
    if (type == T_COLOR) {
        DevPrefixSampler<kPrefixDraws> cc;
        cc.init(mine + 3 * kStride, 0, 2);
        ok &= cc.next(b);
        ok &= cc.next(a);
        f.p[P_C1] = static_cast<int8_t>(a);
        f.p[P_C2] = static_cast<int8_t>(b);
    }
    if (!ok) atomicExch(err, 2);
    cand[static_cast<size_t>(job) * numCand + k] = f;
}

// getSortKey, random_tree_image.h:444-452
__device__ __forceinline__ int featureSortKey(const FeatRec& f) {
    int k = 0;
    k |= static_cast<int>(static_cast<uint8_t>(f.p[P_TYPE] & 0x03)) << 30;
    k |= static_cast<int>(static_cast<uint8_t>(f.p[P_C1] & 0x0F)) << 26;
    k |= static_cast<int>(static_cast<uint8_t>(f.p[P_C2] & 0x0F)) << 22;
    k |= static_cast<int>(static_cast<uint8_t>((f.p[P_O1Y] + 127) & 0xFF)) << 14;
    k |= static_cast<int>(static_cast<uint8_t>((f.p[P_O1X] + 127) & 0xFF)) << 6;
    return k;
}

// A candidate uses at least this many draws: T thresholds, or the 10 NaN responses that reject it.
__host__ __device__ __forceinline__ int minDraws(int T) { return T < 10 ? T : 10; }

// The next words of each job's index generator: as many as the features still missing are expected to
// take, tempered, and per wave the mask of those that uniform_int accepts; and, in the workgroups past the
// first, the job's next candidates, which wait for nothing of it.  MT19937 as the recurrence x[n + 624] =
// mix(x[n], x[n + 1], x[n + 397]) in an LDS ring: no word of the 227 after the last depends on another, and a
// lane's word 227 further on needs its own word and older ones, so four waves make two such steps per barrier
// while eight others temper, test and store the two before.  Bound by the latency of a step, after the 624
// dependent ones that seed the generator (with one step a barrier and all of it in the same four waves, and the
// candidates in a launch of their own: 59 + 13 us for 2000 features x 20 thresholds, 12 + 12 for 100 x 10; now
// 50 and 14).  uniform_int accepts a word w iff w / bucket <= range, that is iff w < bucket (range + 1).
constexpr int kMtStep = 227;
constexpr int kMtRing = 2048;
constexpr int kDrawLanes = 768;
__global__ void __launch_bounds__(kDrawLanes) k_fg_draws(const FeatGenJob* __restrict__ jobs, int F, int T, int ring,
        int fresh, float guess, WalkState* __restrict__ states, uint32_t* __restrict__ mtState, uint32_t* __restrict__ raw,
        unsigned long long* __restrict__ masks, int maxSteps, int numCand, int first, int count, int boxRadius,
        int regionSize, int useDepth, FeatRec* __restrict__ cand, int* __restrict__ err) {
    __shared__ uint32_t x[kMtRing];
    __shared__ int counts[kDrawLanes / 64];
    const int jobIdx = blockIdx.y;
    if (blockIdx.x > 0) {
        drawCandidates(jobs, jobIdx, static_cast<int>(blockIdx.x) - 1, numCand, first, count, boxRadius, regionSize,
                useDepth, cand, err);
        return;
    }
    const FeatGenJob job = jobs[jobIdx];
    WalkState st = states[jobIdx];
    if (fresh) {
        st = WalkState{};
        st.tries = 10;
        st.guess = guess;
    }
    if (st.done) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const UniformIntParams up = uniformIntParams(0, job.n - 1);
    uint32_t* saved = mtState + static_cast<size_t>(jobIdx) * 624;
    if (!fresh) {
        for (int i = tid; i < 624; i += kDrawLanes) x[i] = saved[i];
    } else if (tid == 0) {
        uint32_t v = static_cast<uint32_t>(job.seed);
        x[0] = v;
        for (uint32_t i = 1; i < 624; i++) {
            v = mtInitStep(v, i);
            x[i] = v;
        }
    }
    __syncthreads();
    // draws per feature so far, with the rejected candidates' share
    const double perFeature = st.generated > 0 ? static_cast<double>(st.drawsDone) / st.generated : st.guess;
    const double want = (F - st.generated) * perFeature * 1.06 + 2048.0;
    const int target = st.head + static_cast<int>(fmin(want, static_cast<double>(ring - 512)));
    const int missing = max(0, target - st.tail);
    int steps = 0, made = missing;   // a range of one value takes no words
    if (up.range != 0) {
        const unsigned long long limit = static_cast<unsigned long long>(up.bucket) * (up.range + 1ull);
        const double share = limit >= (1ull << 32) ? 1.0 : static_cast<double>(limit) / 4294967296.0;
        // at least half of the words are accepted, so the ring (at most ring - 512 ahead of the walk before
        // this, and no more than `missing` words over that) never overruns
        steps = min(maxSteps, min(static_cast<int>(missing / share), ring - 512 - (st.tail - st.head)) / kMtStep + (missing > 0 ? 1 : 0));
        uint32_t* out = raw + static_cast<size_t>(jobIdx) * maxSteps * 256;
        unsigned long long* mk = masks + static_cast<size_t>(jobIdx) * maxSteps * 4;
        made = 0;
        // lanes 0 .. 255 make steps s and s + 1, lanes 256 .. 511 and 512 .. 767 test steps s - 2 and s - 1
        const int half = tid >> 8, i = tid & 255;
        for (int s = 0; s < steps + 2; s += 2) {
            const int base = s * kMtStep + i;
            if (half == 0) {
                if (s < steps && i < kMtStep) {
                    const uint32_t a0 = x[base & (kMtRing - 1)], a1 = x[(base + 1) & (kMtRing - 1)];
                    const uint32_t b0 = x[(base + kMtStep) & (kMtRing - 1)], b1 = x[(base + kMtStep + 1) & (kMtRing - 1)];
                    const uint32_t w0 = mtMix(a0, a1, x[(base + 397) & (kMtRing - 1)]);
                    x[(base + 624) & (kMtRing - 1)] = w0;
                    x[(base + kMtStep + 624) & (kMtRing - 1)] = mtMix(b0, b1, w0);
                }
            } else {
                const int step = s - 3 + half;
                if (step >= 0 && step < steps) {
                    bool acc = false;
                    if (i < kMtStep) {
                        const uint32_t v = mtTemper(x[(base + 624 - (3 - half) * kMtStep) & (kMtRing - 1)]);
                        acc = v < limit;
                        out[step * 256 + i] = v;
                    }
                    const unsigned long long mask = __ballot(acc);
                    if (lane == 0) mk[step * 4 + (wave & 3)] = mask;
                    made += __popcll(mask);
                }
            }
            __syncthreads();
        }
        const int base = steps * kMtStep;
        if (lane == 0) counts[wave] = made;
        __syncthreads();
        made = 0;
        for (int w = 4; w < kDrawLanes / 64; w++) made += counts[w];
        for (int i = tid; i < 624; i += kDrawLanes) saved[i] = x[(base + i) & (kMtRing - 1)];
    }
    if (tid == 0) {
        st.recorded = st.tail;
        st.tail += made;
        st.steps = steps;
        states[jobIdx] = st;
    }
}

// The sample records behind the draws produced last, in draw order in the job's ring, so that every
// candidate whose band holds a draw reads its sample coalesced.  A workgroup takes a step's words; their
// place among the accepted ones is the count of the mask bits before them.
__global__ void __launch_bounds__(256) k_fg_records(const FeatGenJob* __restrict__ jobs,
        const WalkState* __restrict__ states, int ring, const uint32_t* __restrict__ raw,
        const unsigned long long* __restrict__ masks, int maxSteps, DrawRec* __restrict__ recs) {
    __shared__ int part[4];
    const WalkState st = states[blockIdx.y];
    if (st.done) return;
    const FeatGenJob job = jobs[blockIdx.y];
    const UniformIntParams up = uniformIntParams(0, job.n - 1);
    DrawRec* out = recs + static_cast<size_t>(blockIdx.y) * ring;
    auto record = [&](int index, int at) {
        const cf_sample s = job.samples[index];
        DrawRec r;
        const bool valid = s.depth_mm > 0;
        r.rinv = valid ? depthReciprocal(depthToFloat(s.depth_mm)) : 0.0;
        r.xy = s.x | (s.y << 16);
        r.image = valid ? static_cast<int>(s.image) : -1;
        out[at & (ring - 1)] = r;
    };
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (up.range == 0) {
        for (int i = st.recorded + blockIdx.x * 256 + tid; i < st.tail; i += gridDim.x * 256) record(up.lo, i);
        return;
    }
    const uint32_t* words = raw + static_cast<size_t>(blockIdx.y) * maxSteps * 256;
    const unsigned long long* mk = masks + static_cast<size_t>(blockIdx.y) * maxSteps * 4;
    for (int s = blockIdx.x; s < st.steps; s += gridDim.x) {
        int before = 0;
        for (int i = tid; i < 4 * s; i += 256) before += __popcll(mk[i]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
        if (lane == 0) part[wave] = before;
        __syncthreads();
        int at = st.recorded + part[0] + part[1] + part[2] + part[3];
        __syncthreads();
        unsigned long long own = 0;
        for (int w = 0; w <= wave; w++) {
            own = mk[4 * s + w];
            if (w < wave) at += __popcll(own);
        }
        if ((own >> lane) & 1ull) {
            record(static_cast<int>(static_cast<uint32_t>(up.lo) + words[s * 256 + tid] / up.bucket),
                    at + __popcll(own & ((1ull << lane) - 1ull)));
        }
    }
}

// position of the n-th set bit of w (n from 1, at most popcount(w))
__device__ __forceinline__ int nthBit(unsigned long long w, int n) {
    int pos = 0;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const int c = __popcll(w & ((1ull << s) - 1ull));
        if (n > c) {
            n -= c;
            w >>= s;
            pos += s;
        }
    }
    return pos;
}

constexpr int kBandMax = 2048;            // draws of the widest band
constexpr int kRoundCandMax = 224;        // candidates of a round
constexpr int kAdvanceLanes = 1024;
constexpr int kGroup = 8;                 // consecutive candidates that k_fg_advance composes
// What a candidate started at a draw of its band comes to, 16 bits: kAccept if it ends with its T-th threshold
// (else rejected) and, in the value bits, the place of its successor's first draw in the successor's band; with
// kLeave, that draw lies outside the successor's band and the value is where the candidate ends in its own;
// kOpen: it does not end inside its band.
constexpr uint16_t kOpen = 0x8000, kAccept = 0x4000, kLeave = 0x1000, kPlace = 0x0fff;
static_assert(kBandMax <= kPlace, "places and ends of a band fit the value bits");

// Band of a round for T thresholds: a power of two of at least 8 T draws.  A candidate uses about 1.25 T
// draws with a spread of T / 8, so the start of the round's j-th candidate is known to about sqrt(j) T / 8:
// 112 candidates are covered to their end (measured on 640x480 frames: T = 32, starts within 80 draws of the
// mean in nine rounds of ten).  Rounds of twice as many with bands of 256 draws often ended early and cost twice
// as much each (21 frames, 3 trees, 2000 x 20: 117.3 against 116.1 ms a training).
static int bandDraws(int T) {
    int b = 128;
    while (b < 8 * T && b < kBandMax) b *= 2;
    return b;
}

// Candidates of a round: 224 with the narrowest band, else 112 as far as their tables (two bytes an entry) fit
// the walker's LDS with the composed ones, and no more than a small feature table can need.
static int roundCandidates(int band, int F) {
    const int most = std::max(28672 / band, std::min(112, 57344 / band));
    return std::min(most, (F + F / 8 + 2 * kGroup) / kGroup * kGroup);
}

// The band of a round's candidate j, in draws from the walk's next one: around j times the draws that a candidate
// has used so far, wider the later the candidate.  The round and the walk over its tables both form it, in
// operations that no compilation contracts.
struct RoundBand {
    int lo, width;
};
__device__ __forceinline__ RoundBand roundBand(const WalkState& st, int j, int T, int band, int numCand, int drawn) {
    const float avg = __fdiv_rn(__fadd_rn(static_cast<float>(st.drawsDone), __fmul_rn(16.0f, st.guess)),
            __fadd_rn(static_cast<float>(st.candsDone), 16.0f));
    const float dev = __fadd_rn(8.0f, __fmul_rn(__fmul_rn(0.19f, avg), __fsqrt_rn(static_cast<float>(j))));
    RoundBand b;
    b.lo = j == 0 ? 0 : max(j * minDraws(T), static_cast<int>(__fsub_rn(__fmul_rn(static_cast<float>(j), avg), dev)));
    b.width = j == 0 ? band
                     : min(band, static_cast<int>(__fadd_rn(__fmul_rn(2.0f, dev), __fmul_rn(1.25f, avg))) + 8);
    b.width = max(0, min(b.width, st.tail - st.head - b.lo));
    if (st.k + j >= min(drawn, numCand)) b.width = 0;   // not drawn yet, or past the last: the walk stops here
    return b;
}

// One candidate of a round on its band (see the head of this file).  Bound by the latency of the corner
// gathers, which the round's candidates x trees workgroups overlap on all CUs.
__global__ void __launch_bounds__(256) k_fg_round(const WalkState* __restrict__ states, ImageSet imgs,
        const FeatRec* __restrict__ cand, int numCand, int drawn, int T, int ring, int band, const DrawRec* __restrict__ recs,
        float* __restrict__ resp, uint16_t* __restrict__ next, int2* __restrict__ firsts) {
    constexpr int kWords = kBandMax / 64;
    __shared__ unsigned long long finite[kWords], rejects[kWords];   // not NaN; tenth NaN of a run
    const WalkState st = states[blockIdx.y];
    const int j = blockIdx.x;
    if (st.done || st.k + j >= numCand) return;
    const size_t row = static_cast<size_t>(blockIdx.y) * gridDim.x + j;
    const RoundBand own = roundBand(st, j, T, band, numCand, drawn), after = roundBand(st, j + 1, T, band, numCand, drawn);
    const int lo = own.lo, width = own.width;
    const Feat f = loadFeat(cand + static_cast<size_t>(blockIdx.y) * numCand + st.k + j);
    const DrawRec* rec = recs + static_cast<size_t>(blockIdx.y) * ring;
    const size_t plane = static_cast<size_t>(imgs.W) * imgs.H;
    for (int i = threadIdx.x; i < band; i += blockDim.x) {
        float v = __builtin_nanf("");
        if (i < width) {
            const DrawRec r = rec[(st.head + lo + i) & (ring - 1)];
            int idx[8];
            if (r.image >= 0 && responseCorners(f, r.xy & 0xffff, static_cast<int>(static_cast<uint32_t>(r.xy) >> 16),
                    imgs.W, imgs.H, r.rinv, false, idx)) {
                if (f.type == T_DEPTH) {
                    const int2* dep = imgs.dep + static_cast<size_t>(r.image) * plane;
                    int2 cv[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) cv[e] = planeAt(dep, idx[e]);
                    v = static_cast<float>(depthResponseFromCorners(cv));
                } else {
                    const float* col = imgs.col + static_cast<size_t>(r.image) * 3 * plane;
                    const float* colA = col + static_cast<size_t>(f.c1) * plane;
                    const float* colB = col + static_cast<size_t>(f.c2) * plane;
                    float c8[8];
#pragma unroll
                    for (int e = 0; e < 4; e++) c8[e] = planeAt(colA, idx[e]);
#pragma unroll
                    for (int e = 4; e < 8; e++) c8[e] = planeAt(colB, idx[e]);
                    v = static_cast<float>(colorResponseFromCorners(c8));
                }
            }
            resp[row * band + i] = v;
        }
        const unsigned long long fm = __ballot(i < width && !__builtin_isnan(v));
        if ((i & 63) == 0) finite[i >> 6] = fm;
    }
    __syncthreads();
    const int words = band / 64;
    // NaN draws of word w inside the band
    auto nanWord = [&](int w) -> unsigned long long {
        if (w < 0 || width <= w * 64) return 0ull;
        const int n = width - w * 64;
        return ~finite[w] & (n >= 64 ? ~0ull : ((1ull << n) - 1ull));
    };
    if (static_cast<int>(threadIdx.x) < words) {
        // runs of 10 on the pair (previous word, word): ends of runs of 2, 4, 8, then 8 + 2
        unsigned long long hi = nanWord(threadIdx.x), lw = nanWord(static_cast<int>(threadIdx.x) - 1);
        auto andShifted = [&](int s, unsigned long long h2, unsigned long long l2) {
            hi &= (h2 << s) | (l2 >> (64 - s));
            lw &= l2 << s;
        };
        andShifted(1, hi, lw);
        const unsigned long long h2 = hi, l2 = lw;
        andShifted(2, hi, lw);
        andShifted(4, hi, lw);
        andShifted(8, h2, l2);
        rejects[threadIdx.x] = hi;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < width; i += blockDim.x) {
        // the first of: the T-th finite draw from i on, the tenth NaN of a run that starts at i or later
        int need = T, end = 0;
        uint16_t how = kOpen;
        if (j == 0 && i == 0) {
            // thresholds found and tries left when the candidate ran past the last round's band
            need = T - st.t;
            const unsigned long long n0 = nanWord(0);
            const int lead = ~n0 ? __builtin_ctzll(~n0) : 64;
            if (lead >= st.tries) {
                end = st.tries;
                how = 0;
            }
        }
        for (int w = i >> 6; how == kOpen && w < words; w++) {
            unsigned long long fw = finite[w], rw = rejects[w];
            const int from = i - w * 64, rejFrom = from + 9;
            if (from > 0) fw &= ~0ull << from;
            if (rejFrom >= 64) rw = 0ull;
            else if (rejFrom > 0) rw &= ~0ull << rejFrom;
            const int c = __popcll(fw);
            const int a = c >= need ? nthBit(fw, need) : 64;
            const int r = rw ? __builtin_ctzll(rw) : 64;
            if (a < 64 || r < 64) {
                how = a < r ? kAccept : 0;
                end = w * 64 + min(a, r) + 1;
            }
            need -= c;
        }
        if (how != kOpen) {
            const int place = lo + end - after.lo;
            how |= place >= 0 && place < after.width ? place : (kLeave | end);
        }
        next[row * band + i] = how;
    }
    if (threadIdx.x == 0 && j == 0) {
        // the band's finite draws and the NaN draws after the last of them, for a candidate that runs past it
        int found = 0, last = -1;
        for (int w = 0; w < words; w++) {
            found += __popcll(finite[w]);
            if (finite[w]) last = w * 64 + 63 - __clzll(finite[w]);
        }
        firsts[blockIdx.y] = make_int2(found, width - 1 - last);
    }
}

// What the walk did with candidate j of a round: it used the band's draws [begin, end) and ended with
// st = 1 (accepted into output slot `slot`), 0 (still open at its band's end), or 2 (rejected, or not
// reached).
struct WalkStep {
    int st, begin, end, t0, slot;
};

// Follows the candidates of a round through their tables, from the state's next draw and candidate on.  The
// round ends at the first candidate that starts outside its band or does not end inside it; the round's first
// candidate, which starts at its band's first draw, then carries its thresholds and tries into the next.
// Bound by the chain of dependent LDS reads.  The chain is shortened by composing the tables of kGroup
// consecutive candidates for every start of the first's band, all in parallel: the walk then takes a read per
// group, checks all groups at once, and the groups it passed are expanded in parallel.  An entry is the place of
// the next entry to read, so that a step of a chain is one read and two operations (with the draw's number in
// the entry, and each candidate's band read beside it to find the place: F = 4000, T = 32 18 us a launch, of
// them 6.6 composing and 3.8 walking; now 11, 2.3 and 1.9).
__global__ void __launch_bounds__(kAdvanceLanes) k_fg_advance(const FeatGenJob* __restrict__ jobs,
        WalkState* __restrict__ states, const FeatRec* __restrict__ cand, int numCand, int drawn, int F, int T,
        int band, int m, const float* __restrict__ resp, const uint16_t* __restrict__ next,
        const int2* __restrict__ firsts, FeatRec* __restrict__ outFeat, float* __restrict__ outThr,
        int* __restrict__ outKey) {
    // uint16 [m][band], then per group of kGroup candidates uint32 [band]: the place after the group's last
    // candidate, its accepted candidates << 16, or kGroupStop if the walk leaves the bands inside the group
    extern __shared__ uint4 tableWords[];
    __shared__ RoundBand bd[kRoundCandMax + 1];
    __shared__ WalkStep steps[kRoundCandMax];
    __shared__ int groupStart[kRoundCandMax / kGroup], groupGen[kRoundCandMax / kGroup];   // start -1: not passed whole
    constexpr uint32_t kGroupStop = 0xffffffffu;
    constexpr int kHold = 4;   // table words loaded while the state is
    const int tid = threadIdx.x, lane = tid & 63;
    const size_t row0 = static_cast<size_t>(blockIdx.x) * m;
    const uint4* src = reinterpret_cast<const uint4*>(next + row0 * band);
    const int words = m * band / 8, groups = m / kGroup;
    uint4 hold[kHold];
#pragma unroll
    for (int u = 0; u < kHold; u++) hold[u] = src[min(tid + u * kAdvanceLanes, words - 1)];
    const WalkState st = states[blockIdx.x];
#pragma unroll
    for (int u = 0; u < kHold; u++) __asm__ volatile("" : : "v"(hold[u].x), "v"(hold[u].y), "v"(hold[u].z), "v"(hold[u].w));
    if (st.done) return;
#pragma unroll
    for (int u = 0; u < kHold; u++) {
        if (tid + u * kAdvanceLanes < words) tableWords[tid + u * kAdvanceLanes] = hold[u];
    }
    for (int i = tid + kHold * kAdvanceLanes; i < words; i += kAdvanceLanes) tableWords[i] = src[i];
    for (int i = tid; i <= m; i += kAdvanceLanes) {
        bd[i] = roundBand(st, i, T, band, numCand, drawn);
        if (i < m) steps[i].st = 2;
    }
    for (int i = tid; i < groups; i += kAdvanceLanes) groupStart[i] = -1;
    __syncthreads();
    const uint16_t* table = reinterpret_cast<const uint16_t*>(tableWords);
    uint32_t* composed = reinterpret_cast<uint32_t*>(tableWords + words);
    constexpr int kChains = 4;   // chains that a lane follows together
    const int bandShift = 31 - __clz(band);
    for (int i0 = tid; i0 < groups * band; i0 += kAdvanceLanes * kChains) {
        const uint16_t* row[kChains];
        int at[kChains];
        uint32_t seen[kChains], accepted[kChains];
#pragma unroll
        for (int u = 0; u < kChains; u++) {
            const int i = i0 + u * kAdvanceLanes, g = min(i >> bandShift, groups - 1);
            row[u] = table + ((g * kGroup) << bandShift);
            at[u] = i & (band - 1);
            // (rows hold entries up to their band's width only)
            seen[u] = at[u] < bd[g * kGroup].width ? 0u : kOpen;
            if (seen[u]) at[u] = 0;
            accepted[u] = 0;
        }
#pragma unroll
        for (int q = 0; q < kGroup; q++) {
            uint32_t e[kChains];
#pragma unroll
            for (int u = 0; u < kChains; u++) e[u] = row[u][(q << bandShift) + at[u]];
#pragma unroll
            for (int u = 0; u < kChains; u++) {
                seen[u] |= e[u];
                accepted[u] += e[u] & kAccept;
                at[u] = seen[u] & (kOpen | kLeave) ? 0 : static_cast<int>(e[u] & kPlace);
            }
        }
#pragma unroll
        for (int u = 0; u < kChains; u++) {
            const int i = i0 + u * kAdvanceLanes;
            if (i < groups * band) {
                composed[i] = seen[u] & (kOpen | kLeave) ? kGroupStop
                                                         : static_cast<uint32_t>(at[u]) | (accepted[u] / kAccept << 16);
            }
        }
    }
    __syncthreads();
    const int outOffset = jobs[blockIdx.x].outOffset;
    if (tid < 64) {
        // wave 0: the groups that are passed whole.  Lane g keeps where group g starts and what it accepts; past a
        // stop the reads go on at place 0 and count for nothing.
        int start = 0, at = 0;
        uint32_t mine = kGroupStop;
        bool inside = bd[0].width > 0;
        for (int g = 0; g < groups; g++) {
            const uint32_t c = composed[(g << bandShift) + at];
            if (lane == g) {
                start = at;
                mine = inside ? c : kGroupStop;
            }
            inside = inside && c != kGroupStop;
            at = inside ? static_cast<int>(c & kPlace) : 0;
        }
        // features accepted before group `lane`: a group counts only if the features and candidates cannot run
        // out in it
        int before = mine == kGroupStop ? 0 : static_cast<int>(mine >> 16);
        const int own = before;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(before, d, 64);
            if (lane >= d) before += o;
        }
        before += st.generated - own;
        const bool pass = mine != kGroupStop && before + kGroup < F && st.k + (lane + 1) * kGroup < 3 * F;
        const unsigned long long fails = __ballot(!pass);
        const int passed = fails ? __builtin_ctzll(fails) : 64;   // lanes past the groups fail
        if (lane < passed) {
            groupStart[lane] = start;
            groupGen[lane] = before;
        }
        // the candidates one by one from there on, all lanes in step: the walk's state is uniform
        int j = passed * kGroup, gen = __shfl(before, passed, 64), err = 0;
        at = 0;
        if (passed > 0) at = static_cast<int>(__shfl(mine, passed - 1, 64) & kPlace);
        j = __builtin_amdgcn_readfirstlane(j);
        gen = __builtin_amdgcn_readfirstlane(gen);
        at = __builtin_amdgcn_readfirstlane(at);
        int left = j > 0 || bd[0].width > 0 ? -1 : 0;   // the draw at which the walk left the bands
        bool open = false;
        while (j < m) {
            // `--maxLoops <= 0` with maxLoops = 3F, checked right after sampling candidate k
            if (gen >= F || st.k + j + 1 >= 3 * F) {
                err = gen < F;
                break;
            }
            if (left >= 0) break;   // its first draw was not evaluated: the next round starts here
            const int e = __builtin_amdgcn_readfirstlane(table[(j << bandShift) + at]);
            const int p = bd[j].lo + at;
            if (e & kOpen) {
                open = j == 0;
                left = open ? bd[0].width : p;
                if (open && lane == 0) steps[0] = WalkStep{0, p, left, st.t, outOffset + gen};
                break;
            }
            const int value = e & kPlace;
            const int end = e & kLeave ? bd[j].lo + value : bd[j + 1].lo + value;
            if (e & kLeave) left = end;
            at = value;
            if (e & kAccept) {
                if (lane == 0) steps[j] = WalkStep{1, p, end, j == 0 ? st.t : 0, outOffset + gen};
                gen++;
            }
            j++;
        }
        const int p = left >= 0 ? left : bd[j].lo + at;
        if (lane == 0) {
            WalkState ns = st;
            ns.head = st.head + p;
            ns.k = st.k + j;
            ns.generated = gen;
            ns.err = err;
            ns.done = gen >= F || err != 0;
            if (open) {   // its draws count once it has ended
                const int2 first = firsts[blockIdx.x];
                ns.openDraws = st.openDraws + p;
                ns.t = st.t + first.x;
                ns.tries = first.x > 0 ? 10 - first.y : st.tries - first.y;
            } else if (j > 0) {
                ns.drawsDone = st.drawsDone + st.openDraws + p;
                ns.candsDone = st.candsDone + j;
                ns.openDraws = 0;
                ns.t = 0;
                ns.tries = 10;
            }
            states[blockIdx.x] = ns;
        }
    }
    __syncthreads();
    if (tid < groups && groupStart[tid] >= 0) {
        int at = groupStart[tid], slot = outOffset + groupGen[tid];
        for (int j = tid * kGroup; j < tid * kGroup + kGroup; j++) {
            const int e = table[(j << bandShift) + at], after = e & kPlace;
            if (e & kAccept) {
                steps[j] = WalkStep{1, bd[j].lo + at, bd[j + 1].lo + after, j == 0 ? st.t : 0, slot++};
            }
            at = after;
        }
    }
    __syncthreads();
    for (int j = tid; j < m; j += kAdvanceLanes) {
        if (steps[j].st != 1) continue;
        const FeatRec fr = cand[static_cast<size_t>(blockIdx.x) * numCand + st.k + j];
        outFeat[steps[j].slot] = fr;
        outKey[steps[j].slot] = featureSortKey(fr);
    }
    // thresholds of the accepted and the still open candidates: their finite draws in order, a wave per
    // candidate, the first 64 draws of kAhead candidates loaded together
    constexpr int kWaves = kAdvanceLanes / 64, kAhead = 7;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int ja = tid >> 6; ja < m; ja += kWaves * kAhead) {
        float v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const int j = ja + u * kWaves;
            v[u] = __builtin_nanf("");
            if (j < m && steps[j].st != 2) {
                const int i = steps[j].begin + lane;
                if (i < steps[j].end) v[u] = resp[(row0 + j) * band + (i - bd[j].lo)];
            }
        }
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const int j = ja + u * kWaves;
            if (j >= m || steps[j].st == 2) continue;
            const WalkStep ws = steps[j];
            float* to = outThr + static_cast<size_t>(ws.slot) * T + ws.t0;
            float cur = v[u];
            for (int i0 = ws.begin;;) {
                const unsigned long long fm = __ballot(!__builtin_isnan(cur));
                if (!__builtin_isnan(cur)) to[__popcll(fm & below)] = cur;
                to += __popcll(fm);
                i0 += 64;
                if (i0 >= ws.end) break;
                cur = i0 + lane < ws.end ? resp[(row0 + j) * band + (i0 + lane - bd[j].lo)] : __builtin_nanf("");
            }
        }
    }
}

// #{k : th[k] < th[t]} of threshold t among its feature's T.  A sample with float key q goes left at threshold
// t iff q <= th[t] iff #{k : th[k] < q} is at most that.
__device__ __forceinline__ uint16_t thresholdRank(const float* __restrict__ th, int T, int t) {
    const float v = th[t];
    int r = 0;
#pragma unroll 8
    for (int k = 0; k < T; k++) r += (th[k] < v) ? 1 : 0;
    return static_cast<uint16_t>(r);
}

// Stable sort of each job's F features by key (rank = #smaller keys + #equal keys earlier), scattering the
// features and their threshold tables: values, ranks, the rows padded to TM with +inf that the
// evaluation kernels compare against (a NaN threshold becomes +inf and -0 becomes +0; neither changes any comparison
// th < q), and, where asked for, the reference's layouts.  The keys start with (type, channel1, channel2), so
// the sorted order also groups the features by the planes they read.
//
// A workgroup ranks kSortFeat features against all keys, which lie in LDS, 16 lanes a feature, and the features'
// thresholds against one another, in LDS too.  Bound by those reads: 12 us for 3 x 2000
// features with 20 thresholds, 9.5 for 2 x 500 with 50 (21 and 29 with 64 features a workgroup, a lane a feature,
// thresholds read from memory).
constexpr int kSortFeat = 16, kSortLanes = 16;   // features of a workgroup, lanes of a feature
__global__ void __launch_bounds__(kSortFeat * kSortLanes) k_fg_sort(const int* __restrict__ keys,
        const FeatRec* __restrict__ inFeat, const float* __restrict__ inThr, int F, int T, int TM,
        FeatRec* __restrict__ feat, float* __restrict__ thrFT, uint16_t* __restrict__ rank, float* __restrict__ thrPad,
        float* __restrict__ thrTF, int8_t* __restrict__ soa) {
    extern __shared__ int sk[];                       // [F] keys
    float* th = reinterpret_cast<float*>(sk + F);     // [kSortFeat][T]
    __shared__ int place[kSortFeat];
    constexpr int kLanes = kSortFeat * kSortLanes;
    const size_t jobF = static_cast<size_t>(blockIdx.y) * F;
    const int i0 = blockIdx.x * kSortFeat, nf = min(kSortFeat, F - i0);
    for (int i = threadIdx.x; i < F; i += kLanes) sk[i] = keys[jobF + i];
    for (int e = threadIdx.x; e < nf * T; e += kLanes) th[e] = inThr[(jobF + i0) * T + e];
    __syncthreads();
    const int own = threadIdx.x / kSortLanes, sub = threadIdx.x % kSortLanes;
    if (own < nf) {
        const int i = i0 + own, ki = sk[i];
        int r = 0;
#pragma unroll 8
        for (int j = sub; j < F; j += kSortLanes) r += (sk[j] < ki || (sk[j] == ki && j < i)) ? 1 : 0;
#pragma unroll
        for (int o = kSortLanes / 2; o > 0; o >>= 1) r += __shfl_xor(r, o, kSortLanes);
        if (sub == 0) {
            place[own] = r;
            const FeatRec fr = inFeat[jobF + i];
            feat[jobF + r] = fr;
            if (soa) {
                for (int p = 0; p < kFeatParams; p++) {
                    soa[(static_cast<size_t>(blockIdx.y) * kFeatParams + p) * F + r] = fr.p[p];
                }
            }
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nf * T; e += kLanes) {
        const int l = e / T, t = e - l * T, dst = place[l];
        const float v = th[e];
        const size_t row = (jobF + dst) * T;
        thrFT[row + t] = v;
        rank[row + t] = thresholdRank(th + l * T, T, t);
        thrPad[(jobF + dst) * TM + t] = (v != v) ? __builtin_inff() : v + 0.0f;
        if (thrTF) thrTF[(static_cast<size_t>(blockIdx.y) * T + t) * F + dst] = v;
    }
    const int padT = TM - T;
    for (int e = threadIdx.x; e < nf * padT; e += kLanes) {
        const int l = e / padT;
        thrPad[(jobF + place[l]) * TM + T + (e - l * padT)] = __builtin_inff();
    }
}

// Reference layout in (soa [trees][11][F], thrTF [trees][T][F]) -> feat, thrFT.
__global__ void __launch_bounds__(256) k_tables_from_reference(const int8_t* __restrict__ soa,
        const float* __restrict__ thrTF, int trees, int F, int T, FeatRec* __restrict__ feat,
        float* __restrict__ thrFT) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= trees * F) return;
    const int job = i / F, f = i % F;
    FeatRec fr;
#pragma unroll
    for (int p = 0; p < 16; p++) fr.p[p] = 0;
    for (int p = 0; p < kFeatParams; p++) fr.p[p] = soa[(static_cast<size_t>(job) * kFeatParams + p) * F + f];
    feat[i] = fr;
    for (int t = 0; t < T; t++) thrFT[static_cast<size_t>(i) * T + t] = thrTF[(static_cast<size_t>(job) * T + t) * F + f];
}

// The ranks and the padded rows of every feature's thresholds, one lane per entry of a padded row.
__global__ void __launch_bounds__(256) k_threshold_ranks(const float* __restrict__ thrFT, int total, int T, int TM,
        uint16_t* __restrict__ rank, float* __restrict__ thrPad) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<size_t>(total) * TM) return;
    const size_t f = i / TM;
    const int t = static_cast<int>(i - f * TM);
    const float* th = thrFT + f * T;
    const float v = t < T ? th[t] : __builtin_inff();
    thrPad[i] = (v != v) ? __builtin_inff() : v + 0.0f;
    if (t < T) rank[f * T + t] = thresholdRank(th, T, t);
}

void launchFeatureGeneration(hipStream_t s, const ImageSet& imgs, const FeatGenJob* jobsDev, int numJobs, int F,
        int T, int boxRadius, int regionSize, int useDepth, FeatTables& tabs, bool referenceLayouts) {
    if (T > kMaxThresholds) throw Error(CF_ERR_ARG, "too many thresholds (max 256)");
    if (F > 8192) throw Error(CF_ERR_ARG, "too many features (max 8192)");
    if (boxRadius > 127 || regionSize > 127) throw Error(CF_ERR_ARG, "boxRadius/regionSize must fit int8");
    // a candidate's second offset is drawn until it differs from the first: with one offset to draw, for ever
    if (boxRadius < 1) throw Error(CF_ERR_ARG, "boxRadius must be at least 1");
    const int numCand = 3 * F;
    tabs.trees = numJobs;
    tabs.F = F;
    tabs.T = T;
    tabs.cand.resize(static_cast<size_t>(numJobs) * numCand);
    tabs.unsortedFeat.resize(static_cast<size_t>(numJobs) * F);
    tabs.unsortedThr.resize(static_cast<size_t>(numJobs) * F * T);
    tabs.unsortedKey.resize(static_cast<size_t>(numJobs) * F);
    tabs.feat.resize(static_cast<size_t>(numJobs) * F);
    tabs.thrFT.resize(static_cast<size_t>(numJobs) * F * T);
    if (referenceLayouts) {
        tabs.thrTF.resize(static_cast<size_t>(numJobs) * F * T);
        tabs.soa.resize(static_cast<size_t>(numJobs) * F * kFeatParams);
    }
    tabs.rank.resize(static_cast<size_t>(numJobs) * F * T);
    const int TM = binThresholdWidth(T);
    tabs.thrPad.resize(static_cast<size_t>(numJobs) * F * TM);
    const int band = bandDraws(T);
    const int m = roundCandidates(band, F);
    int ring = 1 << 14;
    while (ring < (1 << 19) && ring < 2.0 * F * T) ring *= 2;
    const int maxSteps = ring / kMtStep + 1;
    // the walk's buffers in one allocation (hipMalloc and hipFree cost a small training more than the walk)
    const size_t n = static_cast<size_t>(numJobs), perRound = n * m * band;
    size_t bytes = 0;
    auto part = [&](size_t b) {
        const size_t at = bytes;
        bytes += (b + 255) & ~static_cast<size_t>(255);
        return at;
    };
    const size_t oWalk = part(n * sizeof(WalkState) + sizeof(int)), oMt = part(n * 624 * sizeof(uint32_t)),
            oRaw = part(n * maxSteps * 256 * sizeof(uint32_t)), oMasks = part(n * maxSteps * 4 * sizeof(uint64_t)),
            oRecs = part(n * ring * sizeof(DrawRec)), oResp = part(perRound * sizeof(float)),
            oNext = part(perRound * sizeof(uint16_t)), oFirsts = part(n * sizeof(int2));
    tabs.walkSpace.resize(bytes);
    uint8_t* space = tabs.walkSpace.get();
    WalkState* dWalk = reinterpret_cast<WalkState*>(space + oWalk);
    int* dErr = reinterpret_cast<int*>(dWalk + numJobs);   // read back with the states
    CF_HIP(hipMemsetAsync(dErr, 0, sizeof(int), s));
    uint32_t* dMt = reinterpret_cast<uint32_t*>(space + oMt);
    uint32_t* dRaw = reinterpret_cast<uint32_t*>(space + oRaw);
    unsigned long long* dMasks = reinterpret_cast<unsigned long long*>(space + oMasks);
    DrawRec* dRecs = reinterpret_cast<DrawRec*>(space + oRecs);
    float* dResp = reinterpret_cast<float*>(space + oResp);
    uint16_t* dNext = reinterpret_cast<uint16_t*>(space + oNext);
    int2* dFirsts = reinterpret_cast<int2*>(space + oFirsts);
    // a candidate in twenty or fewer is rejected on ordinary frames: the rest are drawn if they are needed
    int drawnBefore = 0, drawn = std::min(numCand, F + F / 8 + 64);
    const size_t stateBytes = n * sizeof(WalkState) + sizeof(int);
    uint8_t* host = tabs.walkHost.resize(stateBytes);
    std::memset(host, 0, stateBytes);
    const WalkState* states = reinterpret_cast<const WalkState*>(host);
    int errHost = 0;
    // draws of a candidate: the mean of these tables' last generation (the level before), or 5/4 T
    const float guess = tabs.meanDraws > 0 ? tabs.meanDraws : 1.25f * T;
    // The rounds the missing features are expected to take are enqueued together with the sort that
    // follows (rounds after a job's last feature return at once); in the rare case that a job needs
    // more, they and the sort are enqueued again.
    for (bool fresh = true, more = true; more; fresh = false) {
        int missing = 0;
        for (int j = 0; j < numJobs; j++) missing = std::max(missing, states[j].done ? 0 : F - states[j].generated);
        // (without a table before this one to go by, the first rounds are short: a candidate's mean use is
        // only guessed)
        const int rounds = std::min(64, missing / std::max(1, m * 9 / 10) + (fresh && tabs.meanDraws > 0 ? 2 : 4));
        const int candBlocks = (drawn - drawnBefore + kCandBlock - 1) / kCandBlock;
        hipLaunchKernelGGL(k_fg_draws, dim3(1 + candBlocks, numJobs), dim3(kDrawLanes), 0, s, jobsDev, F, T, ring,
                fresh ? 1 : 0, guess, dWalk, dMt, dRaw, dMasks, maxSteps, numCand, drawnBefore, drawn - drawnBefore,
                boxRadius, regionSize, useDepth, tabs.cand.get(), dErr);
        drawnBefore = drawn;
        const int steps = static_cast<int>(std::min<double>(maxSteps, 1.4 * missing * T / kMtStep + 12));
        hipLaunchKernelGGL(k_fg_records, dim3(steps, numJobs), dim3(256), 0, s, jobsDev, dWalk, ring, dRaw,
                dMasks, maxSteps, dRecs);
        const size_t lds = static_cast<size_t>(m) * band * 2 + static_cast<size_t>(m / kGroup) * band * 4;
        allowLds(reinterpret_cast<const void*>(&k_fg_advance), lds);
        const size_t sortLds = F * sizeof(int) + kSortFeat * T * sizeof(float);   // 48 KiB at most
        for (int r = 0; r < rounds; r++) {
            hipLaunchKernelGGL(k_fg_round, dim3(m, numJobs), dim3(std::min(band, 256)), 0, s, dWalk, imgs,
                    tabs.cand.get(), numCand, drawn, T, ring, band, dRecs, dResp, dNext, dFirsts);
            hipLaunchKernelGGL(k_fg_advance, dim3(numJobs), dim3(kAdvanceLanes), lds, s, jobsDev, dWalk,
                    tabs.cand.get(), numCand, drawn, F, T, band, m, dResp, dNext, dFirsts,
                    tabs.unsortedFeat.get(), tabs.unsortedThr.get(), tabs.unsortedKey.get());
        }
        hipLaunchKernelGGL(k_fg_sort, dim3((F + kSortFeat - 1) / kSortFeat, numJobs), dim3(kSortFeat * kSortLanes),
                sortLds, s,
                tabs.unsortedKey.get(), tabs.unsortedFeat.get(), tabs.unsortedThr.get(), F, T, TM, tabs.feat.get(),
                tabs.thrFT.get(), tabs.rank.get(), tabs.thrPad.get(),
                referenceLayouts ? tabs.thrTF.get() : nullptr, referenceLayouts ? tabs.soa.get() : nullptr);
        CF_HIP(hipMemcpyAsync(host, dWalk, stateBytes, hipMemcpyDeviceToHost, s));
        CF_HIP(hipStreamSynchronize(s));
        std::memcpy(&errHost, host + n * sizeof(WalkState), sizeof(int));
        more = false;
        for (int j = 0; j < numJobs; j++) {
            if (states[j].err != 0 && errHost == 0) errHost = states[j].err;
            more = more || !states[j].done;
        }
        if (errHost != 0) break;
        if (more) drawn = numCand;
    }
    double draws = 0, cands = 0;
    for (int j = 0; j < numJobs; j++) {
        draws += states[j].drawsDone;
        cands += states[j].candsDone;
    }
    tabs.meanDraws = cands > 0 ? static_cast<float>(draws / cands) : 0.0f;
    if (errHost == 1) throw Error(CF_ERR_RUNTIME, "failed to generate random features. max loops exceeded");
    if (errHost == 2) throw Error(CF_ERR_RUNTIME, "feature sampler needed more engine outputs than provisioned");
}

void launchPrepareTables(hipStream_t s, int trees, int F, int T, FeatTables& tabs) {
    if (T > kMaxThresholds) throw Error(CF_ERR_ARG, "too many thresholds (max 256)");
    tabs.trees = trees;
    tabs.F = F;
    tabs.T = T;
    tabs.feat.resize(static_cast<size_t>(trees) * F);
    tabs.thrFT.resize(static_cast<size_t>(trees) * F * T);
    tabs.rank.resize(static_cast<size_t>(trees) * F * T);
    const int total = trees * F;
    hipLaunchKernelGGL(k_tables_from_reference, dim3((total + 255) / 256), dim3(256), 0, s, tabs.soa.get(),
            tabs.thrTF.get(), trees, F, T, tabs.feat.get(), tabs.thrFT.get());
    const int TM = binThresholdWidth(T);
    tabs.thrPad.resize(static_cast<size_t>(total) * TM);
    const size_t entries = static_cast<size_t>(total) * TM;
    hipLaunchKernelGGL(k_threshold_ranks, dim3(static_cast<unsigned>((entries + 255) / 256)), dim3(256), 0, s,
            tabs.thrFT.get(), total, T, TM, tabs.rank.get(), tabs.thrPad.get());
}

}  // namespace cf
