// Split evaluation of a frontier of nodes:
//
//   k_eval_hist   one workgroup per (node chunk, feature tile): the double
//                 response of every (sample, feature), mapped to its interval
//                 among the feature's thresholds, counted per class in LDS
//                 ("interval histogram", T+1 bins x C classes per feature),
//                 then added to the node's global bins.
//                 Replaces featureResponseKernel + aggregateHistogramsKernel
//                 (random_tree_image_gpu.cu:1455-1720) and the CPU counter
//                 loop (random_tree_image.cpp:97-153): the response is never
//                 stored and never re-read per threshold.
//   k_scores      one thread per (node, feature, threshold): prefix sums over the bins
//                 give every threshold's left/right class counts; FP64
//                 NormalizedInformationGainScore (score.h:45-216) in the
//                 reference's operation order; per-feature best / second best
//                 (scoreFeatures; small nodes are scored by k_eval_hist itself).
//   k_reduce      per node: the reference's threshold-major sequential argmax
//                 with its 1e-13 tie rule (random_tree_image.cpp:445-457,
//                 random_tree.cpp:36-52) as max + first occurrence, valid
//                 whenever no score lies within 1e-13 below the maximum; such
//                 nodes are flagged and replayed sequentially (k_seq_argmax).
//
// Left at threshold t  <=>  r <= t  <=>  q := roundUpToFloat(r) <= t
//                      <=>  bin(q) := #{k : thr[k] < q} <= rank[t]
// with NaN responses in bin T (always right), so left(t, c) is the prefix sum
// of the bins up to rank[t].
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "cf_score.h"

namespace cf {

constexpr int kEvalThreads = 256;
constexpr int kEvalStep = 4;           // features whose corner gathers are issued together
constexpr int kEvalTile = 16;          // features of a workgroup
constexpr int kEvalSmallTile = 4;      // the same where there are few workgroups

// One training pixel held in registers for the feature loop.
struct RegSample {
    double rinv;   // depthReciprocal(depth in metres)
    int img;
    int xy;        // x | y << 16
    int lab;       // label | flip << 8 | (invalid depth) << 10;  < 0: empty slot
};

// #{t : th[t] < q} over a row padded with +inf, T for NaN.
template<int TM>
__device__ __forceinline__ int binOf(float q, const float (&th)[TM], int T) {
    uint32_t b = 0;
#pragma unroll
    for (int t = 0; t < TM; t++) b += (th[t] < q) ? 1u : 0u;
    return (q != q) ? T : static_cast<int>(b);
}

// What a workgroup that counts a node completely needs to score it: the node's class counts, the tables' ranks, the
// node's summaries (null: it does not).
struct NodeScoring {
    const uint32_t* hist = nullptr;
    const uint16_t* rank = nullptr;
    FeatSummary* summ = nullptr;
};

// All images of a set share W x H and are stored back to back, so a sample's
// integrals are found from its image index.
//
// Work mapping: the (chunk, feature tile) pairs, chunk by chunk, are cut into
// eighths, one per XCD (workgroup L runs on XCD L % 8), so that an XCD sweeps
// all feature tiles of one chunk (a region of one image or a few) before the
// next and its L2 holds that region's integrals; with a single chunk it takes
// neighbouring features, which read the same planes.  A node's chunks dealt to
// the XCDs tile by tile had each of them read every image: 7.8 ms for the 117
// nodes of 8 frames, 1000 x 20, now 5.2; groups of 2, 4, 8 chunks swept tile by
// tile 5.4, 5.7, 5.9.
//
// A lane holds one sample and issues the gathers of kEvalStep features before the
// first response is formed: a small node is bound by their latency, and four
// samples of one feature per lane left three quarters of the lanes of a
// 256-sample chunk idle.
//
// With full tiles the four waves take the same 64 samples at a time and a quarter
// of the features each, whose corners fall on the same lines of the L1 (3.30 ->
// 3.11 lines fetched per response; the nodes above 5.2 -> 4.95 ms).  With small
// tiles each wave takes its own samples.
template<int TM>
__global__ void __launch_bounds__(kEvalThreads) k_eval_hist(const float* __restrict__ colBase,
        const int2* __restrict__ depBase, int W, int H, const cf_sample* __restrict__ samples,
        const Chunk* __restrict__ chunks, Chunk node, int chunkLen, int numChunks, int tile, int tiles,
        const FeatRec* __restrict__ feat, const float* __restrict__ thrPad, int F, int T, int C,
        uint32_t* __restrict__ G, NodeScoring scoring) {
    extern __shared__ double evalLds[];   // scoreFeatures' part where the tile is scored, the bins
    uint32_t* h = reinterpret_cast<uint32_t*>(evalLds) + (scoring.summ ? scoreLdsBytes(tile, T, C) / sizeof(uint32_t) : 0);
    const int total = numChunks * tiles, per = (total + kNumXcds - 1) / kNumXcds;
    const int item = static_cast<int>(blockIdx.x % kNumXcds) * per + static_cast<int>(blockIdx.x / kNumXcds);
    if (item >= total) return;
    const int chunkIdx = item / tiles, tileIdx = item - chunkIdx * tiles;
    Chunk ch = node;
    if (chunks) {
        ch = chunks[chunkIdx];
    } else {
        ch.begin += chunkIdx * chunkLen;
        ch.count = min(chunkLen, ch.count - chunkIdx * chunkLen);
    }
    const int f0 = tileIdx * tile;
    const int nf = min(tile, F - f0);
    const int binsPerF = (T + 1) * C;
    const int nb = nf * binsPerF;
    const size_t plane = static_cast<size_t>(W) * H;
    for (int k = threadIdx.x; k < nb; k += kEvalThreads) h[k] = 0;
    __syncthreads();
    const FeatRec* fp = feat + static_cast<size_t>(ch.tree) * F + f0;
    const float* tp = thrPad + (static_cast<size_t>(ch.tree) * F + f0) * TM;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool shared = tile == kEvalTile;
    const int step = shared ? 64 : kEvalThreads, own = shared ? threadIdx.x & 63 : threadIdx.x;
    const int fBegin = shared ? wave * kEvalStep : 0, fEnd = shared ? min(nf, fBegin + kEvalStep) : nf;
    for (int base = 0; base < ch.count; base += step) {
        RegSample rs;
        const int i = base + own;
        rs.lab = -1;
        rs.img = 0;
        rs.xy = 0;
        rs.rinv = 0.0;
        if (i < ch.count) {
            const cf_sample s = samples[ch.begin + i];
            const bool valid = s.depth_mm > 0;
            rs.rinv = valid ? depthReciprocal(depthToFloat(s.depth_mm)) : 0.0;
            rs.img = static_cast<int>(s.image);
            rs.xy = s.x | (s.y << 16);
            rs.lab = s.label | (s.flip << 8) | ((valid ? 0 : 1) << 10);
        }
        const int2* dep = depBase + static_cast<size_t>(rs.img) * plane;
        const float* col = colBase + static_cast<size_t>(rs.img) * 3 * plane;
        const bool live = rs.lab >= 0, valid = live && (rs.lab >> 10) == 0;
        // orientation 0: the sample's own (Both: unflipped); 1: the flipped evaluation of Both samples
        auto evaluate = [&](bool on, bool flip) {
            for (int fi = fBegin; fi < fEnd; fi += kEvalStep) {
                Feat fr[kEvalStep];
                int2 cv[kEvalStep][8];   // depth corners, or colour corners' bits in .x
                bool ok[kEvalStep];
#pragma unroll
                for (int j = 0; j < kEvalStep; j++) {
                    // past a partial tile's end (uniform): the tile's last feature, not counted
                    fr[j] = loadFeat(fp + min(fi + j, nf - 1));
                    int idx[8];
                    ok[j] = on && valid && fi + j < nf &&
                            responseCorners(fr[j], rs.xy & 0xffff, rs.xy >> 16, W, H, rs.rinv, flip, idx);
                    if (ok[j]) {
                        if (fr[j].type == T_DEPTH) {
#pragma unroll
                            for (int c = 0; c < 8; c++) cv[j][c] = planeAt(dep, idx[c]);
                        } else {
                            const float* colA = col + static_cast<size_t>(fr[j].c1) * plane;
                            const float* colB = col + static_cast<size_t>(fr[j].c2) * plane;
#pragma unroll
                            for (int c = 0; c < 4; c++) cv[j][c].x = __float_as_int(planeAt(colA, idx[c]));
#pragma unroll
                            for (int c = 4; c < 8; c++) cv[j][c].x = __float_as_int(planeAt(colB, idx[c]));
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < kEvalStep; j++) {
                    if (fi + j >= nf) break;
                    float th[TM];
                    const float* tf = tp + static_cast<size_t>(fi + j) * TM;
#pragma unroll
                    for (int t = 0; t < TM; t++) th[t] = tf[t];
                    int b = T;
                    if (ok[j]) {
                        double r;
                        if (fr[j].type == T_DEPTH) {
                            r = depthResponseFromCorners(cv[j]);
                        } else {
                            float c8[8];
#pragma unroll
                            for (int c = 0; c < 8; c++) c8[c] = __int_as_float(cv[j][c].x);
                            r = colorResponseFromCorners(c8);
                        }
                        b = binOf<TM>(roundUpToFloat(r), th, T);
                    }
                    if (on) atomicAdd(&h[(fi + j) * binsPerF + b * C + (rs.lab & 0xff)], 1u);
                }
            }
        };
        evaluate(live, ((rs.lab >> 8) & 3) == 1);
        const bool both = live && ((rs.lab >> 8) & 3) == 2;
        if (__any(both)) evaluate(both, true);
    }
    __syncthreads();
    if (scoring.summ) {
        scoreFeatures(h, nf, F, T, C, scoring.hist, scoring.rank + (static_cast<size_t>(ch.tree) * F + f0) * T, evalLds,
                scoring.summ + f0, nullptr);
        return;
    }
    uint32_t* g = G + (static_cast<size_t>(ch.slot) * F + f0) * binsPerF;
    for (int k = threadIdx.x; k < nb; k += kEvalThreads) {
        const uint32_t v = h[k];
        if (v) atomicAdd(&g[k], v);
    }
}

template<int CM>
__device__ double nigScore(int C, const uint32_t* L, const uint32_t* R, const uint32_t* A) {
    double totalLeft = 0, totalRight = 0;
#pragma unroll
    for (int c = 0; c < CM; c++) {
        if (c < C) {
            totalLeft += static_cast<double>(L[c]);
            totalRight += static_cast<double>(R[c]);
        }
    }
    const double total = totalLeft + totalRight;
    const double leftProb = totalLeft / total;
    const double rightProb = totalRight / total;
    double score = 0;
#pragma unroll
    for (int c = 0; c < CM; c++) {
        if (c < C) {
            const uint32_t l = L[c], r = R[c];
            const double classProb = static_cast<double>(A[c]) / total;
            if (l > 0) {
                const double p = static_cast<double>(l) / total;
                score = __dadd_rn(score, __dmul_rn(p, log2(p / (leftProb * classProb))));
            }
            if (r > 0) {
                const double p = static_cast<double>(r) / total;
                score = __dadd_rn(score, __dmul_rn(p, log2(p / (rightProb * classProb))));
            }
        }
    }
    const double ig = clamp01(score);
    if (ig == 0) return 0;
    const double Hs = (entropyOf(totalLeft) + entropyOf(totalRight) - entropyOf(total)) / total;
    double Hc = 0;
#pragma unroll
    for (int c = 0; c < CM; c++) {
        if (c < C && A[c] > 0) Hc += entropyOf(static_cast<double>(A[c]));
    }
    Hc -= entropyOf(total);
    Hc /= total;
    return clamp01((2 * ig) / (Hs + Hc));
}

// Scores of a workgroup's features of one slot from their bins, which come into LDS in one run.  Bound by the
// double divisions and logarithms.  A thread per feature that walked its thresholds took 96 us for one node of
// 1000 features x 20 thresholds (now 10) and 866 us for 206 nodes x 4000 x 32 (now 709).
struct ScoreShape {
    int feats;      // features of a workgroup
    size_t lds;     // their bins (and prefix sums) and scoreFeatures' own
};
static ScoreShape scoreShape(int T, int C) {
    ScoreShape s;
    const int words = (T + 1) * C;
    s.feats = std::max(1, std::min({256 / T, 64, 8192 / words}));
    s.lds = scoreLdsBytes(s.feats, T, C) + static_cast<size_t>(s.feats) * words * sizeof(uint32_t);
    return s;
}

__global__ void __launch_bounds__(256) k_scores(const uint32_t* __restrict__ G, const uint32_t* __restrict__ nodeHist,
        const int* __restrict__ slotTree, const uint16_t* __restrict__ rank, int F, int T, int C, int feats, int blocks,
        int first, FeatSummary* __restrict__ summ, double* __restrict__ allScores, int onlySlot, int fOffset, int Fb,
        const int* __restrict__ listed, int listBase) {
    extern __shared__ double scoreLds[];
    uint32_t* pre = reinterpret_cast<uint32_t*>(scoreLds) + scoreLdsBytes(feats, T, C) / sizeof(uint32_t);   // [feats][T + 1][C]
    // G holds Fb features per slot starting at feature fOffset
    const int at = first + static_cast<int>(blockIdx.x) / blocks;
    const int slot = onlySlot >= 0 ? onlySlot : (listed ? listed[at] - listBase : at);
    const int j0 = (static_cast<int>(blockIdx.x) % blocks) * feats;
    const int nf = min(feats, min(Fb - j0, F - fOffset - j0));
    if (nf <= 0) return;
    const int tid = threadIdx.x, words = (T + 1) * C;
    const uint32_t* g = G + (static_cast<size_t>(slot) * Fb + j0) * words;
    for (int i = tid; i < nf * words; i += 256) pre[i] = g[i];
    __syncthreads();
    scoreFeatures(pre, nf, F, T, C, nodeHist + static_cast<size_t>(slot) * C,
            rank + (static_cast<size_t>(slotTree[slot]) * F + fOffset + j0) * T, scoreLds,
            summ + static_cast<size_t>(slot) * F + fOffset + j0,
            allScores ? allScores + (onlySlot >= 0 ? 0 : static_cast<size_t>(slot) * T * F) + fOffset + j0 : nullptr);
}

// scores[T][F] of one node straight from counters [F][T][C][2]
// (ImageFeatureEvaluation::calculateScores, random_tree_image.cpp:188-237).
template<int CM>
__global__ void __launch_bounds__(256) k_scores_counters(const uint32_t* __restrict__ counters,
        const uint32_t* __restrict__ hist, int F, int T, int C, double* __restrict__ scores) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= F * T) return;
    const int f = i / T, t = i % T;
    uint32_t L[CM], R[CM], A[CM];
#pragma unroll
    for (int c = 0; c < CM; c++) {
        const size_t k = ((static_cast<size_t>(f) * T + t) * C + c) * 2;
        L[c] = c < C ? counters[k] : 0u;
        R[c] = c < C ? counters[k + 1] : 0u;
        A[c] = c < C ? hist[c] : 0u;
    }
    scores[static_cast<size_t>(t) * F + f] = nigScore<CM>(C, L, R, A);
}

void launchScoresFromCounters(hipStream_t s, const uint32_t* counters, const uint32_t* hist, int F, int T, int C,
        double* scores) {
    const dim3 grid((F * T + 255) / 256);
    if (C <= 8) {
        hipLaunchKernelGGL(k_scores_counters<8>, grid, dim3(256), 0, s, counters, hist, F, T, C, scores);
    } else {
        hipLaunchKernelGGL(k_scores_counters<kMaxClasses>, grid, dim3(256), 0, s, counters, hist, F, T, C, scores);
    }
}

__device__ __forceinline__ double waveMax(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ long long waveMinLL(long long v) {
    for (int o = 32; o > 0; o >>= 1) {
        const long long u = __shfl_xor(v, o, 64);
        v = u < v ? u : v;
    }
    return v;
}

// One workgroup per node, one pass over its features' summaries: a lane keeps the largest of its scores, where the
// scan meets it first, and the largest below it; a node is flagged if any score lies within 1e-13 below its
// maximum.  Bound by latency (one wave and two passes per node took 7.3 us for 1000 features and 41 us for 200
// nodes of 4000; now 3.9 and 11).
constexpr int kReduceLanes = 256;
__global__ void __launch_bounds__(kReduceLanes) k_reduce(const FeatSummary* __restrict__ summ, int numSlots, int F,
        NodeBest* __restrict__ out) {
    constexpr int kWaves = kReduceLanes / 64;
    __shared__ double waveBest[kWaves];
    __shared__ long long waveKey[kWaves];
    __shared__ int waveBand[kWaves];
    const int slot = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const FeatSummary* s = summ + static_cast<size_t>(slot) * F;
    double best = -DBL_MAX, below = -DBL_MAX;
    long long key = 0x7fffffffffffffffll;
    for (int f = threadIdx.x; f < F; f += kReduceLanes) {
        const FeatSummary x = s[f];
        const long long k = static_cast<long long>(x.thresh) * F + f;
        if (x.best > best) {
            below = fmax(best, x.second);
            best = x.best;
            key = k;
        } else if (x.best == best) {
            key = k < key ? k : key;
            below = fmax(below, x.second);
        } else {
            below = fmax(below, x.best);
        }
    }
    const double m1 = waveMax(best);
    if (lane == 0) waveBest[wave] = m1;
    __syncthreads();
    double m = waveBest[0];
#pragma unroll
    for (int w = 1; w < kWaves; w++) m = fmax(m, waveBest[w]);
    const bool mine = best == m;
    const int band = __any((!mine && (m - best) < 1e-13) || (below > -DBL_MAX && below < m && (m - below) < 1e-13)) ? 1 : 0;
    const long long k1 = waveMinLL(mine ? key : 0x7fffffffffffffffll);
    if (lane == 0) {
        waveKey[wave] = k1;
        waveBand[wave] = band;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        long long first = waveKey[0];
        int flag = waveBand[0];
        for (int w = 1; w < kWaves; w++) {
            first = waveKey[w] < first ? waveKey[w] : first;
            flag |= waveBand[w];
        }
        NodeBest nb;
        nb.score = m;
        nb.thresh = static_cast<int>(first / F);
        nb.feat = static_cast<int>(first % F);
        nb.flag = flag;
        nb.pad = 0;
        out[slot] = nb;
    }
}

// The literal scan of random_tree_image.cpp:445-457 for one node.
// detail::isScoreBetter (random_tree.cpp:36-52) as used by the scan.
__device__ __forceinline__ bool scoreBetter(double best, double score) {
    if (__builtin_isnan(best)) return true;
    return !(fabs(score - best) < 1e-13) && (score > best);
}

// The scan of random_tree_image.cpp:445-457 for one node.  A score is taken only if it lies above all earlier
// ones: an earlier one was taken, or did not lie above the best of its time by 1e-13, and then neither does one
// that is not larger against a best that has only grown (rounding a difference keeps order).  The waves of the
// workgroup take a segment of the scan each and list its windows of 64 scores that hold one above all before it in
// the segment; the windows that the maxima of the earlier segments do not rule out, a dozen of some thousand, are
// then resolved in order with the reference's predicate.  A segment whose list is full is scanned whole.
// Bound by latency (one wave over all scores: 49 us for 500 x 50, 223 for 4000 x 32; now 16 and
// 31).
// Up to kSeqAlone scores one wave resolves all windows and lists none (a call on 1, 512, 1024, 2048, 5000 random
// scores takes 29, 34, 34, 37, 48 us with one wave, 31, 41, 39, 40, 46 with sixteen; ascending ones 29, 74, 120, 214,
// 490 and 31, 83, 136, 225, 479).
constexpr int kSeqWaves = 16, kSeqList = 64, kSeqAhead = 8, kSeqAlone = 48 * 64;
__global__ void __launch_bounds__(64 * kSeqWaves) k_seq_argmax(const double* __restrict__ allScores, int T, int F,
        NodeBest* __restrict__ allOut) {
    __shared__ int list[kSeqWaves][kSeqList], listed[kSeqWaves];   // windows of a segment, -1: all of them
    __shared__ double listMax[kSeqWaves][kSeqList], segMax[kSeqWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long n = static_cast<long long>(T) * F;
    // one node per workgroup: scores[T][F] and its result
    const double* scores = allScores + static_cast<size_t>(blockIdx.x) * n;
    const int waves = static_cast<int>(blockDim.x >> 6);   // 1 or kSeqWaves
    const int windows = static_cast<int>((n + 63) / 64), per = (windows + waves - 1) / waves;
    auto scoreAt = [&](int w) {
        const long long i = static_cast<long long>(w) * 64 + lane;
        return i < n ? scores[i] : -__builtin_inf();
    };
    if (waves == 1) {
        if (lane == 0) listed[0] = -1;
        __syncthreads();
    } else {
        const int first = min(wave * per, windows), end = min(first + per, windows);
        double run = -__builtin_inf();
        int count = 0;
        for (int w0 = first; w0 < end; w0 += kSeqAhead) {
            double sc[kSeqAhead];
#pragma unroll
            for (int u = 0; u < kSeqAhead; u++) sc[u] = w0 + u < end ? scoreAt(w0 + u) : -__builtin_inf();
#pragma unroll
            for (int u = 0; u < kSeqAhead; u++) {
                if (__any(sc[u] > run)) {
                    const double m = waveMax(sc[u]);
                    if (lane == 0 && count < kSeqList) {
                        list[wave][count] = w0 + u;
                        listMax[wave][count] = m;
                    }
                    count++;
                    run = fmax(run, m);
                }
            }
        }
        if (lane == 0) {
            segMax[wave] = run;
            listed[wave] = count;
        }
        __syncthreads();
        double before = -__builtin_inf();
        for (int w = 0; w < wave; w++) before = fmax(before, segMax[w]);
        if (count <= kSeqList) {
            const int w = lane < count ? list[wave][lane] : 0;
            const bool keep = lane < count && listMax[wave][lane] > before;
            const unsigned long long kept = __ballot(keep);
            if (keep) list[wave][__popcll(kept & ((1ull << lane) - 1ull))] = w;
            if (lane == 0) listed[wave] = __popcll(kept);
        } else if (lane == 0) {
            listed[wave] = -1;
        }
        __syncthreads();
    }
    if (wave != 0) return;
    double best = -__builtin_inf();
    long long pos = 0;
    for (int s = 0; s < waves; s++) {
        const int first = min(s * per, windows), end = min(first + per, windows);
        const int count = listed[s] < 0 ? end - first : listed[s];
        for (int k0 = 0; k0 < count; k0 += kSeqAhead) {
            int win[kSeqAhead];
            double sc[kSeqAhead];
#pragma unroll
            for (int u = 0; u < kSeqAhead; u++) {
                const int k = min(k0 + u, count - 1);
                win[u] = listed[s] < 0 ? first + k : list[s][k];
                sc[u] = k0 + u < count ? scoreAt(win[u]) : -__builtin_inf();
            }
#pragma unroll
            for (int u = 0; u < kSeqAhead; u++) {
                unsigned long long m = __ballot(scoreBetter(best, sc[u]));
                while (m) {
                    const int l = __ffsll(static_cast<long long>(m)) - 1;
                    const double c = __shfl(sc[u], l, 64);
                    if (scoreBetter(best, c)) {
                        best = c;
                        pos = static_cast<long long>(win[u]) * 64 + l;
                    }
                    m &= m - 1;
                }
            }
        }
    }
    if (lane == 0) {
        NodeBest nb;
        nb.score = best;
        nb.feat = static_cast<int>(pos % F);
        nb.thresh = static_cast<int>(pos / F);
        nb.flag = 0;
        nb.pad = 0;
        allOut[blockIdx.x] = nb;
    }
}

// counters[F][T][C][2] of one node (slot 0) from its bins: a workgroup's features come into LDS and become prefix
// sums there, then a lane writes a (threshold, class)'s two counters (a lane per threshold that summed its bins
// from memory: 20 us for 500 x 50 with 5 classes; now 5.8).
__global__ void __launch_bounds__(256) k_counters_from_bins(const uint32_t* __restrict__ G,
        const uint16_t* __restrict__ rank, int F, int T, int C, int feats, uint32_t* __restrict__ counters) {
    extern __shared__ uint32_t pre[];   // [feats][T + 1][C]
    const int f0 = blockIdx.x * feats, nf = min(feats, F - f0), words = (T + 1) * C;
    const uint32_t* g = G + static_cast<size_t>(f0) * words;
    for (int i = threadIdx.x; i < nf * words; i += 256) pre[i] = g[i];
    __syncthreads();
    for (int i = threadIdx.x; i < nf * C; i += 256) {
        uint32_t* row = pre + (i / C) * words + i % C;
        uint32_t run = 0;
#pragma unroll 8
        for (int b = 0; b <= T; b++) {
            run += row[b * C];
            row[b * C] = run;
        }
    }
    __syncthreads();
    uint2* out = reinterpret_cast<uint2*>(counters) + static_cast<size_t>(f0) * T * C;
    for (int i = threadIdx.x; i < nf * T * C; i += 256) {
        const int ft = i / C, c = i - ft * C, fi = ft / T;
        const uint32_t* p = pre + fi * words + c;
        const uint32_t left = p[rank[static_cast<size_t>(f0) * T + ft] * C];
        out[i] = make_uint2(left, p[T * C] - left);
    }
}

__global__ void __launch_bounds__(256) k_responses(const DevImage* __restrict__ imgs,
        const cf_sample* __restrict__ samples, int n, const FeatRec* __restrict__ feats, int F,
        double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * F) return;
    const int f = i / n, k = i % n;
    const cf_sample s = samples[k];
    out[i] = featureResponse(imgs[s.image], loadFeat(feats + f), s.x, s.y, s.depth_mm, s.flip == 1);
}

// response of sample i to feature i
__global__ void __launch_bounds__(256) k_responses_paired(const DevImage* __restrict__ imgs,
        const cf_sample* __restrict__ samples, int n, const FeatRec* __restrict__ feats, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const cf_sample s = samples[i];
    out[i] = featureResponse(imgs[s.image], loadFeat(feats + i), s.x, s.y, s.depth_mm, s.flip == 1);
}

// Chunks of at least 256 samples (one per lane) and at most 4096 (over which the zeroing and flushing of a
// workgroup's histograms no longer shows), of a size that in between
// gives 2048 to 4096 workgroups: 8 to 16 per CU.
int evalChunkSamples(size_t samples, int F) {
    const size_t tiles = (static_cast<size_t>(F) + kEvalTile - 1) / kEvalTile;
    int c = 256;
    while (c < 4096 && samples * tiles > static_cast<size_t>(c) * 4096) c *= 2;
    return c;
}

static void launchEval(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk* chunks,
        const Chunk& node, int chunkLen, int numChunks, const FeatTables& tabs, int C, uint32_t* G,
        const NodeScoring& scoring) {
    if (numChunks == 0) return;
    // under two workgroups per CU with full tiles: tiles of one step
    const int tile = static_cast<int64_t>(numChunks) * ((tabs.F + kEvalTile - 1) / kEvalTile) < 512 ? kEvalSmallTile : kEvalTile;
    const int tiles = (tabs.F + tile - 1) / tile;
    const size_t lds = static_cast<size_t>(tile) * (tabs.T + 1) * C * sizeof(uint32_t) +
            (scoring.summ ? scoreLdsBytes(tile, tabs.T, C) : 0);
    const int64_t blocks = (static_cast<int64_t>(numChunks) * tiles + kNumXcds - 1) / kNumXcds * kNumXcds;
    if (blocks > INT32_MAX) throw Error(CF_ERR_UNSUPPORTED, "too many samples in one evaluation launch");
    const dim3 grid(static_cast<unsigned>(blocks)), block(kEvalThreads);
    auto launch = [&](auto tm) {
        constexpr int TM = decltype(tm)::value;
        // the limit is that of a full tile, whatever the tile
        const size_t full = static_cast<size_t>(kEvalTile) * (tabs.T + 1) * C * sizeof(uint32_t);
        allowLds(reinterpret_cast<const void*>(&k_eval_hist<TM>), std::max(full, lds));
        hipLaunchKernelGGL(k_eval_hist<TM>, grid, block, lds, s, imgs.col, imgs.dep, imgs.W, imgs.H, samples, chunks, node,
                chunkLen, numChunks, tile, tiles, tabs.feat.get(), tabs.thrPad.get(), tabs.F, tabs.T, C, G, scoring);
    };
    switch (binThresholdWidth(tabs.T)) {
        case 8: launch(std::integral_constant<int, 8>{}); break;
        case 12: launch(std::integral_constant<int, 12>{}); break;
        case 16: launch(std::integral_constant<int, 16>{}); break;
        case 20: launch(std::integral_constant<int, 20>{}); break;
        case 24: launch(std::integral_constant<int, 24>{}); break;
        case 32: launch(std::integral_constant<int, 32>{}); break;
        case 64: launch(std::integral_constant<int, 64>{}); break;
        default: launch(std::integral_constant<int, kMaxThresholds>{}); break;
    }
}

void launchEvalHistograms(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk* chunks,
        int numChunks, const FeatTables& tabs, int C, uint32_t* G) {
    launchEval(s, imgs, samples, chunks, Chunk{}, 0, numChunks, tabs, C, G, NodeScoring{});
}

// A node of few samples is taken as one chunk and scored by the workgroups that count it: no histogram is cleared,
// added to and read again, and there is no second launch.  Where the line lies: 117 nodes of 8 frames, 1000 x 20, half
// of them below 256 samples, took 10.7 ms without, 10.4 up to 256, 10.2 up to 512, 1024 and 2048 (with more samples the
// single chunk leaves CUs idle for as long as the second launch takes).
constexpr int kScoredSamples = 512;
bool evalScoresNode(int count, int F, int T, int C) {
    const int tile = (F + kEvalTile - 1) / kEvalTile < 512 ? kEvalSmallTile : kEvalTile;
    return count <= kScoredSamples &&
            static_cast<size_t>(tile) * (T + 1) * C * sizeof(uint32_t) + scoreLdsBytes(tile, T, C) <= kScoreFusedLds;
}

void launchEvalNode(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk& node,
        const FeatTables& tabs, int C, uint32_t* G, const uint32_t* nodeHist, FeatSummary* summ) {
    const int chunkLen = summ ? std::max(node.count, 1) : evalChunkSamples(node.count, tabs.F);
    launchEval(s, imgs, samples, nullptr, node, chunkLen, (node.count + chunkLen - 1) / chunkLen, tabs, C, G,
            NodeScoring{nodeHist, tabs.rank.get(), summ});
}

void launchScores(hipStream_t s, const uint32_t* G, const uint32_t* nodeHist, const int* slotTree, int numSlots,
        const FeatTables& tabs, int C, FeatSummary* summ, double* allScores, int onlySlot, int fOffset, int Fb,
        const int* listed, int listBase) {
    if (Fb < 0) Fb = tabs.F;
    const int slots = onlySlot >= 0 ? 1 : numSlots;
    if (slots == 0 || Fb <= 0) return;
    const ScoreShape shape = scoreShape(tabs.T, C);
    const int blocks = (Fb + shape.feats - 1) / shape.feats;
    allowLds(reinterpret_cast<const void*>(&k_scores), shape.lds);
    const int most = std::max(1, static_cast<int>(kMaxLaunchBlocks / blocks));
    for (int i = 0; i < slots; i += most) {
        const int n = std::min(most, slots - i);
        hipLaunchKernelGGL(k_scores, dim3(static_cast<unsigned>(n) * blocks), dim3(256), shape.lds, s, G, nodeHist,
                slotTree, tabs.rank.get(), tabs.F, tabs.T, C, shape.feats, blocks, i, summ, allScores, onlySlot, fOffset,
                Fb, listed, listBase);
    }
}

void launchReduce(hipStream_t s, const FeatSummary* summ, int numSlots, int F, NodeBest* best) {
    if (numSlots == 0) return;
    hipLaunchKernelGGL(k_reduce, dim3(numSlots), dim3(kReduceLanes), 0, s, summ, numSlots, F, best);
}

void launchSequentialArgmax(hipStream_t s, const double* scores, int T, int F, NodeBest* best, int numNodes) {
    if (numNodes <= 0) return;
    const int waves = static_cast<int64_t>(T) * F <= kSeqAlone ? 1 : kSeqWaves;
    hipLaunchKernelGGL(k_seq_argmax, dim3(static_cast<unsigned>(numNodes)), dim3(64 * waves), 0, s, scores, T, F, best);
}

void launchCountersFromBins(hipStream_t s, const uint32_t* G, const FeatTables& tabs, int C, uint32_t* counters) {
    const int words = (tabs.T + 1) * C, feats = std::max(1, std::min(4, 8192 / words));
    const size_t lds = static_cast<size_t>(feats) * words * sizeof(uint32_t);
    hipLaunchKernelGGL(k_counters_from_bins, dim3((tabs.F + feats - 1) / feats), dim3(256), lds, s, G, tabs.rank.get(),
            tabs.F, tabs.T, C, feats, counters);
}

void launchResponses(hipStream_t s, const DevImage* imgs, const cf_sample* samples, int n, const FeatRec* feats,
        int F, double* out) {
    const int total = n * F;
    if (total == 0) return;
    hipLaunchKernelGGL(k_responses, dim3((total + 255) / 256), dim3(256), 0, s, imgs, samples, n, feats, F, out);
}

void launchResponsesPaired(hipStream_t s, const DevImage* imgs, const cf_sample* samples, int n, const FeatRec* feats,
        double* out) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_responses_paired, dim3((n + 255) / 256), dim3(256), 0, s, imgs, samples, n, feats, out);
}

}  // namespace cf
