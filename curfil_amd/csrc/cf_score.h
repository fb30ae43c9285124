// Scores of features whose class counts per threshold interval lie in LDS: the shared end of the kernels that
// score (k_scores, and k_eval_hist and k_hist_bins for nodes that one workgroup counts completely).
#pragma once

#include <cfloat>

#include "cf_internal.h"

namespace cf {

// NormalizedInformationGainScore::calculateScore (score.h:191-215) over
// InformationGainScore::calculateScore (score.h:87-139); the operation order
// follows the reference so host and device round identically apart from log2.
__device__ __forceinline__ double entropyOf(double p) {
    if (p == 0.0) return 0.0;
    return -p * log2(p);
}
__device__ __forceinline__ double clamp01(double s) {
    if (s > 1.0) return 1.0;
    if (s < 0.0) return 0.0;
    return s;
}

// nigScore of the split that sends L[c] of the node's A[c] samples left, with the terms that the node's
// thresholds share: classProb[c] = A[c] / total, entropyOf(total) and Hc.  The totals are integers, exact in
// double however they are summed.  A caller's class counts below the bins' wrap as nigScore's do.
__device__ __forceinline__ double splitScore(int C, const uint32_t* L, const uint32_t* A, const double* classProb,
        double totalEntropy, double classEntropy) {
    double totalLeft = 0, totalRight = 0, total = 0;
    for (int c = 0; c < C; c++) {
        totalLeft += static_cast<double>(L[c]);
        totalRight += static_cast<double>(A[c] - L[c]);
        total += static_cast<double>(A[c]);
    }
    const bool wraps = totalLeft + totalRight != total;
    total = totalLeft + totalRight;
    const double leftProb = totalLeft / total;
    const double rightProb = totalRight / total;
    double score = 0;
    for (int c = 0; c < C; c++) {
        const uint32_t l = L[c], r = A[c] - l;
        const double prob = wraps ? static_cast<double>(A[c]) / total : classProb[c];
        if (l > 0) {
            const double p = static_cast<double>(l) / total;
            score = __dadd_rn(score, __dmul_rn(p, log2(p / (leftProb * prob))));
        }
        if (r > 0) {
            const double p = static_cast<double>(r) / total;
            score = __dadd_rn(score, __dmul_rn(p, log2(p / (rightProb * prob))));
        }
    }
    const double ig = clamp01(score);
    if (ig == 0) return 0;
    double Ht = totalEntropy, Hc = classEntropy;
    if (wraps) {
        Ht = entropyOf(total);
        Hc = 0;
        for (int c = 0; c < C; c++) {
            if (A[c] > 0) Hc += entropyOf(static_cast<double>(A[c]));
        }
        Hc -= Ht;
        Hc /= total;
    }
    const double Hs = (entropyOf(totalLeft) + entropyOf(totalRight) - Ht) / total;
    return clamp01((2 * ig) / (Hs + Hc));
}

// LDS that scoreFeatures takes beside the bins, at their front: the scores [nf][T], the class probabilities [C],
// entropyOf(total) and Hc, the node's class counts [C].
__host__ __device__ __forceinline__ size_t scoreLdsBytes(int nf, int T, int C) {
    return (static_cast<size_t>(nf) * T + C + 2) * sizeof(double) + static_cast<size_t>((C + 1) / 2 * 2) * sizeof(uint32_t);
}
// A workgroup that counts a node completely scores it too while that takes no more LDS than this (four
// workgroups of 40 KiB fill a CU's).
constexpr size_t kScoreFusedLds = 40 * 1024;

// Scores and summaries of nf features, by a workgroup of at least 64 lanes, a lane per (feature, threshold).  `pre`
// holds the features' bins [nf][T + 1][C], all written before a barrier; they become prefix sums, so that threshold
// t's left counts are row rank[t].  allScores (may be null): the features' scores, [T] rows of F apart.
// What all thresholds of a node share (the class probabilities, the entropies of the classes and of the total, 7
// of 19 logarithms with 5 classes) is formed once per workgroup, by the same operations as nigScore.
__device__ __forceinline__ void scoreFeatures(uint32_t* pre, int nf, int F, int T, int C,
        const uint32_t* __restrict__ nodeHist, const uint16_t* __restrict__ rank, double* lds,
        FeatSummary* __restrict__ summ, double* __restrict__ allScores) {
    double* scores = lds;                         // [nf][T]
    double* classProb = scores + nf * T;          // [C]
    double* terms = classProb + C;                // entropyOf(total), Hc
    uint32_t* A = reinterpret_cast<uint32_t*>(terms + 2);   // [C]
    const int tid = threadIdx.x, lanes = blockDim.x, words = (T + 1) * C;
    if (tid < 64) {
        // total of the node, exact in double; lane c: class c, lane C: the total
        double total = 0;
        for (int c = 0; c < C; c++) total += static_cast<double>(nodeHist[c]);
        const uint32_t a = tid < C ? nodeHist[tid] : 0u;
        const double e = entropyOf(tid < C ? static_cast<double>(a) : total);
        if (tid < C) {
            A[tid] = a;
            classProb[tid] = static_cast<double>(a) / total;
        }
        double Hc = 0;
        for (int c = 0; c < C; c++) {
            const double ec = __shfl(e, c, 64);
            if (__shfl(a, c, 64) > 0u) Hc += ec;
        }
        const double et = __shfl(e, C, 64);
        Hc -= et;
        if (tid == 0) {
            terms[0] = et;
            terms[1] = Hc / total;
        }
    }
    for (int i = tid; i < nf * C; i += lanes) {
        uint32_t* row = pre + (i / C) * words + i % C;
        uint32_t run = 0;
#pragma unroll 8
        for (int b = 0; b <= T; b++) {
            run += row[b * C];
            row[b * C] = run;
        }
    }
    __syncthreads();
    for (int i = tid; i < nf * T; i += lanes) {
        const int fi = i / T, t = i - fi * T;
        const uint32_t* left = pre + fi * words + rank[i] * C;
        const double sc = splitScore(C, left, A, classProb, terms[0], terms[1]);
        scores[i] = sc;
        if (allScores) allScores[static_cast<size_t>(t) * F + fi] = sc;
    }
    __syncthreads();
    if (tid < nf) {
        double best = -DBL_MAX, second = -DBL_MAX;
        int bestT = 0x7fffffff;
        for (int t = 0; t < T; t++) {
            const double sc = scores[tid * T + t];
            if (sc > best) {
                second = best;
                best = sc;
                bestT = t;
            } else if (sc < best && sc > second) {
                second = sc;
            }
        }
        FeatSummary s;
        s.best = best;
        s.second = second;
        s.thresh = bestT;
        s.pad = 0;
        summ[tid] = s;
    }
}

}  // namespace cf
