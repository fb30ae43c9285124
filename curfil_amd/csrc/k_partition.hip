// Stable partition of every split node's samples into its children
// (RandomTreeTrain::train, random_tree.h:1295-1360: a sample goes LEFT iff its
// response is <= the split threshold, children keep the parent's order).
//
// Horizontal flipping (SplitFunction::split, random_tree.h:122-144): a sample
// with flip setting Both whose flipped response falls on the other side is
// split in two: the sample itself, now NoFlip, goes to its side, and a Flip
// copy goes to the other side, at the same position in that child's order.
// So every sample gives at most one entry to each child; an entry weighs 2 in
// the child's histogram iff it is still Both.
//
//   k_part_dir      per chunk: the entries of each sample (bit 0: the sample
//                   goes left, bit 1: it is split), the chunk's left and right
//                   entry counts and the node's left class histogram; the
//                   node's split record
//   k_part_scatter  per chunk: order-preserving compaction of left and right
//                   entries to the destinations the host assigned (children
//                   that stop growing get no destination)
#include "cf_internal.h"

namespace cf {

// A workgroup takes one of the `parts` equal parts of a chunk's places, so that the few chunks of an upper level
// (4096 samples each) spread over the chip: the corner gathers are cache misses nearly all, and a CU looks up
// one line a cycle (a level of 13 flipped frames: 42 us with a workgroup per
// chunk, 14 in parts; of 21 frames and 3 trees, where the lines come from HBM, 52 and 28).
int partitionParts(int numChunks) {
    int parts = 1;
    while (parts < 8 && 2 * parts * numChunks <= 1024) parts *= 2;
    return parts;
}

// The directions of a part of a chunk.  A lane has the gathers of two samples out together; the class and child
// counts come from ballots.  The node's split record is formed here from its argmax (feature of the sorted
// table, threshold index) and written by the first part of its first chunk.
constexpr int kDirLanes = 256, kDirAhead = 2;
__global__ void __launch_bounds__(kDirLanes) k_part_dir(ImageSet imgs, const cf_sample* __restrict__ samples,
        const Chunk* __restrict__ chunks, const NodeBest* __restrict__ best, const int* __restrict__ nodeTree,
        const FeatRec* __restrict__ feat, const float* __restrict__ thrFT, int F, int T, int C, int parts,
        int partLen, SplitRec* __restrict__ splits, uint8_t* __restrict__ dir, int2* __restrict__ partCounts,
        uint32_t* __restrict__ leftHist) {
    __shared__ uint32_t hist[kMaxClasses];
    __shared__ int totalL, totalR;
    const int chunk = static_cast<int>(blockIdx.x) / parts, part = static_cast<int>(blockIdx.x) - chunk * parts;
    Chunk ch = chunks[chunk];
    ch.begin += part * partLen;
    ch.count = min(ch.count - part * partLen, partLen);
    if (ch.count <= 0) {
        if (threadIdx.x == 0) partCounts[blockIdx.x] = make_int2(0, 0);
        return;
    }
    const NodeBest nb = best[ch.slot];
    const size_t tf = static_cast<size_t>(nodeTree[ch.slot]) * F + nb.feat;
    const float threshold = thrFT[tf * T + nb.thresh];
    const Feat f = loadFeat(feat + tf);
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < kMaxClasses) hist[tid] = 0;
    if (tid == 0) {
        totalL = 0;
        totalR = 0;
        if (part == 0 && (chunk == 0 || chunks[chunk - 1].slot != ch.slot)) {
            SplitRec sr;
            sr.feat = feat[tf];
            sr.threshold = threshold;
            sr.flags = 0;
            sr.pad0 = sr.pad1 = 0;
            splits[ch.slot] = sr;
        }
    }
    __syncthreads();
    const double thr = static_cast<double>(threshold);
    const size_t plane = static_cast<size_t>(imgs.W) * imgs.H;
    // whether each sample's response is at most the threshold (NaN is not); flipped for samples of setting Flip,
    // or for all
    auto goesLeft = [&](const cf_sample (&smp)[kDirAhead], bool flipAll, bool (&left)[kDirAhead]) {
        int idx[kDirAhead][8];
        bool ok[kDirAhead];
#pragma unroll
        for (int u = 0; u < kDirAhead; u++) {
            const cf_sample& s = smp[u];
            ok[u] = s.depth_mm > 0;
            const double rinv = depthReciprocal(depthToFloat(ok[u] ? s.depth_mm : 1000));
            const bool inside = responseCorners(f, s.x, s.y, imgs.W, imgs.H, rinv,
                    flipAll || s.flip == 1, idx[u]);
            ok[u] = ok[u] && inside;
#pragma unroll
            for (int e = 0; e < 8; e++) idx[u][e] = ok[u] ? idx[u][e] : 0;
        }
        if (f.type == T_DEPTH) {
            int2 cv[kDirAhead][8];
#pragma unroll
            for (int u = 0; u < kDirAhead; u++) {
                const int2* dep = imgs.dep + static_cast<size_t>(smp[u].image) * plane;
#pragma unroll
                for (int e = 0; e < 8; e++) cv[u][e] = dep[idx[u][e]];
            }
#pragma unroll
            for (int u = 0; u < kDirAhead; u++) left[u] = ok[u] && depthResponseFromCorners(cv[u]) <= thr;
        } else {
            float cv[kDirAhead][8];
#pragma unroll
            for (int u = 0; u < kDirAhead; u++) {
                const float* col = imgs.col + static_cast<size_t>(smp[u].image) * 3 * plane;
#pragma unroll
                for (int e = 0; e < 8; e++) cv[u][e] = (col + static_cast<size_t>(e < 4 ? f.c1 : f.c2) * plane)[idx[u][e]];
            }
#pragma unroll
            for (int u = 0; u < kDirAhead; u++) left[u] = ok[u] && colorResponseFromCorners(cv[u]) <= thr;
        }
    };
    int cntL = 0, cntR = 0;     // of the wave
    uint32_t classCount = 0;    // lane c: the wave's weight of class c
    for (int base = 0; base < ch.count; base += kDirLanes * kDirAhead) {
        if (base + (tid & ~63) >= ch.count) break;   // none of the wave's samples
        cf_sample smp[kDirAhead];
        bool left[kDirAhead], flipped[kDirAhead];
        bool both = false;
#pragma unroll
        for (int u = 0; u < kDirAhead; u++) {
            smp[u] = samples[ch.begin + min(base + u * kDirLanes + tid, ch.count - 1)];
            both = both || smp[u].flip == 2;
        }
        goesLeft(smp, false, left);
#pragma unroll
        for (int u = 0; u < kDirAhead; u++) flipped[u] = left[u];
        if (__any(both)) goesLeft(smp, true, flipped);
#pragma unroll
        for (int u = 0; u < kDirAhead; u++) {
            const int i = base + u * kDirLanes + tid;
            const bool in = i < ch.count;
            const bool goes = left[u], split = smp[u].flip == 2 && flipped[u] != goes;
            if (in) dir[ch.begin + i] = static_cast<uint8_t>((goes ? 1 : 0) | (split ? 2 : 0));
            cntL += __popcll(__ballot(in && (goes || split)));
            cntR += __popcll(__ballot(in && (!goes || split)));
            // left entry: the sample (weight 2 if still Both) or its Flip copy (weight 1)
            const uint32_t wL = !in ? 0u : (split ? 1u : (goes ? (smp[u].flip == 2 ? 2u : 1u) : 0u));
            for (int c = 0; c < C; c++) {
                const int n = __popcll(__ballot(wL != 0 && smp[u].label == c)) +
                        __popcll(__ballot(wL == 2 && smp[u].label == c));
                if (lane == c) classCount += static_cast<uint32_t>(n);
            }
        }
    }
    if (lane == 0) {
        atomicAdd(&totalL, cntL);
        atomicAdd(&totalR, cntR);
    }
    if (lane < C && classCount) atomicAdd(&hist[lane], classCount);
    __syncthreads();
    if (tid == 0) partCounts[blockIdx.x] = make_int2(totalL, totalR);
    if (tid < C && hist[tid]) atomicAdd(&leftHist[static_cast<size_t>(ch.slot) * C + tid], hist[tid]);
}

__global__ void __launch_bounds__(256) k_part_scatter(const cf_sample* __restrict__ samples,
        const Chunk* __restrict__ chunks, const uint8_t* __restrict__ dir, const int2* __restrict__ partCounts,
        int parts, int partLen, const int2* __restrict__ dst, cf_sample* __restrict__ out) {
    __shared__ int waveL[4], waveR[4];
    const int chunk = static_cast<int>(blockIdx.x) / parts, part = static_cast<int>(blockIdx.x) - chunk * parts;
    Chunk ch = chunks[chunk];
    ch.begin += part * partLen;
    ch.count = min(ch.count - part * partLen, partLen);
    if (ch.count <= 0) return;
    const int2 d = dst[chunk];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    int doneL = 0, doneR = 0;   // entries of the chunk's earlier parts, then of this part's earlier samples
    for (int q = 0; q < part; q++) {
        const int2 c = partCounts[chunk * parts + q];
        doneL += c.x;
        doneR += c.y;
    }
    for (int base = 0; base < ch.count; base += 256) {
        const int i = base + threadIdx.x;
        const bool valid = i < ch.count;
        const uint8_t dr = valid ? dir[ch.begin + i] : 0;
        const bool left = dr & 1, split = dr & 2;
        const bool hasL = valid && (left || split);
        const bool hasR = valid && (!left || split);
        const unsigned long long mL = __ballot(hasL), mR = __ballot(hasR);
        if (lane == 0) {
            waveL[wave] = __popcll(mL);
            waveR[wave] = __popcll(mR);
        }
        __syncthreads();
        int preL = __popcll(mL & below), preR = __popcll(mR & below), totL = 0, totR = 0;
        for (int w = 0; w < 4; w++) {
            if (w < wave) {
                preL += waveL[w];
                preR += waveR[w];
            }
            totL += waveL[w];
            totR += waveR[w];
        }
        if (valid) {
            const cf_sample s = samples[ch.begin + i];
            if (hasL && d.x >= 0) {
                cf_sample e = s;
                if (split) e.flip = left ? 0 : 1;   // the sample itself (NoFlip) or its Flip copy
                out[d.x + doneL + preL] = e;
            }
            if (hasR && d.y >= 0) {
                cf_sample e = s;
                if (split) e.flip = left ? 1 : 0;
                out[d.y + doneR + preR] = e;
            }
        }
        doneL += totL;
        doneR += totR;
        __syncthreads();
    }
}

void launchPartitionDirections(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk* chunks,
        int numChunks, int parts, int partLen, const NodeBest* best, const int* nodeTree, const FeatTables& tabs, int C,
        SplitRec* splits, uint8_t* dir, int2* partCounts, uint32_t* leftHist) {
    if (numChunks == 0) return;
    hipLaunchKernelGGL(k_part_dir, dim3(static_cast<unsigned>(numChunks) * parts), dim3(kDirLanes), 0, s, imgs, samples,
            chunks, best, nodeTree, tabs.feat.get(), tabs.thrFT.get(), tabs.F, tabs.T, C, parts, partLen, splits, dir,
            partCounts, leftHist);
}

void launchPartitionScatter(hipStream_t s, const cf_sample* samples, const Chunk* chunks, int numChunks, int parts,
        int partLen, const uint8_t* dir, const int2* partCounts, const int2* dst, cf_sample* out) {
    if (numChunks == 0) return;
    hipLaunchKernelGGL(k_part_scatter, dim3(static_cast<unsigned>(numChunks) * parts), dim3(256), 0, s, samples, chunks,
            dir, partCounts, parts, partLen, dst, out);
}

}  // namespace cf
