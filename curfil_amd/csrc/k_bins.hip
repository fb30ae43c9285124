// Two-pass split evaluation of a whole level (batched training):
//
//   k_eval_bins   pass 1, image-major: the level's samples ordered by
//                 (image, tree, place) are cut into blocks of <= 256 within
//                 each (image, tree) segment; one workgroup per
//                 (block, group of 16 features) computes every response's
//                 interval among the feature's thresholds (the bin used by the
//                 interval histograms) and stores the 16 bins of a sample as
//                 one 16-byte row, bins[group][level index].
//   k_hist_bins   pass 2, node-major: one workgroup per (part of a node
//                 chunk, group) streams the part's bin rows and labels into LDS
//                 interval histograms and adds them to the node's global bins.
//                 Nodes of a single chunk are scored from LDS there and then;
//                 only the others' bins go through memory to k_scores (50
//                 frames, 5 trees, 4000 x 32: 47 ms of clears, histograms and
//                 scores per training, 40 with this; 21 frames, 3 trees,
//                 2000 x 20: 5.25 and 4.7).
//
// Counting is order-independent, so the histograms equal those of the direct
// path (k_eval_hist), whose single kernel gathers the integrals in node order:
// at deep levels a node's samples come from every image and the gathers miss
// in L2.  In pass 1 a workgroup's samples come from one image, the
// workgroups of one XCD sweep one image (the segments of all trees, tree by
// tree within each feature group) for all feature groups of a batch before
// the next, and every tree visits its features in an order grouped by the
// integral planes they read (depth, then colour channel pairs), so the
// trees' workgroups of one feature group read the same planes of one image
// and an XCD's L2 holds them.
//
// Pass 1 is bound by the vector memory path (58 lines in flight per CU times the
// L2's latency of 152 cycles under this load; the L1 is stalled on them in 55% of
// the cycles), not by arithmetic or HBM; its lookups are not far behind (0.90 per
// CU and cycle).  What counts is lines fetched per response: 3.33 with samples
// ordered by row, 3.06 in strips, 2.77 with the waves of a workgroup on the same
// samples (21 frames, 3 trees, 2000 x 20, shape 0; 2.62 with shape 2).  Eight
// waves per CU, each lane with one sample's 8 corner loads in flight, beat
// configurations with more in flight: the blocks an XCD runs at once cover a few
// feature groups of a segment, the planes they read fit the XCD's L2 (0.4%
// misses) and requests return sooner.  The launch reserves LDS the kernel does
// not use to hold the CU at the shape's workgroups.
#include <algorithm>
#include <map>
#include <mutex>

#include "cf_score.h"

namespace cf {

namespace {

struct BinSample {
    double rinv;   // depthReciprocal(depth in metres)
    int xy;        // x | y << 16
    int lab;       // flip << 8 | (invalid depth) << 10 | (flip entry) << 12;  < 0: empty slot
};

// #{t : th[t] < q} over a row padded with +inf (never below q), T for NaN.
// One compare and one add-with-carry per threshold: the compare's lane mask is
// the carry-in of the count.
template<int TM>
__device__ __forceinline__ int binOfT(float q, const float (&th)[TM], int T) {
    uint32_t b = 0;
#pragma unroll
    for (int t = 0; t < TM; t++) b += (th[t] < q) ? 1u : 0u;
    return (q != q) ? T : static_cast<int>(b);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The 8 corners of one (sample, feature) response: depth corners as {sum, count}, colour corners'
// float bits in .x.  Returns false (and issues no load) when the sample has no valid depth or a box
// leaves the image.
__device__ __forceinline__ bool gatherCorners(const Feat& fr, const BinSample& rs, const float* col,
        const int2* dep, int W, int H, size_t plane, int2 (&cv)[8]) {
    const int lab = rs.lab;
    int idx[8];
    const bool ok = lab >= 0 && ((lab >> 10) & 1) == 0 &&
            responseCorners(fr, rs.xy & 0xffff, rs.xy >> 16, W, H, rs.rinv, ((lab >> 8) & 3) == 1, idx);
    if (ok) {
        if (fr.type == T_DEPTH) {
#pragma unroll
            for (int c = 0; c < 8; c++) cv[c] = planeAt(dep, idx[c]);
        } else {
            const float* colA = col + static_cast<size_t>(fr.c1) * plane;
            const float* colB = col + static_cast<size_t>(fr.c2) * plane;
#pragma unroll
            for (int c = 0; c < 4; c++) cv[c].x = __float_as_int(planeAt(colA, idx[c]));
#pragma unroll
            for (int c = 4; c < 8; c++) cv[c].x = __float_as_int(planeAt(colB, idx[c]));
        }
    }
    return ok;
}

template<int TM>
__device__ __forceinline__ uint32_t binFromCorners(const Feat& fr, bool ok, const int2 (&cv)[8],
        const float (&th)[TM], int T) {
    if (!ok) return static_cast<uint32_t>(T);
    double r;
    if (fr.type == T_DEPTH) {
        r = depthResponseFromCorners(cv);
    } else {
        float c8[8];
#pragma unroll
        for (int c = 0; c < 8; c++) c8[c] = __int_as_float(cv[c].x);
        r = colorResponseFromCorners(c8);
    }
    return static_cast<uint32_t>(binOfT<TM>(roundUpToFloat(r), th, T));
}

}  // namespace

// A workgroup's block in LDS: its samples, their bin rows in the making, their level indices.
constexpr int kBlockSampleBytes = sizeof(BinSample) + kBinGroup + sizeof(int);

// Pass 1 with the launch shape <WAVES waves, FPS features whose corner gathers are issued together>.  A workgroup
// covers one block of samples and a group of 16 features.  All its waves take the same 64 samples at a time,
// wave w the features w, w + WAVES, ... of the group: neighbouring features of the table read the same plane with
// nearly the same row offset, so the waves' corners fall on the same lines of a small patch, and a line that one
// wave brought into the L1 serves the others.  (Waves with samples of their own and the same feature share nothing:
// 3.06 lines a response in place of 2.77.)  A wave's features and thresholds are uniform and stay in scalar registers over the block.
template<int TM, int WAVES, int FPS>
__global__ void __launch_bounds__(WAVES * 64) k_eval_bins(const float* __restrict__ colBase,
        const int2* __restrict__ depBase, int W, int H, const cf_sample* __restrict__ samples,
        const uint32_t* __restrict__ perm, const BinBlock* __restrict__ blocks, const int2* __restrict__ work,
        int g0, const FeatRec* __restrict__ feat, const float* __restrict__ thrPad, int F, int T, int N,
        uint4* __restrict__ bins, size_t flipOffset, int blockMax) {
    constexpr int kPerWave = kBinGroup / WAVES;
    static_assert(kPerWave % FPS == 0, "features per step divide a wave's features");
    extern __shared__ uint4 blockLds[];
    BinSample* smp = reinterpret_cast<BinSample*>(blockLds);                  // [blockMax]
    uint8_t* rows = reinterpret_cast<uint8_t*>(smp + blockMax);               // [blockMax][16]
    int* outIdx = reinterpret_cast<int*>(rows + blockMax * kBinGroup);        // [blockMax]
    // work[blockIdx] = (sample block, feature group within the batch); the
    // XCDs' lists are interleaved (workgroup w runs on XCD w % 8) so each XCD
    // sweeps one image (the segments of all trees) for every group of the
    // batch before the next image.  Padding entries have a negative block.
    // Every XCD takes an eighth of the items, in order: an image whose groups
    // cross a boundary is read by two XCDs.  (Whole images per XCD left XCDs
    // idle unless the images divide by 8: 21 frames, 3 trees, 2000 x 20
    // took 7.5 ms a level against 6.5, 50 frames, 5 trees, 4000 x 32 59.8
    // against 52.3.)
    const int2 wk = work[blockIdx.x];
    if (wk.x < 0) return;
    const int g = wk.y;
    const BinBlock bb = blocks[wk.x];
    const size_t plane = static_cast<size_t>(W) * H;
    // all samples of a block belong to image bb.image: the plane bases are uniform
    const int2* dep = depBase + static_cast<size_t>(bb.image) * plane;
    const float* col = colBase + static_cast<size_t>(bb.image) * 3 * plane;

    const int count64 = (bb.count + 63) & ~63;
    for (int i = threadIdx.x; i < count64; i += WAVES * 64) {
        // empty lanes keep in-range fields (they issue no gathers)
        BinSample b{0.0, 0, -1};
        if (i < bb.count) {
            const uint32_t v = perm[bb.begin + i];
            const int s = static_cast<int>(v & ~kFlipEntry);
            const cf_sample x = samples[s];
            const bool valid = x.depth_mm > 0;
            // a flip entry evaluates a Both sample flipped; other entries in the sample's own
            // orientation (Both: unflipped); bit 12 selects the flipped bin rows
            const bool flipEntry = (v & kFlipEntry) != 0;
            outIdx[i] = s;
            b.rinv = valid ? depthReciprocal(depthToFloat(x.depth_mm)) : 0.0;
            b.xy = x.x | (x.y << 16);
            b.lab = ((flipEntry ? 1 : x.flip) << 8) | ((valid ? 0 : 1) << 10) | (flipEntry ? 1 << 12 : 0);
        }
        smp[i] = b;
    }
    __syncthreads();

    const int pos0 = (g0 + g) * kBinGroup;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), lane = threadIdx.x & 63;
    for (int f0 = 0; f0 < kPerWave; f0 += FPS) {
        Feat fr[FPS];
        float th[FPS][TM];
        int pos[FPS];
#pragma unroll
        for (int j = 0; j < FPS; j++) {
            pos[j] = wave + (f0 + j) * WAVES;
            // past the table's end (uniform): the last feature again, its bins are not read
            const size_t tp = static_cast<size_t>(bb.tree) * F + min(pos0 + pos[j], F - 1);
            fr[j] = loadFeat(feat + tp);
#pragma unroll
            for (int t = 0; t < TM; t++) th[j][t] = thrPad[tp * TM + t];
        }
        for (int base = 0; base < bb.count; base += 64) {
            const BinSample rs = smp[base + lane];
            int2 cv[FPS][8];
            bool ok[FPS];
            // the gathers of FPS features are all issued before any response is formed
#pragma unroll
            for (int j = 0; j < FPS; j++) ok[j] = gatherCorners(fr[j], rs, col, dep, W, H, plane, cv[j]);
#pragma unroll
            for (int j = 0; j < FPS; j++) {
                rows[(base + lane) * kBinGroup + pos[j]] =
                        static_cast<uint8_t>(binFromCorners<TM>(fr[j], ok[j], cv[j], th[j], T));
            }
        }
    }
    __syncthreads();
    uint4* out = bins + static_cast<size_t>(g) * N;
    uint4* outFlip = bins + flipOffset + static_cast<size_t>(g) * N;
    for (int i = threadIdx.x; i < bb.count; i += WAVES * 64) {
        // rows are read once, by pass 2: streaming stores keep them from evicting image planes from L2
        const u32x4 v = reinterpret_cast<const u32x4*>(rows)[i];
        uint4* o = (smp[i].lab & (1 << 12)) ? outFlip : out;
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(o + outIdx[i]));
    }
}

// What pass 2 needs to score the nodes of a single chunk where it counts them, by slot of the level: their class
// counts, the tables' ranks, their summaries (null: it does not).
struct LevelScoring {
    const uint32_t* hist;
    const uint16_t* rank;
    FeatSummary* summ;
};

// Pass 2: interval histograms of (part of a node chunk, feature group) from the bin rows.
// G holds the batch's groups: G[slot][ng * 16][T + 1][C].  Bound by the LDS atomics and the instructions that
// form their addresses: a lane takes four features of a sample in one word, 16 samples a wave, and its features in
// an order rotated by the sample, so that one LDS atomic instruction covers 4 samples of each of the 16
// features: their histograms lie in different banks and at most 4 lanes can hit one address (all lanes counting
// one feature, as for samples of an almost pure node, would collide on few bins).  Features past the table's last
// hold anything in the rows; they are counted into histograms that nothing reads.  With the scores of the
// small nodes (50 frames, 5 trees, 4000 x 32) the LDS works in half of the cycles, two thirds of them conflicts, a
// third on equal addresses (samples of one class in one bin).
// One feature of a sample a lane took a byte load and three times the instructions for each atomic, and a
// chunk was not cut into parts: 13 flipped frames, 500 x 50 108 us a level (now 36); 4 small frames 19 (5); 21
// frames, 3 trees, 2000 x 20 199 (151); 50 frames, 5 trees, 4000 x 32 1562 (1245).
__global__ void __launch_bounds__(256) k_hist_bins(const uint4* __restrict__ bins, const uint8_t* __restrict__ labels,
        const Chunk* __restrict__ chunks, int numChunks, int parts, int partLen, int slotBase, int g0, int ng, int F,
        int T, int C, int N, uint32_t* __restrict__ G, size_t flipOffset, LevelScoring scoring) {
    extern __shared__ double histLds[];   // scoreFeatures' part where nodes are scored, the bins
    uint32_t* h = reinterpret_cast<uint32_t*>(histLds) +
            (scoring.summ ? scoreLdsBytes(kBinGroup, T, C) / sizeof(uint32_t) : 0);
    const int partIdx = blockIdx.x / ng;
    const int g = blockIdx.x % ng;
    Chunk ch = chunks[partIdx / parts];
    const int from = partIdx % parts * partLen;
    ch.begin += from;
    ch.count = min(ch.count - from, partLen);
    if (ch.count <= 0) return;
    const int nf = min(kBinGroup, F - (g0 + g) * kBinGroup);
    const int binsPerF = (T + 1) * C;
    for (int k = threadIdx.x; k < kBinGroup * binsPerF; k += 256) h[k] = 0;
    __syncthreads();
    constexpr int kWords = kBinGroup / 4;   // words of a row, lanes of a sample
    const int word = threadIdx.x % kWords;
    const int sub = threadIdx.x / kWords;   // 64 samples per pass of the workgroup
    const size_t row0 = static_cast<size_t>(g) * N + ch.begin;
    const uint32_t* row = reinterpret_cast<const uint32_t*>(bins + row0) + word;
    const uint32_t* rowFlip = reinterpret_cast<const uint32_t*>(bins + flipOffset + row0) + word;
    const uint8_t* lab = labels + ch.begin;
    int shift[4];
    uint32_t* hf[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int byte = (k + sub) & 3;
        shift[k] = 8 * byte;
        hf[k] = h + (word * 4 + byte) * binsPerF;
    }
    // bins are 0..T; the clamp keeps the LDS index inside the histogram whatever a row holds
    auto count = [&](uint32_t v, int label) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int bin = min(static_cast<int>((v >> shift[k]) & 0xffu), T);
            atomicAdd(&hf[k][bin * C + label], 1u);
        }
    };
    constexpr int kUnroll = 8;   // words loaded ahead of their atomics
    constexpr int kPass = 256 / kWords;
    for (int base = 0; base < ch.count; base += kPass * kUnroll) {
        uint32_t v[kUnroll];
        int l[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const int i = base + u * kPass + sub;
            l[u] = -1;
            if (i < ch.count) {
                v[u] = row[static_cast<size_t>(i) * kWords];
                l[u] = lab[i];
            }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            if (l[u] >= 0) {
                count(v[u], l[u] & 0x7f);
                // still Both: its flipped evaluation counts too
                if (l[u] & 0x80) count(rowFlip[static_cast<size_t>(base + u * kPass + sub) * kWords], l[u] & 0x7f);
            }
        }
    }
    __syncthreads();
    const int chunk = partIdx / parts;
    if (scoring.summ && (chunk == 0 || chunks[chunk - 1].slot != ch.slot) &&
            (chunk == numChunks - 1 || chunks[chunk + 1].slot != ch.slot)) {
        const int f0 = (g0 + g) * kBinGroup;
        scoreFeatures(h, nf, F, T, C, scoring.hist + static_cast<size_t>(ch.slot) * C,
                scoring.rank + (static_cast<size_t>(ch.tree) * F + f0) * T, histLds,
                scoring.summ + static_cast<size_t>(ch.slot) * F + f0, nullptr);
        return;
    }
    uint32_t* out = G + (static_cast<size_t>(ch.slot - slotBase) * ng + g) * kBinGroup * binsPerF;
    for (int k = threadIdx.x; k < nf * binsPerF; k += 256) {
        const uint32_t v = h[k];
        if (v) atomicAdd(&out[k], v);
    }
}

// A sample's place within its (image, tree) segment: strips of kStripWidth columns, each top to bottom in steps
// of 4 rows.  The 64 consecutive samples of a wave (one in 77 pixels) then lie in a patch about as high as it
// is wide, and where their corners for a feature fall on one cache line the reads merge: 3.16 lines per response
// over a wave's 8 corners, against 3.51 for samples ordered by row and 3.14 for the best strips of single rows
// (80 to 128 columns; corner addresses of 4 frames of 640x480, offsets to 120, regions to 20).  Pass 1 takes as
// long as its L1 misses: 50 frames, 5 trees, 4000 x 32 987 -> 910 ms a training, 21 frames, 3 trees, 2000 x 20
// 108 -> 100 ms (3.33 -> 3.06 L2 requests per response).
constexpr int kStripWidth = 128, kStripRows = 4;

int levelPlaces(int W, int H) {
    return ((W + kStripWidth - 1) / kStripWidth) * ((H + kStripRows - 1) / kStripRows);
}

// Past 2^26 buckets a place loses low bits (steps of 8, 16 ... rows of a strip) rather than all of them: 50 frames of
// 640x480, 5 trees, 1000 x 32 take 131 ms of pass 1 with whole places, 132, 133, 136, 140 with 1, 2, 3, 4 bits
// dropped, 153 with 8, 163 with none kept.  Whole places fit 65534 (image, tree) segments of 640x480.
int levelPlaceBits(uint64_t segments, int places, int* shift) {
    constexpr uint64_t kMaxBuckets = 1ull << 26;
    int bits = 0;
    while ((1 << bits) < places) bits++;
    int kept = bits;
    while (kept > 0 && ((segments + 2) << kept) > kMaxBuckets) kept--;
    *shift = bits - kept;
    return kept;
}

// Sort keys (segment << placeBits | place) and values (level index) of one tree's level segment.
__global__ void __launch_bounds__(256) k_level_keys(const cf_sample* __restrict__ samples, int begin, int n,
        uint32_t keyBase, uint32_t keyMul, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals, int flipN,
        uint32_t absentKey, int placeBits, int placeShift, int stripPlaces) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const cf_sample x = samples[begin + i];
    const uint32_t place = placeBits > 0 ? ((x.x / kStripWidth) * stripPlaces + x.y / kStripRows) >> placeShift : 0u;
    const uint32_t seg = static_cast<uint32_t>(x.image) * keyMul + keyBase;
    keys[begin + i] = (seg << placeBits) | place;
    vals[begin + i] = static_cast<uint32_t>(begin + i);
    if (flipN > 0) {
        keys[flipN + begin + i] = x.flip == 2 ? ((seg << placeBits) | place) : (absentKey << placeBits);
        vals[flipN + begin + i] = static_cast<uint32_t>(begin + i) | kFlipEntry;
    }
}

// One thread per (XCD list position, XCD): item x * per + pos of the level's work in (image group, feature
// group, block) order; the image group by binary search over the block prefix counts.
__global__ void __launch_bounds__(256) k_build_work(const int* __restrict__ segFirst, const int* __restrict__ segCount,
        const int* __restrict__ segPrefix, int numSegs, int ngb, long long total, int per, int2* __restrict__ work) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<size_t>(per) * kNumXcds) return;
    const long long pos = static_cast<long long>(i % kNumXcds) * per + static_cast<long long>(i / kNumXcds);
    int2 item = make_int2(-1, 0);
    if (pos < total) {
        int lo = 0, hi = numSegs;   // the last segment with segPrefix * ngb <= pos
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (static_cast<long long>(segPrefix[mid]) * ngb <= pos) lo = mid;
            else hi = mid;
        }
        const long long local = pos - static_cast<long long>(segPrefix[lo]) * ngb;
        const int nb = segCount[lo];
        item = make_int2(segFirst[lo] + static_cast<int>(local % nb), static_cast<int>(local / nb));
    }
    work[i] = item;
}

__global__ void __launch_bounds__(256) k_level_labels(const cf_sample* __restrict__ samples, int n,
        uint8_t* __restrict__ labels) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) labels[i] = static_cast<uint8_t>(samples[i].label | (samples[i].flip == 2 ? 0x80 : 0));
}

size_t deviceLdsLimit() {
    static std::mutex mu;
    static std::map<int, size_t> limits;
    int dev = 0;
    CF_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> g(mu);
    auto it = limits.find(dev);
    if (it != limits.end()) return it->second;
    int v = 0;
    CF_HIP(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    return limits[dev] = static_cast<size_t>(v);
}

void allowLds(const void* kernel, size_t bytes) {
    if (bytes <= 64 * 1024) return;
    if (bytes > deviceLdsLimit()) {
        throw Error(CF_ERR_UNSUPPORTED, "(thresholds + 1) x classes too large for the LDS histograms of 16 features (" +
                std::to_string(bytes) + " bytes)");
    }
    CF_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
}

int binThresholdWidth(int T) {
    static const int widths[] = {8, 12, 16, 20, 24, 32, 64, kMaxThresholds};
    for (int w : widths) {
        if (T <= w) return w;
    }
    throw Error(CF_ERR_ARG, "too many thresholds (max 256)");
}

void launchLevelKeys(hipStream_t s, const cf_sample* samples, int begin, int n, uint32_t keyBase, uint32_t keyMul,
        uint32_t* keys, uint32_t* vals, int flipN, uint32_t absentKey, int placeBits, int placeShift, int H) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_level_keys, dim3((n + 255) / 256), dim3(256), 0, s, samples, begin, n, keyBase, keyMul, keys,
            vals, flipN, absentKey, placeBits, placeShift, (H + kStripRows - 1) / kStripRows);
}

int buildWorkLength(int blocks, int ngb) {
    const long long per = (static_cast<long long>(blocks) * ngb + kNumXcds - 1) / kNumXcds;
    if (per * kNumXcds > INT32_MAX) throw Error(CF_ERR_UNSUPPORTED, "too much work in one pass-1 launch");
    return static_cast<int>(per) * kNumXcds;
}

void launchBuildWork(hipStream_t s, const int* segFirst, const int* segCount, const int* segPrefix, int numSegs,
        int blocks, int ngb, int2* work) {
    const int n = buildWorkLength(blocks, ngb);
    if (n == 0) return;
    hipLaunchKernelGGL(k_build_work, dim3((n + 255) / 256), dim3(256), 0, s, segFirst, segCount, segPrefix, numSegs, ngb,
            static_cast<long long>(blocks) * ngb, n / kNumXcds, work);
}

void launchLevelLabels(hipStream_t s, const cf_sample* samples, int n, uint8_t* labels) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_level_labels, dim3((n + 255) / 256), dim3(256), 0, s, samples, n, labels);
}

// Launch shapes of pass 1 the tuner chooses from: {lanes, samples of a block per lane, features whose gathers
// are issued together, workgroups per CU}.  Shape 0 is the default.  Which is ahead turns on the threshold rows:
// with up to 32 thresholds the shapes of two workgroups, within 2% of each other, with more the compares count and
// the last two overlap them with the gathers.  Pass 1 of 70 frames, 5 trees, 1.4 million entries in this order, ms:
// 512 x 8 69.9, 68.6, 68.4, 72.5, 74.8; 512 x 32 70.1, 70.1, 70.9, 72.7, 75.0; 512 x 50 72.4, 76.0, 78.7, 73.0,
// 75.2 and flipped 133.0, 141.6, 145.6, 127.8, 130.4; 256 x 100 79.7, 84.6, 86.5, 69.5, 66.5.  (Levels below the
// tuner's smallest class run shape 0 whatever their rows.)
constexpr EvalShape kEvalShapes[] = {
    {256, 1, 1, 2},
    {256, 1, 2, 2},
    {256, 1, 4, 2},
    {256, 1, 1, 3},
    {256, 1, 1, 4},
};
constexpr int kNumEvalShapes = static_cast<int>(sizeof(kEvalShapes) / sizeof(kEvalShapes[0]));
static_assert(kNumEvalShapes <= 16, "TrainStats counts launches of at most 16 shapes");

int numEvalShapes() { return kNumEvalShapes; }

const EvalShape& evalShape(int i) {
    if (i < 0 || i >= kNumEvalShapes) throw Error(CF_ERR_ARG, "unknown pass-1 launch shape");
    return kEvalShapes[i];
}

// Dynamic LDS that k_eval_bins reserves (and does not use) so that exactly
// w workgroups fit a CU: more than 1 / (w + 1) and at most 1 / w of the CU's
// LDS; 64 KB where that lies inside (w = 2 on 160 KB CUs), else the middle of
// the interval.
static size_t evalBinsLdsBytes(int w) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, size_t> bytes;
    int dev = 0;
    CF_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> g(mu);
    auto it = bytes.find({dev, w});
    if (it != bytes.end()) return it->second;
    int perCu = 0;
    CF_HIP(hipDeviceGetAttribute(&perCu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev));
    const size_t lo = static_cast<size_t>(perCu) / (w + 1) + 1;
    const size_t hi = static_cast<size_t>(perCu) / w;
    size_t b = 64 * 1024;
    if (b < lo || b > hi) b = ((lo + hi) / 2) & ~static_cast<size_t>(255);
    return bytes[{dev, w}] = b;
}

template<int WAVES, int FPS>
static void launchEvalBinsShape(hipStream_t s, int TM, size_t lds, const ImageSet& imgs, const cf_sample* samples,
        const uint32_t* perm, const BinBlock* blocks, const int2* work, int numWork, int g0, const FeatTables& tabs,
        int N, uint4* bins, size_t flipOffset, int blockMax) {
    const dim3 grid(static_cast<unsigned>(numWork)), block(WAVES * 64);
#define CF_EVAL_BINS(TMV)                                                                                        \
    allowLds(reinterpret_cast<const void*>(&k_eval_bins<TMV, WAVES, FPS>), lds);                                 \
    hipLaunchKernelGGL((k_eval_bins<TMV, WAVES, FPS>), grid, block, lds, s, imgs.col, imgs.dep, imgs.W, imgs.H,  \
            samples, perm, blocks, work, g0, tabs.feat.get(), tabs.thrPad.get(), tabs.F, tabs.T, N, bins,         \
            flipOffset, blockMax)
    switch (TM) {
        case 8: CF_EVAL_BINS(8); break;
        case 12: CF_EVAL_BINS(12); break;
        case 16: CF_EVAL_BINS(16); break;
        case 20: CF_EVAL_BINS(20); break;
        case 24: CF_EVAL_BINS(24); break;
        case 32: CF_EVAL_BINS(32); break;
        case 64: CF_EVAL_BINS(64); break;
        default: CF_EVAL_BINS(kMaxThresholds); break;
    }
#undef CF_EVAL_BINS
}

void launchEvalBins(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const uint32_t* perm,
        const BinBlock* blocks, const int2* work, int numWork, int g0,
        const FeatTables& tabs, int N, uint4* bins, size_t flipOffset, int shape) {
    if (numWork == 0) return;
    const int TM = binThresholdWidth(tabs.T);
    const EvalShape& sh = evalShape(shape);
    const int blockMax = sh.lanes * sh.perLane;
    const size_t lds = std::max(evalBinsLdsBytes(sh.wgPerCu), static_cast<size_t>(blockMax) * kBlockSampleBytes);
#define CF_SHAPE(L, F)                                                                                            \
    if (sh.lanes == L && sh.featPerStep == F) {                                                                  \
        launchEvalBinsShape<L / 64, F>(s, TM, lds, imgs, samples, perm, blocks, work, numWork, g0, tabs, N, bins,  \
                flipOffset, blockMax);                                                                           \
        return;                                                                                                  \
    }
    CF_SHAPE(256, 1)
    CF_SHAPE(256, 2)
    CF_SHAPE(256, 4)
#undef CF_SHAPE
    throw Error(CF_ERR_RUNTIME, "pass-1 launch shape without a kernel");
}

// The histograms of the listed slots, cleared.
__global__ void __launch_bounds__(256) k_clear_slots(uint4* __restrict__ G, const int* __restrict__ slots, int slotBase,
        int words, int blocks) {
    uint4* g = G + static_cast<size_t>(slots[blockIdx.x / blocks] - slotBase) * words;
    const int i = static_cast<int>(blockIdx.x % blocks) * 256 + threadIdx.x;
    if (i < words) g[i] = make_uint4(0, 0, 0, 0);
}

void launchClearSlots(hipStream_t s, uint32_t* G, const int* slots, int numSlots, int slotBase, size_t perSlot) {
    if (numSlots == 0) return;
    const int words = static_cast<int>(perSlot / 4), blocks = (words + 255) / 256;
    const int most = std::max(1, static_cast<int>(kMaxLaunchBlocks / blocks));
    for (int i = 0; i < numSlots; i += most) {
        const int n = std::min(most, numSlots - i);
        hipLaunchKernelGGL(k_clear_slots, dim3(static_cast<unsigned>(blocks) * n), dim3(256), 0, s,
                reinterpret_cast<uint4*>(G), slots + i, slotBase, words, blocks);
    }
}

// few chunks and groups: chunks cut into parts while that gives at most 2048 workgroups
static int histParts(int numChunks, int ng) {
    int parts = 1;
    while (parts < 8 && static_cast<int64_t>(2) * parts * numChunks * ng <= 2048) parts *= 2;
    return parts;
}

bool histScoresNodes(int numChunks, int ng, int T, int C) {
    return histParts(numChunks, ng) == 1 &&
            static_cast<size_t>(kBinGroup) * (T + 1) * C * sizeof(uint32_t) + scoreLdsBytes(kBinGroup, T, C) <= kScoreFusedLds;
}

void launchHistBins(hipStream_t s, const uint4* bins, const uint8_t* labels, const Chunk* chunks, int numChunks,
        int slotBase, int g0, int ng, const FeatTables& tabs, int C, int N, uint32_t* G, size_t flipOffset,
        const uint32_t* nodeHist, FeatSummary* summ) {
    if (numChunks == 0 || ng == 0) return;
    const size_t bytes = static_cast<size_t>(kBinGroup) * (tabs.T + 1) * C * sizeof(uint32_t);
    const size_t lds = bytes + (summ ? scoreLdsBytes(kBinGroup, tabs.T, C) : 0);
    allowLds(reinterpret_cast<const void*>(&k_hist_bins), std::max(bytes, lds));
    const int parts = histParts(numChunks, ng), partLen = (kChunk + parts - 1) / parts;
    hipLaunchKernelGGL(k_hist_bins, dim3(static_cast<unsigned>(numChunks) * parts * ng), dim3(256), lds, s, bins, labels,
            chunks, numChunks, parts, partLen, slotBase, g0, ng, tabs.F, tabs.T, C, N, G, flipOffset,
            LevelScoring{nodeHist, tabs.rank.get(), summ});
}

}  // namespace cf
