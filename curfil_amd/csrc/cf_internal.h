// Internal host-side declarations: handles, device buffers, kernel launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "cf_common.h"

namespace cf {

// XCDs of an MI355X: the dispatcher sends workgroup i of a launch to XCD i % kNumXcds, each XCD with
// its own L2.
constexpr int kNumXcds = 8;

// Workgroups of 256 lanes in one launch over node histograms: a grid of 2^32 work-items or more is refused, and
// a histogram budget of 16 GiB (CURFIL_EVAL_BUDGET_MB) holds 2^32 words, so these launches loop or are cut above
// this number (the fill of the default budget's 2 GiB takes one pass).
constexpr unsigned kMaxLaunchBlocks = 1u << 21;

// Thrown inside the library, turned into a status at the C ABI.
struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define CF_HIP(call)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (call);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            throw ::cf::Error(CF_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_));          \
    } while (0)

// Owning device buffer.
template<class T>
class DevBuf {
public:
    DevBuf() = default;
    explicit DevBuf(size_t n) { resize(n); }
    ~DevBuf() { release(); }
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p_(o.p_), n_(o.n_), cap_(o.cap_) { o.p_ = nullptr; o.n_ = o.cap_ = 0; }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) {
            release();
            p_ = o.p_; n_ = o.n_; cap_ = o.cap_;
            o.p_ = nullptr; o.n_ = o.cap_ = 0;
        }
        return *this;
    }
    // grows (never shrinks) the allocation; contents are not preserved
    void resize(size_t n) {
        if (n > cap_) {
            release();
            if (n > 0) {
                hipError_t e = hipMalloc(reinterpret_cast<void**>(&p_), n * sizeof(T));
                if (e != hipSuccess) {
                    p_ = nullptr;
                    throw Error(e == hipErrorOutOfMemory ? CF_ERR_NOMEM : CF_ERR_HIP,
                            std::string("hipMalloc of ") + std::to_string(n * sizeof(T)) + " bytes: " +
                            hipGetErrorString(e));
                }
            }
            cap_ = n;
        }
        n_ = n;
    }
    void release() {
        if (p_) (void)hipFree(p_);
        p_ = nullptr;
        n_ = cap_ = 0;
    }
    T* get() const { return p_; }
    size_t size() const { return n_; }
    size_t bytes() const { return n_ * sizeof(T); }
    size_t capacityBytes() const { return cap_ * sizeof(T); }

private:
    T* p_ = nullptr;
    size_t n_ = 0, cap_ = 0;
};

// Owning page-locked host buffer.
class PinnedBuf {
public:
    PinnedBuf() = default;
    ~PinnedBuf() { release(); }
    PinnedBuf(const PinnedBuf&) = delete;
    PinnedBuf& operator=(const PinnedBuf&) = delete;
    // grows (never shrinks) the allocation; contents are not preserved
    uint8_t* resize(size_t n) {
        if (n > cap_) {
            release();
            CF_HIP(hipHostMalloc(reinterpret_cast<void**>(&p_), n, hipHostMallocDefault));
            cap_ = n;
        }
        return p_;
    }
    void release() {
        if (p_) (void)hipHostFree(p_);
        p_ = nullptr;
        cap_ = 0;
    }
    uint8_t* get() const { return p_; }
    size_t capacityBytes() const { return cap_; }

private:
    uint8_t* p_ = nullptr;
    size_t cap_ = 0;
};

struct TrainWorkspace;   // trainer.cpp
struct FeatTables;

// Uniform-size image set: image i's planes start at col + i*3*W*H and dep + i*W*H.
struct ImageSet {
    const float* col;
    const int2* dep;
    int W, H;
};

}  // namespace cf

struct cf_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    // batched prediction to host memory: one event per launch, whose results are copied while the next runs,
    // and one per copy into the page-locked staging (two halves) for outputs in pageable memory
    std::vector<hipEvent_t> launchDone, copyDone;
    void* hostStage = nullptr;
    size_t hostStageBytes = 0;
    std::string error;
    std::recursive_mutex mu;
    bool profiling = false;
    // scratch buffers reused across calls
    cf::DevBuf<uint8_t> scratch0, scratch1, scratch2;
    // device and page-locked memory of training calls, kept between them (bounded: trainer.cpp)
    std::shared_ptr<cf::TrainWorkspace> trainWorkspace;
    // feature tables of the calls on one node, kept between them up to 64 MiB (NodeTables, capi.cpp)
    std::shared_ptr<cf::FeatTables> nodeTables;
};

struct cf_images {
    cf_ctx* ctx = nullptr;
    int count = 0, W = 0, H = 0;
    cf::DevBuf<float> col;         // [count][3][H][W]
    cf::DevBuf<int2> dep;          // [count][H][W]
    cf::DevBuf<cf::DevImage> desc; // [count]
    std::vector<uint8_t> labels;   // host [count][H][W]
    std::vector<uint8_t> labelsSet;
    std::vector<int32_t> depthHost; // host raw depth mm [count][H][W] (pixel validity for sampling)
    std::vector<uint8_t> depthSet;
    cf::ImageSet set() const;
};

namespace cf {

// ---- launchers (implemented in the .hip files) ----
void launchIntegralU8(hipStream_t s, const uint8_t* rgb, const uint16_t* depth, int W, int H, uint32_t* tmp,
        float* col, int2* dep);
void launchIntegralF32(hipStream_t s, const float* color, const int32_t* depth, int W, int H, uint32_t* tmp,
        double* work, float* col, int2* dep);
// integral of a w x h image (srcCol [3][h][w], srcDep [h][w]) into a W x H slot, NaN / 0 outside
void launchIntegralPad(hipStream_t s, const float* srcCol, const int2* srcDep, int w, int h, int W, int H, float* col,
        int2* dep);

// Feature generation job of one (tree, level).
struct FeatGenJob {
    const cf_sample* samples; // the level's samples of this tree, frontier order
    int n;                    // number of samples
    int seed;                 // seed of the level's RandomSource
    int outOffset;            // feature slot offset (tree * F)
};

// A feature generation job's place in its candidates and its stream of sample-index draws (absolute draw
// numbers; draw i lies in slot i mod the ring's size).
struct WalkState {
    int head, tail;             // next draw of the walk, draws produced
    int recorded, steps;        // draws produced before the last production, and the steps of that
    int k, generated;           // next candidate, features generated
    int t, tries;               // thresholds found and tries left of a candidate that ran past its band
    int drawsDone, candsDone;   // draws used by the candidates that have ended
    int openDraws;              // draws used so far by the candidate that ran past its band
    int err, done;
    float guess;                // expected draws of a candidate before any has ended
};

// the sample behind a draw: depthReciprocal of its depth, x | y << 16, its image (-1: no valid depth)
struct DrawRec {
    double rinv;
    int xy;
    int image;
};

// Per-(tree, level) feature tables on the device, slot = tree * F + f.
struct FeatTables {
    DevBuf<FeatRec> feat;      // sorted features [trees*F]
    DevBuf<float> thrFT;       // thresholds feature-major [trees*F][T]
    DevBuf<float> thrTF;       // thresholds threshold-major [trees][T][F] (reference layout)
    DevBuf<uint16_t> rank;     // rank[tf*T + t] = #{k : thr[k] < thr[t]} within the feature
    DevBuf<float> thrPad;      // thresholds padded with +inf to binThresholdWidth(T), for the evaluation kernels [trees*F][width]
    DevBuf<int8_t> soa;        // [trees][11][F] (reference SoA layout)
    // candidate / unsorted staging
    DevBuf<FeatRec> cand;
    DevBuf<FeatRec> unsortedFeat;
    DevBuf<float> unsortedThr;
    DevBuf<int> unsortedKey;
    // the walk over the draws (k_features.hip)
    DevBuf<uint8_t> walkSpace;
    PinnedBuf walkHost;
    float meanDraws = 0;       // draws per candidate in the last generation (0: none yet)
    int trees = 0, F = 0, T = 0;

    template<class Fn>
    void each(Fn&& fn) {
        fn(feat); fn(thrFT); fn(thrTF); fn(rank); fn(thrPad); fn(soa); fn(cand); fn(unsortedFeat); fn(unsortedThr);
        fn(unsortedKey); fn(walkSpace); fn(walkHost);
    }
};

void launchFeatureGeneration(hipStream_t s, const ImageSet& imgs, const FeatGenJob* jobsDev, int numJobs,
        int F, int T, int boxRadius, int regionSize, int useDepth, FeatTables& tabs, bool referenceLayouts = false);
// thresholds given in reference layout [trees][T][F] + features SoA [trees][11][F] -> tables
void launchPrepareTables(hipStream_t s, int trees, int F, int T, FeatTables& tabs);

// Evaluation work item: a chunk of one node's samples.
constexpr int kChunk = 4096;   // samples of a batched level's chunks
struct Chunk {
    int slot;   // node slot within the launch batch
    int tree;   // tree index (feature table)
    int begin;  // first sample (index into the level sample array)
    int count;  // samples in this chunk
};

struct NodeBest {
    double score;
    int feat;     // sorted feature index
    int thresh;   // threshold index
    int flag;     // 1: near-tie band not clean -> sequential replay needed
    int pad;
};

struct FeatSummary {
    double best;   // max score over thresholds
    double second; // largest score strictly below best (-inf if none)
    int thresh;    // smallest threshold index reaching best
    int pad;
};

// histogram bins G[slot][F][T+1][C] (interval histograms) of the chunks' samples; evalChunkSamples: the chunk
// size for a launch over so many samples
int evalChunkSamples(size_t samples, int F);
void launchEvalHistograms(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk* chunks,
        int numChunks, const FeatTables& tabs, int C, uint32_t* G);
// the same for one node, its chunks of evalChunkSamples formed from the whole (node.slot 0).  With summ, for a node
// that evalScoresNode tells to be scored where it is counted: its features' summaries instead of its bins.
bool evalScoresNode(int count, int F, int T, int C);
void launchEvalNode(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk& node,
        const FeatTables& tabs, int C, uint32_t* G, const uint32_t* nodeHist = nullptr, FeatSummary* summ = nullptr);

// ---- two-pass level evaluation (k_bins.hip)
// LDS a workgroup may use on the current device (MI355X: 160 KB); kernels whose
// histograms need more than the default 64 KB opt in before launch
size_t deviceLdsLimit();
void allowLds(const void* kernel, size_t bytes);

constexpr int kBinGroup = 16;            // features per bin row (16 x 8-bit bins = one uint4 per sample)
constexpr int kMaxBinThresholds = 255;   // bins 0..T must fit in 8 bits
// a block of consecutive entries of the image-major permutation (at most a pass-1 workgroup's samples),
// all of one (tree, image)
struct BinBlock {
    int tree;
    int begin;   // first position in the permutation
    int count;
    int image;   // the image of every sample in the block
};
// keys ((image * keyMul + keyBase) << placeBits | the sample's place in the image, below levelPlaces, >> placeShift)
// and values (level index) of one tree's level segment;
// with flipN > 0 also the flipped evaluation of every Both sample at flipN + index (value |
// kFlipEntry), and segment absentKey for the other samples there
constexpr uint32_t kFlipEntry = 0x80000000u;
void launchLevelKeys(hipStream_t s, const cf_sample* samples, int begin, int n, uint32_t keyBase, uint32_t keyMul,
        uint32_t* keys, uint32_t* vals, int flipN, uint32_t absentKey, int placeBits, int placeShift, int H);
int levelPlaces(int W, int H);
// Bits of a place in the keys of so many segments, and in *shift the low bits that are dropped from the place:
// as many as the buckets have to be fewer than 2^26 (their counts are cleared and scanned at every level).
int levelPlaceBits(uint64_t segments, int places, int* shift);
// label per level index, bit 7 set for samples still set to Both (counted in both orientations)
void launchLevelLabels(hipStream_t s, const cf_sample* samples, int n, uint8_t* labels);
// Counting sort of the n level entries with a key below numSegs << placeBits (the others are not placed): out =
// their values in key order, starts[seg] = first position of segment seg (key >> placeBits) or -1 if it is
// empty, starts[numSegs] = the number of placed entries.  count and cursor hold levelSortBuckets entries,
// blockSum levelSortScanBlocks.
size_t levelSortBuckets(int numSegs, int placeBits);
// p[0 .. n) = v by a kernel (usable inside a captured graph, where memset nodes are avoided)
void launchFillU32(hipStream_t s, uint32_t* p, size_t n, uint32_t v);
size_t levelSortScanBlocks(int numSegs, int placeBits);
void levelCountingSort(hipStream_t s, const uint32_t* keys, const uint32_t* vals, int n, int numSegs, int placeBits,
        uint32_t* count, uint32_t* cursor, uint32_t* blockSum, uint32_t* out, int* starts);
// Work list of pass 1 for ngb feature groups, built on the device.  The items are ordered by image group
// (segment i: its blocks segFirst[i] .. + segCount[i], segPrefix[i] blocks before them), feature group and
// block; XCD x takes the x-th eighth of them, and workgroup w of the launch runs on XCD w % 8, so
// work[pos * 8 + x] is XCD x's item pos, (-1, 0) past the end.  buildWorkLength: entries of the list.
int buildWorkLength(int blocks, int ngb);
void launchBuildWork(hipStream_t s, const int* segFirst, const int* segCount, const int* segPrefix, int numSegs,
        int blocks, int ngb, int2* work);
// bins[g][level index] for the work items (block, g) of feature groups g0 + g;
// permutation entries with kFlipEntry are evaluated flipped into bins[flipOffset + g * N + index]
// with launch shape `shape` (evalShape): blocks of shape.lanes * shape.perLane samples
void launchEvalBins(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const uint32_t* perm,
        const BinBlock* blocks, const int2* work, int numWork, int g0,
        const FeatTables& tabs, int N, uint4* bins, size_t flipOffset, int shape);
// A launch shape of pass 1: lanes per workgroup, samples of its block per lane (the block holds
// lanes * perLane samples), features whose corner gathers are issued together, workgroups per CU (held
// by an LDS reservation).
struct EvalShape {
    int lanes, perLane, featPerStep, wgPerCu;
};
int numEvalShapes();
const EvalShape& evalShape(int i);
// Pass-1 shape tuner: the shape for a launch of threshold width TM at a level of `entries`
// permutation entries.  *measure asks the caller to time the launch and report it with
// evalTunerRecord.  CURFIL_EVAL_SHAPE=i pins shape i, CURFIL_TUNE=0 keeps shape 0,
// CURFIL_TUNE_FILE keeps the choices between runs.
int evalTunerChoose(int TM, size_t entries, bool* measure);
void evalTunerRecord(int TM, size_t entries, int shape, double ms, double responses);
// padded threshold width of the evaluation kernels for T thresholds
int binThresholdWidth(int T);
// G[slot][ng * 16][T + 1][C] from the bin rows of the chunks' samples
// (samples still set to Both also count their flipped row at flipOffset; the chunks' slots count from slotBase)
void launchHistBins(hipStream_t s, const uint4* bins, const uint8_t* labels, const Chunk* chunks, int numChunks,
        int slotBase, int g0, int ng, const FeatTables& tabs, int C, int N, uint32_t* G, size_t flipOffset,
        const uint32_t* nodeHist, FeatSummary* summ);
// Whether launchHistBins over so many chunks may score the nodes of a single chunk where it counts them (with the
// level's nodeHist and summ given, which start at slot 0; their G stays as it is)
bool histScoresNodes(int numChunks, int ng, int T, int C);
// clears the perSlot words of each listed slot in G, which starts at slotBase
void launchClearSlots(hipStream_t s, uint32_t* G, const int* slots, int numSlots, int slotBase, size_t perSlot);
// Scores and per-feature summaries of the slots' histograms.  With allScores, also every score:
// allScores[T][F] of slot onlySlot alone, or allScores[slot][T][F] of all slots (onlySlot < 0).  With `listed`, only
// the numSlots slots listed[i] - listBase.
void launchScores(hipStream_t s, const uint32_t* G, const uint32_t* nodeHist, const int* slotTree, int numSlots,
        const FeatTables& tabs, int C, FeatSummary* summ, double* allScores, int onlySlot, int fOffset = 0,
        int Fb = -1, const int* listed = nullptr, int listBase = 0);
void launchScoresFromCounters(hipStream_t s, const uint32_t* counters, const uint32_t* hist, int F, int T, int C,
        double* scores);
void launchReduce(hipStream_t s, const FeatSummary* summ, int numSlots, int F, NodeBest* best);
// The reference's sequential argmax of scores[node][T][F] into best[node], for numNodes nodes.
void launchSequentialArgmax(hipStream_t s, const double* scores, int T, int F, NodeBest* best, int numNodes = 1);
void launchCountersFromBins(hipStream_t s, const uint32_t* G, const FeatTables& tabs, int C, uint32_t* counters);
void launchResponses(hipStream_t s, const DevImage* imgs, const cf_sample* samples, int n, const FeatRec* feats,
        int F, double* out);
void launchResponsesPaired(hipStream_t s, const DevImage* imgs, const cf_sample* samples, int n, const FeatRec* feats,
        double* out);

// Partition
// the parts that a level's chunks are cut into, of partLen places each (the last may be shorter, or empty)
int partitionParts(int numChunks);
// the split records of the level's nodes from their argmax, every sample's direction, the left and right entries
// of every chunk's parts
void launchPartitionDirections(hipStream_t s, const ImageSet& imgs, const cf_sample* samples, const Chunk* chunks,
        int numChunks, int parts, int partLen, const NodeBest* best, const int* nodeTree, const FeatTables& tabs, int C,
        SplitRec* splits, uint8_t* dir, int2* partCounts, uint32_t* leftHist);
void launchPartitionScatter(hipStream_t s, const cf_sample* samples, const Chunk* chunks, int numChunks, int parts,
        int partLen, const uint8_t* dir, const int2* partCounts, const int2* dst, cf_sample* out);

// Prediction
//
// The split nodes of a forest, packed in 128-byte blocks (one cache line): a block holds a subtree of up to
// three split levels, its nodes at heap positions 0..6 (position p's children at 2p+1 and 2p+2).  Slots 0..6
// are node records {threshold bits, offsets o1x o1y o2x o2y, regions r1x r1y r2x r2y, type c1 c2 -} (signed
// bytes, as in FeatRec); slot 7 is the block's tail {first child block, first leaf, leaf mask, child-block
// mask | first exit position << 16}.  A child position q below the first exit position (7, or 1 / 3 for a
// tree's top block of one or two levels) holds a split of the block; at or past it, a child that is a
// split starts another block.  Bit q of the leaf mask marks a leaf child, numbered from the first leaf in
// position order; bit q of the child-block mask a child block, numbered from the first child block in
// position order.
struct NodeBlock {
    uint4 slot[8];
};
// doubles per posterior row of a packed forest: C rounded up to even, so rows are 16-byte aligned
__host__ __device__ constexpr int postStride(int C) { return (C + 1) & ~1; }
struct DevForest {
    const NodeBlock* blocks;    // all trees' blocks, each tree's breadth-first from its root block
    const double* post;         // [leaves][postStride(C)], a block's leaves together
    const int32_t* treeRoot;    // root block of each tree, or -(leaf index)-1 for a one-node tree
    int numTrees;
    int C;
};
// probs [frames][C][H][W] and labels [frames][H][W] may be null
void launchClassify(hipStream_t s, const DevImage* imgs, const int* frameIdx, int numFrames, int W, int H,
        const DevForest& forest, float* probs, uint8_t* labels);
// one frame of a serving batch: its integrals and its outputs ([C][H][W] posteriors, [H][W] labels)
// Frames of any sizes share a launch: job i classifies rows rowBegin .. rowEnd - 1 of its frame (its
// whole integral image is there) with the tiles firstTile .. (job i + 1's firstTile) - 1 of the launch,
// firstTile ascending from 0 in job order (set by planClassifyJobs).
struct FrameJob {
    DevImage im;
    float* probs;
    uint8_t* labels;
    int firstTile;
    int rowBegin, rowEnd;
    int pad;
};
// the shape of a launch over jobs: the tree-split kernel for few pixels, and the launch's tiles
struct ClassifyPlan {
    int splitWaves = 0;   // waves that share a tile's trees, 0: one thread per pixel
    int totalTiles = 0;
};
// chooses the shape by the jobs' pixels (the tree-split kernel up to splitMaxPixels) and sets their firstTile
// (host copies of the jobs)
ClassifyPlan planClassifyJobs(FrameJob* jobs, int numJobs, const DevForest& forest, double splitMaxPixels);
// the bound below which launches split the trees (CURFIL_CLASSIFY_SPLIT_MPIX or the default)
double classifySplitPixels();
void launchClassifyJobs(hipStream_t s, const FrameJob* jobs, int numJobs, const ClassifyPlan& plan,
        const DevForest& forest);

}  // namespace cf
