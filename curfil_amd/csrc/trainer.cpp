// Level-wise training driver (host side of the hot path).
//
// Semantics follow RandomTreeTrain::train (random_tree.h:1249-1415) and
// ImageFeatureEvaluation::evaluateBestSplits (random_tree_image.cpp:239-502):
//   * the root is level 1; a level equal to maxDepth is not evaluated;
//   * one seed per (tree, level) from the tree's RandomSource, one feature
//     table per (tree, level) generated from all of the level's samples in
//     frontier order;
//   * children ids are ++idNode (left, right), rolled back by 2 when a side is
//     empty (the node stays a leaf);
//   * a child keeps growing iff its histogram is not pure and it holds at
//     least minSampleCount samples;
//   * with horizontal flipping, samples set to Both count twice in the
//     histograms and are evaluated in both orientations; a Both sample that the
//     split separates from its flipped self continues as NoFlip plus a Flip
//     copy on the other side (random_tree.h:1295-1360).
// The device keeps the level's samples contiguous per node; evaluation runs
// either node by node (CF_MODE_PLAIN, the reference GPU path's shape: one
// launch sequence and one host sync per node) or for every node of every
// tree of the level together (CF_MODE_BATCHED).
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>

#include "cf_host.h"

namespace cf {

namespace {

struct ActiveTree {
    int job;                  // index into jobs / out
    int idNode;               // last assigned node id
    std::vector<int> nodes;   // frontier: node indices into out[job].nodes
    std::vector<int> counts;  // samples per frontier node
    int begin = 0, n = 0;     // segment of the level buffer
};

// The pass-1 blocks of one block size at the current level, and the work list of a batch size.
struct BlockSet {
    int level = -1;        // level the blocks were built for
    // in the level's staged tables
    const BinBlock* dBlocks = nullptr;
    const int* dSegInfo = nullptr;   // per image group: first block, block count, blocks before it
    int numSegs = 0, numBlocks = 0;
    DevBuf<int2> work;
    int workGroups = -1;   // feature groups the work list was built for
    int numWork = 0;
};

// An event pair for timing launches the tuner measures.
class EventPair {
public:
    EventPair() {
        CF_HIP(hipEventCreate(&a));
        CF_HIP(hipEventCreate(&b));
    }
    ~EventPair() {
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
    }
    EventPair(const EventPair&) = delete;
    EventPair& operator=(const EventPair&) = delete;
    hipEvent_t a = nullptr, b = nullptr;
};

// A level's evaluation captured from the stream into a graph, instantiated and launched once.  The
// capture holds kernels only (buffers are cleared by a fill kernel, not a memset node; tables are
// uploaded before it), so nothing in it depends on host memory.
class LevelGraph {
public:
    explicit LevelGraph(hipStream_t s) : s_(s) {}
    ~LevelGraph() {
        if (capturing_) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(s_, &g);
            if (g) (void)hipGraphDestroy(g);
        }
        if (launched_) (void)hipStreamSynchronize(s_);   // normally done already: the level waits for its argmax
        if (exec_) (void)hipGraphExecDestroy(exec_);
        if (graph_) (void)hipGraphDestroy(graph_);
    }
    LevelGraph(const LevelGraph&) = delete;
    LevelGraph& operator=(const LevelGraph&) = delete;
    void beginCapture() {
        CF_HIP(hipStreamBeginCapture(s_, hipStreamCaptureModeThreadLocal));
        capturing_ = true;
    }
    void launch() {
        capturing_ = false;
        CF_HIP(hipStreamEndCapture(s_, &graph_));
        CF_HIP(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0));
        CF_HIP(hipGraphLaunch(exec_, s_));
        launched_ = true;
    }
    bool launched() const { return launched_; }

private:
    hipStream_t s_;
    bool capturing_ = false, launched_ = false;
    hipGraph_t graph_ = nullptr;
    hipGraphExec_t exec_ = nullptr;
};

struct LevelNode {
    int active;  // index into the active list (feature table)
    int node;    // node index in its tree
    int begin, count;
    int chunkBegin, chunkEnd;
};

// a node's samples in chunks of at most `per` for slot `slot` of a direct evaluation
void appendChunks(std::vector<Chunk>& out, const LevelNode& ln, int slot, int per) {
    for (int b = 0; b < ln.count; b += per) out.push_back(Chunk{slot, ln.active, ln.begin + b, std::min(per, ln.count - b)});
}

// Device time of the work enqueued between begin() and end() on the stream.  The events are read by
// flush(), called where the host waits for the stream anyway, so timing adds no host waits between
// the kernels of a level.
class PhaseTimer {
public:
    PhaseTimer(hipStream_t s, bool on) : s_(s), on_(on) {}
    ~PhaseTimer() {
        for (hipEvent_t e : pool_) (void)hipEventDestroy(e);
        for (const Pending& p : pending_) {
            (void)hipEventDestroy(p.a);
            (void)hipEventDestroy(p.b);
        }
        if (cur_) (void)hipEventDestroy(cur_);
    }
    void begin() {
        if (!on_) return;
        if (!cur_) cur_ = take();
        CF_HIP(hipEventRecord(cur_, s_));
    }
    // the phase's elapsed milliseconds are added to `acc` at the next flush()
    void end(double& acc) {
        if (!on_) return;
        hipEvent_t b = take();
        CF_HIP(hipEventRecord(b, s_));
        pending_.push_back(Pending{cur_, b, &acc});
        cur_ = nullptr;
    }
    // waits for the last ended phase and accumulates every ended phase
    void flush() {
        if (!on_ || pending_.empty()) return;
        CF_HIP(hipEventSynchronize(pending_.back().b));
        for (const Pending& p : pending_) {
            float ms = 0;
            CF_HIP(hipEventElapsedTime(&ms, p.a, p.b));
            *p.acc += ms;
            pool_.push_back(p.a);
            pool_.push_back(p.b);
        }
        pending_.clear();
    }

private:
    struct Pending {
        hipEvent_t a, b;
        double* acc;
    };
    hipEvent_t take() {
        if (!pool_.empty()) {
            hipEvent_t e = pool_.back();
            pool_.pop_back();
            return e;
        }
        hipEvent_t e = nullptr;
        CF_HIP(hipEventCreate(&e));
        return e;
    }
    hipStream_t s_;
    bool on_;
    hipEvent_t cur_ = nullptr;
    std::vector<hipEvent_t> pool_;
    std::vector<Pending> pending_;
};

// Device memory budgets of a batched level.  CURFIL_*_BUDGET_MB sets them in MiB
// (at least 16); CURFIL_*_BUDGET_KB in KiB without that floor, so that small
// workloads can be made to run the evaluation in several feature-group and
// node-slot batches, as the full-size workloads do.
size_t budgetBytes(const char* mbVar, const char* kbVar, size_t defaultMb) {
    if (const char* kb = std::getenv(kbVar)) {
        const long long v = std::atoll(kb);
        return static_cast<size_t>(std::max(1LL, v)) << 10;
    }
    const char* e = std::getenv(mbVar);
    size_t mb = e ? static_cast<size_t>(std::atoll(e)) : defaultMb;
    if (mb < 16) mb = 16;
    return mb << 20;
}

size_t evalBudgetBytes() { return budgetBytes("CURFIL_EVAL_BUDGET_MB", "CURFIL_EVAL_BUDGET_KB", 2048); }

size_t binsBudgetBytes() { return budgetBytes("CURFIL_BINS_BUDGET_MB", "CURFIL_BINS_BUDGET_KB", 4096); }

bool isPure(const uint32_t* h, int C) {
    int nz = 0;
    for (int c = 0; c < C; c++) {
        if (h[c] == 0) continue;
        if (++nz > 1) return false;
    }
    return nz == 1;
}

// Small host tables on their way to the device: put() copies one into page-locked memory and returns where it
// will lie on the device, flush() enqueues the copies (one per block, in practice one).  reset() when the
// copies and the kernels that read them are done.
class StageArena {
public:
    void reset() {
        if (blocks_.size() > 1) {   // one block of the size that was needed
            size_t n = 0;
            for (const auto& b : blocks_) n += b->cap;
            blocks_.clear();
            addBlock(n);
        }
        for (auto& b : blocks_) b->used = b->flushed = 0;
    }
    template<class V>
    V* put(const V* p, size_t n) {
        const size_t bytes = (n * sizeof(V) + 255) & ~static_cast<size_t>(255);
        if (blocks_.empty() || blocks_.back()->used + bytes > blocks_.back()->cap) addBlock(bytes);
        Block& b = *blocks_.back();
        V* d = reinterpret_cast<V*>(b.dev.get() + b.used);
        if (n > 0) std::memcpy(b.host.get() + b.used, p, n * sizeof(V));
        b.used += bytes;
        return d;
    }
    template<class V>
    V* put(const std::vector<V>& v) { return put(v.data(), v.size()); }
    void flush(hipStream_t s) {
        for (auto& b : blocks_) {
            if (b->used == b->flushed) continue;
            CF_HIP(hipMemcpyAsync(b->dev.get() + b->flushed, b->host.get() + b->flushed, b->used - b->flushed,
                    hipMemcpyHostToDevice, s));
            b->flushed = b->used;
        }
    }
    void release() { blocks_.clear(); }
    size_t capacityBytes() const {
        size_t n = 0;
        for (const auto& b : blocks_) n += b->cap;
        return n;
    }

private:
    struct Block {
        PinnedBuf host;
        DevBuf<uint8_t> dev;
        size_t cap = 0, used = 0, flushed = 0;
    };
    void addBlock(size_t bytes) {
        auto b = std::make_unique<Block>();
        b->cap = std::max<size_t>(bytes, 256 * 1024);
        b->host.resize(b->cap);
        b->dev.resize(b->cap);
        blocks_.push_back(std::move(b));
    }
    std::vector<std::unique_ptr<Block>> blocks_;
};

}  // namespace

// What a training call allocates.  It stays with the context for the next call (hipMalloc and hipFree took 7.6
// of 22 ms of a small training: 13 flipped frames of 320x240, 2 trees, 500 x 50), under the context's mutex, on
// the context's stream; contents never carry over.  After a call the buffers over kKeepBytes in all are given
// back, the largest first; the rest with the context.
struct TrainWorkspace {
    static constexpr size_t kKeepBytes = size_t{1} << 30;
    DevBuf<cf_sample> level[2];
    DevBuf<uint8_t> dir;
    FeatTables tabs;
    DevBuf<int2> graphWork[2];   // work lists of a captured level: full and last feature-group batch
    DevBuf<uint32_t> G;
    DevBuf<FeatSummary> summ, repSumm;
    DevBuf<double> allScores;
    DevBuf<NodeBest> repBest;
    DevBuf<uint32_t> keys, vals, perm, sortCount, sortCursor, sortBlocks;
    DevBuf<uint8_t> lab8;
    std::map<int, BlockSet> blockSets;   // by pass-1 block size
    DevBuf<int> starts;
    DevBuf<uint4> bins;
    DevBuf<uint8_t> results;     // a level's argmax, split records, chunk counts and left histograms
    PinnedBuf hostResults, hostStarts;
    StageArena arena[2];         // by level parity

    template<class Fn>
    void each(Fn&& fn) {
        fn(level[0]); fn(level[1]); fn(dir); fn(graphWork[0]); fn(graphWork[1]); fn(G); fn(summ); fn(repSumm);
        fn(allScores); fn(repBest); fn(keys); fn(vals); fn(perm); fn(sortCount); fn(sortCursor); fn(sortBlocks);
        fn(lab8); fn(starts); fn(bins); fn(results); fn(hostResults); fn(hostStarts); fn(arena[0]); fn(arena[1]);
        tabs.each(fn);
        for (auto& kv : blockSets) fn(kv.second.work);
    }
    void trim() {
        for (;;) {
            size_t sum = 0, most = 0;
            each([&](auto& b) {
                sum += b.capacityBytes();
                most = std::max(most, b.capacityBytes());
            });
            if (sum <= kKeepBytes) return;
            each([&](auto& b) {
                if (b.capacityBytes() == most) b.release();
            });
        }
    }
};

namespace {
// the workspace of one call, trimmed at its end (also when the call throws: after its enqueued work)
struct WorkspaceUse {
    TrainWorkspace& ws;
    hipStream_t s;
    ~WorkspaceUse() {
        (void)hipStreamSynchronize(s);
        ws.trim();
    }
};
}  // namespace

void trainTrees(cf_ctx* ctx, cf_images* images, const cf_train_config& cfg, int C, std::vector<TreeJob>& jobs,
        int mode, std::vector<TreeBuild>& out, TrainStats& stats) {
    if (cfg.max_depth <= 0) throw Error(CF_ERR_ARG, "maxDepth must be positive");
    if (C < 1 || C > kMaxClasses) throw Error(CF_ERR_ARG, "number of classes must be in [1, 32]");
    if (cfg.feature_count == 0 || cfg.thresholds == 0) throw Error(CF_ERR_ARG, "featureCount and thresholds must be positive");
    if (mode != CF_MODE_PLAIN && mode != CF_MODE_BATCHED) throw Error(CF_ERR_ARG, "unknown training mode");
    const int F = static_cast<int>(cfg.feature_count);
    const int T = cfg.thresholds;
    hipStream_t s = ctx->stream;
    const auto t0 = std::chrono::steady_clock::now();

    out.assign(jobs.size(), TreeBuild());
    size_t total = 0;
    bool anyBoth = false;
    for (auto& j : jobs) {
        total += j.roots->size();
        for (const cf_sample& x : *j.roots) anyBoth = anyBoth || x.flip == 2;
    }
    // a Both sample splits at most once into a NoFlip sample and a Flip copy, which
    // never split again: a level holds at most twice the root samples
    const size_t capacity = std::max<size_t>(anyBoth ? 2 * total : total, 1);
    if (!ctx->trainWorkspace) ctx->trainWorkspace = std::make_shared<TrainWorkspace>();
    TrainWorkspace& ws = *ctx->trainWorkspace;
    WorkspaceUse use{ws, s};
    DevBuf<cf_sample>* level = ws.level;
    level[0].resize(capacity);
    level[1].resize(capacity);
    DevBuf<uint8_t>& dir = ws.dir;
    dir.resize(capacity);

    std::vector<ActiveTree> active;
    {
        size_t offset = 0;   // each tree's roots are copied straight from the forest into level 0
        for (size_t j = 0; j < jobs.size(); j++) {
            TreeBuild& tb = out[j];
            cf_tree_node root{};
            root.id = jobs[j].treeId;
            root.level = 1;
            root.parent = -1;
            root.left = root.right = -1;
            root.num_samples = static_cast<int32_t>(jobs[j].roots->size());
            root.is_leaf = 1;
            tb.nodes.push_back(root);
            tb.hist.assign(C, 0u);
            for (const cf_sample& x : *jobs[j].roots) {
                if (x.label >= C) throw Error(CF_ERR_ARG, "sample label >= number of classes");
                if (x.image >= static_cast<uint32_t>(images->count)) throw Error(CF_ERR_ARG, "sample image out of range");
                if (x.x >= images->W || x.y >= images->H) throw Error(CF_ERR_ARG, "sample position outside the image");
                tb.hist[x.label] += 1;
                if (x.flip == 2) tb.hist[x.label] += 1;
            }
            if (jobs[j].roots->empty()) continue;
            ActiveTree a;
            a.job = static_cast<int>(j);
            a.idNode = jobs[j].treeId;
            a.nodes.push_back(0);
            a.counts.push_back(static_cast<int>(jobs[j].roots->size()));
            a.begin = static_cast<int>(offset);
            a.n = static_cast<int>(jobs[j].roots->size());
            CF_HIP(hipMemcpyAsync(level[0].get() + offset, jobs[j].roots->data(), jobs[j].roots->size() * sizeof(cf_sample),
                    hipMemcpyHostToDevice, s));
            offset += jobs[j].roots->size();
            active.push_back(std::move(a));
        }
    }
    int cur = 0;

    // Batched levels use the two-pass evaluation (image-major bins, then
    // node histograms; samples set to Both get a second, flipped bin row)
    // unless T exceeds the 8-bit bins or CURFIL_EVAL_DIRECT is set.
    const bool twoPass = mode == CF_MODE_BATCHED && T <= kMaxBinThresholds &&
            std::getenv("CURFIL_EVAL_DIRECT") == nullptr;

    FeatTables& tabs = ws.tabs;
    tabs.meanDraws = 0;
    DevBuf<int2>* dGraphWork = ws.graphWork;
    DevBuf<uint32_t>& dG = ws.G;
    DevBuf<FeatSummary>& dSumm = ws.summ;
    DevBuf<FeatSummary>& dRepSumm = ws.repSumm;
    DevBuf<double>& dAllScores = ws.allScores;
    DevBuf<NodeBest>& dRepBest = ws.repBest;
    DevBuf<uint32_t>&dKeys = ws.keys, &dVals = ws.vals, &dPerm = ws.perm, &dSortCount = ws.sortCount,
            &dSortCursor = ws.sortCursor, &dSortBlocks = ws.sortBlocks;
    DevBuf<uint8_t>& dLab8 = ws.lab8;
    std::map<int, BlockSet>& blockSets = ws.blockSets;
    EventPair tuneEvents;
    const hipEvent_t tuneStart = tuneEvents.a, tuneEnd = tuneEvents.b;
    DevBuf<int>& dStarts = ws.starts;
    DevBuf<uint4>& dBins = ws.bins;
    const size_t binsBudget = binsBudgetBytes();
    // CURFIL_LEVEL_GRAPH=1: levels whose pass-1 shape is settled run as one captured graph.  Off by default:
    // once a graph has been instantiated the HIP runtime holds one of the process's hardware queues
    // (GPU_MAX_HW_QUEUES, 4 by default), so streams created later share queues (the serving loop's three
    // lost a fifth of their capacity), and a level launched kernel by kernel is as fast: its host reads
    // wait for nothing between kernels.  Not while the context profiles either: the phase timers' events
    // have to be recorded on the stream (events recorded inside a captured graph give no elapsed times).
    const char* lg = std::getenv("CURFIL_LEVEL_GRAPH");
    const bool levelGraphs = lg && std::strcmp(lg, "1") == 0 && !ctx->profiling;
    PhaseTimer timer(s, ctx->profiling);
    const size_t perSlot = static_cast<size_t>(F) * (T + 1) * C;
    const size_t budget = evalBudgetBytes();
    size_t maxSlots = std::max<size_t>(1, budget / (perSlot * sizeof(uint32_t)));

    // per-level evaluation log on stderr (with profiling on), like the reference's per-level INFO lines
    const bool levelLog = ctx->profiling && std::getenv("CURFIL_LEVEL_LOG") != nullptr;
    for (int levelNr = 1; !active.empty(); levelNr++) {
        if (levelNr == cfg.max_depth) break;
        stats.levels++;
        const int numActive = static_cast<int>(active.size());
        // the level before the last has been read back, and with it everything that its tables fed
        StageArena& up = ws.arena[levelNr & 1];
        up.reset();
        // ---- feature generation jobs, one per tree
        std::vector<FeatGenJob> fj(numActive);
        for (int a = 0; a < numActive; a++) {
            fj[a].samples = level[cur].get() + active[a].begin;
            fj[a].n = active[a].n;
            fj[a].seed = jobs[active[a].job].rs.uniformSampler(0xFFFFFF).next();
            fj[a].outOffset = a * F;
        }
        // ---- nodes and chunks of the level (slot = position in `nodes`)
        std::vector<LevelNode> nodes;
        std::vector<Chunk> chunks;
        std::vector<uint32_t> nodeHist;   // class histograms and trees of the level's nodes
        std::vector<int> nodeTree;
        std::vector<int> multiSlots;      // the nodes of more than one chunk
        for (int a = 0; a < numActive; a++) {
            int off = active[a].begin;
            for (size_t k = 0; k < active[a].nodes.size(); k++) {
                LevelNode ln;
                ln.active = a;
                ln.node = active[a].nodes[k];
                ln.begin = off;
                ln.count = active[a].counts[k];
                ln.chunkBegin = static_cast<int>(chunks.size());
                appendChunks(chunks, ln, static_cast<int>(nodes.size()), kChunk);
                ln.chunkEnd = static_cast<int>(chunks.size());
                off += ln.count;
                nodes.push_back(ln);
                const uint32_t* h = &out[active[a].job].hist[static_cast<size_t>(ln.node) * C];
                nodeHist.insert(nodeHist.end(), h, h + C);
                nodeTree.push_back(a);
                if (ln.chunkEnd - ln.chunkBegin > 1) multiSlots.push_back(static_cast<int>(nodes.size()) - 1);
                stats.evaluations += static_cast<double>(ln.count) * F * T;
                stats.responses += static_cast<double>(ln.count) * F;
                stats.nodes += 1;
            }
        }
        const FeatGenJob* dJobs = up.put(fj);
        const Chunk* dChunks = up.put(chunks);
        const uint32_t* dNodeHist = up.put(nodeHist);
        const int* dNodeTree = up.put(nodeTree);
        const int* dMulti = up.put(multiSlots);
        up.flush(s);
        const int numNodes = static_cast<int>(nodes.size());
        const int numChunks = static_cast<int>(chunks.size());
        const double evalMsBefore = stats.evalKernelMs;
        // what the host reads of a level, in one buffer: split record and argmax per node, left and right
        // entries per part of a chunk, left class histogram per node
        const int parts = partitionParts(numChunks), partLen = (kChunk + parts - 1) / parts;
        const size_t splitsAt = 0, bestAt = splitsAt + numNodes * sizeof(SplitRec),
                countsAt = bestAt + numNodes * sizeof(NodeBest), histAt = countsAt + static_cast<size_t>(numChunks) * parts * sizeof(int2),
                resultBytes = histAt + static_cast<size_t>(numNodes) * C * sizeof(uint32_t);
        static_assert(sizeof(SplitRec) % 8 == 0 && sizeof(NodeBest) % 8 == 0, "alignment of the parts that follow");
        ws.results.resize(resultBytes + 16);
        NodeBest* dBest = reinterpret_cast<NodeBest*>(ws.results.get() + bestAt);
        SplitRec* dSplits = reinterpret_cast<SplitRec*>(ws.results.get() + splitsAt);
        int2* dPartCounts = reinterpret_cast<int2*>(ws.results.get() + countsAt);
        uint32_t* dLeftHist = reinterpret_cast<uint32_t*>(ws.results.get() + histAt);
        uint8_t* hostResults = ws.hostResults.resize(resultBytes + 16);
        NodeBest* best = reinterpret_cast<NodeBest*>(hostResults + bestAt);

        // image-major order of a level that is evaluated in two passes; the segments' starts are read at the
        // feature generation's wait
        int N = 0, M = 0, numKeys = 0;
        auto sortLevel = [&]() {
            for (int a = 0; a < numActive; a++) N = std::max(N, active[a].begin + active[a].n);
            // image-major order of the level: (image, tree, place) keys, counting sort of level indices.
            // With Both samples a second entry per level index evaluates it flipped; the entries of samples
            // that are not Both get the key one past the last (tree, image) and sort to the end.
            M = anyBoth ? 2 * N : N;
            dKeys.resize(M);
            dVals.resize(M);
            dPerm.resize(M);
            dLab8.resize(N);
            const uint64_t keyRange = static_cast<uint64_t>(numActive) * static_cast<uint64_t>(images->count);
            if (keyRange >= (1ull << 27)) throw Error(CF_ERR_UNSUPPORTED, "too many (tree, image) segments in one level");
            // within a segment, samples ordered by place, as finely as the number of segments allows
            // (CURFIL_ROW_ORDER=0: not at all)
            int placeShift = 0;
            int placeBits = levelPlaceBits(keyRange, levelPlaces(images->W, images->H), &placeShift);
            const char* rowOrder = std::getenv("CURFIL_ROW_ORDER");
            if (rowOrder && std::strcmp(rowOrder, "0") == 0) placeBits = 0;
            // segments (image, tree) in image-major order: the trees' segments of one image are adjacent
            for (int a = 0; a < numActive; a++) {
                launchLevelKeys(s, level[cur].get(), active[a].begin, active[a].n, static_cast<uint32_t>(a),
                        static_cast<uint32_t>(numActive), dKeys.get(), dVals.get(), anyBoth ? N : 0,
                        static_cast<uint32_t>(keyRange), placeBits, placeShift, images->H);
            }
            numKeys = static_cast<int>(keyRange);
            dSortCount.resize(levelSortBuckets(numKeys, placeBits));
            dSortCursor.resize(levelSortBuckets(numKeys, placeBits));
            dSortBlocks.resize(levelSortScanBlocks(numKeys, placeBits));
            dStarts.resize(numKeys + 1);
            levelCountingSort(s, dKeys.get(), dVals.get(), M, numKeys, placeBits, dSortCount.get(), dSortCursor.get(),
                    dSortBlocks.get(), dPerm.get(), dStarts.get());
            launchLevelLabels(s, level[cur].get(), N, dLab8.get());
            int* hostStarts = reinterpret_cast<int*>(ws.hostStarts.resize((static_cast<size_t>(numKeys) + 1) * sizeof(int)));
            CF_HIP(hipMemcpyAsync(hostStarts, dStarts.get(), (static_cast<size_t>(numKeys) + 1) * sizeof(int),
                    hipMemcpyDeviceToHost, s));
        };
        if (twoPass) sortLevel();

        timer.begin();
        launchFeatureGeneration(s, images->set(), dJobs, numActive, F, T, cfg.box_radius, cfg.region_size,
                cfg.use_depth_images, tabs);
        timer.end(stats.featGenMs);

        // ---- evaluation
        auto evalSlots = [&](int s0, int s1) {
            const int ns = s1 - s0;
            const uint32_t* slotHist = dNodeHist + static_cast<size_t>(s0) * C;
            dG.resize(static_cast<size_t>(ns) * perSlot);
            dSumm.resize(static_cast<size_t>(ns) * F);
            const Chunk node{0, nodes[s0].active, nodes[s0].begin, nodes[s0].count};
            const bool scored = ns == 1 && evalScoresNode(node.count, F, T, C);
            auto histograms = [&]() {
                CF_HIP(hipMemsetAsync(dG.get(), 0, static_cast<size_t>(ns) * perSlot * sizeof(uint32_t), s));
                if (ns == 1) {
                    launchEvalNode(s, images->set(), level[cur].get(), node, tabs, C, dG.get());
                    return;
                }
                size_t slotSamples = 0;
                for (int i = s0; i < s1; i++) slotSamples += nodes[i].count;
                const int per = evalChunkSamples(slotSamples, F);
                std::vector<Chunk> bc;
                for (int i = s0; i < s1; i++) appendChunks(bc, nodes[i], i - s0, per);
                const Chunk* dEval = up.put(bc);
                up.flush(s);
                launchEvalHistograms(s, images->set(), level[cur].get(), dEval, static_cast<int>(bc.size()), tabs, C,
                        dG.get());
            };
            timer.begin();
            if (scored) {
                launchEvalNode(s, images->set(), level[cur].get(), node, tabs, C, nullptr, slotHist, dSumm.get());
            } else {
                histograms();
            }
            timer.end(stats.evalKernelMs);
            stats.evalLaunches += 1;
            timer.begin();
            if (!scored) launchScores(s, dG.get(), slotHist, dNodeTree + s0, ns, tabs, C, dSumm.get(), nullptr, -1);
            launchReduce(s, dSumm.get(), ns, F, dBest + s0);
            timer.end(stats.scoreMs);
            CF_HIP(hipMemcpyAsync(&best[s0], dBest + s0, ns * sizeof(NodeBest), hipMemcpyDeviceToHost, s));
            CF_HIP(hipStreamSynchronize(s));
            timer.flush();
            for (int i = 0; i < ns; i++) {
                if (!best[s0 + i].flag) continue;
                // near-tie band: replay the reference's sequential scan for this node
                dAllScores.resize(static_cast<size_t>(T) * F);
                if (scored) histograms();
                launchScores(s, dG.get(), slotHist, dNodeTree + s0, ns, tabs, C, dSumm.get(), dAllScores.get(), i);
                launchSequentialArgmax(s, dAllScores.get(), T, F, dBest + s0 + i);
                stats.replays++;
            }
        };
        // the literal sequential argmax of flagged nodes from their direct-path histograms, as many nodes
        // per launch as the histogram budget holds
        auto replayNodes = [&](const std::vector<int>& flagged) {
            for (size_t a = 0; a < flagged.size();) {
                const int ns = static_cast<int>(std::min<size_t>(flagged.size() - a, maxSlots));
                std::vector<Chunk> bc;
                std::vector<uint32_t> nh(static_cast<size_t>(ns) * C);
                std::vector<int> st(ns);
                size_t flaggedSamples = 0;
                for (int k = 0; k < ns; k++) flaggedSamples += nodes[flagged[a + k]].count;
                const int per = evalChunkSamples(flaggedSamples, F);
                for (int k = 0; k < ns; k++) {
                    const LevelNode& ln = nodes[flagged[a + k]];
                    appendChunks(bc, ln, k, per);
                    std::memcpy(&nh[static_cast<size_t>(k) * C],
                            &out[active[ln.active].job].hist[static_cast<size_t>(ln.node) * C], C * sizeof(uint32_t));
                    st[k] = ln.active;
                }
                const Chunk* dRepChunks = up.put(bc);
                const uint32_t* dRepHist = up.put(nh);
                const int* dRepTree = up.put(st);
                up.flush(s);
                dG.resize(static_cast<size_t>(ns) * perSlot);
                dAllScores.resize(static_cast<size_t>(ns) * T * F);
                dRepSumm.resize(static_cast<size_t>(ns) * F);
                dRepBest.resize(ns);
                CF_HIP(hipMemsetAsync(dG.get(), 0, static_cast<size_t>(ns) * perSlot * sizeof(uint32_t), s));
                launchEvalHistograms(s, images->set(), level[cur].get(), dRepChunks, static_cast<int>(bc.size()), tabs, C,
                        dG.get());
                launchScores(s, dG.get(), dRepHist, dRepTree, ns, tabs, C, dRepSumm.get(), dAllScores.get(), -1);
                launchSequentialArgmax(s, dAllScores.get(), T, F, dRepBest.get(), ns);
                for (int k = 0; k < ns; k++) {
                    CF_HIP(hipMemcpyAsync(dBest + flagged[a + k], dRepBest.get() + k, sizeof(NodeBest),
                            hipMemcpyDeviceToDevice, s));
                }
                stats.replays += ns;
                a += ns;
            }
        };
        auto evalTwoPass = [&]() {
            // (image, tree) segments of the sorted order -> blocks of at most the launch shape's samples within a
            // segment; the segments of one image form a group of consecutive blocks
            int* starts = reinterpret_cast<int*>(ws.hostStarts.get());
            timer.flush();
            if (starts[numKeys] < 0) starts[numKeys] = M;   // the end of the last segment
            // blocks of one pass-1 block size: consecutive runs of <= blockSamples entries within a (image, tree)
            // segment; the segments of one image form a group of consecutive blocks.  Built on the host from the
            // segment starts for each block size the tuner asks for; the work list of a batch of ngb feature
            // groups is then built on the device: each XCD takes an eighth of it in order, all feature groups of an
            // image group (feature group major, then tree, then block) before the next image group, so the trees'
            // workgroups of one feature group read the same planes of one image from the XCD's L2; workgroup w runs on
            // XCD w % 8, so the lists are interleaved
            for (auto& kv : blockSets) kv.second.level = -1;
            auto blocksFor = [&](int blockSamples) -> BlockSet& {
                BlockSet& bs = blockSets[blockSamples];
                if (bs.level == levelNr) return bs;
                bs.level = levelNr;
                bs.workGroups = -1;
                std::vector<BinBlock> blocks;
                std::vector<std::pair<int, int>> segBlocks;   // per image group: first block, block count
                int k = 0;
                while (k < numKeys && starts[k] < 0) k++;
                while (k < numKeys) {
                    int k2 = k + 1;
                    while (k2 < numKeys && starts[k2] < 0) k2++;
                    const int b = starts[k], e = starts[k2];
                    const int first = static_cast<int>(blocks.size());
                    for (int p = b; p < e; p += blockSamples) {
                        blocks.push_back(BinBlock{k % numActive, p, std::min(blockSamples, e - p), k / numActive});
                    }
                    const int image = k / numActive;
                    if (!segBlocks.empty() && blocks[segBlocks.back().first].image == image) {
                        segBlocks.back().second += static_cast<int>(blocks.size()) - first;
                    } else {
                        segBlocks.emplace_back(first, static_cast<int>(blocks.size()) - first);
                    }
                    k = k2;
                }
                bs.dBlocks = up.put(blocks);
                bs.numSegs = static_cast<int>(segBlocks.size());
                bs.numBlocks = static_cast<int>(blocks.size());
                std::vector<int> segInfo(3 * static_cast<size_t>(bs.numSegs), 0);
                for (int i = 0, before = 0; i < bs.numSegs; i++) {
                    segInfo[i] = segBlocks[i].first;
                    segInfo[bs.numSegs + i] = segBlocks[i].second;
                    segInfo[2 * static_cast<size_t>(bs.numSegs) + i] = before;
                    before += segBlocks[i].second;
                }
                bs.dSegInfo = up.put(segInfo);
                up.flush(s);
                return bs;
            };
            // the work list of a batch of ngb feature groups into `work`; returns its length
            auto buildWork = [&](BlockSet& bs, int ngb, DevBuf<int2>& work) {
                const int numWork = buildWorkLength(bs.numBlocks, ngb);
                work.resize(std::max<size_t>(static_cast<size_t>(numWork), 1));
                const int ns = bs.numSegs;
                launchBuildWork(s, bs.dSegInfo, bs.dSegInfo + ns, bs.dSegInfo + 2 * ns, ns, bs.numBlocks, ngb,
                        work.get());
                return numWork;
            };
            auto workFor = [&](BlockSet& bs, int ngb) {
                if (bs.workGroups == ngb) return;
                bs.workGroups = ngb;
                bs.numWork = buildWork(bs, ngb, bs.work);
            };
            dSumm.resize(static_cast<size_t>(numNodes) * F);
            // feature groups in batches that fit the bin-row budget; node slots in batches that fit the histogram budget
            const int groupsTotal = (F + kBinGroup - 1) / kBinGroup;
            // a group's rows: one per level index, and a second (flipped) one with Both samples
            const size_t rowBytes = static_cast<size_t>(N) * sizeof(uint4) * (anyBoth ? 2 : 1);
            const int ng = static_cast<int>(std::max<size_t>(1, std::min<size_t>(groupsTotal, binsBudget / rowBytes)));
            const size_t flipOffset = anyBoth ? static_cast<size_t>(ng) * N : 0;
            dBins.resize(static_cast<size_t>(ng) * N * (anyBoth ? 2 : 1));
            stats.groupBatchesMax = std::max(stats.groupBatchesMax, (groupsTotal + ng - 1) / ng);
            const int TM = binThresholdWidth(T);
            bool tuning = false;
            const int levelShape = evalTunerChoose(TM, static_cast<size_t>(M), &tuning);
            // node-slot batches of a batch of ngb feature groups: the slots whose histograms fit the budget
            auto slotBatches = [&](int ngb) {
                const size_t perSlot = static_cast<size_t>(ngb) * kBinGroup * (T + 1) * C;
                const int maxSlots = static_cast<int>(std::max<size_t>(1, budget / (perSlot * sizeof(uint32_t))));
                std::vector<std::pair<int, int>> out;
                for (int s0 = 0; s0 < numNodes; s0 += maxSlots) out.emplace_back(s0, std::min(numNodes, s0 + maxSlots));
                return out;
            };
            // pass 2 and the scores of the slots [s0, s1) for the feature groups [g0, g0 + ngb): nodes of a single chunk
            // are scored where they are counted, the others' histograms cleared, added to and read
            auto countAndScore = [&](int s0, int s1, int g0, int ngb) {
                const int nc = nodes[s1 - 1].chunkEnd - nodes[s0].chunkBegin;
                const size_t perSlotB = static_cast<size_t>(ngb) * kBinGroup * (T + 1) * C;
                const bool scored = histScoresNodes(nc, ngb, T, C);
                int ns = s1 - s0;
                const int* listed = nullptr;
                if (scored) {
                    const auto m0 = std::lower_bound(multiSlots.begin(), multiSlots.end(), s0);
                    listed = dMulti + (m0 - multiSlots.begin());
                    ns = static_cast<int>(std::lower_bound(m0, multiSlots.end(), s1) - m0);
                    launchClearSlots(s, dG.get(), listed, ns, s0, perSlotB);
                } else {
                    launchFillU32(s, dG.get(), ns * perSlotB, 0u);
                }
                timer.begin();
                launchHistBins(s, dBins.get(), dLab8.get(), dChunks + nodes[s0].chunkBegin, nc, s0, g0, ngb, tabs, C, N,
                        dG.get(), flipOffset, scored ? dNodeHist : nullptr, scored ? dSumm.get() : nullptr);
                timer.end(stats.histMs);
                timer.begin();
                launchScores(s, dG.get(), dNodeHist + static_cast<size_t>(s0) * C, dNodeTree + s0, ns, tabs, C,
                        dSumm.get() + static_cast<size_t>(s0) * F, nullptr, -1, g0 * kBinGroup, ngb * kBinGroup, listed, s0);
                timer.end(stats.scoreMs);
            };
            LevelGraph graph(s);
            if (!tuning && levelGraphs) {
                // The shape is settled: the level's evaluation (every batch's pass 1; per node-slot batch the
                // histogram clear, pass 2 and the scores; the argmax) is captured into one graph and launched
                // once, so the device runs it back to back with no host work between its kernels.  Work
                // lists, chunk tables and buffers are set up before the capture.
                const EvalShape& es = evalShape(levelShape);
                BlockSet& bs = blocksFor(es.lanes * es.perLane);
                struct Batch {
                    int g0, ngb;
                    const DevBuf<int2>* work;
                    int numWork;
                    std::vector<std::pair<int, int>> slots;
                };
                const int lastNgb = groupsTotal - ((groupsTotal - 1) / ng) * ng;
                const int numWorkFull = buildWork(bs, ng, dGraphWork[0]);
                const int numWorkLast = lastNgb == ng ? numWorkFull : buildWork(bs, lastNgb, dGraphWork[1]);
                bs.workGroups = -1;
                std::vector<Batch> batches;
                size_t maxG = 1;
                for (int g0 = 0; g0 < groupsTotal; g0 += ng) {
                    const int ngb = std::min(ng, groupsTotal - g0);
                    Batch b{g0, ngb, ngb == ng ? &dGraphWork[0] : &dGraphWork[1], ngb == ng ? numWorkFull : numWorkLast,
                            slotBatches(ngb)};
                    const size_t perSlotB = static_cast<size_t>(ngb) * kBinGroup * (T + 1) * C;
                    for (const auto& sb : b.slots) {
                        maxG = std::max(maxG, static_cast<size_t>(sb.second - sb.first) * perSlotB);
                    }
                    batches.push_back(std::move(b));
                }
                dG.resize(maxG);
                graph.beginCapture();
                for (const Batch& b : batches) {
                    timer.begin();
                    launchEvalBins(s, images->set(), level[cur].get(), dPerm.get(), bs.dBlocks, b.work->get(),
                            b.numWork, b.g0, tabs, N, dBins.get(), flipOffset, levelShape);
                    timer.end(stats.evalKernelMs);
                    stats.evalLaunches += 1;
                    stats.shapeLaunches[levelShape] += 1;
                    stats.slotBatchesMax = std::max(stats.slotBatchesMax, static_cast<int>(b.slots.size()));
                    for (const auto& sb : b.slots) countAndScore(sb.first, sb.second, b.g0, b.ngb);
                }
                timer.begin();
                launchReduce(s, dSumm.get(), numNodes, F, dBest);
                timer.end(stats.scoreMs);
                graph.launch();
                stats.levelGraphs += 1;
            }
            for (int g0 = 0; g0 < (graph.launched() ? 0 : groupsTotal); g0 += ng) {
                const int ngb = std::min(ng, groupsTotal - g0);
                bool measure = false;
                const int shape = evalTunerChoose(TM, static_cast<size_t>(M), &measure);
                const EvalShape& es = evalShape(shape);
                BlockSet& bs = blocksFor(es.lanes * es.perLane);
                workFor(bs, ngb);
                if (measure) CF_HIP(hipEventRecord(tuneStart, s));
                timer.begin();
                launchEvalBins(s, images->set(), level[cur].get(), dPerm.get(), bs.dBlocks, bs.work.get(),
                        bs.numWork, g0, tabs, N, dBins.get(), flipOffset, shape);
                timer.end(stats.evalKernelMs);
                if (measure) {
                    CF_HIP(hipEventRecord(tuneEnd, s));
                    CF_HIP(hipEventSynchronize(tuneEnd));
                    float ms = 0;
                    CF_HIP(hipEventElapsedTime(&ms, tuneStart, tuneEnd));
                    // responses of the launch: every entry of the permutation for each feature of the batch
                    const int feats = std::min(F - g0 * kBinGroup, ngb * kBinGroup);
                    evalTunerRecord(TM, static_cast<size_t>(M), shape, ms, static_cast<double>(M) * feats);
                }
                stats.evalLaunches += 1;
                stats.shapeLaunches[shape] += 1;
                const size_t perSlotB = static_cast<size_t>(ngb) * kBinGroup * (T + 1) * C;
                const int maxSlotsB = static_cast<int>(std::max<size_t>(1, budget / (perSlotB * sizeof(uint32_t))));
                stats.slotBatchesMax = std::max(stats.slotBatchesMax, (numNodes + maxSlotsB - 1) / maxSlotsB);
                for (int s0 = 0; s0 < numNodes;) {
                    const int s1 = std::min(numNodes, s0 + maxSlotsB);
                    dG.resize(static_cast<size_t>(s1 - s0) * perSlotB);
                    countAndScore(s0, s1, g0, ngb);
                    s0 = s1;
                }
            }
            if (!graph.launched()) {
                timer.begin();
                launchReduce(s, dSumm.get(), numNodes, F, dBest);
                timer.end(stats.scoreMs);
            }
        };
        if (mode == CF_MODE_PLAIN) {
            for (int i = 0; i < numNodes; i++) evalSlots(i, i + 1);
        } else if (twoPass) {
            evalTwoPass();
        } else {
            for (int s0 = 0; s0 < numNodes;) {
                const int s1 = static_cast<int>(std::min<size_t>(numNodes, s0 + maxSlots));
                evalSlots(s0, s1);
                s0 = s1;
            }
        }

        if (levelLog) {
            double levelSamples = 0;
            for (const auto& ln : nodes) levelSamples += ln.count;
            std::fprintf(stderr, "[curfil] level %d: trees %d nodes %d samples %.0f chunks %zu eval %.2f ms (%.3g responses/s)\n",
                    levelNr, numActive, numNodes, levelSamples, chunks.size(), stats.evalKernelMs - evalMsBefore,
                    levelSamples * F / ((stats.evalKernelMs - evalMsBefore) * 1e-3));
        }

        // ---- split records, built on the device from the argmax and the level's feature tables, and the samples'
        // directions; the level's one read-back.  Nodes of a two-pass level whose argmax has to be replayed show
        // up in it: they are replayed, and the records and directions made again.
        for (bool again = twoPass;; again = false) {
            CF_HIP(hipMemsetAsync(dLeftHist, 0, static_cast<size_t>(numNodes) * C * sizeof(uint32_t), s));
            timer.begin();
            launchPartitionDirections(s, images->set(), level[cur].get(), dChunks, numChunks, parts, partLen, dBest,
                    dNodeTree, tabs, C, dSplits, dir.get(), dPartCounts, dLeftHist);
            timer.end(stats.partitionMs);
            CF_HIP(hipMemcpyAsync(hostResults, ws.results.get(), resultBytes, hipMemcpyDeviceToHost, s));
            CF_HIP(hipStreamSynchronize(s));
            timer.flush();
            if (!again) break;
            std::vector<int> flagged;
            for (int i = 0; i < numNodes; i++) {
                if (best[i].flag) flagged.push_back(i);
            }
            if (flagged.empty()) break;
            replayNodes(flagged);
        }
        const SplitRec* splits = reinterpret_cast<const SplitRec*>(hostResults + splitsAt);
        int2* chunkCounts = reinterpret_cast<int2*>(hostResults + countsAt);   // of the parts, then of the chunks
        for (int c = 0; c < numChunks; c++) {
            int2 sum = make_int2(0, 0);
            for (int q = 0; q < parts; q++) {
                sum.x += chunkCounts[c * parts + q].x;
                sum.y += chunkCounts[c * parts + q].y;
            }
            chunkCounts[c] = sum;
        }
        const uint32_t* leftHist = reinterpret_cast<const uint32_t*>(hostResults + histAt);

        // ---- tree growth on the host, next frontier and sample destinations
        std::vector<int2> dst(chunks.size(), make_int2(-1, -1));
        std::vector<ActiveTree> next;
        int nextOff = 0;
        int slot = 0;
        for (int a = 0; a < numActive; a++) {
            ActiveTree& at = active[a];
            TreeBuild& tb = out[at.job];
            ActiveTree na;
            na.job = at.job;
            na.begin = nextOff;
            for (size_t k = 0; k < at.nodes.size(); k++, slot++) {
                const LevelNode& ln = nodes[slot];
                int nL = 0, nR = 0;
                for (int c = ln.chunkBegin; c < ln.chunkEnd; c++) {
                    nL += chunkCounts[c].x;
                    nR += chunkCounts[c].y;
                }
                const int leftId = ++at.idNode;
                const int rightId = ++at.idNode;
                if (nL == 0 || nR == 0) {
                    at.idNode -= 2;
                    continue;
                }
                const int pi = ln.node;
                const int li = static_cast<int>(tb.nodes.size());
                for (int side = 0; side < 2; side++) {
                    cf_tree_node cn{};
                    cn.id = side == 0 ? leftId : rightId;
                    cn.level = tb.nodes[pi].level + 1;
                    cn.parent = pi;
                    cn.left = cn.right = -1;
                    cn.num_samples = side == 0 ? nL : nR;
                    cn.is_leaf = 1;
                    tb.nodes.push_back(cn);
                    for (int c = 0; c < C; c++) {
                        const uint32_t l = leftHist[static_cast<size_t>(slot) * C + c];
                        tb.hist.push_back(side == 0 ? l : tb.hist[static_cast<size_t>(pi) * C + c] - l);
                    }
                }
                cf_tree_node& p = tb.nodes[pi];
                p.is_leaf = 0;
                p.left = li;
                p.right = li + 1;
                p.feature_id = best[slot].feat;
                p.threshold = splits[slot].threshold;
                p.score = best[slot].score;
                for (int q = 0; q < kFeatParams; q++) p.feature[q] = splits[slot].feat.p[q];
                int childBegin[2] = {-1, -1};
                for (int side = 0; side < 2; side++) {
                    const int ci = li + side;
                    const int cnt = side == 0 ? nL : nR;
                    if (!isPure(&tb.hist[static_cast<size_t>(ci) * C], C) &&
                            cnt >= static_cast<int>(cfg.min_sample_count)) {
                        childBegin[side] = nextOff;
                        na.nodes.push_back(ci);
                        na.counts.push_back(cnt);
                        nextOff += cnt;
                    }
                }
                int doneL = 0, doneR = 0;
                for (int c = ln.chunkBegin; c < ln.chunkEnd; c++) {
                    const int cl = chunkCounts[c].x;
                    const int cr = chunkCounts[c].y;
                    dst[c].x = childBegin[0] >= 0 ? childBegin[0] + doneL : -1;
                    dst[c].y = childBegin[1] >= 0 ? childBegin[1] + doneR : -1;
                    doneL += cl;
                    doneR += cr;
                }
            }
            na.n = nextOff - na.begin;
            na.idNode = at.idNode;
            if (!na.nodes.empty()) next.push_back(std::move(na));
        }
        if (nextOff > 0) {
            const int2* dDst = up.put(dst);
            up.flush(s);
            timer.begin();
            launchPartitionScatter(s, level[cur].get(), dChunks, numChunks, parts, partLen, dir.get(), dPartCounts, dDst,
                    level[1 - cur].get());
            timer.end(stats.partitionMs);
            cur = 1 - cur;
        }
        active.swap(next);
    }
    CF_HIP(hipStreamSynchronize(s));
    timer.flush();
    stats.seconds += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace cf
