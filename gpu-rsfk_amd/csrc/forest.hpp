// Internal interfaces between the translation units of the library.
#pragma once
#include "rsfk_common.hpp"
#include <atomic>
#include <thread>
#include "bf16.hpp"
#include "join_copy.hpp"
#include <vector>

namespace rsfk {

struct TreeBatchWorkspace;

// tree_build.hip
size_t tree_ws_bytes(int N, int D, int MIN, int B);
int tree_ws_alloc(TreeBatchWorkspace** out, int N, int D, int MIN, int B);
void tree_ws_free(TreeBatchWorkspace* w);
int tree_ws_enable_index(TreeBatchWorkspace* w, int MIN, int MAX_DEPTH);
const TreeRec* tree_ws_recs(const TreeBatchWorkspace* w, int t);
int tree_ws_leaf_cap(const TreeBatchWorkspace* w);
const int* tree_ws_perm(const TreeBatchWorkspace* w, int t);
const int* tree_ws_leaf_start(const TreeBatchWorkspace* w, int t);
const int* tree_ws_leaf_size(const TreeBatchWorkspace* w, int t);
const int* tree_ws_stats(const TreeBatchWorkspace* w, int t);      // ints: buckets of at most kBucketSplit points, larger ones, ...; those of tree t + 1 kTreeStatPitch further on
int tree_small_threshold(int D, int N, int B);
const float* tree_ws_phase_seconds(const TreeBatchWorkspace* w);
const unsigned long long* tree_ws_counts(const TreeBatchWorkspace* w);
int tree_screen_row_bytes(int D, bool q8);
int build_tree_batch(TreeBatchWorkspace* w, const float* points, const uint16_t* pb16, const uint8_t* q8, int N, int D,
                     int MIN, int MAX,
                     int MAX_DEPTH, int seed0, int nb, int* host_stats, hipStream_t stream);

// bucket_knn.hip
int launch_bucket_knn(const float* points, int N, int D, int K, const int* ids, const int* starts,
                      const int* sizes, int n_buckets, int stride, int max_bucket, int* knn_idx, float* knn_dist,
                      hipStream_t stream);

// bucket_knn_gram.hip
int launch_bucket_knn_gram(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                           int n_buckets, int stride, int min_size, int max_size, int* knn_idx, float* knn_dist,
                           hipStream_t stream);
// trees from this index on take the kernel that screens the pair matrix on the matrix cores (RSFK_GRAM_FROM)
int bucket_gram_from();

// Kernels a tree's buckets can go to (bits of *launched of launch_bucket_knn_tree, and of the report of a build)
enum : int {
    kBucketKernelSmall = 1,      // k_bucket_knn_small<64>: two wavefronts per bucket of up to 64 points, every pair exact
    kBucketKernelScreen = 2,     // k_bucket_knn_screen: the same with the pair matrix bounded on the matrix cores first
    kBucketKernelAuto = 128,     // k_bucket_knn_auto: one of the two, chosen on the device from the previous tree's pairs
    kBucketKernelMedium = 4,     // k_bucket_knn_small<72>: three wavefronts, buckets of 65..72 points
    kBucketKernelRows = 8,       // k_bucket_knn_rows: a bucket's points resident in LDS
    kBucketKernelTiled = 16,     // k_bucket_knn<SL, false>: 64 x 64 tiles, a workgroup per bucket
    kBucketKernelStrip = 32,     // k_bucket_knn<SL, true>: 64 x 64 tiles, a workgroup per 64 members of a bucket
    kBucketKernelGram = 64,      // k_bucket_knn_gram: any bucket size, pair matrix bounded on the matrix cores
    kBucketKernelForest = 512,   // k_forest_pairs + k_forest_merge: the buckets of several trees at once
    kBucketKernelPairs = 256,    // k_bucket_pairs + k_bucket_merge_pairs: 64 x 64 tiles, every pair once, distances through memory
};
// Working memory of k_bucket_pairs / k_bucket_merge_pairs: the pair matrices of as many buckets as fit are in it at a
// time.  One per stream of launches; p == null: the forms of the general kernel that need none are taken.
struct PairScratch {
    float* p = nullptr;
    size_t floats = 0;
};
// Floats of working memory the buckets of a launch would like (0: none of them reaches the general kernel, or the
// form is switched off); at most pair_scratch_max() (512 MB; RSFK_BUCKET_PAIRS_MB overrides), the launch then goes in
// several parts.
size_t pair_scratch_max();
size_t bucket_pairs_scratch_floats(int D, int K, int n_buckets, int max_bucket);
// Form of k_bucket_knn_auto (every pair exact, or bounded on the matrix cores first), from what the tree before left in kFormWords
// words, in a sample of its buckets: words 0..3, pairs << 32 | offered, the pairs that are not above the last slot of one of their rows;
// words 4..7, pairs << 32 | listed, the pairs that the bound of the screened form left to the exact test, if that form ran.
constexpr int kFormWords = 8;
constexpr unsigned int kScreenAlways = 0xffffffffu;
struct BucketFormRule {
    unsigned int share_q16;      // screened below this share of offered pairs (in 1 / 65536); kScreenAlways: always
    unsigned int least_q16;      // ... and not below this one, unless
    unsigned int few_q16;        // ... it is below this one,
    unsigned int vain_q16;       // ... and not once listed less offered pairs were at least this share (twice few_q16 where few are offered)
};
struct BucketForm {
    bool screened, vain;
};
__host__ __device__ __forceinline__ BucketForm bucket_form(const unsigned long long* __restrict__ words, BucketFormRule rule)
{
    if (rule.share_q16 == kScreenAlways) return {true, false};
    unsigned long long a = 0, b = 0;                     // (the halves cannot carry into each other: a tree has < 2^32 pairs)
#pragma unroll
    for (int i = 0; i < kFormWords / 2; ++i) {
        a += words[i];
        b += words[kFormWords / 2 + i];
    }
    const unsigned long long offered = a & 0xffffffffull, pairs = a >> 32, listed = b & 0xffffffffull, bounded = b >> 32;
    const unsigned long long o = offered << 16, nothing = (listed - offered) << 16;      // (listed pairs that no row can take)
    const bool few = o < pairs * rule.few_q16;
    const bool vain = bounded > 0 && nothing >= bounded * (few ? 2 * rule.few_q16 : rule.vain_q16);
    return {!vain && (few || (o < pairs * rule.share_q16 && o >= pairs * rule.least_q16)), vain};
}
// mean: points of a small bucket of the tree
BucketFormRule bucket_form_rule(double mean, int D);
// The small buckets of a tree with sorted rows: words of the tree before (null: first tree) and, zeroed, of this one
struct SmallBucketForm {
    const unsigned long long* prev;
    unsigned long long* words;
    BucketFormRule rule;
};
int launch_bucket_knn_tree(const float* points, const SmallBucketForm* form,
                           bool rows_sorted, bool gram, int D, int K, const int* ids, const int* starts, const int* sizes,
                           int leaf_cap, int n_small, int n_big, int max_bucket, int* knn_idx, float* knn_dist,
                           hipStream_t stream, int part = 0, int trees_before = 0, int* launched = nullptr,
                           const PairScratch* pairs = nullptr);

// bucket_knn_forest.hip: the buckets of several trees at once (small inputs)
bool bucket_forest_wanted(int n_trees);
int bucket_forest_group(int N, int D, int K, int max_bucket, int n_trees, int all_trees);
size_t bucket_forest_floats(int N, int max_bucket, int n_trees);
int launch_bucket_knn_forest(const float* points, int N, int D, int K, int T, const int* perm, const int* leaf_start, const int* leaf_size,
                             int leaf_cap, const int* stats, const int* host_stats, int max_bucket, float* pair_dist, int* info,
                             int* knn_idx, float* knn_dist, hipStream_t stream);

// What the last K-NN-graph build of this process did, as a line of JSON (rsfk_last_build_report): which bucket
// kernels every tree went to, the counts the algorithmic bytes of the tree build and of the exploration are made of,
// and the time of each of the three steps.  Returns the length of the text (without the final zero), which is
// truncated to cap - 1 characters.
int build_report_json(char* buf, int cap);

// bucket_knn_screen.hip
int launch_sort_rows(int* knn_idx, float* knn_dist, int N, int K, hipStream_t stream);
int launch_bucket_knn_screen(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                             int n_buckets, int stride, int* knn_idx, float* knn_dist, hipStream_t stream);
// Buckets of up to 64 points of one tree of a forest, the form of the kernel (every pair exact, or bounded on the matrix
// cores first) chosen on the device (bucket_form).
int launch_bucket_knn_auto(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                           int n_buckets, int* knn_idx, float* knn_dist, const SmallBucketForm& form, hipStream_t stream);
// share of the pairs (in 1 / 65536) below which the screened form is taken (RSFK_BUCKET_SCREEN); kScreenAlways: always
unsigned int bucket_screen_share_q16();

// bucket_knn_rows.hip
int bucket_rows_cap(int D, int K);
int bucket_rows_pitch(int D);
int launch_bucket_knn_rows(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes, int n_buckets,
                           int stride, int min_size, int max_size, bool rows_sorted, bool young_rows, int* knn_idx,
                           float* knn_dist, hipStream_t stream);

// bucket_knn_rows_screen.hip
int launch_bucket_knn_rows_screen(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                                  int n_buckets, int min_size, int max_size, int* knn_idx, float* knn_dist, hipStream_t stream);

// bucket_knn_small.hip
int small_bucket_cap();
int medium_bucket_cap();
int launch_bucket_knn_medium(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                             int n_buckets, int stride, bool rows_sorted, int* knn_idx, float* knn_dist, hipStream_t stream);
int launch_bucket_knn_small(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                            int n_buckets, int stride, bool rows_sorted, int* knn_idx, float* knn_dist, hipStream_t stream);

// host_copy.hip: pageable host memory <-> device memory through pinned buffers, large arrays on several threads
struct HostArray {
    void* dev;
    void* host;
    size_t bytes;
};
// The arrays a call takes to the device.  Small ones are only queued on the stream; the pinned block they pass through
// is held until the object goes (after the call has waited for the stream).
class HostStage {
public:
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage();
    int to_device(const HostArray* a, int n, hipStream_t stream);      // once per object for small arrays

private:
    void* block_ = nullptr;
    hipStream_t stream_ = nullptr;
};
// Everything queued on the stream first, then the copies; complete on return.
int copy_to_host(const HostArray* a, int n, hipStream_t stream);
// The same for results into arrays that may be fresh: begin() once the call's work has started (addresses and sizes on the host count),
// so that a thread makes the arrays' pages while the device works; it ends with finish() or the object.
class HostResult {
public:
    HostResult() = default;
    HostResult(const HostResult&) = delete;
    HostResult& operator=(const HostResult&) = delete;
    ~HostResult();
    void begin(const HostArray* a, int n);
    int finish(const HostArray* a, int n, hipStream_t stream);         // complete on return

private:
    std::thread pages_;
    std::atomic<bool> stop_{false};
};
void release_copy_buffers();

// explore_join.hip
struct ExploreWorkspace;
bool explore_join_enabled(int N, int K);
bool explore_merge_fits(int D, int K);
// graph_only: room for the reversed graph alone (launch_reversed_graph), as blocks the caller can do without (ws_try_alloc)
int explore_ws_alloc(ExploreWorkspace** out, int N, int K, bool with_bounds = false, bool graph_only = false);
bool explore_ws_takes(int N, int K);
int launch_reversed_graph(ExploreWorkspace* w, const int* idx, int N, int K, hipStream_t stream);
const int* explore_ws_offs(const ExploreWorkspace* w);       // N + 1
int* explore_ws_rev(const ExploreWorkspace* w);        // entry numbers p K + k, in compressed rows by the neighbour
void explore_ws_free(ExploreWorkspace* w);
const uint32_t* explore_ws_pass(const ExploreWorkspace* w);
struct JoinBounds;
const JoinBounds& explore_ws_bounds(const ExploreWorkspace* w);
int* explore_ws_todo(ExploreWorkspace* w, int which);
// A list that many points may go to at once is kept in shares, a counter each: additions to one cache line are carried out one after
// the other, about 14 ns each.  Point number i of a launch (of at most N points) has share i % kTodoShares.
constexpr int kTodoShares = 32;
inline int todo_share(int N) { return (N + kTodoShares - 1) / kTodoShares; }
int* explore_ws_share_lists(ExploreWorkspace* w);
int* explore_ws_shares(ExploreWorkspace* w);               // numbers, 32 words apart
// order: null, or a permutation of the points that keeps nearby points together (the buckets of a tree): the points
// are then worked on in that order, a contiguous eighth of it per die (die_local_place)
int launch_explore_join(ExploreWorkspace* w, const JoinCopy& jc, int N, int D, int K, const int* knn_idx, int* old_idx,
                        const float* knn_dist, hipStream_t stream, const int* order = nullptr);

// explore.hip
// true when rows of K neighbours of D-dimensional points get the merge kernel that takes a point's candidates in the
// order of their lower bounds (the workspace should then be allocated with room for the bounds)
bool explore_merge_uses_bounds(int D, int K);
bool explore_join_keeps_bounds(int N, int D, int K);
int launch_explore(const float* points, const Bf16Copy* bf, const JoinCopy* jc, int N, int D, int K, int* knn_idx,
                   float* knn_dist, int* old_idx, ExploreWorkspace* ws, hipStream_t stream, bool rows_sorted = false,
                   unsigned long long* stat = nullptr,       // stat: kExploreStatWords words, or null (count_exact)
                   const int* order = nullptr,               // order: see launch_explore_join
                   bool one_tree = false);                   // the rows come from the buckets of one tree (which kernels are faster)
constexpr int kExploreStatWords = 32 * 256;

// graph_export.hip
int symmetrize_device(const int* d_idx, const float* d_dist, int N, int K, int drop_self, int* d_indptr, int* d_cols,
                      float* d_vals, long long cap, long long* nnz, hipStream_t stream);
// Count-only form of symmetrize_device (d_indptr and *nnz) whose working memory is a fixed device array of the
// library: no allocation of any kind.  At most 2^20 points and 2^25 slots.
int symmetrize_count_noalloc(const int* d_idx, int N, int K, int drop_self, int* d_indptr, long long* nnz, hipStream_t stream);
int symmetrize_host(const int* idx, const float* dist, int N, int K, int drop_self, int* indptr, int* cols, float* vals,
                    long long cap, long long* nnz);

// ann.hip
size_t ann_ws_ints(int NQ, int rec_cap);
int ann_plane_pitch(int N, int NQ, int D);
bool ann_low_wanted(int n_trees, int N, int NQ, int D);
unsigned int ann_half_share_q16(int N, int NQ, int D, int n_trees, unsigned int share_q16);
// Does the float16 copy of the queries, for their way through the trees, take less than what it gives?  (x 50 300,000 / 120,000 3 trees 1.94 -> 1.99 ms
// with it, 8 3.44 -> 3.43, 20 6.52 -> 6.37; 100,000 / 100,000 x 100 1.54 -> 1.57, 2.63 -> 2.63, 5.14 -> 4.95; 300,000 / 600,000 x 80 one tree 2.35 -> 2.46, 3
// 4.83 -> 4.77, 8 9.16 -> 8.75.)
inline bool ann_copy_pays(int n_trees, int NQ) { return (long long)n_trees * NQ >= 1500000; }
unsigned int ann_screen_share_q16(int N, int NQ, int D, int K, int n_leaves);
size_t ann_stat_words(int n_trees);
int launch_ann_ws_init(int* ws, int NQ, int rec_cap, unsigned long long* stats, int n_trees, hipStream_t stream);
int launch_ann_tree(const float* points, const float* queries, int N, int NQ, int D, int K, const int* perm, const TreeRec* recs,
                    const int* n_rec_dev, int rec_cap, int n_leaves, const JoinCopy* q_copy, const JoinCopy* p_copy,
                    int n_trees, const int* start, int* ws, float* planes, int* q_idx, float* q_dist,
                    const unsigned long long* prev, unsigned long long* stats, hipStream_t stream);
// ann_top.hip: the first levels of the trees of a batch
bool ann_top_wanted(int n_trees, int NQ, int D);
size_t ann_top_bytes(int n_trees, int D);
int launch_ann_top(const float* points, const JoinCopy& jc, int NQ, int D, int n_trees, const TreeRec* recs, const int* n_rec_dev, int rec_cap,
                   void* ws, int* start, hipStream_t stream);
int ann_forest_group(int N, int NQ, int D, int K, int MAX, int max_bucket, int rec_cap, int nb);
int launch_ann_forest(const float* points, const float* queries, int N, int NQ, int D, int K, int T, const int* perm, const TreeRec* recs,
                      const int* n_rec_dev, int rec_cap, float* planes, int* reached, int* q_idx, float* q_dist, hipStream_t stream);
int knn_ann_forest_device(int n_trees, int K, int N, int NQ, int D, int MIN, int MAX, int MAX_DEPTH, int verbose, int seed,
                          const float* d_points, const float* d_queries, int* d_qidx, float* d_qdist, float* log_forest,
                          hipStream_t stream);
int knn_ann_forest_host(int n_trees, int K, int N, int NQ, int D, int MIN, int MAX, int MAX_DEPTH, int verbose, int seed,
                        const float* points, const float* queries, int* q_idx, float* q_dist, float* log_forest);
int tree_ws_rec_cap(const TreeBatchWorkspace* w);
const int* tree_ws_n_rec(const TreeBatchWorkspace* w, int t);     // device address of the number of records of tree t
int knn_forest_device(int n_trees, int K, int N, int D, int MIN, int MAX, int MAX_DEPTH, int verbose, int seed,
                      int nnef, const float* d_points, int* d_idx, float* d_dist, float* log_forest,
                      hipStream_t stream);
int knn_forest_host(int n_trees, int K, int N, int D, int MIN, int MAX, int MAX_DEPTH, int verbose, int seed,
                    int nnef, const float* points, int* knn_idx, float* knn_dist, float* log_forest, int fresh_rows = 0);
int build_tree_host(const float* d_points, int N, int D, int MIN, int MAX, int MAX_DEPTH, int seed,
                    std::vector<int>& perm, std::vector<int>& leaf_start, std::vector<int>& leaf_size, int stats[5]);

}  // namespace rsfk
