// ovx_batch_host.hpp -- host-side pieces shared by batches and the server.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "ovx_batch.hpp"
#include "ovx_plan.hpp"

namespace ovx {

// Kernel path (and its twiddles) of length n in `variant`, created on first
// use and shared.  The (n, rows) form takes batch_variant(n, rows).
const LineFFT *shared_path(long n, int variant, int *status);
const LineFFT *shared_path(long n, long rows, int *status);
// Variant of the tile bodies an (n, rows) job runs in a batch or the server:
// the autotuner's batch entry, else the default.
int batch_variant(long n, long rows);
// Batch tile autotuner (ovx_tune.cpp): the variants whose device body a
// batch tile can run for length n, the cached choice for (n, rows) or -1,
// and the tuning itself (records the choice).
std::vector<int> batch_candidates(long n, long rows);
int tuned_batch_variant(long n, long rows);
int autotune_batch(long n, long rows, int *best_variant, double *best_us);
int batch_path_of(const LineFFT &f);
int device_cu_count();
int make_batch_job(const LineFFT &f, long rows, const float2 *x, long ldx, float2 *y, long ldy, const float2 *wprep,
                   BatchJob *job);
// Middle-pass workgroups of one row each that `rows` rows of a four-step job
// of n = n1 * n2 points make (fs_conv_rows turns their sum over a launch into
// rows per tile).
long batch_conv_workgroups(int n1, int n2, long rows);
// Prepared spectrum of a resident replica in the layout of path `f`.
int replica_prepared(int id, const float2 **prep, long *n, const LineFFT *f);

// One launch of a batch: a persistent kernel over LDS-resident tiles
// (line == 0: the 1024-thread one, line == kMidLine: the 512-thread one) or
// four-step pass `pass` over lines of length `line`.
constexpr int kMidLine = -1;
struct TileQueue {
  int line = 0;
  int pass = 0;
  std::vector<BatchSpan> spans;
  int tiles = 0;
  size_t bytes = 0; // four-step: rows of the chunk
  // `count` tiles of operation `op` over rows [row0, row1) of job `job`
  void push(int job, int op, long row0, long row1, long count, int conv_rows = 0);
};
// Launch queue `q` whose spans are at `spans` in device memory.
hipError_t launch_queue(const TileQueue &q, const BatchJob *jobs, const BatchSpan *spans, hipStream_t s);
// Append job `ji`, whose rows are LDS-resident, to the queue of its persistent
// launch: fastconv rows, or a forward Fftm's.
void push_row_tiles(const BatchJob &j, int ji, bool fft, TileQueue &big, TileQueue &mid);

// Four-step passes of a batch in chunks of about kFsChunkBytes of rows
// (rows of one job may fall into different chunks), each chunk's three passes
// launched back to back: a chunk's matrix then stays in the 256 MB Infinity
// Cache from one pass to the next, X and the result passing it by
// (fs_streams_in, fs_streams_out).  Chunks of 96 / 128 / 160 / 192 / 224 / 256 /
// 512 MB, us: 400 rows of 65536 247 / 228 / 230 / 222 / 207 / 212 / 209, 800 rows
// 467 / 437 / 425 / 422 / 402 / 413 / 431, 2000 rows 1118 / 1050 / 1032 / 1011 /
// 995 / 1002 / 1072, 240 rows of 262144 567 / 543 / 524 / 532 / 538 / 527 / 563.
// (224 MB is the fastest on three of the four lists; with 192, 400 rows of 65536
// stay two chunks, as the tests of a batch's launches count them.)
constexpr size_t kFsChunkBytes = (size_t)192 << 20;
// Four-step queues (in launch order) of jobs order[0], order[1], ... that
// take the four-step path; a job with a workspace is a forward Fftm.
std::vector<TileQueue> chunked_fs_queues(const std::vector<BatchJob> &jobs, const std::vector<int> &order,
                                         size_t chunk_bytes);

// Device job/span tables plus the batch's launches (queues in launch order)
// captured in one hipGraph.
struct GraphBatch {
  DevBuf d_jobs, d_spans;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int nlaunch = 0;
  size_t ntiles = 0;
  ~GraphBatch();
  void release_graph();
  int build(const std::vector<BatchJob> &jobs, const std::vector<TileQueue> &queues, hipStream_t s);
  int launch(hipStream_t s) const;
};

} // namespace ovx
