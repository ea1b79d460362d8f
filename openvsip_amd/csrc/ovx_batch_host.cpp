// ovx_batch_host.cpp -- batches of uneven fastconv jobs (C-ABI part):
// tile-queue construction, device tables, the persistent launches over the
// LDS-resident tiles and the four-step pass launches captured once into a
// hipGraph and replayed, and the plain one-launch-per-job path it is
// compared with.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <vector>

#include "ovx_batch.hpp"
#include "ovx_batch_host.hpp"
#include "ovx_fourstep.hpp"
#include "ovx_plan.hpp"

namespace ovx {

// ---------------------------------------------------------------- shared paths
// Kernel paths (twiddle tables) per (transform length, variant), shared by
// batches, replicas and the server.
static std::mutex g_path_mu;
static std::map<std::pair<long, int>, std::unique_ptr<LineFFT>> g_paths;

// Variant the batch tiles of an (n, rows) job run: the autotuner's batch
// entry for (n, rows) when it names a tile body (an older cache file may hold
// other variant numbers), else the last candidate, a plan's own default where
// it has a tile.  Lengths without a tile run the standalone default.
int batch_variant(long n, long rows)
{
  const std::vector<int> cands = batch_candidates(n, rows);
  if (cands.empty()) return LineFFT::default_variant(n, rows);
  const int v = tuned_batch_variant(n, rows);
  return std::find(cands.begin(), cands.end(), v) != cands.end() ? v : cands.back();
}

const LineFFT *shared_path(long n, int variant, int *status)
{
  std::lock_guard<std::mutex> g(g_path_mu);
  auto it = g_paths.find({ n, variant });
  if (it != g_paths.end()) {
    *status = OVX_OK;
    return it->second.get();
  }
  std::unique_ptr<LineFFT> f(new (std::nothrow) LineFFT());
  if (!f) {
    *status = fail(OVX_ERR_NOMEM, "host allocation");
    return nullptr;
  }
  *status = f->init(n, variant);
  if (*status) return nullptr;
  const LineFFT *p = f.get();
  g_paths[{ n, variant }] = std::move(f);
  return p;
}

const LineFFT *shared_path(long n, long rows, int *status) { return shared_path(n, batch_variant(n, rows), status); }

int batch_path_of(const LineFFT &f)
{
  if (f.kind == LineFFT::HIER) return BP_HIER;
  if (f.kind == LineFFT::LDS) return BP_ROW;
  if (f.kind == LineFFT::FOURSTEP) return BP_FS;
  return 0;
}

int device_cu_count()
{
  static int cus = 0;
  if (!cus) {
    hipDeviceProp_t p;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&p, dev) != hipSuccess) return 256;
    cus = p.multiProcessorCount;
  }
  return cus;
}

// Fill `job` for a fastconv of n x rows against a prepared spectrum.
int make_batch_job(const LineFFT &f, long rows, const float2 *x, long ldx, float2 *y, long ldy, const float2 *wprep,
                   BatchJob *job)
{
  BatchJob j{};
  j.path = batch_path_of(f);
  j.n = (int)f.n;
  j.p = j.path == BP_ROW ? f.rc.p : 0;
  if (!batch_supported(j.path, j.n, j.p))
    return fail(OVX_ERR_UNSUPPORTED, "length %ld has no batch tile (path %d)", f.n, j.path);
  if (!f.tables_ready()) return fail(OVX_ERR_STATE, "length %ld: twiddle tables missing", f.n);
  if (rows > 0x7fffffff) return fail(OVX_ERR_UNSUPPORTED, "too many rows in one job");
  j.rows = rows;
  j.x = x;
  j.ldx = ldx;
  j.y = y;
  j.ldy = ldy;
  j.w = wprep;
  j.scale = 1.0f;
  if (j.path == BP_HIER) {
    j.tw0 = f.tw_outer;
    j.tw1 = f.tw_wave;
  } else if (j.path == BP_ROW) {
    j.tw0 = (const float2 *)f.tw.p;
  } else {
    j.tw0 = (const float2 *)f.tw1.p;
    j.tw1 = (const float2 *)f.tw2.p;
    j.tw2c = f.tw2c;
    j.tlo = (const float2 *)f.tlo.p;
    j.thi = (const float2 *)f.thi.p;
    j.sbits = f.sbits;
    j.tfull = (const float2 *)f.tfull.p;
    j.n1 = (int)f.n1;
    j.n2 = (int)f.n2;
  }
  *job = j;
  return OVX_OK;
}

long batch_conv_workgroups(int n1, int n2, long rows) { return rows * (n1 / batch_fs_conv_lines_per_group(n2)); }

void TileQueue::push(int job, int op, long row0, long row1, long count, int conv_rows)
{
  if (count <= 0) return;
  spans.push_back(BatchSpan{ tiles, job, op, (int)row0, (int)row1, conv_rows });
  tiles += (int)count;
}

hipError_t launch_queue(const TileQueue &q, const BatchJob *jobs, const BatchSpan *spans, hipStream_t s)
{
  if (q.tiles <= 0) return hipSuccess;
  const BatchQueue bq{ jobs, spans, (int)q.spans.size(), q.tiles };
  if (q.line == 0) return launch_batch(bq, std::min(q.tiles, device_cu_count()), s);
  if (q.line == kMidLine) return launch_batch_mid(bq, std::min(q.tiles, kBatchMidBlocksPerCu * device_cu_count()), s);
  // A chunk's first and last pass go past the caches by its bytes, as a standalone
  // call's do; rows off the 128-byte lines, which standalone calls then keep in the
  // caches (fs_whole_lines), are not told apart here.
  const bool stream = q.pass == 0 ? fs_streams_in(q.bytes) : fs_streams_out(q.bytes);
  return launch_batch_fs(q.line, q.pass, stream, bq, s);
}

void push_row_tiles(const BatchJob &j, int ji, bool fft, TileQueue &big, TileQueue &mid)
{
  const int rpt = batch_rows_per_tile(j.path, j.n, j.p);
  const int op = j.path == BP_HIER ? (fft ? BT_HIER_FFT_FWD : BT_HIER_FASTCONV) : (fft ? BT_ROW_FFT_FWD : BT_ROW_FASTCONV);
  TileQueue &q = batch_queue(j.path, j.n, j.p) == kMidQueue ? mid : big;
  q.push(ji, op, 0, j.rows, (j.rows + rpt - 1) / rpt);
}

// The passes of rows [r0, r1) of a four-step job: a fastconv's three, with
// `conv_rows` rows per middle-pass tile, or an Fftm's two.
static void push_fs_tiles(const BatchJob &j, int ji, long r0, long r1, int conv_rows, TileQueue q[kBatchQueues])
{
  const bool fft = j.ws != nullptr;
  const long rows = r1 - r0, cols = j.n2 / batch_fs_lines_per_group(j.n1);
  q[fs_queue(0, j.n1)].push(ji, fft ? BT_FS_FFT_A : BT_FS_A, r0, r1, rows * cols);
  if (fft) {
    q[fs_queue(1, j.n2)].push(ji, BT_FS_FFT_B, r0, r1, rows * (j.n1 / batch_fs_lines_per_group(j.n2)));
    return;
  }
  const long sets = (rows + conv_rows - 1) / conv_rows;
  q[fs_queue(1, j.n2)].push(ji, BT_FS_B, r0, r1, sets * (j.n1 / batch_fs_conv_lines_per_group(j.n2)), conv_rows);
  q[fs_queue(2, j.n1)].push(ji, BT_FS_C, r0, r1, rows * cols);
}

std::vector<TileQueue> chunked_fs_queues(const std::vector<BatchJob> &jobs, const std::vector<int> &order,
                                         size_t chunk_bytes)
{
  struct Part {
    int ji;
    long r0, r1;
  };
  std::vector<TileQueue> out;
  std::vector<Part> chunk;
  size_t used = 0;
  auto flush = [&] {
    long workgroups = 0; // of the fastconvs' middle pass
    for (const Part &p : chunk)
      if (!jobs[p.ji].ws) workgroups += batch_conv_workgroups(jobs[p.ji].n1, jobs[p.ji].n2, p.r1 - p.r0);
    TileQueue cq[kBatchQueues];
    for (const Part &p : chunk) push_fs_tiles(jobs[p.ji], p.ji, p.r0, p.r1, fs_conv_rows(workgroups, false), cq);
    for (int k = 1; k < kFsQueueEnd; ++k) {
      if (!cq[k].tiles) continue;
      cq[k].line = fs_queue_line(k);
      cq[k].pass = fs_queue_pass(k);
      cq[k].bytes = used;
      out.push_back(std::move(cq[k]));
    }
    chunk.clear();
    used = 0;
  };
  for (int ji : order) {
    const BatchJob &j = jobs[(size_t)ji];
    if (j.path != BP_FS) continue;
    const size_t row_bytes = (size_t)j.n * 8;
    for (long r = 0; r < j.rows;) {
      // as many rows as the chunk takes, at least one into an empty chunk
      long fit = used < chunk_bytes ? (long)((chunk_bytes - used) / row_bytes) : 0;
      if (fit == 0 && used > 0) {
        flush();
        continue;
      }
      fit = std::min(std::max(fit, 1l), j.rows - r);
      chunk.push_back(Part{ ji, r, r + fit });
      used += (size_t)fit * row_bytes;
      r += fit;
    }
  }
  if (!chunk.empty()) flush();
  return out;
}

GraphBatch::~GraphBatch() { release_graph(); }

void GraphBatch::release_graph()
{
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  exec = nullptr;
  graph = nullptr;
}

// Upload jobs and the queues' spans; capture the launches once, in queue order.
int GraphBatch::build(const std::vector<BatchJob> &jobs, const std::vector<TileQueue> &queues, hipStream_t s)
{
  release_graph();
  std::vector<BatchSpan> all;
  nlaunch = 0;
  ntiles = 0;
  for (const auto &q : queues) {
    all.insert(all.end(), q.spans.begin(), q.spans.end());
    ntiles += (size_t)q.tiles;
    if (q.tiles) ++nlaunch;
  }
  int st;
  if ((st = d_jobs.alloc(std::max<size_t>(jobs.size(), 1) * sizeof(BatchJob))) ||
      (st = d_spans.alloc(std::max<size_t>(all.size(), 1) * sizeof(BatchSpan))))
    return st;
  hipError_t e = hipSuccess;
  if (!jobs.empty()) e = hipMemcpyAsync(d_jobs.p, jobs.data(), jobs.size() * sizeof(BatchJob), hipMemcpyHostToDevice, s);
  if (e == hipSuccess && !all.empty())
    e = hipMemcpyAsync(d_spans.p, all.data(), all.size() * sizeof(BatchSpan), hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return hip_fail(e, "batch table upload");
  if (nlaunch == 0) return OVX_OK;

  hipStream_t cap;
  e = hipStreamCreateWithFlags(&cap, hipStreamNonBlocking);
  if (e != hipSuccess) return hip_fail(e, "capture stream");
  e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
  if (e == hipSuccess) {
    const BatchSpan *spans = (const BatchSpan *)d_spans.p;
    for (const auto &q : queues) {
      if (e == hipSuccess) e = launch_queue(q, (const BatchJob *)d_jobs.p, spans, cap);
      spans += q.spans.size();
    }
    hipError_t e2 = hipStreamEndCapture(cap, &graph);
    if (e == hipSuccess) e = e2;
  }
  if (e == hipSuccess) e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipStreamDestroy(cap);
  if (e != hipSuccess) {
    release_graph();
    return hip_fail(e, "batch graph capture");
  }
  return OVX_OK;
}

int GraphBatch::launch(hipStream_t s) const
{
  if (nlaunch == 0) return OVX_OK;
  hipError_t e = hipGraphLaunch(exec, s);
  if (e != hipSuccess) return hip_fail(e, "batch graph launch");
  return OVX_OK;
}

} // namespace ovx

using namespace ovx;

// ---------------------------------------------------------------- C-ABI
struct ovx_batch_s {
  struct HostJob {
    long n, rows;
    const void *x;
    long ldx;
    int replica;
    void *y;
    long ldy;
  };
  std::vector<HostJob> jobs;
  std::vector<BatchJob> djobs;
  std::vector<const LineFFT *> paths;
  std::vector<const float2 *> preps;
  GraphBatch gb;
  bool committed = false;
};

extern "C" int ovx_batch_create(ovx_batch *b)
{
  if (!b) return fail(OVX_ERR_INVALID, "null batch pointer");
  *b = new (std::nothrow) ovx_batch_s();
  if (!*b) return fail(OVX_ERR_NOMEM, "host allocation");
  return OVX_OK;
}

extern "C" int ovx_batch_destroy(ovx_batch b)
{
  if (!b) return fail(OVX_ERR_INVALID, "null batch");
  delete b;
  return OVX_OK;
}

extern "C" int ovx_batch_add_fastconv(ovx_batch b, long n, long rows, const void *x, long ldx, int replica, void *y,
                                      long ldy)
{
  if (!b) return fail(OVX_ERR_INVALID, "null batch");
  if (b->committed) return fail(OVX_ERR_STATE, "batch already committed");
  if (!x || !y) return fail(OVX_ERR_INVALID, "null data pointer");
  if (n < 1 || rows < 0) return fail(OVX_ERR_INVALID, "bad job size");
  if (rows > 1 && (ldx < n || ldy < n)) return fail(OVX_ERR_INVALID, "row stride shorter than n");
  b->jobs.push_back(ovx_batch_s::HostJob{ n, rows, x, ldx, replica, y, ldy });
  return OVX_OK;
}

extern "C" int ovx_batch_commit(ovx_batch b, void *stream)
{
  if (!b) return fail(OVX_ERR_INVALID, "null batch");
  if (b->committed) return fail(OVX_ERR_STATE, "batch already committed");
  hipStream_t s = (hipStream_t)stream;
  b->djobs.clear();
  b->paths.clear();
  b->preps.clear();
  // tile bodies for the (n, rows) keys the autotuner has not seen yet
  if (!getenv("OVX_NO_BATCH_TUNE")) {
    for (size_t i = 0; i < b->jobs.size(); ++i) {
      const auto &h = b->jobs[i];
      if (batch_candidates(h.n, h.rows).size() > 1 && tuned_batch_variant(h.n, h.rows) < 0) {
        int st = autotune_batch(h.n, h.rows, nullptr, nullptr);
        if (st) return st;
      }
    }
  }
  for (size_t i = 0; i < b->jobs.size(); ++i) {
    const auto &h = b->jobs[i];
    int st;
    const LineFFT *f = shared_path(h.n, h.rows, &st);
    if (!f) return st;
    const float2 *prep = nullptr;
    long rn = 0;
    if ((st = replica_prepared(h.replica, &prep, &rn, f))) return st;
    if (rn != h.n) return fail(OVX_ERR_INVALID, "replica %d has length %ld, job %zu has %ld", h.replica, rn, i, h.n);
    BatchJob j;
    if ((st = make_batch_job(*f, h.rows, (const float2 *)h.x, h.ldx, (float2 *)h.y, h.ldy, prep, &j))) return st;
    b->djobs.push_back(j);
    b->paths.push_back(f);
    b->preps.push_back(prep);
  }
  // largest jobs first inside each queue
  std::vector<int> order(b->djobs.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
  std::stable_sort(order.begin(), order.end(), [&](int a, int c) { return b->djobs[a].n > b->djobs[c].n; });
  // Launch order: the two persistent launches over the LDS-resident tiles
  // (1024-thread rows, then the shorter ones), then the four-step jobs' rows
  // in Infinity-Cache-sized chunks, one launch per non-empty (pass, line
  // length) queue of a chunk, in pass order.
  std::vector<TileQueue> queues(2);
  queues[1].line = kMidLine;
  for (int i : order)
    if (b->djobs[i].path != BP_FS) push_row_tiles(b->djobs[i], i, false, queues[0], queues[1]);
  for (auto &fq : chunked_fs_queues(b->djobs, order, kFsChunkBytes)) queues.push_back(std::move(fq));
  int st = b->gb.build(b->djobs, queues, s);
  if (st) return st;
  b->committed = true;
  return OVX_OK;
}

extern "C" int ovx_batch_exec(ovx_batch b, void *stream)
{
  if (!b) return fail(OVX_ERR_INVALID, "null batch");
  if (!b->committed) return fail(OVX_ERR_STATE, "batch not committed");
  return b->gb.launch((hipStream_t)stream);
}

extern "C" int ovx_batch_exec_plain(ovx_batch b, void *stream)
{
  if (!b) return fail(OVX_ERR_INVALID, "null batch");
  if (!b->committed) return fail(OVX_ERR_STATE, "batch not committed");
  hipStream_t s = (hipStream_t)stream;
  for (size_t i = 0; i < b->jobs.size(); ++i) {
    const auto &h = b->jobs[i];
    int st = b->paths[i]->fastconv_prepared((const float2 *)h.x, h.ldx, b->preps[i], (float2 *)h.y, h.ldy, h.rows, s);
    if (st) return st;
  }
  return OVX_OK;
}

extern "C" long ovx_batch_tiles(ovx_batch b)
{
  if (!b) return -1;
  return (long)b->gb.ntiles;
}

extern "C" int ovx_batch_launches(ovx_batch b)
{
  if (!b) return -1;
  return b->gb.nlaunch;
}

extern "C" int ovx_batch_job_variant(ovx_batch b, long job)
{
  if (!b || !b->committed || job < 0 || job >= (long)b->paths.size()) return -1;
  return b->paths[(size_t)job]->variant;
}
