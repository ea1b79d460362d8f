// ovx_batch.hpp -- persistent tile-queue kernel for batches of uneven jobs.
#pragma once
#include <hip/hip_runtime.h>

#include "ovx_ols.hpp"

namespace ovx {

// Kernel path of one job (which device body its tiles run).
enum BatchPath { BP_HIER = 1, BP_ROW = 2, BP_FS = 3 };
// Tile operations.
enum BatchOp {
  BT_HIER_FASTCONV = 1, // a tile's worth of rows of a hierarchical-path job
  BT_ROW_FASTCONV = 2,  // the same of a register-Stockham-path job
  BT_FS_A = 3,          // four-step fastconv pass 1: a column group of a row
  BT_FS_B = 4,          // pass 2: a line group of conv_rows rows
  BT_FS_C = 5,          // pass 3: a column group of a row
  BT_HIER_FFT_FWD = 6,  // forward Fftm rows of a hierarchical-path job
  BT_ROW_FFT_FWD = 7,   // forward Fftm rows of a register-Stockham-path job
  BT_FS_FFT_A = 8,      // four-step forward Fftm pass 1: x -> workspace
  BT_FS_FFT_B = 9,      // pass 2: workspace -> y (natural order)
  BT_OLS = 10           // a tile's worth of overlap-save segments
};

struct alignas(16) BatchJob { // spans may follow a table of jobs
  int path;
  int n;
  int p;             // ROW: values per thread
  long rows;
  const float2 *x;
  long ldx;
  float2 *y;
  long ldy;
  const float2 *w;   // prepared spectrum (path layout, 1/n folded in)
  const float2 *tw0; // HIER: outer table; ROW: engine table; FS: n1 line table
  const float2 *tw1; // HIER: 1024-point wave table; FS: n2 line table
  const float2 *tw2c; // FS: n2 line table of a fastconv's middle pass
  const float2 *tlo, *thi;
  int sbits;
  const float2 *tfull; // FS: full twiddle table or null
  int n1, n2;
  float scale;       // forward Fftm scale
  float2 *ws;        // four-step Fftm workspace (rows x n)
  OlsArgs ols;       // overlap-save segment parameters
  int ols_len;       // segment length L
};

// Consecutive tiles of a queue: one operation over rows (or segments) [row0,
// row1) of one job.  A workgroup finds the span of its tile and works out rows
// and line group itself.  The host wrote and copied a table of the tiles, 160 KB
// for 32 mixed requests: with that, a copy per queue and a graph that launched
// empty queues too the server took 340 us for them, now 262.
struct alignas(16) BatchSpan {
  int tile0; // first tile in the queue
  int job;
  int op;
  int row0, row1;
  int conv_rows; // BT_FS_B: rows per tile
};

// Tile queues of a batch: queue 0 holds the LDS-resident tiles (rows,
// overlap-save segments) of the 1024-thread persistent launch, queue
// kMidQueue those of the 512-thread one; the four-step passes get one queue
// per (pass, line length 256 or 512), queues 1 .. kFsQueueEnd - 1, run in
// pass order, one line group per workgroup.
constexpr int kBatchQueues = 8;
constexpr int kFsQueueEnd = 7;
constexpr int kMidQueue = 7;
constexpr int kFsLines[2] = { 256, 512 };
inline int fs_queue(int pass, int n_line) { return 1 + 2 * pass + (n_line == 512 ? 1 : 0); }
inline int fs_queue_line(int q) { return kFsLines[(q - 1) % 2]; }

// X(N, P): the register-Stockham tile bodies, N points with P values per
// thread.  A length has the configurations that a fastconv plan of it runs by
// default (row_pick), so that a job gives the same floats in a batch as alone:
// at 1024 points that is the hierarchical body (16 values a thread, the same
// operations).  6144 and 12288 points, whose plans run 24 values a thread, have
// 12, which fit the 128-VGPR budget of both kernels.  16 values a thread for
// every power of two / the plans' own: 47 jobs of 512 points 20.2 / 20.1 us, 50
// of 2048 60.5 / 72.3, 47 of 256 13.2 / 14.6, the 512-job benchmark 5.93 / 5.95
// ms.
#define OVX_ROW_TILES(X)                                                                        \
  X(256, 4) X(512, 8) X(2048, 16) X(2048, 8) X(4096, 16) X(3072, 12) X(6144, 12) X(12288, 12)
constexpr bool batch_row_tile(int n, int p)
{
#define X(N, P) \
  if (n == N && p == P) return true;
  OVX_ROW_TILES(X)
#undef X
  return false;
}

// Threads per persistent workgroup.  Rows whose line takes at most 512
// threads (every LDS-resident length up to 8192; overlap-save segments up to
// 8192) run in the 512-thread launch, two workgroups per CU, so that one
// workgroup's loads and stores overlap the other's arithmetic; 12288 and
// 16384 need the 1024-thread workgroup, one per CU.
constexpr int kBatchThreads = 1024;
constexpr int kBatchMidThreads = 512;
constexpr int batch_line_threads(int path, int n, int p) // threads of one row's transform
{
  return path == BP_HIER ? 64 * (n / 1024) : n / p;
}
constexpr bool batch_mid_routed(int path, int n, int p) { return batch_line_threads(path, n, p) <= kBatchMidThreads; }
constexpr bool batch_ols_mid_routed(int L) { return L / 16 <= kBatchMidThreads; }
inline int batch_queue(int path, int n, int p) { return batch_mid_routed(path, n, p) ? kMidQueue : 0; }
inline int batch_ols_queue(int L) { return batch_ols_mid_routed(L) ? kMidQueue : 0; }
int batch_rows_per_tile(int path, int n, int p);
int batch_ols_segments_per_tile(int L);
int batch_fs_lines_per_group(int n_line); // C of a four-step group of lines of length n_line
int batch_fs_conv_lines_per_group(int n_line); // of a fastconv's middle pass
bool batch_supported(int path, int n, int p);

// A queue in device memory: spans by first tile, `tiles` tiles in all.
struct BatchQueue {
  const BatchJob *jobs;
  const BatchSpan *spans;
  int nspans, tiles;
};
// One persistent launch over a queue of LDS-resident tiles: `grid` workgroups,
// workgroup w taking tiles w, w + grid, ...
hipError_t launch_batch(const BatchQueue &q, int grid, hipStream_t s);
// The same over the 512-thread queue (two workgroups per CU).
hipError_t launch_batch_mid(const BatchQueue &q, int grid, hipStream_t s);
constexpr int kBatchMidBlocksPerCu = 2;
// Four-step pass `pass` (0, 1, 2) over a queue of line length n_line (256 or
// 512), one tile per workgroup; `stream`: a column pass with non-temporal access
// (fs_streams_in, fs_streams_out).
hipError_t launch_batch_fs(int n_line, int pass, bool stream, const BatchQueue &q, hipStream_t s);
inline int fs_queue_pass(int q) { return (q - 1) / 2; }

} // namespace ovx
