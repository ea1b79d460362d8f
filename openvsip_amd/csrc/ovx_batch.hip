// ovx_batch.hip -- persistent launches over (instance, rows) tile queues.
//
// A batch of uneven fast-convolution jobs (different N and row counts) is cut
// into tiles: a few whole rows of an LDS-resident job (one workgroup's worth
// of threads), or one column/line group of one row of a four-step job.  The
// LDS-resident tiles run in two persistent launches, one of 1024-thread
// workgroups (one per CU; rows of 12288 and 16384 points) and one of
// 512-thread workgroups (two per CU; every shorter row), whose fixed grids
// stride over their queues, workgroup w taking tiles w, w + grid, ...  Every
// tile runs the same device body as the standalone kernel of its variant, so a
// job's result is bitwise the same alone and in a batch.  Four-step jobs need their
// three passes in order; each pass is a launch of its own over its queue.  A
// batch's launches are captured in one hipGraph; the server issues its own.
#include "ovx_batch.hpp"
#include "ovx_fs_dev.hpp"
#include "ovx_hier_dev.hpp"
#include "ovx_ols_dev.hpp"
#include "ovx_row_dev.hpp"

namespace ovx {

// LDS of the largest tile of each persistent launch.  1024 threads: 64
// register-Stockham rows of 256 (17408 float2), four-step groups
// 4 x 16 x 273.  512 threads: every tile routed there (rows of up to 8192
// points, overlap-save segments) needs 16 lines' worth of 512 threads,
// 16 * 512 * 33 / 32 = 8448 float2 (67.6 KB: two workgroups per CU).  Every
// tile function checks its need against its launch's figure.
constexpr int kBatchLds = 4 * 16 * 273 > 17408 ? 4 * 16 * 273 : 17408;
constexpr int kBatchMidLds = 8448;
template <int NT>
struct BatchLds {
  static constexpr int value = NT == kBatchThreads ? kBatchLds : kBatchMidLds;
};

// A tile function's thread number, taken anew for each tile: what it computes
// from it (LDS and memory offsets, table entries) cannot be moved out of the
// loop over tiles, where the offsets of every size at once would not fit the
// registers.  (Inlined without this the two kernels keep 268 and 1048 bytes a
// thread in scratch memory; as functions that are called, the tile functions
// each save and restore up to 49 registers a tile: 24 uneven instances,
// 694 MB, 356 us called and 352 inlined.)
__device__ __forceinline__ int tile_thread()
{
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Tile `ti` of a queue: its span and its number in the span.  (Jobs and spans
// are kernel arguments of their own, __restrict__: only so are the descriptor's
// fields read by scalar loads, and the kernels free of scratch memory.)  The lanes of each
// wave read 64 spans at once.
struct Tile {
  int job, op, row0, row1, conv_rows, k;
};
__device__ __forceinline__ Tile find_tile(const BatchSpan *__restrict__ spans, int nspans, int ti)
{
  const int lane = tile_thread() & 63;
  for (int base = 0;; base += 64) {
    int4 a = make_int4(0x7fffffff, 0, 0, 0);
    int2 b = make_int2(0, 0);
    if (base + lane < nspans) {
      const BatchSpan *sp = spans + base + lane;
      a = *(const int4 *)sp;
      b = *(const int2 *)&sp->row1;
    }
    const int n = __popcll(__ballot(a.x <= ti)); // the spans that begin here or before
    if (n == 64 && base + 64 < nspans && spans[base + 64].tile0 <= ti) continue;
    auto of = [&](int v) { return __builtin_amdgcn_readlane(v, n - 1); };
    return Tile{ of(a.y), of(a.z), of(a.w), of(b.x), of(b.y), ti - of(a.x) };
  }
}

// Tile functions of a workgroup of NT threads: NT / (threads of a row) rows
// (or overlap-save segments) per tile.
template <int NT, int N>
__device__ __forceinline__ void tile_hier_fastconv(const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  using H = Hier<N>;
  const int row0 = tile.row0 + tile.k * (NT / H::TR);
  static_assert(NT % H::TR == 0 && (NT / H::TR) * H::LROW <= BatchLds<NT>::value, "tile LDS");
  HierArgs a{};
  a.x = j.x;
  a.ldx = j.ldx;
  a.y = j.y;
  a.ldy = j.ldy;
  a.w = j.w;
  a.rows = j.rows;
  a.tw_outer = j.tw0;
  a.tw_wave = j.tw1;
  const int tid = tile_thread();
  const int lrow = tid / H::TR;
  const int t = tid % H::TR;
  // a tile of one row is only made for a row that exists
  hier_fastconv_body<N, NT / H::TR == 1, false, N == 16384>(a, row0, lrow, t, lds + lrow * H::LROW);
}

template <int NT, int N>
__device__ __forceinline__ void tile_hier_fwd(const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  using H = Hier<N>;
  const int row0 = tile.row0 + tile.k * (NT / H::TR);
  static_assert(NT % H::TR == 0 && (NT / H::TR) * H::LROW <= BatchLds<NT>::value, "tile LDS");
  HierArgs a{};
  a.x = j.x;
  a.ldx = j.ldx;
  a.y = j.y;
  a.ldy = j.ldy;
  a.rows = j.rows;
  a.tw_outer = j.tw0;
  a.tw_wave = j.tw1;
  a.scale = j.scale;
  const int tid = tile_thread();
  const int lrow = tid / H::TR;
  const int t = tid % H::TR;
  hier_fwd_body<N>(a, row0, lrow, t, lds + lrow * H::LROW);
}

template <int NT, int N, int P>
__device__ __forceinline__ void tile_row_fastconv(const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  using E = Engine<N, P, line_in_wave(N / P)>;
  const int row0 = tile.row0 + tile.k * (NT / E::T);
  static_assert(NT % E::T == 0 && (NT / E::T) * E::LROW <= BatchLds<NT>::value, "tile LDS");
  const int tid = tile_thread();
  const int lrow = tid / E::T;
  const int t = tid % E::T;
  // 3 * 2^k rows, one or two a workgroup, load faster past the caches (19 jobs,
  // 184 MB, half of it 6144 and 12288: 84.0 us ordinary, 81.5 so), powers of two
  // the ordinary way (15 jobs, 222 MB: 108.1 and 110.0)
  row_fastconv_body<N, P, P == 12>(j.x, j.ldx, j.w, 0, j.y, j.ldy,
                          j.rows, j.tw0, 1.0f, row0, lrow, t, lds + lrow * E::LROW);
}

template <int NT, int N, int P>
__device__ __forceinline__ void tile_row_fwd(const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  using E = Engine<N, P, line_in_wave(N / P)>;
  const int row0 = tile.row0 + tile.k * (NT / E::T);
  static_assert(NT % E::T == 0 && (NT / E::T) * E::LROW <= BatchLds<NT>::value, "tile LDS");
  const int tid = tile_thread();
  const int lrow = tid / E::T;
  const int t = tid % E::T;
  row_fft_body<N, P, -1>(j.x, j.ldx, j.y, j.ldy, j.rows,
                         j.tw0, j.scale, row0, lrow, t, lds + lrow * E::LROW);
}

// Overlap-save segments seg0, seg0 + 1, ... (NT / (L/16) of them per tile);
// those past the last store nothing.
template <int NT, int L>
__device__ __forceinline__ void tile_ols(const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  const OlsArgs a = j.ols;
  constexpr int T = L / 16;
  static_assert(NT % T == 0 && (NT / T) * Engine<L, 16>::LROW <= BatchLds<NT>::value, "tile LDS");
  const int tid = tile_thread();
  const int t = tid % T;
  const int copy = tid / T;
  ols_body<L, 16>(a, tile.row0 + tile.k * (NT / T), copy, t, lds + copy * Engine<L, 16>::LROW);
}

int batch_ols_segments_per_tile(int L)
{
  return (batch_ols_mid_routed(L) ? kBatchMidThreads : kBatchThreads) / (L / 16);
}

template <typename J>
__device__ __forceinline__ FsArgs fs_args_of(const J &j)
{
  FsArgs a{};
  a.n1 = j.n1;
  a.n2 = j.n2;
  a.nbig = j.n;
  a.tw1 = j.tw0;
  a.tw2 = j.tw1;
  a.tw2c = j.tw2c;
  a.tlo = j.tlo;
  a.thi = j.thi;
  a.sbits = j.sbits;
  a.tfull = j.tfull;
  a.wp = j.w;
  a.ldwp = 0;
  a.scale = 1.0f;
  return a;
}

// Whether a tile of (path, n) -- or an overlap-save segment of length L --
// runs in the launch of NT threads: the host routes each to exactly one of
// the two (batch_queue, batch_ols_queue), and the other launch's switch has
// no code for it.
template <int NT, int PATH, int N, int P = 0>
constexpr bool runs_in() { return batch_mid_routed(PATH, N, P) == (NT == kBatchMidThreads); }
template <int NT, int L>
constexpr bool ols_runs_in() { return batch_ols_mid_routed(L) == (NT == kBatchMidThreads); }
static_assert(batch_mid_routed(BP_HIER, 8192, 0) && !batch_mid_routed(BP_HIER, 16384, 0) &&
                  batch_mid_routed(BP_ROW, 6144, 12) && !batch_mid_routed(BP_ROW, 12288, 12) &&
                  batch_ols_mid_routed(8192) && !batch_ols_mid_routed(16384),
              "rows of 12288 and 16384 points (and segments of 16384) need the 1024-thread launch, all others "
              "run in the 512-thread one");

template <int NT, int N>
__device__ __forceinline__ void run_hier(bool fwd_only, const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  if constexpr (runs_in<NT, BP_HIER, N>()) {
    if (fwd_only) tile_hier_fwd<NT, N>(j, tile, lds);
    else tile_hier_fastconv<NT, N>(j, tile, lds);
  }
}
template <int NT, int N, int P>
__device__ __forceinline__ void run_row(bool fwd_only, const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  if constexpr (runs_in<NT, BP_ROW, N, P>()) {
    if (fwd_only) tile_row_fwd<NT, N, P>(j, tile, lds);
    else tile_row_fastconv<NT, N, P>(j, tile, lds);
  }
}
template <int NT, int L>
__device__ __forceinline__ void run_ols(const BatchJob &j, const Tile &tile, lds_ptr lds)
{
  if constexpr (ols_runs_in<NT, L>()) tile_ols<NT, L>(j, tile, lds);
}

// The persistent loop of a launch of NT threads: workgroup w takes tiles w,
// w + grid, ...: consecutive tiles (rows of one job, jobs of like size next to
// each other) go to different workgroups, so each gets a like share of the
// queue (a shared atomic counter cost each workgroup a cross-XCD round trip
// per tile).
template <int NT>
__device__ __forceinline__ void batch_loop(const BatchJob *__restrict__ jobs, const BatchSpan *__restrict__ spans,
                                           int nspans, int tiles, float2 *lds_mem)
{
  const lds_ptr lds = as_lds(lds_mem);
  for (int ti = blockIdx.x; ti < tiles; ti += gridDim.x) {
    const Tile tile = find_tile(spans, nspans, ti);
    const BatchJob &j = jobs[tile.job]; // the same for every lane: scalar loads
    switch (tile.op) {
    case BT_HIER_FASTCONV:
    case BT_HIER_FFT_FWD: {
      const bool fwd = tile.op == BT_HIER_FFT_FWD;
      switch (j.n) {
      case 1024: run_hier<NT, 1024>(fwd, j, tile, lds); break;
      case 2048: run_hier<NT, 2048>(fwd, j, tile, lds); break;
      case 4096: run_hier<NT, 4096>(fwd, j, tile, lds); break;
      case 8192: run_hier<NT, 8192>(fwd, j, tile, lds); break;
      case 16384: run_hier<NT, 16384>(fwd, j, tile, lds); break;
      default: break;
      }
      break;
    }
    case BT_ROW_FASTCONV:
    case BT_ROW_FFT_FWD: {
      const bool fwd = tile.op == BT_ROW_FFT_FWD;
      switch (j.n + j.p) { // lengths are multiples of 256, values per thread fewer
#define X(N, P) \
      case N + P: run_row<NT, N, P>(fwd, j, tile, lds); break;
      OVX_ROW_TILES(X)
#undef X
      default: break;
      }
      break;
    }
    case BT_OLS:
      switch (j.ols_len) {
      case 1024: run_ols<NT, 1024>(j, tile, lds); break;
      case 2048: run_ols<NT, 2048>(j, tile, lds); break;
      case 4096: run_ols<NT, 4096>(j, tile, lds); break;
      case 8192: run_ols<NT, 8192>(j, tile, lds); break;
      case 16384: run_ols<NT, 16384>(j, tile, lds); break;
      default: break;
      }
      break;
    default: break; // four-step tiles run in k_batch_fs
    }
    __syncthreads(); // LDS reuse by the next tile
  }
}

__global__ __launch_bounds__(kBatchThreads) void k_batch(
    const BatchJob *__restrict__ jobs, const BatchSpan *__restrict__ spans, int nspans, int tiles)
{
  __shared__ float2 lds_mem[kBatchLds];
  batch_loop<kBatchThreads>(jobs, spans, nspans, tiles, lds_mem);
}

// Two workgroups per CU: four waves per SIMD (the second launch bound is
// waves per SIMD: 128 VGPRs) and
// 2 x 67.6 KB of LDS.
__global__ __launch_bounds__(kBatchMidThreads, kBatchMidBlocksPerCu * kBatchMidThreads / 256) void k_batch_mid(
    const BatchJob *__restrict__ jobs, const BatchSpan *__restrict__ spans, int nspans, int tiles)
{
  __shared__ float2 lds_mem[kBatchMidLds];
  batch_loop<kBatchMidThreads>(jobs, spans, nspans, tiles, lds_mem);
}

hipError_t launch_batch(const BatchQueue &q, int grid, hipStream_t s)
{
  hipLaunchKernelGGL(k_batch, dim3(grid), dim3(kBatchThreads), 0, s, q.jobs, q.spans, q.nspans, q.tiles);
  return hipGetLastError();
}

hipError_t launch_batch_mid(const BatchQueue &q, int grid, hipStream_t s)
{
  hipLaunchKernelGGL(k_batch_mid, dim3(grid), dim3(kBatchMidThreads), 0, s, q.jobs, q.spans, q.nspans, q.tiles);
  return hipGetLastError();
}

// ---------------------------------------------------------------- four-step passes
// Row and line group of tile k of a column pass over rows [row0, row1): eight
// rows at a time, their tiles in turn, so that the workgroups of a row land on
// one XCD (the standalone passes' placement).
__device__ __forceinline__ void fs_col_tile(const Tile &t, int groups, int &row, int &group)
{
  const int rows = t.row1 - t.row0, whole = rows & ~7;
  if (t.k < whole * groups) {
    const int e = t.k / 8;
    row = t.row0 + e / groups * 8 + t.k % 8;
    group = e % groups;
  } else {
    const int e = t.k - whole * groups, left = rows - whole;
    row = t.row0 + whole + e % left;
    group = e / left;
  }
}

// One line group per workgroup (the standalone kernels' shape; four waves per
// SIMD, the occupancy the LDS of L = 256 groups allows), so co-resident
// workgroups run independently and overlap their loads with other groups'
// arithmetic.  The job descriptor is read from global memory (uniform per tile,
// scalar loads).
template <int L, int PASS, bool STREAM>
__global__ __launch_bounds__(FsCfg<L>::NT, 4) void k_batch_fs(
    const BatchJob *__restrict__ jobs, const BatchSpan *__restrict__ spans, int nspans)
{
  using F = FsCfg<L>;
  constexpr int CC = F::NT / FsConv<L>::T; // lines of a middle-pass tile
  static_assert(CC * FsConv<L>::LROW <= F::LDS, "middle pass LDS");
  __shared__ float2 lds[F::LDS];
  const int tid = (int)threadIdx.x;
  const Tile tile = find_tile(spans, nspans, blockIdx.x);
  const BatchJob &j = jobs[tile.job];
  FsArgs a = fs_args_of(j);
  int row, group;
  if constexpr (PASS == 0) { // column FFT: fastconv x -> y, Fftm x -> workspace
    const bool fft = tile.op == BT_FS_FFT_A;
    a.in = j.x;
    a.ld_in = j.ldx;
    a.out = fft ? j.ws : j.y;
    a.ld_out = fft ? (long)j.n : j.ldy;
    fs_col_tile(tile, j.n2 / F::C, row, group);
    fs_col_body<L, F::P, F::C, -1, false, false, STREAM>(a, row, group, tid, lds);
  } else if constexpr (PASS == 1) {
    if (tile.op == BT_FS_B) { // fastconv: middle pass in place on y
      a.in = j.y;
      a.ld_in = j.ldy;
      a.out = j.y;
      a.ld_out = j.ldy;
      const int groups = j.n1 / CC;
      row = tile.row0 + tile.k / groups * tile.conv_rows;
      fs_conv_body<L, CC>(a, row, min(tile.conv_rows, tile.row1 - row), 1, tile.k % groups, tid, lds);
    } else { // Fftm: workspace -> y in natural order, scaled
      a.scale = j.scale;
      a.in = j.ws;
      a.ld_in = j.n;
      a.out = j.y;
      a.ld_out = j.ldy;
      const int groups = j.n1 / F::C;
      fs_row_body<L, F::P, F::C, -1>(a, tile.row0 + tile.k / groups, tile.k % groups, tid, lds);
    }
  } else { // fastconv pass 3: column IFFT in place on y
    a.in = j.y;
    a.ld_in = j.ldy;
    a.out = j.y;
    a.ld_out = j.ldy;
    fs_col_tile(tile, j.n2 / F::C, row, group);
    fs_col_body<L, F::P, F::C, +1, false, false, STREAM, STREAM>(a, row, group, tid, lds);
  }
}

template <int L, int PASS, bool STREAM>
static hipError_t launch_fs(const BatchQueue &q, hipStream_t s)
{
  hipLaunchKernelGGL((k_batch_fs<L, PASS, STREAM>), dim3(q.tiles), dim3(FsCfg<L>::NT), 0, s, q.jobs, q.spans,
                     q.nspans);
  return hipGetLastError();
}

template <int L>
static hipError_t launch_fs_pass(int pass, bool stream, const BatchQueue &q, hipStream_t s)
{
  if (pass == 0) return stream ? launch_fs<L, 0, true>(q, s) : launch_fs<L, 0, false>(q, s);
  if (pass == 1) return launch_fs<L, 1, false>(q, s);
  return stream ? launch_fs<L, 2, true>(q, s) : launch_fs<L, 2, false>(q, s);
}

hipError_t launch_batch_fs(int n_line, int pass, bool stream, const BatchQueue &q, hipStream_t s)
{
  if (q.tiles <= 0) return hipSuccess;
  if (n_line == 256) return launch_fs_pass<256>(pass, stream, q, s);
  if (n_line == 512) return launch_fs_pass<512>(pass, stream, q, s);
  return hipErrorInvalidValue;
}

bool batch_supported(int path, int n, int p)
{
  if (path == BP_HIER) return hier_supported(n);
  if (path == BP_ROW) return batch_row_tile(n, p);
  if (path == BP_FS) return n == 65536 || n == 131072 || n == 262144;
  return false;
}

int batch_rows_per_tile(int path, int n, int p)
{
  if (path != BP_HIER && path != BP_ROW) return 1;
  return (batch_mid_routed(path, n, p) ? kBatchMidThreads : kBatchThreads) / batch_line_threads(path, n, p);
}

int batch_fs_lines_per_group(int n_line)
{
  if (n_line == 256) return FsCfg<256>::C;
  if (n_line == 512) return FsCfg<512>::C;
  return 0;
}

int batch_fs_conv_lines_per_group(int n_line)
{
  if (n_line == 256) return FsCfg<256>::NT / FsConv<256>::T;
  if (n_line == 512) return FsCfg<512>::NT / FsConv<512>::T;
  return 0;
}

} // namespace ovx
