// util.hip — exclusive prefix sums (one, two or four launches by size; deterministic) and small helpers.
#include "swr_internal.h"
#include "swr_device.h"

#include <mutex>

namespace {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 4;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

std::mutex g_err_mu;
std::string g_err;

// Block-wide exclusive scan of one value per thread; returns the exclusive
// prefix and writes the block total.
template <class T>
__device__ T block_excl_scan(T v, T *lds, T *total) {
  const int w = wave_in_block(), l = lane_id();
  T inc = wave_incl_scan(v);
  if (l == SWR_WAVE - 1) lds[w] = inc;
  __syncthreads();
  T wave_off = 0, tot = 0;
  for (int k = 0; k < SCAN_THREADS / SWR_WAVE; k++) {
    if (k < w) wave_off += lds[k];
    tot += lds[k];
  }
  __syncthreads();
  *total = tot;
  return wave_off + inc - v;
}

template <class TI, class TO>
__global__ void __launch_bounds__(SCAN_THREADS) k_tile_sums(const TI *in, int n, TO *tile_sums) {
  __shared__ TO lds[SCAN_THREADS / SWR_WAVE];
  const long long base = (long long)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_ITEMS;
  TO s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++)
    if (base + k < n) s += (TO)in[base + k];
  TO tot;
  block_excl_scan<TO>(s, lds, &tot);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// A tile's exclusive scan, after the sum of everything before it: every
// workgroup adds up the earlier tiles' sums or, while there are few tiles,
// their items; of many tiles the sums were scanned before.  The last one
// writes the total.
enum { SCAN_BY_ITEMS, SCAN_BY_SUMS, SCAN_BY_OFFSETS };
template <class TI, class TO, int BY>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_apply(const TI *in, int n, const TO *tile_sums, TO *out,
                                                             TO *total) {
  __shared__ TO lds[SCAN_THREADS / SWR_WAVE];
  const long long base = (long long)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_ITEMS;
  TO before = 0;
  if (BY == SCAN_BY_OFFSETS) {
    if (threadIdx.x == 0) before = tile_sums[blockIdx.x];
  } else if (BY == SCAN_BY_SUMS) {
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += SCAN_THREADS) before += tile_sums[k];
  } else {
    const int first = blockIdx.x * SCAN_TILE;
#pragma unroll 8
    for (int k = threadIdx.x; k < first; k += SCAN_THREADS) before += (TO)in[k];
  }
  TO vals[SCAN_ITEMS];
  TO s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    vals[k] = (base + k < n) ? (TO)in[base + k] : 0;
    s += vals[k];
  }
  TO off, tot;
  block_excl_scan<TO>(before, lds, &off);
  TO ex = block_excl_scan<TO>(s, lds, &tot) + off;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0 && total) *total = off + tot;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    if (base + k < n) out[base + k] = ex;
    ex += vals[k];
  }
}

// Tiles up to which one launch does (16,384 items: the last workgroup reads 60
// items a thread first, about a launch's time).
constexpr int SCAN_DIRECT = 16;
// Tiles up to which every workgroup adds up the sums before its own: that
// reading grows with the square of the tiles, and from about four million
// items on two launches over the sums are cheaper (a neighbour build on a grid
// of 4.2 million bins 123 us either way, of 14 million 178 and 161, of 33
// million 349 and 229, of 112 million 1,878 and 549).
constexpr int SCAN_FLAT = 4096;

template <class TI, class TO>
int scan_impl(swr_system *S, const TI *in, TO *out, int n, TO *total_dev) {
  if (n <= 0) {
    if (total_dev) HIP_CHECK(hipMemsetAsync(total_dev, 0, sizeof(TO), S->stream));
    return SWR_OK;
  }
  const int ntiles = div_up(n, SCAN_TILE);
  if (ntiles <= SCAN_DIRECT && (const void *)in != (const void *)out) {
    hipLaunchKernelGGL((k_scan_apply<TI, TO, SCAN_BY_ITEMS>), dim3(ntiles), dim3(SCAN_THREADS), 0, S->stream, in, n,
                       (const TO *)nullptr, out, total_dev);
    HIP_CHECK(hipGetLastError());
    return SWR_OK;
  }
  const int ntiles2 = div_up(ntiles, SCAN_TILE);
  const size_t need = sizeof(TO) * (2 * (size_t)ntiles + ntiles2);
  if (need > S->scan_tmp_bytes) {
    if (S->scan_tmp) (void)hipFree(S->scan_tmp);
    S->scan_tmp = nullptr;
    S->scan_tmp_bytes = 0;
    HIP_CHECK(hipMalloc(&S->scan_tmp, need * 2));
    S->scan_tmp_bytes = need * 2;
  }
  TO *tiles = (TO *)S->scan_tmp;
  hipLaunchKernelGGL((k_tile_sums<TI, TO>), dim3(ntiles), dim3(SCAN_THREADS), 0, S->stream, in, n, tiles);
  if (ntiles <= SCAN_FLAT) {
    hipLaunchKernelGGL((k_scan_apply<TI, TO, SCAN_BY_SUMS>), dim3(ntiles), dim3(SCAN_THREADS), 0, S->stream, in, n,
                       (const TO *)tiles, out, total_dev);
  } else {
    TO *offs = tiles + ntiles, *tiles2 = offs + ntiles;
    hipLaunchKernelGGL((k_tile_sums<TO, TO>), dim3(ntiles2), dim3(SCAN_THREADS), 0, S->stream, (const TO *)tiles, ntiles,
                       tiles2);
    hipLaunchKernelGGL((k_scan_apply<TO, TO, SCAN_BY_SUMS>), dim3(ntiles2), dim3(SCAN_THREADS), 0, S->stream,
                       (const TO *)tiles, ntiles, (const TO *)tiles2, offs, (TO *)nullptr);
    hipLaunchKernelGGL((k_scan_apply<TI, TO, SCAN_BY_OFFSETS>), dim3(ntiles), dim3(SCAN_THREADS), 0, S->stream, in, n,
                       (const TO *)offs, out, total_dev);
  }
  HIP_CHECK(hipGetLastError());
  return SWR_OK;
}

}  // namespace

void swr_set_error_msg(const std::string &m) {
  std::lock_guard<std::mutex> g(g_err_mu);
  g_err = m;
}

extern "C" const char *swr_last_error(void) {
  static thread_local std::string copy;
  std::lock_guard<std::mutex> g(g_err_mu);
  copy = g_err;
  return copy.c_str();
}

// Exclusive scan of n ints into int64 offsets; out has n+1 entries
// (out[n] = total).
int swr_scan_i32_to_i64(swr_system *S, const int *in, long long *out, int n) {
  return scan_impl<int, long long>(S, in, out, n, out + n);
}

// Exclusive scan of n ints into ints; total written to *total_dev (device).
int swr_scan_i32(swr_system *S, const int *in, int *out, int n, int *total_dev) {
  return scan_impl<int, int>(S, in, out, n, total_dev);
}

const char *const swr_kt_names[KT_COUNT] = {"verlet", "far", "build_H", "cg_iter", "cg_setup", "bo",
                                            "validate", "spmv", "reset", "qeq_q", "bins", "mixed_inner",
                                            "mixed_outer", "bonds", "cg_scalars", "mark", "cg_update", "nonbonded",
                                            "atom_energy", "dbond", "hbonds", "valence",
                                            "torsion", "panel"};

// Records a start event for kernel slot k on the system stream.
void swr_kt_begin(swr_system *S, int k) {
  if (!S->ktime) return;
  swr_system::KTimer &t = S->kt[k];
  if ((size_t)(2 * t.used + 2) > t.ev.size()) {
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return;
    t.ev.push_back(a);
    t.ev.push_back(b);
  }
  (void)hipEventRecord(t.ev[2 * t.used], S->stream);
}

void swr_kt_end(swr_system *S, int k) {
  if (!S->ktime) return;
  swr_system::KTimer &t = S->kt[k];
  if ((size_t)(2 * t.used + 2) > t.ev.size()) return;
  (void)hipEventRecord(t.ev[2 * t.used + 1], S->stream);
  t.used++;
}

extern "C" int swr_ktimer_enable(swr_system *S, int on) {
  if (!S) return SWR_ERR_ARG;
  S->ktime = on != 0;
  return SWR_OK;
}

// Accumulates the recorded launches of slot `name` (synchronises) and
// returns the total milliseconds and launch count since the last reset.
extern "C" int swr_ktimer_read(swr_system *S, const char *name, double *ms, long long *count, int reset) {
  if (!S || !name) return SWR_ERR_ARG;
  int k = -1;
  for (int i = 0; i < KT_COUNT; i++)
    if (std::string(name) == swr_kt_names[i]) k = i;
  if (k < 0) return SWR_ERR_ARG;
  swr_system::KTimer &t = S->kt[k];
  if (t.used) {
    HIP_CHECK(hipEventSynchronize(t.ev[2 * t.used - 1]));
    for (int u = 0; u < t.used; u++) {
      float e = 0.f;
      if (hipEventElapsedTime(&e, t.ev[2 * u], t.ev[2 * u + 1]) == hipSuccess) t.ms += e;
    }
    t.count += t.used;
    t.used = 0;
  }
  if (ms) *ms = t.ms;
  if (count) *count = t.count;
  if (reset) { t.ms = 0; t.count = 0; }
  return SWR_OK;
}

int swr_ensure_tmp(swr_system *S, size_t bytes) {
  size_t count = (bytes + sizeof(int) - 1) / sizeof(int);
  if (count <= S->tmp_i_cap) return SWR_OK;
  int rc = swr_alloc(&S->tmp_i, count);
  if (rc) return rc;
  S->tmp_i_cap = count;
  return SWR_OK;
}
