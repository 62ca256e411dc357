// libteahip.so: chunk handle, field access, timing and the final pass of
// every reduction.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <string>

#include "tea_hip_impl.h"

namespace tea {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string& msg) { g_last_error = msg; }

const char* const kKernelNames[K_NUM] = {
    "set_chunk_data", "set_chunk_state", "store_energy", "local_halos",
    "field_summary",  "cg_init_u",       "cg_init_k",    "cg_init_others",
    "cg_calc_w",      "cg_calc_ur",      "cg_calc_p",    "cg_fused_w",
    "cg_fused_r",     "cg_apply_pending", "copy_u",      "calculate_residual",
    "calculate_2norm", "finalise",       "mpcg_convert", "mpcg_w",
    "mpcg_r",         "mpcg_apply_u",    "mpcg_refresh",  "fcg_w",
    "fcg_jacobi",     "fcg_restrict",    "fcg_net",       "fcg_prolong",
    "span_finish",    "jacobi_init",     "jacobi_copy_u", "jacobi_iterate",
    "jacobi_fused",   "cheby_init",      "cheby_iterate", "cheby_calc_u",
    "cheby_fused",    "ppcg_init",       "ppcg_calc_ur",  "ppcg_calc_sd",
    "ppcg_fused",     "ppcg_two_step",   "cheby_two_step", "fcg_sweeps",
    "cg_ra_finish"};

Timed::Timed(tea_hip_chunk* c_, int kid_, hipStream_t s)
    : c(c_), kid(kid_), stream(s ? s : c_->stream) {
  if (!c->timing || !c->time_kernel[kid]) return;
  if (c->event_pool.size() < 2) {
    for (int i = 0; i < 64; ++i) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return;
      c->event_pool.push_back(e);
    }
  }
  start = c->event_pool.back();
  c->event_pool.pop_back();
  stop = c->event_pool.back();
  c->event_pool.pop_back();
  (void)hipEventRecord(start, stream);
}

Timed::~Timed() {
  if (!start) return;
  (void)hipEventRecord(stop, stream);
  c->inflight.push_back({kid, start, stop});
}

int resolve_timing(tea_hip_chunk* c) {
  for (auto& p : c->inflight) {
    float ms = 0.0f;
    TEA_HIP_TRY(hipEventElapsedTime(&ms, p.start, p.stop));
    c->launches[p.kid] += 1;
    c->total_ms[p.kid] += ms;
    c->event_pool.push_back(p.start);
    c->event_pool.push_back(p.stop);
  }
  c->inflight.clear();
  return TEA_HIP_OK;
}

int sync_chunk(tea_hip_chunk* c) {
  TEA_HIP_TRY(hipStreamSynchronize(c->stream));
  c->poll_nr = 0;
  c->ra_dirty = false;
  return resolve_timing(c);
}

int resolve_ready(tea_hip_chunk* c) {
  size_t k = 0;
  for (; k < c->inflight.size(); ++k) {
    const auto& p = c->inflight[k];
    const hipError_t e = hipEventQuery(p.stop);
    if (e == hipErrorNotReady) break;
    TEA_HIP_TRY(e);
    float ms = 0.0f;
    TEA_HIP_TRY(hipEventElapsedTime(&ms, p.start, p.stop));
    c->launches[p.kid] += 1;
    c->total_ms[p.kid] += ms;
    c->event_pool.push_back(p.start);
    c->event_pool.push_back(p.stop);
  }
  c->inflight.erase(c->inflight.begin(), c->inflight.begin() + k);
  return TEA_HIP_OK;
}

// A signalling NaN.  Every partial is a sum, and IEEE 754 arithmetic never
// returns a signalling NaN (a NaN operand comes out quiet), so no partial
// can equal it; the wait below would still end when the stream goes idle.
constexpr uint64_t kPollSentinel = 0x7ff4c0ffee5e4d1dull;

// Spins until none of the nr x len values at v (arrays stride apart) holds
// the sentinel.  The stream is queried only after about 2^22 spins
// (milliseconds, longer than a pass over an 8192^2 chunk) and then every
// 2^16 spins, a few queries per pass even over the largest chunks: a query
// every few hundred spins slowed the kernels it overlapped.  An idle stream
// with a sentinel left means a kernel wrote fewer values than were waited
// for: an error naming the value.
static int wait_values(tea_hip_chunk* c, const volatile uint64_t* v, size_t stride, int nr,
                       int len) {
  int q = 0, i = 0;
  for (uint64_t spins = 1;; ++spins) {
    while (q < nr) {
      while (i < len && v[q * stride + i] != kPollSentinel) ++i;
      if (i < len) break;
      ++q;
      i = 0;
    }
    if (q == nr) break;
    if (spins >= (1ull << 22) && (spins & 0xffff) == 0) {
      const hipError_t e = hipStreamQuery(c->stream);
      if (e == hipSuccess) {
        std::atomic_thread_fence(std::memory_order_acquire);
        for (int qq = 0; qq < nr; ++qq)
          for (int ii = 0; ii < len; ++ii)
            if (v[qq * stride + ii] == kPollSentinel) {
              set_error("reduction " + std::to_string(qq) + " left partial " +
                        std::to_string(ii) + " unwritten");
              return TEA_HIP_EINVAL;
            }
        break;
      }
      if (e != hipErrorNotReady) TEA_HIP_TRY(e);
    }
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return resolve_ready(c);
}

// The host's view of the partials is coherent, mapped memory: the finisher's
// stores reach it while the kernel is still retiring, so the host can form
// the next scalar and launch the next kernel before the stream reports
// completion.
static int wait_partials(tea_hip_chunk* c) {
  if (c->poll_nr == 0) return sync_chunk(c);
  const int nr = c->poll_nr;
  c->poll_nr = 0;
  TEA_RETURN_IF(wait_values(c, reinterpret_cast<const volatile uint64_t*>(c->host_partials),
                            (size_t)c->nspan, nr, 1));
  // Every pass queued before the one waited for has ended, a dropped
  // run-ahead too.
  c->ra_dirty = false;
  return TEA_HIP_OK;
}

void arm_host_values(double* host, int count) {
  uint64_t* v = reinterpret_cast<uint64_t*>(host);
  for (int i = 0; i < count; ++i) v[i] = kPollSentinel;
}

int wait_host_values(tea_hip_chunk* c, const double* host, int count) {
  return wait_values(c, reinterpret_cast<const volatile uint64_t*>(host), 0, 1, count);
}

// Final passes of the reference's reduceArray (TeaLeaf/c_kernels/sycl/
// sycl_shared.hpp:43-75) over one launch's level-2 partials, on the host:
// the kernels write one partial per 4096-cell span straight into pinned host
// memory, so after the stream is synchronised the remaining passes (e.g.
// 4105 -> 65 -> 2 -> 1 at 4096^2) are a few thousand host additions, with
// no extra launch.  Each pass cuts the array into zero-padded groups of 64
// and sums each group with the pairwise tree.
static double host_tree_passes(double* v, size_t len) {
  while (len != 1) {
    const size_t groups = (len + kWave - 1) / kWave;
    for (size_t g = 0; g < groups; ++g) {
      double a[kWave];
      for (int l = 0; l < kWave; ++l) {
        const size_t i = g * kWave + l;
        a[l] = i < len ? v[i] : 0.0;
      }
      for (int st = 1; st < kWave; st *= 2)
        for (int i = 0; i + st < kWave; i += 2 * st) a[i] = a[i] + a[i + st];
      v[g] = a[0];  // g <= 64g: earlier groups never read it again
    }
    len = groups;
  }
  return v[0];
}

// A sum's last pass, the run-ahead's scalar and where they go (RaTail, or the
// sums alone), by one lane.
template <int NR, bool TAIL>
__device__ inline void finish_out(const double (&sum)[NR], double* out, int out_stride,
                                  const RaTail& tail) {
  if (!TAIL) {
#pragma unroll
    for (int q = 0; q < NR; ++q) out[(size_t)q * out_stride] = sum[q];
    return;
  }
  double x;
  if (NR == 1) {
    const double r0 = tail.from_dev ? tail.ra[2] : tail.rro;
    x = tail.mode == 0 ? r0 / sum[0] : sum[0] / r0;
    if (tail.mode == 1) tail.ra[2] = sum[0];
  } else {
    x = tail.mode == 0 ? sum[NR - 1] / sum[0] : -sum[NR - 1] / tail.ra[2];
    if (tail.mode == 0) tail.ra[2] = sum[0];
    out[1] = sum[NR - 1];
  }
  tail.ra[tail.mode] = x;
  out[0] = sum[0];
  out[NR] = x;
}

// One group of 512 block sums (64 spans): lane l takes span l's 8 blocks.
__device__ inline double group_sum(const double* __restrict__ p) {
  const int lane = threadIdx.x & (kWave - 1);
  const double2 a = ld2(p, kSubPerSpan * lane), b = ld2(p, kSubPerSpan * lane + 2);
  const double2 c = ld2(p, kSubPerSpan * lane + 4), d = ld2(p, kSubPerSpan * lane + 6);
  return wave_tree_dpp(((a.x + a.y) + (b.x + b.y)) + ((c.x + c.y) + (d.x + d.y)));
}

// The rest of the tree over the block sums of at most 16 groups, a wave per
// group in one block, wave 0 the last pass: 3.4 us at 1024^2, all latency,
// against 4.8 us for a block per group with a last-block pass.
constexpr int kFinishWaves = 16;
template <int NR, bool TAIL>
__global__ __launch_bounds__(kFinishWaves * kWave) void span_finish_kernel(
    const double* __restrict__ sub, int nblk, double* out, int out_stride, RaTail tail) {
  __shared__ double gs[NR][kFinishWaves];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const size_t stride = sub_stride(nblk);
  double t[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q)
    t[q] = wv * kGroupBlocks < nblk ? group_sum(sub + q * stride + wv * kGroupBlocks) : 0.0;
#pragma unroll
  for (int q = 0; q < NR; ++q)
    if (lane == 0) gs[q][wv] = t[q];
  __syncthreads();
  if (wv != 0) return;
  double sum[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) sum[q] = wave_tree_dpp(lane < kFinishWaves ? gs[q][lane] : 0.0);
  if (lane == 0) finish_out<NR, TAIL>(sum, out, out_stride, tail);
}

// More groups (grids above 8192 blocks): a wave and block per group; the last
// one to count itself done runs the remaining passes over the group sums in
// part.  Those are stored and read at device scope (past the XCDs' own L2s),
// and the count follows its sum's store, so no fence is needed: a release
// fence writes back a whole L2.  That order rests on the hardware, not on the
// language's memory model (all these accesses are relaxed): s_waitcnt vmcnt(0)
// ends once the device-scope store is out, and the last block's loads are issued
// only after the branch on the count it read.
__device__ inline void st_agent(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline double ld_agent(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int NR, bool TAIL>
__global__ __launch_bounds__(kWave) void span_finish_groups_kernel(
    const double* __restrict__ sub, int nblk, double* part, unsigned* count, double* out,
    int out_stride, RaTail tail) {
  const int lane = threadIdx.x, g = blockIdx.x, ngrp = gridDim.x;
  const size_t stride = sub_stride(nblk);
  double t[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) t[q] = group_sum(sub + q * stride + (size_t)g * kGroupBlocks);
  unsigned prev = 0;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < NR; ++q) st_agent(part + (size_t)q * ngrp + g, t[q]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the sums are out before the count
    prev = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  prev = __builtin_amdgcn_readfirstlane(prev);
  if (prev != gridDim.x - 1) return;
  // At most 8192 groups (a chunk has fewer than 2^31 cells): up to 128 sums
  // of 64 groups, held one per lane in w[0] and w[1].
  double sum[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    double w[2] = {0.0, 0.0};
    for (int i = 0; i * kWave < ngrp; ++i) {
      const int k = i * kWave + lane;
      const double u = wave_tree_dpp(k < ngrp ? ld_agent(part + (size_t)q * ngrp + k) : 0.0);
      if (lane == (i & (kWave - 1))) {
        if (i < kWave)
          w[0] = u;
        else
          w[1] = u;
      }
    }
    sum[q] = wave_tree_dpp(w[0]);
    if (ngrp > kWave * kWave) sum[q] = sum[q] + wave_tree_dpp(w[1]);
  }
  if (lane != 0) return;
  __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  finish_out<NR, TAIL>(sum, out, out_stride, tail);
}

template <int NR, bool TAIL>
static void launch_finish(tea_hip_chunk* c, const double* sub, double* out, int out_stride,
                          const RaTail& tail) {
  const int ngrp = sub_stride(c->nblk) / kGroupBlocks;
  if (ngrp <= kFinishWaves)
    hipLaunchKernelGGL((span_finish_kernel<NR, TAIL>), dim3(1), dim3(kFinishWaves * kWave), 0,
                       c->stream, sub, c->nblk, out, out_stride, tail);
  else
    hipLaunchKernelGGL((span_finish_groups_kernel<NR, TAIL>), dim3(ngrp), dim3(kWave), 0,
                       c->stream, sub,
                       c->nblk, c->grp_sum, c->done_count, out, out_stride, tail);
}

int launch_span_finish(tea_hip_chunk* c, int nr, int* len, int slot, bool poll,
                       const double* sub) {
  TEA_CHECK_ARG(nr >= 1 && nr <= kSubMaxNr, "span_finish: bad reduction count");
  TEA_CHECK_ARG(slot >= 0 && slot + nr <= 4, "span_finish: bad partials slot");
  if (!sub) sub = c->sub;
  *len = 1;
  c->poll_nr = 0;
  if (poll && c->poll && slot == 0) {
    for (int q = 0; q < nr; ++q) arm_host_values(c->host_partials + (size_t)q * c->nspan, 1);
    c->poll_nr = nr;
  }
  Timed t(c, K_SPAN_FINISH);
  const auto launch = nr == 1   ? launch_finish<1, false>
                      : nr == 2 ? launch_finish<2, false>
                      : nr == 3 ? launch_finish<3, false>
                                : launch_finish<4, false>;
  launch(c, sub, c->partials + (size_t)slot * c->nspan, c->nspan, RaTail{});
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

int launch_span_finish_ra(tea_hip_chunk* c, int nr, double* out, const RaTail& tail) {
  TEA_CHECK_ARG(nr == 1 || nr == 2, "span_finish: bad reduction count");
  Timed t(c, nr == 1 ? K_CG_RA_FINISH : K_SPAN_FINISH);
  const auto launch = nr == 1 ? launch_finish<1, true> : launch_finish<2, true>;
  launch(c, c->sub, out, 1, tail);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

bool dev_alloc_bytes(tea_hip_chunk* c, void** p, size_t bytes) {
  *p = nullptr;
  if (bytes > c->dev_limit - c->dev_bytes) return false;
  if (hipMalloc(p, bytes) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return false;
  }
  c->dev_sizes[*p] = bytes;
  c->dev_bytes += bytes;
  return true;
}

int release_spares(tea_hip_chunk* c, bool keep_pair) {
  TEA_RETURN_IF(drop_ahead(c, kAheadNone));
  if (c->hold) TEA_RETURN_IF(apply_mp_hold(c));
  TEA_RETURN_IF(apply_held_u(c));
  TEA_RETURN_IF(sync_chunk(c));
  for (double** b : {&c->p_alt[1], &c->p_alt[2], &c->r_alt, &c->w_alt, &c->u_alt})
    dev_free(c, *b);
  if (c->mp_cur == 3) {
    std::swap(c->mp_p[0], c->mp_p[3]);
    c->mp_cur = 0;
  }
  for (float** b : {&c->mp_p[3], &c->mp_r_alt, &c->mp_w_alt, &c->fcg_z_alt}) dev_free(c, *b);
  c->p_ring_off = c->ra_off = c->mra_off = true;
  if (keep_pair) return TEA_HIP_OK;
  dev_free(c, c->spare);
  dev_free(c, c->spare2);
  c->j_off = true;
  return TEA_HIP_OK;
}

double* host_slots(int n, double** dev) {
  double* host = nullptr;
  if (hipHostMalloc(&host, n * sizeof(double), hipHostMallocMapped | hipHostMallocCoherent) ==
      hipSuccess) {
    if (hipHostGetDevicePointer((void**)dev, host, 0) == hipSuccess) return host;
    (void)hipHostFree(host);
  }
  (void)hipGetLastError();
  return nullptr;
}

void dev_free_bytes(tea_hip_chunk* c, void* p) {
  if (!p) return;
  const auto it = c->dev_sizes.find(p);
  c->dev_bytes -= it->second;
  c->dev_sizes.erase(it);
  (void)hipFree(p);
}

// dst = src in 16-byte pieces, one per thread, nontemporal both ways: the
// streaming ceiling for tea_hip_copy_bandwidth.
__global__ __launch_bounds__(kBlock) void stream_copy_kernel(const double* __restrict__ src,
                                                             double* __restrict__ dst,
                                                             size_t n2) {
  typedef double dv2 __attribute__((ext_vector_type(2)));
  const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n2) return;
  const dv2 v = __builtin_nontemporal_load(reinterpret_cast<const dv2*>(src) + i);
  __builtin_nontemporal_store(v, reinterpret_cast<dv2*>(dst) + i);
}

int finish_reduction_n(tea_hip_chunk* c, int nr, int len, double* out) {
  TEA_RETURN_IF(wait_partials(c));
  for (int q = 0; q < nr; ++q)
    out[q] = host_tree_passes(c->host_partials + (size_t)q * c->nspan,
                              (size_t)len);
  return TEA_HIP_OK;
}

int finish_reduction_lens(tea_hip_chunk* c, int nr, const int* lens, double* out) {
  TEA_RETURN_IF(sync_chunk(c));
  for (int q = 0; q < nr; ++q)
    out[q] = host_tree_passes(c->host_partials + (size_t)q * c->nspan,
                              (size_t)lens[q]);
  return TEA_HIP_OK;
}

int finish_reduction(tea_hip_chunk* c, int nr, double* out) {
  return finish_reduction_n(c, nr, c->nspan, out);
}

}  // namespace tea

using namespace tea;

#define TEA_CHECK_CHUNK(c) TEA_CHECK_ARG((c) != nullptr, "null chunk handle")

extern "C" {

const char* tea_hip_last_error(void) { return g_last_error.c_str(); }

int tea_hip_chunk_create(int device, int x, int y, int halo_depth,
                         tea_hip_chunk** out) {
  TEA_CHECK_ARG(out != nullptr, "null output handle");
  *out = nullptr;
  TEA_CHECK_ARG(halo_depth >= 1, "halo_depth must be >= 1");
  TEA_CHECK_ARG(x > 2 * halo_depth && y > 2 * halo_depth,
                "x and y must exceed 2*halo_depth");
  const long n = (long)x * (long)y;
  TEA_CHECK_ARG(n < (1L << 31) - kSpan, "chunk too large (x*y >= 2^31)");
  int ndev = 0;
  TEA_HIP_TRY(hipGetDeviceCount(&ndev));
  TEA_CHECK_ARG(device >= 0 && device < ndev, "no such HIP device");
  TEA_HIP_TRY(hipSetDevice(device));

  tea_hip_chunk* c = new tea_hip_chunk();
  c->device = device;
  c->geo.x = x;
  c->geo.y = y;
  c->geo.h = halo_depth;
  c->geo.n = (int)n;
  c->geo.nt = n > kStreamCells;
  c->geo.nt_half = n > kStreamCellsHalf;
  c->geo.bands = bands_for(x);
  c->geo.dx = FastDiv((uint32_t)x);
  c->ngroup = (int)((n + kWave - 1) / kWave);
  c->nspan = (int)((n + kSpan - 1) / kSpan);
  if (const char* b = getenv("TEA_HIP_BATCH")) c->batch = atoi(b);
  c->pairs = y >= 3;
  if (const char* pv = getenv("TEA_HIP_PAIRS")) c->pairs = c->pairs && atoi(pv) != 0;
  c->quads = c->pairs && x % 4 == 0;
  if (const char* qv = getenv("TEA_HIP_QUADS")) c->quads = c->quads && atoi(qv) != 0;
  if (const char* hv = getenv("TEA_HIP_HOLD_U")) c->hold_ok = atoi(hv) != 0;
  c->nblk = (int)((n + kPairBlock - 1) / kPairBlock);
  if (const char* pb = getenv("TEA_HIP_PAIR_BLOCKS")) c->pair_blocks = atoi(pb);
  for (int k = 0; k < K_NUM; ++k) c->time_kernel[k] = true;
  if (const char* only = getenv("TEA_HIP_STATS_ONLY")) {
    for (int k = 0; k < K_NUM; ++k) {
      const std::string name = kKernelNames[k];
      const std::string list = std::string(",") + only + ",";
      c->time_kernel[k] = list.find("," + name + ",") != std::string::npos;
    }
  }
  if (const char* pv = getenv("TEA_HIP_POLL")) c->poll = atoi(pv) != 0;
  if (const char* rv = getenv("TEA_HIP_RUN_AHEAD")) c->ra_enabled = atoi(rv) != 0;
  if (const char* sv = getenv("TEA_HIP_STACK")) c->stack = atoi(sv);
  if (const char* sp = getenv("TEA_HIP_SPIN"))
    if (atoi(sp) != 0) (void)hipSetDeviceFlags(hipDeviceScheduleSpin);

  auto fail = [&](int code) {
    tea_hip_chunk_destroy(c);
    return code;
  };

  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    set_error("hipStreamCreateWithFlags failed");
    return fail(TEA_HIP_EHIP);
  }

  const size_t xy = (size_t)n;
  const size_t X = (size_t)x, Y = (size_t)y;
  for (int f = 0; f < TEA_NUM_FIELDS; ++f) c->field_len[f] = xy;
  c->field_len[TEA_FIELD_X_AREA] = (X + 1) * Y;
  c->field_len[TEA_FIELD_Y_AREA] = X * (Y + 1);
  c->field_len[TEA_FIELD_CELL_X] = X;
  c->field_len[TEA_FIELD_CELL_Y] = Y;
  c->field_len[TEA_FIELD_CELL_DX] = X;
  c->field_len[TEA_FIELD_CELL_DY] = Y;
  c->field_len[TEA_FIELD_VERTEX_DX] = X + 1;
  c->field_len[TEA_FIELD_VERTEX_DY] = Y + 1;
  c->field_len[TEA_FIELD_VERTEX_X] = X + 1;
  c->field_len[TEA_FIELD_VERTEX_Y] = Y + 1;
  c->field_len[TEA_FIELD_COMMS_BUFFER] = std::max(X, Y) * (size_t)halo_depth;

  for (int f = 0; f < TEA_NUM_FIELDS; ++f) {
    const size_t bytes = pair_bytes((long)c->field_len[f], sizeof(double));
    if (!dev_alloc(c, &c->field[f], bytes)) {
      set_error("hipMalloc of a field failed");
      return fail(TEA_HIP_ENOMEM);
    }
    if (hipMemsetAsync(c->field[f], 0, bytes, c->stream) != hipSuccess) {
      set_error("hipMemsetAsync failed");
      return fail(TEA_HIP_EHIP);
    }
  }
  if (!dev_alloc(c, &c->p_alt[0], pair_bytes(n, sizeof(double)))) {
    set_error("hipMalloc of the second p buffer failed");
    return fail(TEA_HIP_ENOMEM);
  }
  // One allocation, zero: two sets of block sums, the group sums and the
  // finisher's counter.
  const size_t ns = (size_t)kSubMaxNr * sub_stride(c->nblk), ng = ns / kGroupBlocks;
  const size_t rbytes = (2 * ns + ng + 1) * sizeof(double);
  if (!dev_alloc(c, &c->sub, rbytes)) {
    set_error("hipMalloc of the reduction workspace failed");
    return fail(TEA_HIP_ENOMEM);
  }
  c->sub2 = c->sub + ns;
  c->grp_sum = c->sub2 + ns;
  c->done_count = reinterpret_cast<unsigned*>(c->grp_sum + ng);
  if (hipMemsetAsync(c->sub, 0, rbytes, c->stream) != hipSuccess) {
    set_error("hipMemsetAsync failed");
    return fail(TEA_HIP_EHIP);
  }
  const size_t pbytes = 4 * (size_t)c->nspan * sizeof(double);
  if (hipHostMalloc(&c->host_partials, pbytes,
                    hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
    c->host_partials = nullptr;
    set_error("hipHostMalloc of the reduction partials failed");
    return fail(TEA_HIP_ENOMEM);
  }
  std::memset(c->host_partials, 0, pbytes);
  if (hipHostGetDevicePointer((void**)&c->partials, c->host_partials, 0) !=
      hipSuccess) {
    set_error("hipHostGetDevicePointer failed");
    return fail(TEA_HIP_EHIP);
  }
  if (hipStreamSynchronize(c->stream) != hipSuccess) {
    set_error("hipStreamSynchronize failed");
    return fail(TEA_HIP_EHIP);
  }
  if (const char* ev = getenv("TEA_HIP_EXTRA_BYTES")) {
    const size_t extra = strtoull(ev, nullptr, 10);
    if (extra < SIZE_MAX - c->dev_bytes) c->dev_limit = c->dev_bytes + extra;
  }
  *out = c;
  return TEA_HIP_OK;
}

int tea_hip_chunk_destroy(tea_hip_chunk* c) {
  if (!c) return TEA_HIP_OK;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& p : c->inflight) {
    (void)hipEventDestroy(p.start);
    (void)hipEventDestroy(p.stop);
  }
  for (auto e : c->event_pool) (void)hipEventDestroy(e);
  for (int f = 0; f < TEA_NUM_FIELDS; ++f)
    if (c->field[f]) (void)hipFree(c->field[f]);
  for (double* b : c->p_alt)
    if (b) (void)hipFree(b);
  for (double* b : {c->r_alt, c->u_alt, c->w_alt, c->ra_dev})
    if (b) (void)hipFree(b);
  if (c->ra_host) (void)hipHostFree(c->ra_host);
  if (c->spare) (void)hipFree(c->spare);
  if (c->spare2) (void)hipFree(c->spare2);
  if (c->sub) (void)hipFree(c->sub);
  for (float* b : c->mp_p)
    if (b) (void)hipFree(b);
  for (float* b : {c->mp_r, c->mp_w, c->mp_kx, c->mp_ky, c->fcg_z, c->mp_r_alt, c->mp_w_alt,
                   c->fcg_z_alt})
    if (b) (void)hipFree(b);
  if (c->mra_dev) (void)hipFree(c->mra_dev);
  if (c->mra_host) (void)hipHostFree(c->mra_host);
  if (c->j_host) (void)hipHostFree(c->j_host);
  if (c->fcg_xsum) (void)hipFree(c->fcg_xsum);
  if (c->fcg_g) (void)hipFree(c->fcg_g);
  for (FcgLevel& L : c->fcg_lv) {
    for (float* b : {L.feat, L.rbar, L.kc, L.dis, L.sig, L.y})
      if (b) (void)hipFree(b);
    if (L.rms) (void)hipFree(L.rms);
    if (L.tpart) (void)hipFree(L.tpart);
    if (L.net) tea_nn_destroy(L.net);
  }
  if (c->host_partials) (void)hipHostFree(c->host_partials);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return TEA_HIP_OK;
}

int tea_hip_field(tea_hip_chunk* c, int field, double** dev_ptr,
                  size_t* count) {
  TEA_CHECK_CHUNK(c);
  TEA_CHECK_ARG(field >= 0 && field < TEA_NUM_FIELDS, "bad field id");
  if (dev_ptr) *dev_ptr = c->field[field];
  if (count) *count = c->field_len[field];
  return TEA_HIP_OK;
}

int tea_hip_field_write(tea_hip_chunk* c, int field, const double* host,
                        size_t count) {
  TEA_CHECK_CHUNK(c);
  TEA_CHECK_ARG(field >= 0 && field < TEA_NUM_FIELDS, "bad field id");
  TEA_CHECK_ARG(count <= c->field_len[field], "count exceeds field length");
  TEA_CHECK_ARG(host != nullptr || count == 0, "null host buffer");
  TEA_HIP_TRY(hipSetDevice(c->device));
  TEA_RETURN_IF(apply_pending(c));
  TEA_HIP_TRY(hipMemcpyAsync(c->field[field], host, count * sizeof(double),
                             hipMemcpyHostToDevice, c->stream));
  if (field == TEA_FIELD_P) c->p_alt_synced = false;
  c->faces_ok_u = c->faces_ok_p = false;
  return sync_chunk(c);
}

int tea_hip_field_read(tea_hip_chunk* c, int field, double* host,
                       size_t count) {
  TEA_CHECK_CHUNK(c);
  TEA_CHECK_ARG(field >= 0 && field < TEA_NUM_FIELDS, "bad field id");
  TEA_CHECK_ARG(count <= c->field_len[field], "count exceeds field length");
  TEA_CHECK_ARG(host != nullptr || count == 0, "null host buffer");
  TEA_HIP_TRY(hipSetDevice(c->device));
  TEA_RETURN_IF(apply_pending(c));
  TEA_HIP_TRY(hipMemcpyAsync(host, c->field[field], count * sizeof(double),
                             hipMemcpyDeviceToHost, c->stream));
  return sync_chunk(c);
}

int tea_hip_synchronize(tea_hip_chunk* c) {
  TEA_CHECK_CHUNK(c);
  TEA_HIP_TRY(hipSetDevice(c->device));
  return sync_chunk(c);
}

int tea_hip_set_fused(tea_hip_chunk* c, int fused) {
  TEA_CHECK_CHUNK(c);
  TEA_HIP_TRY(hipSetDevice(c->device));
  TEA_RETURN_IF(apply_pending(c));
  c->fused = fused ? 1 : 0;
  return TEA_HIP_OK;
}

int tea_hip_flush(tea_hip_chunk* c) {
  TEA_CHECK_CHUNK(c);
  TEA_HIP_TRY(hipSetDevice(c->device));
  TEA_RETURN_IF(apply_pending(c));
  return sync_chunk(c);
}

int tea_hip_timing_enable(tea_hip_chunk* c, int enable) {
  TEA_CHECK_CHUNK(c);
  TEA_RETURN_IF(sync_chunk(c));
  c->timing = enable != 0;
  return TEA_HIP_OK;
}

int tea_hip_kernel_stats(tea_hip_chunk* c, int kernel_id, long* launches,
                         double* total_ms) {
  TEA_CHECK_CHUNK(c);
  TEA_CHECK_ARG(kernel_id >= 0 && kernel_id < K_NUM, "bad kernel id");
  TEA_RETURN_IF(sync_chunk(c));
  if (launches) *launches = c->launches[kernel_id];
  if (total_ms) *total_ms = c->total_ms[kernel_id];
  return TEA_HIP_OK;
}

int tea_hip_ahead_taken(tea_hip_chunk* c, long taken[3]) {
  TEA_CHECK_CHUNK(c);
  TEA_CHECK_ARG(taken != nullptr, "null output");
  for (int k = 0; k < 3; ++k) taken[k] = c->taken[k];
  return TEA_HIP_OK;
}

int tea_hip_timing_reset(tea_hip_chunk* c) {
  TEA_CHECK_CHUNK(c);
  TEA_RETURN_IF(sync_chunk(c));
  for (int k = 0; k < K_NUM; ++k) {
    c->launches[k] = 0;
    c->total_ms[k] = 0.0;
  }
  return TEA_HIP_OK;
}

int tea_hip_copy_bandwidth(int device, size_t bytes, int reps, double* gbs) {
  TEA_CHECK_ARG(gbs != nullptr, "null output");
  TEA_CHECK_ARG(bytes >= 16 && bytes % 16 == 0, "bytes must be a positive multiple of 16");
  TEA_CHECK_ARG(reps >= 1, "reps must be positive");
  TEA_HIP_TRY(hipSetDevice(device));
  const size_t n2 = bytes / 16;
  double *src = nullptr, *dst = nullptr;
  if (hipMalloc(&src, bytes) != hipSuccess) {
    set_error("hipMalloc of the copy source failed");
    return TEA_HIP_ENOMEM;
  }
  if (hipMalloc(&dst, bytes) != hipSuccess) {
    (void)hipFree(src);
    set_error("hipMalloc of the copy destination failed");
    return TEA_HIP_ENOMEM;
  }
  hipStream_t st = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int status = TEA_HIP_OK;
  float ms = 0.0f;
  const dim3 grid((unsigned)((n2 + kBlock - 1) / kBlock));
  if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess ||
      hipMemsetAsync(src, 0, bytes, st) != hipSuccess) {
    set_error("copy bandwidth: stream, event or memset failed");
    status = TEA_HIP_EHIP;
  } else {
    for (int k = 0; k < 2; ++k)  // warm-up
      hipLaunchKernelGGL(stream_copy_kernel, grid, dim3(kBlock), 0, st, src, dst, n2);
    (void)hipEventRecord(e0, st);
    for (int k = 0; k < reps; ++k)
      hipLaunchKernelGGL(stream_copy_kernel, grid, dim3(kBlock), 0, st, src, dst, n2);
    (void)hipEventRecord(e1, st);
    if (hipGetLastError() != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
        hipEventElapsedTime(&ms, e0, e1) != hipSuccess || ms <= 0.0f) {
      set_error("copy bandwidth: launch or timing failed");
      status = TEA_HIP_EHIP;
    } else {
      *gbs = 2.0 * (double)bytes / ((double)ms * 1e-3 / reps) / 1e9;
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (st) (void)hipStreamDestroy(st);
  (void)hipFree(src);
  (void)hipFree(dst);
  return status;
}

int tea_hip_num_kernels(void) { return K_NUM; }

const char* tea_hip_kernel_name(int kernel_id) {
  if (kernel_id < 0 || kernel_id >= K_NUM) return "";
  return kKernelNames[kernel_id];
}

}  // extern "C"
