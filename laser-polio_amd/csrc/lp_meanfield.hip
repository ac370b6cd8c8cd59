// Mean-field rollout of the node-level transmission map and its adjoint
// (C ABI in include/lp_meanfield.h).
#include "../../include/lp_meanfield.h"
#include <mutex>

namespace lp_mf {

constexpr int WG = 256;

// Scratch of lp_mf_adjoint_days_noalloc: the two work rows of a launch per day (the
// mixed-weight adjoints of a day and of the one after it), 2 * LP_MF_NOALLOC_MAX_NODES
// floats = 256 KiB held by every GPU the library runs on until the process ends.
static __device__ __align__(256) float scratch[2 * LP_MF_NOALLOC_MAX_NODES];

constexpr int kMaxDevices = 64;
float* g_scratch[kMaxDevices] = {};   // device address of `scratch` on each device
std::mutex g_scratch_mu;

// Device address of `scratch` on the current device, looked up once per device
// (each device holds its own copy of the array at its own address).
int scratch_of_current_device(float** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return LP_ERR_HIP;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return LP_ERR_HIP;
    g_scratch[dev] = static_cast<float*>(ptr);
  }
  *out = g_scratch[dev];
  return LP_OK;
}

// A workgroup barrier that orders LDS only: global stores of the trajectories stay in
// flight across it (nothing in the launch reads them back).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Three ways to roll the days, chosen by the number of nodes (mf_path):
//   one workgroup (n <= 256)     every day in one launch: the network's rows in registers, the
//                                state exchanged through LDS, one barrier a day;
//   resident workgroups          every day in one cooperative launch of up to 128
//   (n <= 2048)                  workgroups, 16 rows each in registers, the state exchanged
//                                through the trajectory rows themselves (below);
//   one launch per day           larger networks, and under stream capture or where a
//                                cooperative launch is not to be had.
// One launch per day costs its dispatch and a chain of dependent loads for every day: 5.6
// us at 774 nodes forward, and 9 more for the adjoint's two.  Resident workgroups take 1.8
// us for either, one workgroup of 23 nodes 0.36 and 0.53 us (a launch per day: about 6 and 11).
// The network's adjoint N_bar[j][i] += beta_j (mbar_i - mbar_j) of all days is summed
// by one pass afterwards (k_mf_net_bar) instead of read and written once a day.
// In the adjoint, mbar_i = ((g_bar_i season_t) r0_i) / pop_i of a day goes to its season_part
// row first (h below; see day_adjoint): the network sees it there, and at the end
// season_part_i = mbar_i / season_t m_i takes its place.

// x plus the other lanes' of its row of 16, in every lane of the row.
template <int N>
__device__ __forceinline__ float add_row_ror(float x) {
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 | N, 0xf, 0xf, false));
}
__device__ __forceinline__ float row_sum(float x) {
  x = add_row_ror<8>(x);
  x = add_row_ror<4>(x);
  x = add_row_ror<2>(x);
  return add_row_ror<1>(x);
}
// The sum over the wavefront, in every lane.
__device__ __forceinline__ float wave_sum(float x) {
  x = row_sum(x);
  x = x + __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}

// Node i's constants.
struct Node {
  float keep, r0, rho, inv_pop;
};
__device__ __forceinline__ Node node_of(const lp_mf_model& m, int i) {
  return Node{m.keep[i], m.r0_scalar[i], m.rho[i], m.inv_pop[i]};
}

// One day of a node forward from its S, E, I and its mix sum_j N_ji I_j.
struct DayOut {
  float S, E, I, lam, mm, g;
};
__device__ __forceinline__ DayOut day_forward(const lp_mf_model& m, const Node& c, float season, float mix, float S,
                                              float E, float I) {
  DayOut o;
  o.mm = m.iota * fmaf(I, c.keep, mix);
  o.g = ((o.mm * season) * c.r0) * c.inv_pop;
  const float p = -lp::expm1f_lp(-o.g);
  o.lam = (c.rho * S) * p;
  o.S = S - o.lam;
  o.E = (E + o.lam) - E * m.inv_tau_e;
  o.I = (I + E * m.inv_tau_e) - I * m.inv_tau_i;
  return o;
}

// The elementwise part of a day's adjoint: from the adjoints of the state after the day,
// updates aS and aE to the day's start, adds to r0_bar, returns the day's row entry: mbar, the
// adjoint of the mixed weight, whose rounding every node and day shares through the network
// (((g_bar r0) inv_pop) season in its place, the same product in another order, moved the
// gradients of E and I by 1e-6 of their size, away from float64 on some inputs: 2.6e-6 for
// 1.9e-6).  season_part is mbar / season times m; a season so small that the quotient could
// be lost keeps the row without its factor.
__device__ __forceinline__ bool row_has_season(float season) { return fabsf(season) >= 0x1p-20f; }
__device__ __forceinline__ float row_scale(float season) { return row_has_season(season) ? 1.0f : season; }   // mbar / row
__device__ __forceinline__ float day_adjoint(const lp_mf_model& m, const Node& c, float season, float S0, float mm,
                                             float g, float ainc, float& aS, float& aE, float aI, float& r0_bar) {
  const float p = -lp::expm1f_lp(-g);
  const float q = lp::expf_lp(-g);
  const float lam_bar = (ainc - aS) + aE;
  const float g_bar = ((lam_bar * c.rho) * S0) * q;
  r0_bar += ((g_bar * mm) * season) * c.inv_pop;
  aS = aS + (lam_bar * c.rho) * p;
  aE = aE * (1.0f - m.inv_tau_e) + aI * m.inv_tau_e;
  return ((row_has_season(season) ? g_bar * season : g_bar) * c.r0) * c.inv_pop;
}
// aI at the day's start from aI after it and s = sum_i N_ji mbar_i.
__device__ __forceinline__ float adjoint_i(const lp_mf_model& m, const Node& c, float aI, float mbar, float s) {
  return aI * (1.0f - m.inv_tau_i) + m.iota * fmaf(c.keep, mbar, s);
}

// The seasonality of a call's days, 64 of them in the lanes of every wavefront (a load per day
// would wait, in order, for the trajectory stores before it).
struct Season {
  float v;
  __device__ __forceinline__ void load(const float* season, int t0, int days, int d) {   // the 64 days d is among
    const int j = (d & ~63) + (int)(threadIdx.x & 63);
    v = j < days ? season[t0 + j] : 0.0f;
  }
  __device__ __forceinline__ float at(int d) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), d & 63));
  }
};

// ---- one workgroup -------------------------------------------------------------------
// Sixteen lanes per network row: row group g holds rows g + G q (q < RW, G row groups),
// lane l of it columns l + 16 k (k < K), in registers; lane q of the group is the owner of
// node g + G q and keeps its state.  Bound by the chain of a day (LDS read, K multiply-adds, a row
// sum, the node's formula, LDS write, barrier).
template <int RW, int K>
struct Rows {
  float w[RW][K];
  __device__ __forceinline__ void load(const float* net, int n, int g, int G, int l) {
#pragma unroll
    for (int q = 0; q < RW; ++q) {
      const int i = g + G * q;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int j = l + 16 * k;
        w[q][k] = i < n && j < n ? net[(size_t)i * n + j] : 0.0f;
      }
    }
  }
  // Row l's (l < RW) product with v, in lane l of the group.
  __device__ __forceinline__ float apply(const float* v, int l) const {
    float a[RW], b[RW];
#pragma unroll
    for (int q = 0; q < RW; ++q) a[q] = b[q] = 0.0f;
#pragma unroll
    for (int k = 0; k < K; k += 2) {
      const float x = v[l + 16 * k], y = v[l + 16 * (k + 1)];
#pragma unroll
      for (int q = 0; q < RW; ++q) {
        a[q] = fmaf(w[q][k], x, a[q]);
        b[q] = fmaf(w[q][k + 1], y, b[q]);
      }
    }
    float r = 0.0f;
#pragma unroll
    for (int q = 0; q < RW; ++q) {
      const float s = row_sum(a[q] + b[q]);
      r = l == q ? s : r;
    }
    return r;
  }
};

template <int RW, int K>
__global__ void __launch_bounds__(1024) k_mf_days_wg(lp_mf_model m, int t0, int days, float* S, float* E, float* I,
                                                     float* inc, float* msave, float* gsave) {
  __shared__ float v[2][16 * K];
  const int n = m.n, l = threadIdx.x & 15, g = threadIdx.x >> 4, G = blockDim.x >> 4;
  Rows<RW, K> rows;
  rows.load(m.net_t, n, g, G, l);
  const int i = g + G * l;
  const bool own = l < RW && i < n;
  for (int j = threadIdx.x; j < 2 * 16 * K; j += blockDim.x) (&v[0][0])[j] = 0.0f;
  __syncthreads();
  Node c{};
  float s = 0.0f, e = 0.0f, x = 0.0f;
  if (own) {
    c = node_of(m, i);
    s = S[i]; e = E[i]; x = I[i];
    v[0][i] = x;
  }
  __syncthreads();
  Season seasons;
  for (int d = 0; d < days; ++d) {
    if ((d & 63) == 0) seasons.load(m.season, t0, days, d);
    const float season = seasons.at(d);
    const float mix = rows.apply(v[d & 1], l);
    if (own) {
      const DayOut o = day_forward(m, c, season, mix, s, e, x);
      s = o.S; e = o.E; x = o.I;
      v[(d + 1) & 1][i] = x;
      const size_t r0 = (size_t)d * n + i, r1 = r0 + n;
      S[r1] = s; E[r1] = e; I[r1] = x;
      inc[r0] = o.lam;
      if (msave) msave[r0] = o.mm;
      if (gsave) gsave[r0] = o.g;
    }
    lds_barrier();
  }
}

// A node's inputs of PF days in the adjoint, day hi - 1 first; the next PF days' load while
// these are used.
template <int PF>
struct AdjIn {
  float S0[PF], mm[PF], g[PF], ainc[PF];
  __device__ __forceinline__ void load(bool own, int hi, int n, int i, const float* S, const float* msave, const float* gsave,
                                       const float* a) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const bool on = own && hi - 1 - u >= 0;
      const size_t r = on ? (size_t)(hi - 1 - u) * n + i : 0;
      S0[u] = on ? S[r] : 0.0f;
      mm[u] = on ? msave[r] : 0.0f;
      g[u] = on ? gsave[r] : 0.0f;
      ainc[u] = on ? a[r] : 0.0f;
    }
  }
};

template <int RW, int K>
__global__ void __launch_bounds__(1024) k_mf_adj_wg(lp_mf_model m, int t0, int days, const float* S, const float* msave,
                                                    const float* gsave, const float* ainc, float* aS, float* aE,
                                                    float* aI, float* r0_bar, float* h) {
  constexpr int PF = RW * K >= 64 ? 2 : 8;   // by the registers the network leaves
  __shared__ float v[2][16 * K];
  const int n = m.n, l = threadIdx.x & 15, g = threadIdx.x >> 4, G = blockDim.x >> 4;
  Rows<RW, K> rows;
  rows.load(m.net, n, g, G, l);
  const int i = g + G * l;
  const bool own = l < RW && i < n;
  for (int j = threadIdx.x; j < 2 * 16 * K; j += blockDim.x) (&v[0][0])[j] = 0.0f;
  __syncthreads();
  Node c{};
  float s = 0.0f, e = 0.0f, x = 0.0f, r0 = 0.0f;
  if (own) {
    c = node_of(m, i);
    s = aS[i]; e = aE[i]; x = aI[i]; r0 = r0_bar[i];
  }
  AdjIn<PF> in, next;
  in.load(own, days, n, i, S, msave, gsave, ainc);
  Season seasons;
  seasons.load(m.season, t0, days, days - 1);
  for (int hi = days; hi > 0; hi -= PF) {
    next.load(own, hi - PF, n, i, S, msave, gsave, ainc);
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int d = hi - 1 - u;
      if (d < 0) break;
      const float season = seasons.at(d);
      float mbar = 0.0f;
      if (own) {
        const float hd = day_adjoint(m, c, season, in.S0[u], in.mm[u], in.g[u], in.ainc[u], s, e, x, r0);
        mbar = hd * row_scale(season);
        v[d & 1][i] = mbar;
        h[(size_t)d * n + i] = hd;
      }
      lds_barrier();
      const float sum = rows.apply(v[d & 1], l);
      if (own) x = adjoint_i(m, c, x, mbar, sum);
      if ((d & 63) == 0 && d > 0) seasons.load(m.season, t0, days, d - 1);
    }
    in = next;
  }
  if (own) {
    aS[i] = s; aE[i] = e; aI[i] = x;
    r0_bar[i] = r0;
  }
}

// ---- resident workgroups ---------------------------------------------------------------
// Workgroup b owns rows 16 b .. + 15, wavefront w of its eight rows 16 b + 2 w and + 1, lane l
// columns l + 64 k (k < K) in registers; lanes 0 and 1 own the two nodes.  The vector a day
// needs (the day's I row, or in the adjoint its h row) is passed through its own global
// row: cleared to PENDING (a NaN no owner stores) beforehand, every element is stored
// once by its owner and read by everyone until it has come, both as relaxed agent-scope
// atomics, so no flag, fence or barrier between the workgroups is needed, only that all
// are resident at once (a cooperative launch).  The trajectories are stored after the next
// row has come: a wavefront's memory operations complete in order, so its reads would
// wait for the stores.  Reads that come too early hold up the stores they wait for (all of
// them go to the same lines past the L2s): without the sleep before the first read a day
// took 3.6 us instead of 2.2, and four wavefronts that only waited, or 256- or
// 1024-thread workgroups, were slower too.  A wait ends after `wait_ticks` of the 100 MHz
// clock in any case (a workgroup not resident, or preempted).  The workgroup's owners then store
// NaN everywhere they have not stored yet and return; the rows that others wait for keep
// PENDING, a NaN itself.  So a call that gave up leaves right values and NaN, never what the
// memory held before.
constexpr int RES_WG = 512, RES_ROWS = 16;
constexpr uint32_t PENDING = 0xFFFFFFFFu;
constexpr int64_t TICKS_PER_US = 100;
constexpr int32_t WAIT_US = 10000000;   // 10 s

__global__ void __launch_bounds__(WG) k_mf_pending(uint32_t* p, int64_t n) {
  for (int64_t j = (int64_t)blockIdx.x * WG + threadIdx.x; j < n; j += (int64_t)gridDim.x * WG) p[j] = PENDING;
}
__device__ __forceinline__ void publish(float* p, float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  __hip_atomic_store(reinterpret_cast<uint32_t*>(p), u == PENDING ? 0x7fc00000u : u, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// Elements [0, n) of `row` into LDS vector v, times `scale`; false (in every thread of the
// workgroup) if one did not come within `wait_ticks`, or *s_late was set.  Ends with a barrier.
template <int K>
__device__ __forceinline__ bool await_row(const float* row, int n, float scale, float* v, int* s_late,
                                          int64_t wait_ticks) {
  constexpr int PER = 64 * K / RES_WG;
  const int w = threadIdx.x;
  __builtin_amdgcn_s_sleep(16);   // 16 x 64 cycles: what a row needs to come at least
  uint32_t u[PER];
#pragma unroll
  for (int a = 0; a < PER; ++a) {
    const int j = w + a * RES_WG;
    u[a] = j < n ? __hip_atomic_load(reinterpret_cast<const uint32_t*>(row + j), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
  }
  int64_t t_end = 0;
#pragma unroll
  for (int a = 0; a < PER; ++a) {
    const int j = w + a * RES_WG;
    while (u[a] == PENDING) {
      __builtin_amdgcn_s_sleep(1);
      u[a] = __hip_atomic_load(reinterpret_cast<const uint32_t*>(row + j), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (u[a] != PENDING) break;
      const int64_t now = (int64_t)wall_clock64();
      if (t_end == 0) t_end = now + wait_ticks;
      if (now - t_end > 0) { *s_late = 1; break; }
    }
    v[j] = j < n ? __builtin_bit_cast(float, u[a]) * scale : 0.0f;
  }
  lds_barrier();
  return *s_late == 0;
}

template <int K>
struct TwoRows {
  float w[2][K];
  __device__ __forceinline__ void load(const float* net, int n, int i0, int lane) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int i = i0 + q, j = lane + 64 * k;
        w[q][k] = i < n && j < n ? net[(size_t)i * n + j] : 0.0f;
      }
  }
  // Row `lane`'s (0 or 1) product with v.
  __device__ __forceinline__ float apply(const float* v, int lane) const {
    float a0 = 0.0f, a1 = 0.0f, b0 = 0.0f, b1 = 0.0f;
#pragma unroll
    for (int k = 0; k < K; k += 2) {
      const float x = v[lane + 64 * k], y = v[lane + 64 * (k + 1)];
      a0 = fmaf(w[0][k], x, a0); b0 = fmaf(w[0][k + 1], y, b0);
      a1 = fmaf(w[1][k], x, a1); b1 = fmaf(w[1][k + 1], y, b1);
    }
    const float r0 = wave_sum(a0 + b0), r1 = wave_sum(a1 + b1);
    return lane == 0 ? r0 : r1;
  }
};

template <int K>
__global__ void __launch_bounds__(RES_WG) k_mf_days_res(lp_mf_model m, int t0, int days, float* S, float* E, float* I,
                                                        float* inc, float* msave, float* gsave, int64_t wait_ticks) {
  __shared__ float v[2][64 * K];
  __shared__ int s_late;
  const int n = m.n, lane = threadIdx.x & 63;
  const int i0 = blockIdx.x * RES_ROWS + (threadIdx.x >> 6) * 2, i = i0 + lane;
  if (threadIdx.x == 0) s_late = wait_ticks == 0;
  for (int j = threadIdx.x; j < 64 * K; j += RES_WG) v[0][j] = j < n ? I[j] : 0.0f;
  __syncthreads();
  TwoRows<K> rows;
  rows.load(m.net_t, n, i0, lane);
  const bool own = lane < 2 && i < n;
  Node c{};
  float s = 0.0f, e = 0.0f, x = 0.0f;
  if (own) {
    c = node_of(m, i);
    s = S[i]; e = E[i]; x = I[i];
  }
  DayOut o{};
  auto store = [&](int d) {                               // the trajectories of day d
    if (!own) return;
    const size_t r0 = (size_t)d * n + i, r1 = r0 + n;
    S[r1] = o.S; E[r1] = o.E;
    inc[r0] = o.lam;
    if (msave) msave[r0] = o.mm;
    if (gsave) gsave[r0] = o.g;
  };
  Season seasons;
  for (int d = 0; d < days; ++d) {
    if (d > 0) {
      const bool came = await_row<K>(I + (size_t)d * n, n, 1.0f, v[d & 1], &s_late, wait_ticks);
      store(d - 1);
      if (!came) {
        const float lost = __builtin_nanf("");
        o = DayOut{lost, lost, lost, lost, lost, lost};
        for (; d < days; ++d) store(d);
        return;
      }
    }
    if ((d & 63) == 0) seasons.load(m.season, t0, days, d);
    const float mix = rows.apply(v[d & 1], lane);
    if (own) {
      o = day_forward(m, c, seasons.at(d), mix, s, e, x);
      publish(I + (size_t)(d + 1) * n + i, o.I);
      s = o.S; e = o.E; x = o.I;
    }
  }
  store(days - 1);
}

template <int K>
__global__ void __launch_bounds__(RES_WG) k_mf_adj_res(lp_mf_model m, int t0, int days, const float* S, const float* msave,
                                                       const float* gsave, const float* ainc, float* aS, float* aE,
                                                       float* aI, float* r0_bar, float* h, int64_t wait_ticks) {
  constexpr int PF = 4;
  __shared__ float v[2][64 * K];
  __shared__ int s_late;
  const int n = m.n, lane = threadIdx.x & 63;
  const int i0 = blockIdx.x * RES_ROWS + (threadIdx.x >> 6) * 2, i = i0 + lane;
  if (threadIdx.x == 0) s_late = wait_ticks == 0;
  __syncthreads();
  Season seasons;
  seasons.load(m.season, t0, days, days - 1);
  TwoRows<K> rows;
  rows.load(m.net, n, i0, lane);
  const bool own = lane < 2 && i < n;
  Node c{};
  float s = 0.0f, e = 0.0f, x = 0.0f, r0 = 0.0f;
  if (own) {
    c = node_of(m, i);
    s = aS[i]; e = aE[i]; x = aI[i]; r0 = r0_bar[i];
  }
  AdjIn<PF> in, next;
  in.load(own, days, n, i, S, msave, gsave, ainc);
  for (int hi = days; hi > 0; hi -= PF) {
    next.load(own, hi - PF, n, i, S, msave, gsave, ainc);
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int d = hi - 1 - u;
      if (d < 0) break;
      const float season = seasons.at(d);
      float mbar = 0.0f;
      if (own) {
        const float hd = day_adjoint(m, c, season, in.S0[u], in.mm[u], in.g[u], in.ainc[u], s, e, x, r0);
        publish(h + (size_t)d * n + i, hd);
        mbar = hd * row_scale(season);
      }
      if (!await_row<K>(h + (size_t)d * n, n, row_scale(season), v[d & 1], &s_late, wait_ticks)) {
        if (own) aS[i] = aE[i] = aI[i] = r0_bar[i] = __builtin_nanf("");
        return;
      }
      const float sum = rows.apply(v[d & 1], lane);
      if (own) x = adjoint_i(m, c, x, mbar, sum);
      if ((d & 63) == 0 && d > 0) seasons.load(m.season, t0, days, d - 1);
    }
    in = next;
  }
  if (own) {
    aS[i] = s; aE[i] = e; aI[i] = x;
    r0_bar[i] = r0;
  }
}

// ---- one launch per day -------------------------------------------------------------------
// Fixed-order sum of the 256 per-thread partials of a workgroup.
__device__ __forceinline__ float wg_sum(float v, float* sh) {
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  for (int o = WG / 2; o > 0; o >>= 1) {
    if (tid < o) sh[tid] = sh[tid] + sh[tid + o];
    __syncthreads();
  }
  return sh[0];
}

// One day forward (one workgroup per node): row t of S/E/I -> row t+1; inc, m, g of the day.
__global__ void __launch_bounds__(WG) k_mf_day(lp_mf_model m, int t, const float* S0, const float* E0,
                                               const float* I0, float* S1, float* E1, float* I1, float* inc,
                                               float* msave, float* gsave) {
  __shared__ float sh[WG];
  const int i = blockIdx.x, n = m.n;
  const float* row = m.net_t + (size_t)i * n;
  float acc = 0.0f;
  for (int j = threadIdx.x; j < n; j += WG) acc = fmaf(row[j], I0[j], acc);
  const float mix = wg_sum(acc, sh);
  if (threadIdx.x != 0) return;
  const DayOut o = day_forward(m, node_of(m, i), m.season[t], mix, S0[i], E0[i], I0[i]);
  S1[i] = o.S;
  E1[i] = o.E;
  I1[i] = o.I;
  inc[i] = o.lam;
  if (msave) msave[i] = o.mm;
  if (gsave) gsave[i] = o.g;
}

// The adjoint a day per launch, one workgroup per node: with d < days the network part of
// day d (mbar of that day read from mb_in), then with d > 0 the node's elementwise part
// of day d - 1, whose mbar goes to mb_out.
__global__ void __launch_bounds__(WG) k_mf_adj_day(lp_mf_model m, int t0, int days, int d, const float* S,
                                                   const float* msave, const float* gsave, const float* ainc, float* aS,
                                                   float* aE, float* aI, float* r0_bar, float* h, const float* mb_in,
                                                   float* mb_out) {
  __shared__ float sh[WG];
  const int j = blockIdx.x, n = m.n;
  float s = 0.0f;
  if (d < days) {
    const float* row = m.net + (size_t)j * n;
    float acc = 0.0f;
    for (int i = threadIdx.x; i < n; i += WG) acc = fmaf(row[i], mb_in[i], acc);
    s = wg_sum(acc, sh);
  }
  if (threadIdx.x != 0) return;
  const Node c = node_of(m, j);
  float x = aI[j];
  if (d < days) x = adjoint_i(m, c, x, mb_in[j], s);
  aI[j] = x;
  if (d == 0) return;
  const float season = m.season[t0 + d - 1];
  const size_t r = (size_t)(d - 1) * n + j;
  float a = aS[j], e = aE[j], r0 = r0_bar[j];
  const float hj = day_adjoint(m, c, season, S[r], msave[r], gsave[r], ainc[r], a, e, x, r0);
  aS[j] = a;
  aE[j] = e;
  r0_bar[j] = r0;
  h[r] = hj;
  mb_out[j] = hj * row_scale(season);
}

// ---- after the days --------------------------------------------------------------------
// N_bar[j][i] += sum over the days of beta_j (mbar_i - mbar_j), one workgroup per 32 x 32
// tile, four rows of one column per thread, NB_DAYS days staged in LDS at a time.  The
// day-by-day form read and wrote all of N_bar once a day (2 x 2.4 MB at 774 nodes, 5.3 us a
// day with the product it rode on); this is 19 us for 180 days.
constexpr int NB_TILE = 32, NB_DAYS = 64;
__global__ void __launch_bounds__(WG) k_mf_net_bar(lp_mf_model m, int t0, int days, const float* I, const float* h,
                                                   float* net_bar) {
  __shared__ float s_i[NB_DAYS][NB_TILE];
  __shared__ float4 s_j[NB_DAYS][NB_TILE / 4], s_b[NB_DAYS][NB_TILE / 4];
  const int n = m.n, c = threadIdx.x & (NB_TILE - 1), q = threadIdx.x / NB_TILE;   // column, group of four rows
  const int i0 = blockIdx.x * NB_TILE, j0 = blockIdx.y * NB_TILE, i = i0 + c;
  const int ci = i < n ? i : 0, cj = j0 + c < n ? j0 + c : 0;   // (columns past the last one go unused)
  constexpr int PER = NB_DAYS * NB_TILE / WG;
  // sums go on from N_bar, latest day first: days in one call or several give the same bits
  float acc[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int j = j0 + 4 * q + a;
    acc[a] = i < n && j < n ? net_bar[(size_t)j * n + i] : 0.0f;
  }
  for (int hi = days; hi > 0; hi -= NB_DAYS) {
    const int lo = hi > NB_DAYS ? hi - NB_DAYS : 0;
    __syncthreads();
    float x[PER], y[PER], b[PER], season[PER];   // every load of the stage in flight at once
#pragma unroll
    for (int a = 0; a < PER; ++a) {
      const int day = lo + q + a * (WG / NB_TILE);
      const size_t r = (size_t)(day < hi ? day : hi - 1) * n;
      season[a] = row_scale(m.season[t0 + (day < hi ? day : hi - 1)]);
      x[a] = h[r + ci];
      y[a] = h[r + cj];
      b[a] = I[r + cj];
    }
#pragma unroll
    for (int a = 0; a < PER; ++a) {
      const int d = q + a * (WG / NB_TILE);
      s_i[d][c] = x[a] * season[a];
      reinterpret_cast<float*>(s_j[d])[c] = y[a] * season[a];
      reinterpret_cast<float*>(s_b[d])[c] = m.iota * b[a];
    }
    __syncthreads();
    for (int d = hi - lo - 1; d >= 0; --d) {
      const float x = s_i[d][c];
      const float4 y = s_j[d][q], b = s_b[d][q];
      acc[0] = fmaf(b.x, x - y.x, acc[0]);
      acc[1] = fmaf(b.y, x - y.y, acc[1]);
      acc[2] = fmaf(b.z, x - y.z, acc[2]);
      acc[3] = fmaf(b.w, x - y.w, acc[3]);
    }
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int j = j0 + 4 * q + a;
    if (i < n && j < n && i != j) net_bar[(size_t)j * n + i] = acc[a];
  }
}

// season_part from the rows, in place.
__global__ void __launch_bounds__(WG) k_mf_season(lp_mf_model m, int t0, int days, float* h, const float* msave) {
  const int i = blockIdx.x * WG + threadIdx.x;
  if (i >= m.n) return;
  for (int d = blockIdx.y; d < days; d += gridDim.y) {
    const float season = m.season[t0 + d], mm = msave[(size_t)d * m.n + i];
    float* p = h + (size_t)d * m.n + i;
    *p = (row_has_season(season) ? *p / season : *p) * mm;
  }
}

// Which way a call goes.  The one-workgroup kernels lead the resident ones up to the 256
// nodes whose rows their registers hold; above 2048 nodes two rows a wavefront no longer fit.
// A cooperative launch costs about 20 us more than an ordinary one, so calls of few days
// were faster a launch per day (774 nodes, forward 1 / 5 / 30 / 180 days: 36 / 43 / 84 / 340 us
// against 16 / 32 / 165 / 850; adjoint 45 / 53 / 98 / 367 against 21 / 76 / 267 / 1555).
// The choice goes by the nodes alone all the same: the ways add in different orders, and days
// in one call or in several are to give the same bits.
enum class Path { kOneWorkgroup, kResident, kPerDay };
constexpr int ONE_WG_MAX = 256, RES_MAX = 2048;

Path mf_path(int n, hipStream_t s) {
  if (n <= ONE_WG_MAX) return Path::kOneWorkgroup;
  if (n > RES_MAX) return Path::kPerDay;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) { (void)hipGetLastError(); return Path::kPerDay; }
  if (st != hipStreamCaptureStatusNone) return Path::kPerDay;
  int dev = 0, coop = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess)
    return Path::kPerDay;
  return coop ? Path::kResident : Path::kPerDay;
}

template <typename F>
void one_workgroup(int n, F&& f) {   // f(rows per group, columns per lane as constants; threads)
  const int t = (n + 3) / 4 * 64;    // n <= 64: a row group of 16 lanes per node, whole wavefronts
  if (n <= 32) f(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{}, t);
  else if (n <= 64) f(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{}, t);
  else if (n <= 128) f(std::integral_constant<int, 2>{}, std::integral_constant<int, 8>{}, 1024);
  else f(std::integral_constant<int, 4>{}, std::integral_constant<int, 16>{}, 1024);
}
template <typename F>
hipError_t resident(int n, F&& f) {   // f(columns per lane)
  if (n <= 512) return f(std::integral_constant<int, 8>{});
  if (n <= 1024) return f(std::integral_constant<int, 16>{});
  return f(std::integral_constant<int, 32>{});
}
int fill_grid(int64_t n) { return (int)std::min<int64_t>((n + WG - 1) / WG, 2048); }

}  // namespace lp_mf

extern "C" {

int lp_mf_days_bounded(const lp_mf_model* model, int32_t t0, int32_t t1, float* S, float* E, float* I, float* inc,
                       float* m_save, float* g_save, int32_t wait_us, void* hip_stream) {
  if (!model || model->n <= 0 || t1 < t0 || !S || !E || !I || !inc || wait_us < 0) return LP_ERR_ARG;
  int64_t wait_ticks = wait_us * lp_mf::TICKS_PER_US;
  lp_mf_model m = *model;
  int n = m.n, days = t1 - t0;
  if (days == 0) return LP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(hip_stream);
  switch (lp_mf::mf_path(n, s)) {
    case lp_mf::Path::kOneWorkgroup:
      lp_mf::one_workgroup(n, [&](auto rw, auto k, int threads) {
        hipLaunchKernelGGL((lp_mf::k_mf_days_wg<decltype(rw)::value, decltype(k)::value>), dim3(1), dim3(threads), 0, s, m,
                           t0, days, S, E, I, inc, m_save, g_save);
      });
      break;
    case lp_mf::Path::kResident: {
      const int64_t cells = (int64_t)days * n;
      hipLaunchKernelGGL(lp_mf::k_mf_pending, dim3(lp_mf::fill_grid(cells)), dim3(lp_mf::WG), 0, s,
                         reinterpret_cast<uint32_t*>(I + n), cells);
      const hipError_t e = lp_mf::resident(n, [&](auto k) {
        void* args[] = {&m, &t0, &days, &S, &E, &I, &inc, &m_save, &g_save, &wait_ticks};
        return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&lp_mf::k_mf_days_res<decltype(k)::value>),
                                          dim3((n + lp_mf::RES_ROWS - 1) / lp_mf::RES_ROWS), dim3(lp_mf::RES_WG), args, 0, s);
      });
      if (e == hipSuccess) break;
      (void)hipGetLastError();   // not to be had now: a launch per day
      [[fallthrough]];
    }
    case lp_mf::Path::kPerDay:
      for (int d = 0; d < days; ++d) {
        const size_t r0 = (size_t)d * n, r1 = (size_t)(d + 1) * n;
        hipLaunchKernelGGL(lp_mf::k_mf_day, dim3(n), dim3(lp_mf::WG), 0, s, m, t0 + d, S + r0, E + r0, I + r0,
                           S + r1, E + r1, I + r1, inc + r0, m_save ? m_save + r0 : nullptr, g_save ? g_save + r0 : nullptr);
      }
      break;
  }
  return hipGetLastError() == hipSuccess ? LP_OK : LP_ERR_HIP;
}

int lp_mf_days(const lp_mf_model* model, int32_t t0, int32_t t1, float* S, float* E, float* I, float* inc,
               float* m_save, float* g_save, void* hip_stream) {
  return lp_mf_days_bounded(model, t0, t1, S, E, I, inc, m_save, g_save, lp_mf::WAIT_US, hip_stream);
}

int lp_mf_adjoint_days_noalloc(const lp_mf_model* model, int32_t t0, int32_t t1, const float* S, const float* I,
                               const float* m_save, const float* g_save, const float* a_inc, float* aS, float* aE,
                               float* aI, float* r0_bar, float* net_bar, float* season_part, void* hip_stream) {
  if (!model || model->n <= 0 || model->n > LP_MF_NOALLOC_MAX_NODES) return LP_ERR_ARG;
  float* work = nullptr;
  const int rc = lp_mf::scratch_of_current_device(&work);
  if (rc) return rc;
  // every work row is written before it is read, so the previous call's contents need
  // no clearing
  return lp_mf_adjoint_days(model, t0, t1, S, I, m_save, g_save, a_inc, aS, aE, aI, r0_bar, net_bar,
                            season_part, work, hip_stream);
}

int lp_mf_adjoint_days(const lp_mf_model* model, int32_t t0, int32_t t1, const float* S, const float* I,
                       const float* m_save, const float* g_save, const float* a_inc, float* aS, float* aE,
                       float* aI, float* r0_bar, float* net_bar, float* season_part, float* work,
                       void* hip_stream) {
  return lp_mf_adjoint_days_bounded(model, t0, t1, S, I, m_save, g_save, a_inc, aS, aE, aI, r0_bar, net_bar,
                                    season_part, work, lp_mf::WAIT_US, hip_stream);
}

int lp_mf_adjoint_days_bounded(const lp_mf_model* model, int32_t t0, int32_t t1, const float* S, const float* I,
                               const float* m_save, const float* g_save, const float* a_inc, float* aS, float* aE,
                               float* aI, float* r0_bar, float* net_bar, float* season_part, float* work,
                               int32_t wait_us, void* hip_stream) {
  if (!model || model->n <= 0 || t1 < t0 || !S || !I || !m_save || !g_save || !a_inc || !aS || !aE || !aI ||
      !r0_bar || !net_bar || !season_part || !work || wait_us < 0)
    return LP_ERR_ARG;
  int64_t wait_ticks = wait_us * lp_mf::TICKS_PER_US;
  lp_mf_model m = *model;
  int n = m.n, days = t1 - t0;
  if (days == 0) return LP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(hip_stream);
  float* h = season_part;
  const int64_t cells = (int64_t)days * n;
  switch (lp_mf::mf_path(n, s)) {
    case lp_mf::Path::kOneWorkgroup:
      lp_mf::one_workgroup(n, [&](auto rw, auto k, int threads) {
        hipLaunchKernelGGL((lp_mf::k_mf_adj_wg<decltype(rw)::value, decltype(k)::value>), dim3(1), dim3(threads), 0, s, m,
                           t0, days, S, m_save, g_save, a_inc, aS, aE, aI, r0_bar, h);
      });
      break;
    case lp_mf::Path::kResident: {
      hipLaunchKernelGGL(lp_mf::k_mf_pending, dim3(lp_mf::fill_grid(cells)), dim3(lp_mf::WG), 0, s,
                         reinterpret_cast<uint32_t*>(h), cells);
      const hipError_t e = lp_mf::resident(n, [&](auto k) {
        void* args[] = {&m, &t0, &days, &S, &m_save, &g_save, &a_inc, &aS, &aE, &aI, &r0_bar, &h, &wait_ticks};
        return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&lp_mf::k_mf_adj_res<decltype(k)::value>),
                                          dim3((n + lp_mf::RES_ROWS - 1) / lp_mf::RES_ROWS), dim3(lp_mf::RES_WG), args, 0, s);
      });
      if (e == hipSuccess) break;
      (void)hipGetLastError();   // not to be had now: a launch per day
      [[fallthrough]];
    }
    case lp_mf::Path::kPerDay:
      // launch d takes the network part of day d and the elementwise part of day d - 1
      for (int d = days; d >= 0; --d)
        hipLaunchKernelGGL(lp_mf::k_mf_adj_day, dim3(n), dim3(lp_mf::WG), 0, s, m, t0, days, d, S, m_save, g_save, a_inc,
                           aS, aE, aI, r0_bar, h, work + (size_t)(d & 1) * n, work + (size_t)((d + 1) & 1) * n);
      break;
  }
  const int tiles = (n + lp_mf::NB_TILE - 1) / lp_mf::NB_TILE;
  hipLaunchKernelGGL(lp_mf::k_mf_net_bar, dim3(tiles, tiles), dim3(lp_mf::WG), 0, s, m, t0, days, I, h, net_bar);
  hipLaunchKernelGGL(lp_mf::k_mf_season, dim3((n + lp_mf::WG - 1) / lp_mf::WG, std::min(days, 1024)), dim3(lp_mf::WG), 0, s, m, t0,
                     days, h, m_save);
  return hipGetLastError() == hipSuccess ? LP_OK : LP_ERR_HIP;
}

}  // extern "C"
