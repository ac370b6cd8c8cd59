#pragma once
// Population initialisation on the device (lp_init_population, include/lp_step.h):
// the per-agent columns that SEIR_ABM and its components draw at construction
// (model.py:561-713 ages, immunity, initial infections; 816-866 heterogeneity;
// 568-587 disease timers; 1548-1669 death dates; 1887-1894 RI timers), for every
// slot of every node segment, from counter-based Philox streams keyed by (init seed,
// sim-local slot).  Draws use float32 samplers of the named distributions; they are
// the same distributions as the host generator's, not the same numbers.
#include "lp_kernels.hip"

namespace lp {

constexpr uint32_t ST_INIT = 9;   // Philox stream of the initial draws (sub-stream << 8)
enum : uint32_t { SI_AGE = 0, SI_AGE2, SI_EXP, SI_INF, SI_PAR, SI_HET, SI_STATE, SI_RI, SI_MISSED };

// Uniform in (0, 1) from the top 24 bits.
__device__ __forceinline__ float u01o(uint32_t r) { return ((float)(r >> 8) + 0.5f) * 5.9604644775390625e-08f; }

// Standard normal by Box-Muller from two 32-bit draws.
__device__ __forceinline__ float normal_bm(uint32_t r1, uint32_t r2) {
  const float u1 = u01o(r1), u2 = u01o(r2);
  return sqrtf(-2.0f * logf(u1)) * cosf(6.2831853071795865f * u2);
}

// Draw j of sub-stream `sub` for agent `slot` (the day word holds -1 - j: no step
// of a run uses negative days).
__device__ __forceinline__ uint4 init_draw(uint64_t seed, uint64_t slot, uint32_t sub, uint32_t j) {
  return philox((uint32_t)slot, (uint32_t)(slot >> 32), (uint32_t)(-1 - (int32_t)j), ST_INIT | (sub << 8), seed);
}

// Gamma(shape k, scale theta) by Marsaglia & Tsang (ACM TOMS 26(3), 2000): for k >= 1
// d = k - 1/3, c = 1/sqrt(9d), x ~ N(0,1), v = (1 + c x)^3, accept d v when
// log u < x^2/2 + d - d v + d log v; for k < 1, Gamma(k + 1) * u^(1/k).  One attempt, the j-th;
// false if it is rejected.
__device__ __forceinline__ bool gamma_try(float dd, float c, uint64_t seed, uint64_t slot, uint32_t sub, uint32_t j, float& g) {
  const uint4 o = init_draw(seed, slot, sub, j);
  const float x = normal_bm(o.x, o.y);
  const float t = 1.0f + c * x;
  if (t <= 0.0f) return false;
  const float v = t * t * t;
  const float u = u01o(o.z);
  if (!(logf(u) < 0.5f * x * x + dd - dd * v + dd * logf(v))) return false;
  g = dd * v;
  return true;
}

// Per wavefront: a sample of each of its 256 agents (agent 4 l + a is slot a of lane l), and the
// agents whose first gamma attempt was rejected.  The samples go through LDS so that the
// loops over a lane's agents need not be unrolled: fewer registers, more wavefronts.
struct WaveSamples {
  float g[256];
  uint16_t list[256];
};
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Gamma samples of the wave's agents (slots slot0 + agent) into w.g.  Every agent's first attempt,
// then the agents it was rejected for (1 in 20 at shape 4.5) gathered one per lane: a
// wavefront repeating its 64 agents until the last one is accepted takes 2.2 attempts of
// every lane, this way 1.1.
__device__ __forceinline__ void gamma_mt4(float k, float theta, uint64_t seed, uint64_t slot0, uint32_t sub, int lane,
                                          WaveSamples& w) {
  const bool boost = k < 1.0f;
  const float kk = boost ? k + 1.0f : k;
  const float dd = kk - 1.0f / 3.0f, c = 1.0f / sqrtf(9.0f * dd);
  int tot = 0;
#pragma unroll 1
  for (int a = 0; a < 4; ++a) {
    const int at = 4 * lane + a;
    float g = dd;
    const bool r = !gamma_try(dd, c, seed, slot0 + (uint64_t)at, sub, 0, g);
    w.g[at] = g;
    const uint64_t mk = __ballot(r);
    if (r) w.list[tot + __popcll(mk & ((1ull << lane) - 1ull))] = (uint16_t)at;
    tot += __popcll(mk);
  }
  if (tot) {                                              // uniform
    wave_lds_fence();
    for (int b = lane; b < tot; b += 64) {
      const int at = w.list[b];
      float g = dd;
      for (uint32_t j = 1; j < 64; ++j)
        if (gamma_try(dd, c, seed, slot0 + (uint64_t)at, sub, j, g)) break;
      w.g[at] = g;
    }
    wave_lds_fence();
  }
#pragma unroll 1
  for (int a = 0; a < 4; ++a) {
    const int at = 4 * lane + a;
    float g = w.g[at];
    if (boost) {
      const uint4 o = init_draw(seed, slot0 + (uint64_t)at, sub, 64);
      g *= powf(u01o(o.x), 1.0f / k);
    }
    w.g[at] = g * theta;
  }
}

// A sample of duration distribution `ds` (lp_dist, but for gamma: gamma_mt4) for agent `slot`.
__device__ float dist_sample(const lp_dist& ds, uint64_t seed, uint64_t slot, uint32_t sub) {
  switch (ds.kind) {
    case LP_DIST_CONSTANT: return ds.a;
    case LP_DIST_NORMAL: { const uint4 o = init_draw(seed, slot, sub, 0); return ds.a + ds.b * normal_bm(o.x, o.y); }
    case LP_DIST_LOGNORMAL: {
      if (!(ds.a > 0.0f)) return 0.0f;
      const float m = ds.a, s = ds.b;
      const float mu = logf((m * m) / sqrtf(s * s + m * m)), sg = sqrtf(logf((s * s) / (m * m) + 1.0f));
      const uint4 o = init_draw(seed, slot, sub, 0);
      return expf(mu + sg * normal_bm(o.x, o.y));
    }
    case LP_DIST_POISSON: {                                // inversion (small means: durations)
      const uint4 o = init_draw(seed, slot, sub, 0);
      const float u = u01o(o.x);
      float p = expf(-ds.a), F = p;
      int k = 0;
      while (u > F && k < 1000) { k += 1; p = p * ds.a / (float)k; F += p; }
      return (float)k;
    }
    case LP_DIST_EXPONENTIAL: { const uint4 o = init_draw(seed, slot, sub, 0); return -ds.a * logf(u01o(o.x)); }
    case LP_DIST_UNIFORM_INT: {
      const uint4 o = init_draw(seed, slot, sub, 0);
      return floorf(ds.a + u01o(o.x) * (ds.b - ds.a));
    }
    default: return 0.0f;
  }
}

// Samples of `ds` for the wave's agents (slots slot0 + agent): this lane's four.
__device__ __forceinline__ float4 dist_sample4(const lp_dist& ds, uint64_t seed, uint64_t slot0, uint32_t sub, int lane,
                                               WaveSamples& w) {
  if (ds.kind == LP_DIST_GAMMA) {                         // uniform
    gamma_mt4(ds.a, ds.b, seed, slot0, sub, lane, w);
  } else {
#pragma unroll 1
    for (int a = 0; a < 4; ++a) w.g[4 * lane + a] = dist_sample(ds, seed, slot0 + (uint64_t)(4 * lane + a), sub);
  }
  return reinterpret_cast<const float4*>(w.g)[lane];
}

// Float duration -> timer: truncated toward zero, clipped to [0, 127] (model.py:575-579).
__device__ __forceinline__ uint32_t to_timer(float x) {
  const float tr = truncf(x);
  return tr <= 0.0f ? 0u : tr >= 127.0f ? 127u : (uint32_t)tr;
}

// Age in days of an initial agent (exponential capped, or a pyramid bin then a day in it).
__device__ int32_t init_age(const lp_init_sim& sp, uint64_t seed, uint64_t slot) {
  const uint4 o = init_draw(seed, slot, SI_AGE, 0);
  int32_t age;
  if (sp.age_model == 0) {
    float a = -sp.age_mean_days * logf(u01o(o.x));
    if (a > sp.age_cap_days) a = sp.age_cap_days;
    age = (int32_t)a;
  } else {
    const float u = u01o(o.x);
    int b = 0;
    while (b < sp.n_pyr - 1 && u >= sp.pyr_cdf[b]) ++b;
    const int32_t lo = sp.pyr_lo[b], hi = sp.pyr_hi[b];
    age = lo + (int32_t)floorf(u01o(o.y) * (float)(hi - lo));
  }
  return age == 0 ? 1 : age;
}

// One workgroup per tile, one quad of slots per thread: every slot's timers and multipliers;
// the initial agents' ages, death dates, immunity, RI timers and node ids; unborn slots'
// defaults.  Each group of columns is stored before the next is drawn and the loops over a
// thread's agents are not unrolled, so few registers are live (68; 117 with everything
// in one unrolled body).  Bound by the draws (eight Philox blocks and the samplers'
// logarithms, roots and cosines per agent): 4.9 ms for 269 M slots, of which 2.0 ms are
// the 32 bytes a slot; 7.5 ms before, 5.4 with the shorter Philox rounds alone.
__global__ void __launch_bounds__(WG) k_init(Dev d, const lp_init_sim* specs) {
  const int tile = d.tiles[blockIdx.x], u = tile & ((1 << d.tpw_sh) - 1);
  const int4 span = d.spans[tile >> d.tpw_sh];
  const int node = span.x, sim = span.w;
  const lp_sim_params& simp = d.sims[sim];
  const lp_init_sim& sp = specs[sim];
  const uint64_t seed = sp.seed;
  const int64_t live_hi = d.live_end[node];
  __shared__ __align__(16) WaveSamples s_w[WG / 64];
  __shared__ int64_t s_km[LP_KM_LEN];   // the simulation's mortality table: a search of dependent loads per agent
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x < LP_KM_LEN) s_km[threadIdx.x] = d.km_cd[(size_t)sim * LP_KM_LEN + threadIdx.x];
  __syncthreads();
  const int64_t i0 = ((int64_t)span.y + u) * LP_TILE + (int64_t)threadIdx.x * 4;
  const int64_t q0 = i0 >> 2;
  const uint64_t slot0 = (uint64_t)(i0 - 4 * lane - simp.slot_base);   // the wave's first slot
  auto pack2 = [](const uint32_t (&v)[4]) {
    return make_uint2((v[0] & 0xffffu) | (v[1] << 16), (v[2] & 0xffffu) | (v[3] << 16));
  };
  // disease timers: every slot (newborns inherit theirs)
  {
    uint32_t et[4], it[4], pt[4];
    float4 f = dist_sample4(sp.dur_exp, seed, slot0, SI_EXP, lane, s_w[wave]);
#pragma unroll
    for (int a = 0; a < 4; ++a) et[a] = to_timer(lane_of(f, a));
    reinterpret_cast<uint2*>(d.exp_timer)[q0] = pack2(et);
    f = dist_sample4(sp.dur_inf, seed, slot0, SI_INF, lane, s_w[wave]);
#pragma unroll
    for (int a = 0; a < 4; ++a) it[a] = to_timer(lane_of(f, a));
    reinterpret_cast<uint2*>(d.inf_timer)[q0] = pack2(it);
    f = dist_sample4(sp.t_to_paralysis, seed, slot0, SI_PAR, lane, s_w[wave]);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float pr = lane_of(f, a) - (float)et[a];
      const float pmax = (float)it[a];
      pr = pr < 0.0f ? 0.0f : pr > pmax ? pmax : pr;
      pt[a] = (uint32_t)pr;
    }
    reinterpret_cast<uint2*>(d.par_timer)[q0] = pack2(pt);
  }
  // heterogeneity: every slot
  {
    float4 inf = make_float4(sp.inf_mean, sp.inf_mean, sp.inf_mean, sp.inf_mean), risk = make_float4(1.f, 1.f, 1.f, 1.f);
    if (sp.het_model != 0) {                              // uniform
      float* s_risk = s_w[wave].g + 4 * lane;
#pragma unroll 1
      for (int a = 0; a < 4; ++a) {
        const uint4 o = init_draw(seed, slot0 + (uint64_t)(4 * lane + a), SI_HET, 0);
        const float z0 = normal_bm(o.x, o.y), z1 = normal_bm(o.z, o.w);
        const float y1 = sp.rho * z0 + sqrtf(1.0f - sp.rho * sp.rho) * z1;   // Cholesky of [[1, rho], [rho, 1]]
        s_risk[a] = expf(sp.risk_mu + sp.risk_sigma * z0);
        float v;
        if (sp.het_model == 1) {
          v = sp.inf_mean * expf(sp.risk_mu + sp.risk_sigma * y1);
        } else {
          // Gamma(shape 1) quantile of Phi(y1): -mean * log(1 - Phi(y1)) = -mean * log(Phi(-y1))
          v = -sp.inf_mean * logf(0.5f * erfcf(y1 * 0.70710678118654752f));
        }
        inf = make_float4(inf.y, inf.z, inf.w, v);
      }
      risk = reinterpret_cast<const float4*>(s_w[wave].g)[lane];
    }
    reinterpret_cast<float4*>(d.risk)[q0] = risk;
    reinterpret_cast<float4*>(d.infect)[q0] = inf;
  }
  // the initial agents; unborn slots keep the defaults (agent a enters at the top of each
  // pack, three more rotations bring it to its place)
  uint32_t st = 0, mi = 0;
  uint64_t nid = 0, ri = 0;
  int4 dob = make_int4(0, 0, 0, 0), dod = dob;
#pragma unroll 1
  for (int a = 0; a < 4; ++a) {
    int32_t b_day = -1, d_day = sp.vd ? 0 : INT_MAX;
    int16_t n_id = -1, r_t = -1;
    int8_t s = -1, missed = 0;
    if (i0 + a < live_hi) {
      const uint64_t slot = slot0 + (uint64_t)(4 * lane + a);
      const int32_t age = init_age(sp, seed, slot);
      b_day = -age;
      s = 0;
      const uint4 o = init_draw(seed, slot, SI_STATE, 0);
      if (sp.init_immun > 0.0f && u01o(o.x) < sp.init_immun) s = 3;
      const float ub = u01o(o.y);                        // one draw for all age bands
      for (int b = 0; b < sp.n_bands; ++b)
        if (age >= sp.band_lo[b] && age < sp.band_hi[b] && ub < sp.band_frac[b]) s = 3;
      if (sp.vd) d_day = km_age_at_death(s_km, seed, slot, -1, age) - age;
      if (sp.ri) {
        const float days = sp.ri_hi > sp.ri_lo ? sp.ri_lo + u01o(init_draw(seed, slot, SI_RI, 0).x) * (sp.ri_hi - sp.ri_lo)
                                               : sp.ri_lo;
        r_t = (int16_t)(int32_t)((float)b_day + days);
      }
      if (sp.missed_frac > 0.0f && u01o(o.z) < sp.missed_frac) missed = 1;
      n_id = (int16_t)(node - simp.node_begin);
    }
    st = (st >> 8) | ((uint32_t)(uint8_t)s << 24);
    mi = (mi >> 8) | ((uint32_t)(uint8_t)missed << 24);
    nid = (nid >> 16) | ((uint64_t)(uint16_t)n_id << 48);
    ri = (ri >> 16) | ((uint64_t)(uint16_t)r_t << 48);
    dob = make_int4(dob.y, dob.z, dob.w, b_day);
    dod = make_int4(dod.y, dod.z, dod.w, d_day);
  }
  reinterpret_cast<uint32_t*>(d.state)[q0] = st;
  reinterpret_cast<uint32_t*>(d.strain)[q0] = 0u;
  reinterpret_cast<uint32_t*>(d.pp)[q0] = 0xFFFFFFFFu;  // potentially_paralyzed -1
  reinterpret_cast<uint32_t*>(d.paralyzed)[q0] = 0u;
  reinterpret_cast<uint32_t*>(d.ipv)[q0] = 0u;
  reinterpret_cast<uint32_t*>(d.missed)[q0] = mi;
  reinterpret_cast<uint64_t*>(d.node_id)[q0] = nid;
  reinterpret_cast<uint64_t*>(d.ri_timer)[q0] = ri;
  reinterpret_cast<int4*>(d.dob)[q0] = dob;
  reinterpret_cast<int4*>(d.dod)[q0] = dod;
}

// The initial infections chosen by the host (exact counts per node): state I.
__global__ void k_init_infected(Dev d, const int64_t* slots, int64_t n) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = slots[j];
    if (i >= 0 && i < d.capacity && d.state[i] >= 0) d.state[i] = 2;
  }
}

}  // namespace lp
