// The gravity migration network built on the device (lp_build_network,
// include/lp_step.h), per simulation of the context, into the bound "network_t"
// (float32, each simulation's n x n block transposed) and "keep" (1 - row sum):
//   w_ij = k p_i^a p_j^b / d_ij^c for j != i (non-finite -> 0)     laser_core gravity as
//   w_ij /= (sum_j p_j)^c                                         model.py:1243-1251 calls it
//   rows whose sum exceeds max_rowsum scaled down to it           row_normalizer, model.py:1258
// in float64, cast to float32 at the end, as the host builds it (network.py).  Three
// passes: the powers of the populations and of their sum, one per node and simulation;
// one workgroup per row for the entries, row sums, scales and keep, the entries kept in
// float64; then 64 x 64 tiles staged in LDS so both the reads (row-major) and the
// network_t writes (transposed) are contiguous.  Bound by the float64 power of each
// distance, one per entry (five per entry when each pass took the powers it needed itself:
// 120 us for 4 networks of 774 nodes, 44 us now).
#include "lp_kernels.hip"

namespace lp {

constexpr int NET_TILE = 64;

// w_ij before the row scale, from kpa_i = k p_i^a and pb_j = p_j^b.
__device__ __forceinline__ double gravity_w(const lp_gravity_spec& g, double kpa_i, double pb_j, double d_ij,
                                            double inv_sc, bool diag) {
  if (diag) return 0.0;
  double w = kpa_i * pb_j / pow(d_ij, g.c);
  if (!isfinite(w)) w = 0.0;
  return w * inv_sc;
}

// Sum of v over the workgroup, in a fixed order (lane partials, then a tree in LDS).
__device__ double block_sum_f64(double v, double* red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int s = WG / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  const double out = red[0];
  __syncthreads();
  return out;
}

// Scratch of a build: per node k p^a, p^b and the row scale, per simulation 1 / S^c, and, when
// there is room, every entry before the row scale (at its network_t offset's row-major place).
struct NetScratch {
  double *kpa, *pb, *row_scale, *inv_sc, *w;
};

// Simulation blockIdx.x, nodes blockIdx.y * WG + thread.
__global__ void __launch_bounds__(WG) k_net_pow(Dev d, const lp_gravity_spec* specs, const double* pop, NetScratch x) {
  __shared__ double red[WG];
  const int sim = blockIdx.x;
  const lp_sim_params& sp = d.sims[sim];
  const lp_gravity_spec g = specs[sim];
  const int nb = sp.node_begin, m = sp.n_nodes, j = (int)blockIdx.y * WG + (int)threadIdx.x;
  if (j < m) {
    const double p = pop[nb + j];
    x.kpa[nb + j] = g.k * pow(p, g.a);
    x.pb[nb + j] = pow(p, g.b);
  }
  if (blockIdx.y != 0) return;
  double s = 0.0;
  for (int i = threadIdx.x; i < m; i += WG) s += pop[nb + i];
  const double total = block_sum_f64(s, red);
  if (threadIdx.x == 0) x.inv_sc[sim] = 1.0 / pow(total, g.c);
}

// One workgroup per node i (global index): its row's entries, their sum, the row scale and
// keep[i].
__global__ void __launch_bounds__(WG) k_net_rows(Dev d, const lp_gravity_spec* specs, const double* dist, NetScratch x) {
  __shared__ double red[WG];
  const int n = blockIdx.x;
  const int sim = d.node_sim[n];
  const lp_sim_params& sp = d.sims[sim];
  const lp_gravity_spec g = specs[sim];
  const int nb = sp.node_begin, m = sp.n_nodes, i = n - nb;
  const double inv_sc = x.inv_sc[sim], kpa = x.kpa[n];
  const int64_t row = sp.net_off + (int64_t)i * m;
  double acc = 0.0;
  for (int j = threadIdx.x; j < m; j += WG) {
    const double w = gravity_w(g, kpa, x.pb[nb + j], dist[row + j], inv_sc, j == i);
    if (x.w) x.w[row + j] = w;
    acc += w;
  }
  const double rs = block_sum_f64(acc, red);
  if (threadIdx.x == 0) {
    const double scale = rs > g.max_rowsum ? g.max_rowsum / rs : 1.0;
    x.row_scale[n] = scale;
    const_cast<float*>(d.keep)[n] = (float)(1.0 - rs * scale);
  }
}

// Tile (ti, tj) of simulation blockIdx.y: rows i0..i0+63, columns j0..j0+63 of its network,
// written transposed into network_t[net_off + j * m + i].
__global__ void __launch_bounds__(WG) k_net_tiles(Dev d, const lp_gravity_spec* specs, const double* dist, NetScratch x) {
  __shared__ float tile[NET_TILE][NET_TILE + 1];
  const int sim = blockIdx.y;
  const lp_sim_params& sp = d.sims[sim];
  const int m = sp.n_nodes, nb = sp.node_begin;
  const int tiles = (m + NET_TILE - 1) / NET_TILE;
  if ((int)blockIdx.x >= tiles * tiles) return;
  const lp_gravity_spec g = specs[sim];
  const int i0 = ((int)blockIdx.x / tiles) * NET_TILE, j0 = ((int)blockIdx.x % tiles) * NET_TILE;
  const int c = threadIdx.x & (NET_TILE - 1), r0 = threadIdx.x / NET_TILE;   // 4 rows per pass
  // rows of the tile: contiguous reads along j
#pragma unroll 4
  for (int r = r0; r < NET_TILE; r += WG / NET_TILE) {
    const int i = i0 + r, j = j0 + c;
    float v = 0.0f;
    if (i < m && j < m) {
      const int64_t at = sp.net_off + (int64_t)i * m + j;
      const double w = x.w ? x.w[at] : gravity_w(g, x.kpa[nb + i], x.pb[nb + j], dist[at], x.inv_sc[sim], i == j);
      v = (float)(w * x.row_scale[nb + i]);
    }
    tile[r][c] = v;
  }
  __syncthreads();
  // columns of the tile: contiguous network_t writes along i
  float* out = const_cast<float*>(d.network_t) + sp.net_off;
  for (int r = r0; r < NET_TILE; r += WG / NET_TILE) {
    const int j = j0 + r, i = i0 + c;
    if (i < m && j < m) out[(int64_t)j * m + i] = tile[c][r];
  }
}

}  // namespace lp
