// mpm_kernels.hip -- gfx950 kernels of the explicit MPM substep and their host launchers.
//
// Data layout in HBM (a context holds one scene, or several scenes side by side):
//   particles   two ping-pong buffers of NPLANES float planes of `cap` floats each (SoA):
//               x(3) v(3) B(9) F(9) plastic m V phi id(int bits) V*tau(6). After the first substep
//               the planes are kept physically sorted by cell key, so every particle pass streams
//               them. A cloth's vertices and elements are particles of the same buffers.
//   keys        uint32 cell key per particle in the current physical order (written by G2P).
//   sort        per-cell counts of the next sort (made by G2P, zero from a sort to the next G2P), by state
//               buffer a flag per tile and per scan block of cells, cell_start over all cells plus one, scan
//               block totals; LSD radix besides: K1/K2 keys and V1/V2 index ping-pong buffers, tickets and
//               per-pass look-back status words.
//   grid        dense planes m, mom(3) and interleaved float4 pairs (v, v_BF) over the nodes; only
//               the 4x4x4 node blocks around active tiles are written each substep.
//   tiles       4x4x4-cell tiles: slot per tile (-1 = inactive), active list, per-slot P2G partials
//               over the tile's 7x7x7 node footprint.
//
// Substep (stress at F^n): scan block totals and tile lists -> cell scan (small grids: in the first launch) ->
// cell scatter -> cell rank (bins) -> p2g -> grid -> g2p (counts the next sort's cells) -> apex finish.
// Reference-compatible substep (stress at predicted F^): p2g(momentum) -> grid(normalise) -> stress at F^ ->
// p2g(force) -> grid(force update) replace the p2g -> grid pair. A cloth adds its vertex forces before P2G, the
// fixed-vertex node stops after the grid update, and the element update (directions, QR return map, the next
// substep's element forces) after G2P. The surrogate adds the position lists and its kernel after G2P.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "mpm_device.hpp"
#include "mpm_kernels.h"
#include "mpm_mlp_device.hpp"

namespace mpm {

// ================================================================== small helpers
__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }

// Indices read from device buffers are kept inside [0, n) so that an inconsistent buffer can only
// produce wrong values, never an out-of-bounds access.
__device__ __forceinline__ int clamp_index(int i, int n) { return i < 0 ? 0 : (i >= n ? n - 1 : i); }

// Element i of a plane whose address is uniform, through a 32-bit byte offset: one vector register and no
// 64-bit address arithmetic per access (a state plane holds fewer than 2^30 particles: 35 planes of as many
// floats would not fit any device).
__device__ __forceinline__ float plane_load(const float* plane, uint32_t i) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(plane) + (size_t)(uint32_t)(4u * i));
}

// wave-uniform float held in a scalar register (the readfirstlane builtin works on 32-bit integers)
__device__ __forceinline__ float uniform_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}

// The scene parameters of a workgroup-uniform scene, read once and held in scalar registers for the
// whole kernel (the table lives in global memory, which the compiler reads with a vector load at
// every use otherwise). The level-set primitives are not copied: kernels that use this copy do not
// evaluate level sets.
__device__ __forceinline__ DevParams uniform_params(const DevParams& G) {
  DevParams P;
  const auto ui = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  P.order = ui(G.order);
  P.material = ui(G.material);
  P.predicted = ui(G.predicted);
  P.friction_model = ui(G.friction_model);
  P.lambda0 = uniform_f(G.lambda0);
  P.mu0 = uniform_f(G.mu0);
  P.theta_c = uniform_f(G.theta_c);
  P.theta_s = uniform_f(G.theta_s);
  P.xi = uniform_f(G.xi);
  P.h0 = uniform_f(G.h0);
  P.h1 = uniform_f(G.h1);
  P.h2 = uniform_f(G.h2);
  P.h3 = uniform_f(G.h3);
  P.per_particle_phi = ui(G.per_particle_phi);
  P.alpha_f = uniform_f(G.alpha_f);
  const long long ad = __builtin_bit_cast(long long, G.alpha_d);
  P.alpha_d = __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)ui((int)(ad >> 32)) << 32) |
                                                    (unsigned)ui((int)ad)));
  P.friction = uniform_f(G.friction);
  P.damping = uniform_f(G.damping);
  P.svd_ratio = uniform_f(G.svd_ratio);
  P.apex_radius = uniform_f(G.apex_radius);
  P.dinv = uniform_f(G.dinv);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    P.gravity[d] = uniform_f(G.gravity[d]);
    P.gmin[d] = uniform_f(G.gmin[d]);
    P.h[d] = uniform_f(G.h[d]);
    P.inv_h[d] = uniform_f(G.inv_h[d]);
    P.res[d] = ui(G.res[d]);
    P.tiles[d] = ui(G.tiles[d]);
  }
  P.nls = 0;
  P.mesh_v0 = ui(G.mesh_v0);
  P.mesh_e0 = ui(G.mesh_e0);
  P.mesh_e1 = ui(G.mesh_e1);
  P.c_mu = uniform_f(G.c_mu);
  P.c_lambda = uniform_f(G.c_lambda);
  P.c_gamma = uniform_f(G.c_gamma);
  P.c_k = uniform_f(G.c_k);
  P.c_cf = uniform_f(G.c_cf);
  return P;
}

// Exact cell index along one axis: the number of thresholds thr[c] <= x, where thr[c] is the
// smallest float f with (double(f) - min)/h >= c. This equals static_cast<int>((x - min)/h) of the
// reference evaluated in double (HybridSolver.cpp:33-36) for x >= min, using FP32 compares only.
// The FP32 quotient t is within inv_h (2^-24 |gmin| + 2^-24 |x - gmin|) + 2^-24 |t| (rounded bounds, difference,
// spacing and product), less than 2^-22 (|gmin| inv_h + |t|), of the exact one: where t is farther than that
// from a whole number, floor(t) is the cell, and the thresholds of the cell itself are not gathered (k_g2p with
// them 386 -> 365 us at 2^22 particles, 185 -> 177 us for 16 scenes of 1.8 M).
// lo, hi: thr[0] and thr[res].
__device__ __forceinline__ int axis_cell(const float* thr, float lo, float hi, int res, float x, float gmin, float inv_h,
                                         int& oob) {
  if (!(x >= lo)) { oob = 1; return 0; }
  if (x >= hi) { oob = 1; return res - 1; }
  const float t = (x - gmin) * inv_h, tf = floorf(t), near = 0x1p-22f * (fabsf(gmin) * inv_h + fabsf(t));
  int c = (int)tf;
  c = c < 0 ? 0 : (c > res - 1 ? res - 1 : c);
  if (t - tf <= near || t - tf >= 1.0f - near) {
    while (c > 0 && x < thr[c]) --c;
    while (c < res - 1 && x >= thr[c + 1]) ++c;
  }
  return c;
}

// Lowest stencil node along one axis of a particle at grid coordinate g: floor(g - 0.5) for the
// quadratic kernel, floor(g) - 1 for the cubic one. The floor is clamped to [-8, res + 8] before the
// conversion, so that a non-finite or far out-of-grid position (an unstable run) gives a stencil whose
// nodes all lie outside the grid instead of an integer overflow: every index formed from it as
// base + o (o <= 3) stays far inside the int range, and every node is then dropped as out of grid.
template <int ORDER>
__device__ __forceinline__ int stencil_base(float g, int res) {
  float b = ORDER == 2 ? floorf(g - 0.5f) : floorf(g) - 1.0f;
  b = fminf(fmaxf(b, -8.0f), (float)res + 8.0f);  // NaN gives -8
  return (int)b;
}

// A scene's thresholds and its grid's bounds among them. Formed at a kernel's start, where the compiler reads
// uniform data through the scalar cache; after a kernel's first stores it would read each bound as a vector and
// wait for it: six round trips one after another in every G2P wave (k_g2p 362 -> 328 us at 2^22 particles, 172 ->
// 157 for 16 scenes, 90 -> 86 at 2^20).
struct CellThr {
  const float* thr[3];
  float lo[3], hi[3];
};
__device__ __forceinline__ CellThr cell_thr(const float* thr, const int* res) {
  CellThr t;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    t.thr[d] = thr;
    t.lo[d] = thr[0];
    t.hi[d] = thr[res[d]];
    thr += res[d] + 1;
  }
  return t;
}
__device__ __forceinline__ uint32_t cell_key(const DevParams& P, const CellThr& t, float x0, float x1, float x2, int& oob,
                                             int (&c)[3]) {
  c[0] = axis_cell(t.thr[0], t.lo[0], t.hi[0], P.res[0], x0, P.gmin[0], P.inv_h[0], oob);
  c[1] = axis_cell(t.thr[1], t.lo[1], t.hi[1], P.res[1], x1, P.gmin[1], P.inv_h[1], oob);
  c[2] = axis_cell(t.thr[2], t.lo[2], t.hi[2], P.res[2], x2, P.gmin[2], P.inv_h[2], oob);
  return (uint32_t)(c[2] * P.res[0] * P.res[1] + c[1] * P.res[0] + c[0]);
}

// Tile (within the scene) of cell (c0, c1, c2).
__device__ __forceinline__ int tile_of(const DevParams& P, int c0, int c1, int c2) {
  return ((c2 >> 2) * P.tiles[1] + (c1 >> 2)) * P.tiles[0] + (c0 >> 2);
}

// Adds the wave's particles (active lanes with valid set) to the next sort's counts; `tile` is the key's tile
// over all scenes. Called with the wave's first lanes active. The lanes hold particles in the order of the cells
// they come from, and few change their cell in a substep, so runs of one key in consecutive lanes are taken
// together: a run's first lane adds its length with one atomic, all of them in the same instruction, and the
// wave does not wait for the round trip before the ticket is used. (Grouping all lanes of a key, not only
// consecutive ones, takes a loop over the keys: k_g2p 383 instead of 371 us at 2^22 particles. The scan blocks' totals are
// not counted here: one more atomic per wave, on words that few cells share, took k_g2p from 74 to 153 us at
// 2^20 particles.)
struct CountTicket {
  int base, head;
};
__device__ __forceinline__ CountTicket count_wave(const BinCounts& b, bool valid, uint32_t key, int tile) {
  const int lane = (int)lane_id();
  const uint32_t k = valid ? key : 0xFFFFFFFFu;  // no cell's key
  const uint32_t prev = (uint32_t)__shfl_up((int)k, 1);
  const uint64_t heads = __ballot(lane == 0 || k != prev), ends = heads | ~__ballot(true);
  const uint64_t upto = heads & (~0ull >> (63 - lane)), above = ends & ~(~0ull >> (63 - lane));
  CountTicket t{0, 63 - __clzll((long long)upto)};
  if (valid && t.head == lane) {
    t.base = atomicAdd(&b.cell_count[key], (above ? __ffsll((long long)above) - 1 : 64) - lane);
    b.tile_flag[tile] = 1;
    b.scan_flag[key / SCAN_TILE] = 1;
  }
  return t;
}
// The lane's number in its cell.
__device__ __forceinline__ uint32_t count_rank(const CountTicket& t) {
  return (uint32_t)(__shfl(t.base, t.head) + (int)lane_id() - t.head);
}

// ================================================================== keys of the caller order
// keys[id] = cell key of caller particle id (physical index pos[id]); the radix sort consumes the
// keys in caller order, so that equal keys keep caller order as in the reference.
__global__ __launch_bounds__(256) void k_keys(SceneTable T, const float* __restrict__ st, int64_t cap, int n,
                                              const float* __restrict__ thr, uint32_t* __restrict__ keys,
                                              int* __restrict__ status) {
  const PBlock b = particle_block(T);  // physical slots are scene-major like the caller ids
  const DevParams& P = T.params[b.s];
  const int j = b.j;
  int oob = 0;
  const CellThr t = cell_thr(thr + T.thr_off[b.s], P.res);
  int c[3];
  if (j < b.end)
    keys[j] = (uint32_t)T.node_off[b.s] +
              cell_key(P, t, st[PX * cap + j], st[(PX + 1) * cap + j], st[(PX + 2) * cap + j], oob, c);
  if (__ballot(oob) && lane_id() == 0) atomicOr(status, MPM_STATUS_OUT_OF_DOMAIN);
}

// Volume-weighted Kirchhoff stress of the current F (after the caller sets particles or parameters).
__global__ __launch_bounds__(256) void k_stress_init(SceneTable T, float* __restrict__ st, int64_t cap, int n,
                                                     unsigned long long* __restrict__ fallback) {
  const PBlock b = particle_block(T);
  const DevParams& P = T.params[b.s];
  const int i = b.j;
  if (i >= b.end) return;
  float F[9], K[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < 9; ++c) F[c] = st[(PF + c) * cap + i];
  int fb = 0;
  // cloth vertices and elements carry no particle stress (their F planes hold D for elements)
  const int pid = reinterpret_cast<const int*>(st + (size_t)PID * cap)[i];
  if (particle_kind(P, pid) == KIND_PARTICLE) kirchhoff_of_F(P, F, st[PPL * cap + i], st[PVOL * cap + i], K, fb);
#pragma unroll
  for (int e = 0; e < 6; ++e) st[(PK + e) * cap + i] = K[e];
  if (fb) atomicAdd(fallback, (unsigned long long)fb);
}

// ================================================================== radix sort (stable LSD, 8-bit digits)
// Per substep: one histogram launch for all three digit positions, then one launch per digit.
// A pass block ranks its 4096 keys stably with wave ballots (per-wave, per-digit running counts in
// LDS), publishes its per-digit counts and finds its global offsets by decoupled look-back over the
// preceding blocks (blocks take tickets in start order, so a block only waits on running blocks).
constexpr uint32_t FLAG_AGG = 1u << 30, FLAG_PREFIX = 2u << 30, VALUE_MASK = (1u << 30) - 1u;

__global__ __launch_bounds__(256) void k_reset(uint32_t* __restrict__ zero_words, int64_t n_zero, const Clock* clk) {
  if (clock_skip(clk)) return;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_zero; i += stride) zero_words[i] = 0u;
}

// Lanes of a wave that share a digit are grouped with 8 ballots; one lane per group adds the count.
__device__ __forceinline__ uint64_t digit_peers(bool valid, uint32_t d) {
  uint64_t peers = __ballot(valid);
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) {
    bool set = (d >> bit) & 1u;
    uint64_t bb = __ballot(valid && set);
    peers &= set ? bb : ~bb;
  }
  return peers;
}

__global__ __launch_bounds__(256) void k_sort_hist(const uint32_t* __restrict__ keys, int n, int passes,
                                                   uint32_t* __restrict__ hist, const Clock* clk) {
  if (clock_skip(clk)) return;
  __shared__ uint32_t h[4][256];
  for (int i = threadIdx.x; i < 1024; i += 256) (&h[0][0])[i] = 0u;
  __syncthreads();
  const int base = blockIdx.x * HIST_TILE;
  for (int k = 0; k < HIST_IPT; ++k) {
    const int i = base + k * 256 + threadIdx.x;
    const bool valid = i < n;
    const uint32_t key = valid ? keys[i] : 0u;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0ull) continue;
    const int first = __ffsll((long long)vmask) - 1;
    for (int p = 0; p < passes; ++p) {
      const uint32_t d = (key >> (8 * p)) & 255u;
      const uint32_t d0 = __shfl(d, first);
      if (__ballot(valid && d == d0) == vmask) {  // one digit across the wave: one add
        if ((int)lane_id() == first) atomicAdd(&h[p][d0], (uint32_t)__popcll(vmask));
      } else if (valid) {
        atomicAdd(&h[p][d], 1u);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 256 * passes; i += 256) {
    uint32_t c = (&h[0][0])[i];
    if (c) atomicAdd(&hist[i], c);
  }
}

constexpr int LOOKBACK = 8;  // predecessor status words read per look-back step

__global__ __launch_bounds__(256) void k_sort_pass(const uint32_t* __restrict__ kin, const int* __restrict__ vin,
                                                   uint32_t* __restrict__ kout, int* __restrict__ vout, int n, int pass,
                                                   const uint32_t* __restrict__ hist, uint32_t* __restrict__ tickets,
                                                   uint32_t* __restrict__ status, const Clock* clk) {
  if (clock_skip(clk)) return;
  __shared__ uint32_t s_k[SORT_TILE];
  __shared__ int s_v[SORT_TILE];
  __shared__ uint32_t s_wh[4][256];
  __shared__ uint32_t s_off[256];
  __shared__ uint32_t s_loc[256];
  __shared__ uint32_t s_scan[256];
  __shared__ int s_tile;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  if (tid == 0) s_tile = (int)atomicAdd(&tickets[pass], 1u);
  for (int i = tid; i < 1024; i += 256) (&s_wh[0][0])[i] = 0u;
  __syncthreads();
  const int b = s_tile;
  if (b >= (int)gridDim.x) return;  // tickets are zeroed per substep; uniform across the block
  const int base = b * SORT_TILE + w * (64 * SORT_IPT);
  const int shift = 8 * pass;
  uint32_t kr[SORT_IPT];
  int vr[SORT_IPT];
  uint32_t rr[SORT_IPT];
  const uint64_t lt = (1ull << lane) - 1ull;
  // stable rank of every key among the equal digits before it in the block (waves in order,
  // 64-key chunks in order, lanes in order)
#pragma unroll
  for (int i = 0; i < SORT_IPT; ++i) {
    int pos = base + i * 64 + lane;
    bool valid = pos < n;
    uint32_t k = valid ? kin[pos] : 0u;
    int v = valid ? (vin ? vin[pos] : pos) : 0;
    uint32_t d = (k >> shift) & 255u;
    const uint64_t peers = digit_peers(valid, d);
    uint32_t prev = s_wh[w][d];
    if (valid && (peers >> lane) == 1ull) s_wh[w][d] = prev + (uint32_t)__popcll(peers);
    kr[i] = k;
    vr[i] = v;
    rr[i] = prev + (uint32_t)__popcll(peers & lt);
  }
  __syncthreads();
  {
    const int d = tid;
    uint32_t t0 = s_wh[0][d], t1 = s_wh[1][d], t2 = s_wh[2][d], t3 = s_wh[3][d];
    s_wh[0][d] = 0u;
    s_wh[1][d] = t0;
    s_wh[2][d] = t0 + t1;
    s_wh[3][d] = t0 + t1 + t2;
    const uint32_t total = t0 + t1 + t2 + t3;
    uint32_t* my = status + (size_t)b * 256 + d;
    uint32_t excl = 0u;
    if (b == 0) {
      __hip_atomic_store(my, FLAG_PREFIX | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      __hip_atomic_store(my, FLAG_AGG | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // look back over the predecessors LOOKBACK at a time (independent loads), summing published
      // aggregates nearest first until an inclusive prefix is found; an unpublished entry is
      // polled again. Every block publishes its aggregate before it looks back, so the wait ends.
      int bb = b - 1;
      while (true) {
        uint32_t sv[LOOKBACK];
#pragma unroll
        for (int j = 0; j < LOOKBACK; ++j)
          sv[j] = bb - j >= 0 ? __hip_atomic_load(status + (size_t)(bb - j) * 256 + d, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : FLAG_PREFIX;
        int used = 0;
        bool found = false;
#pragma unroll
        for (int j = 0; j < LOOKBACK; ++j) {
          if (found || used < j) continue;           // stop at the first prefix or unpublished entry
          const uint32_t fl = sv[j] & ~VALUE_MASK;
          if (fl == 0u) continue;
          excl += sv[j] & VALUE_MASK;
          used = j + 1;
          if (fl == FLAG_PREFIX) found = true;
        }
        if (found) break;
        bb -= used;
      }
      __hip_atomic_store(my, FLAG_PREFIX | (excl + total), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // exclusive scans over the digits: global histogram of this pass, and this block's totals
    const uint32_t gh = hist[pass * 256 + d];
    s_scan[d] = gh;
    s_loc[d] = total;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      uint32_t a1 = d >= off ? s_scan[d - off] : 0u;
      uint32_t a2 = d >= off ? s_loc[d - off] : 0u;
      __syncthreads();
      s_scan[d] += a1;
      s_loc[d] += a2;
      __syncthreads();
    }
    const uint32_t loc = s_loc[d] - total;
    __syncthreads();
    s_loc[d] = loc;
    s_off[d] = (s_scan[d] - gh) + excl - loc;  // global destination = s_off[d] + block-local position
  }
  __syncthreads();
  // place the block's keys in LDS in output order, then write contiguous runs
#pragma unroll
  for (int i = 0; i < SORT_IPT; ++i) {
    int pos = base + i * 64 + lane;
    if (pos < n) {
      uint32_t d = (kr[i] >> shift) & 255u;
      uint32_t lp = s_loc[d] + s_wh[w][d] + rr[i];
      if (lp < (uint32_t)SORT_TILE) {
        s_k[lp] = kr[i];
        s_v[lp] = vr[i];
      }
    }
  }
  __syncthreads();
  const int cnt = min(SORT_TILE, n - b * SORT_TILE);
#pragma unroll
  for (int i = 0; i < SORT_IPT; ++i) {
    const int t = i * 256 + tid;
    if (t < cnt) {
      const uint32_t k = s_k[t];
      const uint32_t dst = s_off[(k >> shift) & 255u] + (uint32_t)t;
      if (dst < (uint32_t)n) {  // always true for a consistent histogram; keeps a bad one in bounds
        kout[dst] = k;
        vout[dst] = s_v[t];
      }
    }
  }
}

// ------------------------------------------------------------------ one-digit counting sort
// The cell key itself is the single digit: the particles of every cell are counted where they are moved
// (count_wave: atomic ranks, in no particular order), the counts are scanned into cell offsets, the caller
// ids are scattered into their cells, and each cell is ordered by caller id (the rank of id i in its cell is
// the number of smaller ids there). The result equals the LSD passes' stable sort bit for bit. The count and
// the scatter run over physical slots, where the previous sort left the particles in cell order: lanes of a
// wave share few distinct keys, and the scatter's writes land close to where they are read; the scatter puts
// each id's slot and key beside it, so that the rank pass loads a position's id, slot and key together (gathering
// the key through the slot, the sort took 83 us instead of 78 at 2^22 particles, 56 instead of 52 for 16 scenes).
__global__ __launch_bounds__(256) void k_clear_counts(BinCounts b, int64_t nscan, int64_t ntiles, int64_t ncells,
                                                      int* __restrict__ counters) {
  const int64_t stride = (int64_t)gridDim.x * 256, t0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t q = t0; q < nscan; q += stride) b.scan_flag[q] = 0;
  for (int64_t q = t0; q < ntiles; q += stride) b.tile_flag[q] = 0;
  for (int64_t q = t0; q < ncells; q += stride) b.cell_count[q] = 0;
  if (t0 < 2) counters[t0] = 0;
}

// The counts of particles by their keys (those that no G2P has counted).
__global__ __launch_bounds__(256) void k_cell_count(SceneTable T, BinCounts b, const uint32_t* __restrict__ keys, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const bool valid = i < n;
  const uint32_t key = valid ? keys[i] : 0u;
  const int sc = scene_of(T.node_off, T.nscenes, (int64_t)key);
  const DevParams& P = T.params[sc];
  const uint32_t lk = key - (uint32_t)T.node_off[sc];
  const int r01 = P.res[0] * P.res[1];
  const int c2 = (int)(lk / (uint32_t)r01), rem = (int)(lk % (uint32_t)r01);
  const int c1 = rem / P.res[0], c0 = rem % P.res[0];
  const CountTicket t = count_wave(b, valid, key, T.tile_off[sc] + tile_of(P, c0, c1, c2));
  const uint32_t r = count_rank(t);
  if (valid) b.rank[i] = r;
}

// The tiles that hold particles: their flags, then the number of flags, which are cleared (new particles or a new
// grid; a substep's tiles are counted by claim_block).
__global__ __launch_bounds__(256) void k_flag_tiles(SceneTable T, const float* __restrict__ st, int64_t cap,
                                                    const float* __restrict__ thr, uint8_t* __restrict__ flag) {
  const PBlock b = particle_block(T);
  if (b.j >= b.end) return;
  const DevParams& P = T.params[b.s];
  const CellThr t = cell_thr(thr + T.thr_off[b.s], P.res);
  int oob = 0, c[3];
  (void)cell_key(P, t, st[PX * cap + b.j], st[(PX + 1) * cap + b.j], st[(PX + 2) * cap + b.j], oob, c);
  flag[T.tile_off[b.s] + tile_of(P, c[0], c[1], c[2])] = 1;
}
__global__ __launch_bounds__(256) void k_sum_flags(uint8_t* __restrict__ flag, int64_t ntiles, int* __restrict__ count) {
  int sum = 0;
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < ntiles; q += (int64_t)gridDim.x * 256) {
    sum += flag[q];
    flag[q] = 0;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if (lane_id() == 0 && sum) atomicAdd(count, sum);
}

// Total of a scan block's SCAN_TILE cell counts (the blocks are independent).
__device__ __forceinline__ void sum_block(const SortBufs& a, int b) {
  __shared__ uint32_t s_wsum[4];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  if (tid == 0) a.scan_flag_clear[b] = 0;
  if (!a.bins.scan_flag[b]) {  // no particle in the block's cells: nothing to read
    if (tid == 0) a.scan_sum[b] = 0u;
    return;
  }
  const int* cnt = a.bins.cell_count;
  const int64_t base = (int64_t)b * SCAN_TILE + (int64_t)tid * SCAN_IPT;
  uint32_t t = 0;
  if (base + SCAN_IPT <= a.ncells) {
    const int4* p4 = reinterpret_cast<const int4*>(cnt + base);
#pragma unroll
    for (int q = 0; q < SCAN_IPT / 4; ++q) {
      const int4 v = p4[q];
      t += (uint32_t)v.x + (uint32_t)v.y + (uint32_t)v.z + (uint32_t)v.w;
    }
  } else {
    for (int q = 0; q < SCAN_IPT; ++q)
      if (base + q < a.ncells) t += (uint32_t)cnt[base + q];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off);
  if (lane == 0) s_wsum[w] = t;
  __syncthreads();
  if (tid == 0) a.scan_sum[b] = s_wsum[0] + s_wsum[1] + s_wsum[2] + s_wsum[3];
}

// Thread per tile t (tiles and node blocks share one index space). A flagged tile receives the
// next slot of the active tile list. Node block t is active when any of its 27 neighbour tiles is
// (the 7x7x7-node P2G footprint of those tiles covers it) and receives the next slot of the active
// block list. A workgroup takes one atomic per list. Slot numbers depend on the order in which waves
// run; no result depends on them. The other buffer's flags are cleared.
__device__ __forceinline__ void claim_block(const SortBufs& a, int b) {
  __shared__ int s_cnt[2][4];
  __shared__ int s_base[2];
  const int64_t t = (int64_t)b * 256 + threadIdx.x;
  bool tile_on = false, block_on = false;
  if (t < a.ntiles) {
    // the scene: uniform where the workgroup's tiles are one scene's
    const int t_first = b * 256, t_last = (int)min((int64_t)t_first + 255, a.ntiles - 1);
    const auto tile_off = as_const(a.T.tile_off);
    const int sf = scene_of(tile_off, a.T.nscenes, t_first);
    int off = tile_off[sf], tl[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) tl[d] = as_const(a.T.params)[sf].tiles[d];
    if (sf + 1 < a.T.nscenes && t_last >= tile_off[sf + 1]) {
      const int sc = scene_of(a.T.tile_off, a.T.nscenes, (int)t);
      off = a.T.tile_off[sc];
#pragma unroll
      for (int d = 0; d < 3; ++d) tl[d] = a.T.params[sc].tiles[d];
    }
    const int lt = (int)t - off;
    const int t0 = lt % tl[0], t1 = (lt / tl[0]) % tl[1], t2 = lt / (tl[0] * tl[1]);
    uint8_t v[27];
#pragma unroll
    for (int q = 0; q < 27; ++q) {  // all 27 loads issued together
      const int b0 = t0 + q % 3 - 1, b1 = t1 + (q / 3) % 3 - 1, b2 = t2 + q / 9 - 1;
      const bool in = b0 >= 0 && b1 >= 0 && b2 >= 0 && b0 < tl[0] && b1 < tl[1] && b2 < tl[2];
      v[q] = in ? a.bins.tile_flag[off + (b2 * tl[1] + b1) * tl[0] + b0] : 0;
    }
    tile_on = v[13] != 0;
#pragma unroll
    for (int q = 0; q < 27; ++q) block_on |= v[q] != 0;
  }
  const uint64_t mt = __ballot(tile_on), mb = __ballot(block_on);
  const int lane = (int)lane_id(), w = (int)threadIdx.x >> 6;
  if (lane == 0) {
    s_cnt[0][w] = __popcll(mt);
    s_cnt[1][w] = __popcll(mb);
  }
  __syncthreads();
  // one atomic per list and workgroup (a single counter takes many device-scope atomics slowly across XCDs)
  if (threadIdx.x < 2) {
    const int k = (int)threadIdx.x;
    const int total = s_cnt[k][0] + s_cnt[k][1] + s_cnt[k][2] + s_cnt[k][3];
    s_base[k] = total ? atomicAdd(&a.counters[k == 0 ? CNT_TILES : CNT_BLOCKS], total) : 0;
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
  int slot_t = -1, slot_b = -1;
  if (tile_on) {
    int base = s_base[0];
    for (int k = 0; k < w; ++k) base += s_cnt[0][k];
    slot_t = base + __popcll(mt & below);
    a.active_tiles[slot_t] = (int)t;
  }
  if (block_on) {
    int base = s_base[1];
    for (int k = 0; k < w; ++k) base += s_cnt[1][k];
    slot_b = base + __popcll(mb & below);
    a.active_blocks[slot_b] = (int)t;
  }
  if (t < a.ntiles) {
    a.tile_slot[t] = slot_t;
    a.block_slot[t] = slot_b;
    a.tile_flag_clear[t] = 0;
  }
}

// Exclusive scan of the cell counts into cell_start[0 .. ncells]: block b starts at the sum of the
// totals of the blocks before it (read and summed by the block itself) and scans its SCAN_TILE cells;
// the blocks are independent. A block without particles writes nothing: its cells are empty, which every reader learns from scan_flag (the getter of the bins fills them, k_fill_bins). A
// block with particles also writes the start of the next block's first cell (its own end), which
// the next block, if it has particles, writes with the same value. The last block writes
// cell_start[ncells].
// With few scan blocks (SMALL) a block adds up the cells of the occupied blocks before it, instead of reading
// their totals.
template <bool SMALL>
__device__ __forceinline__ void scan_block(const SortBufs& a, int b) {
  const int* cnt = a.bins.cell_count;
  const int64_t ncells = a.ncells;
  int* cell_start = a.cell_start;
  __shared__ uint32_t s_wsum[4];
  __shared__ uint32_t s_boff[4];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const bool last = (int64_t)(b + 1) * SCAN_TILE >= ncells;
  if (SMALL && tid == 0) a.scan_flag_clear[b] = 0;
  if (!a.bins.scan_flag[b] && !last) return;
  {
    uint32_t p = 0;
    if constexpr (SMALL) {
      // every fourth of them a wave, with all of a block's loads in flight (every block before b is whole)
      uint64_t todo = __ballot(lane < b && a.bins.scan_flag[lane < b ? lane : 0]);
      for (int r = 0; todo; ++r, todo &= todo - 1) {
        if ((r & 3) != w) continue;
        const int4* p4 = reinterpret_cast<const int4*>(cnt + (int64_t)(__ffsll((long long)todo) - 1) * SCAN_TILE);
#pragma unroll
        for (int q = 0; q < SCAN_TILE / 256; ++q) {
          const int4 v = p4[64 * q + lane];
          p += (uint32_t)v.x + (uint32_t)v.y + (uint32_t)v.z + (uint32_t)v.w;
        }
      }
    } else {
      for (int q = tid; q < b; q += 256) p += a.scan_sum[q];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
    if (lane == 0) s_boff[w] = p;
  }
  const int64_t base = (int64_t)b * SCAN_TILE + (int64_t)tid * SCAN_IPT;
  int c[SCAN_IPT];
  if (base + SCAN_IPT <= ncells) {
    const int4* p4 = reinterpret_cast<const int4*>(cnt + base);
#pragma unroll
    for (int q = 0; q < SCAN_IPT / 4; ++q) {
      const int4 v = p4[q];
      c[4 * q] = v.x; c[4 * q + 1] = v.y; c[4 * q + 2] = v.z; c[4 * q + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int q = 0; q < SCAN_IPT; ++q) c[q] = base + q < ncells ? cnt[base + q] : 0;
  }
  uint32_t tsum = 0;
#pragma unroll
  for (int q = 0; q < SCAN_IPT; ++q) tsum += (uint32_t)c[q];
  uint32_t x = tsum;  // inclusive scan over the wave's threads
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_wsum[w] = x;
  __syncthreads();
  const uint32_t boff = s_boff[0] + s_boff[1] + s_boff[2] + s_boff[3];
  uint32_t wpre = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) wpre += k < w ? s_wsum[k] : 0u;
  uint32_t run = boff + wpre + (x - tsum);
  if (base + SCAN_IPT <= ncells) {
    int4* ps = reinterpret_cast<int4*>(cell_start + base);
#pragma unroll
    for (int q = 0; q < SCAN_IPT / 4; ++q) {
      int4 vs;
      vs.x = (int)run; run += (uint32_t)c[4 * q];
      vs.y = (int)run; run += (uint32_t)c[4 * q + 1];
      vs.z = (int)run; run += (uint32_t)c[4 * q + 2];
      vs.w = (int)run; run += (uint32_t)c[4 * q + 3];
      ps[q] = vs;
    }
  } else {
#pragma unroll
    for (int q = 0; q < SCAN_IPT; ++q) {
      if (base + q < ncells) {
        cell_start[base + q] = (int)run;
        run += (uint32_t)c[q];
      }
    }
  }
  if (base < ncells && base + SCAN_IPT >= ncells) cell_start[ncells] = (int)run;  // the total
  if (tid == 255 && !last) cell_start[(int64_t)(b + 1) * SCAN_TILE] = (int)run;  // the next block's first cell
}

// The scan blocks' totals (workgroups below nscan) and the tile lists (the others): independent of each other,
// so one launch hides one's latency behind the other's. With the counts made by G2P a substep sorts in four
// launches (this one, scan, scatter, rank) where a separate count, totals and claim took six: sort 117 -> 83 us and
// G2P 356 -> 328 at 2^22 particles (of which 55 us less by the cell_key changes), sort 30 -> 22 us at 2^15.
// Up to SMALL_SCAN scan blocks (a 64^3 grid's), the scan itself takes the totals' place and the sort has three launches:
// 30 substeps of 2^15 particles on 64^3 1.50 -> 1.46 ms, 20 of a tiny scene on 24^3 1.59 -> 1.54.
constexpr int SMALL_SCAN = 64;
template <bool SMALL>
__global__ __launch_bounds__(256) void k_sums_claim(SortBufs a, int nscan) {
  if (clock_skip(a.clk)) return;
  const int b = (int)blockIdx.x;
  if (b < nscan) {
    if (b == 0 && threadIdx.x < 2) a.counters_clear[threadIdx.x] = 0;
    if (b == 0 && threadIdx.x == 2) *a.cand_count = 0;
    if constexpr (SMALL) scan_block<true>(a, b);
    else sum_block(a, b);
  } else {
    claim_block(a, b - nscan);
  }
}

__global__ __launch_bounds__(256) void k_cell_scan(SortBufs a) {
  if (clock_skip(a.clk)) return;
  scan_block<false>(a, (int)blockIdx.x);
}

// The bins of the last sort for the host: cell_start[c] = the first sorted position whose key is at
// least c (a binary search of the sorted keys), for every cell c in [0, ncells]. The sort's own scan
// writes only the scan blocks that hold particles, which is all the substep reads; the keys, unlike
// the block flags, belong to the last sort that ran, also when the device clock skipped a later
// captured substep.
__global__ __launch_bounds__(256) void k_fill_bins(const uint32_t* __restrict__ ks, int n, int64_t ncells,
                                                   int* __restrict__ cell_start) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c > ncells) return;
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = lo + ((hi - lo) >> 1);
    if ((int64_t)ks[mid] < c) lo = mid + 1;
    else hi = mid;
  }
  cell_start[c] = lo;
}

// The caller id -> physical slot map from the state's id plane and, when kc is given, the keys by
// caller id from the keys by physical slot (the input of the radix passes).
__global__ __launch_bounds__(256) void k_caller_keys(const uint32_t* __restrict__ keys, const int* __restrict__ pid, int n,
                                                     uint32_t* __restrict__ kc, int* __restrict__ pos, const Clock* clk) {
  if (clock_skip(clk)) return;
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  const int i = pid[j];
  if ((unsigned)i < (unsigned)n) {  // always true for a consistent id plane
    if (kc) kc[i] = keys[j];
    pos[i] = j;
  }
}

__global__ __launch_bounds__(256) void k_cell_scatter(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ rank,
                                                      int n, const int* __restrict__ cell_start,
                                                      const int* __restrict__ pid, int* __restrict__ tmp,
                                                      int* __restrict__ tslot, uint32_t* __restrict__ ks,
                                                      const Clock* clk) {
  if (clock_skip(clk)) return;
  const int j = blockIdx.x * 256 + threadIdx.x;  // physical slot
  if (j >= n) return;
  const uint32_t k = keys[j];
  const int id = pid[j], p = cell_start[k] + (int)rank[j];
  if ((unsigned)p < (unsigned)n) {  // always true for consistent counts
    tmp[p] = id;
    tslot[p] = j;
    ks[p] = k;  // final: every position of a cell holds its key
  }
}

// Thread per sorted position: the caller id placed there by the scatter moves to its stable rank
// within the cell (a cell of c particles costs c comparisons per particle). It also does the bin
// pass's work (k_bounds) for its new position: src = the particle's physical slot, and the cell's
// first particle clears the cell's count.
// The workgroup first copies the ids of its 256 positions and RANK_HALO on either side into LDS (one
// coalesced round trip): a cell of at most RANK_HALO particles around any of its positions lies in
// that window, and its ids are compared there; a larger cell reads them from global memory.
constexpr int RANK_HALO = 64;
__global__ __launch_bounds__(256) void k_cell_rank(const uint32_t* __restrict__ ks, const int* __restrict__ tmp,
                                                   const int* __restrict__ tslot, int n,
                                                   const int* __restrict__ cell_start,
                                                   int* __restrict__ vs, int* __restrict__ cnt, int* __restrict__ src,
                                                   const Clock* clk) {
  if (clock_skip(clk)) return;
  constexpr int WIN = 256 + 2 * RANK_HALO;
  __shared__ int s_ids[WIN];
  const int wlo = (int)blockIdx.x * 256 - RANK_HALO;  // the window holds positions wlo .. wlo + WIN - 1
  const int j = blockIdx.x * 256 + threadIdx.x;
  // the position's slot and key are loaded with the window
  const int jc = min(j, n - 1);
  const int pi = tslot[jc];
  const uint32_t k = ks[jc];
  for (int q = (int)threadIdx.x; q < WIN; q += 256) {
    const int p = wlo + q;
    s_ids[q] = (p >= 0 && p < n) ? tmp[p] : 0;
  }
  const int s0 = cell_start[k], e0 = min(cell_start[k + 1], n);
  __syncthreads();
  if (j >= n) return;
  const int i = clamp_index(s_ids[j - wlo], n);
  int r = 0;
  if (s0 >= wlo && e0 <= wlo + WIN) {
    for (int m = s0 - wlo; m < e0 - wlo; ++m) r += s_ids[m] < i ? 1 : 0;
  } else {
    // 8 ids per step, loaded together (past the cell's end the loads read its last entry, in
    // bounds, and are not counted)
    for (int m0 = s0; m0 < e0; m0 += 8) {
      int t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = tmp[min(m0 + u, e0 - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) r += (m0 + u < e0 && t[u] < i) ? 1 : 0;
    }
  }
  const int d = s0 + r;
  if ((unsigned)d >= (unsigned)n) return;  // never, for consistent counts
  vs[d] = i;
  src[d] = clamp_index(pi, n);
  if (r == 0) cnt[k] = 0;
}

// ================================================================== bins
// Thread per sorted position (the digit passes only): src = the particle's physical slot; the first position of
// each run of equal keys clears the cell's count for the next substep.
__global__ __launch_bounds__(256) void k_bounds(SceneTable T, const uint32_t* __restrict__ ks, int n,
                                                int* __restrict__ cnt, const int* __restrict__ perm,
                                                const int* __restrict__ pos, int* __restrict__ src, const Clock* clk) {
  if (clock_skip(clk)) return;
  const PBlock b = particle_block(T);  // sorted positions are scene-major as well
  const int j = b.j;
  if (j >= b.end) return;
  src[j] = clamp_index(pos[clamp_index(perm[j], n)], n);
  const uint32_t k = ks[j];
  if (j == 0 || ks[j - 1] != k) cnt[k] = 0;
}

// ================================================================== P2G
// One workgroup (8 waves) per active 4x4x4-cell tile; wave w owns the cell layer z = w & 3 and walks
// rows (y) 2 (w >> 2) and 2 (w >> 2) + 1 one after another, with no workgroup barrier until the
// tile is done. (Two row halves per layer halve a tile's latency, which evens out the last round
// when the active tiles do not divide evenly over the resident workgroups.)
//
// Row pass. The four cells of a row (x = 0..3) are contiguous in the sorted order. In chunk k,
// lane (cx, r), r < RANKS, stages the particle of rank RANKS k + r of cell cx: it loads the
// particle (one chunk ahead) and writes a 48-float payload (B-spline weights of the window's 4 nodes
// per axis, mass, affine momentum terms, stress impulse, and the x-column terms every lane of the
// cell needs) into the wave's LDS slots. Then lane (cx, zo, oy) adds the chunk's particles of cell
// cx, in ascending rank, to its 4 register sums: nodes (cx-1+ox, cy-1+oy, z-1+zo), ox = 0..3, of the
// cell's 4x4x4 node window c-1 .. c+2 (a superset of the quadratic stencil and exactly the cubic
// one). At the end of the row the sums are added into the wave's own LDS node slab (7 x 7 x 4 nodes)
// in four phases ox = 0..3; within a phase every lane has a different node, so the slab receives
// the row sums in a fixed order.
//
// When all waves are done, node (X, Y, Z) of the tile's 7x7x7 footprint is the sum of the slabs of
// the waves of layers l with 0 <= Z - l <= 3, in ascending l and row half, and is stored as the
// tile's partial. k_grid sums the covering tiles' partials in ascending tile order: every node value
// is a sum in a fixed order, without float atomics on global memory, and reruns are bitwise identical.
constexpr int PAY = 48;                 // payload floats per staged particle (12 x float4)
// LDS floats between consecutive ranks' payloads: 52 = 20 (mod 32), so the 128-bit payload writes of
// the eight staging lanes of a cell fall on distinct groups of the 32 banks (48 would give 4-way
// bank conflicts).
constexpr int PAY_STRIDE = 52;
// RANKS (2, 4 or 8, chosen by the autotuner) = ranks per cell staged per chunk; one cell's staged
// payloads take RANKS * PAY_STRIDE + 4 floats (the 4 shift the cells of a row onto different banks).
// The chunk size does not change the order in which a lane adds its cell's particles, so results do
// not depend on it.
template <int RANKS>
constexpr int pay_cell() { return RANKS * PAY_STRIDE + 4; }
constexpr int SLAB = FOOT * FOOT * 4;   // nodes of a wave's slab
constexpr int P2G_SLABS = 8;            // slabs of a tile: 4 cell layers x 2 row halves
// payload layout (floats): the x weights of window nodes c-1 .. c+2, the y and z weights and
// derivatives (per cell width), the x-column terms g[ox][r] = ox wx[ox] Q[r][0] - dwx[ox] S[r][0]
// that every lane of the cell adds with weight wy wz, the mass, q0 (a cloth vertex's force in the
// force pass), and the y and z columns of Q and of the scaled stress matrix S.
constexpr int PY_WX = 0, PY_WY = 4, PY_DWY = 8, PY_WZ = 12, PY_DWZ = 16, PY_G = 20;
constexpr int PY_M = 32, PY_Q0 = 33, PY_Q12 = 36, PY_S12 = 42;

// Weights and derivatives (per cell width) of the window nodes c-1 .. c+2 of a particle at fraction
// f of cell c. Quadratic: the three nodes from base = floor(c + f - 0.5) (c - 1 for f < 0.5, else c),
// fx = c + f - base in [0.5, 1.5): N = 0.5 (1.5 - fx)^2, 0.75 - (fx - 1)^2, 0.5 (fx - 0.5)^2, in
// closed form and without branches (HybridSolver.cpp:18-97, interpolation.cpp:9-33).
template <int ORDER>
__device__ __forceinline__ void window_weights(float f, float* w, float* dw) {
  if constexpr (ORDER == 2) {
    const bool hi = f >= 0.5f;
    const float fx = hi ? f : f + 1.0f;
    const float a = 1.5f - fx, b = fx - 1.0f, c = fx - 0.5f;
    const float w0 = 0.5f * a * a, w1 = 0.75f - b * b, w2 = 0.5f * c * c;
    const float d0 = -a, d1 = -2.0f * b, d2 = c;
    w[0] = hi ? 0.0f : w0;
    w[1] = hi ? w0 : w1;
    w[2] = hi ? w1 : w2;
    w[3] = hi ? w2 : 0.0f;
    dw[0] = hi ? 0.0f : d0;
    dw[1] = hi ? d0 : d1;
    dw[2] = hi ? d1 : d2;
    dw[3] = hi ? d2 : 0.0f;
  } else {
#pragma unroll
    for (int o = 0; o < 4; ++o) spline<ORDER>(f + 1.0f - (float)o, w[o], dw[o]);
  }
}

// Scene constants of the tile being transferred, held in registers for the whole tile.
struct P2GScene {
  float gmin[3], inv_h[3], h[3], dinv;
  int res[3];
  int mesh_v0, mesh_e0, mesh_e1;
};


template <class PP>
__device__ __forceinline__ P2GScene p2g_scene(PP& P) {
  P2GScene S;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    S.gmin[d] = uniform_f(P.gmin[d]);
    S.inv_h[d] = uniform_f(P.inv_h[d]);
    S.h[d] = uniform_f(P.h[d]);
    S.res[d] = __builtin_amdgcn_readfirstlane(P.res[d]);
  }
  S.dinv = uniform_f(P.dinv);
  S.mesh_v0 = __builtin_amdgcn_readfirstlane(P.mesh_v0);
  S.mesh_e0 = __builtin_amdgcn_readfirstlane(P.mesh_e0);
  S.mesh_e1 = __builtin_amdgcn_readfirstlane(P.mesh_e1);
  return S;
}

// Particle data a staging lane needs, loaded one chunk ahead of its use (the loads of the next
// chunk are in flight while the wave accumulates the current one). In the force pass of the
// predicted-stress mode B holds the stress matrix that k_stress_predicted left at the sorted position.
struct StageIn {
  int pid;  // the particle's id when the scene has a cloth mesh (else that of slot 0)
  float x[3], m, v[3], B[9], K[6];
};

// The physical slot of sorted position idx, loaded a chunk before the particle's own data so that
// the two dependent loads do not stall the wave back to back; it is clamped where it is used.
__device__ __forceinline__ int p2g_slot(const P2GArgs& a, int idx) { return a.src[idx]; }

template <int MODE>
__device__ __forceinline__ void p2g_load_at(const P2GArgs& a, const P2GScene& S, int slot, int idx, StageIn& in) {
  const uint32_t pi = (uint32_t)clamp_index(slot, a.n);
  const float* st = a.state;
  const int64_t cap = a.cap;
  // a scene without a mesh loads word 0 of the id plane in every lane (one cache line) instead of a
  // branch around the load: a branch here makes the wave wait for this chunk's loads before the
  // accumulation of the previous one
  in.pid = __float_as_int(plane_load(st + PID * cap, S.mesh_e1 > S.mesh_v0 ? pi : 0u));
#pragma unroll
  for (int d = 0; d < 3; ++d) in.x[d] = plane_load(st + (PX + d) * cap, pi);
  if constexpr (MODE != P2G_FORCE) {
    in.m = plane_load(st + PM * cap, pi);
#pragma unroll
    for (int d = 0; d < 3; ++d) in.v[d] = plane_load(st + (PV + d) * cap, pi);
#pragma unroll
    for (int i = 0; i < 9; ++i) in.B[i] = plane_load(st + (PB + i) * cap, pi);
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) in.B[i] = plane_load(a.stress + i * cap, (uint32_t)idx);
  }
  if constexpr (MODE == P2G_MOM_STRESS) {
#pragma unroll
    for (int i = 0; i < 6; ++i) in.K[i] = plane_load(st + (PK + i) * cap, pi);
  }
}

template <int MODE>
__device__ __forceinline__ void p2g_load(const P2GArgs& a, const P2GScene& S, int idx, StageIn& in) {
  p2g_load_at<MODE>(a, S, p2g_slot(a, idx), idx, in);
}

template <int ORDER, int MODE>
__device__ __forceinline__ void p2g_stage(const P2GArgs& a, const P2GScene& S, float dt, const StageIn& in, int g0, int g1,
                                          int g2, float4* dst) {
  // No FMA contraction: the row and the layer pass inline this function into different kernels, and
  // the payload must have the same bits in both (contraction is decided per kernel otherwise).
#pragma clang fp contract(off)
  float pay[PAY];
#pragma unroll
  for (int i = 0; i < PAY; ++i) pay[i] = 0.0f;
  // kind of the point from its id (loaded with the rest of its data, used only here)
  const int kind = (S.mesh_e1 <= S.mesh_v0 || in.pid < S.mesh_v0) ? KIND_PARTICLE
                                                                    : (in.pid < S.mesh_e0 ? KIND_VERTEX : KIND_ELEMENT);
  const int mid = in.pid - (kind == KIND_VERTEX ? S.mesh_v0 : S.mesh_e0);
  const int cc[3] = {g0, g1, g2};
  float f[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) f[d] = (in.x[d] - S.gmin[d]) * S.inv_h[d] - (float)cc[d];
  float wx[4], dwx[4], wy[4], dwy[4], wz[4], dwz[4];
  window_weights<ORDER>(f[0], wx, dwx);
  window_weights<ORDER>(f[1], wy, dwy);
  window_weights<ORDER>(f[2], wz, dwz);
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    pay[PY_WX + o] = wx[o];
    pay[PY_WY + o] = wy[o];
    pay[PY_DWY + o] = dwy[o];
    pay[PY_WZ + o] = wz[o];
    pay[PY_DWZ + o] = dwz[o];
  }
  // the weights leave their registers before the rest is formed (the layer pass holds 64 sums meanwhile)
#pragma unroll
  for (int i = 0; i < PY_G / 4; ++i) dst[i] = make_float4(pay[4 * i], pay[4 * i + 1], pay[4 * i + 2], pay[4 * i + 3]);
  __builtin_amdgcn_sched_barrier(0);
  float Q0[3] = {0.0f, 0.0f, 0.0f}, S0[3] = {0.0f, 0.0f, 0.0f};  // x columns of Q and of S
  if constexpr (MODE != P2G_FORCE) {
    // momentum w*(q0 + Q o): Q = m D^-1 B diag(h), q0 = m v - Q (1 + f)  (HybridSolver.cpp:134,169-170)
    const float mp = in.m;
    float Q[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) Q[3 * r + c] = mp * S.dinv * in.B[3 * r + c] * S.h[c];
    pay[PY_M] = mp;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      float q0 = mp * in.v[r] - (Q[3 * r] * (1.0f + f[0]) + Q[3 * r + 1] * (1.0f + f[1]) + Q[3 * r + 2] * (1.0f + f[2]));
      if (MODE == P2G_MOM_STRESS && kind == KIND_VERTEX) q0 += dt * a.vert_force[3 * mid + r];  // in-plane impulse (:378)
      pay[PY_Q0 + r] = q0;
      Q0[r] = Q[3 * r];
      pay[PY_Q12 + 2 * r] = Q[3 * r + 1];
      pay[PY_Q12 + 2 * r + 1] = Q[3 * r + 2];
    }
  }
  float Sm[9];  // stress matrix, columns scaled by 1/h (and by dt when folded into the momentum)
#pragma unroll
  for (int i = 0; i < 9; ++i) Sm[i] = 0.0f;
  if constexpr (MODE == P2G_MOM_STRESS) {
    // stress at F^n: the Kirchhoff stress V P(F) F^T written by the previous G2P (or by k_stress_init)
    const int R[9] = {0, 3, 4, 3, 1, 5, 4, 5, 2};  // symmetric 3x3 from (xx yy zz xy xz yz)
    if (kind == KIND_PARTICLE) {
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) Sm[3 * r + c] = dt * in.K[R[3 * r + c]] * S.inv_h[c];
    } else if (kind == KIND_ELEMENT) {  // element stress of the normal/shear response (:434-454)
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) Sm[3 * r + c] = dt * a.elem_stress[9 * mid + 3 * r + c] * S.inv_h[c];
    }
  }
  if constexpr (MODE == P2G_FORCE) {
    if (kind == KIND_VERTEX) {
#pragma unroll
      for (int r = 0; r < 3; ++r) pay[PY_Q0 + r] = a.vert_force[3 * mid + r];
    } else if (kind == KIND_ELEMENT) {
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) Sm[3 * r + c] = a.elem_stress[9 * mid + 3 * r + c] * S.inv_h[c];
    } else {
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) Sm[3 * r + c] = in.B[3 * r + c] * S.inv_h[c];
    }
  }
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    S0[r] = Sm[3 * r];
    pay[PY_S12 + 2 * r] = Sm[3 * r + 1];
    pay[PY_S12 + 2 * r + 1] = Sm[3 * r + 2];
  }
#pragma unroll
  for (int ox = 0; ox < 4; ++ox)
#pragma unroll
    for (int r = 0; r < 3; ++r) pay[PY_G + 3 * ox + r] = (float)ox * wx[ox] * Q0[r] - dwx[ox] * S0[r];
#pragma unroll
  for (int i = PY_G / 4; i < PAY / 4; ++i) dst[i] = make_float4(pay[4 * i], pay[4 * i + 1], pay[4 * i + 2], pay[4 * i + 3]);
}

// Stress matrix V P(F^) F^n^T of every particle at the predicted F^ = F + dt (sum_i v_i grad w_ip^T) F from
// the post-P2G grid velocity (HybridSolver.cpp:269-339), thread per sorted position j, written to
// stress[9 planes][j] for the force pass of P2G. As G2P, the gather factors over the axes (row sums of v
// with w and w' along x) and loads one z plane of nodes at a time.
// The force pass used to do this inside its staging, where only the staging lanes of a wave (a quarter to a
// half) gathered, node after node, and nothing overlapped the wait: 203 us for the force pass of 321k cubic
// particles, now 33 us for this kernel and 35 us for the force pass (MI355X).
template <int ORDER>
__global__ __launch_bounds__(256) void k_stress_predicted(P2GArgs a) {
  if (clock_skip(a.clk)) return;
  const float dt = clock_dt(a.clk, a.dt);
  const PBlock pb = particle_block(a.T);
  const DevParams P = uniform_params(a.T.params[pb.s]);
  const float4* gvel = a.gvel + 2 * a.T.node_off[pb.s];
  const int j = pb.j;
  int fb = 0;
  if (j < pb.end) {
    const float* st = a.state;
    const int64_t cap = a.cap;
    const int pi = clamp_index(a.src[j], a.n);
    const int pid = reinterpret_cast<const int*>(st + (size_t)PID * cap)[P.mesh_e1 > P.mesh_v0 ? pi : 0];
    float Fn[9], g[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) g[d] = (st[(PX + d) * cap + pi] - P.gmin[d]) * P.inv_h[d];
#pragma unroll
    for (int i = 0; i < 9; ++i) Fn[i] = st[(PF + i) * cap + pi];
    const float Jp = st[PPL * cap + pi], vol = st[PVOL * cap + pi];
    int nid[3][ORDER + 1];
    float w[3][4], dw[3][4];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int base = stencil_base<ORDER>(g[d], P.res[d]);
#pragma unroll
      for (int o = 0; o < ORDER + 1; ++o) {
        const int nn = base + o;
        const bool in = nn >= 0 && nn < P.res[d];  // out-of-grid nodes: zero weight, clamped index
        spline<ORDER>(g[d] - (float)nn, w[d][o], dw[d][o]);
        w[d][o] = in ? w[d][o] : 0.0f;
        dw[d][o] = in ? dw[d][o] * P.inv_h[d] : 0.0f;
        nid[d][o] = nn < 0 ? 0 : (nn >= P.res[d] ? P.res[d] - 1 : nn);
      }
    }
    const int64_t res0 = P.res[0], res01 = (int64_t)P.res[0] * P.res[1];
    float G[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) G[i] = 0.0f;
#pragma unroll 1
    for (int oz = 0; oz < ORDER + 1; ++oz) {
      float wz = w[2][0], dwz = dw[2][0];
      int nz = nid[2][0];
#pragma unroll
      for (int o = 1; o < ORDER + 1; ++o) {
        wz = oz == o ? w[2][o] : wz;
        dwz = oz == o ? dw[2][o] : dwz;
        nz = oz == o ? nid[2][o] : nz;
      }
      float4 q[ORDER + 1][ORDER + 1];
#pragma unroll
      for (int oy = 0; oy < ORDER + 1; ++oy) {
        const float4* rp = gvel + 2 * (nz * res01 + nid[1][oy] * res0);
#pragma unroll
        for (int ox = 0; ox < ORDER + 1; ++ox) q[oy][ox] = rp[2 * nid[0][ox]];
      }
#pragma unroll
      for (int oy = 0; oy < ORDER + 1; ++oy) {
        float A[3] = {0.0f, 0.0f, 0.0f}, Ad[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ox = 0; ox < ORDER + 1; ++ox) {
          const float vi[3] = {q[oy][ox].x, q[oy][ox].y, q[oy][ox].z};
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            A[r] += w[0][ox] * vi[r];
            Ad[r] += dw[0][ox] * vi[r];
          }
        }
        const float wyz = w[1][oy] * wz, dyz = dw[1][oy] * wz, ydz = w[1][oy] * dwz;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          G[3 * r] += wyz * Ad[r];
          G[3 * r + 1] += dyz * A[r];
          G[3 * r + 2] += ydz * A[r];
        }
      }
    }
    if (particle_kind(P, pid) == KIND_PARTICLE) {
      float GF[9], Fh[9], Sp[9];
      mat_mul(G, Fn, GF);
#pragma unroll
      for (int i = 0; i < 9; ++i) Fh[i] = Fn[i] + dt * GF[i];
      stress_matrix(P, Fh, Fn, Jp, vol, Sp, fb);
#pragma unroll
      for (int i = 0; i < 9; ++i) a.stress[i * cap + j] = Sp[i];
    }
  }
  if (__ballot(fb != 0)) {  // one atomic per wave
    unsigned long long c = (unsigned long long)fb;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if (lane_id() == 0) atomicAdd(a.fallback_svd, c);
  }
}

// Constants of a tile's scene.
struct TileScene {
  P2GScene S;
  int64_t noff;
  int sc, toff, nt0, nt1;
};
__device__ __forceinline__ TileScene tile_scene(const P2GArgs& a, int sc) {
  TileScene n;
  const auto P = as_const(a.T.params) + sc;
  n.sc = sc;
  n.S = p2g_scene(*P);
  n.noff = as_const(a.T.node_off)[sc];
  n.toff = as_const(a.T.tile_off)[sc];
  n.nt0 = P->tiles[0];
  n.nt1 = P->tiles[1];
  return n;
}

// A tile's first cell (uniform) and, of a wave's ROWS rows from row0, the lane's cells as loaded (lo, hi hold
// something else where occ is 0), in one round trip.
struct TileRows {
  int t0, t1, t2;
  uint32_t occ[2];
  int lo[2], hi[2];
};
template <int ROWS>
__device__ __forceinline__ TileRows tile_rows(const P2GArgs& a, const TileScene& n, int gtile, int cx, int layer, int row0) {
  TileRows b;
  const int tile = gtile - n.toff;
  b.t0 = tile % n.nt0;
  b.t1 = (tile / n.nt0) % n.nt1;
  b.t2 = tile / (n.nt0 * n.nt1);
  const int g0 = 4 * b.t0 + cx, g2 = 4 * b.t2 + layer;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int g1 = 4 * b.t1 + row0 + r;
    const bool in = g0 < n.S.res[0] && g1 < n.S.res[1] && g2 < n.S.res[2];
    const int64_t key = n.noff + (in ? (g2 * n.S.res[1] + g1) * n.S.res[0] + g0 : 0);
    b.occ[r] = a.occ[key / SCAN_TILE];
    b.lo[r] = a.cell_start[key];
    b.hi[r] = a.cell_end[key];
    if (!in) b.occ[r] = 0u;
  }
  return b;
}


template <int ORDER, int MODE, int RANKS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_p2g(P2GArgs a) {
  if (clock_skip(a.clk)) return;
  const float dt = clock_dt(a.clk, a.dt);
  constexpr int P2G_RANKS = RANKS;
  constexpr int PAY_CELL = pay_cell<RANKS>();
  constexpr int ROWS = 16 / WAVES;  // rows per wave
  __shared__ float4 s_pay[WAVES][4 * PAY_CELL / 4];
  __shared__ float s_slab[P2G_SLABS][4][SLAB];  // [layer + 4 row half][quantity][node]
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  // wave w owns cell layer z = w & 3 and ROWS rows from row0
  const int layer = w & 3, row0 = __builtin_amdgcn_readfirstlane(ROWS * (w >> 2));
  const int ntile = as_const(a.counters)[CNT_TILES];
  constexpr int NQ = (MODE == P2G_FORCE) ? 3 : 4;
  // staging role: lane (cx, sr), sr < RANKS; accumulation role: lane (cx, zo, oy)
  const int cx = lane >> 4, sr = lane & 15;
  const int zo = (lane >> 2) & 3, oy = lane & 3;
  const float foy = (float)oy, fzo = (float)zo;
  float* slab = &s_slab[layer + 4 * (row0 >> 1)][0][0];
  for (int i = tid; i < P2G_SLABS * 4 * SLAB; i += 64 * WAVES) (&s_slab[0][0][0])[i] = 0.0f;
  __syncthreads();
  // the tiles of one XCD are a contiguous range of the (ascending) active tiles
  const XcdRange tr = xcd_range(ntile);
  if (tr.first >= tr.end) return;  // uniform: no tile for this workgroup
  const auto tiles = as_const(a.active_tiles);
  auto scene_at = [&](int gtile) {
    return a.T.nscenes == 1 ? 0 : __builtin_amdgcn_readfirstlane(scene_of(as_const(a.T.tile_off), a.T.nscenes, gtile));
  };
  const int last = tr.first + (tr.end - 1 - tr.first) / tr.stride * tr.stride;  // this workgroup's last list entry
  int gtile = tiles[tr.first];
  int gtile_next = tiles[min(tr.first + tr.stride, last)];
  TileScene n = tile_scene(a, scene_at(gtile));
  TileRows rows = tile_rows<ROWS>(a, n, gtile, cx, layer, row0);
  // the lane's cell of each of the wave's rows, and each row's largest count (uniform)
  int rstart0, rcnt0, rstart1, rcnt1, rmax0, rmax1;
  auto take_rows = [&]() {
    rstart0 = rows.lo[0];
    rcnt0 = rows.occ[0] ? rows.hi[0] - rows.lo[0] : 0;
    rstart1 = ROWS == 2 ? rows.lo[1] : 0;
    rcnt1 = ROWS == 2 && rows.occ[1] ? rows.hi[1] - rows.lo[1] : 0;
    rmax0 = max(max(__builtin_amdgcn_readlane(rcnt0, 0), __builtin_amdgcn_readlane(rcnt0, 16)),
                max(__builtin_amdgcn_readlane(rcnt0, 32), __builtin_amdgcn_readlane(rcnt0, 48)));
    rmax1 = max(max(__builtin_amdgcn_readlane(rcnt1, 0), __builtin_amdgcn_readlane(rcnt1, 16)),
                max(__builtin_amdgcn_readlane(rcnt1, 32), __builtin_amdgcn_readlane(rcnt1, 48)));
  };
  for (int slot = tr.first; slot < tr.end; slot += tr.stride) {
    const int g0 = 4 * rows.t0 + cx, t1 = rows.t1, g2 = 4 * rows.t2 + layer;  // this lane's cell of each row (both roles)
    const P2GScene S = n.S;  // this tile's
    take_rows();
    if (slot + tr.stride < tr.end) {  // the next tile's cells
      gtile = gtile_next;
      gtile_next = tiles[min(slot + 2 * tr.stride, last)];
      const int sc_next = scene_at(gtile);
      if (sc_next != n.sc) n = tile_scene(a, sc_next);
      rows = tile_rows<ROWS>(a, n, gtile, cx, layer, row0);
    }
    auto rmax_of = [&](int r) { return r == 0 ? rmax0 : rmax1; };
    auto rcnt_of = [&](int r) { return r == 0 ? rcnt0 : rcnt1; };
    auto rstart_of = [&](int r) { return r == 0 ? rstart0 : rstart1; };
    // walk the (row, chunk) steps in order (row 2 = done), loading the particles ahead
    auto next_row = [&](int r) { return (r == 0 && rmax0 > 0) ? 0 : ((r <= 1 && rmax1 > 0) ? 1 : 2); };
    auto advance = [&](int& r, int& kk) {
      if (r >= 2) return;
      if (P2G_RANKS * (kk + 1) >= rmax_of(r)) {
        r = next_row(r + 1);
        kk = 0;
      } else {
        ++kk;
      }
    };
    int cr = next_row(0), k = 0;
    StageIn in;
    // slot of this lane's particle two steps ahead (step after the next)
    int cr2 = cr, k2 = k;
    advance(cr2, k2);
    int pi2 = 0;
    if (cr < 2 && sr < P2G_RANKS && sr < rcnt_of(cr)) p2g_load<MODE>(a, S, rstart_of(cr) + sr, in);
    if (cr2 < 2 && sr < P2G_RANKS && P2G_RANKS * k2 + sr < rcnt_of(cr2))
      pi2 = p2g_slot(a, rstart_of(cr2) + P2G_RANKS * k2 + sr);
    float acc[4][NQ];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[i][q] = 0.0f;
    // row sums into the slab: phase ox, node (cx + ox, cy + oy, zo)
    auto add_row = [&](int cy) {
#pragma unroll
      for (int ox = 0; ox < 4; ++ox) {
        const int ln = (cx + ox) + FOOT * (cy + oy) + FOOT * FOOT * zo;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {  // no other wave's at this time, and a different node per lane: no atomics
          slab[q * SLAB + ln] += acc[ox][q];
          acc[ox][q] = 0.0f;
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      }
    };
    while (cr < 2) {
      const int cy = row0 + cr;
      const int g1 = 4 * t1 + cy;
      const int cnt = rcnt_of(cr);
      // ---- stage ranks RANKS k .. RANKS k + RANKS - 1 of each cell of the row
      if (sr < P2G_RANKS) {
        const int rank = P2G_RANKS * k + sr;
        if (rank < cnt) {
          p2g_stage<ORDER, MODE>(a, S, dt, in, g0, g1, g2, &s_pay[w][(cx * PAY_CELL + sr * PAY_STRIDE) / 4]);
        }
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      // ---- the next step: its particles' data (their slots arrived during this step), and the
      // slots of the step after it
      const int ncr = cr2, nk = k2;
      if (ncr < 2 && sr < P2G_RANKS && P2G_RANKS * nk + sr < rcnt_of(ncr))
        p2g_load_at<MODE>(a, S, pi2, rstart_of(ncr) + P2G_RANKS * nk + sr, in);
      advance(cr2, k2);
      if (cr2 < 2 && sr < P2G_RANKS && P2G_RANKS * k2 + sr < rcnt_of(cr2))
        pi2 = p2g_slot(a, rstart_of(cr2) + P2G_RANKS * k2 + sr);
      // ---- accumulate this lane's cell, ascending rank
      const int nr = min(P2G_RANKS, cnt - P2G_RANKS * k);
      for (int r = 0; r < nr; ++r) {
        const float4* src = &s_pay[w][(cx * PAY_CELL + r * PAY_STRIDE) / 4];
        const float* pf = reinterpret_cast<const float*>(src);
        const float4 WX = src[0];
        const float wxs[4] = {WX.x, WX.y, WX.z, WX.w};
        const float wy = pf[PY_WY + oy], dwy = pf[PY_DWY + oy], wz = pf[PY_WZ + zo], dwz = pf[PY_DWZ + zo];
        float g[12];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const float4 t = src[PY_G / 4 + i];
          g[4 * i] = t.x; g[4 * i + 1] = t.y; g[4 * i + 2] = t.z; g[4 * i + 3] = t.w;
        }
        float qs[16];  // m, q0(3), Q12(6), S12(6)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 t = src[PY_M / 4 + i];
          qs[4 * i] = t.x; qs[4 * i + 1] = t.y; qs[4 * i + 2] = t.z; qs[4 * i + 3] = t.w;
        }
        const float wyz = wy * wz, dyz = dwy * wz, ydz = wy * dwz;
        float e[3];
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) {
          float qrow = qs[1 + rr];
          if constexpr (MODE != P2G_FORCE)
            qrow = __builtin_fmaf(qs[4 + 2 * rr + 1], fzo, __builtin_fmaf(qs[4 + 2 * rr], foy, qrow));
          e[rr] = wyz * qrow;
          if constexpr (MODE != P2G_MOM)
            e[rr] = __builtin_fmaf(-qs[10 + 2 * rr + 1], ydz, __builtin_fmaf(-qs[10 + 2 * rr], dyz, e[rr]));
        }
        const float mw = qs[0] * wyz;
#pragma unroll
        for (int ox = 0; ox < 4; ++ox) {
          const float wx = wxs[ox];
          constexpr int q1 = (MODE != P2G_FORCE) ? 1 : 0;
          if constexpr (MODE != P2G_FORCE) acc[ox][0] = __builtin_fmaf(wx, mw, acc[ox][0]);
#pragma unroll
          for (int rr = 0; rr < 3; ++rr)
            acc[ox][q1 + rr] = __builtin_fmaf(wyz, g[3 * ox + rr], __builtin_fmaf(wx, e[rr], acc[ox][q1 + rr]));
        }
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (ROWS == 2 && ncr != cr) add_row(cy);
      cr = ncr;
      k = nk;
    }
    if constexpr (ROWS == 1) {  // the two waves of a slab one after the other, in row order
      if (row0 % 2 == 0 && rmax0 > 0) add_row(row0);
      __syncthreads();
      if (row0 % 2 == 1 && rmax0 > 0) add_row(row0);
    }
    __syncthreads();
    // ---- tile partial: node (X, Y, Z) = sum over layers l, 0 <= Z - l <= 3, ascending, and within a
    // layer over the row halves in order; slabs cleared
    float* part = a.partials + (size_t)slot * PART_STRIDE + (MODE == P2G_FORCE ? 4 * FOOT3 : 0);
    for (int i = tid; i < FOOT3; i += 64 * WAVES) {
      const int X = i % FOOT, Y = (i / FOOT) % FOOT, Z = i / (FOOT * FOOT);
      float s[NQ];
#pragma unroll
      for (int q = 0; q < NQ; ++q) s[q] = 0.0f;
#pragma unroll
      for (int ww = 0; ww < P2G_SLABS; ++ww) {
        const int l = ww >> 1, hh = ww & 1, wv = l + 4 * hh;
        const int z = Z - l;
        if (z < 0 || z > 3) continue;
        const int ln = X + FOOT * Y + FOOT * FOOT * z;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          s[q] += s_slab[wv][q][ln];
          s_slab[wv][q][ln] = 0.0f;
        }
      }
      if constexpr (NQ == 4) {
        reinterpret_cast<float4*>(part)[i] = make_float4(s[0], s[1], s[2], s[3]);
      } else {
#pragma unroll
        for (int q = 0; q < NQ; ++q) part[q * FOOT3 + i] = s[q];
      }
    }
    __syncthreads();
  }
}

// The first cell of a wave's layer of a tile (uniform), and the lane's cell: occ, lo and hi as loaded (lo, hi
// hold something else where occ is 0).
struct TileCell {
  int g0, g1, g2;
  uint32_t occ;
  int lo, hi;
};
__device__ __forceinline__ TileCell tile_cell(const P2GArgs& a, const TileScene& n, int gtile, int cx, int cy, int cz) {
  TileCell b;
  const int tile = gtile - n.toff;
  const int t0 = tile % n.nt0, t1 = (tile / n.nt0) % n.nt1, t2 = tile / (n.nt0 * n.nt1);
  b.g0 = 4 * t0;
  b.g1 = 4 * t1;
  b.g2 = 4 * t2 + cz;
  const bool in = b.g0 + cx < n.S.res[0] && b.g1 + cy < n.S.res[1] && b.g2 < n.S.res[2];
  const int64_t key = n.noff + (in ? (b.g2 * n.S.res[1] + b.g1 + cy) * n.S.res[0] + b.g0 + cx : 0);
  b.occ = a.occ[key / SCAN_TILE];
  b.lo = a.cell_start[key];
  b.hi = a.cell_end[key];
  if (!in) b.occ = 0u;
  return b;
}

// Layer pass (the other P2G schedule). One workgroup (4 waves) per
// active tile; wave w owns cell layer z = w and all 16 cells of it at once. Staging lane (c, r),
// c = lane >> 2 (cell x = c & 3, y = c >> 2), r < RANKS, stages rank RANKS k + r of cell c; then
// lane (c, zo) adds the chunk's particles of cell c, in ascending rank, to 16 x 4 register sums:
// nodes (x-1+ox, y-1+oy, z-1+zo) of the cell's 4x4x4 window. Four lanes read each payload, instead
// of the row pass's sixteen. The arithmetic per particle and node, the split of a layer into two
// row halves with a slab each, the order in which a slab node receives the cell sums (rows
// ascending, then ox ascending: phases oy = 3..0, ox = 0..3) and the order of the slab sums are
// those of the row pass, so both passes give the same bits.
//
// Bound by vector instructions (two thirds of the VALU's cycles) and by what is exposed of each tile's chain
// of loads (list entry, bins, slots, particles) before its first particle. So the next tile's bins are loaded
// before this tile's chunks, its first slots after them, and its first particles before the slab sums are
// stored; and a wave's slabs take the place of its payloads, which are done with by then: 52 KB a workgroup
// instead of 71, three on a CU instead of two. P2G at 2^22 particles (7.5 per cell) 302 -> 272 us; 16 scenes
// of 1.8 M in all 157 -> 148 us. Three on a CU leave a wave 168 registers; with momentum and stress in one pass that is
// two too few, and the compiler stores one pair before the loop over the tiles and loads it once per tile (12 bytes of
// scratch a lane, nothing in the particle loops).
template <int ORDER, int MODE, int RANKS>
__global__ __launch_bounds__(256, 3) void k_p2g_layer(P2GArgs a) {
  if (clock_skip(a.clk)) return;
  const float dt = clock_dt(a.clk, a.dt);
  constexpr int PAY_CELL = RANKS * PAY_STRIDE;
  constexpr int NQ = (MODE == P2G_FORCE) ? 3 : 4;
  constexpr int WAVE_FLOATS = 16 * PAY_CELL > 2 * NQ * SLAB ? 16 * PAY_CELL : 2 * NQ * SLAB;
  __shared__ float4 s_wave[4][WAVE_FLOATS / 4];
  static_assert(WAVE_FLOATS % 4 == 0 && (2 * NQ * SLAB) % 4 == 0, "float4 slots");
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int ntile = as_const(a.counters)[CNT_TILES];
  const int c = lane >> 2, sr = lane & 3, zo = lane & 3;  // staging (c, sr); accumulation (c, zo)
  const int cx = c & 3, cy = c >> 2;
  const float fzo = (float)zo;
  float4* pay = &s_wave[w][0];
  float* slab = reinterpret_cast<float*>(pay) + (cy >> 1) * NQ * SLAB;  // [row half][quantity][node]
  const XcdRange tr = xcd_range(ntile);
  if (tr.first >= tr.end) return;  // uniform: no tile for this workgroup
  auto scene_at = [&](int gtile) {
    return a.T.nscenes == 1 ? 0 : __builtin_amdgcn_readfirstlane(scene_of(as_const(a.T.tile_off), a.T.nscenes, gtile));
  };
  const int last = tr.first + (tr.end - 1 - tr.first) / tr.stride * tr.stride;  // this workgroup's last list entry
  const auto tiles = as_const(a.active_tiles);
  int gtile = tiles[tr.first];
  int gtile_next = tiles[min(tr.first + tr.stride, last)];
  TileScene n = tile_scene(a, scene_at(gtile));
  TileCell cell = tile_cell(a, n, gtile, cx, cy, w);
  int start = cell.lo, cnt = cell.occ ? cell.hi - cell.lo : 0;
  StageIn in;
  int pi2 = 0;  // slot of this lane's particle in the chunk after the next
  if (sr < RANKS && sr < cnt) p2g_load<MODE>(a, n.S, start + sr, in);
  if (sr < RANKS && RANKS + sr < cnt) pi2 = p2g_slot(a, start + RANKS + sr);
  for (int slot = tr.first; slot < tr.end; slot += tr.stride) {
    // the next tile's cells (the last tile's own again at the end: loaded, not used)
    gtile = gtile_next;
    gtile_next = tiles[min(slot + 2 * tr.stride, last)];
    const P2GScene S = n.S;  // this tile's
    const int sc_next = scene_at(gtile);
    if (sc_next != n.sc) n = tile_scene(a, sc_next);
    const TileCell next = tile_cell(a, n, gtile, cx, cy, w);
    int cmax = cnt;
#pragma unroll
    for (int off = 4; off < 64; off <<= 1) cmax = max(cmax, __shfl_xor(cmax, off));
    cmax = __builtin_amdgcn_readfirstlane(cmax);
    float acc[4][4][NQ];  // [oy][ox][quantity]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[i][j][q] = 0.0f;
    for (int k = 0; k * RANKS < cmax; ++k) {
      if (sr < RANKS && RANKS * k + sr < cnt)
        p2g_stage<ORDER, MODE>(a, S, dt, in, cell.g0 + cx, cell.g1 + cy, cell.g2, pay + (c * PAY_CELL + sr * PAY_STRIDE) / 4);
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (sr < RANKS) {  // the next chunk's data and the slots of the one after
        if (RANKS * (k + 1) + sr < cnt) p2g_load_at<MODE>(a, S, pi2, start + RANKS * (k + 1) + sr, in);
        if (RANKS * (k + 2) + sr < cnt) pi2 = p2g_slot(a, start + RANKS * (k + 2) + sr);
      }
      const int nr = min(RANKS, cnt - RANKS * k);
      for (int r = 0; r < nr; ++r) {
        const float4* src = pay + (c * PAY_CELL + r * PAY_STRIDE) / 4;
        const float* pf = reinterpret_cast<const float*>(src);
        const float4 WX = src[PY_WX / 4], WY = src[PY_WY / 4], DWY = src[PY_DWY / 4];
        const float wxs[4] = {WX.x, WX.y, WX.z, WX.w};
        const float wys[4] = {WY.x, WY.y, WY.z, WY.w};
        const float dwys[4] = {DWY.x, DWY.y, DWY.z, DWY.w};
        const float wz = pf[PY_WZ + zo], dwz = pf[PY_DWZ + zo];
        float g[12];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const float4 t = src[PY_G / 4 + i];
          g[4 * i] = t.x; g[4 * i + 1] = t.y; g[4 * i + 2] = t.z; g[4 * i + 3] = t.w;
        }
        float qs[16];  // m, q0(3), Q12(6), S12(6)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 t = src[PY_M / 4 + i];
          qs[4 * i] = t.x; qs[4 * i + 1] = t.y; qs[4 * i + 2] = t.z; qs[4 * i + 3] = t.w;
        }
#pragma unroll
        for (int oy = 0; oy < 4; ++oy) {
          const float wy = wys[oy], dwy = dwys[oy];
          const float wyz = wy * wz, dyz = dwy * wz, ydz = wy * dwz;
          float e[3];
#pragma unroll
          for (int rr = 0; rr < 3; ++rr) {
            float qrow = qs[1 + rr];
            if constexpr (MODE != P2G_FORCE)
              qrow = __builtin_fmaf(qs[4 + 2 * rr + 1], fzo, __builtin_fmaf(qs[4 + 2 * rr], (float)oy, qrow));
            e[rr] = wyz * qrow;
            if constexpr (MODE != P2G_MOM)
              e[rr] = __builtin_fmaf(-qs[10 + 2 * rr + 1], ydz, __builtin_fmaf(-qs[10 + 2 * rr], dyz, e[rr]));
          }
          const float mw = qs[0] * wyz;
#pragma unroll
          for (int ox = 0; ox < 4; ++ox) {
            const float wx = wxs[ox];
            constexpr int q1 = (MODE != P2G_FORCE) ? 1 : 0;
            if constexpr (MODE != P2G_FORCE) acc[oy][ox][0] = __builtin_fmaf(wx, mw, acc[oy][ox][0]);
#pragma unroll
            for (int rr = 0; rr < 3; ++rr)
              acc[oy][ox][q1 + rr] =
                  __builtin_fmaf(wyz, g[3 * ox + rr], __builtin_fmaf(wx, e[rr], acc[oy][ox][q1 + rr]));
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    // the slots of the next tile's first two chunks
    cell = next;
    start = cell.lo;
    cnt = cell.occ && slot + tr.stride < tr.end ? cell.hi - cell.lo : 0;
    int pi1 = 0;
    if (sr < RANKS && sr < cnt) pi1 = p2g_slot(a, start + sr);
    if (sr < RANKS && RANKS + sr < cnt) pi2 = p2g_slot(a, start + RANKS + sr);
    // ---- the payloads are done with: clear the wave's slabs, then the cells' sums into the slab of their
    // row half: phase (oy descending, ox ascending), node (cx + ox, cy + oy, zo); a node receives its cells
    // in ascending row, then ascending ox
    for (int i = lane; i < 2 * NQ * SLAB / 4; i += 64) pay[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (cmax > 0) {
#pragma unroll
      for (int oy = 3; oy >= 0; --oy)
#pragma unroll
        for (int ox = 0; ox < 4; ++ox) {
          const int ln = (cx + ox) + FOOT * (cy + oy) + FOOT * FOOT * zo;
#pragma unroll
          for (int q = 0; q < NQ; ++q) slab[q * SLAB + ln] += acc[oy][ox][q];  // own slab, a node per lane
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    if (sr < RANKS && sr < cnt) p2g_load_at<MODE>(a, n.S, pi1, start + sr, in);  // the next tile's first chunk
    __syncthreads();
    // ---- tile partial: layers l ascending, row halves in order
    float* part = a.partials + (size_t)slot * PART_STRIDE + (MODE == P2G_FORCE ? 4 * FOOT3 : 0);
    for (int i = tid; i < FOOT3; i += 256) {
      const int X = i % FOOT, Y = (i / FOOT) % FOOT, Z = i / (FOOT * FOOT);
      float sum[NQ];
#pragma unroll
      for (int q = 0; q < NQ; ++q) sum[q] = 0.0f;
#pragma unroll
      for (int ww = 0; ww < 8; ++ww) {
        const int l = ww >> 1, hh = ww & 1, z = Z - l;
        if (z < 0 || z > 3) continue;
        const float* p = reinterpret_cast<const float*>(&s_wave[l][0]) + hh * NQ * SLAB + X + FOOT * Y + FOOT * FOOT * z;
#pragma unroll
        for (int q = 0; q < NQ; ++q) sum[q] += p[q * SLAB];
      }
      if constexpr (NQ == 4) {
        reinterpret_cast<float4*>(part)[i] = make_float4(sum[0], sum[1], sum[2], sum[3]);
      } else {
#pragma unroll
        for (int q = 0; q < NQ; ++q) part[q * FOOT3 + i] = sum[q];
      }
    }
    __syncthreads();
  }
}

// ================================================================== grid update
// One 64-thread workgroup per active 4x4x4 node block; each node sums the partials of the (at most
// 2 per axis) tiles whose footprint covers it, in ascending tile order, then applies
// v = p/m (HybridSolver.cpp:233-240), v += dt (f/m + g) (:457, :725-737) and collision (:460-511).
template <int MODE>
__global__ __launch_bounds__(64) void k_grid(GridArgs a) {
  if (clock_skip(a.clk)) return;
  const float dt = clock_dt(a.clk, a.dt);
  const int nblk = as_const(a.counters)[CNT_BLOCKS];
  float vmax = 0.0f;  // max |v| over this lane's nodes after the velocity update
  const int lx = threadIdx.x & 3, ly = (threadIdx.x >> 2) & 3, lz = threadIdx.x >> 4;
  const XcdRange br = xcd_range(nblk);
  for (int s = br.first; s < br.end; s += br.stride) {
    const int gblk = as_const(a.active_blocks)[s];
    const int sc = __builtin_amdgcn_readfirstlane(scene_of(as_const(a.T.tile_off), a.T.nscenes, gblk));
    const auto& P = as_const(a.T.params)[sc];
    const int toff = as_const(a.T.tile_off)[sc];
    const int blk = gblk - toff;
    const int nt0 = P.tiles[0], nt1 = P.tiles[1], nt2 = P.tiles[2];
    const int b0 = blk % nt0, b1 = (blk / nt0) % nt1, b2 = blk / (nt0 * nt1);
    // the slots of the 27 tiles around the block (b - 1 .. b + 1 per axis), one lane each; every
    // node of the block is covered by tiles among them
    int slot27 = -1;
    {
      const int q = (int)threadIdx.x;
      const int u0 = b0 - 1 + q % 3, u1 = b1 - 1 + (q / 3) % 3, u2 = b2 - 1 + q / 9;
      if (q < 27 && u0 >= 0 && u1 >= 0 && u2 >= 0 && u0 < nt0 && u1 < nt1 && u2 < nt2)
        slot27 = a.tile_slot[toff + (u2 * nt1 + u1) * nt0 + u0];
    }
    const int r0 = P.res[0], r1 = P.res[1], r2 = P.res[2];
    const int n0 = 4 * b0 + lx, n1 = 4 * b1 + ly, n2 = 4 * b2 + lz;
    const bool in_grid = n0 < r0 && n1 < r1 && n2 < r2;
    const int64_t node = as_const(a.T.node_off)[sc] + ((int64_t)n2 * r1 + n1) * r0 + n0;
    const int nn[3] = {n0, n1, n2}, ntl[3] = {nt0, nt1, nt2};
    // covering tiles of this node along each axis: tlo and tlo + 1 (if <= thi), both in b - 1 .. b + 1
    int tlo[3], thi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      int lo = (nn[d] - 5 + 3) / 4;  // ceil((n-5)/4) for n >= 2; clamped below
      if (nn[d] - 5 < 0) lo = 0;
      int hi = (nn[d] + 1) / 4;
      thi[d] = hi < ntl[d] - 1 ? hi : ntl[d] - 1;
      tlo[d] = lo;
    }
    const int qoff = (MODE == GRID_FORCE_UPDATE) ? 4 : 0;
    constexpr int NQ = (MODE == GRID_FORCE_UPDATE) ? 3 : 4;
    // all partial loads of the node first (at most 2 x 2 x 2 tiles), then the sums in ascending tile
    // order (t2, t1, t0), as a loop over the covering tiles would add them
    float val[8][NQ];
    bool use[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int t0 = tlo[0] + (k & 1), t1 = tlo[1] + ((k >> 1) & 1), t2 = tlo[2] + (k >> 2);
      const int q27 = (t2 - (b2 - 1)) * 9 + (t1 - (b1 - 1)) * 3 + (t0 - (b0 - 1));
      const int sl = __shfl(slot27, q27);  // q27 is in [0, 27): lanes 0..26 hold the slots
      use[k] = in_grid && t0 <= thi[0] && t1 <= thi[1] && t2 <= thi[2] && q27 >= 0 && q27 < 27 && sl >= 0;
      const int ln = (n0 - (4 * t0 - 1)) + FOOT * (n1 - (4 * t1 - 1)) + FOOT * FOOT * (n2 - (4 * t2 - 1));
      const float* part = a.partials + (size_t)(use[k] ? sl : 0) * PART_STRIDE + qoff * FOOT3;
      const int pn = use[k] ? ln : 0;
      // unconditional loads (an unused tile reads slot 0, node 0: in bounds) keep them all in flight
      if constexpr (NQ == 4) {  // m, p of a node: one float4
        const float4 p4 = reinterpret_cast<const float4*>(part)[pn];
        val[k][0] = p4.x;
        val[k][1] = p4.y;
        val[k][2] = p4.z;
        val[k][3] = p4.w;
      } else {
#pragma unroll
        for (int q = 0; q < NQ; ++q) val[k][q] = part[q * FOOT3 + pn];
      }
    }
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int q = 0; q < NQ; ++q) sum[q] = use[k] ? sum[q] + val[k][q] : sum[q];
    if (!in_grid) continue;
    float v[3], vbf[3];
    if constexpr (MODE == GRID_FORCE_UPDATE) {
      const float m = a.gm[node];
      const float4 g4 = a.gvel[2 * node];
      v[0] = g4.x; v[1] = g4.y; v[2] = g4.z;
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (m > 0.0f) v[d] += dt * (sum[d] / m + P.gravity[d]);
    } else {
      const float m = sum[0];
      a.gm[node] = m;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        a.gmom[d * a.ng + node] = sum[1 + d];
        v[d] = m > 0.0f ? sum[1 + d] / m : 0.0f;
        if (MODE == GRID_FUSED && m > 0.0f) v[d] += dt * P.gravity[d];
      }
    }
    vmax = fmaxf(vmax, sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
    if constexpr (MODE == GRID_NORMALIZE) {
      vbf[0] = v[0]; vbf[1] = v[1]; vbf[2] = v[2];
    } else {
      const float xn[3] = {P.gmin[0] + (float)n0 * P.h[0], P.gmin[1] + (float)n1 * P.h[1], P.gmin[2] + (float)n2 * P.h[2]};
      collide(P, xn, v, vbf);
    }
    a.gvel[2 * node] = make_float4(v[0], v[1], v[2], vbf[0]);
    a.gvel[2 * node + 1] = make_float4(vbf[1], vbf[2], 0.0f, 0.0f);
  }
  if (a.vmax_out != nullptr) {
    // max over the wave, one atomic per wave (non-negative floats order as their bit patterns)
    for (int off = 32; off > 0; off >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, off));
    // (only a new maximum, as far as this wave can see: the waves' atomics on one word run one after another)
    if (threadIdx.x == 0 && vmax > 0.0f &&
        __hip_atomic_load(a.vmax_out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < __float_as_uint(vmax))
      atomicMax(a.vmax_out, __float_as_uint(vmax));
  }
}

// ================================================================== adaptive time step
// Dt = CFL / max(300, max|v| / h_min) (HybridSolver.cpp:860,878; RegularGrid.cpp:188-200,
// RegularGrid.h:60), evaluated in double as in the reference from the max node speed after the
// velocity update; then the frame clamp to 1/60 s (:880-892): a substep that reaches the frame end
// is shortened to it, t advances by 1/60 and the frame time restarts.
// The new Dt from the velocities after the grid update, and whether it ends the frame: G2P forms it for itself,
// k_clock_end stores it.
struct ClockStep {
  double dt;
  bool frame;
};
__device__ __forceinline__ ClockStep clock_step(const Clock* c, bool init) {
  const double vmax = (double)__uint_as_float(c->vmax_bits);
  const double rate = vmax / c->hmin;
  ClockStep s{c->cfl / (rate > 300.0 ? rate : 300.0), false};
  if (!init && c->inner + s.dt >= 1.0 / 60.0) {
    s.dt = 1.0 / 60.0 - c->inner;
    s.frame = true;
  }
  return s;
}

// The first Dt, before any substep.
__global__ void k_clock_init(Clock* c) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  c->dt = clock_step(c, true).dt;
  c->dt_f = (float)c->dt;
  c->vmax_bits = 0u;
}

// End of a substep: the clock advances by the Dt that its G2P took; the reference closes a frame after the
// substep that completed it (output at HybridSolver.cpp:990-1029) and leaves its loop when t > maxt (:867).
__global__ void k_clock_end(Clock* c, const int* tiles) {
  if (threadIdx.x != 0 || blockIdx.x != 0 || c->skip) return;
  const ClockStep s = clock_step(c, false);
  c->dt = s.dt;
  c->dt_f = (float)s.dt;
  c->vmax_bits = 0u;
  c->tiles = *tiles;
  c->executed += 1;
  c->substeps += 1;
  if (s.frame) {
    c->t += 1.0 / 60.0;
    c->inner = 0.0;
    c->frame += 1;
    c->frame_done = 1;
    c->skip = 1;
  } else {
    c->inner += s.dt;
  }
  if (c->t > c->maxt) {
    c->done = 1;
    c->skip = 1;
  }
}

// ================================================================== G2P + F update + return map
constexpr int G2P_BX = 12;               // x extent of a wave's node box (nodes)
constexpr int G2P_BOX = G2P_BX * 4 * 4;  // nodes of the box: G2P_BX x 4 (y) x 4 (z)

// A node box's nodes, G2P_BOX / 64 per lane (slot i = it * 64 + lane: x = i % G2P_BX, then y, then
// z), in the grid's record layout; slots outside the box read the box's corner (in bounds).
__device__ __forceinline__ void g2p_box_load(const float4* gvel, int lane, int x0, int y0, int z0, int nx, int ny,
                                             int nz, int64_t res0, int64_t res01, float4 (&t)[2 * G2P_BOX / 64]) {
#pragma unroll
  for (int it = 0; it < G2P_BOX / 64; ++it) {
    const int i = it * 64 + lane;
    const int ix = i % G2P_BX, row = i / G2P_BX, iy = row & 3, iz = row >> 2;
    const bool in = ix < nx && iy < ny && iz < nz;
    const int64_t node = (z0 + (in ? iz : 0)) * res01 + (y0 + (in ? iy : 0)) * res0 + (x0 + (in ? ix : 0));
    t[2 * it] = gvel[2 * node];
    t[2 * it + 1] = gvel[2 * node + 1];
  }
}
__device__ __forceinline__ void g2p_box_store(float4* box, int lane, const float4 (&t)[2 * G2P_BOX / 64]) {
#pragma unroll
  for (int it = 0; it < G2P_BOX / 64; ++it) {
    const int i = it * 64 + lane;
    box[2 * i] = t[2 * it];
    box[2 * i + 1] = t[2 * it + 1];
  }
}

// floor(a / d) for 0 <= a < 2^31 with the multiplier m and shift l of d (integer arithmetic only;
// l = 0 means d = 1): t = floor(a m / 2^32), then (t + ((a - t) >> 1)) >> (l - 1).
__device__ __forceinline__ int floor_div(int a, uint32_t m, int l) {
  if (l == 0) return a;
  const uint32_t n = (uint32_t)a, t = __umulhi(n, m);
  return (int)((t + ((n - t) >> 1)) >> (l - 1));
}

// Thread per sorted position j (caller id pid = perm[j]): gathers the stencil of grid v
// (post-collision) and v_BF (pre-friction), computes v_p, APIC B (HybridSolver.cpp:739-825),
// x += dt sum w v_BF (:942-950), F^ = (I + dt sum v_BF grad w^T) F (:553-577) and the return map
// (:612-681), and writes the particle to slot j of the other buffer, so that the buffers stay
// physically sorted by cell. It also records where pid now lives and pid's next cell key.
template <int ORDER>
__global__ __launch_bounds__(256) void k_g2p(G2PArgs a) {
  if (clock_skip(a.clk)) return;
  const float dt = a.clk != nullptr ? (float)clock_step(a.clk, false).dt : a.dt;
  const int pblk = (int)blockIdx.x;
  const PBlock pb = particle_block(a.T, pblk);
  const DevParams P = uniform_params(a.T.params[pb.s]);
  const int64_t noff = a.T.node_off[pb.s];
  const float4* gvel = a.gvel + 2 * noff;
  const int j = pb.j;
  const CellThr thr = cell_thr(a.thr + a.T.thr_off[pb.s], P.res);
  const int toff = a.T.tile_off[pb.s];
  int oob = 0, bad = 0, cfl = 0, fb_svd = 0, fb_apex = 0;
  bool cand = false, apex = false;
  const int wv = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  const int64_t res0 = P.res[0], res01 = (int64_t)P.res[0] * P.res[1];
  // The wave's node boxes. When the wave's positions lie in one row of cells, or in two consecutive
  // rows of one z plane (the sorted cell keys of its positions tell), the nodes c-1 .. c+2 around
  // each row's cells (at most G2P_BX x 4 x 4 per row) are copied into the wave's LDS area, in the
  // grid's own record layout, and the stencil gathers read them there: one round trip to HBM, made
  // together with the particle loads, instead of one per z plane. The keys only place the boxes: a
  // wave uses them only if every lane's stencil lies inside its row's box, and they are clamped to
  // the grid whatever the keys hold.
  __shared__ float4 s_box[4][2][2 * G2P_BOX];
  const uint32_t dm0 = a.T.params[pb.s].div_m[0], dm1 = a.T.params[pb.s].div_m[1];
  const int ds0 = a.T.params[pb.s].div_s[0], ds1 = a.T.params[pb.s].div_s[1];
  // The particle's state and its sorted key, loaded by every lane (lanes past the end read the
  // last position), so that the box below is placed while they are in flight.
  const int jc = j < pb.end ? j : pb.end - 1;
  const uint32_t kj = a.ks[jc];
  const int perm_j = a.perm[jc], src_j = a.src[jc];
  asm volatile("" ::: "memory");  // the three coalesced loads are issued together, first
  const int pid = clamp_index(perm_j, a.n);
  const int pi = clamp_index(src_j, a.n);
  const float* st = a.sin;
  const int64_t cap = a.cap;
  float xp[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) xp[d] = st[(PX + d) * cap + pi];
  float Fn[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) Fn[i] = st[(PF + i) * cap + pi];
  float plastic = st[PPL * cap + pi];
  const float phi_p = st[PPHI * cap + pi];
  const float vol = st[PVOL * cap + pi];
  const float mass = st[PM * cap + pi];
  // Box q covers x bx0q .. +bnxq, y by0q .. +bnyq, z bz0 .. +bnz (uniform). One box when the wave's
  // cells are in one row; two when they are in two consecutive rows of one z plane (lanes below
  // `split` in the first). nbox = 0: the wave gathers from the grid.
  int bx00 = 0, by00 = 0, bnx0 = 0, bny0 = 0, bx01 = 0, by01 = 0, bnx1 = 0, bny1 = 0;
  int bz0 = 0, bnz = 0, nbox = 0, split = 64;
  const int jw = __builtin_amdgcn_readfirstlane(j - lane);
  if (jw < pb.end) {
    const int64_t ncell = (int64_t)P.res[0] * P.res[1] * P.res[2];
    const int64_t lf = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)kj, 0) - noff;
    const int64_t ll = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)kj, 63) - noff;
    if (lf >= 0 && ll >= lf && ll < ncell && ll <= INT32_MAX) {
      const int rf = floor_div((int)lf, dm0, ds0);
      const int rl = floor_div((int)ll, dm0, ds0);
      const int zc = floor_div(rf, dm1, ds1), yc = rf - zc * P.res[1];
      const int xf = (int)lf - rf * P.res[0], xl = (int)ll - rl * P.res[0];
      int xa = xl, xb = xf;  // last x of the first row, first x of the second
      if (rf == rl) {
        nbox = 1;
      } else if (rl == rf + 1 && yc + 1 < P.res[1]) {
        // keys are sorted: the lanes whose cell precedes row rl's first cell are the first row's
        const int64_t r0 = P.res[0], row_end = (int64_t)rl * r0;
        split = __popcll(__ballot((int64_t)(uint32_t)kj - noff < row_end));
        if (split >= 1 && split <= 63) {
          // (clamped to the row: only keys that are not sorted could fall outside it)
          const int64_t ka = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)kj, split - 1) - noff - (int64_t)rf * r0;
          const int64_t kb = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)kj, split) - noff - row_end;
          xa = (int)(ka < 0 ? 0 : (ka >= r0 ? r0 - 1 : ka));
          xb = (int)(kb < 0 ? 0 : (kb >= r0 ? r0 - 1 : kb));
          nbox = 2;
        }
      }
      if (nbox == 1) split = 64;
      bz0 = max(zc - 1, 0);
      bnz = min(zc + 2, P.res[2] - 1) - bz0 + 1;
      bx00 = max(xf - 1, 0);
      bnx0 = min((nbox == 2 ? xa : xl) + 2, P.res[0] - 1) - bx00 + 1;
      by00 = max(yc - 1, 0);
      bny0 = min(yc + 2, P.res[1] - 1) - by00 + 1;
      bx01 = max(xb - 1, 0);
      bnx1 = min(xl + 2, P.res[0] - 1) - bx01 + 1;
      by01 = max(yc, 0);
      bny1 = min(yc + 3, P.res[1] - 1) - by01 + 1;
      bool ok = bnz >= 1 && bnx0 >= 1 && bnx0 <= G2P_BX && bny0 >= 1;
      if (nbox == 2) ok = ok && bnx1 >= 1 && bnx1 <= G2P_BX && bny1 >= 1;
      if (!ok) nbox = 0;
    }
  }
  if (nbox > 0) {
    // the second row's box after the first (one more round trip for those waves, but no more live
    // registers than one box needs)
    {
      float4 t[2 * G2P_BOX / 64];
      g2p_box_load(gvel, lane, bx00, by00, bz0, bnx0, bny0, bnz, res0, res01, t);
      g2p_box_store(&s_box[wv][0][0], lane, t);
    }
    if (nbox == 2) {
      float4 t[2 * G2P_BOX / 64];
      g2p_box_load(gvel, lane, bx01, by01, bz0, bnx1, bny1, bnz, res0, res01, t);
      g2p_box_store(&s_box[wv][1][0], lane, t);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (j < pb.end) {
    float g[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) g[d] = (xp[d] - P.gmin[d]) * P.inv_h[d];
    int base[3];
    float w[3][4], dw[3][4];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      base[d] = stencil_base<ORDER>(g[d], P.res[d]);
      if constexpr (ORDER == 2) {
        quad_weights(g[d] - (float)base[d], w[d], dw[d]);
      } else {
#pragma unroll
        for (int o = 0; o < ORDER + 1; ++o) spline<ORDER>(g[d] - (float)(base[d] + o), w[d][o], dw[d][o]);
      }
    }
    // Out-of-grid nodes are dropped (HybridSolver.cpp:44-47): they get zero weight and an in-range
    // (clamped) index, so every load stays inside the stencil's active node blocks.
    int nid[3][ORDER + 1];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int o = 0; o < ORDER + 1; ++o) {
        const int nn = base[d] + o;
        const bool in = nn >= 0 && nn < P.res[d];
        w[d][o] = in ? w[d][o] : 0.0f;
        dw[d][o] = in ? dw[d][o] : 0.0f;
        nid[d][o] = nn < 0 ? 0 : (nn >= P.res[d] ? P.res[d] - 1 : nn);
      }
    // The stencil sums factor over the axes: along each x row of nodes (fixed y, z) the row sums
    //   A = sum wx v, Ax = sum wx (x_i - x_p) v, C = sum wx v_BF, Cd = sum wx' v_BF
    // are formed first, then weighted by the row's y and z factors:
    //   v_p += wyz A, B[:,0] += wyz Ax, B[:,1] += wyz dy A, B[:,2] += wyz dz A,
    //   sum w v_BF += wyz C, grad v_BF[:,0] += wyz/h Cd, [:,1] += wy' wz/h C, [:,2] += wy wz'/h C.
    float wdx[ORDER + 1];
#pragma unroll
    for (int ox = 0; ox < ORDER + 1; ++ox) wdx[ox] = w[0][ox] * (((float)(base[0] + ox) - g[0]) * P.h[0]);
    float vp[3] = {0.0f, 0.0f, 0.0f}, vb[3] = {0.0f, 0.0f, 0.0f};
    float Bn[9], Gv[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) { Bn[i] = 0.0f; Gv[i] = 0.0f; }
    // node addressing: the wave's box when every lane's stencil lies inside it, else the grid
    const int mb = lane >= split ? 1 : 0;  // this lane's box
    const int lx0 = mb ? bx01 : bx00, ly0 = mb ? by01 : by00, lnx = mb ? bnx1 : bnx0, lny = mb ? bny1 : bny0;
    const bool inside = nid[0][0] >= lx0 && nid[0][ORDER] < lx0 + lnx && nid[1][0] >= ly0 &&
                        nid[1][ORDER] < ly0 + lny && nid[2][0] >= bz0 && nid[2][ORDER] < bz0 + bnz;
    const bool use_box = nbox > 0 && __ballot(!inside) == 0;
    // LDS offsets (in float4, from the wave's first box) of the stencil's x and y nodes in its box
    int bxo[ORDER + 1], byo[ORDER + 1];
#pragma unroll
    for (int o = 0; o < ORDER + 1; ++o) {
      bxo[o] = 2 * (nid[0][o] - lx0);
      byo[o] = 2 * G2P_BOX * mb + 2 * G2P_BX * (nid[1][o] - ly0);
    }
    // one z plane of rows per iteration (not unrolled): its loads are in flight together without
    // holding the whole stencil in registers
#pragma unroll 1
    for (int oz = 0; oz < ORDER + 1; ++oz) {
      float wz = w[2][0], dwz = dw[2][0];
      int nz = nid[2][0];
#pragma unroll
      for (int o = 1; o < ORDER + 1; ++o) {
        wz = oz == o ? w[2][o] : wz;
        dwz = oz == o ? dw[2][o] : dwz;
        nz = oz == o ? nid[2][o] : nz;
      }
      const float dz = ((float)(base[2] + oz) - g[2]) * P.h[2];
      // the plane's (ORDER+1)^2 nodes are loaded together and waited for once (v and v_BF of a
      // node are its two float4, of which the second holds v_BF y, z in x, y), from the wave's box
      // in LDS or from the grid (the branch is uniform)
      float4 qa[ORDER + 1][ORDER + 1];
      float2 qb[ORDER + 1][ORDER + 1];
      if (use_box) {
        const float4* pp = &s_box[wv][0][0] + 2 * (4 * G2P_BX) * (nz - bz0);
#pragma unroll
        for (int oy = 0; oy < ORDER + 1; ++oy)
#pragma unroll
          for (int ox = 0; ox < ORDER + 1; ++ox) {
            qa[oy][ox] = pp[byo[oy] + bxo[ox]];
            qb[oy][ox] = *reinterpret_cast<const float2*>(pp + byo[oy] + bxo[ox] + 1);
          }
      } else {
        const float4* pp = gvel + 2 * (nz * res01);
#pragma unroll
        for (int oy = 0; oy < ORDER + 1; ++oy) {
          const float4* rp = pp + 2 * (nid[1][oy] * res0);
#pragma unroll
          for (int ox = 0; ox < ORDER + 1; ++ox) {
            qa[oy][ox] = rp[2 * nid[0][ox]];
            qb[oy][ox] = *reinterpret_cast<const float2*>(rp + 2 * nid[0][ox] + 1);
          }
        }
      }
#pragma unroll
      for (int oy = 0; oy < ORDER + 1; ++oy) {
        const float dy = ((float)(base[1] + oy) - g[1]) * P.h[1];
        float A[3], Ax[3], C[3], Cd[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) { A[r] = 0.0f; Ax[r] = 0.0f; C[r] = 0.0f; Cd[r] = 0.0f; }
#pragma unroll
        for (int ox = 0; ox < ORDER + 1; ++ox) {
          const float4 q0 = qa[oy][ox];
          const float2 q1 = qb[oy][ox];
          const float vi[3] = {q0.x, q0.y, q0.z};
          const float bi[3] = {q0.w, q1.x, q1.y};
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            A[r] += w[0][ox] * vi[r];
            Ax[r] += wdx[ox] * vi[r];
            C[r] += w[0][ox] * bi[r];
            Cd[r] += dw[0][ox] * bi[r];
          }
        }
        const float wyz = w[1][oy] * wz;
        const float wyzy = wyz * dy, wyzz = wyz * dz;
        const float gx = wyz * P.inv_h[0];
        const float gy = dw[1][oy] * wz * P.inv_h[1];
        const float gz = w[1][oy] * dwz * P.inv_h[2];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          vp[r] += wyz * A[r];
          Bn[3 * r] += wyz * Ax[r];
          Bn[3 * r + 1] += wyzy * A[r];
          Bn[3 * r + 2] += wyzz * A[r];
          vb[r] += wyz * C[r];
          Gv[3 * r] += gx * Cd[r];
          Gv[3 * r + 1] += gy * C[r];
          Gv[3 * r + 2] += gz * C[r];
        }
      }
    }
    float xn[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      xn[d] = xp[d] + dt * vb[d];
      if (fabsf(xn[d] - xp[d]) > P.h[d]) cfl = 1;
    }
    // the next sort's key and counts (of a cloth element: k_cloth_elements, which moves it to its vertices);
    // the atomics are in flight during the return map
    const int kind = particle_kind(P, pid);
    int cell[3];
    const uint32_t key = (uint32_t)noff + cell_key(P, thr, xn[0], xn[1], xn[2], oob, cell);
    const CountTicket ticket =
        count_wave(a.bins, kind != KIND_ELEMENT, key, toff + tile_of(P, cell[0], cell[1], cell[2]));
    // cloth vertices and elements keep only the skew part of B (damping 1, HybridSolver.cpp:926-932)
    const float damping = kind == KIND_PARTICLE ? P.damping : 1.0f;
    if (damping != 0.0f) {
      float C[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) C[i] = Bn[i];
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          float sym = 0.5f * (C[3 * r + c] + C[3 * c + r]);
          Bn[3 * r + c] = (C[3 * r + c] - sym) + (1.0f - damping) * sym;
        }
    }
    float Fh[9], GF[9];
    mat_mul(Gv, Fn, GF);
#pragma unroll
    for (int i = 0; i < 9; ++i) Fh[i] = Fn[i] + dt * GF[i];
    float K[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    SurrogateIO io;
    io.mode = a.sur_mode;
    io.pair_log = a.pair_log;
    io.pair_cap = a.pair_cap;
    io.pair_count = a.pair_count;
    io.deferred = false;
    io.defer_apex = a.apex_mask != nullptr;
    io.apex_deferred = false;
    // particles: return mapping. A cloth element's F planes hold D, of which F^ updates d3
    // (HybridSolver.cpp:599-603); its d1, d2 and return mapping follow in k_cloth_elements.
    if (kind == KIND_PARTICLE) return_map(P, Fh, plastic, phi_p, vol, K, fb_svd, fb_apex, io);
    // A deferred particle's trial SVD goes to its record: the wave's deferred lanes write next to
    // each other from the position of lane 0 (coalesced even where few lanes defer); the wave's mask
    // below lists the particle, and the list carries the record index.
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t dmask = __ballot(io.deferred), amask = __ballot(io.apex_deferred);
    if (io.deferred) {  // a candidate of the surrogate
      cand = true;
      const int64_t n = a.n, r = (j - lane) + __popcll(dmask & below);
#pragma unroll
      for (int k = 0; k < 3; ++k) a.cand[(CAND_SIGMA + k) * n + r] = io.sigma[k];
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        a.cand[(CAND_U + k) * n + r] = io.U[k];
        a.cand[(CAND_V + k) * n + r] = io.V[k];
      }
    }
    if (io.apex_deferred) {  // an FP64 apex projection for k_apex_finish
      apex = true;
      const int64_t n = a.n, r = (j - lane) + __popcll(amask & below);
#pragma unroll
      for (int k = 0; k < 3; ++k) a.apex_usv[(CAND_SIGMA + k) * n + r] = io.sigma[k];
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        a.apex_usv[(CAND_U + k) * n + r] = io.U[k];
        a.apex_usv[(CAND_V + k) * n + r] = io.V[k];
      }
    }
    float* so = a.sout;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      so[(PX + d) * cap + j] = xn[d];
      so[(PV + d) * cap + j] = vp[d];
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      so[(PB + i) * cap + j] = Bn[i];
      so[(PF + i) * cap + j] = Fh[i];
    }
    if (a.write_stress) {
#pragma unroll
      for (int e = 0; e < 6; ++e) so[(PK + e) * cap + j] = K[e];
    }
    so[PPL * cap + j] = plastic;
    so[PM * cap + j] = mass;
    so[PVOL * cap + j] = vol;
    so[PPHI * cap + j] = phi_p;
    reinterpret_cast<int*>(so + (size_t)PID * cap)[j] = pid;
    if (a.pos_out) a.pos_out[pid] = j;
    a.keys[j] = key;
    const uint32_t rank = count_rank(ticket);
    if (kind != KIND_ELEMENT) a.bins.rank[j] = rank;
    bad = !(isfinite(xn[0]) && isfinite(xn[1]) && isfinite(xn[2]) && isfinite(vp[0]) && isfinite(vp[1]) &&
            isfinite(vp[2]) && isfinite(Fh[0]) && isfinite(Fh[4]) && isfinite(Fh[8]) && isfinite(plastic));
  }
  // every wave records its deferred lanes (none past the end of the scene) for the position lists
  if (a.apex_mask || a.sur_mode == 2) {
    const uint64_t am = __ballot(apex), dm = __ballot(cand);
    if (lane == 0) {
      a.wave_pos[4 * pblk + wv] = j;
      if (a.apex_mask) a.apex_mask[4 * pblk + wv] = am;
      if (a.sur_mode == 2) a.cand_mask[4 * pblk + wv] = dm;
    }
  }
  const int flags = (oob ? MPM_STATUS_OUT_OF_DOMAIN : 0) | (bad ? MPM_STATUS_NONFINITE : 0) | (cfl ? MPM_STATUS_CFL : 0);
  if (__ballot(flags != 0)) {
    if (flags) atomicOr(a.status, flags);
  }
  // fallback counts: one atomic per wave
  if (__ballot(fb_svd != 0)) {
    unsigned long long c = (unsigned long long)fb_svd;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if (lane_id() == 0) atomicAdd(a.fallback_svd, c);
  }
  if (__ballot(fb_apex != 0)) {
    unsigned long long c = (unsigned long long)fb_apex;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if (lane_id() == 0) atomicAdd(a.fallback_apex, c);
  }
}

// The FP64 apex projections deferred by k_g2p, gathered into full waves: from the trial SVD that
// k_g2p stored and the particle's q, phi and V, the FP64 projection and F_E and V tau (the same
// function return_map calls, on the same operands), stored over the trial F^ left in the output
// buffer. The result equals computing it inside k_g2p. j: the particle's sorted position, r: its record.
__device__ __forceinline__ void apex_particle(const ApexArgs& a, int j, int r, int& fb_apex) {
  const int sc = scene_of(a.T.part_off, a.T.nscenes, j);
  const DevParams& P = a.T.params[sc];
  float* st = a.st;
  const int64_t cap = a.cap, n = a.n;
  float S[3], U[9], V[9];
#pragma unroll
  for (int k = 0; k < 3; ++k) S[k] = a.apex_usv[(CAND_SIGMA + k) * n + r];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    U[k] = a.apex_usv[(CAND_U + k) * n + r];
    V[k] = a.apex_usv[(CAND_V + k) * n + r];
  }
  float plastic = st[PPL * cap + j];
  const float phi_p = st[PPHI * cap + j];
  const float vol = st[PVOL * cap + j];
  SurrogateIO io;
  io.mode = a.log_pairs ? 1 : 0;
  io.pair_log = a.pair_log;
  io.pair_cap = a.pair_cap;
  io.pair_count = a.pair_count;
  // the FP32 trial strains, as the return map computed them (used by the pair log only)
  float l[3] = {0.0f, 0.0f, 0.0f};
  if (io.mode == 1) {
    l[0] = logf(S[0]);
    l[1] = logf(S[1]);
    l[2] = logf(S[2]);
  }
  float Fe[9], K[6];
  sand_apex_finish(P, U, S, V, l, P.per_particle_phi ? phi_p : P.h0, phi_p, plastic, vol, Fe, K, fb_apex, io);
#pragma unroll
  for (int i = 0; i < 9; ++i) st[(PF + i) * cap + j] = Fe[i];
  st[PPL * cap + j] = plastic;
  if (a.write_stress) {
#pragma unroll
    for (int e = 0; e < 6; ++e) st[(PK + e) * cap + j] = K[e];
  }
}
// One atomic per wave.
__device__ __forceinline__ void apex_fallbacks(const ApexArgs& a, int fb_apex) {
  unsigned long long c = (unsigned long long)fb_apex;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(a.fallback_apex, c);
}

// Without the surrogate, from G2P's masks: a workgroup takes those of `gw` G2P waves at a time (4, a G2P workgroup's,
// where that gives few groups; else 32, which gathers fuller waves), lists their flagged positions in LDS and works the
// list off. Bound by the launch and one round trip of the masks where few particles are flagged, and by scattered writes
// where many are (410k of 2^22: 63 us; in groups of 16 and 64 waves 65-68 and 72, with two list launches before it and
// waves filled over the whole state 53 + 11). With few flagged, G2P and what follows it took 95 us with the list launches
// and 92 without at 2^20 particles, 177 and 171 for 16 scenes.
__global__ __launch_bounds__(256) void k_apex_finish(ApexArgs a) {
  if (clock_skip(a.clk)) return;
  __shared__ int s_slot[64 * APEX_GROUP], s_idx[64 * APEX_GROUP];
  const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
  int fb_apex = 0;
  for (int w0 = (int)blockIdx.x * a.gw; w0 < a.nwaves; w0 += (int)gridDim.x * a.gw) {
    const int nw = min(a.gw, a.nwaves - w0);
    // wave wv lists the masks wv, wv + 4, ...; every wave forms the offsets (lane l: mask l) by itself
    const uint64_t ml = lane < nw ? a.mask[w0 + lane] : 0ull;
    int off = __popcll(ml);
    const int own = off;
#pragma unroll
    for (int d = 1; d < APEX_GROUP; d <<= 1) {
      const int y = __shfl_up(off, d);
      if (lane >= d) off += y;
    }
    const int count = __builtin_amdgcn_readlane(off, APEX_GROUP - 1);
    if (count == 0) continue;  // uniform over the workgroup
    off -= own;
    for (int q = wv; q < nw; q += 4) {
      const uint64_t m = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(ml >> 32), q) << 32) |
                         (uint32_t)__builtin_amdgcn_readlane((int)ml, q);
      const int o = __builtin_amdgcn_readlane(off, q), p = a.wave_pos[w0 + q];
      if ((m >> lane) & 1ull) {
        const int rank = __popcll(m & ((1ull << lane) - 1ull));
        s_slot[o + rank] = p + lane;
        s_idx[o + rank] = p + rank;
      }
    }
    __syncthreads();
    for (int c = (int)threadIdx.x; c < count; c += 256)
      apex_particle(a, clamp_index(s_slot[c], a.n), clamp_index(s_idx[c], a.n), fb_apex);
    __syncthreads();
  }
  apex_fallbacks(a, fb_apex);
}

// Beside the surrogate, whose candidates are listed by launches of their own, from the list that these make as well:
// waves full over the whole state. Both with the lists, 2^22 particles: 75.3 us from the masks, 71.6 so (MI355X).
__global__ __launch_bounds__(256) void k_apex_list(ApexArgs a) {
  if (clock_skip(a.clk)) return;
  const int count = min(*a.count, a.n);
  int fb_apex = 0;
  for (int c = (int)blockIdx.x * 256 + (int)threadIdx.x; c < count; c += (int)gridDim.x * 256)
    apex_particle(a, clamp_index(a.list[c], a.n), clamp_index(a.idx[c], a.n), fb_apex);
  apex_fallbacks(a, fb_apex);
}

// ================================================================== position lists
// Lists of the sorted positions that G2P flagged, in ascending order and without atomics: the surrogate's candidates
// and, beside them, the deferred FP64 apex projections (two lists, one set of launches).
// Every G2P wave w stores the ballots of its flagged lanes (mask[l][w]) and the position of its
// lane 0 (wpos[w]). Waves form groups of 64: k_list_sums totals each group; k_list_write (one
// workgroup per group) adds up the totals of the groups before its own, places each wave's
// positions after that offset and the waves before it in the group, and the last group's
// workgroup writes the list lengths.
__global__ __launch_bounds__(256) void k_list_sums(ListArgs a) {
  const int ng = (a.nwaves + 63) / 64;
  const int g = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (g >= ng) return;
  const int w = g * 64 + lane;
  for (int l = 0; l < a.nlists; ++l) {
    int c = w < a.nwaves ? __popcll(a.mask[l][w]) : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if (lane == 0) a.gsum[l * ng + g] = c;
  }
}

__global__ __launch_bounds__(256) void k_list_write(ListArgs a) {
  __shared__ uint64_t s_m[2][64];
  __shared__ int s_off[2][64], s_p[64], s_red[2][4];
  const int ng = (a.nwaves + 63) / 64;
  const int g = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int w = g * 64 + lane;
  // each list's offset of this group: the totals of the groups before it, summed by the workgroup
  // itself (integer sums, so the order does not matter)
  for (int l = 0; l < a.nlists; ++l) {
    int sum = 0;
    for (int i = t; i < g; i += 256) sum += a.gsum[l * ng + i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == 0) s_red[l][wv] = sum;
  }
  __syncthreads();
  if (wv < a.nlists) {  // wave l: the offsets of list l's 64 masks of the group
    const int pre = s_red[wv][0] + s_red[wv][1] + s_red[wv][2] + s_red[wv][3];
    const uint64_t m = w < a.nwaves ? a.mask[wv][w] : 0ull;
    const int c = __popcll(m);
    int x = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off);
      if (lane >= off) x += y;
    }
    s_m[wv][lane] = m;
    s_off[wv][lane] = pre + x - c;
    // the last group's workgroup writes the list's length
    if (g == ng - 1 && lane == 63) *a.count[wv] = pre + x;
  } else if (wv == 3) {
    s_p[lane] = w < a.nwaves ? a.wpos[w] : 0;
  }
  __syncthreads();
  // wave wv writes the positions of masks 16 wv .. 16 wv + 15 of each list, one mask at a time
  for (int l = 0; l < a.nlists; ++l)
    for (int i = 16 * wv; i < 16 * wv + 16; ++i) {
      const uint64_t mi = s_m[l][i];
      if ((mi >> lane) & 1ull) {
        const int rank = __popcll(mi & ((1ull << lane) - 1ull));
        a.list[l][s_off[l][i] + rank] = s_p[i] + lane;
        a.idx[l][s_off[l][i] + rank] = s_p[i] + rank;
      }
    }
}

// ================================================================== surrogate return map
// Cone-branch particles deferred by k_g2p (sur_mode 2) are finished by k_surrogate. Each wave takes
// 64 listed candidates, one per lane, evaluates the MLP for them with BF16 MFMA (weights staged once
// per workgroup in LDS, activations in registers) and then gates each prediction H = eps + 1e-3 y
// of the projected Hencky strains:
//   yield equality   | |dev H| + c alpha tr H | <= tol       (c = (3 lambda + 2 mu) / (2 mu))
//   volume           | tr H - tr eps | <= tol                (the cone return is deviatoric)
//   flow direction   the deviatoric correction eps - H is parallel to dev eps (orthogonal part <= tol)
//                    and points along it
// An accepted prediction gives Sigma' = exp(H), dq = |eps - H|; a rejected one runs the exact
// projection (HybridSolver.cpp:646-673) through the same code as k_g2p, so rejecting every
// prediction reproduces the exact path bit for bit. With a decision log, candidate row r < dec_cap
// records (slot bits, eps, phi, K/mu, H, accepted) at dec_log[10 r ..].
// The gate and the update of a wave's candidates follow its network evaluation in the same kernel:
// their loads and stores (the trial SVD, the new F, q and stress) overlap the other waves' network
// arithmetic, which is bound by the SiLU's transcendentals, instead of taking a pass of their own.

// Gate and state update of candidate `row` at sorted slot j (S, U, V: its trial SVD, eps = log S,
// y: the network's outputs, vol: its volume). Returns whether the prediction was accepted.
__device__ __forceinline__ bool surrogate_update(const SurrogateArgs& a, int row, int j, const DevParams& P,
                                                 const float S[3], const float eps[3], const float y[3], float q,
                                                 float phi_p, float phi, float kmu, const float U[9], const float V[9],
                                                 float vol) {
#pragma clang fp contract(off)
  const int64_t cap = a.cap;
  const float c_yield = (3.0f * P.lambda0 + 2.0f * P.mu0) / (2.0f * P.mu0);
  float H[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) H[k] = eps[k] + MLP_CORR_SCALE * y[k];
  const float fa = phi * 3.14159265358979323846f / 180.0f;
  const float sf = sinf(fa);
  const float alpha = sqrtf(2.0f / 3.0f) * 2.0f * sf / (3.0f - sf);
  const float trH = H[0] + H[1] + H[2], trE = eps[0] + eps[1] + eps[2];
  float dH[3], dE[3], d[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    dH[k] = H[k] - trH / 3.0f;
    dE[k] = eps[k] - trE / 3.0f;
  }
  const float nH = sqrtf(dH[0] * dH[0] + dH[1] * dH[1] + dH[2] * dH[2]);
  const float nE = sqrtf(dE[0] * dE[0] + dE[1] * dE[1] + dE[2] * dE[2]);
#pragma unroll
  for (int k = 0; k < 3; ++k) d[k] = dE[k] - dH[k];  // deviatoric part of eps - H
  const float along = (d[0] * dE[0] + d[1] * dE[1] + d[2] * dE[2]) / nE;
  float ortho2 = 0.0f;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float o = d[k] - along * dE[k] / nE;
    ortho2 += o * o;
  }
  const float tol = a.gate_tol;
  const bool accepted = fabsf(nH + c_yield * alpha * trH) <= tol && fabsf(trH - trE) <= tol && along > 0.0f &&
                        sqrtf(ortho2) <= tol;
  if (a.dec_log && row < a.dec_cap) {
    float* rec = a.dec_log + (int64_t)10 * row;
    rec[0] = __int_as_float(j);
    rec[1] = eps[0];
    rec[2] = eps[1];
    rec[3] = eps[2];
    rec[4] = phi;
    rec[5] = kmu;
    rec[6] = H[0];
    rec[7] = H[1];
    rec[8] = H[2];
    rec[9] = accepted ? 1.0f : 0.0f;
  }
  float Sn[3], lnSn[3], dq;
  if (accepted) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      Sn[k] = expf(H[k]);
      lnSn[k] = H[k];
    }
    dq = sqrtf((eps[0] - H[0]) * (eps[0] - H[0]) + (eps[1] - H[1]) * (eps[1] - H[1]) + (eps[2] - H[2]) * (eps[2] - H[2]));
  } else {
    const float phi0 = P.per_particle_phi ? phi_p : P.h0;
    float lnS[3];
    sand_project(P, phi0, q, S, Sn, lnS, lnSn, dq);
  }
  float Fe[9], K[6];
  sand_finish(P, U, V, Sn, lnSn, dq, q, vol, Fe, K);
#pragma unroll
  for (int k = 0; k < 9; ++k) a.st[(PF + k) * cap + j] = Fe[k];
  a.st[PPL * cap + j] = q;
  if (a.write_stress) {
#pragma unroll
    for (int e = 0; e < 6; ++e) a.st[(PK + e) * cap + j] = K[e];
  }
  return accepted;
}

__global__ __launch_bounds__(MLP_FWD_THREADS) void k_surrogate(SurrogateArgs a) {
  if (clock_skip(a.clk)) return;
  extern __shared__ __align__(16) unsigned char smem[];
  MLPShared& sh = *reinterpret_cast<MLPShared*>(smem);
  // the counter is cleared by the sort stage; a G2P stage repeated without it cannot list more than n
  const int count = min(*a.cand_count, a.n);
  if (blockIdx.x == 0 && threadIdx.x == 0 && count > 0) atomicAdd(a.candidates, (unsigned long long)count);
  const int nw = blockDim.x >> 6;
  // uniform per workgroup: nothing to do, skip the weight staging
  if ((int64_t)blockIdx.x * nw * 64 >= count) return;
  stage_weights(sh, a.wbf, a.master);
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t cap = a.cap, n = a.n;
  unsigned n_acc = 0;
  for (int g = blockIdx.x * nw + w; (int64_t)g * 64 < count; g += gridDim.x * nw) {
    const int row = g * 64 + lane;
    float S[3] = {1.0f, 1.0f, 1.0f}, eps[3] = {0.0f, 0.0f, 0.0f}, phi = 0.0f, kmu = 0.0f, q = 0.0f, phi_p = 0.0f;
    int j = 0, sc = 0;
    float U[9], V[9], vol = 0.0f;
#pragma unroll
    for (int k = 0; k < 9; ++k) U[k] = V[k] = 0.0f;
    if (row < count) {
      j = clamp_index(a.cand_slot[row], (int)n);
      const int r = clamp_index(a.cand_idx[row], (int)n);
      sc = scene_of(a.T.part_off, a.T.nscenes, j);
      const DevParams& P = a.T.params[sc];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        S[k] = a.cand[(CAND_SIGMA + k) * n + r];
        eps[k] = logf(S[k]);
      }
      q = a.st[PPL * cap + j];
      phi_p = a.st[PPHI * cap + j];
      phi = dp_phi(P, phi_p, q);
      kmu = bulk_over_shear(P);
      // what the update needs after the network: these loads complete under its arithmetic
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        U[k] = a.cand[(CAND_U + k) * n + r];
        V[k] = a.cand[(CAND_V + k) * n + r];
      }
      vol = a.st[PVOL * cap + j];
    }
    const float x[5] = {eps[0], eps[1], eps[2], phi, kmu};
    float y[3];
    wave_forward64<MLP_FWD_TILES>(sh, x, y, nullptr, 0, 0);
    // the network's registers are free from here on: keep the update's loads below this point
    __builtin_amdgcn_sched_barrier(0);
    bool accepted = false;
    if (row < count)
      accepted = surrogate_update(a, row, j, a.T.params[sc], S, eps, y, q, phi_p, phi, kmu, U, V, vol);
    n_acc += (unsigned)__popcll(__ballot(accepted));
    __builtin_amdgcn_sched_barrier(0);
  }
  // one atomic per wave
  if (lane == 0 && n_acc) atomicAdd(a.accepted, (unsigned long long)n_acc);
}

// ================================================================== cloth
// Element forces from the current directions (per element), then each vertex sums the forces of
// its incident elements in ascending element order (deterministic).
__device__ __forceinline__ void element_forces(const ClothArgs& a, int e, const float* D, float vol, int& fb) {
  float fv[9], M[9];
  cloth_element_forces(a.P, D, a.rest + 9 * (size_t)e, vol, fv, M, fb);
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    a.elem_fv[9 * (size_t)e + i] = fv[i];
    a.elem_stress[9 * (size_t)e + i] = M[i];
  }
}
// The element forces of directions that no substep has advanced; else k_cloth_elements has formed them.
__global__ __launch_bounds__(256) void k_cloth_element_forces(ClothArgs a) {
  if (clock_skip(a.clk)) return;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  int fb = 0;
  if (e < a.ne) {
    const DevParams& P = a.P;
    const int pi = clamp_index(a.pos[P.mesh_e0 + e], a.n);
    float D[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) D[i] = a.st[(PF + i) * a.cap + pi];
    element_forces(a, e, D, a.st[PVOL * a.cap + pi], fb);
  }
  if (fb) atomicAdd(a.fallback, (unsigned long long)fb);
}

// The rest in-plane QR factor of each element, from its undeformed directions (set-up only).
__global__ __launch_bounds__(256) void k_cloth_rest(ClothArgs a, float* __restrict__ rest) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.ne) return;
  const int pi = clamp_index(a.pos[a.P.mesh_e0 + e], a.n);
  float D[9], Q[9], R[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) D[i] = a.st[(PF + i) * a.cap + pi];
  int fb = 0;
  qr3_guarded(D, Q, R, a.P.svd_ratio, fb);
  rest[9 * (size_t)e + 6] = R[0];
  rest[9 * (size_t)e + 7] = R[1];
  rest[9 * (size_t)e + 8] = R[4];
}

__global__ __launch_bounds__(256) void k_cloth_vertex_forces(ClothArgs a) {
  if (clock_skip(a.clk)) return;
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v == 0 && *a.fallback_next) {  // the element forces are used now
    *a.fallback += *a.fallback_next;
    *a.fallback_next = 0;
  }
  if (v >= a.nv) return;
  float f[3] = {0.0f, 0.0f, 0.0f};
  for (int k = a.vcsr_off[v]; k < a.vcsr_off[v + 1]; ++k) {
    const int ent = a.vcsr[k];  // 3 e + corner
    const int e = ent / 3, c = ent - 3 * e;
    if (e < 0 || e >= a.ne) continue;
#pragma unroll
    for (int r = 0; r < 3; ++r) f[r] += a.elem_fv[9 * (size_t)e + 3 * c + r];
  }
#pragma unroll
  for (int r = 0; r < 3; ++r) a.vert_force[3 * (size_t)v + r] = f[r];
}

// Fixed vertices (HybridSolver.cpp:513-550): for every in-grid node with positive weight for a fixed
// vertex, the 27 nodes (i, j, k) around it are stopped (v = v_BF = 0) through their linear index
// k r0 r1 + j r0 + i, which is checked against [0, gridNumber) only (:536-539). The union of those
// neighbourhoods is the stencil box widened by one node per axis; a neighbour one step outside the
// grid in x or y therefore stops the node its linear index names, e.g. (-1, j, k) stops
// (r0 - 1, j - 1, k), as in the reference.
template <int ORDER>
__global__ __launch_bounds__(64) void k_cloth_fixed(ClothArgs a) {
  if (clock_skip(a.clk)) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.nfixed) return;
  const DevParams& P = a.P;
  const int pi = clamp_index(a.pos[clamp_index(a.fixed[k], a.n)], a.n);
  int lo[3], hi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float g = (a.st[(PX + d) * a.cap + pi] - P.gmin[d]) * P.inv_h[d];
    const int base = stencil_base<ORDER>(g, P.res[d]);
    lo[d] = base + ORDER + 1;
    hi[d] = base - 1;
    for (int o = 0; o <= ORDER; ++o) {
      float w, dw;
      spline<ORDER>(g - (float)(base + o), w, dw);
      if (w > 0.0f) {
        lo[d] = min(lo[d], base + o);
        hi[d] = max(hi[d], base + o);
      }
    }
    // the weight matrix holds in-grid nodes only (HybridSolver.cpp:44-47)
    lo[d] = max(lo[d], 0);
    hi[d] = min(hi[d], P.res[d] - 1);
  }
  if (lo[0] > hi[0] || lo[1] > hi[1] || lo[2] > hi[2]) return;
  const int64_t ng = (int64_t)P.res[0] * P.res[1] * P.res[2];
  const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int n2 = lo[2] - 1; n2 <= hi[2] + 1; ++n2)
    for (int n1 = lo[1] - 1; n1 <= hi[1] + 1; ++n1)
      for (int n0 = lo[0] - 1; n0 <= hi[0] + 1; ++n0) {
        const int64_t node = ((int64_t)n2 * P.res[1] + n1) * P.res[0] + n0;
        if (node < 0 || node >= ng) continue;
        a.gvel[2 * node] = z;
        a.gvel[2 * node + 1] = z;
      }
}

// After G2P: element position = centroid and velocity = mean of its vertices' new values
// (LagrangianMesh::updateElementPositions, HybridSolver.cpp:750-756), d1 = x2 - x1, d2 = x3 - x1
// (:584-590), d3 as updated by G2P, then the return mapping; the element's next key.
__global__ __launch_bounds__(256) void k_cloth_elements(ClothArgs a) {
  if (clock_skip(a.clk)) return;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  int fb = 0, fb_next = 0, oob = 0;
  const DevParams& P = a.P;
  const CellThr thr = cell_thr(a.thr, P.res);
  if (e < a.ne) {
    const int id = P.mesh_e0 + e;
    // the element's and its vertices' slots, then all of their data in one round of loads
    const int pe = clamp_index(a.pos[id], a.n);
    int pv[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) pv[c] = clamp_index(a.pos[clamp_index(a.faces[3 * e + c], a.n)], a.n);
    float xv[3][3], vv[3][3], d3[3];
    const float vol = a.st[PVOL * a.cap + pe];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      d3[d] = a.st[(PF + 3 * d + 2) * a.cap + pe];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        xv[c][d] = a.st[(PX + d) * a.cap + pv[c]];
        vv[c][d] = a.st[(PV + d) * a.cap + pv[c]];
      }
    }
    float D[9], xe[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      xe[d] = (xv[0][d] + xv[1][d] + xv[2][d]) / 3.0f;
      a.st[(PX + d) * a.cap + pe] = xe[d];
      a.st[(PV + d) * a.cap + pe] = (vv[0][d] + vv[1][d] + vv[2][d]) / 3.0f;
      D[3 * d] = xv[1][d] - xv[0][d];
      D[3 * d + 1] = xv[2][d] - xv[0][d];
      D[3 * d + 2] = d3[d];
    }
    cloth_return_map(P, D, fb);
#pragma unroll
    for (int i = 0; i < 9; ++i) a.st[(PF + i) * a.cap + pe] = D[i];
    // the forces that the next P2G scatters, from D while it is at hand (a lookup, ten scattered loads and a launch
    // fewer: 30 substeps of 0.69 M entries with a 256 x 256-vertex cloth 8.27 -> 7.93 ms)
    element_forces(a, e, D, vol, fb_next);
    int cell[3];
    const uint32_t key = cell_key(P, thr, xe[0], xe[1], xe[2], oob, cell);
    const CountTicket ticket = count_wave(a.bins, true, key, tile_of(P, cell[0], cell[1], cell[2]));
    a.keys[pe] = key;
    a.bins.rank[pe] = count_rank(ticket);
  }
  if (fb) atomicAdd(a.fallback, (unsigned long long)fb);
  if (fb_next) atomicAdd(a.fallback_next, (unsigned long long)fb_next);
  if (oob) atomicOr(a.status, MPM_STATUS_OUT_OF_DOMAIN);
}

// ================================================================== auxiliary kernels
// rho_p = sum_i w_ip m_i / h^3, V_p = m_p / rho_p (HybridSolver.cpp:242-249), at the current positions.
template <int ORDER>
__global__ __launch_bounds__(256) void k_volumes(SceneTable T, float* __restrict__ st, int64_t cap, int n,
                                                 const float* __restrict__ gm_all) {
  const PBlock pb = particle_block(T);
  const int i = pb.j;
  if (i >= pb.end) return;
  const DevParams& P = T.params[pb.s];
  const float* gm = gm_all + T.node_off[pb.s];
  // particles only: a cloth's vertices and elements keep their mesh volumes (HybridSolver.cpp:242-249)
  if (particle_kind(P, reinterpret_cast<const int*>(st + (size_t)PID * cap)[i]) != KIND_PARTICLE) return;
  float g[3];
  int base[3];
  float w[3][4], dw[3][4];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    g[d] = (st[(PX + d) * cap + i] - P.gmin[d]) * P.inv_h[d];
    base[d] = stencil_base<ORDER>(g[d], P.res[d]);
#pragma unroll
    for (int o = 0; o < ORDER + 1; ++o) spline<ORDER>(g[d] - (float)(base[d] + o), w[d][o], dw[d][o]);
  }
  float rho = 0.0f;
  for (int oz = 0; oz < ORDER + 1; ++oz)
    for (int oy = 0; oy < ORDER + 1; ++oy)
      for (int ox = 0; ox < ORDER + 1; ++ox) {
        int n0 = base[0] + ox, n1 = base[1] + oy, n2 = base[2] + oz;
        if (n0 < 0 || n1 < 0 || n2 < 0 || n0 >= P.res[0] || n1 >= P.res[1] || n2 >= P.res[2]) continue;
        rho += w[0][ox] * w[1][oy] * w[2][oz] * gm[((int64_t)n2 * P.res[1] + n1) * P.res[0] + n0];
      }
  rho /= P.h[0] * P.h[1] * P.h[2];
  st[PVOL * cap + i] = st[PM * cap + i] / rho;
}

// Copy planes [p0, p0+np) of the device order into caller order (out[plane][id] = st[plane][i]).
__global__ __launch_bounds__(256) void k_unpermute(const float* __restrict__ st, int64_t cap, int n, int p0, int np,
                                                   float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int id = reinterpret_cast<const int*>(st + (size_t)PID * cap)[i];
  if (id < 0 || id >= n) return;
  for (int p = 0; p < np; ++p) out[(size_t)p * n + id] = st[(p0 + p) * cap + i];
}

// Inverse of k_unpermute: planes [p0, p0+np) of the device order from caller order
// (st[plane][pos[id]] = in[plane][id]).
__global__ __launch_bounds__(256) void k_permute_in(float* __restrict__ st, int64_t cap, int n, int p0, int np,
                                                    const float* __restrict__ in, const int* __restrict__ pos) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n) return;
  const int i = pos[id];
  if (i < 0 || i >= n) return;
  for (int p = 0; p < np; ++p) st[(p0 + p) * cap + i] = in[(size_t)p * n + id];
}

// Dense planar copy of one grid quantity (0 = m, 1 = momentum, 2 = v, 3 = v_BF), with nodes
// outside the active blocks set to zero.
__global__ __launch_bounds__(256) void k_grid_export(SceneTable T, const float* __restrict__ grid, int64_t ng, int which,
                                                     const int* __restrict__ block_slot, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ng) return;
  const int sc = scene_of(T.node_off, T.nscenes, i);
  const DevParams& P = T.params[sc];
  const int64_t li = i - T.node_off[sc];
  const int n0 = (int)(li % P.res[0]), n1 = (int)((li / P.res[0]) % P.res[1]), n2 = (int)(li / ((int64_t)P.res[0] * P.res[1]));
  const int b = T.tile_off[sc] + ((n2 >> 2) * P.tiles[1] + (n1 >> 2)) * P.tiles[0] + (n0 >> 2);
  const bool on = block_slot[b] >= 0;
  if (which == 0) {
    out[i] = on ? grid[GRID_M * ng + i] : 0.0f;
  } else if (which == 1) {
    for (int d = 0; d < 3; ++d) out[d * ng + i] = on ? grid[(GRID_MOM + d) * ng + i] : 0.0f;
  } else {
    const float* vel = grid + GRID_VEL * ng + 8 * i;
    for (int d = 0; d < 3; ++d) out[d * ng + i] = on ? vel[which == 2 ? d : 3 + d] : 0.0f;
  }
}

__global__ __launch_bounds__(256) void k_iota(int* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

// Number of nodes with m > 0 in the active blocks.
__global__ __launch_bounds__(64) void k_count_nodes(SceneTable T, const float* __restrict__ gm, const int* __restrict__ counters,
                                                    const int* __restrict__ active_blocks, unsigned long long* __restrict__ out) {
  const int nblk = counters[CNT_BLOCKS];
  const int lx = threadIdx.x & 3, ly = (threadIdx.x >> 2) & 3, lz = threadIdx.x >> 4;
  unsigned long long c = 0;
  for (int s = blockIdx.x; s < nblk; s += gridDim.x) {
    const int gblk = active_blocks[s];
    const int sc = scene_of(T.tile_off, T.nscenes, gblk);
    const DevParams& P = T.params[sc];
    const int blk = gblk - T.tile_off[sc];
    const int b0 = blk % P.tiles[0], b1 = (blk / P.tiles[0]) % P.tiles[1], b2 = blk / (P.tiles[0] * P.tiles[1]);
    const int n0 = 4 * b0 + lx, n1 = 4 * b1 + ly, n2 = 4 * b2 + lz;
    if (n0 >= P.res[0] || n1 >= P.res[1] || n2 >= P.res[2]) continue;
    if (gm[T.node_off[sc] + ((int64_t)n2 * P.res[1] + n1) * P.res[0] + n0] > 0.0f) ++c;
  }
  if (c) atomicAdd(out, c);
}

// Plain copy (measurement reference for the PMC byte counters).
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, int64_t n4) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

__global__ __launch_bounds__(256) void k_fill_int(int* __restrict__ p, int64_t n, int v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ================================================================== launchers
static inline int blocks_for(int64_t n, int t) { return (int)((n + t - 1) / t); }

void launch_pos_of_ids(hipStream_t s, const int* pid, int n, int* pos) {
  if (n > 0) hipLaunchKernelGGL(k_caller_keys, dim3(blocks_for(n, 256)), dim3(256), 0, s, nullptr, pid, n, nullptr, pos, nullptr);
}

void launch_keys(hipStream_t s, const SceneTable& T, int nblocks, const float* st, int64_t cap, int n,
                 const float* thr, uint32_t* keys, int* status) {
  if (n > 0) hipLaunchKernelGGL(k_keys, dim3(nblocks), dim3(256), 0, s, T, st, cap, n, thr, keys, status);
}

void launch_stress_init(hipStream_t s, const SceneTable& T, int nblocks, float* st, int64_t cap, int n,
                        unsigned long long* fallback) {
  if (n > 0) hipLaunchKernelGGL(k_stress_init, dim3(nblocks), dim3(256), 0, s, T, st, cap, n, fallback);
}

void launch_count_tiles(hipStream_t s, const SceneTable& T, int nblocks, const float* st, int64_t cap, const float* thr,
                        uint8_t* flag, int64_t ntiles, int* count) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(k_flag_tiles, dim3(nblocks), dim3(256), 0, s, T, st, cap, thr, flag);
  hipLaunchKernelGGL(k_sum_flags, dim3(std::min(1024, blocks_for(ntiles, 256))), dim3(256), 0, s, flag, ntiles, count);
}

void launch_count(hipStream_t s, const SceneTable& T, const BinCounts& b, const uint32_t* keys, int n, int64_t ncells,
                  int64_t ntiles, int* counters, bool dirty) {
  const int64_t nscan = blocks_for(ncells, SCAN_TILE), work = dirty ? ncells : std::max(nscan, ntiles);
  hipLaunchKernelGGL(k_clear_counts, dim3(std::min(4096, blocks_for(work, 256))), dim3(256), 0, s, b, nscan, ntiles,
                     dirty ? ncells : 0, counters);
  if (n > 0) hipLaunchKernelGGL(k_cell_count, dim3(blocks_for(n, 256)), dim3(256), 0, s, T, b, keys, n);
}

void launch_sort(hipStream_t s, const SortBufs& b, const uint32_t* keys_in, int n, int nblocks, int passes, int mode) {
  if (n <= 0) return;
  const int nscan = blocks_for(b.ncells, SCAN_TILE);
  const dim3 first(nscan + blocks_for(b.ntiles, 256));
  if (nscan <= SMALL_SCAN) {
    hipLaunchKernelGGL(k_sums_claim<true>, first, dim3(256), 0, s, b, nscan);
  } else {
    hipLaunchKernelGGL(k_sums_claim<false>, first, dim3(256), 0, s, b, nscan);
    hipLaunchKernelGGL(k_cell_scan, dim3(nscan), dim3(256), 0, s, b);
  }
  if (mode == SORT_COUNTING) {
    uint32_t* kf = (passes & 1) ? b.k1 : b.k2;  // the result goes where the digit passes put it
    int* vf = (passes & 1) ? b.v1 : b.v2;
    int* tmp = (passes & 1) ? b.v2 : b.v1;
    hipLaunchKernelGGL(k_cell_scatter, dim3(blocks_for(n, 256)), dim3(256), 0, s, keys_in, b.bins.rank, n, b.cell_start,
                       b.pid, tmp, b.tslot, kf, b.clk);
    hipLaunchKernelGGL(k_cell_rank, dim3(blocks_for(n, 256)), dim3(256), 0, s, kf, tmp, b.tslot, n, b.cell_start, vf,
                       b.bins.cell_count, b.src, b.clk);
    return;
  }
  hipLaunchKernelGGL(k_reset, dim3(std::min(4096, blocks_for(b.radix_words, 256))), dim3(256), 0, s, b.hist,
                     b.radix_words, b.clk);
  // the digit passes are stable in their input order, which must be the caller order: the keys
  // (by physical slot) go to caller order first, and the caller id -> slot map comes with them
  uint32_t* kc = reinterpret_cast<uint32_t*>(b.tslot);
  hipLaunchKernelGGL(k_caller_keys, dim3(blocks_for(n, 256)), dim3(256), 0, s, keys_in, b.pid, n, kc, b.pos, b.clk);
  const int nb = blocks_for(n, SORT_TILE);
  hipLaunchKernelGGL(k_sort_hist, dim3(blocks_for(n, HIST_TILE)), dim3(256), 0, s, kc, n, passes, b.hist, b.clk);
  const uint32_t* kin = kc;
  const int* vin = nullptr;
  for (int p = 0; p < passes; ++p) {
    uint32_t* ko = (p & 1) ? b.k2 : b.k1;
    int* vo = (p & 1) ? b.v2 : b.v1;
    hipLaunchKernelGGL(k_sort_pass, dim3(nb), dim3(256), 0, s, kin, vin, ko, vo, n, p, b.hist, b.tickets,
                       b.status + (size_t)p * nb * 256, b.clk);
    kin = ko;
    vin = vo;
  }
  hipLaunchKernelGGL(k_bounds, dim3(nblocks), dim3(256), 0, s, b.T, kin, n, b.bins.cell_count, vin, b.pos, b.src, b.clk);
}

void launch_fill_bins(hipStream_t s, const uint32_t* ks, int n, int64_t ncells, int* cell_start) {
  if (ncells <= 0) return;
  hipLaunchKernelGGL(k_fill_bins, dim3(blocks_for(ncells + 1, 256)), dim3(256), 0, s, ks, n, ncells, cell_start);
}

template <int RANKS, int WAVES>
static void launch_p2g_r(hipStream_t s, const P2GArgs& a, int order, int mode, int grid) {
  if (mode == P2G_MOM_STRESS) {
    if (order == 2) hipLaunchKernelGGL((k_p2g<2, P2G_MOM_STRESS, RANKS, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, a);
    else hipLaunchKernelGGL((k_p2g<3, P2G_MOM_STRESS, RANKS, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, a);
  } else if (mode == P2G_MOM) {
    if (order == 2) hipLaunchKernelGGL((k_p2g<2, P2G_MOM, RANKS, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, a);
    else hipLaunchKernelGGL((k_p2g<3, P2G_MOM, RANKS, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, a);
  } else {
    if (order == 2) hipLaunchKernelGGL((k_p2g<2, P2G_FORCE, RANKS, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, a);
    else hipLaunchKernelGGL((k_p2g<3, P2G_FORCE, RANKS, WAVES>), dim3(grid), dim3(64 * WAVES), 0, s, a);
  }
}

template <int RANKS>
static void launch_p2g_l(hipStream_t s, const P2GArgs& a, int order, int mode, int grid) {
  if (mode == P2G_MOM_STRESS) {
    if (order == 2) hipLaunchKernelGGL((k_p2g_layer<2, P2G_MOM_STRESS, RANKS>), dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_p2g_layer<3, P2G_MOM_STRESS, RANKS>), dim3(grid), dim3(256), 0, s, a);
  } else if (mode == P2G_MOM) {
    if (order == 2) hipLaunchKernelGGL((k_p2g_layer<2, P2G_MOM, RANKS>), dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_p2g_layer<3, P2G_MOM, RANKS>), dim3(grid), dim3(256), 0, s, a);
  } else {
    if (order == 2) hipLaunchKernelGGL((k_p2g_layer<2, P2G_FORCE, RANKS>), dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_p2g_layer<3, P2G_FORCE, RANKS>), dim3(grid), dim3(256), 0, s, a);
  }
}

void launch_p2g(hipStream_t s, const P2GArgs& a, int order, int mode, int grid, int ranks, int pass) {
  if (pass == P2G_LAYERS) {
    if (ranks == 2) launch_p2g_l<2>(s, a, order, mode, grid);
    else launch_p2g_l<4>(s, a, order, mode, grid);
  } else if (pass == P2G_WIDE_ROWS) {
    launch_p2g_r<8, 16>(s, a, order, mode, grid);
  } else {
    if (ranks == 4) launch_p2g_r<4, 8>(s, a, order, mode, grid);
    else launch_p2g_r<8, 8>(s, a, order, mode, grid);
  }
}

void launch_stress_predicted(hipStream_t s, const P2GArgs& a, int order, int nblocks) {
  if (a.n <= 0) return;
  if (order == 2) hipLaunchKernelGGL(k_stress_predicted<2>, dim3(nblocks), dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_stress_predicted<3>, dim3(nblocks), dim3(256), 0, s, a);
}

void launch_clock_init(hipStream_t s, Clock* c) { hipLaunchKernelGGL(k_clock_init, dim3(1), dim3(64), 0, s, c); }

void launch_clock_end(hipStream_t s, Clock* c, const int* tiles) {
  hipLaunchKernelGGL(k_clock_end, dim3(1), dim3(64), 0, s, c, tiles);
}

void launch_grid(hipStream_t s, const GridArgs& a, int mode, int grid) {
  if (mode == GRID_FUSED) hipLaunchKernelGGL(k_grid<GRID_FUSED>, dim3(grid), dim3(64), 0, s, a);
  else if (mode == GRID_NORMALIZE) hipLaunchKernelGGL(k_grid<GRID_NORMALIZE>, dim3(grid), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_grid<GRID_FORCE_UPDATE>, dim3(grid), dim3(64), 0, s, a);
}

void launch_g2p(hipStream_t s, const G2PArgs& a, int order, int nblocks, hipEvent_t ev_start, hipEvent_t ev_stop) {
  if (a.n <= 0) return;
  if (ev_start) {  // timed launch: the events take the dispatch's own start and end times
    if (order == 2) hipExtLaunchKernelGGL(k_g2p<2>, dim3(nblocks), dim3(256), 0, s, ev_start, ev_stop, 0, a);
    else hipExtLaunchKernelGGL(k_g2p<3>, dim3(nblocks), dim3(256), 0, s, ev_start, ev_stop, 0, a);
    return;
  }
  if (order == 2) hipLaunchKernelGGL(k_g2p<2>, dim3(nblocks), dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_g2p<3>, dim3(nblocks), dim3(256), 0, s, a);
}

void launch_volumes(hipStream_t s, const SceneTable& T, int order, int nblocks, float* st, int64_t cap, int n,
                    const float* gm) {
  if (n <= 0) return;
  if (order == 2) hipLaunchKernelGGL(k_volumes<2>, dim3(nblocks), dim3(256), 0, s, T, st, cap, n, gm);
  else hipLaunchKernelGGL(k_volumes<3>, dim3(nblocks), dim3(256), 0, s, T, st, cap, n, gm);
}

void launch_unpermute(hipStream_t s, const float* st, int64_t cap, int n, int p0, int np, float* out) {
  if (n > 0) hipLaunchKernelGGL(k_unpermute, dim3(blocks_for(n, 256)), dim3(256), 0, s, st, cap, n, p0, np, out);
}

void launch_permute_in(hipStream_t s, float* st, int64_t cap, int n, int p0, int np, const float* in, const int* pos) {
  if (n > 0) hipLaunchKernelGGL(k_permute_in, dim3(blocks_for(n, 256)), dim3(256), 0, s, st, cap, n, p0, np, in, pos);
}

void launch_grid_export(hipStream_t s, const SceneTable& T, const float* grid, int64_t ng, int which, const int* block_slot,
                        float* out) {
  hipLaunchKernelGGL(k_grid_export, dim3(blocks_for(ng, 256)), dim3(256), 0, s, T, grid, ng, which, block_slot, out);
}

void launch_iota(hipStream_t s, int* p, int n) {
  if (n > 0) hipLaunchKernelGGL(k_iota, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, n);
}

void launch_count_nodes(hipStream_t s, const SceneTable& T, const float* gm, const int* counters, const int* active_blocks,
                        unsigned long long* out, int grid) {
  hipLaunchKernelGGL(k_count_nodes, dim3(grid), dim3(64), 0, s, T, gm, counters, active_blocks, out);
}

void launch_copy(hipStream_t s, const float4* src, float4* dst, int64_t n4) {
  int grid = blocks_for(n4, 256);
  if (grid > 8192) grid = 8192;
  if (n4 > 0) hipLaunchKernelGGL(k_copy, dim3(grid), dim3(256), 0, s, src, dst, n4);
}

static size_t surrogate_smem() { return sizeof(MLPShared); }

void surrogate_set_smem_limit() {
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_surrogate),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)surrogate_smem());
}

void launch_position_lists(hipStream_t s, const ListArgs& a) {
  if (a.nwaves <= 0 || a.nlists <= 0) return;
  const int ng = (a.nwaves + 63) / 64;
  hipLaunchKernelGGL(k_list_sums, dim3((ng + 3) / 4), dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_list_write, dim3(ng), dim3(256), 0, s, a);
}

void launch_surrogate(hipStream_t s, const SurrogateArgs& a, int n_cu, hipEvent_t* ev) {
  if (ev && ev[0]) {  // a timed launch: the dispatch records its own start and end
    hipExtLaunchKernelGGL(k_surrogate, dim3(n_cu), dim3(MLP_FWD_THREADS), surrogate_smem(), s, ev[0], ev[1], 0, a);
    return;
  }
  hipLaunchKernelGGL(k_surrogate, dim3(n_cu), dim3(MLP_FWD_THREADS), surrogate_smem(), s, a);
}

void launch_apex_finish(hipStream_t s, ApexArgs a, int n_cu) {
  if (a.list) {
    hipLaunchKernelGGL(k_apex_list, dim3(2 * n_cu), dim3(256), 0, s, a);
    return;
  }
  const int small = blocks_for(a.nwaves, 4);
  a.gw = small <= 8 * n_cu ? 4 : APEX_GROUP;
  hipLaunchKernelGGL(k_apex_finish, dim3(a.gw == 4 ? small : std::min(4 * n_cu, blocks_for(a.nwaves, APEX_GROUP))),
                     dim3(256), 0, s, a);
}

void launch_fill_int(hipStream_t s, int* p, int64_t n, int v) {
  if (n > 0) hipLaunchKernelGGL(k_fill_int, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, n, v);
}

void launch_cloth_rest(hipStream_t s, const ClothArgs& a, float* rest) {
  if (a.ne > 0) hipLaunchKernelGGL(k_cloth_rest, dim3(blocks_for(a.ne, 256)), dim3(256), 0, s, a, rest);
}

void launch_cloth_element_forces(hipStream_t s, const ClothArgs& a) {
  if (a.ne > 0) hipLaunchKernelGGL(k_cloth_element_forces, dim3(blocks_for(a.ne, 256)), dim3(256), 0, s, a);
}

void launch_cloth_vertex_forces(hipStream_t s, const ClothArgs& a) {
  if (a.nv > 0) hipLaunchKernelGGL(k_cloth_vertex_forces, dim3(blocks_for(a.nv, 256)), dim3(256), 0, s, a);
}

void launch_cloth_fixed(hipStream_t s, const ClothArgs& a) {
  if (a.nfixed <= 0) return;
  if (a.P.order == 2) hipLaunchKernelGGL(k_cloth_fixed<2>, dim3(blocks_for(a.nfixed, 64)), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_cloth_fixed<3>, dim3(blocks_for(a.nfixed, 64)), dim3(64), 0, s, a);
}

void launch_cloth_elements(hipStream_t s, const ClothArgs& a) {
  if (a.ne > 0) hipLaunchKernelGGL(k_cloth_elements, dim3(blocks_for(a.ne, 256)), dim3(256), 0, s, a);
}

}  // namespace mpm
