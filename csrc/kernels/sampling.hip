// Per-row token sampling over the full vocabulary (V ~ 128k-152k) on gfx950:
// temperature -> top-k -> top-p -> categorical, or argmax when temperature == 0.
//
// Parallel layout: each row is split into NSEG segments, one block of 512 threads (1024 where segments are long) per
// (segment, row), so a batch-8 step spreads its 8 x 600 KB of logits over 192 CUs
// instead of 8. After each pass the blocks of a row exchange tagged partials (sample_gran_kernel:
// NSEG is chosen on the host so that B * NSEG <= 256 blocks, all co-resident, and every wait has a
// give-up bound). With NSEG == 1 (large batches) a row is one block (sample_row_kernel).
//
// Exact sampling, no sort, no histogram atomics:
//   pass 0: per segment (max, Z = sum e^{(x-max)/T}, argmax) and the Gumbel-max draw
//           argmax_i (x_i / T + G_i) — an exact sample of the tempered distribution.
//   Without top-k/top-p the Gumbel winner is the answer (one pass).
//   With them, rejection on the pivot: candidate j is accepted iff
//     #{x_i > x_j} < top_k  and  sum_{x_i > x_j} e_i < top_p * Z
//   (j is inside both prefix sets). Every pass computes those two counts for the
//   current candidate AND, speculatively, the next candidate = Gumbel-max restricted
//   to {x_i > x_j} with fresh noise (if j is rejected, every token <= x_j is outside
//   the nucleus too). So each rejection round costs one parallel pass; accepted
//   samples are distributed exactly as the renormalised filtered distribution.
// RNG: Philox4x32-10 keyed by the per-row seed, counter (float4 index, offset, round),
// so results are reproducible for a given (seed, offset) and independent of NSEG.
// Merges read the segments' partials in a fixed order: bit-reproducible.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "launchers.h"
#include "sampling_common.h"

namespace vgate {

// Lane exchange on the VALU (no LDS round trip per step, unlike __shfl_xor's ds_bpermute): DPP
// quad permutes for partners 1 and 2, row rotations by 4 and 8 (after the quad steps every lane of
// a quad holds the quad's merge, so rotations complete the 16-lane row), permlane swaps for 16 / 32.
template <int K>
__device__ __forceinline__ uint32_t lane_x(uint32_t v) {
  if constexpr (K == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, false);   // quad_perm [1,0,3,2]
  else if constexpr (K == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, false);  // [2,3,0,1]
  else if constexpr (K == 4) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x124, 0xf, 0xf, false);  // row_ror:4
  else if constexpr (K == 8) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, false);  // row_ror:8
  else if constexpr (K == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (threadIdx.x & 16) ? r[0] : r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32) ? r[0] : r[1];
  }
}
// a wave's values under a commutative operation, the same in every lane
template <typename T, typename F>
__device__ __forceinline__ T wave_all(T v, F f) {
  auto other = [](T x, auto k) { return __builtin_bit_cast(T, lane_x<decltype(k)::value>(__builtin_bit_cast(uint32_t, x))); };
  v = f(v, other(v, std::integral_constant<int, 1>{}));
  v = f(v, other(v, std::integral_constant<int, 2>{}));
  v = f(v, other(v, std::integral_constant<int, 4>{}));
  v = f(v, other(v, std::integral_constant<int, 8>{}));
  v = f(v, other(v, std::integral_constant<int, 16>{}));
  v = f(v, other(v, std::integral_constant<int, 32>{}));
  return __builtin_bit_cast(T, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float wave_max(float v) { return wave_all(v, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ float wave_sum(float v) { return wave_all(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ int wave_min(int v) { return wave_all(v, [](int a, int b) { return a < b ? a : b; }); }

using Mode0 = std::integral_constant<int, 0>;
using Mode1 = std::integral_constant<int, 1>;

// The merge of a wave's partials, in every lane. Maxima first, then one rescaling per lane and plain sums: merged pairwise, each of the six
// steps waits for two exponentials (1.2 us a merge and three merges a pass).
template <typename Mode>
__device__ __forceinline__ Acc wave_merge(const Acc& a, float c, Mode) {
  Acc r = acc_init();
  r.gk = wave_max(a.gk);
  r.gi = wave_min(a.gi >= 0 && a.gk == r.gk ? a.gi : 0x7fffffff);  // (equal keys: the lower index)
  const uint64_t at = __ballot(a.gi == r.gi);
  if (at == 0) {
    r.gi = -1;
  } else {
    r.gx = __uint_as_float(__builtin_amdgcn_readlane((int)__float_as_uint(a.gx), __builtin_ctzll(at)));
  }
  if constexpr (Mode::value == 0) {
    r.mx = wave_max(a.mx);
    r.amx = wave_min(a.mx == r.mx ? a.amx : 0x7fffffff);
    r.z = wave_sum(a.mx == r.mx ? a.z : a.mx == -INFINITY ? 0.f : a.z * __builtin_amdgcn_exp2f((a.mx - r.mx) * c));
  } else {
    r.cnt = wave_sum(a.cnt);
    r.q = wave_sum(a.q);
  }
  return r;
}

// The merge of the waves' results that `red` holds, in every lane of the calling wave
template <typename Mode>
__device__ __forceinline__ Acc merge_waves(const Acc* red, int nw, float c, Mode mode) {
  const int lane = threadIdx.x & 63;
  Acc a = red[lane < nw ? lane : 0];
  if (lane >= nw) a = acc_init();
  return wave_merge(a, c, mode);
}

// Block-wide reduction (the first wave holds the result).
template <typename Mode>
__device__ __forceinline__ Acc block_reduce_acc(const Acc& a, float c, Acc* red, Mode mode) {
  __syncthreads();  // `red` may still be read by the first wave from a previous reduction
  const Acc w = wave_merge(a, c, mode);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  __syncthreads();
  return threadIdx.x < 64 ? merge_waves(red, blockDim.x >> 6, c, mode) : w;
}

// Per-row sampling parameters (row-uniform).
struct RowParams {
  float T, c, cn, topp;
  bool greedy, use_k, use_p;
  int topk;
  uint64_t seed, off;
};

__device__ __forceinline__ RowParams row_params(const SampleArgs& a, int row) {
  RowParams r;
  r.T = a.temperature ? a.temperature[row] : 0.f;
  r.greedy = !(r.T > 1e-5f);
  r.c = r.greedy ? LOG2E_S : LOG2E_S / r.T;  // log2-domain scale
  r.cn = r.greedy ? 1.f : 1.f / r.T;         // natural-domain scale (Gumbel keys)
  r.seed = a.seeds ? a.seeds[row] : 0ull;
  r.off = a.offsets ? (uint64_t)a.offsets[row] : 0ull;
  r.topk = a.top_k ? a.top_k[row] : -1;
  r.topp = a.top_p ? a.top_p[row] : 1.f;
  r.use_k = r.topk > 0 && r.topk < a.V;
  r.use_p = r.topp < 1.f;
  return r;
}

// Four logits' contribution to a pass (shared by the memory sweep and the register-resident
// segments, so both produce the same bits): mode 0 (max / Z / argmax + Gumbel key), mode 1
// (count and mass above xj + the key restricted to x > xj). L = logf(fmaxf(-logf(u), 1e-30f)) of
// each logit's uniform for the pass's round (key = v / T - L: a Gumbel draw). The maximum of the four comes first, so that the sum over them
// waits for one rescaling and not for four (the exponents are those of the maximum so far; v == mx counts 1 also where both are infinite).
// (Modes are known when this is compiled: with one that is not, stores into either mode's fields are merged into one through a pointer,
// and the accumulator moves to memory.)
template <int mode>
__device__ __forceinline__ void accum4(const float (&v)[4], int i, const float (&L)[4], float xj, float rmx, const RowParams& rp, Acc& acc) {
  if constexpr (mode == 0) {
    const float m = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
    if (m > acc.mx) {
      // (nothing yet: the exponent may be no number, -inf times the scale 0 of an infinite temperature)
      acc.z = acc.mx == -INFINITY ? 0.f : acc.z * __builtin_amdgcn_exp2f((acc.mx - m) * rp.c);
      acc.mx = m;
      acc.amx = i + (v[0] == m ? 0 : v[1] == m ? 1 : v[2] == m ? 2 : 3);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (mode == 0) {
      acc.z += v[j] > -INFINITY ? (v[j] == acc.mx ? 1.f : __builtin_amdgcn_exp2f((v[j] - acc.mx) * rp.c)) : 0.f;
    } else {
      acc.cnt += v[j] > xj ? 1.f : 0.f;
      acc.q += v[j] > xj ? __builtin_amdgcn_exp2f((v[j] - rmx) * rp.c) : 0.f;
    }
    const float g = v[j] * rp.cn - L[j];
    const bool take = !rp.greedy && (mode == 0 || v[j] > xj) && v[j] > -INFINITY && g > acc.gk;
    acc.gk = take ? g : acc.gk;
    acc.gi = take ? i + j : acc.gi;
    acc.gx = take ? v[j] : acc.gx;
  }
}

// accurate logs: a fast log rounding -log(u) to 0 near u = 1 would make an infinite key
__device__ __forceinline__ float gumbel_log(float u) { return logf(fmaxf(-logf(u), 1e-30f)); }

// One sweep of float4 range [v_lo, v_hi) of a row by this block (8 float4 loads in flight per
// thread). mode 0: max / Z / argmax + Gumbel keys; mode 1: acceptance statistics of candidate
// value xj (count and mass of x > xj, mass relative to the row max rmx) + Gumbel keys restricted
// to x > xj with the noise of `round`.
template <int mode>
__device__ __forceinline__ void sweep_range(const float4* x4, int v_lo, int v_hi, float xj, float rmx,
                                            uint32_t round, const RowParams& rp, Acc& acc) {
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int v0 = v_lo + tid; v0 < v_hi; v0 += nt * 8) {
    // lanes past the range load nothing (a clamped re-read of the last float4 cost a wave load
    // per lane: ~40 % of a 32-segment pass's loads at V = 152k)
    float4 q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int vi = v0 + u * nt;
      q[u] = vi < v_hi ? x4[vi] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int vi = v0 + u * nt;
      if (vi >= v_hi) break;
      const float e[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
      float uu[4] = {0.5f, 0.5f, 0.5f, 0.5f};
      if (!rp.greedy) philox4(rp.seed, rp.off, (uint32_t)vi, round, uu);
      float L[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        L[j] = (!rp.greedy && (mode == 0 || e[j] > xj) && e[j] > -INFINITY) ? gumbel_log(uu[j]) : 0.f;
      accum4<mode>(e, 4 * vi, L, xj, rmx, rp, acc);
    }
  }
}

// The host ring's words past the sampled ids: the sticky fault word, if it is set (the host clears its copies after a recovery), and the
// custom all-reduce's {error, ticks, calls}. What earlier launches of the step raised is final here; a wait of this launch that gives up
// hands its own bit over (fault_to_host).
__device__ __forceinline__ void ring_store(const SampleArgs& a, int at, uint32_t v) {
  __hip_atomic_store(reinterpret_cast<uint32_t*>(a.ring) + (size_t)*a.ring_slot * a.ring_stride + at, v, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void fault_to_host(const SampleArgs& a, uint32_t more) {
  if (a.fault == nullptr || a.ring == nullptr) return;
  const uint32_t f = __hip_atomic_load(a.fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) | more;
  if (f != 0) ring_store(a, a.ring_stride - 1, f);
}

__device__ __forceinline__ void finish_row(const SampleArgs& a, int row, int chosen, float mx, float z, float c) {
  a.out[row] = chosen;
  if (a.ring != nullptr) {
    ring_store(a, row, (uint32_t)chosen);
    fault_to_host(a, 0u);
    if (a.ar != nullptr && row == 0) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        ring_store(a, a.ring_stride - 4 + i, __hip_atomic_load(a.ar + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM));
    }
    drain_stores();
  }
  if (a.out_logprob) a.out_logprob[row] = ((a.logits[(size_t)row * a.ldl + chosen] - mx) * c - log2f(z)) / LOG2E_S;
}

// ---- one block per row (NSEG == 1: batches above SAMPLE_MAX_BLOCKS / 2 rows, or no workspace) ----
// Every pass sweeps the whole row and ends at a block barrier; same passes, noise and acceptance
// tests as the segmented kernel below.
template <int NT>
__global__ __launch_bounds__(NT) void sample_row_kernel(SampleArgs a) {
  TLScope tl_scope(a.tl);
  __shared__ Acc red[NT / 64];
  __shared__ Acc merged;
  const int row = blockIdx.y, tid = threadIdx.x;
  const int V4 = a.V >> 2;  // host guarantees V % 4 == 0 and 16-B aligned rows
  const float* x = a.logits + (size_t)row * a.ldl;
  const float4* x4 = reinterpret_cast<const float4*>(x);
  const RowParams rp = row_params(a, row);
  const float c = rp.c;
  auto pass = [&](auto mode, float xj, float rmx, uint32_t round) {
    Acc acc = acc_init();
    sweep_range<decltype(mode)::value>(x4, 0, V4, xj, rmx, round, rp, acc);
    acc = block_reduce_acc(acc, c, red, mode);
    if (tid == 0) merged = acc;
    __syncthreads();
  };
  pass(Mode0{}, 0.f, 0.f, 0u);
  const float mx = merged.mx, z = merged.z;
  int chosen = merged.amx, j = merged.gi;
  if (!rp.greedy) {
    if (rp.use_k || rp.use_p) {
      const float pmass = rp.topp * z;
      for (uint32_t round = 1; round <= SAMPLE_MAX_ROUNDS && j >= 0; ++round) {
        pass(Mode1{}, merged.gx, mx, round);
        const bool ok_k = !rp.use_k || merged.cnt < (float)rp.topk;
        const bool ok_p = !rp.use_p || merged.q < pmass;
        if (ok_k && ok_p) break;
        j = merged.gi;  // next candidate, drawn from {x > x_j}
      }
    }
    if (j >= 0) chosen = j;
  }
  if (tid == 0) finish_row(a, row, chosen, mx, z, c);
}

// ---- single launch: tagged granules instead of tickets / counters ----
// What a pass takes: the noise, and the merges and meetings, 3 us of them (6.5 before the merges of wave_merge; us, top-p 0.95, rows half
// greedy, before -> now: 8 rows of 32000 21.7 -> 13.2, 32 rows 23.5 -> 15.3, 64 rows 33.8 -> 21.3; greedy, one row 9.7 -> 6.9).
// The pass kernels' meetings cost a launch boundary per pass, the in-launch ones a serialised
// atomic per arriving block (~0.5 us each, 32 per row). Here every block of a row publishes its
// pass partial as two 16-B granules {.., tag} (device-coherent sc1 stores, one transaction each),
// and EVERY block of the row gathers all of the row's granules itself (lane s polls segment s
// until both tags carry this pass's tag), merges them in the same fixed lane order and takes the
// same accept / reject decision — no counter, no merger block, one memory round trip after the
// last partial lands. Tags = (row epoch << 6) | pass: the epoch advances once per launch (one store
// by the row's segment 0 at its exit, see the end of the kernel), so a granule of an earlier launch
// never matches; granules alternate two buffers by pass parity (a block reaches pass g + 2,
// rewriting parity g, only after every block of the row published g + 1, i.e. finished reading g).
// Each row owns a FIXED granule region of SAMPLE_GRAN_SEGS segments whatever the launch's (B, nseg):
// a slot is only ever written by its own row, under that row's monotonic epoch. (A layout that moved
// with nseg let row r read row r' < r's leftovers from a launch of another batch size whose tag
// happened to equal r's current one.)
// Every wait is bounded: a give-up sets fault bit 16 (the engine fails the step) and the row
// falls back to its argmax. B x nseg <= 256 blocks: all co-resident.
template <typename Mode>
__device__ __forceinline__ void gran_publish(uint4* g, const Acc& a, Mode, uint32_t tag) {
  // mode 0 (pass 0): {mx, z, amx}, mode 1 (rounds): {cnt, q}; then {gk, gi, gx}. (Word by word out of the struct: put together as one vector
  // from it, the struct is read as a vector and lives in memory.)
  float p0 = Mode::value == 0 ? +a.mx : +a.cnt, p1 = Mode::value == 0 ? +a.z : +a.q, p2 = __int_as_float(a.amx);
  float k0 = a.gk, k1 = __int_as_float(a.gi), k2 = a.gx;
  asm volatile("" : "+v"(p0), "+v"(p1), "+v"(p2), "+v"(k0), "+v"(k1), "+v"(k2));
  st_sc1_x4(reinterpret_cast<float*>(g), 0u, f32x4{p0, p1, p2, __uint_as_float(tag)});
  st_sc1_x4(reinterpret_cast<float*>(g), 16u, f32x4{k0, k1, k2, __uint_as_float(tag)});
}

// one wave: gather the nseg granule pairs of (row, parity) and merge them, in every lane. Returns false if a wait gave up.
template <typename Mode>
__device__ __forceinline__ bool gran_gather(const SampleArgs& args, const uint4* gbase, int nseg, Mode mode, uint32_t tag, float c,
                                            Acc& out) {
  const int lane = threadIdx.x & 63;
  Acc a = acc_init();
  bool ok = true;
  if (lane < nseg) {
    const float* gp = reinterpret_cast<const float*>(gbase + 2 * lane);
    f32x4 g0, g1;
    uint32_t spins = 0;
    while (true) {
      g0 = ld_sc1_x4(gp, 0u);
      g1 = ld_sc1_x4(gp, 16u);
      if (__float_as_uint(g0[3]) == tag && __float_as_uint(g1[3]) == tag) break;
      if (++spins > (1u << 22)) { ok = false; break; }
      __builtin_amdgcn_s_sleep(1);
    }
    if (ok) {
      if constexpr (Mode::value == 0) {
        a.mx = g0[0];
        a.z = g0[1];
        a.amx = __float_as_int(g0[2]);
      } else {
        a.cnt = g0[0];
        a.q = g0[1];
      }
      a.gk = g1[0]; a.gi = __float_as_int(g1[1]); a.gx = g1[2];
    }
  }
  const bool all_ok = __all(ok);
  if (!all_ok && lane == 0 && args.fault != nullptr) {
    atomicOr(args.fault, 16u);
    fault_to_host(args, 16u);
  }
  out = wave_merge(a, c, mode);
  return all_ok;
}

template <int NT>
__global__ __launch_bounds__(NT) void sample_gran_kernel(SampleArgs a) {
  TLScope tl_scope(a.tl);
  __shared__ Acc red[NT / 64];
  __shared__ Acc merged;
  __shared__ int s_ok;
  const int seg = blockIdx.x, nseg = gridDim.x, row = blockIdx.y, tid = threadIdx.x;
  const int V4 = a.V >> 2;
  const int v_lo = (int)(((long long)V4 * seg) / nseg), v_hi = (int)(((long long)V4 * (seg + 1)) / nseg);
  const float* x = a.logits + (size_t)row * a.ldl;
  const float4* x4 = reinterpret_cast<const float4*>(x);
  const RowParams rp = row_params(a, row);
  const float c = rp.c;
  const uint32_t ep = __builtin_amdgcn_readfirstlane(__float_as_uint(ld_sc1(reinterpret_cast<const float*>(a.epoch + row))));
  uint4* rowg = reinterpret_cast<uint4*>(a.gran) + (size_t)row * SAMPLE_GRAN_ROW;  // [parity][SEGS][2]
  // one pass: sweep, block merge, publish, gather every segment's granules, share the row merge
  auto pass = [&](auto mode, float xj, float rmx, uint32_t round, uint32_t gen) -> bool {
    Acc acc = acc_init();
    sweep_range<decltype(mode)::value>(x4, v_lo, v_hi, xj, rmx, round, rp, acc);
    acc = block_reduce_acc(acc, c, red, mode);
    const uint32_t tag = (ep << 6) | gen;
    uint4* pg = rowg + (size_t)(gen & 1) * SAMPLE_GRAN_SEGS * 2;
    if (tid == 0) {
      gran_publish(pg + 2 * seg, acc, mode, tag);
    }
    if (tid < 64) {
      Acc r;
      const bool ok = gran_gather(a, pg, nseg, mode, tag, c, r);
      if (tid == 0) {
        merged = r;
        s_ok = ok;
      }
    }
    __syncthreads();
    return s_ok != 0;
  };
  uint32_t gen = 1;
  bool ok = pass(Mode0{}, 0.f, 0.f, 0u, gen);
  const float mx = merged.mx, z = merged.z;
  int chosen = merged.amx, j = merged.gi;
  float xj = merged.gx;
  if (ok && !rp.greedy) {
    if (rp.use_k || rp.use_p) {
      const float pmass = rp.topp * z;
      for (uint32_t round = 1; round <= SAMPLE_MAX_ROUNDS && j >= 0; ++round) {
        ok = pass(Mode1{}, xj, mx, round, ++gen);
        if (!ok) { j = -1; break; }
        const bool ok_k = !rp.use_k || merged.cnt < (float)rp.topk;
        const bool ok_p = !rp.use_p || merged.q < pmass;
        if (ok_k && ok_p) break;
        j = merged.gi;  // next candidate, drawn from {x > x_j}
        xj = merged.gx;
      }
    }
    if (j >= 0) chosen = j;
  }
  if (tid == 0 && seg == 0) {
    finish_row(a, row, chosen, mx, z, c);
    // advance the row's epoch for the next launch: one store by segment 0, no exit ticket (32 device-scope
    // atomics or same-word stores per row serialise at the memory side). Safe: no block gets here before
    // it gathered pass 1 from EVERY block of its row, i.e. after every block read the epoch
    st_sc1(reinterpret_cast<float*>(a.epoch + row), __uint_as_float((ep + 1u) & 0x03ffffffu));
  }
}

int g_sample_nseg = SAMPLE_GRAN_SEGS;  // segments per row cap (set_sample_nseg; benchmarks/sampler_stress.py)
void set_sample_nseg(int n) { g_sample_nseg = n < 1 ? 1 : (n > SAMPLE_GRAN_SEGS ? SAMPLE_GRAN_SEGS : n); }

// At least 1024 logits in a segment, and no more than 8 to 24 segments of 2048: each block of a row polls all of the row's partials, which
// takes 1 us with 8 of them and 2.8 with 31 (us, top-p 0.95, 8 rows of 32000: 31 segments 19.4, 16 14.7, 8 15.3; of 151936: 31 25, 24 19.6,
// 16 21.5, 8 29.3).
int sample_segments(int B, int V) {
  const int V4 = V >> 2;
  int nseg = SAMPLE_MAX_BLOCKS / (B > 0 ? B : 1);
  if (nseg > g_sample_nseg) nseg = g_sample_nseg;
  nseg = std::min(nseg, std::min(V4 / 256, std::max(8, std::min(SAMPLE_GRAN_SEGS, V4 / 512))));
  return nseg < 1 ? 1 : nseg;
}

// More waves where a thread of 256 would have more than 12 pieces of 16 B: the noise of a segment (Philox, two logarithms per logit)
// then takes longer than the meeting (us, top-p 0.95, 512 -> 1024 threads: vocabulary 151936, 32 rows 29.4 -> 27.6, 64 rows 68.6 -> 62.9, 16 rows
// 24.0, 23.7; 32000, 64 rows 21.3, 21.6, 128 rows 34.5 -> 33.0, 8 rows 14.7, 15.5. 256 threads: 15.2 and 24.4 at 8 and 64 rows of 32000).
static bool long_rows(int V, int nseg) { return (V >> 2) > 3072 * nseg; }
// More whole rows than CUs: two workgroups of 1024 threads share a CU, of 256 eight, and only a long row makes up for that (us, 256 ->
// 1024 threads, greedy and top-p: 512 rows of 32000 27, 104 -> 35, 114, of 65536 44, 179 -> 48, 180, of 128256 76, 347 -> 71, 295; 768 rows of
// 128256 93, 493 -> 108, 512).
static bool long_whole_rows(int V, int B) { return B <= SAMPLE_MAX_BLOCKS ? long_rows(V, 1) : B <= 2 * SAMPLE_MAX_BLOCKS && V > 65536; }

void launch_sample(const SampleArgs& s, hipStream_t st) {
  if (s.B <= 0) return;
  const int nseg = sample_segments(s.B, s.V);
  SampleArgs a = s;
  if (nseg > 1 && s.gran != nullptr && s.epoch != nullptr && s.B <= SAMPLE_GRAN_ROWS) {
    a.tl = tl_take("sample_gran", nseg * s.B);
    if (long_rows(s.V, nseg)) hipLaunchKernelGGL(sample_gran_kernel<1024>, dim3(nseg, s.B), dim3(1024), 0, st, a);
    else hipLaunchKernelGGL(sample_gran_kernel<512>, dim3(nseg, s.B), dim3(512), 0, st, a);
    return;
  }
  a.tl = tl_take("sample", s.B);
  if (long_whole_rows(s.V, s.B)) hipLaunchKernelGGL(sample_row_kernel<1024>, dim3(1, s.B), dim3(1024), 0, st, a);
  else hipLaunchKernelGGL(sample_row_kernel<SAMPLE_THREADS>, dim3(1, s.B), dim3(SAMPLE_THREADS), 0, st, a);
}

}  // namespace vgate
