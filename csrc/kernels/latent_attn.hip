// Latent attention over a paged cache that holds, per token, one normed latent vector (rank) and one
// rotated key part (rot) shared by all heads. The per-head key and value up-projections are absorbed
// into the query and the output (q' = W_uk^T q, out = W_uv (sum_j p_j c_j)), so prompt portions and
// single decoded tokens run the same kernel on the cached rows alone:
//   score(t, h, j) = scale * (q'[t][h] . c_j + rope(q_rot[t][h]) . k_rot_j),   0 <= position(t) - j < window
//   ol[t][h]       = sum_j softmax_j(score) c_j
// A sink (one logit per head) only enters the softmax denominator: the running max starts at it, the sum at 1.
// Key tiles sit at absolute positions whatever the window's start, so a row's sums keep their order.
// latent_write: RMS norm of the latent (fp32 statistics) + rotation of the shared key part (interleaved or half-split
// pairs, cos and sin times a factor) + the paged store, one launch. Angles are position * inv_freq in fp32 with
// full-range sin / cos.
// latent_attn, fp32 caches (and shapes the MFMA kernel does not take): one workgroup per (token, group
// of heads); key tiles of 16 rows staged in LDS as fp32, scores, running max / sum and the weighted
// latent sum all in fp32 FMA.
// latent_attn, bf16 caches: MFMA kernel. Query rows are (token, head) pairs of one sequence, 16 per wave
// (4 independent waves per workgroup), keys in tiles of 32 = two pages:
//   S = Q K^T    v_mfma 16x16x32, Q fragments stationary in registers, K fragments (16 B of one cached
//                row per lane) straight from the cache
//   online softmax in fp32 (exp2 of log2(e)-scaled scores, per-lane partial row sums)
//   O += P C     P goes C-layout -> A-layout through a 16 x 32 bf16 tile in LDS; the B operand needs
//                eight consecutive KEYS of one latent column per lane, which the cache's second,
//                transposed copy of the latent part ([page][column][16 keys], written by latent_write)
//                delivers as one 16-B load: no transposition in the kernel
// Waves of a workgroup never meet at a barrier (each loops to its own causal limit), except for a
// sequence whose rows fit one wave (a decoded token): there the four waves take every fourth key tile
// of the same rows and merge their partial (max, sum, weighted latent) through LDS, so a lone token's
// keys are streamed by four waves instead of one. With parts > 1 (steps of decoded tokens: few workgroups), blockIdx.y
// of up to eight workgroups share such a sequence's key tiles (tile t goes to workgroup (t / 4) mod parts, wave
// t mod 4); each leaves its merged (max, sum, weighted latent) in an fp32 scratch and latent_attn_merge_kernel
// rescales and adds them in part order. The number of parts depends on the step's shape alone.
// latent_attn, bf16 caches, prompt portions: tiled kernel. A workgroup owns 64 (token, head) rows and its four waves split
// the columns instead of the rows, so that every cached element is read once per workgroup, by one wave, straight into
// that wave's registers: wave w multiplies every fourth 32-wide piece of the query rows with the same piece of the keys
// (partial scores of all 64 rows, summed over the waves through LDS in wave order), each wave takes the softmax of one of
// the four row tiles, and wave w accumulates the w-th quarter of the latent for all 64 rows (P comes from LDS). A key
// tile's fragments are asked for as soon as the ones before have been used, a phase ahead of their use; the barriers
// (two per tile) wait for LDS traffic only. A row's running max moves only when a tile exceeds it by more than 2^8 (the
// weights stay below 2^8 then, and the accumulators are rarely rescaled); that is decided per row, so a row's result does
// not depend on its neighbours. The workgroups with the most keys start first.
// latent_attn, bf16 caches, prompt portions, latents of 128, 256 or 512 with a rotated part of 64: staged kernel. Pages come into LDS by
// DMA a step ahead and each wave carries 16 or 32 rows from scores to weighted latents in registers (latent_attn_staged_kernel).
#include <stdlib.h>

#include <type_traits>

#include "lds_rows.h"
#include "locate.h"
#include "row_norm.h"
#include "seq_launchers.h"

namespace vgate {
namespace {

__device__ __forceinline__ float ldx(const void* p, int64_t i, int f32) {
  return f32 ? reinterpret_cast<const float*>(p)[i] : bf2f(reinterpret_cast<const bf16_t*>(p)[i]);
}
__device__ __forceinline__ void stx(void* p, int64_t i, int f32, float v) {
  if (f32) reinterpret_cast<float*>(p)[i] = v;
  else reinterpret_cast<bf16_t*>(p)[i] = f2bf(v);
}

// entry i (< rot_dims) of the row at x + base, turned by the position: pairs (2j, 2j + 1), or (j, j + rot_dims / 2)
__device__ __forceinline__ float turned(const LatentArgs& a, const void* x, int64_t base, int i, float pos) {
  const int hr = a.rot_dims >> 1;
  const bool second = a.rot_half ? i >= hr : (i & 1);
  const int j = a.rot_half ? (second ? i - hr : i) : (i >> 1);
  const int i0 = a.rot_half ? j : (i & ~1), i1 = a.rot_half ? j + hr : (i | 1);
  const float ang = pos * a.inv_freq[j];
  const float cs = cosf(ang) * a.rot_amp, sn = sinf(ang) * a.rot_amp;
  const float u = ldx(x, base + i0, a.f32), v = ldx(x, base + i1, a.f32);
  return second ? (v * cs + u * sn) : (u * cs - v * sn);
}

// grid (token, 2 with the query's latent): the key's row and the query's norm read the same projection and nothing of each other, so
// they share a launch (us, latents of 256 and 512, two launches -> one: 32 rows 4.7 + 3.9 -> 4.2, 2048 rows 8.4 + 5.9 -> 9.9). NI
// columns of the query's latent per thread in registers.
template <int NI>
__global__ __launch_bounds__(256) void latent_write_kernel(LatentArgs a, LatentWriteArgs b) {
  __shared__ float red[16];
  const int t = blockIdx.x;
  if (blockIdx.y == 1) {  // (uniform)
    const int64_t src = t * b.ldq, dst = (int64_t)t * b.qn;
    float v[NI], w[NI];
    load_row(b.qx, src, a.f32, b.qn, v);
    load_row(b.qw, 0, 1, b.qn, w);
    norm_row(v, b.qn, b.eps, 0, red, [&](int c) { return ldx(b.qx, src + c, a.f32); },
             [&](int c, int i, float r) { stx(b.qy, dst + c, a.f32, r * (i >= 0 ? w[i] : b.qw[c])); });
    return;
  }
  const int slot = a.slots[t];
  if (slot < 0) return;  // uniform per block
  const int64_t src = t * b.ldkv;
  const int64_t dst = (int64_t)slot * (a.rank + a.rot);
  bf16_t* cache_t = reinterpret_cast<bf16_t*>(b.cache_t);
  float v[2], w[2];
  load_row(b.kv, src, a.f32, a.rank, v);
  load_row(b.w, 0, 1, a.rank, w);
  norm_row(v, a.rank, b.eps, 0, red, [&](int c) { return ldx(b.kv, src + c, a.f32); }, [&](int c, int i, float r) {
    r *= i >= 0 ? w[i] : b.w[c];
    stx(a.cache, dst + c, a.f32, r);
    if (cache_t != nullptr)  // [page][column][key in page]
      cache_t[((int64_t)(slot / b.page) * a.rank + c) * b.page + slot % b.page] = f2bf(r);
  });
  const float pos = (float)a.positions[t];
  for (int i = threadIdx.x; i < a.rot; i += blockDim.x) {
    float o;
    if (i < a.rot_dims) {
      o = turned(a, b.kv, src + a.rank, i, pos);
    } else {
      o = ldx(b.kv, src + a.rank + i, a.f32);
    }
    stx(a.cache, dst + a.rank + i, a.f32, o);
  }
}

__global__ __launch_bounds__(256) void latent_qrope_kernel(LatentArgs a, const void* __restrict__ q, int H, int dim,
                                                            void* __restrict__ qa) {
  const int t = blockIdx.x;
  const float pos = (float)a.positions[t];
  for (int e = threadIdx.x; e < H * a.rot; e += blockDim.x) {
    const int h = e / a.rot, i = e % a.rot;
    const int64_t src = ((int64_t)t * H + h) * (dim + a.rot) + dim;
    float o;
    if (i < a.rot_dims) {
      o = turned(a, q, src, i, pos);
    } else {
      o = ldx(q, src + i, a.f32);
    }
    stx(qa, ((int64_t)t * H + h) * (a.rank + a.rot) + a.rank + i, a.f32, o);
  }
}

constexpr int KT = 16;      // keys per tile
constexpr int MAXACC = 16;  // latent outputs per thread: heads-per-block * rank <= 256 * MAXACC

__global__ __launch_bounds__(256) void latent_attn_kernel(LatentArgs a, const void* __restrict__ qa, int H, int HC,
                                                           float scale, const int32_t* __restrict__ block_tables,
                                                           int max_blocks, int page,
                                                           const int32_t* __restrict__ context_lens,
                                                           const int32_t* __restrict__ query_start, int S,
                                                           void* __restrict__ ol, int window,
                                                           const float* __restrict__ sink) {
  extern __shared__ float lds[];
  const int E = a.rank + a.rot, EP = E + 1;
  float* qs = lds;                  // [HC][EP]
  float* ks = qs + HC * EP;         // [KT][EP]
  float* sc = ks + KT * EP;         // [HC][KT] scores, then weights
  float* mrun = sc + HC * KT;       // [HC]
  float* lrun = mrun + HC;          // [HC]
  float* alpha = lrun + HC;         // [HC]
  const int t = blockIdx.x;
  if (t >= query_start[S]) return;
  int lo = 0, hi = S - 1;           // the sequence of token t: query_start[s] <= t < query_start[s + 1]
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (query_start[mid] <= t) lo = mid; else hi = mid - 1;
  }
  const int s = lo;
  const int nkeys = context_lens[s] - (query_start[s + 1] - t) + 1;
  const int first = max(0, nkeys - window);  // the oldest key the token sees
  const int h0 = blockIdx.y * HC;
  const int nh = min(HC, H - h0);
  const int tid = threadIdx.x;
  for (int e = tid; e < nh * E; e += 256) {
    const int h = e / E, c = e % E;
    qs[h * EP + c] = ldx(qa, ((int64_t)t * H + h0 + h) * E + c, a.f32);
  }
  if (tid < HC) {
    const bool sk = sink != nullptr && tid < nh;
    mrun[tid] = sk ? sink[h0 + tid] : -INFINITY;
    lrun[tid] = sk ? 1.f : 0.f;
    alpha[tid] = 1.f;
  }
  float acc[MAXACC];
#pragma unroll
  for (int i = 0; i < MAXACC; ++i) acc[i] = 0.f;
  const int32_t* bt = block_tables + (int64_t)s * max_blocks;
  for (int j0 = (first / KT) * KT; j0 < nkeys; j0 += KT) {
    __syncthreads();  // previous tile fully consumed (and q / running stats written)
    for (int e = tid; e < KT * E; e += 256) {
      const int jj = e / E, c = e % E;
      const int kj = j0 + jj;
      float v = 0.f;
      if (kj < nkeys && kj >= first) {
        const int64_t row = (int64_t)bt[kj / page] * page + kj % page;
        v = ldx(a.cache, row * E + c, a.f32);
      }
      ks[jj * EP + c] = v;
    }
    __syncthreads();
    {  // scores: two threads per (head, key), each half of the dot product
      const int wi = tid >> 1, half = tid & 1;
      float d = 0.f;
      const bool on = wi < nh * KT;
      const int h = on ? wi / KT : 0, jj = on ? wi % KT : 0;
      if (on) {
        const int c0 = half ? (E >> 1) : 0, c1 = half ? E : (E >> 1);
        const float* qp = qs + h * EP;
        const float* kp = ks + jj * EP;
        for (int c = c0; c < c1; ++c) d = fmaf(qp[c], kp[c], d);
      }
      d += __shfl_xor(d, 1, 64);
      if (on && half == 0) sc[h * KT + jj] = (j0 + jj < nkeys && j0 + jj >= first) ? d * scale : -INFINITY;
    }
    __syncthreads();
    if (tid < nh) {
      const float m0 = mrun[tid];
      float m1 = m0;
      for (int jj = 0; jj < KT; ++jj) m1 = fmaxf(m1, sc[tid * KT + jj]);
      const float al = expf(m0 - m1);  // m0 = -inf on the first tile: 0
      float l = 0.f;  // the tile's own sum first: the running sum takes one rounding per tile, not per key
      for (int jj = 0; jj < KT; ++jj) {
        const float pj = expf(sc[tid * KT + jj] - m1);
        sc[tid * KT + jj] = pj;
        l += pj;
      }
      mrun[tid] = m1; lrun[tid] = fmaf(lrun[tid], al, l); alpha[tid] = al;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MAXACC; ++i) {
      const int o = tid + i * 256;
      if (o < nh * a.rank) {
        const int h = o / a.rank, c = o % a.rank;
        float v = 0.f;
        const float* pp = sc + h * KT;
#pragma unroll
        for (int jj = 0; jj < KT; ++jj) v = fmaf(pp[jj], ks[jj * EP + c], v);
        acc[i] = fmaf(acc[i], alpha[h], v);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MAXACC; ++i) {
    const int o = tid + i * 256;
    if (o < nh * a.rank) {
      const int h = o / a.rank, c = o % a.rank;
      stx(ol, ((int64_t)t * H + h0 + h) * a.rank + c, a.f32, acc[i] / lrun[h]);
    }
  }
}


// ---------------------------------------------------------------------------------- MFMA (bf16)
__device__ __forceinline__ bf16x8 frag16(const bf16_t* rowp, int k, int K, bool valid) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (valid && k < K) {
    const bf16_t* q = rowp + k;
    if (k + 8 <= K && (reinterpret_cast<uintptr_t>(q) & 15) == 0) {
      v = ld16(q);
    } else {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = (k + 2 * j < K) ? q[2 * j] : 0;
        const uint32_t hi = (k + 2 * j + 1 < K) ? q[2 * j + 1] : 0;
        w[j] = lo | (hi << 16);
      }
      v = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  return as_bf16x8(v);
}

// reductions over the 16 lanes that share l >> 4: rotations by 8, 4, 2, 1 inside the DPP row (VALU, no LDS)
template <int CTRL>
__device__ __forceinline__ float row_rot(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float group16_max(float v) {
  v = fmaxf(v, row_rot<0x128>(v)); v = fmaxf(v, row_rot<0x124>(v));
  v = fmaxf(v, row_rot<0x122>(v)); v = fmaxf(v, row_rot<0x121>(v));
  return v;
}
__device__ __forceinline__ float group16_sum(float v) {
  v += row_rot<0x128>(v); v += row_rot<0x124>(v); v += row_rot<0x122>(v); v += row_rot<0x121>(v);
  return v;
}

// NCT: 16-column tiles of the latent (rank <= 16 NCT); NQF: 32-wide fragments of a query row (E <= 32 NQF).
// E % 8 == 0 (host-checked): every cache fragment is one unconditional 16-B load; a fragment past the row's
// end or the latent's last column is read from a clamped address: its partner (zero Q fragment) or its
// output column (never stored) makes the value irrelevant, and cached values are always finite.
// A decoded token's wave sees one or two key tiles, so what bounds it is how often it waits for memory: all of a tile's keys are asked
// for together, all of its values while the softmax runs (by groups of 4 and 8 before, nine waits a tile), and the four waves' results meet
// in LDS areas of their own, summed by all threads. us, 32 sequences: 12 heads, latent 512, some 700 keys 31.0 -> 22.7 and the merge 10.7 ->
// 4.6; 8 heads, latent 256, 512 keys 16.2 -> 11.5 and 6.6 -> 4.6.
// EXACT: rows of whole fragments and a latent of whole tiles (E = 32 NQF, rank = 16 NCT), nothing is clamped. The others read and multiply
// by what their rows do not have, too: leaving it out takes branches between the loads (us, 32 sequences, 12 heads, 700 keys, loads by groups of 4
// and 8 -> now, and now with branches: latent 264 of 328 29.6 -> 20.6, 21.2; 384 of 448 32.0 -> 21.8, 22.8; 512 of 512 35.7 -> 22.9, 24.2; 200
// of 224, 3 tokens beside 31 102 -> 78, 112).
template <int NCT, int NQF, bool EXACT>
__global__ __launch_bounds__(256, NCT > 16 ? 1 : 2) void latent_attn_mfma_kernel(LatentArgs a, const bf16_t* __restrict__ qa, int H,
                                                                float scale_log2e,
                                                                const int32_t* __restrict__ block_tables,
                                                                int max_blocks, int num_pages,
                                                                const int32_t* __restrict__ context_lens,
                                                                const int32_t* __restrict__ query_start, int S,
                                                                const bf16_t* __restrict__ cache_t,
                                                                bf16_t* __restrict__ ol, int window,
                                                                const float* __restrict__ sink, int parts,
                                                                float* __restrict__ part_o, float* __restrict__ part_ml) {
  __shared__ __attribute__((aligned(16))) bf16_t pl[4][16][40];
  __shared__ float mrg_m[4][16], mrg_l[4][16], mrg_f[4][16], row_l[16];
  constexpr int OS = 16 * NCT + 4;        // row stride of the area (the four rows of an instruction in different banks)
  extern __shared__ __attribute__((aligned(16))) float mrg_o[];  // split mode: the waves' weighted latents [4][16][OS]
  const int E = a.rank + a.rot, KR = a.rank;
  int tile;
  // (sequence, 64-row tile) of this workgroup
  const int s = locate_item(S, (int)blockIdx.x, tile, [&](int i) { return ((query_start[i + 1] - query_start[i]) * H + 63) / 64; });
  if (s < 0) return;
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lg = l >> 4;
  const int t0 = query_start[s], ntok = query_start[s + 1] - t0;
  const int pos0 = context_lens[s] - ntok;
  const int nrows = ntok * H;
  const bool split = nrows <= 16;  // workgroup-uniform: one row tile, keys shared out over the four waves
  const int part = blockIdx.y;     // (only sequences in split mode are shared out over several workgroups)
  if (!split && part > 0) return;
  const int np = split ? parts : 1;
  const int row0 = split ? 0 : tile * 64 + wv * 16;
  if (row0 >= nrows) return;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  const int nqf = (E + 31) >> 5, nct = (KR + 15) >> 4;
  // stationary Q fragments: A operand, lane holds Q[row lr][32 kk + 8 lg ..]
  bf16x8 qf[NQF];
  {
    const int r = row0 + lr;
    const bool ok = r < nrows;
    const bf16_t* qrow = qa + ((int64_t)(t0 + (ok ? r / H : 0)) * H + (ok ? r % H : 0)) * E;
#pragma unroll
    for (int kk = 0; kk < NQF; ++kk) qf[kk] = frag16(qrow, 32 * kk + 8 * lg, E, ok && kk < nqf);
  }
  // C-layout rows of this lane: row0 + 4 lg + i; keys visible to each
  int limit[4], lowest[4];
  float m[4], lsum[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = row0 + 4 * lg + i;
    const bool ok = r < nrows;
    limit[i] = ok ? pos0 + r / H + 1 : 0;   // keys [lowest, limit); a row past the last sees none
    lowest[i] = max(0, limit[i] - window);
    const bool sk = ok && sink != nullptr && (!split || (wv == 0 && part == 0));  // the sink counts once
    m[i] = sk ? sink[r % H] * 1.4426950408889634f : -INFINITY;
    lsum[i] = (sk && lr == 0) ? 1.f : 0.f;
  }
  const int last = min(row0 + 15, nrows - 1);
  const int kmax = pos0 + last / H + 1;  // wave-uniform
  const int kmin = max(0, pos0 + row0 / H + 1 - window) & ~31;  // first tile any row of the wave sees
  f32x4 O[NCT];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) O[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int32_t* bt = block_tables + (int64_t)s * max_blocks;
  for (int j0 = kmin + (split ? 32 * (wv + 4 * part) : 0); j0 < kmax; j0 += split ? 128 * np : 32) {
    int pg0 = bt[j0 >> 4];
    int pg1 = (j0 + 16 < kmax) ? bt[(j0 >> 4) + 1] : pg0;
    pg0 = __builtin_amdgcn_readfirstlane(min(max(pg0, 0), num_pages - 1));
    pg1 = __builtin_amdgcn_readfirstlane(min(max(pg1, 0), num_pages - 1));
    int kr = lr;
    if (!EXACT) asm volatile("" : "+v"(kr));  // (opaque: clamped offsets are worked out here and not kept in registers over the loop)
    f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16_t* k0p = cache + (int64_t)pg0 * 16 * E;   // (the page is the wave's: a scalar base and 32-bit offsets)
    const bf16_t* k1p = cache + (int64_t)pg1 * 16 * E;
    // fragments asked for together, as registers allow without spilling (clamped addresses take one more each)
    constexpr int KG = !EXACT ? 4 : (NCT > 16 ? NQF / 2 : NQF), VG = !EXACT ? 8 : (NCT > 16 ? NCT / 2 : NCT);
#pragma unroll
    for (int g = 0; g < NQF; g += KG) {
      uint4 b0[KG], b1[KG];
#pragma unroll
      for (int u = 0; u < KG; ++u)
        if (g + u < NQF) {
          const int off = kr * E + (EXACT ? 32 * (g + u) + 8 * lg : min(32 * (g + u) + 8 * lg, E - 8));
          b0[u] = ld16(k0p + off);
          b1[u] = ld16(k1p + off);
        }
#pragma unroll
      for (int u = 0; u < KG; ++u)
        if (g + u < NQF) {
          s0 = mfma16(qf[g + u], as_bf16x8(b0[u]), s0);
          s1 = mfma16(qf[g + u], as_bf16x8(b1[u]), s1);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    const bf16_t* tp = cache_t + ((int64_t)((lg >> 1) ? pg1 : pg0) * KR + kr) * 16 + 8 * (lg & 1);
    uint4 vb[VG];
    auto values = [&](int c0) {
#pragma unroll
      for (int u = 0; u < VG; ++u)
        if (c0 + u < NCT) vb[u] = ld16(tp + (EXACT ? 256 * (c0 + u) : 16 * (min(16 * (c0 + u) + kr, KR - 1) - kr)));
      __builtin_amdgcn_sched_barrier(0);
    };
    values(0);  // (asked for here, ahead of the softmax)
    float al[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v0 = (j0 + lr < limit[i] && j0 + lr >= lowest[i]) ? s0[i] * scale_log2e : -INFINITY;
      const float v1 = (j0 + 16 + lr < limit[i] && j0 + 16 + lr >= lowest[i]) ? s1[i] * scale_log2e : -INFINITY;
      const float mnew = fmaxf(m[i], group16_max(fmaxf(v0, v1)));
      const float ms = (mnew == -INFINITY) ? 0.f : mnew;  // a row that has seen no key yet (split mode)
      al[i] = exp2f(m[i] - ms);
      const float p0 = exp2f(v0 - ms), p1 = exp2f(v1 - ms);
      lsum[i] = lsum[i] * al[i] + p0 + p1;
      m[i] = mnew;
      pl[wv][4 * lg + i][lr] = f2bf(p0);
      pl[wv][4 * lg + i][16 + lr] = f2bf(p1);
    }
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) O[ct][i] *= al[i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's P tile is written (LDS is in order per wave)
    const bf16x8 pf = as_bf16x8(*reinterpret_cast<const uint4*>(&pl[wv][lr][8 * lg]));
#pragma unroll
    for (int c0 = 0; c0 < NCT; c0 += VG) {
      if (c0 > 0) values(c0);
#pragma unroll
      for (int u = 0; u < VG; ++u)
        if (c0 + u < NCT) O[c0 + u] = mfma16(pf, as_bf16x8(vb[u]), O[c0 + u]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // P tile read before the next tile overwrites it
  }
  if (split) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float tot = group16_sum(lsum[i]);
      if (lr == 0) { mrg_m[wv][4 * lg + i] = m[i]; mrg_l[wv][4 * lg + i] = tot; }
    }
    __syncthreads();
    const int64_t slot = (int64_t)part * gridDim.x + blockIdx.x;
    float* area = mrg_o + wv * 16 * OS;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * lg + i;
      float M = mrg_m[0][r];
#pragma unroll
      for (int w = 1; w < 4; ++w) M = fmaxf(M, mrg_m[w][r]);
      const float Ms = (M == -INFINITY) ? 0.f : M;  // (rows past the sequence's last)
      float L = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) L += mrg_l[w][r] * exp2f(mrg_m[w][r] - Ms);  // a wave that saw no key: l = 0, exp2(-inf) = 0
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) area[r * OS + 16 * ct + lr] = O[ct][i];
      if (lr == 0) mrg_f[wv][r] = exp2f(m[i] - Ms);
      if (wv == 0 && lr == 0) {
        row_l[r] = L;
        if (np > 1) {
          part_ml[(slot * 16 + r) * 2] = M;
          part_ml[(slot * 16 + r) * 2 + 1] = L;
        }
      }
    }
    __syncthreads();
    // four columns a thread and turn, the waves' parts scaled and added in wave order, each by one fused step; np > 1 (workgroup-uniform):
    // handed on, the merge kernel finishes the rows
#pragma unroll 4
    for (int e = threadIdx.x; e < 16 * 4 * NCT; e += 256) {
      const int r = e / (4 * NCT), col = 4 * (e % (4 * NCT));
      const float* o = mrg_o + r * OS + col;
      f32x4 y = *reinterpret_cast<const f32x4*>(o) * mrg_f[0][r];
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(o + 16 * w * OS);
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = fmaf(v[j], mrg_f[w][r], y[j]);
      }
      if (np > 1) {
        *reinterpret_cast<f32x4*>(part_o + slot * (16 * 16 * NCT) + r * (16 * NCT) + col) = y;
      } else if (r < nrows) {
        const float inv = 1.f / row_l[r];
        bf16_t* orow = ol + ((int64_t)(t0 + r / H) * H + r % H) * KR;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (col + j < KR) orow[col + j] = f2bf(y[j] * inv);
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float tot = group16_sum(lsum[i]);
    const float inv = 1.f / tot;
    const int r = row0 + 4 * lg + i;
    if (r < nrows) {
      bf16_t* orow = ol + ((int64_t)(t0 + r / H) * H + r % H) * KR;
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const int col = 16 * ct + lr;
        if (ct < nct && col < KR) orow[col] = f2bf(O[ct][i] * inv);
      }
    }
  }
}

// NC: 16-column tiles of the latent per wave (rank <= 64 NC); NK: 32-wide query / key pieces per wave (E <= 128 NK).
// E % 8 == 0 (host-checked). Pieces past the row's end and columns past the latent's last are read from clamped addresses:
// a zero query piece or an output column that is never stored makes their value irrelevant.
constexpr float LAZY_MAX = 8.f;
template <int NC, int NK>
__global__ __launch_bounds__(256) void latent_attn_tiled_kernel(LatentArgs a, const bf16_t* __restrict__ qa, int H,
                                                                 float scale_log2e, const int32_t* __restrict__ block_tables,
                                                                 int max_blocks, int num_pages,
                                                                 const int32_t* __restrict__ context_lens,
                                                                 const int32_t* __restrict__ query_start, int S,
                                                                 const bf16_t* __restrict__ cache_t, bf16_t* __restrict__ ol,
                                                                 int window, const float* __restrict__ sink) {
  __shared__ __attribute__((aligned(16))) f32x4 sp[4][8][64];     // [wave][row tile, key half][lane]: partial scores
  __shared__ __attribute__((aligned(16))) bf16_t pl[64][40];      // weights
  __shared__ __attribute__((aligned(16))) float fac[64];          // rescaling factors, at the end 1 / row sums
  const int E = a.rank + a.rot, KR = a.rank;
  const int bx = gridDim.x - 1 - blockIdx.x;
  int tile;
  // (sequence, 64-row tile) of this workgroup
  const int s = locate_item(S, bx, tile, [&](int i) { return ((query_start[i + 1] - query_start[i]) * H + 63) / 64; });
  if (s < 0) return;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lg = l >> 4;
  const int t0 = query_start[s], ntok = query_start[s + 1] - t0;
  const int pos0 = context_lens[s] - ntok;
  const int nrows = ntok * H, row0 = tile * 64;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(a.cache);
  bf16x8 qf[4][NK];  // A operands: lane holds Q[row 16 rt + lr][32 (w + 4 i) + 8 lg ..]
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int r = row0 + 16 * rt + lr;
    const bool ok = r < nrows;
    const bf16_t* qrow = qa + ((int64_t)(t0 + (ok ? r / H : 0)) * H + (ok ? r % H : 0)) * E;
#pragma unroll
    for (int i = 0; i < NK; ++i) qf[rt][i] = frag16(qrow, 32 * (w + 4 * i) + 8 * lg, E, ok);
  }
  // softmax rows of this lane: row0 + 16 w + 4 lg + i; keys [lowest, limit) are visible
  int limit[4], lowest[4];
  float m[4], lsum[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = row0 + 16 * w + 4 * lg + i;
    const bool ok = r < nrows;
    limit[i] = ok ? pos0 + r / H + 1 : 0;
    lowest[i] = max(0, limit[i] - window);
    const bool sk = ok && sink != nullptr;
    m[i] = sk ? sink[r % H] * 1.4426950408889634f : -INFINITY;
    lsum[i] = (sk && lr == 0) ? 1.f : 0.f;
  }
  const int kmax = pos0 + min(row0 + 63, nrows - 1) / H + 1;       // workgroup-uniform
  const int kmin = max(0, pos0 + row0 / H + 1 - window) & ~31;
  const int32_t* bt = block_tables + (int64_t)s * max_blocks;
  auto page_of = [&](int j) { return min(max(bt[min(j, kmax - 1) >> 4], 0), num_pages - 1); };
  uint4 kf[2][NK], cf[NC];
  auto load_k = [&](int p0, int p1) {
    const bf16_t* k0 = cache + ((int64_t)p0 * 16 + lr) * E;
    const bf16_t* k1 = cache + ((int64_t)p1 * 16 + lr) * E;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int off = min(32 * (w + 4 * i) + 8 * lg, E - 8);
      kf[0][i] = ld16(k0 + off);
      kf[1][i] = ld16(k1 + off);
    }
  };
  auto load_c = [&](int p0, int p1) {  // eight consecutive keys of one latent column per lane
    const bf16_t* tp = cache_t + (int64_t)((lg >> 1) ? p1 : p0) * KR * 16 + 8 * (lg & 1);
#pragma unroll
    for (int c = 0; c < NC; ++c) cf[c] = ld16(tp + (int64_t)min(16 * (w * NC + c) + lr, KR - 1) * 16);
  };
  f32x4 O[4][NC];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int c = 0; c < NC; ++c) O[rt][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  int p0 = page_of(kmin), p1 = page_of(kmin + 16);
  int n0 = page_of(kmin + 32), n1 = page_of(kmin + 48);   // the next tile's pages (past the last: a page that is there)
  load_k(p0, p1);
  load_c(p0, p1);
  for (int j0 = kmin; j0 < kmax; j0 += 32) {
    f32x4 sc[4][2];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) sc[rt][0] = sc[rt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NK; ++i)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        sc[rt][0] = mfma16(qf[rt][i], as_bf16x8(kf[0][i]), sc[rt][0]);
        sc[rt][1] = mfma16(qf[rt][i], as_bf16x8(kf[1][i]), sc[rt][1]);
      }
    load_k(n0, n1);   // the next tile's keys: under way during the softmax and the weighted sum
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      sp[w][2 * rt][l] = sc[rt][0];
      sp[w][2 * rt + 1][l] = sc[rt][1];
    }
    lds_barrier();
    f32x4 s0 = sp[0][2 * w][l], s1 = sp[0][2 * w + 1][l];
#pragma unroll
    for (int u = 1; u < 4; ++u) { s0 += sp[u][2 * w][l]; s1 += sp[u][2 * w + 1][l]; }
    f32x4 al;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v0 = (j0 + lr < limit[i] && j0 + lr >= lowest[i]) ? s0[i] * scale_log2e : -INFINITY;
      const float v1 = (j0 + 16 + lr < limit[i] && j0 + 16 + lr >= lowest[i]) ? s1[i] * scale_log2e : -INFINITY;
      const float top = group16_max(fmaxf(v0, v1));
      const bool move = top > m[i] + LAZY_MAX;   // (m = -inf: the first visible keys; the same in the row's 16 lanes)
      const float mo = m[i];
      m[i] = move ? top : mo;
      const float ms = (m[i] == -INFINITY) ? 0.f : m[i];   // a row that has seen no key yet
      al[i] = move ? exp2f(mo - top) : 1.f;
      const float e0 = exp2f(v0 - ms), e1 = exp2f(v1 - ms);
      lsum[i] = lsum[i] * al[i] + e0 + e1;
      pl[16 * w + 4 * lg + i][lr] = f2bf(e0);
      pl[16 * w + 4 * lg + i][16 + lr] = f2bf(e1);
    }
    if (lr == 0) *reinterpret_cast<f32x4*>(&fac[16 * w + 4 * lg]) = al;
    lds_barrier();
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const f32x4 f = *reinterpret_cast<const f32x4*>(&fac[16 * rt + 4 * lg]);
      if (__any(f[0] != 1.f || f[1] != 1.f || f[2] != 1.f || f[3] != 1.f)) {
#pragma unroll
        for (int c = 0; c < NC; ++c) O[rt][c] *= f;
      }
      const bf16x8 pf = as_bf16x8(*reinterpret_cast<const uint4*>(&pl[16 * rt + lr][8 * lg]));
#pragma unroll
      for (int c = 0; c < NC; ++c) O[rt][c] = mfma16(pf, as_bf16x8(cf[c]), O[rt][c]);
    }
    load_c(n0, n1);
    __builtin_amdgcn_sched_barrier(0);
    n0 = page_of(j0 + 64);
    n1 = page_of(j0 + 80);
  }
  {
    f32x4 inv;
#pragma unroll
    for (int i = 0; i < 4; ++i) inv[i] = 1.f / group16_sum(lsum[i]);
    __syncthreads();   // every wave has read the last tile's factors
    if (lr == 0) *reinterpret_cast<f32x4*>(&fac[16 * w + 4 * lg]) = inv;
    __syncthreads();
  }
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rl = 16 * rt + 4 * lg + i, r = row0 + rl;
      if (r < nrows) {
        const float inv = fac[rl];
        bf16_t* orow = ol + ((int64_t)(t0 + r / H) * H + r % H) * KR;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int col = 16 * (w * NC + c) + lr;
          if (col < KR) orow[col] = f2bf(O[rt][c][i] * inv);
        }
      }
    }
}

// Prompt portions, rows of whole 128-B lines (E = 64 NE, rank = 16 NCT): a workgroup owns 64 (token, head) rows, KW of its waves share 16 KW of
// them and take every KW-th tile of 32 keys (absolute positions, so that a row's sums keep their order). The pages of a step are staged
// by LDS-DMA, keys as rows of lines (lds_rows.h) and the transposed latents as they lie, one step ahead. A wave computes K Q^T, so that a
// lane holds eight keys of one row: the row's maximum takes two exchanges, and the weights are the B operand of C^T P as they are, once
// the latents are read in the same order of keys: nothing but the stages goes through LDS until the KW waves' results are added.
// What bounds it is the chain of a lone wave per SIMD (products, softmax, products: some 400 instructions between two barriers for 72
// products) and LDS, per wave and tile of 32 keys 2 NE + NCT KiB of fragments for KW row tiles. The sums stay in AGPRs (mfma_acc, and a
// read only inside the rare rescaling: hoisted before its branch it was 128 moves per step), latents are asked for before the softmax,
// masks are a branch (most tiles have none hidden).
// (latent_attn_tiled_kernel, which this one replaces there: keys straight into registers, 64 lanes on 16 lines for 64 B each, scores and
// weights through LDS between barriers. 1999 tokens of 8 heads, rank 256: 131 -> 66 us; 3 x 601 tokens of 12 heads among 5 decoded,
// rank 512: 94 -> 55. On the way: with the builtin products 102 / 90, in AGPRs 83 / 57.)
template <int NE, int NCT, int KW>
__global__ __launch_bounds__(256, 1) void latent_attn_staged_kernel(LatentArgs a, const bf16_t* __restrict__ qa, int H,
                                                                    float scale_log2e, const int32_t* __restrict__ block_tables,
                                                                    int max_blocks, int num_pages,
                                                                    const int32_t* __restrict__ context_lens,
                                                                    const int32_t* __restrict__ query_start, int S,
                                                                    const bf16_t* __restrict__ cache_t, bf16_t* __restrict__ ol,
                                                                    int window, const float* __restrict__ sink) {
  constexpr int E = 64 * NE, KR = 16 * NCT, PP = 2 * NE + NCT / 2;   // 1 KiB pieces of a page: keys, transposed latents
  constexpr int PPW = KW == 2 ? PP : (2 * NE > NCT / 2 ? 2 * NE : NCT / 2), STAGE = 2 * KW * PP * 1024, STEP = 32 * KW;
  static_assert(NCT % 8 == 0 && PPW % 2 == 0 && (KW == 1 || KW == 2) && 2 * PPW < 64, "whole pieces, vmcnt");
  extern __shared__ __attribute__((aligned(16))) char smem[];   // two stages; at the end the KW waves' results
  int tile;
  const int s = __builtin_amdgcn_readfirstlane(
      locate_item(S, (int)(gridDim.x - 1 - blockIdx.x), tile, [&](int i) { return ((query_start[i + 1] - query_start[i]) * H + 63) / 64; }));
  if (s < 0) return;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, lr = l & 15, lg = l >> 4;
  const int kw = KW == 2 ? wid & 1 : 0, rw = KW == 2 ? wid >> 1 : wid;
  const int t0 = query_start[s], ntok = query_start[s + 1] - t0;
  const int pos0 = context_lens[s] - ntok;
  const int nrows = ntok * H, row0 = __builtin_amdgcn_readfirstlane(tile) * 64, wrow = row0 + 16 * KW * rw;
  bf16x8 qf[KW][2 * NE];   // B operands: lane holds Q[row wrow + 16 r + lr][32 i + 8 lg ..]
  int limit[KW], lowest[KW];   // the row's visible keys: [lowest, limit)
  float m[KW], lsum[KW];
#pragma unroll
  for (int r = 0; r < KW; ++r) {
    const int row = wrow + 16 * r + lr;
    const bool ok = row < nrows;
    const bf16_t* qrow = qa + ((int64_t)(t0 + (ok ? row / H : 0)) * H + (ok ? row % H : 0)) * E;
#pragma unroll
    for (int i = 0; i < 2 * NE; ++i) qf[r][i] = as_bf16x8(ld16(qrow + 32 * i + 8 * lg));
    limit[r] = ok ? pos0 + row / H + 1 : 0;
    lowest[r] = max(0, limit[r] - window);
    const bool sk = ok && sink != nullptr && kw == 0;
    m[r] = sk ? sink[row % H] * 1.4426950408889634f : -INFINITY;
    lsum[r] = (sk && lg == 0) ? 1.f : 0.f;
  }
  const int kmax = __builtin_amdgcn_readfirstlane(pos0 + min(row0 + 63, nrows - 1) / H + 1);
  const int first = __builtin_amdgcn_readfirstlane(max(0, pos0 + row0 / H + 1 - window)), kmin = first & ~(STEP - 1);
  const int open = pos0 + row0 / H + 1;   // below: every row's limit is further on
  const int nsteps = (kmax - kmin + STEP - 1) / STEP;
  const int32_t* bt = block_tables + (int64_t)s * max_blocks;
  // this wave's share of a step's pages: page pgw, or (KW = 1) its keys or its latents, the fewer of them some twice
  const int pgw = KW == 2 ? wid : wid >> 1;
  auto page_of = [&](int t) {
    const int j = kmin + STEP * t + 16 * pgw;
    return min(max(bt[min(j, kmax - 1) >> 4], 0), num_pages - 1);
  };
  const uint32_t lds0 = lds_addr_of(smem), cvo = l * 16;
  uint32_t kvo[2];   // (x_piece_col(), the second page of a tile turned by two chunks: a fragment has rows of both)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * i + (l >> 3);
    kvo[i] = (uint32_t)r * (2u * E) - 1024u * i + (uint32_t)(((l & 7) ^ x_swz(r) ^ ((pgw & 1) << 1)) << 4);
  }
  auto issue = [&](int page, int buf) {
    const u32x4 krs = rsrc_words(reinterpret_cast<const bf16_t*>(a.cache) + (int64_t)page * 16 * E);
    const u32x4 crs = rsrc_words(cache_t + (int64_t)page * 16 * KR);
    const uint32_t dst = lds0 + buf * STAGE + (uint32_t)(pgw * PP) * 1024u;
    constexpr int NK = KW == 2 ? 2 * NE : PPW, NC = KW == 2 ? NCT / 2 : PPW;
    if (KW == 2 || (wid & 1) == 0) {
#pragma unroll
      for (int q = 0; q < NK; q += 2) {
        const int x = q % (2 * NE);
        blds16_run<2>(krs, kvo, (uint32_t)(x >> 1) * 128u, dst + x * 1024u);
      }
    }
    if (KW == 2 || (wid & 1) == 1) {
#pragma unroll
      for (int q = 0; q < NC; q += q + 4 <= NC ? 4 : 2) {
        const int x = q % (NCT / 2);
        if (q + 4 <= NC) blds16_run<4>(crs, {cvo, cvo, cvo, cvo}, (uint32_t)x * 1024u, dst + (2 * NE + x) * 1024u);
        else blds16_run<2>(crs, {cvo, cvo}, (uint32_t)x * 1024u, dst + (2 * NE + x) * 1024u);
      }
    }
  };
  f32x4 O[KW][NCT];
#pragma unroll
  for (int r = 0; r < KW; ++r)
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      O[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(O[r][c]));
    }
  // row lr of key fragment k is the tile's key 8 (lr / 4) + 4 k + lr % 4: a lane's scores are then those of keys 8 lg .. 8 lg + 7, which it
  // meets again as 16 B of a transposed latent
  int ko[2][2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int pg = lr >> 3, r = ((8 * (lr >> 2)) & 15) + 4 * k + (lr & 3);
      ko[k][i] = pg * PP * 1024 + r * 128 + (((4 * i + lg) ^ x_swz(r) ^ (pg << 1)) << 4);
    }
  const int co = (2 * NE + (lg >> 1) * PP) * 1024 + lr * 32 + (lg & 1) * 16;
  // the loads above are waited for here, and the compiler sees that: from now on the counter holds DMA alone (a wait for the queries inside
  // the loop waits for the next step's pages too)
#pragma unroll
  for (int r = 0; r < KW; ++r) {
#pragma unroll
    for (int i = 0; i < 2 * NE; ++i) asm volatile("" : "+v"(qf[r][i]));
    asm volatile("" : "+v"(m[r]));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  issue(page_of(0), 0);
  issue(page_of(1), 1);
  int next = page_of(2);
  for (int t = 0; t < nsteps; ++t) {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PPW) : "memory");   // the step's pages are there, for every wave
    const int j0 = kmin + STEP * t + 32 * kw;
    const char* sb = smem + (t & 1) * STAGE + 2 * kw * PP * 1024;
    if (j0 < kmax && j0 + 32 > first) {
      f32x4 sc[KW][2];
#pragma unroll
      for (int r = 0; r < KW; ++r) sc[r][0] = sc[r][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 2 * NE; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const bf16x8 kf = as_bf16x8(*reinterpret_cast<const uint4*>(sb + (i >> 1) * 2048 + ko[k][i & 1]));
#pragma unroll
          for (int r = 0; r < KW; ++r) sc[r][k] = mfma16(kf, qf[r][i], sc[r][k]);
        }
      constexpr int CA = 16 < NCT ? 16 : NCT;   // latents asked for before the softmax
      uint4 cf[CA];
#pragma unroll
      for (int c = 0; c < CA; ++c) cf[c] = *reinterpret_cast<const uint4*>(sb + co + c * 512);
      __builtin_amdgcn_sched_barrier(0xf);   // (arithmetic may pass)
      float v[KW][8], al[KW];
#pragma unroll
      for (int r = 0; r < KW; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[r][e] = sc[r][e >> 2][e & 3] * scale_log2e;
      if (j0 + 32 > open || j0 < kmax - window) {   // a key that one of the rows doesn't see
        asm volatile("");   // (a branch)
#pragma unroll
        for (int r = 0; r < KW; ++r)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int j = j0 + 8 * lg + e;
            v[r][e] = (j < limit[r] && j >= lowest[r]) ? v[r][e] : -INFINITY;
          }
      }
      uint4 pf[KW];
      bool moved = false;
#pragma unroll
      for (int r = 0; r < KW; ++r) {
        float top = v[r][0];
#pragma unroll
        for (int e = 1; e < 8; ++e) top = fmaxf(top, v[r][e]);
        top = fmaxf(top, xor16(top));
        top = fmaxf(top, xor32(top));
        const bool move = top > m[r] + LAZY_MAX;   // (m = -inf: the first visible keys; the same in the row's four lanes)
        moved |= move;
        al[r] = move ? exp2f(m[r] - top) : 1.f;   // (not the bare instruction, for which results below 2^-126 are zero)
        m[r] = move ? top : m[r];
        const float ms = (m[r] == -INFINITY) ? 0.f : m[r];   // a row that has seen no key yet
        lsum[r] = lsum[r] * al[r] + weights8(v[r], ms);
        pf[r] = pack8(v[r]);
      }
      if (__any(moved)) {
#pragma unroll
        for (int r = 0; r < KW; ++r)
#pragma unroll
          for (int c = 0; c < NCT; ++c) {
            asm volatile("" : "+a"(O[r][c]));   // (read here, not before the branch)
            O[r][c] *= al[r];
            asm volatile("" : "+a"(O[r][c]));
          }
      }
#pragma unroll
      for (int r = 0; r < KW; ++r) {
        u32x4 pk = __builtin_bit_cast(u32x4, pf[r]);
        asm volatile("s_nop 1" : "+v"(pk));   // (the wait states that mfma_acc asks for)
        pf[r] = __builtin_bit_cast(uint4, pk);
      }
#pragma unroll
      for (int c = 0; c < NCT; ++c) {
        const uint4 f = c < CA ? cf[c < CA ? c : 0] : *reinterpret_cast<const uint4*>(sb + co + c * 512);
#pragma unroll
        for (int r = 0; r < KW; ++r) mfma_acc(O[r][c], f, pf[r]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // every wave is done with the buffer
    issue(next, t & 1);   // (past the last step: pages that are there, never used)
    next = page_of(t + 3);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int r = 0; r < KW; ++r)
#pragma unroll
    for (int c = 0; c < NCT; ++c) asm volatile("" : "+a"(O[r][c]));
  if constexpr (KW == 2) {   // the odd key tiles' results onto the even ones'
    f32x4* po = reinterpret_cast<f32x4*>(smem) + (rw * 64 + l) ;
    float* pm = reinterpret_cast<float*>(smem + 2 * KW * NCT * 1024);
    if (kw == 1) {
#pragma unroll
      for (int r = 0; r < KW; ++r) {
#pragma unroll
        for (int c = 0; c < NCT; ++c) po[(r * NCT + c) * 128] = O[r][c];
        pm[(r * 2 + rw) * 128 + l] = m[r];
        pm[(r * 2 + rw) * 128 + 64 + l] = lsum[r];
      }
    }
    __syncthreads();
    if (kw == 1) return;
#pragma unroll
    for (int r = 0; r < KW; ++r) {
      const float mo = pm[(r * 2 + rw) * 128 + l], lo = pm[(r * 2 + rw) * 128 + 64 + l];
      const float M = fmaxf(m[r], mo);
      // a half that saw no key: max -inf, factor 0; a sink of +inf, in the even half's maximum: factor 1, the row's weights are zero
      const float f0 = m[r] == M ? 1.f : exp2f(m[r] - M), f1 = mo == M ? 1.f : exp2f(mo - M);
      lsum[r] = lsum[r] * f0 + lo * f1;
#pragma unroll
      for (int c = 0; c < NCT; ++c) O[r][c] = O[r][c] * f0 + po[(r * NCT + c) * 128] * f1;
    }
  }
#pragma unroll
  for (int r = 0; r < KW; ++r) {
    float tot = lsum[r];
    tot += xor16(tot);
    tot += xor32(tot);
    const float inv = 1.f / tot;
    const int row = wrow + 16 * r + lr;
    if (row < nrows) {
      bf16_t* orow = ol + ((int64_t)(t0 + row / H) * H + row % H) * KR + 4 * lg;
#pragma unroll
      for (int c = 0; c < NCT; ++c)
        *reinterpret_cast<uint2*>(orow + 16 * c) =
            make_uint2(pack_bf2(O[r][c][0] * inv, O[r][c][1] * inv), pack_bf2(O[r][c][2] * inv, O[r][c][3] * inv));
    }
  }
}

// The rows of a split sequence from the partial results of `parts` workgroups: M = max of the parts' maxima (log2
// units), sums and weighted latents rescaled by 2^(M_p - M) and added in part order, then normalised and stored.
// vs: the row stride of the parts' weighted latents.
__global__ __launch_bounds__(256) void latent_attn_merge_kernel(int rank, int H, const int32_t* __restrict__ query_start,
                                                                 int S, int parts, int vs, const float* __restrict__ part_o,
                                                                 const float* __restrict__ part_ml,
                                                                 bf16_t* __restrict__ ol) {
  int tile;
  // the sequence of this workgroup, numbered as in the attention kernel
  const int s = locate_item(S, (int)blockIdx.x, tile, [&](int i) { return ((query_start[i + 1] - query_start[i]) * H + 63) / 64; });
  if (s < 0) return;
  const int t0 = query_start[s], nrows = (query_start[s + 1] - t0) * H;
  if (nrows > 16) return;  // (not shared out: the attention kernel has stored its rows)
  constexpr int MAXP = 8;
  // a thread's four columns of the blockIdx.y-th rows of the tile (a workgroup's threads take each column of its rows once at most: one
  // wait for memory)
  const int c4 = (rank + 3) / 4, per = 16 / gridDim.y;
  for (int e = threadIdx.x; e < per * c4; e += blockDim.x) {
    const int r = per * blockIdx.y + e / c4, col = 4 * (e % c4);   // (columns past the latent's last: within the row's stride, never stored)
    if (r >= nrows) continue;
    float pm[MAXP], plv[MAXP], M = -INFINITY;
    f32x4 po[MAXP];
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {  // all parts' loads asked for together
      const int64_t slot = (int64_t)min(p, parts - 1) * gridDim.x + blockIdx.x;
      const float2 ml = *reinterpret_cast<const float2*>(part_ml + (slot * 16 + r) * 2);
      pm[p] = p < parts ? ml.x : -INFINITY;
      plv[p] = ml.y;
      po[p] = *reinterpret_cast<const f32x4*>(part_o + slot * (16 * vs) + r * vs + col);
      M = fmaxf(M, pm[p]);
    }
    float L = 0.f;
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
      const float f = exp2f(pm[p] - M);  // a part that saw no key (or is none): max -inf, factor 0
      L = fmaf(plv[p], f, L);
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = fmaf(po[p][j], f, y[j]);
    }
    bf16_t* o = ol + ((int64_t)(t0 + r / H) * H + r % H) * rank + col;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (col + j < rank) o[j] = f2bf(y[j] / L);
  }
}

// VGATE_LATENT_TILED=0: prompt portions on the kernel whose waves split the rows
bool tiled_prefill() {
  static const bool on = [] {
    const char* e = getenv("VGATE_LATENT_TILED");
    return e == nullptr || e[0] != '0';
  }();
  return on;
}

// Latents of 128, 256 or 512 with a rotated part of 64: rows of whole lines, 16-B aligned (else the tiled kernel)
template <int NCT>
bool staged_takes(const LatentArgs& a, const void* qa, const void* cache_t, const void* ol) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(a.cache) | reinterpret_cast<uintptr_t>(qa) | reinterpret_cast<uintptr_t>(cache_t) |
                       reinterpret_cast<uintptr_t>(ol);
  return a.rank == 16 * NCT && a.rot == 64 && at % 16 == 0;
}

template <int NCT, int NQF>
void launch_mfma(const LatentArgs& a, const void* qa, int H, float scale, const int32_t* block_tables, int max_blocks,
                 int num_pages, const int32_t* context_lens, const int32_t* query_start, int S, const void* cache_t,
                 void* ol, int window, const float* sink, int parts, float* scratch, hipStream_t st) {
  const int blocks = (a.T * H + 63) / 64 + S;
  if ((int64_t)a.T * H > 16 * (int64_t)S && tiled_prefill() && staged_takes<NCT>(a, qa, cache_t, ol)) {
    constexpr int NE = NCT / 4 + 1, KW = NCT <= 16 ? 2 : 1;
    constexpr int LDS = 2 * 2 * KW * (2 * NE + NCT / 2) * 1024;
    auto kern = latent_attn_staged_kernel<NE, NCT, KW>;
    static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
    (void)attr;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), LDS, st, a, reinterpret_cast<const bf16_t*>(qa), H, scale * 1.4426950408889634f,
                       block_tables, max_blocks, num_pages, context_lens, query_start, S, reinterpret_cast<const bf16_t*>(cache_t),
                       reinterpret_cast<bf16_t*>(ol), window, sink);
    return;
  }
  if ((int64_t)a.T * H > 16 * (int64_t)S && tiled_prefill()) {  // (prompt portions among the step's sequences)
    hipLaunchKernelGGL((latent_attn_tiled_kernel<NCT / 4, (NQF + 3) / 4>), dim3(blocks), dim3(256), 0, st, a,
                       reinterpret_cast<const bf16_t*>(qa), H, scale * 1.4426950408889634f, block_tables, max_blocks, num_pages,
                       context_lens, query_start, S, reinterpret_cast<const bf16_t*>(cache_t), reinterpret_cast<bf16_t*>(ol),
                       window, sink);
    return;
  }
  float* part_o = scratch;
  float* part_ml = parts > 1 ? scratch + (size_t)parts * blocks * 16 * 16 * NCT : nullptr;
  auto decode = [&](auto nqf, auto exact) {
    constexpr int LDS = 4 * 16 * (16 * NCT + 4) * 4;
    auto kern = latent_attn_mfma_kernel<NCT, decltype(nqf)::value, decltype(exact)::value>;
    static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
    (void)attr;
    hipLaunchKernelGGL(kern, dim3(blocks, parts), dim3(256), LDS, st, a, reinterpret_cast<const bf16_t*>(qa), H,
                       scale * 1.4426950408889634f, block_tables, max_blocks, num_pages, context_lens, query_start, S,
                       reinterpret_cast<const bf16_t*>(cache_t), reinterpret_cast<bf16_t*>(ol), window, sink, parts, part_o, part_ml);
  };
  if (a.rot == 64 && a.rank == 16 * NCT) decode(std::integral_constant<int, NCT / 2 + 2>{}, std::true_type{});
  else decode(std::integral_constant<int, NQF>{}, std::false_type{});
  if (parts > 1)
    hipLaunchKernelGGL(latent_attn_merge_kernel, dim3(blocks, a.rank <= 256 ? 4 : 8), dim3(256), 0, st, a.rank, H, query_start, S, parts, 16 * NCT,
                       part_o, part_ml, reinterpret_cast<bf16_t*>(ol));
}

// 16-column tiles / 32-wide query fragments of the instantiation that takes a latent of this size
void mfma_shape(int rank, int E, int& nct, int& nqf) {
  if (rank <= 128 && E <= 128) { nct = 8; nqf = 4; }
  else if (rank <= 128 && E <= 192) { nct = 8; nqf = 6; }
  else if (rank <= 256 && E <= 256) { nct = 16; nqf = 8; }
  else if (rank <= 256 && E <= 384) { nct = 16; nqf = 12; }
  else if (E <= 512) { nct = 32; nqf = 16; }
  else { nct = 32; nqf = 20; }
}
bool mfma_takes(int rank, int rot, int f32, int page) {
  const int E = rank + rot;
  return !f32 && page == 16 && rank <= 512 && E <= 640 && E % 8 == 0 && E >= 8;
}

}  // namespace

void launch_latent_write(const LatentArgs& a, const LatentWriteArgs& w, hipStream_t st) {
  if (a.T <= 0) return;
  const dim3 grid(a.T, w.qn > 0 ? 2 : 1);
  if (w.qn <= 512) hipLaunchKernelGGL(latent_write_kernel<2>, grid, dim3(256), 0, st, a, w);
  else if (w.qn <= 1024) hipLaunchKernelGGL(latent_write_kernel<4>, grid, dim3(256), 0, st, a, w);
  else hipLaunchKernelGGL(latent_write_kernel<8>, grid, dim3(256), 0, st, a, w);
}

void launch_latent_qrope(const LatentArgs& a, const void* q, int H, int dim, void* qa, hipStream_t st) {
  if (a.T <= 0) return;
  hipLaunchKernelGGL(latent_qrope_kernel, dim3(a.T), dim3(256), 0, st, a, q, H, dim, qa);
}

void launch_latent_attn(const LatentArgs& a, const void* qa, int H, float scale, const int32_t* block_tables,
                        int max_blocks, int page, const int32_t* context_lens, const int32_t* query_start, int S,
                        void* ol, const void* cache_t, int num_pages, int window, const float* sink, int parts,
                        float* scratch, hipStream_t st) {
  if (a.T <= 0 || S <= 0) return;
  const int E = a.rank + a.rot;
  if (cache_t != nullptr && mfma_takes(a.rank, a.rot, a.f32, page)) {
    int nct, nqf;
    mfma_shape(a.rank, E, nct, nqf);
    if (parts < 1 || scratch == nullptr) parts = 1;
#define VG_LAT(NCT, NQF) if (nct == NCT && nqf == NQF) launch_mfma<NCT, NQF>(a, qa, H, scale, block_tables, max_blocks, \
    num_pages, context_lens, query_start, S, cache_t, ol, window, sink, parts, scratch, st)
    VG_LAT(8, 4); VG_LAT(8, 6); VG_LAT(16, 8); VG_LAT(16, 12); VG_LAT(32, 16); VG_LAT(32, 20);
#undef VG_LAT
    return;
  }
  int HC = H < 8 ? H : 8;
  while (HC > 1 && (HC * a.rank > 256 * MAXACC || (size_t)(HC + KT) * (E + 1) * 4 > 56 * 1024)) --HC;
  const size_t lds = ((size_t)(HC + KT) * (E + 1) + HC * KT + 3 * HC) * sizeof(float);
  hipLaunchKernelGGL(latent_attn_kernel, dim3(a.T, (H + HC - 1) / HC), dim3(256), lds, st, a, qa, H, HC, scale,
                     block_tables, max_blocks, page, context_lens, query_start, S, ol, window, sink);
}

// Decoded tokens on the MFMA kernel: how many workgroups share a sequence's key tiles (1: no split), chosen from the
// step's shape so that the launch has about two workgroups per CU, and the scratch floats their partial results take. A latent of more than
// 256 leaves room for one; fewer parts for it cost as much as they gain (us, latent 512, 12 heads, 700 keys, 512 / wg and 256 / S parts: 33
// sequences in 64 slots 25.2 and 33.9, 48 45.5 and 35.8, 64 52.6 and 47.1, 80 in 128 51.6 and 65.9, 128 90.2 and 72.8).
int latent_attn_parts(int T, int S, int H, int rank, int rot, int f32, int page) {
  if (!mfma_takes(rank, rot, f32, page) || (int64_t)T * H > 16 * (int64_t)S) return 1;
  const int wg = (T * H + 63) / 64 + S;
  const int parts = 512 / (wg > 0 ? wg : 1);
  return parts < 2 ? 1 : (parts > 8 ? 8 : parts);
}
size_t latent_attn_part_floats(int T, int S, int H, int rank, int rot, int parts) {
  if (parts <= 1) return 0;
  int nct, nqf;
  mfma_shape(rank, rank + rot, nct, nqf);
  return (size_t)parts * ((T * H + 63) / 64 + S) * 16 * (16 * nct + 2);
}

}  // namespace vgate
