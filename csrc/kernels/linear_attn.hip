// Linear attention with decay: one fp32 state matrix S [key][value] per (sequence, head) kept in a state
// slot between steps,
//   S <- diag(a_t) S + k_t v_t^T,   o_t = S^T (q_scale q_t)
// with a_t either a constant per head or sigmoid(z_t)^(1 / tau) per key channel (z fp32), optionally
// silu on q, k and v, optionally rotary positions on the leading rot_dims entries of every q / k head
// (entry i paired with i + rot_dims / 2, or 2i with 2i + 1; angle = position * inv_freq in fp32) and a key
// scale after them, then an RMS norm of o (per head, or over the concatenated heads; with or without a
// weight) and an output gate silu(g) or sigmoid(g). Key and value sizes may differ.
// Variants: the decay exp(-exp(z_t)); with a bonus u [H][D] the state is read BEFORE its update and the current
// token's own outer product enters the output through u,
//   o_t = (S_(t-1) + diag(u) k_t v_t^T)^T (q_scale q_t),   then   S_t = diag(a_t) S_(t-1) + k_t v_t^T
// (PRE instantiations of the scan: the prepared vector's fourth entry is u k); a per-head norm whose weight has one
// entry per output channel. Three launches:
//   prep   (token, head) parallel: the fp32 per-channel triples {a, k_scale k, q_scale q} and the values.
//   scan   the recurrence. Column v of S depends on no other column, so a head's value columns are split
//          into slices of 8 NC and every (sequence, head, slice) is one wave: lane = (key group of eight,
//          columns c + 8 n for n < NC), ceil(D / 8) x NC state entries in registers; per token one FMA pair
//          per entry and three lane exchanges per column for o; one LDS read of a key channel's {a, k, q}
//          serves the lane's NC columns (NC = 4 when there are enough waves without the finer split, else 1). Tokens are staged through LDS, the next batch loaded into registers
//          while the current one computes. A sequence's tokens of the step run in order from the slot's
//          state; a portion that starts at position 0 starts from zero, so a reused slot needs no clearing.
//   finish token parallel: norm, norm weight, output gate, store in the activation dtype.
// Long steps (a prompt portion of hundreds of tokens) run the scan over chunks of CH tokens in parallel:
//   local   every chunk from a zero state: its local state L_c and the product A_c of its decays
//   carry   per sequence, chunk after chunk: I_0 = slot state, I_(c+1) = diag(A_c) I_c + L_c (the same
//           recurrence taken CH tokens at a time, all fp32); the slot receives the last one
//   output  every chunk again from its true initial state I_c, now writing o
// Twice the arithmetic, but a lone sequence's dependent chain is CH tokens long instead of the whole portion.
// Decoding steps and long ones of key and value sizes up to 128 take other forms (takes_small() has the line):
//   short  sequences of few tokens (decoding) in ONE launch, a workgroup per (sequence, head): the vectors in LDS, the whole
//          state in registers (lane = four columns, key group), read and written once in whole cache lines; the update
//          does not wait for the outputs, so a token costs no barrier.
//   chunks of CT = 64 tokens, for longer portions. With g_(j..i) = a_j .. a_i per channel (1 if empty) and I the state a chunk starts from
//            o_i = (g_(1..i) q_i)^T I + sum_(j<=i) (q_i . g_(j+1..i) k_j) v_j
//            I' = g_(1..CT) I + sum_j g_(j+1..CT) k_j v_j^T
//          (with a bonus the products stop at i - 1 and the term j = i is q_i . u k_i). Every product of decays is a product
//          of factors <= 1 taken in order. local: the second sum, fp32 MFMA (16x16x4); carry as above; output: the
//          triangle of weighted products (a lane holds k_j g of four D / 32 channels and walks i), then both products
//          with fp32 MFMA, norm and gate. 2048 tokens, 8 heads of 128: 100 us, by the scan in chunks 162.
#include <algorithm>

#include "chunks.h"
#include "seq_launchers.h"

namespace vgate {
namespace {

__device__ __forceinline__ float ldx(const void* p, int64_t i, int f32) {
  return f32 ? reinterpret_cast<const float*>(p)[i] : bf2f(reinterpret_cast<const bf16_t*>(p)[i]);
}
__device__ __forceinline__ float sigm(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x * sigm(x); }
// log(sigmoid(z)) without overflow on either side
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float xor8(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));
}

// one workgroup per token: vec[t][h][d] = {a, k, q}, vals[t][h][c] = v
__global__ __launch_bounds__(256) void linear_prep_kernel(LinearAttnArgs p, float4* __restrict__ vec,
                                                           float* __restrict__ vals) {
  const int t = blockIdx.x;
  if (t >= p.query_start[p.S]) return;  // padding rows of a graph bucket
  const int HD = p.H * p.D, HV = p.H * p.V;
  const float inv_tau = 1.f / p.tau;
  const float pos = p.rot_dims > 0 ? (float)p.positions[t] : 0.f;
  const int half = p.rot_dims >> 1;
  for (int e = threadIdx.x; e < HD; e += blockDim.x) {
    float q = ldx(p.q, (int64_t)t * p.ldq + e, p.f32), k = ldx(p.k, (int64_t)t * p.ldk + e, p.f32);
    if (p.in_silu) { q = silu_f(q); k = silu_f(k); }
    const int d = e % p.D;
    if (d < p.rot_dims) {  // the pair's other entry, then (u, v) -> (u c - v s, v c + u s)
      const bool first = p.rot_half ? d < half : !(d & 1);
      const int eo = p.rot_half ? (first ? e + half : e - half) : (e ^ 1);
      float qo = ldx(p.q, (int64_t)t * p.ldq + eo, p.f32), ko = ldx(p.k, (int64_t)t * p.ldk + eo, p.f32);
      if (p.in_silu) { qo = silu_f(qo); ko = silu_f(ko); }
      const float ang = pos * p.inv_freq[p.rot_half ? (first ? d : d - half) : (d >> 1)];
      const float cs = cosf(ang), sn = sinf(ang);
      q = first ? q * cs - qo * sn : q * cs + qo * sn;
      k = first ? k * cs - ko * sn : k * cs + ko * sn;
    }
    float a;
    if (p.z == nullptr) a = p.head_decay[e / p.D];
    else if (p.decay_exp) a = expf(-expf(p.z[(int64_t)t * p.ldz + e]));
    else a = expf(log_sigmoid(p.z[(int64_t)t * p.ldz + e]) * inv_tau);
    k *= p.k_scale;
    vec[(int64_t)t * HD + e] = make_float4(a, k, q * p.q_scale, p.bonus != nullptr ? p.bonus[e] * k : 0.f);
  }
  for (int e = threadIdx.x; e < HV; e += blockDim.x) {
    const float v = ldx(p.v, (int64_t)t * p.ldv + e, p.f32);
    vals[(int64_t)t * HV + e] = p.in_silu ? silu_f(v) : v;
  }
}

// lane = 8 * q + c: key group q of 8 (keys [q dq, (q + 1) dq) with dq = ceil(D / 8) <= DQ), value column c0 + c
// MODE 0: a sequence's whole portion from its slot. MODE 1 / 2: one chunk of CH tokens per blockIdx.x (chunks
// of all sequences numbered in order), 1 = from zero, writes the chunk's local state and decay product;
// 2 = from cstate[chunk], writes the outputs.
enum { SCAN_WHOLE = 0, SCAN_LOCAL = 1, SCAN_OUTPUT = 2 };

__device__ __forceinline__ bool locate_chunk(const LinearAttnArgs& p, int CH, int bx, int& s, int& t0, int& t1) {
  int local;
  s = locate_item(p.S, bx, local, [&](int i) {
    const int a = p.query_start[i], b = p.query_start[i + 1];
    return (p.state_slots[i] < 0 || b <= a) ? 0 : (b - a + CH - 1) / CH;
  });
  if (s < 0) return false;
  t0 = p.query_start[s] + local * CH;
  t1 = min(p.query_start[s + 1], t0 + CH);
  return true;
}

template <int DQ, int TC, int NC, int MODE, bool PRE>
__global__ __launch_bounds__(64) void linear_scan_kernel(LinearAttnArgs p, const float4* __restrict__ vec,
                                                          const float* __restrict__ vals, float* __restrict__ oraw,
                                                          int CH, float* __restrict__ cstate, float* __restrict__ cdecay) {
  constexpr int QV = DQ + 1;              // padded group stride: the groups' broadcast reads hit different banks
  constexpr int NE = (8 * DQ + 63) / 64;  // channels a lane stages per token
  constexpr int CW = 8 * NC;              // value columns of a wave: lane column + 8 n, n < NC
  constexpr int NVL = (TC * CW + 63) / 64;
  __shared__ float4 lv[2][TC][8 * QV];
  __shared__ float lvv[2][TC][CW];
  const int h = blockIdx.y, c0 = blockIdx.z * CW;
  int s = blockIdx.x, t0, t1;
  if (MODE == SCAN_WHOLE) {
    t0 = p.query_start[s]; t1 = p.query_start[s + 1];
    if (p.state_slots[s] < 0 || t1 <= t0) return;
  } else if (!locate_chunk(p, CH, blockIdx.x, s, t0, t1)) {
    return;
  }
  const int D = p.D, V = p.V, lane = threadIdx.x;
  const int q = lane >> 3, cl = lane & 7;
  const int dq = (D + 7) >> 3;
  const int k0 = q * dq;
  // where this block's state starts from and goes to
  float* sp = MODE == SCAN_WHOLE ? p.state + ((int64_t)p.state_slots[s] * p.H + h) * D * V
                                 : cstate + ((int64_t)blockIdx.x * p.H + h) * D * V;
  const bool from_zero = MODE == SCAN_LOCAL ||
                         (MODE == SCAN_WHOLE && p.context_lens[s] - (t1 - t0) <= 0);
  float S[DQ][NC], A[MODE == SCAN_LOCAL ? DQ : 1];
#pragma unroll
  for (int j = 0; j < DQ; ++j) {
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int c = c0 + cl + 8 * n;
      S[j][n] = (c < V && j < dq && k0 + j < D && !from_zero) ? sp[(int64_t)(k0 + j) * V + c] : 0.f;
    }
    if (MODE == SCAN_LOCAL) A[j] = 1.f;
  }
  float4 pv[TC][NE];
  float pvv[NVL];
  auto fetch = [&](int tb) {
#pragma unroll
    for (int i = 0; i < TC; ++i)
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int d = lane + 64 * e, t = tb + i;
        const bool ok = d < D && t < t1;
        pv[i][e] = ok ? vec[((int64_t)t * p.H + h) * D + d] : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
    for (int r = 0; r < NVL; ++r) {  // TC x CW values, lane -> (token, column)
      const int e = lane + 64 * r;
      const int t = tb + e / CW, cc = c0 + e % CW;
      pvv[r] = (e < TC * CW && t < t1 && cc < V) ? vals[((int64_t)t * p.H + h) * V + cc] : 0.f;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TC; ++i)
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int d = lane + 64 * e;
        if (d < D) lv[buf][i][(d / dq) * QV + (d % dq)] = pv[i][e];
      }
#pragma unroll
    for (int r = 0; r < NVL; ++r) {
      const int e = lane + 64 * r;
      if (e < TC * CW) lvv[buf][e / CW][e % CW] = pvv[r];
    }
  };
  // entries of channels past D are zeroed once and never written: the token loops run DQ iterations with
  // no bounds test (a = k = q = 0 leaves S and o alone)
  for (int e = lane; e < 2 * TC * 8 * QV; e += 64) (&lv[0][0][0])[e] = make_float4(0.f, 0.f, 0.f, 0.f);
  __syncthreads();
  fetch(t0);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int tb = t0; tb < t1; tb += TC) {
    const bool more = tb + TC < t1;
    if (more) fetch(tb + TC);
    const int nt = min(TC, t1 - tb);
#pragma unroll
    for (int i = 0; i < TC; ++i) {
      if (i >= nt) break;
      const float4* tv = &lv[buf][i][q * QV];
      float vv[NC], o[NC];
#pragma unroll
      for (int n = 0; n < NC; ++n) { vv[n] = lvv[buf][i][cl + 8 * n]; o[n] = 0.f; }
#pragma unroll
      for (int j = 0; j < DQ; ++j) {
        const float4 x = tv[j];  // {a, k, q, u k}: one LDS read serves the lane's NC columns
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          if (PRE && MODE != SCAN_LOCAL) o[n] = fmaf(x.z, fmaf(x.w, vv[n], S[j][n]), o[n]);  // the state before its update
          S[j][n] = fmaf(x.y, vv[n], x.x * S[j][n]);
          if (!PRE && MODE != SCAN_LOCAL) o[n] = fmaf(x.z, S[j][n], o[n]);
        }
        if (MODE == SCAN_LOCAL) A[j] *= x.x;
      }
      if (MODE != SCAN_LOCAL) {
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          float r = o[n];
          r += xor8(r);
          r += xor16(r);
          r += xor32(r);
          const int c = c0 + cl + 8 * n;
          if (c < V && q == 0) oraw[((int64_t)(tb + i) * p.H + h) * V + c] = r;
        }
      }
    }
    if (more) {
      put(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
  if (MODE == SCAN_OUTPUT) return;
#pragma unroll
  for (int j = 0; j < DQ; ++j)
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int c = c0 + cl + 8 * n;
      if (c < V && j < dq && k0 + j < D) sp[(int64_t)(k0 + j) * V + c] = S[j][n];
    }
  if (MODE == SCAN_LOCAL && blockIdx.z == 0 && cl == 0) {
#pragma unroll
    for (int j = 0; j < DQ; ++j)
      if (j < dq && k0 + j < D) cdecay[((int64_t)blockIdx.x * p.H + h) * D + k0 + j] = A[MODE == SCAN_LOCAL ? j : 0];
  }
}

// one thread per (sequence, head, state entry): I_0 = slot state (zero at position 0),
// I_(c+1) = diag(A_c) I_c + L_c; cstate[c] becomes I_c, the slot the state after the last chunk
__global__ __launch_bounds__(256) void linear_carry_kernel(LinearAttnArgs p, int CH, float* __restrict__ cstate,
                                                            const float* __restrict__ cdecay) {
  const int s = blockIdx.x, h = blockIdx.y;
  const int slot = p.state_slots[s];
  const int t0 = p.query_start[s], t1 = p.query_start[s + 1];
  if (slot < 0 || t1 <= t0) return;
  const int base = count_items(s, [&](int i) {
    const int a = p.query_start[i], b = p.query_start[i + 1];
    return (p.state_slots[i] < 0 || b <= a) ? 0 : (b - a + CH - 1) / CH;
  });
  const int nc = (t1 - t0 + CH - 1) / CH;
  const int D = p.D, V = p.V;
  const bool from_zero = p.context_lens[s] - (t1 - t0) <= 0;
  float* sp = p.state + ((int64_t)slot * p.H + h) * D * V;
  for (int e = blockIdx.z * blockDim.x + threadIdx.x; e < D * V; e += gridDim.z * blockDim.x) {
    const int k = e / V;
    float cur = from_zero ? 0.f : sp[e];
    for (int c = 0; c < nc; ++c) {
      float* cs = cstate + ((int64_t)(base + c) * p.H + h) * D * V + e;
      const float loc = *cs;
      *cs = cur;
      cur = fmaf(cdecay[((int64_t)(base + c) * p.H + h) * D + k], cur, loc);
    }
    sp[e] = cur;
  }
}

// one workgroup per token; waves take heads in turn
__global__ __launch_bounds__(256) void linear_finish_kernel(LinearAttnArgs p, const float* __restrict__ oraw) {
  __shared__ float red[16];
  const int t = blockIdx.x;
  if (t >= p.query_start[p.S]) return;
  const int H = p.H, V = p.V, HV = H * V;
  const float* o = oraw + (int64_t)t * HV;
  auto emit = [&](int e, float y) {
    const float g = ldx(p.g, (int64_t)t * p.ldg + e, p.f32);
    y *= p.gate_silu ? silu_f(g) : sigm(g);
    const int64_t oi = (int64_t)t * p.ldo + e;
    if (p.f32) reinterpret_cast<float*>(p.out)[oi] = y;
    else reinterpret_cast<bf16_t*>(p.out)[oi] = f2bf(y);
  };
  if (p.norm_all) {
    float ss = 0.f;
    for (int e = threadIdx.x; e < HV; e += blockDim.x) ss = fmaf(o[e], o[e], ss);
    ss = block_reduce_sum(ss, red);
    const float inv = 1.f / sqrtf(ss / (float)HV + p.eps);
    for (int e = threadIdx.x; e < HV; e += blockDim.x) emit(e, o[e] * inv * (p.nw != nullptr ? p.nw[e] : 1.f));
    return;
  }
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int h = wv; h < H; h += 4) {
    float ss = 0.f;
    for (int c = lane; c < V; c += 64) ss = fmaf(o[h * V + c], o[h * V + c], ss);
    ss = wave_reduce_sum(ss);
    const float inv = 1.f / sqrtf(ss / (float)V + p.eps);
    for (int c = lane; c < V; c += 64)
      emit(h * V + c, o[h * V + c] * inv * (p.nw != nullptr ? p.nw[p.norm_full ? h * V + c : c] : 1.f));
  }
}

template <int DQ, int TC, int NC, bool PRE>
void launch_scan_pre(const LinearAttnArgs& a, int T, const float4* vec, const float* vals, float* oraw, int CH, float* cstate,
                 float* cdecay, hipStream_t st) {
  const int cols = (a.V + 8 * NC - 1) / (8 * NC);
  if (CH <= 0) {
    hipLaunchKernelGGL((linear_scan_kernel<DQ, TC, NC, SCAN_WHOLE, PRE>), dim3(a.S, a.H, cols), dim3(64), 0, st, a, vec, vals,
                       oraw, 0, nullptr, nullptr);
    return;
  }
  const int chunks = linear_attn_chunks(T, a.S, CH);
  hipLaunchKernelGGL((linear_scan_kernel<DQ, TC, NC, SCAN_LOCAL, false>), dim3(chunks, a.H, cols), dim3(64), 0, st, a, vec, vals,
                     oraw, CH, cstate, cdecay);
  const int ez = min(64, (a.D * a.V + 255) / 256);
  hipLaunchKernelGGL(linear_carry_kernel, dim3(a.S, a.H, ez), dim3(256), 0, st, a, CH, cstate, cdecay);
  hipLaunchKernelGGL((linear_scan_kernel<DQ, TC, NC, SCAN_OUTPUT, PRE>), dim3(chunks, a.H, cols), dim3(64), 0, st, a, vec, vals,
                     oraw, CH, cstate, cdecay);
}

template <int DQ, int TC, int NC>
void launch_scan(const LinearAttnArgs& a, int T, const float4* vec, const float* vals, float* oraw, int CH, float* cstate,
                 float* cdecay, hipStream_t st) {
  if (a.bonus != nullptr) launch_scan_pre<DQ, TC, NC, true>(a, T, vec, vals, oraw, CH, cstate, cdecay, st);
  else launch_scan_pre<DQ, TC, NC, false>(a, T, vec, vals, oraw, CH, cstate, cdecay, st);
}

// ------------------------------------------------------------------------------- key and value sizes up to 128
// decay, key (scaled) and query (scaled) of N (token, channel) pairs of head h; past t1 or D: 1, 0, 0. Every operand's loads stand
// together, from clamped addresses: behind a test per pair each would be waited for by itself (2048 tokens of 8 heads of 128: the chunks' local pass 46 -> 26 us, their output
// 60 -> 49).
template <bool F32, int N>
__device__ __forceinline__ void decay_key_query(const LinearAttnArgs& p, int h, int t1, const int (&t)[N], const int (&d)[N], float (&a)[N],
                                                float (&k)[N], float (&q)[N]) {
  constexpr int f32 = F32 ? 1 : 0;
  int64_t tt[N];
  int e[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    tt[i] = min(t[i], t1 - 1);
    e[i] = h * p.D + min(d[i], p.D - 1);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q[i] = ldx(p.q, tt[i] * p.ldq + e[i], f32);
    k[i] = ldx(p.k, tt[i] * p.ldk + e[i], f32);
  }
  if (p.z != nullptr) {
#pragma unroll
    for (int i = 0; i < N; ++i) a[i] = p.z[tt[i] * p.ldz + e[i]];
  } else {
    const float hd = p.head_decay[h];
#pragma unroll
    for (int i = 0; i < N; ++i) a[i] = hd;
  }
  if (p.in_silu) {
#pragma unroll
    for (int i = 0; i < N; ++i) { q[i] = silu_f(q[i]); k[i] = silu_f(k[i]); }
  }
  if (p.rot_dims > 0) {  // the pair's other entry, then (u, v) -> (u c - v s, v c + u s)
    const int half = p.rot_dims >> 1;
    float qo[N], ko[N], ang[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const bool turn = d[i] < p.rot_dims, first = p.rot_half ? d[i] < half : !(d[i] & 1);
      const int eo = !turn ? e[i] : (p.rot_half ? (first ? e[i] + half : e[i] - half) : (first ? e[i] + 1 : e[i] - 1));
      qo[i] = ldx(p.q, tt[i] * p.ldq + eo, f32);
      ko[i] = ldx(p.k, tt[i] * p.ldk + eo, f32);
      ang[i] = (float)p.positions[tt[i]] * p.inv_freq[!turn ? 0 : (p.rot_half ? (first ? d[i] : d[i] - half) : (d[i] >> 1))];
    }
    if (p.in_silu) {
#pragma unroll
      for (int i = 0; i < N; ++i) { qo[i] = silu_f(qo[i]); ko[i] = silu_f(ko[i]); }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (d[i] < p.rot_dims) {
        const bool first = p.rot_half ? d[i] < half : !(d[i] & 1);
        const float cs = cosf(ang[i]), sn = sinf(ang[i]);
        q[i] = first ? q[i] * cs - qo[i] * sn : q[i] * cs + qo[i] * sn;
        k[i] = first ? k[i] * cs - ko[i] * sn : k[i] * cs + ko[i] * sn;
      }
  }
  if (p.z != nullptr) {
    if (p.decay_exp) {
#pragma unroll
      for (int i = 0; i < N; ++i) a[i] = expf(-expf(a[i]));
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) a[i] = expf(log_sigmoid(a[i]) * (1.f / p.tau));
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const bool ok = t[i] < t1 && d[i] < p.D;
    a[i] = ok ? a[i] : 1.f;
    k[i] = ok ? k[i] * p.k_scale : 0.f;
    q[i] = ok ? q[i] * p.q_scale : 0.f;
  }
}
// values of N (token, channel) pairs of head h; past t1 or V: 0
template <bool F32, int N>
__device__ __forceinline__ void values_at(const LinearAttnArgs& p, int h, int t1, const int (&t)[N], const int (&c)[N], float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = ldx(p.v, (int64_t)min(t[i], t1 - 1) * p.ldv + h * p.V + min(c[i], p.V - 1), F32 ? 1 : 0);
  if (p.in_silu) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = silu_f(v[i]);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = t[i] < t1 && c[i] < p.V ? v[i] : 0.f;
}
// weight times gate of N (token, output channel) pairs of head h (past t1 or V: some other pair's)
template <bool F32, int N>
__device__ __forceinline__ void weights_gates(const LinearAttnArgs& p, int h, int t1, const int (&t)[N], const int (&c)[N], float (&y)[N]) {
  float w[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    y[i] = ldx(p.g, (int64_t)min(t[i], t1 - 1) * p.ldg + h * p.V + min(c[i], p.V - 1), F32 ? 1 : 0);
    w[i] = 1.f;
  }
  if (p.nw != nullptr) {
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = p.nw[(p.norm_full ? h * p.V : 0) + min(c[i], p.V - 1)];
  }
  if (p.gate_silu) {
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = w[i] * silu_f(y[i]);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = w[i] * sigm(y[i]);
  }
}

constexpr int ST = 8;   // tokens the short kernel stages at a time

// grid (sequence, head): sequences of at most `lim` tokens, key and value size up to P. PRE: with a bonus.
// Bound by the state's bytes once sequences x heads fill the chip: 64 sequences x 8 heads of 128 (67 MB) 16.0 us, three launches
// 35.2; a further token costs 1.1 us.
template <int P, bool F32, bool PRE>
__global__ __launch_bounds__(256) void linear_short_kernel(LinearAttnArgs p, int lim, float* __restrict__ oraw) {
  constexpr int CG = P / 4, KW = 64 / CG, KG = 4 * KW, KP = P / KG;   // column groups, key groups (of a wave; all), keys of a group
  __shared__ __attribute__((aligned(16))) float la[ST][P], lk[ST][P], lq[ST][P], lu[PRE ? ST : 1][P], lv[ST][P], lg[ST][P];
  __shared__ __attribute__((aligned(16))) float lo[ST][4][P];   // the waves' parts of the outputs
  const int s = blockIdx.x, h = blockIdx.y;
  const int slot = p.state_slots[s];
  const int t0 = p.query_start[s], t1 = p.query_start[s + 1];
  if (slot < 0 || t1 <= t0 || t1 - t0 > lim) return;
  const int D = p.D, V = p.V, tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int c = 4 * (lane % CG), k0 = KP * (wv * KW + lane / CG);
  const bool from_zero = p.context_lens[s] - (t1 - t0) <= 0;
  float* sp = p.state + ((int64_t)slot * p.H + h) * D * V;
  const bool vec4 = V % 4 == 0 && reinterpret_cast<uintptr_t>(sp) % 16 == 0;
  f32x4 S[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (from_zero || k0 + j >= D || c >= V) continue;
    const float* x = sp + (int64_t)(k0 + j) * V + c;
    if (vec4) S[j] = ld4(x);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) S[j][e] = c + e < V ? x[e] : 0.f;
  }
  for (int tb = t0; tb < t1; tb += ST) {
    if (tb > t0) __syncthreads();
    {  // 32 lanes per token; channels past D: k = q = 0, a = 1 (their state stays zero)
      constexpr int N = P / 32;
      const int i = tid >> 5, l = tid & 31;
      int t[N], d[N];
      float a[N], k[N], q[N], v[N], y[N];
#pragma unroll
      for (int m = 0; m < N; ++m) { t[m] = tb + i; d[m] = l + 32 * m; y[m] = 0.f; }
      if (t[0] < t1) {   // (uniform per half wave)
        decay_key_query<F32>(p, h, t1, t, d, a, k, q);
        values_at<F32>(p, h, t1, t, d, v);
        if (!p.norm_all) weights_gates<F32>(p, h, t1, t, d, y);
#pragma unroll
        for (int m = 0; m < N; ++m) {
          la[i][d[m]] = a[m]; lk[i][d[m]] = k[m]; lq[i][d[m]] = q[m]; lv[i][d[m]] = v[m];
          if (PRE) lu[i][d[m]] = d[m] < D ? p.bonus[h * D + d[m]] * k[m] : 0.f;
          if (!p.norm_all) lg[i][d[m]] = t[m] < t1 && d[m] < V ? y[m] : 0.f;
        }
      }
    }
    __syncthreads();
    const int nt = min(ST, t1 - tb);
    for (int i = 0; i < nt; ++i) {
      const f32x4 v = ld4(&lv[i][c]);
      f32x4 O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KP; ++j) {
        const float a = la[i][k0 + j], k = lk[i][k0 + j], q = lq[i][k0 + j];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (PRE) O[e] = fmaf(q, fmaf(lu[i][k0 + j], v[e], S[j][e]), O[e]);   // the state before its update
          S[j][e] = fmaf(k, v[e], a * S[j][e]);
          if (!PRE) O[e] = fmaf(q, S[j][e], O[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (KW >= 8) O[e] += row_rot<0x128>(O[e]);
        if (KW >= 4) O[e] += xor16(O[e]);
        O[e] += xor32(O[e]);
      }
      if (lane < CG) *reinterpret_cast<f32x4*>(&lo[i][wv][c]) = O;
    }
    __syncthreads();
    {  // the outputs of the staged tokens: head norm, weight, gate; raw where the norm spans the heads
      const int i = tid >> 5, l = tid & 31, t = tb + i;
      float o[P / 32], ss = 0.f;
#pragma unroll
      for (int m = 0; m < P / 32; ++m) {
        const int d = l + 32 * m;
        o[m] = lo[i][0][d] + lo[i][1][d] + (lo[i][2][d] + lo[i][3][d]);   // (columns past V are zero)
        ss = fmaf(o[m], o[m], ss);
      }
      const float inv = 1.f / sqrtf(half_sum(ss) / (float)V + p.eps);
#pragma unroll
      for (int m = 0; m < P / 32; ++m) {
        const int d = l + 32 * m;
        if (t >= t1 || d >= V) continue;
        if (p.norm_all) {
          oraw[((int64_t)t * p.H + h) * V + d] = o[m];
          continue;
        }
        const float y = o[m] * inv * lg[i][d];
        const int64_t oi = (int64_t)t * p.ldo + h * V + d;
        if (F32) reinterpret_cast<float*>(p.out)[oi] = y;
        else reinterpret_cast<bf16_t*>(p.out)[oi] = f2bf(y);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    if (k0 + j >= D || c >= V) continue;
    float* x = sp + (int64_t)(k0 + j) * V + c;
    if (vec4) *reinterpret_cast<f32x4*>(x) = S[j];
    else
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < V) x[e] = S[j][e];
  }
}

constexpr int CT = 64;         // tokens of a chunk
constexpr int CTP = CT + 4;    // padded rows of tokens: 16 lanes' 16-B pieces of 16 rows fall into all 64 banks

// grid (chunk, head): cstate[chunk][h] = sum_j g_(j+1..CT) k_j v_j^T [D][V], cdecay = g_(1..CT). MFMA operands: the token
// 16 n + 4 kg + e is element e of lane group kg in both operands, so a lane's four steps are one 16-B piece of a row.
template <int DP, bool F32>
__global__ __launch_bounds__(256) void linear_local_kernel(LinearAttnArgs p, int lim, float* __restrict__ cstate,
                                                            float* __restrict__ cdecay) {
  constexpr int DT = (DP / 16 + 3) / 4;   // channel tiles of a wave
  __shared__ __attribute__((aligned(16))) float kt[DP][CTP], vt[128][CTP];
  __shared__ float late[DP];
  int s, t0, t1;
  if (!locate_chunk<CT>(p.query_start, p.state_slots, p.S, lim, blockIdx.x, s, t0, t1)) return;
  const int h = blockIdx.y, D = p.D, V = p.V, tid = threadIdx.x;
  const int half = tid >> 7, j0 = half * (CT / 2);
  {
    const int d = tid & 127;
    float k[CT / 2], g = 1.f;
    if (d < DP) {   // from the half's last token to its first: k_j times the decays after it
      float a[CT / 2];
#pragma unroll
      for (int j = 0; j < CT / 2; j += 8) {
        int t[8], dd[8];
        float an[8], kn[8], qn[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) { t[e] = t0 + j0 + j + e; dd[e] = d; }
        decay_key_query<F32>(p, h, t1, t, dd, an, kn, qn);
#pragma unroll
        for (int e = 0; e < 8; ++e) { a[j + e] = an[e]; k[j + e] = kn[e]; }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = CT / 2 - 1; j >= 0; --j) {
        k[j] *= g;
        g *= a[j];
      }
      if (half == 1) late[d] = g;
    }
#pragma unroll
    for (int j = 0; j < CT / 2; j += 8) {   // values, a column per thread
      int t[8], c[8];
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) { t[e] = t0 + j0 + j + e; c[e] = d; }
      values_at<F32>(p, h, t1, t, c, v);
      *reinterpret_cast<f32x4*>(&vt[d][j0 + j]) = f32x4{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<f32x4*>(&vt[d][j0 + j + 4]) = f32x4{v[4], v[5], v[6], v[7]};
    }
    __syncthreads();
    if (d < DP) {
      const float f = half == 0 ? late[d] : 1.f;
#pragma unroll
      for (int j = 0; j < CT / 2; j += 4)
        *reinterpret_cast<f32x4*>(&kt[d][j0 + j]) = f32x4{k[j] * f, k[j + 1] * f, k[j + 2] * f, k[j + 3] * f};
      if (half == 0 && d < D) cdecay[((int64_t)blockIdx.x * p.H + h) * D + d] = g * f;
    }
  }
  __syncthreads();
  const int w = tid >> 6, l = tid & 63, lr = l & 15, kg = l >> 4;
  float* cs = cstate + ((int64_t)blockIdx.x * p.H + h) * D * V;
  f32x4 acc[DT][8];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < CT / 16; ++n) {
    f32x4 A[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) A[t] = ld4(&kt[min(16 * (w * DT + t), DP - 16) + lr][16 * n + 4 * kg]);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (16 * u >= V) continue;
      const f32x4 B = ld4(&vt[16 * u + lr][16 * n + 4 * kg]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[t][e], B[e], acc[t][u], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * (w * DT + t) + 4 * kg + i, c = 16 * u + lr;
        if (d < D && c < V) cs[(int64_t)d * V + c] = acc[t][u][i];
      }
}

// grid (sequence, head, stretches of 256 state entries): as linear_carry_kernel, over the chunks of CT tokens; eight chunks'
// local states are asked for at a time
__global__ __launch_bounds__(256) void linear_chunk_carry_kernel(LinearAttnArgs p, int lim, float* __restrict__ cstate,
                                                                  const float* __restrict__ cdecay) {
  const int s = blockIdx.x, h = blockIdx.y;
  const int slot = p.state_slots[s];
  const int t0 = p.query_start[s], t1 = p.query_start[s + 1];
  if (slot < 0 || t1 - t0 <= lim) return;
  const int64_t c0 = first_chunk<CT>(p.query_start, p.state_slots, lim, s);   // (whole waves)
  const int D = p.D, V = p.V, e = blockIdx.z * 256 + threadIdx.x;
  if (e >= D * V) return;
  const int nc = (t1 - t0 + CT - 1) / CT;
  float* sp = p.state + ((int64_t)slot * p.H + h) * D * V;
  const int64_t step = (int64_t)p.H * D * V, dstep = (int64_t)p.H * D;
  float* cs = cstate + (c0 * p.H + h) * D * V + e;
  const float* cd = cdecay + (c0 * p.H + h) * D + e / V;
  float cur = p.context_lens[s] - (t1 - t0) <= 0 ? 0.f : sp[e];
  for (int c = 0; c < nc; c += 8) {
    float loc[8], dec[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = min(c + i, nc - 1);
      loc[i] = cs[j * step];
      dec[i] = cd[j * dstep];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (c + i < nc) {
        cs[(c + i) * step] = cur;
        cur = fmaf(dec[i], cur, loc[i]);
      }
  }
  sp[e] = cur;
}

// grid (chunk, head), 512 threads: the outputs of a chunk from the state it starts from. Wave w owns the columns 16 w ..
// Bound by chains through LDS with two waves per SIMD, the triangle's rows first: a row's operands are asked for a row ahead, and the decays'
// products read their 16 tokens together (29 chunks of 8 heads of 128: 43.5 -> 37.0 us).
template <int DP, bool F32, bool PRE>
__global__ __launch_bounds__(512) void linear_output_kernel(LinearAttnArgs p, int lim, const float* __restrict__ cstate,
                                                             float* __restrict__ oraw) {
  constexpr int X = DP / 32, NT = DP / 16, DS = DP + 4;   // (padded rows, as CTP)
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* la = lds;                    // [CT][DS] decays
  float* lk = la + CT * DS;           // keys
  float* lq = lk + CT * DS;           // queries, then times the decays up to them
  float* tr = lq + CT * DS;           // [CT][CTP] the triangle
  float* red = tr + CT * CTP;         // [8][CT] rows' sums of squares; before, [4][DP] decays of 16 tokens
  int s, t0, t1;
  if (!locate_chunk<CT>(p.query_start, p.state_slots, p.S, lim, blockIdx.x, s, t0, t1)) return;
  const int h = blockIdx.y, D = p.D, V = p.V, tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, lr = l & 15, kg = l >> 4;
  const int col = 16 * w + lr;
  const bool con = col < V;
  // B operands straight from memory: the state (channels 16 n + 4 kg + e) and the values (tokens 16 n + 4 kg + e) of the column
  f32x4 B[NT], vb[CT / 16];
  const float* cs = cstate + ((int64_t)blockIdx.x * p.H + h) * D * V;
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = 16 * n + 4 * kg + e;
      B[n][e] = con && d < D ? cs[(int64_t)d * V + col] : 0.f;
    }
  {
    int t[CT / 4], c[CT / 4];
    float v[CT / 4];
#pragma unroll
    for (int u = 0; u < CT / 4; ++u) { t[u] = t0 + 16 * (u / 4) + 4 * kg + u % 4; c[u] = col; }
    values_at<F32>(p, h, t1, t, c, v);
#pragma unroll
    for (int u = 0; u < CT / 4; ++u) vb[u / 4][u % 4] = v[u];
  }
  constexpr int PT = CT * DP / 512, PB = PT < 8 ? PT : 8;   // (token, channel) pairs of a thread, and of a batch
#pragma unroll
  for (int m = 0; m < PT; m += PB) {
    int t[PB], dd[PB];
    float a[PB], k[PB], q[PB];
#pragma unroll
    for (int u = 0; u < PB; ++u) { t[u] = t0 + (tid + 512 * (m + u)) / DP; dd[u] = tid % DP; }
    decay_key_query<F32>(p, h, t1, t, dd, a, k, q);
#pragma unroll
    for (int u = 0; u < PB; ++u) {
      const int at = (t[u] - t0) * DS + dd[u];
      la[at] = a[u]; lk[at] = k[u]; lq[at] = q[u];
    }
  }
  for (int e = tid; e < CT * CTP; e += 512) tr[e] = 0.f;
  __syncthreads();
  {  // the triangle: a wave owns eight columns j, lane = (channel group dg of eight, j). A column has CT - j rows: waves w and
     // w + 4, which share a SIMD, take stretches that add up alike
    const int jb = w < 4 ? w : 11 - w;
    const int dg = l >> 3, j = 8 * jb + (l & 7);
    float x[4 * X], diag = 0.f;
#pragma unroll
    for (int m = 0; m < X; ++m)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int d = 32 * m + 4 * dg + c;
        x[4 * m + c] = lk[j * DS + d];
        if (PRE) diag = fmaf(lq[j * DS + d] * (d < D ? p.bonus[h * D + d] : 0.f), x[4 * m + c], diag);
      }
    if (PRE) diag = key_sum<8>(diag);
    f32x4 na[X], nq[X];   // the next row's, asked for a row ahead (past the last: the last)
    auto row = [&](int i) {
#pragma unroll
      for (int m = 0; m < X; ++m) {
        na[m] = ld4(&la[i * DS + 32 * m + 4 * dg]);
        nq[m] = ld4(&lq[i * DS + 32 * m + 4 * dg]);
      }
    };
    row(8 * jb);
    for (int i = 8 * jb; i < CT; ++i) {
      float r = 0.f;
      f32x4 a[X], q[X];
#pragma unroll
      for (int m = 0; m < X; ++m) { a[m] = na[m]; q[m] = nq[m]; }
      row(min(i + 1, CT - 1));
#pragma unroll
      for (int m = 0; m < X; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (PRE) r = fmaf(q[m][c], x[4 * m + c], r);
          if (i > j) x[4 * m + c] *= a[m][c];
          if (!PRE) r = fmaf(q[m][c], x[4 * m + c], r);
        }
      r = key_sum<8>(r);
      if (PRE && i == j) r = diag;
      if (dg == 0 && i >= j) tr[i * CTP + j] = r;
    }
  }
  __syncthreads();
  {  // q_i g_(1..i) (with a bonus g_(1..i-1)) in place: a channel and 16 tokens per thread
    const int d = tid & 127, part = tid >> 7;
    float g = 1.f, a[16], q[16];   // (read together: a store between them would order the reads)
    if (d < DP) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        a[i] = la[(16 * part + i) * DS + d];
        q[i] = lq[(16 * part + i) * DS + d];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (!PRE) g *= a[i];
        q[i] *= g;
        if (PRE) g *= a[i];
      }
      red[part * DP + d] = g;
    }
    __syncthreads();
    if (d < DP) {
      if (part > 0) {
        float f = 1.f;
        for (int m = 0; m < part; ++m) f *= red[m * DP + d];
#pragma unroll
        for (int i = 0; i < 16; ++i) q[i] *= f;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) lq[(16 * part + i) * DS + d] = q[i];
    }
  }
  __syncthreads();
  f32x4 acc[CT / 16];
#pragma unroll
  for (int r = 0; r < CT / 16; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    f32x4 A[CT / 16];
#pragma unroll
    for (int r = 0; r < CT / 16; ++r) A[r] = ld4(&lq[(16 * r + lr) * DS + 16 * n + 4 * kg]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int r = 0; r < CT / 16; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[r][e], B[n][e], acc[r], 0, 0, 0);
  }
#pragma unroll
  for (int n = 0; n < CT / 16; ++n) {
    f32x4 A[CT / 16];
#pragma unroll
    for (int r = n; r < CT / 16; ++r) A[r] = ld4(&tr[(16 * r + lr) * CTP + 16 * n + 4 * kg]);
    // the zeros above the diagonal would turn an infinity or a NaN into NaN for the tokens before it: such a block goes term by term
    const f32x4 z = vb[n] * 0.f;
    const bool finite = __all(z[0] + z[1] + (z[2] + z[3]) == 0.f);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int r = n; r < CT / 16; ++r)
        if (r > n || finite) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[r][e], vb[n][e], acc[r], 0, 0, 0);
    if (!finite)
      for (int j = 0; j < 16; ++j) {
        const int from = lr + 16 * (j / 4);
        const float v0 = __shfl(vb[n][0], from, 64), v1 = __shfl(vb[n][1], from, 64), v2 = __shfl(vb[n][2], from, 64), v3 = __shfl(vb[n][3], from, 64);
        const float v = j % 4 == 0 ? v0 : (j % 4 == 1 ? v1 : (j % 4 == 2 ? v2 : v3));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (j <= 4 * kg + i) acc[n][i] = fmaf(tr[(16 * n + 4 * kg + i) * CTP + 16 * n + j], v, acc[n][i]);
      }
  }
  // acc[r][i]: token 16 r + 4 kg + i, column col (columns past V are zero)
  if (p.norm_all) {
#pragma unroll
    for (int r = 0; r < CT / 16; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = t0 + 16 * r + 4 * kg + i;
        if (con && t < t1) oraw[((int64_t)t * p.H + h) * V + col] = acc[r][i];
      }
    return;
  }
  float wg[CT / 4];
  {
    int t[CT / 4], c[CT / 4];
#pragma unroll
    for (int u = 0; u < CT / 4; ++u) { t[u] = t0 + 16 * (u / 4) + 4 * kg + u % 4; c[u] = col; }
    weights_gates<F32>(p, h, t1, t, c, wg);
  }
#pragma unroll
  for (int r = 0; r < CT / 16; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float ss = acc[r][i] * acc[r][i];
      ss += row_rot<0x128>(ss);
      ss += row_rot<0x124>(ss);
      ss += row_rot<0x122>(ss);
      ss += row_rot<0x121>(ss);
      if (lr == 0) red[w * CT + 16 * r + 4 * kg + i] = ss;
    }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < CT / 16; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * r + 4 * kg + i, t = t0 + row;
      if (!con || t >= t1) continue;
      float ss = 0.f;
#pragma unroll
      for (int m = 0; m < 8; ++m) ss += red[m * CT + row];
      const float y = acc[r][i] * (1.f / sqrtf(ss / (float)V + p.eps)) * wg[4 * r + i];
      const int64_t oi = (int64_t)t * p.ldo + h * V + col;
      if (F32) reinterpret_cast<float*>(p.out)[oi] = y;
      else reinterpret_cast<bf16_t*>(p.out)[oi] = f2bf(y);
    }
}

// Tokens a sequence may have in a step to be run one by one: a chunk of 64 costs what 50 tokens do, and its three launches more. Decoding
// steps (T <= S), and short ones that may nearly be, take one launch (8 heads of 128, in parentheses with empty or few chunks: 128
// sequences 32 us (53), 256 61 (98); 63 decoded tokens beside a portion of 65 95 (146), 127 beside 65 103 (169), beside 129 183 (170)).
int short_limit(int T, int S) { return T <= std::max(S, 96) || T <= std::min(2 * S, 256) ? T : 64; }
// chunks of a step whose sequences longer than lim tokens have T between them: each has at most one that is not whole. (Workgroups past
// the last chunk leave at once, but push real ones together on fewer CUs: 20 + 700 tokens, 16 heads of 128, with 22 of them per head 127 us,
// without 118.)
int long_chunks(int T, int S, int lim) { return T <= lim ? 0 : (T + std::min(S, T / (lim + 1)) * (CT - 1)) / CT; }
// Decoding steps: one launch instead of three (16 sequences x 8 heads of 128: 25.3 -> 12.2 us). Long steps: chunks with fp32 MFMA
// (2048 tokens 162 -> 100 us, 63 decoded tokens beside a portion of 961 1054 -> 169, 64 portions of 16 62 -> 47). Between them
// the scan below, which spreads a head's columns over several workgroups, is ahead where sequences are few: one portion of
// 96 78 us (here 96; of 128 98 against 84), 8 of 48 54 (59), and where sequences x heads are few besides (16 of 48, 4 heads: 50, here 54).
// With key sizes up to 64 a token of the scan costs half as much, and a long step's own chunks there spread better than the MFMA ones:
// those are ahead where portions are long on average only while their workgroups fill the chip about once (us, scan / MFMA chunks, heads of
// 64: 2048 tokens, 8 heads 98, 68; 16 heads 115, 123; 32 heads 144, 229; 512 tokens, 8 heads 54, 60; 4 x 400, 4 heads 80, 63, 16 heads 103, 123,
// 32 heads 134, 229; 20 + 700, 8 heads 58, 75).
bool takes_small(int T, int S, int H, int D, int V) {
  if (D > 128 || V > 128) return false;
  if (T <= 2 * S) return true;
  if (T < (S == 1 ? 128 : (S < 16 ? 512 : 256)) || (T < 64 * S && S * H < 128)) return false;
  if (D > 64 || T < 96 * S) return true;
  if (S == 1 && T < 256) return T >= 160;   // (the scan has no chunks below 256 tokens)
  const bool tiny = D <= 32 && V <= 32;
  const int64_t work = (int64_t)T * H;      // (a workgroup per 64)
  if (S == 1) return work >= (tiny ? 12288 : 8192) && work <= 16384;
  if (S == 2) return !tiny && work >= 8192 && work <= 16000;
  return work >= (tiny ? 8000 : 4000) && work <= 16000;
}

template <int DP, bool F32, bool PRE>
void launch_small(const LinearAttnArgs& a, int T, const LinearPlan& plan, float* oraw, float* cstate, float* cdecay, hipStream_t st) {
  const int P = max(a.D, a.V), lim = plan.lim, chunks = plan.chunks;
  if (lim > 0) {
    const dim3 grid(a.S, a.H);
    if (P <= 32) hipLaunchKernelGGL((linear_short_kernel<32, F32, PRE>), grid, dim3(256), 0, st, a, lim, oraw);
    else if (P <= 64) hipLaunchKernelGGL((linear_short_kernel<64, F32, PRE>), grid, dim3(256), 0, st, a, lim, oraw);
    else hipLaunchKernelGGL((linear_short_kernel<128, F32, PRE>), grid, dim3(256), 0, st, a, lim, oraw);
  }
  if (chunks > 0) {
    constexpr size_t bytes = ((size_t)3 * CT * (DP + 4) + CT * CTP + 8 * CT) * 4;
    auto out = linear_output_kernel<DP, F32, PRE>;
    static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(out), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)bytes) == hipSuccess;
    (void)attr;
    hipLaunchKernelGGL((linear_local_kernel<DP, F32>), dim3(chunks, a.H), dim3(256), 0, st, a, lim, cstate, cdecay);
    hipLaunchKernelGGL(linear_chunk_carry_kernel, dim3(a.S, a.H, (a.D * a.V + 255) / 256), dim3(256), 0, st, a, lim, cstate, cdecay);
    hipLaunchKernelGGL(out, dim3(chunks, a.H), dim3(512), bytes, st, a, lim, cstate, oraw);
  }
  if (a.norm_all) hipLaunchKernelGGL(linear_finish_kernel, dim3(T), dim3(256), 0, st, a, oraw);
}

template <int DP>
void launch_small_dp(const LinearAttnArgs& a, int T, const LinearPlan& plan, float* oraw, float* cstate, float* cdecay, hipStream_t st) {
  if (a.f32) {
    if (a.bonus != nullptr) launch_small<DP, true, true>(a, T, plan, oraw, cstate, cdecay, st);
    else launch_small<DP, true, false>(a, T, plan, oraw, cstate, cdecay, st);
  } else {
    if (a.bonus != nullptr) launch_small<DP, false, true>(a, T, plan, oraw, cstate, cdecay, st);
    else launch_small<DP, false, false>(a, T, plan, oraw, cstate, cdecay, st);
  }
}

}  // namespace

int linear_attn_chunk_size(int T, int S) {
  // steps of a few tokens per sequence (decoding, short portions): one pass per sequence; long ones: chunks
  return T >= 256 && T >= 64 * S ? 64 : 0;
}
int linear_attn_chunks(int T, int S, int CH) { return CH > 0 ? T / CH + S : 0; }
LinearPlan linear_attn_plan(int T, int S, int H, int D, int V) {
  const int lim = short_limit(T, S);
  // T counts padding rows too, so a sequence may be much shorter. A lone one then takes chunks whatever its length (not more
  // of them than any step of T rows); several are told apart by their lengths on the device.
  const bool lone = S == 1 && T > lim;
  return {takes_small(T, S, H, D, V), lone ? 0 : lim, lone ? (T + CT - 1) / CT : long_chunks(T, S, lim)};
}
size_t linear_attn_scratch_floats(int T, int S, int H, int D, int V) {
  const int CH = linear_attn_chunk_size(T, S);
  const size_t any = (size_t)T * H * (4 * D + 2 * V) + (size_t)linear_attn_chunks(T, S, CH) * H * D * (V + 1);
  const LinearPlan plan = linear_attn_plan(T, S, H, D, V);
  const size_t small = (size_t)T * H * V + (size_t)plan.chunks * H * D * (V + 1);
  return plan.small && small > any ? small : any;
}

// scratch: linear_attn_scratch_floats(): {a, k, q, -} per key channel, the values, the raw outputs, and for
// chunked steps every chunk's state and decay product
void launch_linear_attn(const LinearAttnArgs& a, int T, float* scratch, hipStream_t st) {
  if (a.S <= 0 || a.H <= 0 || T <= 0) return;
  const int64_t nk = (int64_t)T * a.H * a.D, nv = (int64_t)T * a.H * a.V;
  const LinearPlan plan = linear_attn_plan(T, a.S, a.H, a.D, a.V);
  if (plan.small && a.cols_per_lane == 0) {   // scratch: raw outputs, the chunks' states, their decays
    float* states = scratch + nv;
    float* decays = states + (size_t)plan.chunks * a.H * a.D * a.V;
    if (a.D <= 32) launch_small_dp<32>(a, T, plan, scratch, states, decays, st);
    else if (a.D <= 64) launch_small_dp<64>(a, T, plan, scratch, states, decays, st);
    else launch_small_dp<128>(a, T, plan, scratch, states, decays, st);
    return;
  }
  float4* vec = reinterpret_cast<float4*>(scratch);
  float* vals = scratch + 4 * nk;
  float* oraw = vals + nv;
  const int CH = linear_attn_chunk_size(T, a.S);
  float* cstate = oraw + nv;
  float* cdecay = cstate + (size_t)linear_attn_chunks(T, a.S, CH) * a.H * a.D * a.V;
  hipLaunchKernelGGL(linear_prep_kernel, dim3(T), dim3(256), 0, st, a, vec, vals);
  // columns per lane: few columns -> more waves (a small batch of decoded tokens needs them to fill the chip);
  // wide values -> every LDS read of a key channel's {a, k, q} serves four columns
  const bool wide = a.cols_per_lane > 0 ? a.cols_per_lane > 1
                                        : a.V >= 32 && (int64_t)a.S * a.H * ((a.V + 31) / 32) * (CH > 0 ? T / CH + 1 : 1) >= 512;
  if (a.D <= 32) { if (wide) launch_scan<4, 8, 4>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); else launch_scan<4, 8, 1>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); }
  else if (a.D <= 64) { if (wide) launch_scan<8, 8, 4>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); else launch_scan<8, 8, 1>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); }
  else if (a.D <= 128) { if (wide) launch_scan<16, 4, 4>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); else launch_scan<16, 4, 1>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); }
  else { if (wide) launch_scan<32, 4, 2>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); else launch_scan<32, 4, 1>(a, T, vec, vals, oraw, CH, cstate, cdecay, st); }
  hipLaunchKernelGGL(linear_finish_kernel, dim3(T), dim3(256), 0, st, a, oraw);
}

}  // namespace vgate
