// Generalized delta rule with per-channel decay, one fp32 state matrix S [key][value] per (sequence,
// head) kept in a state slot between steps:
//   w = exp(-c * sigmoid(wl + w0))        per key channel decay
//   a = sigmoid(al + ab)                  per key channel removal rate
//   u = k / sqrt(sum(k^2) + unit_eps)
//   S <- diag(w) S - (a * u) (u^T S) + k v^T        (both correction terms read the old S)
//   o  = S^T r;  out = o / rms(o) * nw * sigmoid(g)  (rms over the head)
// Sequences with few tokens in the step (decoding) run them one after another, one workgroup per (sequence, head) and one launch
// for everything (delta_short_kernel): the whole state sits in registers (lane = four columns, key group), is read and
// written once in whole cache lines, and since
//   o = (w r)^T S_old - (b . r) (u^T S_old) + (k . r) v,      b = a u
// both sums over keys are of the old state and take one exchange per token. A sequence's tokens run in order from the
// slot's state; a portion that starts at position 0 starts from zero, so a reused slot needs no clearing.
// Prompt portions take chunks of CN = 32 tokens at once. With b_i = a_i u_i, k_i = n_i u_i (n_i the key's length), S the state a
// chunk starts from, g_(j..i) = w_j .. w_i per channel (1 if empty) and p_i = u_i^T S_(i-1) what token i takes away,
//   S_i = g_(1..i) S + sum_(j<=i) g_(j+1..i) (k_j v_j^T - b_j p_j^T)
// so the p of a chunk solve a unit lower triangular system whose matrix does not involve S:
//   p_i + sum_(j<i) (u_i . g_(j+1..i-1) b_j) p_j = (g_(1..i-1) u_i)^T S + sum_(j<i) (u_i . g_(j+1..i-1) k_j) v_j
// i.e. p = W S + y, and with R = g_(1..i) r_i,  o_i = (R_i - sum_(j<=i) (r_i . g_(j+1..i) b_j) W_j) S + (the same sums of v and y),
//   S <- g_(1..CN) S + sum_j g_(j+1..CN) (k_j v_j^T - b_j p_j^T).
// Every product of decays is a product of factors <= 1 taken in order (nothing is divided by a decay). Three launches, all fp32:
//   chunk  (chunk, head) parallel: the tokens' vectors in LDS, the four triangles (a lane holds b_j g and u_j g of four D / 32
//          channels and walks i), the solve with one column of [W | y] per thread.
//   chunk scan    the only sequential part: per (sequence, head, 16 columns) [W; Q] S and the update as fp32 MFMA (16x16x4);
//          S stays in registers (C layout) and goes round through LDS as B operand; the part of the update that only
//          needs v runs before the wait for p.
//   chunk finish  norm and gate, from the scan's [column][token] tiles.
// Portions in between, of few sequences (takes_scan() has the lines), take three launches of another kind:
//   prep   (token, head) parallel: the per-channel fp32 vectors {w, a u, k, r} and u of every token.
//   scan   the recurrence token by token. Column v of S depends on no other, so a wave owns 8 of a head's value columns: lane =
//          (key group of eight, column), D / 8 state entries in registers, the sums over keys D / 8 FMAs and three lane
//          exchanges. The dependent chain of a token is what bounds it. Tokens are staged through LDS eight at a time, the next eight
//          loaded while the current ones compute.
//   finish (token, head) parallel: head norm, weight, gate.
// 2048 tokens, 8 heads of 128: 69 + 112 + 13 us; the tokens one after another (three launches, one wave per 8 columns) took
// 1060 us, 0.5 us of chain per token. What bounds the chunk scan is its 64 MFMAs per wave and two barriers per 32 tokens.
#include <algorithm>

#include "chunks.h"
#include "seq_launchers.h"

namespace vgate {
namespace {

__device__ __forceinline__ float ldx(const void* p, int64_t i, int f32) {
  return f32 ? reinterpret_cast<const float*>(p)[i] : bf2f(reinterpret_cast<const bf16_t*>(p)[i]);
}
__device__ __forceinline__ float sigm(float x) { return 1.f / (1.f + expf(-x)); }

constexpr int TC = 8;  // tokens staged in LDS at a time

// grid (sequence, head): sequences of at most `lim` tokens, head size up to DP. Bound by the state's bytes once sequences x
// heads fill the chip: 32 sequences x 8 heads of 128 (34 MB) 14.8 us; before, in three launches of which the scan read the
// state in 32-B pieces, 58 us. Further tokens take 1.35 us each: 320 VALU operations and one barrier per wave.
template <int DP, bool F32>
__global__ __launch_bounds__(256) void delta_short_kernel(DeltaArgs p, int lim) {
  constexpr int CG = DP / 4, KW = 64 / CG, KG = 4 * KW, KP = DP / KG;   // column groups, key groups (of a wave; all), keys of a group
  constexpr int f32 = F32 ? 1 : 0;
  __shared__ __attribute__((aligned(16))) float lu[TC][DP], lw[TC][DP], lwr[TC][DP], lb[TC][DP], lv[TC][DP], lg[TC][DP];
  __shared__ float len[TC], br[TC], kr[TC];
  __shared__ __attribute__((aligned(16))) float lp[TC][4][DP], lo[TC][4][DP];   // the waves' parts of u^T S and (w r)^T S
  const int s = blockIdx.x, h = blockIdx.y;
  const int slot = p.state_slots[s];
  const int t0 = p.query_start[s], t1 = p.query_start[s + 1];
  if (slot < 0 || t1 <= t0 || t1 - t0 > lim) return;
  const int D = p.D, tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int c = 4 * (lane % CG), k0 = KP * (wv * KW + lane / CG);
  const bool from_zero = p.context_lens[s] - (t1 - t0) <= 0;
  float* sp = p.state + ((int64_t)slot * p.H + h) * D * D;
  const bool vec4 = D % 4 == 0 && reinterpret_cast<uintptr_t>(sp) % 16 == 0;
  f32x4 S[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (from_zero || k0 + j >= D || c >= D) continue;
    const float* q = sp + (int64_t)(k0 + j) * D + c;
    if (vec4) S[j] = ld4(q);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) S[j][e] = c + e < D ? q[e] : 0.f;
  }
  for (int tb = t0; tb < t1; tb += TC) {
    if (tb > t0) __syncthreads();
    {  // 32 lanes per token; channels past D and tokens past the end: u = b = r = v = 0, w = 1
      const int i = tid >> 5, l = tid & 31, t = tb + i;
      float k[DP / 32], r[DP / 32], a[DP / 32], ss = 0.f;
#pragma unroll
      for (int m = 0; m < DP / 32; ++m) {
        const int d = l + 32 * m, ch = h * D + d;
        const bool ok = t < t1 && d < D;
        const int64_t ix = (int64_t)t * p.ld + ch;
        k[m] = ok ? ldx(p.k, ix, f32) : 0.f;
        r[m] = ok ? ldx(p.r, ix, f32) : 0.f;
        a[m] = ok ? sigm(ldx(p.a, ix, f32) + p.ab[ch]) : 0.f;
        const float w = ok ? expf(-p.decay_c * sigm(ldx(p.wl, (int64_t)t * p.ldw + ch, f32) + p.w0[ch])) : 1.f;
        lw[i][d] = w;
        lwr[i][d] = w * r[m];
        lv[i][d] = ok ? ldx(p.v, ix, f32) : 0.f;
        lg[i][d] = ok ? p.nw[ch] * sigm(ldx(p.g, ix, f32)) : 0.f;
        ss = fmaf(k[m], k[m], ss);
      }
      const float n = sqrtf(half_sum(ss) + p.unit_eps), f = t < t1 ? 1.f / n : 0.f;
      float sb = 0.f, sk = 0.f;
#pragma unroll
      for (int m = 0; m < DP / 32; ++m) {
        const float u = k[m] * f, b = a[m] * u;
        lu[i][l + 32 * m] = u;
        lb[i][l + 32 * m] = b;
        sb = fmaf(b, r[m], sb);
        sk = fmaf(k[m], r[m], sk);
      }
      sb = half_sum(sb);
      sk = half_sum(sk);
      if (l == 0) { len[i] = n; br[i] = sb; kr[i] = sk; }
    }
    __syncthreads();
    const int nt = min(TC, t1 - tb);
    for (int i = 0; i < nt; ++i) {
      f32x4 P = {0.f, 0.f, 0.f, 0.f}, O = P;
      float u[KP], w[KP], b[KP];
#pragma unroll
      for (int j = 0; j < KP; ++j) {
        u[j] = lu[i][k0 + j];
        w[j] = lw[i][k0 + j];
        b[j] = lb[i][k0 + j];
        const float wr = lwr[i][k0 + j];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          P[e] = fmaf(u[j], S[j][e], P[e]);
          O[e] = fmaf(wr, S[j][e], O[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (KW >= 8) { P[e] += row_rot<0x128>(P[e]); O[e] += row_rot<0x128>(O[e]); }
        if (KW >= 4) { P[e] += xor16(P[e]); O[e] += xor16(O[e]); }
        P[e] += xor32(P[e]);
        O[e] += xor32(O[e]);
      }
      if (lane < CG) {
        *reinterpret_cast<f32x4*>(&lp[i][wv][c]) = P;
        *reinterpret_cast<f32x4*>(&lo[i][wv][c]) = O;
      }
      lds_barrier();
      P = ld4(&lp[i][0][c]) + ld4(&lp[i][1][c]) + (ld4(&lp[i][2][c]) + ld4(&lp[i][3][c]));
      const f32x4 nv = ld4(&lv[i][c]) * len[i];
#pragma unroll
      for (int j = 0; j < KP; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[j][e] = fmaf(u[j], nv[e], fmaf(-b[j], P[e], w[j] * S[j][e]));
    }
    __syncthreads();
    {  // the outputs of the staged tokens: head norm, weight, gate (columns past D are zero)
      const int i = tid >> 5, l = tid & 31, t = tb + i;
      float o[DP / 32], ss = 0.f;
#pragma unroll
      for (int m = 0; m < DP / 32; ++m) {
        const int d = l + 32 * m;
        const float P = lp[i][0][d] + lp[i][1][d] + (lp[i][2][d] + lp[i][3][d]);
        const float O = lo[i][0][d] + lo[i][1][d] + (lo[i][2][d] + lo[i][3][d]);
        o[m] = fmaf(kr[i], lv[i][d], fmaf(-br[i], P, O));
        ss = fmaf(o[m], o[m], ss);
      }
      const float inv = 1.f / sqrtf(half_sum(ss) / (float)D + p.eps);
#pragma unroll
      for (int m = 0; m < DP / 32; ++m) {
        const int d = l + 32 * m;
        if (t >= t1 || d >= D) continue;
        const int64_t oi = (int64_t)t * p.ldo + h * D + d;
        const float y = o[m] * inv * lg[i][d];
        if (F32) reinterpret_cast<float*>(p.out)[oi] = y;
        else reinterpret_cast<bf16_t*>(p.out)[oi] = f2bf(y);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    if (k0 + j >= D || c >= D) continue;
    float* q = sp + (int64_t)(k0 + j) * D + c;
    if (vec4) *reinterpret_cast<f32x4*>(q) = S[j];
    else
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < D) q[e] = S[j][e];
  }
}

// ------------------------------------------------------------------------------------------ tokens one by one, a head's columns apart
// token t belongs to a sequence with a slot and at most `lim` tokens (no sequence: a padding row of a graph bucket); whole waves, a lane
// per sequence
__device__ __forceinline__ bool token_of_short(const DeltaArgs& p, int t, int lim) {
  for (int i0 = 0; i0 < p.S; i0 += 64) {
    const int i = i0 + (threadIdx.x & 63);
    const int a = i < p.S ? p.query_start[i] : 0, b = i < p.S ? p.query_start[i + 1] : 0;
    const unsigned long long hit = __ballot(a <= t && t < b), ok = __ballot(i < p.S && p.state_slots[i] >= 0 && b - a <= lim);
    if (hit != 0) return (hit & ok) != 0;
  }
  return false;
}

// one wave per (token, head): vec[t][h][d] = {w, a u, k, r}, un[t][h][d] = u
__global__ __launch_bounds__(64) void delta_prep_kernel(DeltaArgs p, int lim, float4* __restrict__ vec,
                                                         float* __restrict__ un) {
  const int t = blockIdx.x, h = blockIdx.y;
  if (!token_of_short(p, t, lim)) return;
  const int D = p.D, lane = threadIdx.x;
  float kk[2], rr[2], aa[2], ww[2];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int d = lane + 64 * i;
    kk[i] = rr[i] = aa[i] = ww[i] = 0.f;
    if (d < D) {
      const int ch = h * D + d;
      const int64_t ix = (int64_t)t * p.ld + ch;
      kk[i] = ldx(p.k, ix, p.f32);
      rr[i] = ldx(p.r, ix, p.f32);
      aa[i] = sigm(ldx(p.a, ix, p.f32) + p.ab[ch]);
      ww[i] = expf(-p.decay_c * sigm(ldx(p.wl, (int64_t)t * p.ldw + ch, p.f32) + p.w0[ch]));
      ss = fmaf(kk[i], kk[i], ss);
    }
  }
  ss = wave_reduce_sum(ss);
  const float inv = 1.f / sqrtf(ss + p.unit_eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int d = lane + 64 * i;
    if (d < D) {
      const float u = kk[i] * inv;
      const int64_t o = ((int64_t)t * p.H + h) * D + d;
      vec[o] = make_float4(ww[i], aa[i] * u, kk[i], rr[i]);
      un[o] = u;
    }
  }
}

// lane = 8 * q + c: key group q of 8 (keys [q DQ', (q + 1) DQ') with DQ' = ceil(D / 8)), value column c0 + c
template <int DQ>
__global__ __launch_bounds__(64) void delta_scan_kernel(DeltaArgs p, int lim, const float4* __restrict__ vec,
                                                         const float* __restrict__ un, float* __restrict__ oraw) {
  // quarter strides padded (DQ + 1 float4 / DQ + 4 floats): the four quarters' broadcast reads of one
  // instruction fall into different LDS banks. Entries of channels past D are zeroed once and never
  // written, so the token loops run DQ iterations with no bounds test (zeros leave S, u^T S and o alone).
  constexpr int QV = DQ + 1, QU = DQ + 4;
  __shared__ float4 lv[2][TC][8 * QV];
  __shared__ float lu[2][TC][8 * QU];
  __shared__ float lvv[2][TC][8];  // the slice's value columns of each staged token
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 8;
  const int slot = p.state_slots[s];
  const int t0 = p.query_start[s], t1 = p.query_start[s + 1];
  if (slot < 0 || t1 <= t0 || t1 - t0 > lim) return;
  const int D = p.D, lane = threadIdx.x;
  const int q = lane >> 3, c = c0 + (lane & 7);
  const int dq = (D + 7) >> 3;         // keys per group at run time (<= DQ)
  const int k0 = q * dq;
  const bool con = c < D;
  const int pos0 = p.context_lens[s] - (t1 - t0);
  float* sp = p.state + ((int64_t)slot * p.H + h) * D * D;
  float S[DQ];
#pragma unroll
  for (int j = 0; j < DQ; ++j)
    S[j] = (con && j < dq && k0 + j < D && pos0 > 0) ? sp[(int64_t)(k0 + j) * D + c] : 0.f;
  // staging: a token's D channels are D float4 + D floats; lane l moves channels l, l + 64 of each token
  float4 pv[TC][2];
  float pu[TC][2];
  float pvv;
  auto fetch = [&](int tb) {
#pragma unroll
    for (int i = 0; i < TC; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int d = lane + 64 * e, t = tb + i;
        const bool ok = d < D && t < t1;
        const int64_t o = ((int64_t)(ok ? t : t0) * p.H + h) * D + (ok ? d : 0);
        pv[i][e] = ok ? vec[o] : make_float4(0.f, 0.f, 0.f, 0.f);
        pu[i][e] = ok ? un[o] : 0.f;
      }
    {  // TC x 8 values, lane -> (token, column)
      const int t = tb + (lane >> 3), cc = c0 + (lane & 7);
      pvv = (t < t1 && cc < D) ? ldx(p.v, (int64_t)t * p.ld + h * D + cc, p.f32) : 0.f;
    }
  };
  // LDS index of channel d: quarter-major, padded to DQ per quarter
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TC; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int d = lane + 64 * e;
        if (d < D) {
          lv[buf][i][(d / dq) * QV + (d % dq)] = pv[i][e];
          lu[buf][i][(d / dq) * QU + (d % dq)] = pu[i][e];
        }
      }
    lvv[buf][lane >> 3][lane & 7] = pvv;
  };
  for (int e = lane; e < 2 * TC * 8 * QV; e += 64) (&lv[0][0][0])[e] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int e = lane; e < 2 * TC * 8 * QU; e += 64) (&lu[0][0][0])[e] = 0.f;
  __syncthreads();
  fetch(t0);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int tb = t0; tb < t1; tb += TC) {
    const bool more = tb + TC < t1;
    if (more) fetch(tb + TC);
    const int nt = min(TC, t1 - tb);
    // unrolled over the staged tokens, with token i + 1's vectors read from LDS into a second register
    // set before token i's FMAs and lane exchanges (they do not depend on the state)
    float4 xv[2][DQ];
    float xu[2][DQ], xvv[2];
    auto grab = [&](int i, int r) {
      const float4* tv = &lv[buf][i][q * QV];
      const float* tu = &lu[buf][i][q * QU];
#pragma unroll
      for (int j = 0; j < DQ; ++j) { xv[r][j] = tv[j]; xu[r][j] = tu[j]; }
      xvv[r] = lvv[buf][i][lane & 7];
    };
    grab(0, 0);
#pragma unroll
    for (int i = 0; i < TC; ++i) {
      if (i >= nt) break;
      if (i + 1 < TC) grab(i + 1, (i + 1) & 1);  // (past nt: stale but finite LDS, never used)
      const int r = i & 1;
      const float vv = xvv[r];
      float uS = 0.f;
#pragma unroll
      for (int j = 0; j < DQ; ++j) uS = fmaf(xu[r][j], S[j], uS);
      uS += row_rot<0x128>(uS);
      uS += xor16(uS);
      uS += xor32(uS);
      float o = 0.f;
#pragma unroll
      for (int j = 0; j < DQ; ++j) {
        const float4 x = xv[r][j];  // {w, a u, k, r}
        S[j] = fmaf(x.z, vv, fmaf(-x.y, uS, x.x * S[j]));
        o = fmaf(x.w, S[j], o);
      }
      o += row_rot<0x128>(o);
      o += xor16(o);
      o += xor32(o);
      if (con && q == 0) oraw[(int64_t)(tb + i) * p.H * D + h * D + c] = o;
    }
    if (more) {
      put(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
#pragma unroll
  for (int j = 0; j < DQ; ++j)
    if (con && j < dq && k0 + j < D) sp[(int64_t)(k0 + j) * D + c] = S[j];
}

// one wave per (token, head)
__global__ __launch_bounds__(64) void delta_finish_kernel(DeltaArgs p, int lim, const float* __restrict__ oraw) {
  const int t = blockIdx.x, h = blockIdx.y;
  if (!token_of_short(p, t, lim)) return;
  const int D = p.D, lane = threadIdx.x;
  float o[2];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int d = lane + 64 * i;
    o[i] = d < D ? oraw[((int64_t)t * p.H + h) * D + d] : 0.f;
    ss = fmaf(o[i], o[i], ss);
  }
  ss = wave_reduce_sum(ss);
  const float inv = 1.f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int d = lane + 64 * i;
    if (d < D) {
      const int ch = h * D + d;
      const float y = o[i] * inv * p.nw[ch] * sigm(ldx(p.g, (int64_t)t * p.ld + ch, p.f32));
      const int64_t oi = (int64_t)t * p.ldo + ch;
      if (p.f32) reinterpret_cast<float*>(p.out)[oi] = y;
      else reinterpret_cast<bf16_t*>(p.out)[oi] = f2bf(y);
    }
  }
}

// ------------------------------------------------------------------------------------------ chunks of CN tokens
// floats of one (chunk, head) record: [W; Q] (rows, channels), the update's b and k (channels, tokens) each, g_(1..CN) [DP], then y, the
// outputs and v (columns, tokens) each; all but g in the order of frag()
__host__ __device__ inline int64_t delta_chunk_floats(int DP, int D) { return (int64_t)4 * CN * DP + DP + (int64_t)3 * CN * whole16(D); }

// grid (chunk, head). At DP = 128 the LDS comes to half of a CU's.
template <int DP, bool F32>
__global__ __launch_bounds__(256, 2) void delta_chunk_kernel(DeltaArgs p, int lim, float* __restrict__ rec) {
  constexpr int X = DP / 32;   // 16-B pieces of a row a lane of the pair sums holds: channels 32 x + 4 dg ..
  __shared__ __attribute__((aligned(16))) float lw[CN][DP], lu[CN][DP], lb[CN][DP], lr[CN][DP];
  __shared__ __attribute__((aligned(16))) float Ab[tri(CN)], Ak[tri(CN)], Rb[tri(CN + 1)], Rk[tri(CN + 1)];
  __shared__ float len[CN];
  int s, t0, t1;
  if (!locate_chunk(p.query_start, p.state_slots, p.S, lim, blockIdx.x, s, t0, t1)) return;
  const int h = blockIdx.y, D = p.D, H = p.H;
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  float* r0 = rec + ((int64_t)blockIdx.x * H + h) * delta_chunk_floats(DP, D);
  float* kb = r0 + 2 * CN * DP;
  float* kk = kb + CN * DP;
  float* gam = kk + CN * DP;
  float* yy = gam + DP;
  float* oo = yy + CN * whole16(D);
  float* vo = oo + CN * whole16(D);
  constexpr int KT = DP / 16;
  const int DQ4 = (D + 3) & ~3;   // channels in whole quads of lanes (u = b = r = 0, w = 1 in those past D)
  constexpr int f32 = F32 ? 1 : 0;
#pragma unroll 4
  for (int e = tid; e < CN * DP; e += 256) {   // rows past the end: u = b = r = 0, w = 1
    const int i = e / DP, d = e % DP;
    float w = 1.f, a = 0.f, k = 0.f, r = 0.f;
    if (d < D && t0 + i < t1) {
      const int ch = h * D + d;
      const int64_t ix = (int64_t)(t0 + i) * p.ld + ch;
      k = ldx(p.k, ix, f32);
      r = ldx(p.r, ix, f32);
      a = sigm(ldx(p.a, ix, f32) + p.ab[ch]);
      w = expf(-p.decay_c * sigm(ldx(p.wl, (int64_t)(t0 + i) * p.ldw + ch, f32) + p.w0[ch]));
    }
    lw[i][d] = w; lu[i][d] = k; lb[i][d] = a; lr[i][d] = r;
  }
  __syncthreads();
  {  // u = k / its length and b = a u in place: eight threads per row
    const int row = tid >> 3, part = tid & 7;
    float4 v[DP / 32];
    float ss = 0.f;
#pragma unroll
    for (int m = 0; m < DP / 32; ++m) {
      v[m] = *reinterpret_cast<const float4*>(&lu[row][32 * m + 4 * part]);
      ss = fmaf(v[m].x, v[m].x, fmaf(v[m].y, v[m].y, fmaf(v[m].z, v[m].z, fmaf(v[m].w, v[m].w, ss))));
    }
    ss += row_rot<0xB1>(ss);    // (quad_perm [1, 0, 3, 2], then [2, 3, 0, 1], then row_half_mirror)
    ss += row_rot<0x4E>(ss);
    ss += row_rot<0x141>(ss);
    const bool real = t0 + row < t1;
    const float n = sqrtf(ss + p.unit_eps), f = real ? 1.f / n : 0.f;
    if (part == 0) len[row] = real ? n : 0.f;
#pragma unroll
    for (int m = 0; m < DP / 32; ++m) {
      const float4 u = make_float4(v[m].x * f, v[m].y * f, v[m].z * f, v[m].w * f);
      float4* bp = reinterpret_cast<float4*>(&lb[row][32 * m + 4 * part]);
      const float4 a = *bp;
      *reinterpret_cast<float4*>(&lu[row][32 * m + 4 * part]) = u;
      *bp = make_float4(a.x * u.x, a.y * u.y, a.z * u.z, a.w * u.w);
    }
  }
  __syncthreads();
  {  // the triangles: a wave owns eight columns j, lane = (channel group dg of eight, j); the wave with most rows differs
     // between neighbouring chunks, so that workgroups on one CU do not all load the same SIMD
    const int jb = (blockIdx.x & 1) ? 3 - wv : wv;
    const int dg = lane >> 3, j = 8 * jb + (lane & 7);
    float xb[4 * X], xu[4 * X];
#pragma unroll
    for (int x = 0; x < X; ++x) {
      const float4 v = *reinterpret_cast<const float4*>(&lb[j][32 * x + 4 * dg]);
      const float4 u = *reinterpret_cast<const float4*>(&lu[j][32 * x + 4 * dg]);
      xb[4 * x] = v.x; xb[4 * x + 1] = v.y; xb[4 * x + 2] = v.z; xb[4 * x + 3] = v.w;
      xu[4 * x] = u.x; xu[4 * x + 1] = u.y; xu[4 * x + 2] = u.z; xu[4 * x + 3] = u.w;
    }
    const float nj = len[j];
    for (int i = 8 * jb; i < CN; ++i) {
      float ab = 0.f, ak = 0.f, rb = 0.f, rk = 0.f;
#pragma unroll
      for (int x = 0; x < X; ++x) {
        const float4 wq = *reinterpret_cast<const float4*>(&lw[i][32 * x + 4 * dg]);
        const float4 uq = *reinterpret_cast<const float4*>(&lu[i][32 * x + 4 * dg]);
        const float4 rq = *reinterpret_cast<const float4*>(&lr[i][32 * x + 4 * dg]);
        const float w[4] = {wq.x, wq.y, wq.z, wq.w}, u[4] = {uq.x, uq.y, uq.z, uq.w}, r[4] = {rq.x, rq.y, rq.z, rq.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          ab = fmaf(u[c], xb[4 * x + c], ab);
          ak = fmaf(u[c], xu[4 * x + c], ak);
          if (i > j) { xb[4 * x + c] *= w[c]; xu[4 * x + c] *= w[c]; }
          rb = fmaf(r[c], xb[4 * x + c], rb);
          rk = fmaf(r[c], xu[4 * x + c], rk);
        }
      }
      ab = key_sum<8>(ab); ak = key_sum<8>(ak); rb = key_sum<8>(rb); rk = key_sum<8>(rk);
      if (dg == 0 && i > j) { Ab[tri(i) + j] = ab; Ak[tri(i) + j] = ak * nj; }
      if (dg == 0 && i >= j) { Rb[tri(i + 1) + j] = rb; Rk[tri(i + 1) + j] = rk * nj; }
    }
  }
  __syncthreads();
  for (int c = tid; c < DQ4 + D; c += 256) {   // one column of [W | y] per thread
    float x[CN];
    if (c < DQ4) {
      float gm = 1.f;
#pragma unroll
      for (int i = 0; i < CN; ++i) {
        x[i] = gm * lu[i][c] - row_dot(Ab + tri(i), x, i);
        gm *= lw[i][c];
        if (i % 2) __builtin_amdgcn_sched_barrier(0);   // (rows ahead of time would take hundreds of registers)
      }
      gam[c] = gm;
      float gb = 1.f;
#pragma unroll
      for (int j0 = CN - 4; j0 >= 0; j0 -= 4) {
        f32x4 vb, vk;
#pragma unroll
        for (int j = 3; j >= 0; --j) {
          vb[j] = lb[j0 + j][c] * gb;
          vk[j] = lu[j0 + j][c] * len[j0 + j] * gb;
          gb *= lw[j0 + j][c];
        }
        *reinterpret_cast<f32x4*>(kb + frag(c, j0, 2)) = vb;
        *reinterpret_cast<f32x4*>(kk + frag(c, j0, 2)) = vk;
        __builtin_amdgcn_sched_barrier(0);
      }
      gm = 1.f;
#pragma unroll
      for (int i0 = 0; i0 < CN; i0 += 4) {
        f32x4 q;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          gm *= lw[i0 + i][c];
          q[i] = gm * lr[i0 + i][c] - row_dot(Rb + tri(i0 + i + 1), x, i0 + i + 1);
          if (i % 2) __builtin_amdgcn_sched_barrier(0);
        }
        put_rows4(r0, i0, c, KT, f32x4{x[i0], x[i0 + 1], x[i0 + 2], x[i0 + 3]});
        put_rows4(r0, CN + i0, c, KT, q);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      const int vc = c - DQ4;
      float v[CN];
#pragma unroll
      for (int i = 0; i < CN; ++i) v[i] = t0 + i < t1 ? ldx(p.v, (int64_t)(t0 + i) * p.ld + h * D + vc, f32) : 0.f;
#pragma unroll
      for (int i = 0; i < CN; ++i) {
        x[i] = row_dot(Ak + tri(i), v, i) - row_dot(Ab + tri(i), x, i);
        if (i % 2) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i0 = 0; i0 < CN; i0 += 4) {
        f32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = row_dot(Rk + tri(i0 + i + 1), v, i0 + i + 1) - row_dot(Rb + tri(i0 + i + 1), x, i0 + i + 1);
        *reinterpret_cast<f32x4*>(yy + frag(vc, i0, 2)) = f32x4{x[i0], x[i0 + 1], x[i0 + 2], x[i0 + 3]};
        *reinterpret_cast<f32x4*>(oo + frag(vc, i0, 2)) = o;
        *reinterpret_cast<f32x4*>(vo + frag(vc, i0, 2)) = f32x4{v[i0], v[i0 + 1], v[i0 + 2], v[i0 + 3]};
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  for (int e = tid; e < (DP - DQ4) * CN; e += 256) {   // channels past them: zero
    const int d = DQ4 + e / CN, i = e % CN;
    r0[frag(i, d, KT)] = 0.f;
    r0[frag(CN + i, d, KT)] = 0.f;
    kb[frag(d, i, 2)] = 0.f;
    kk[frag(d, i, 2)] = 0.f;
    if (i == 0) gam[d] = 0.f;
  }
  for (int e = tid; e < (whole16(D) - D) * CN; e += 256) {   // columns of a last tile that is not whole: zero
    const int at = frag(D + e / CN, e % CN, 2);
    yy[at] = oo[at] = vo[at] = 0.f;
  }
}

// grid (head, rounded up to the XCDs, 16 columns, sequence): a head's workgroups read the same records on one XCD. NT tiles
// of 16 channels. MFMA operands: the channel (or token) 16 n + 4 kg + e is element e of lane group kg in both operands, so
// a lane's four steps are one 16-B piece of a row.
template <int NT>
__global__ __launch_bounds__(256) void delta_chunk_scan_kernel(DeltaArgs p, int lim, float* __restrict__ rec) {
  constexpr int DP = 16 * NT, TW = (NT + 3) / 4;
  __shared__ __attribute__((aligned(16))) float Sl[16][DP + 4];
  __shared__ __attribute__((aligned(16))) float Pl[16][CN + 4];
  const int s = blockIdx.z, h = blockIdx.x, c0 = blockIdx.y * 16;
  if (h >= p.H) return;
  const int slot = p.state_slots[s];
  const int t0 = p.query_start[s], t1 = p.query_start[s + 1];
  if (slot < 0 || t1 - t0 <= lim) return;
  const int nc = (t1 - t0 + CN - 1) / CN, D = p.D, H = p.H;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, kg = l >> 4;
  const bool con = c0 + lr < D;
  const bool from_zero = p.context_lens[s] - (t1 - t0) <= 0;
  float* sp = p.state + ((int64_t)slot * H + h) * D * D;
  f32x4 S[TW];
#pragma unroll
  for (int t = 0; t < TW; ++t) {
    const int tile = w + 4 * t;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * tile + 4 * kg + i;
      S[t][i] = (!from_zero && tile < NT && d < D && con) ? sp[(int64_t)d * D + c0 + lr] : 0.f;
    }
    if (tile < NT) *reinterpret_cast<f32x4*>(&Sl[lr][16 * tile + 4 * kg]) = S[t];
  }
  const int64_t per = delta_chunk_floats(DP, D);
  float* r0 = rec + ((int64_t)first_chunk(p.query_start, p.state_slots, lim, s) * H + h) * per;
  struct Chunk {   // what a lane needs of one chunk's record
    f32x4 A[NT], B[TW][2], K[TW][2], gm[TW], v[2], add;
    float* out;
  };
  auto fetch = [&](Chunk& x, int ch) {
    float* r = r0 + (int64_t)ch * H * per;
    const float* kb = r + 2 * CN * DP;
    const float* kk = kb + CN * DP;
    float* gam = r + 4 * CN * DP;
    float* yy = gam + DP;
    yy += blockIdx.y * 512 + 4 * l;   // (the workgroup's columns: two pieces)
    x.out = yy + (w < 2 ? 0 : CN * whole16(D)) + 256 * (w & 1);   // y of waves 0, 1; the outputs of 2, 3
#pragma unroll
    for (int n = 0; n < NT; ++n) x.A[n] = ld4(r + (w * NT + n) * 256 + 4 * l);
    x.add = ld4(x.out);
#pragma unroll
    for (int m = 0; m < 2; ++m) x.v[m] = ld4(yy + 2 * CN * whole16(D) + 256 * m);
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int tile = min(w + 4 * t, NT - 1);
      x.gm[t] = ld4(gam + 16 * tile + 4 * kg);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        x.K[t][m] = ld4(kk + (2 * tile + m) * 256 + 4 * l);
        x.B[t][m] = ld4(kb + (2 * tile + m) * 256 + 4 * l);
      }
    }
  };
  // chunk ch from `x`, while chunk ch + 1 is on its way into `y` (the barriers wait for LDS traffic only)
  auto step = [&](Chunk& x, Chunk& y, int ch) {
    fetch(y, min(ch + 1, nc - 1));   // (without a branch: the waits below then count past these loads)
    __builtin_amdgcn_sched_barrier(0);
    f32x4 P0 = f32x4{0.f, 0.f, 0.f, 0.f}, P1 = P0;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(&Sl[lr][16 * n + 4 * kg]);
      P0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.A[n][0], b[0], P0, 0, 0, 0);
      P1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.A[n][1], b[1], P1, 0, 0, 0);
      P0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.A[n][2], b[2], P0, 0, 0, 0);
      P1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.A[n][3], b[3], P1, 0, 0, 0);
    }
    const f32x4 P = x.add + (P0 + P1);
    if (w < 2) *reinterpret_cast<f32x4*>(&Pl[lr][16 * w + 4 * kg]) = -P;
    else if (con) *reinterpret_cast<f32x4*>(x.out) = P;
#pragma unroll
    for (int t = 0; t < TW; ++t) {   // k v^T does not wait for p
      S[t] *= x.gm[t];
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.K[t][m][e], x.v[m][e], S[t], 0, 0, 0);
    }
    lds_barrier();   // p is there, and every wave is done with S
#pragma unroll
    for (int t = 0; t < TW; ++t) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(&Pl[lr][16 * m + 4 * kg]);
#pragma unroll
        for (int e = 0; e < 4; ++e) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.B[t][m][e], b[e], S[t], 0, 0, 0);
      }
      if (w + 4 * t < NT) *reinterpret_cast<f32x4*>(&Sl[lr][16 * (w + 4 * t) + 4 * kg]) = S[t];
    }
    lds_barrier();
  };
  Chunk x, y;
  fetch(x, 0);
  lds_barrier();
  int ch = 0;
  for (; ch + 1 < nc; ch += 2) {
    step(x, y, ch);
    step(y, x, ch + 1);
  }
  if (ch < nc) step(x, y, ch);
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * (w + 4 * t) + 4 * kg + i;
      if (w + 4 * t < NT && d < D && con) sp[(int64_t)d * D + c0 + lr] = S[t][i];
    }
}

// grid (chunk, head)
__global__ __launch_bounds__(256) void delta_chunk_finish_kernel(DeltaArgs p, int lim, int DP, const float* __restrict__ rec) {
  __shared__ float lo[128][CN + 1];
  __shared__ float rn[CN];
  int s, t0, t1;
  if (!locate_chunk(p.query_start, p.state_slots, p.S, lim, blockIdx.x, s, t0, t1)) return;
  const int h = blockIdx.y, D = p.D, H = p.H, tid = threadIdx.x;
  const float* o = rec + ((int64_t)blockIdx.x * H + h) * delta_chunk_floats(DP, D) + 4 * CN * DP + DP + CN * whole16(D);
  for (int e = tid; e < whole16(D) * CN / 4; e += 256) {   // (frag(): column, then token)
    const int c = (e >> 7) * 16 + (e & 15), i = ((e >> 6) & 1) * 16 + ((e >> 4) & 3) * 4;
    const f32x4 v = ld4(o + 4 * e);
#pragma unroll
    for (int j = 0; j < 4; ++j) lo[c][i + j] = v[j];
  }
  __syncthreads();
  {  // eight threads per token
    const int i = tid >> 3, part = tid & 7;
    float ss = 0.f;
    for (int c = part; c < D; c += 8) ss = fmaf(lo[c][i], lo[c][i], ss);
    ss += row_rot<0xB1>(ss);
    ss += row_rot<0x4E>(ss);
    ss += row_rot<0x141>(ss);
    if (part == 0) rn[i] = 1.f / sqrtf(ss / (float)D + p.eps);
  }
  __syncthreads();
  for (int e = tid; e < (t1 - t0) * D; e += 256) {
    const int i = e / D, c = e % D, ch = h * D + c;
    const int64_t t = t0 + i;
    const float y = lo[c][i] * rn[i] * p.nw[ch] * sigm(ldx(p.g, t * p.ld + ch, p.f32));
    const int64_t oi = t * p.ldo + ch;
    if (p.f32) reinterpret_cast<float*>(p.out)[oi] = y;
    else reinterpret_cast<bf16_t*>(p.out)[oi] = f2bf(y);
  }
}

int delta_channels(int D) { return D <= 32 ? 32 : (D <= 64 ? 64 : 128); }
// Few sequences, not all of them decoded tokens: the scan is ahead for portions of some 12 to 128 tokens (D <= 64: 20 to 96), 0.4 to
// 0.5 us a token where all its workgroups run at once (their LDS allows 768 on the chip, 1536 for D <= 64). us, scan / short form / chunks, 8
// heads of 128: one portion of 8 tokens 17, 16, 69; of 16 22, 27, 69; of 64 47, 91, 79; of 96 63, 134, 80; of 128 80, 176, 84; of 160 96, 219, 86;
// 4 x 8 18, 17, 22; 4 x 64 49, 92, 82; 8 x 64 (more than run at once) 92, 92, 97. D = 64: 16 tokens 16, 16, 51; 64 34, 55, 51; 96 46, 81,
// 52; 128 57, 107, 54. The host knows rows and sequences only. In a step of several sequences and more than 128 rows those of more
// tokens take chunks, told apart on the device: three more launches, 6 us, so not once the sequences are so long on average that the scan
// has little to give (4 x 64 tokens 56, without the scan 82; 3 + 253 111, 104, by the scan alone 148).
constexpr int delta_scan_limit(int D) { return D > 64 ? 128 : 96; }
bool takes_scan(int T, int S, int H, int D) {
  const int64_t blocks = (int64_t)S * H * ((D + 7) / 8);
  const int lim = delta_scan_limit(D);
  return blocks <= (D > 64 ? 768 : (D > 32 ? 1536 : 4096)) && T >= std::max(D > 64 ? 12 : 24, 4 * S) &&
         (T <= lim || (S > 1 && T <= (lim - 32) * S));
}
// Else, tokens a sequence may have in a step to be run one by one in the short form: 1.3 us each against about 75 us for the shortest
// portion in chunks. Decoding steps (T <= S) and others of at most 64 rows, which may be too, take one launch (8 heads of 128, with the
// chunks' three empty ones: 128 sequences 35 us, 45; 256 65, 82).
int delta_limit(int T, int S) { return T <= S || T <= 64 ? T : 48; }
// chunks of a step whose sequences longer than lim tokens have T between them: each has at most one that is not whole
int delta_chunks(int T, int S, int lim) { return T <= lim ? 0 : (T + std::min(S, T / (lim + 1)) * (CN - 1)) / CN; }

// {w, a u, k, r}, u, the raw outputs; whole 16-B pieces
size_t scan_floats(int T, int H, int D) { return ((size_t)T * H * D * 6 + 3) / 4 * 4; }

void launch_scan(const DeltaArgs& a, int T, int lim, float* scratch, hipStream_t st) {
  const int64_t n = (int64_t)T * a.H * a.D;
  float4* vec = reinterpret_cast<float4*>(scratch);
  float* un = scratch + 4 * n;
  float* oraw = scratch + 5 * n;
  hipLaunchKernelGGL(delta_prep_kernel, dim3(T, a.H), dim3(64), 0, st, a, lim, vec, un);
  const dim3 grid(a.S, a.H, (a.D + 7) / 8);
  if (a.D <= 32) hipLaunchKernelGGL(delta_scan_kernel<4>, grid, dim3(64), 0, st, a, lim, vec, un, oraw);
  else if (a.D <= 64) hipLaunchKernelGGL(delta_scan_kernel<8>, grid, dim3(64), 0, st, a, lim, vec, un, oraw);
  else hipLaunchKernelGGL(delta_scan_kernel<16>, grid, dim3(64), 0, st, a, lim, vec, un, oraw);
  hipLaunchKernelGGL(delta_finish_kernel, dim3(T, a.H), dim3(64), 0, st, a, lim, oraw);
}

template <int DP, bool F32>
void launch_delta(const DeltaArgs& a, int T, const DeltaPlan& plan, float* scratch, hipStream_t st) {
  // T counts padding rows too, so a sequence may be much shorter. A lone one then takes chunks whatever its length (not more
  // of them than any step of T rows); several are told apart by their lengths on the device.
  const bool lone = a.S == 1 && plan.chunks > 0;
  if (plan.scan) launch_scan(a, T, plan.lim, scratch, st);
  else if (!lone) hipLaunchKernelGGL((delta_short_kernel<DP, F32>), dim3(a.S, a.H), dim3(256), 0, st, a, plan.lim);
  if (plan.chunks == 0) return;
  const int lim = lone ? 0 : plan.lim;
  float* rec = scratch + (plan.scan ? scan_floats(T, a.H, a.D) : 0);
  const dim3 grid(plan.chunks, a.H), scan((a.H + 7) / 8 * 8, (a.D + 15) / 16, a.S);
  hipLaunchKernelGGL((delta_chunk_kernel<DP, F32>), grid, dim3(256), 0, st, a, lim, rec);
  hipLaunchKernelGGL(delta_chunk_scan_kernel<DP / 16>, scan, dim3(256), 0, st, a, lim, rec);
  hipLaunchKernelGGL(delta_chunk_finish_kernel, grid, dim3(256), 0, st, a, lim, DP, rec);
}

template <int DP>
void launch_delta_dp(const DeltaArgs& a, int T, const DeltaPlan& plan, float* scratch, hipStream_t st) {
  if (a.f32) launch_delta<DP, true>(a, T, plan, scratch, st);
  else launch_delta<DP, false>(a, T, plan, scratch, st);
}

}  // namespace

DeltaPlan delta_rule_plan(int T, int S, int H, int D) {
  const bool scan = takes_scan(T, S, H, D);
  const int lim = scan ? (T <= 128 ? T : delta_scan_limit(D)) : delta_limit(T, S);
  return {scan, lim, S == 1 && T > lim ? (T + CN - 1) / CN : delta_chunks(T, S, lim)};
}

size_t delta_rule_scratch_floats(int T, int S, int H, int D) {
  const DeltaPlan plan = delta_rule_plan(T, S, H, D);
  const size_t rows = scan_floats(T, H, D), chunks = (size_t)plan.chunks * H * delta_chunk_floats(delta_channels(D), D);
  return plan.scan ? rows + chunks : std::max(rows, chunks);
}

// scratch: `floats` of them, 6 T H D at least; fewer than delta_rule_scratch_floats(): the scan in place of chunks
void launch_delta_rule(const DeltaArgs& a, int T, float* scratch, size_t floats, hipStream_t st) {
  if (a.S <= 0 || a.H <= 0 || T <= 0) return;
  DeltaPlan plan = delta_rule_plan(T, a.S, a.H, a.D);
  if (plan.chunks > 0 && floats < delta_rule_scratch_floats(T, a.S, a.H, a.D)) plan = DeltaPlan{true, T, 0};
  if (a.D <= 32) launch_delta_dp<32>(a, T, plan, scratch, st);
  else if (a.D <= 64) launch_delta_dp<64>(a, T, plan, scratch, st);
  else launch_delta_dp<128>(a, T, plan, scratch, st);
}

}  // namespace vgate
