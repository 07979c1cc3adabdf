// Row-major GEMM of any shape: out = epi(A W^T) with W stored [N][K] as checkpoints hold it.
//
// It serves what the fragment-packed GEMMs (gemm.hip, gemm_prefill.hip) do not take: fp32 models (true
// fp32 FMA, no reduced-precision matrix mode), sizes that are not multiples of the MFMA tile, one
// product per head (batch = blockIdx.z with strides on A, W and out), one product per expert over a
// device-side row grouping (group_off; tiles are located on the device, so the grid is fixed and
// the launch is graph-capturable), A-row gathers, and gated pairs (two weight matrices, one
// activation in the epilogue).
//   bf16: 64 x 64 block tile, 4 waves of 2 x 2 v_mfma_f32_16x16x32_bf16 tiles, operands read as 16-B
//         fragments straight from global memory (both operands are k-contiguous rows), fp32 accumulate.
//         Large aligned products (hundreds of rows, wide outputs: the expert GEMMs of a prompt portion):
//         128 x 128 block tile (a weight pair: 128 x 64 of each matrix), 4 waves of 4 x 4 MFMA tiles, k-steps of
//         32 staged through two LDS buffers, the loads of the two steps after the current one in flight.
//   fp32: 64 x 64 x 16 LDS-tiled FMA kernel, 4 x 4 outputs per thread, k ascending.
#include <cstdlib>
#include <type_traits>

#include "lds_rows.h"
#include "locate.h"
#include "seq_launchers.h"

namespace vgate {
namespace {

constexpr int BM = 64, BN = 64;

__device__ __forceinline__ bool locate_tile(const AnyGemmArgs& p, int by, int& grp, int& r0, int& rend, int bm = BM) {
  if (p.group_off == nullptr) {
    grp = 0; r0 = by * bm; rend = p.M;
    return r0 < p.M;
  }
  int local;
  grp = locate_item(p.groups, by, local, [&](int g) { return (p.group_off[g + 1] - p.group_off[g] + bm - 1) / bm; });
  if (grp < 0) return false;
  r0 = p.group_off[grp] + local * bm;
  rend = p.group_off[grp + 1];
  return true;
}

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + expf(-x)); }

// the activation of one output (g: the accumulator with its bias, u: the second matrix's); ACT is AnyGemmArgs::act
template <int ACT>
__device__ __forceinline__ float act_val(const AnyGemmArgs& p, float g, float u) {
  if (ACT == 1) return g * sigmoidf_(g) * u;
  if (ACT == 2) {
    const float gg = fminf(g, p.limit);
    const float uu = fminf(fmaxf(u, -p.limit), p.limit);
    return gg * sigmoidf_(p.alpha * gg) * (uu + 1.f);
  }
  if (ACT == 3) return tanhf(g);
  if (ACT == 4) return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
  if (ACT == 5) return 0.5f * g * (1.f + erff(g * 0.70710678118654752f));
  if (ACT == 6) { const float r = fmaxf(g, 0.f); return r * r; }
  return g;
}

// fn<ACT>() for the launch's activation: one uniform branch per tile, so a thread's outputs run through straight code of
// their own activation (a chain of tests per output would jump over every other activation's code each time)
template <int DUAL, typename F>
__device__ __forceinline__ void with_act(const AnyGemmArgs& p, F&& fn) {
  if (DUAL) {
    if (p.act == 1) fn(std::integral_constant<int, 1>{});
    else if (p.act == 2) fn(std::integral_constant<int, 2>{});
    else fn(std::integral_constant<int, 4>{});
  } else {
    if (p.act == 0) fn(std::integral_constant<int, 0>{});
    else if (p.act == 6) fn(std::integral_constant<int, 6>{});
    else if (p.act == 5) fn(std::integral_constant<int, 5>{});
    else fn(std::integral_constant<int, 3>{});
  }
}

__device__ __forceinline__ void store_value(const AnyGemmArgs& p, int64_t i, float v) {
  if (p.out_f32) reinterpret_cast<float*>(p.out)[i] = v;
  else reinterpret_cast<bf16_t*>(p.out)[i] = f2bf(v);
}

__device__ __forceinline__ void store_out(const AnyGemmArgs& p, int64_t b, int m, int n, float v) {
  if (p.gate != nullptr) {
    const int64_t gi = (int64_t)m * p.ldg + b * p.g_bs + (int64_t)n * p.g_cs;
    const float gl = p.gate_f32 ? reinterpret_cast<const float*>(p.gate)[gi]
                                : bf2f(reinterpret_cast<const bf16_t*>(p.gate)[gi]);
    v *= sigmoidf_(gl);
  }
  store_value(p, (int64_t)m * p.ldo + b * p.o_bs + n, v);
}

__device__ __forceinline__ bf16x8 load_frag(const bf16_t* rowp, int k, int K, bool valid) {
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

// AL: K, the row strides and the batch strides are multiples of 8 elements and the bases 16-B aligned
// (host-checked): every fragment is one unconditional 16-B load (rows / columns past the edge read a
// clamped, valid row and are dropped at the store; k past K selects zero), two k-steps are loaded before
// their MFMAs, so the loads of a wave overlap.
// NJ: 16-column tiles per wave (2: 64-column block tile; 4: 128-column block tile for wide outputs, which
// loads 1.5x fewer fragment bytes per MFMA)
// A tile with at most 32 rows (an expert's few rows of a decode step) on the aligned 64-column form: the two
// waves that would split the rows split the k range instead (k-steps of 64 in turn, so each weight fragment is
// loaded by one wave only and a wave's dependent chain of loads is half as long) and add up through LDS.
template <int DUAL, bool AL, int NJ>
__global__ __launch_bounds__(256) void gemm_any_mfma_kernel(AnyGemmArgs p) {
  constexpr bool KS = AL && NJ == 2;
  __shared__ f32x4 red[KS ? 2 : 1][KS ? (DUAL ? 8 : 4) : 1][KS ? 64 : 1];
  int grp, r0, rend;
  if (!locate_tile(p, blockIdx.y, grp, r0, rend)) return;
  const bool ks = KS && rend - r0 <= 32;  // (workgroup-uniform)
  const int64_t b = blockIdx.z;
  const int64_t wsel = (p.group_off != nullptr) ? grp : b;
  const int n0 = blockIdx.x * (32 * NJ);
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wm = wv & 1, wn = wv >> 1;
  const int lr = l & 15, lk = 8 * (l >> 4);
  const int mrow = ks ? 0 : wm * 32;  // first row of this wave
  const bf16_t* A = reinterpret_cast<const bf16_t*>(p.a) + b * p.a_bs;
  const bf16_t* W = reinterpret_cast<const bf16_t*>(p.w) + wsel * p.w_bs;
  const bf16_t* W2 = DUAL ? reinterpret_cast<const bf16_t*>(p.w2) + wsel * p.w_bs : nullptr;
  const bf16_t* arow[2];
  bool aval[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = r0 + mrow + i * 16 + lr;
    aval[i] = m < rend;
    const int src = aval[i] ? (p.a_rows ? p.a_rows[m] : m) : 0;
    arow[i] = A + (int64_t)src * p.lda;
  }
  const bf16_t* wrow[NJ];
  const bf16_t* w2row[NJ];
  bool wval[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int n = n0 + wn * 16 * NJ + j * 16 + lr;
    wval[j] = n < p.N;
    wrow[j] = W + (int64_t)(wval[j] ? n : 0) * p.ldw;
    w2row[j] = DUAL ? W2 + (int64_t)(wval[j] ? n : 0) * p.ldw : nullptr;
  }
  f32x4 acc[2][NJ], acc2[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc2[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  if (AL) {
    const uint4 zero = make_uint4(0, 0, 0, 0);
    const int K = p.K;
    for (int k0 = ks ? 64 * wm : 0; k0 < K; k0 += ks ? 128 : 64) {
      uint4 av[2][2], wv_[2][NJ], uv[2][NJ];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int k = k0 + 32 * st + lk;
        const int kc = min(k, K - 8);
#pragma unroll
        for (int i = 0; i < 2; ++i) av[st][i] = ld16(arow[i] + kc);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          wv_[st][j] = ld16(wrow[j] + kc);
          if (DUAL) uv[st][j] = ld16(w2row[j] + kc);
        }
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bool in = k0 + 32 * st + lk < K;
        if (!in) {
#pragma unroll
          for (int i = 0; i < 2; ++i) av[st][i] = zero;  // a zero A fragment zeroes the product
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            acc[i][j] = mfma16(as_bf16x8(av[st][i]), as_bf16x8(wv_[st][j]), acc[i][j]);
            if (DUAL) acc2[i][j] = mfma16(as_bf16x8(av[st][i]), as_bf16x8(uv[st][j]), acc2[i][j]);
          }
      }
    }
  } else
  for (int k0 = 0; k0 < p.K; k0 += 32) {
    const int k = k0 + lk;
    bf16x8 af[2], bfr[NJ], b2[NJ];
#pragma unroll
    for (int i = 0; i < 2; ++i) af[i] = load_frag(arow[i], k, p.K, aval[i]);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      bfr[j] = load_frag(wrow[j], k, p.K, wval[j]);
      if (DUAL) b2[j] = load_frag(w2row[j], k, p.K, wval[j]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
        if (DUAL) acc2[i][j] = mfma16(af[i], b2[j], acc2[i][j]);
      }
  }
  if (KS && ks) {  // the k halves of a wave pair: wm 1 hands its sums to wm 0
    if (wm == 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          red[KS ? wn : 0][KS ? 2 * i + j : 0][KS ? l : 0] = acc[i][j];
          if (DUAL) red[KS ? wn : 0][KS ? 4 + 2 * i + j : 0][KS ? l : 0] = acc2[i][j];
        }
    }
    __syncthreads();
    if (wm == 1) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        acc[i][j] += red[KS ? wn : 0][KS ? 2 * i + j : 0][KS ? l : 0];
        if (DUAL) acc2[i][j] += red[KS ? wn : 0][KS ? 4 + 2 * i + j : 0][KS ? l : 0];
      }
  }
  float gl[2][NJ][4];   // the gates' logits, asked for together
  if (p.gate != nullptr) {
    const bool gf = p.gate_f32 != 0;
    auto load = [&](auto f32) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int n = min(n0 + wn * 16 * NJ + j * 16 + lr, p.N - 1), m = min(r0 + mrow + i * 16 + 4 * (l >> 4) + e, rend - 1);
            const int64_t gi = (int64_t)m * p.ldg + b * p.g_bs + (int64_t)n * p.g_cs;
            gl[i][j][e] = decltype(f32)::value ? reinterpret_cast<const float*>(p.gate)[gi]
                                               : bf2f(reinterpret_cast<const bf16_t*>(p.gate)[gi]);
          }
    };
    if (gf) load(std::true_type{});
    else load(std::false_type{});
  }
  with_act<DUAL>(p, [&](auto act) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int n = n0 + wn * 16 * NJ + j * 16 + lr;
        if (n >= p.N) continue;
        const float bias = p.bias ? p.bias[n] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = r0 + mrow + i * 16 + 4 * (l >> 4) + e;
          if (m >= rend) continue;
          float v = act_val<decltype(act)::value>(p, acc[i][j][e] + bias, DUAL ? acc2[i][j][e] : 0.f);
          if (p.gate != nullptr) v *= sigmoidf_(gl[i][j][e]);
          store_value(p, (int64_t)m * p.ldo + b * p.o_bs + n, v);
        }
      }
  });
}

// Few rows. Host-checked as AL above. A workgroup owns 16 columns (of both matrices), its four waves take pairs of k-steps (64
// elements: whole 128-B lines of a weight row) in turn and meet in LDS; wave i finishes the i-th 16 rows. A tile's 64 rows go in passes of
// 32. What bounds it is one trip to memory for the weights, 4 to 6 us a launch. UB pairs in flight per wave: one, and eight waves per SIMD
// (with four the registers leave three, and K below 1024 is read in vain: 2048 x 512 with 8 rows each of 8 experts 7.3 us, 12.4); more for
// up to 8 rows and long K, which are one chain of loads (a row of 2048 x 4096 11.9 -> 9.5 us), and for few workgroups.
// ROWS: of a workgroup, 64, or 16 where workgroups are few (narrow outputs: their rows' chains then run side by side).
template <int DUAL, int UB, int ROWS>
__global__ __launch_bounds__(256) void gemm_any_rows_kernel(AnyGemmArgs p) {
  constexpr int NM = 1 + DUAL;
  __shared__ f32x4 red[4][2 * NM][64];
  int grp, r0, rend;
  if (!locate_tile(p, blockIdx.y, grp, r0, rend, ROWS)) return;
  const int64_t b = blockIdx.z, wsel = p.group_off != nullptr ? grp : b;
  const int n0 = blockIdx.x * 16, K = p.K;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = l & 15, lk = 8 * (l >> 4);
  const int n = n0 + lr;
  const bf16_t* A = reinterpret_cast<const bf16_t*>(p.a) + b * p.a_bs;
  const int64_t wo = wsel * p.w_bs + (int64_t)min(n, p.N - 1) * p.ldw;   // (columns past N: the last one's, never stored)
  const bf16_t* w = reinterpret_cast<const bf16_t*>(p.w) + wo;
  const bf16_t* w2 = DUAL ? reinterpret_cast<const bf16_t*>(p.w2) + wo : nullptr;
  rend = min(rend, r0 + ROWS);
  for (; r0 < rend; r0 += 32) {
    const bool two = ROWS > 16 && rend - r0 > 16;   // (workgroup-uniform)
    const bf16_t* ar[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {      // (rows past the end: the pass's first, never stored)
      const int m = r0 + 16 * i + lr < rend ? r0 + 16 * i + lr : r0;
      ar[i] = A + (int64_t)(p.a_rows ? p.a_rows[m] : m) * p.lda;
    }
    f32x4 acc[2][NM];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int d = 0; d < NM; ++d) acc[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto run = [&](auto mt) {
      constexpr int MT = decltype(mt)::value;
      for (int k0 = 64 * wv; k0 < K; k0 += 256 * UB) {
        uint4 wf[UB][2][NM], af[UB][2][MT];
#pragma unroll
        for (int u = 0; u < UB; ++u)
#pragma unroll
          for (int st = 0; st < 2; ++st) {
            const int k = min(k0 + 256 * u + 32 * st + lk, K - 8);   // (past K: a clamped address, A zeroed below)
            wf[u][st][0] = ld16(w + k);
            if (DUAL) wf[u][st][NM - 1] = ld16(w2 + k);
#pragma unroll
            for (int i = 0; i < MT; ++i) af[u][st][i] = ld16(ar[i] + k);
          }
#pragma unroll
        for (int u = 0; u < UB; ++u)
#pragma unroll
          for (int st = 0; st < 2; ++st) {
            const bool in = k0 + 256 * u + 32 * st + lk < K;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              const bf16x8 a = as_bf16x8(in ? af[u][st][i] : make_uint4(0, 0, 0, 0));
#pragma unroll
              for (int d = 0; d < NM; ++d) acc[i][d] = mfma16(a, as_bf16x8(wf[u][st][d]), acc[i][d]);
            }
          }
      }
    };
    if (two) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
    // what the finishing waves need besides is on its way while the others arrive
    const int mw = r0 + 16 * wv + 4 * (l >> 4);   // first of this lane's four rows, if its wave finishes some
    const bool last = wv < 2 && (wv == 0 || two);
    float gl[4] = {0.f, 0.f, 0.f, 0.f}, bias = 0.f;
    if (last && p.bias != nullptr) bias = p.bias[min(n, p.N - 1)];
    if (last && p.gate != nullptr) {
      const int64_t gc = b * p.g_bs + (int64_t)min(n, p.N - 1) * p.g_cs;
      if (p.gate_f32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) gl[e] = reinterpret_cast<const float*>(p.gate)[(int64_t)min(mw + e, rend - 1) * p.ldg + gc];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) gl[e] = bf2f(reinterpret_cast<const bf16_t*>(p.gate)[(int64_t)min(mw + e, rend - 1) * p.ldg + gc]);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int d = 0; d < NM; ++d)
        if (i == 0 || two) red[wv][i * NM + d][l] = acc[i][d];
    __syncthreads();
    if (last && n < p.N) {
      f32x4 s[NM];
#pragma unroll
      for (int d = 0; d < NM; ++d) s[d] = (red[0][wv * NM + d][l] + red[1][wv * NM + d][l]) + (red[2][wv * NM + d][l] + red[3][wv * NM + d][l]);
      with_act<DUAL>(p, [&](auto act) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (mw + e >= rend) continue;
          float v = act_val<decltype(act)::value>(p, s[0][e] + bias, DUAL ? s[NM - 1][e] : 0.f);
          if (p.gate != nullptr) v *= sigmoidf_(gl[e]);
          store_value(p, (int64_t)(mw + e) * p.ldo + b * p.o_bs + n, v);
        }
      });
    }
    __syncthreads();   // (the next pass writes red again)
  }
}

// LDS-tiled form. Host-checked: K, the row strides and the batch strides are multiples of 8 elements, the bases
// 16-B aligned, K >= 8. Block tile 128 rows x 128 weight rows (DUAL: rows 0..63 of the tile are W's, 64..127 the
// same columns of W2, so a lane holds gate and up of one output); wave (wm, wn) owns rows 64 wm .. and 4 x 4 MFMA
// tiles. A k-step's 128 x 32 A and weight tiles are two 16-B pieces per thread each; rows past the group's end
// read the tile's first row and columns past N the last one (both dropped at the store), k past K reads a
// clamped address and zeroes the A piece. What bounds it is a k-step's way from memory, so two of them are under way (AHEAD; us in an
// engine step, one -> two: 8 experts at 4096 rows, pairs of 1024 x 2048 69.8 -> 64.3, 2048 x 1024 53.7 -> 47.8; 2048 rows of 1024 x 1024
// 20.4 -> 20.0, warm 21.8 -> 16.6). Where K is short and workgroups are many, the registers of the second step are better spent on a fourth
// workgroup per CU: 12 products of 512 x 128 at 2048 rows 14.2 -> 13.6, 16 19.0 -> 16.8 (two workgroups per CU: 10.2 -> 10.6).
constexpr int LM = 128, LKS = 32, LPAD = LKS + 8;
// OUT: how the outputs are stored, apart so that one way's work does not slow the others (gates in the plain form: 12 products of 512 x 128
// at 2048 rows 13.4 -> 17.9 us). OUT_GATED: bf16 in whole pieces, times a gate. OUT_F32: fp32, 64 rows at a time through LDS, in whole lines
// (1808 rows of 3072 x 96 19.5 -> 9.7 us, 1801 of 1024 x 128 16.7 -> 6.8 against a store per value).
enum { OUT_PLAIN = 0, OUT_GATED = 1, OUT_F32 = 2 };
constexpr int LDS_TILE_BYTES = 4 * LM * LPAD * 2;   // operand buffers of gemm_any_lds_kernel, the least that lds_store() may use
// The outputs of a 128-row block tile from the waves' accumulators, by way of LDS that nobody reads or writes any more
template <int DUAL, int OUT>
__device__ __forceinline__ void lds_store(const AnyGemmArgs& p, const f32x4 (&acc)[4][4], bf16_t* smem, int64_t b, int r0, int rend, int n0) {
  constexpr int WN = DUAL ? 64 : 128;  // columns of each weight matrix per block
  constexpr int OPAD = WN + 8;         // padded row of the staged outputs
  static_assert(LM * OPAD * 2 <= LDS_TILE_BYTES, "the staged outputs fit the operand buffers");
  const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6;
  const int wm = wv & 1, wn = wv >> 1, lr = l & 15, lg = l >> 4;
  if constexpr (OUT == OUT_F32) {
    constexpr int FP = 128 + 4;
    static_assert(!DUAL && 64 * FP * 4 <= LDS_TILE_BYTES, "64 rows fit the operand buffers");
    float* fs = reinterpret_cast<float*>(smem);
    float* out = reinterpret_cast<float*>(p.out) + b * p.o_bs;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (wm == half)
        with_act<DUAL>(p, [&](auto act) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int col = wn * 64 + j * 16 + lr;
            const float bias = p.bias ? p.bias[min(n0 + col, p.N - 1)] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) fs[(i * 16 + 4 * lg + e) * FP + col] = act_val<decltype(act)::value>(p, acc[i][j][e] + bias, 0.f);
          }
        });
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 64 * 32 / 256; ++u) {
        const int x = tid + 256 * u, row = x >> 5, col = (x & 31) * 4, m = r0 + 64 * half + row;
        if (m < rend && n0 + col < p.N) *reinterpret_cast<f32x4*>(out + (int64_t)m * p.ldo + n0 + col) = *reinterpret_cast<const f32x4*>(&fs[row * FP + col]);
      }
      if (half == 0) __syncthreads();
    }
    return;
  }
  if (OUT == OUT_GATED || p.vec_out) {  // bf16 rows of whole 16-B pieces: staged in LDS, then stored whole
    // a gate: one logit per row, or its tile brought in whole pieces to where the outputs will lie, each lane's to its own
    const bool tiled = OUT == OUT_GATED && p.g_cs != 0, rowed = OUT == OUT_GATED && p.g_cs == 0;
    float rg[4][4];
    if (rowed) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t at = (int64_t)min(r0 + wm * 64 + i * 16 + 4 * lg + e, rend - 1) * p.ldg + b * p.g_bs;
          rg[i][e] = sigmoidf_(p.gate_f32 ? reinterpret_cast<const float*>(p.gate)[at] : bf2f(reinterpret_cast<const bf16_t*>(p.gate)[at]));
        }
    } else if (tiled) {
      const bf16_t* gate = reinterpret_cast<const bf16_t*>(p.gate) + b * p.g_bs;
#pragma unroll
      for (int u = 0; u < LM * WN / 8 / 256; ++u) {
        const int x = tid + 256 * u, row = x / (WN / 8), col = (x % (WN / 8)) * 8;
        if (n0 + col < p.N) *reinterpret_cast<uint4*>(&smem[row * OPAD + col]) = ld16(gate + (int64_t)min(r0 + row, rend - 1) * p.ldg + n0 + col);
      }
      __syncthreads();
    }
    with_act<DUAL>(p, [&](auto act) {
#pragma unroll
      for (int j = 0; j < (DUAL ? 2 : 4); ++j) {
        const int col = (DUAL ? wn * 32 : wn * 64) + j * 16 + lr;
        const float bias = p.bias ? p.bias[min(n0 + col, p.N - 1)] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            bf16_t* at = &smem[(wm * 64 + i * 16 + 4 * lg + e) * OPAD + col];
            float v = act_val<decltype(act)::value>(p, acc[i][j][e] + bias, DUAL ? acc[i][j + 2][e] : 0.f);
            if (rowed) v *= rg[i][e];
            if (tiled) v *= sigmoidf_(bf2f(*at));
            *at = f2bf(v);
          }
      }
    });
    __syncthreads();
    bf16_t* out = reinterpret_cast<bf16_t*>(p.out) + b * p.o_bs;
#pragma unroll
    for (int u = 0; u < LM * WN / 8 / 256; ++u) {
      const int x = tid + 256 * u, row = x / (WN / 8), col = (x % (WN / 8)) * 8;
      if (r0 + row < rend && n0 + col < p.N)
        *reinterpret_cast<uint4*>(out + (int64_t)(r0 + row) * p.ldo + n0 + col) =
            *reinterpret_cast<const uint4*>(&smem[row * OPAD + col]);
    }
    return;
  }
  with_act<DUAL>(p, [&](auto act) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < (DUAL ? 2 : 4); ++j) {
        const int n = n0 + (DUAL ? wn * 32 : wn * 64) + j * 16 + lr, m = r0 + wm * 64 + i * 16 + 4 * lg;
        if (n >= p.N) continue;
        const float bias = p.bias ? p.bias[n] : 0.f;
        float gl[4];   // (asked for together)
        if (p.gate != nullptr) {
          const int64_t gc = b * p.g_bs + (int64_t)n * p.g_cs;
          if (p.gate_f32) {
#pragma unroll
            for (int e = 0; e < 4; ++e) gl[e] = reinterpret_cast<const float*>(p.gate)[(int64_t)min(m + e, rend - 1) * p.ldg + gc];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) gl[e] = bf2f(reinterpret_cast<const bf16_t*>(p.gate)[(int64_t)min(m + e, rend - 1) * p.ldg + gc]);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (m + e >= rend) continue;
          float v = act_val<decltype(act)::value>(p, acc[i][j][e] + bias, DUAL ? acc[i][j + 2][e] : 0.f);
          if (p.gate != nullptr) v *= sigmoidf_(gl[e]);
          store_value(p, (int64_t)(m + e) * p.ldo + b * p.o_bs + n, v);
        }
      }
  });
}

template <int DUAL, int AHEAD, int OUT>
__global__ __launch_bounds__(256, 3) void gemm_any_lds_kernel(AnyGemmArgs p) {
  constexpr int WN = DUAL ? 64 : 128;  // columns of each weight matrix per block
  __shared__ __attribute__((aligned(16))) bf16_t smem[4 * LM * LPAD];  // two A and two weight buffers, then the outputs
  typedef bf16_t Tile[LM][LPAD];
  Tile* As = reinterpret_cast<Tile*>(smem);
  Tile* Ws = As + 2;
  int grp, r0, rend;
  if (!locate_tile(p, blockIdx.y, grp, r0, rend, LM)) return;
  const int64_t b = blockIdx.z;
  const int64_t wsel = (p.group_off != nullptr) ? grp : b;
  const int n0 = blockIdx.x * WN;
  const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6;
  const int wm = wv & 1, wn = wv >> 1, lr = l & 15, lg = l >> 4;
  const bf16_t* A = reinterpret_cast<const bf16_t*>(p.a) + b * p.a_bs;
  const bf16_t* W = reinterpret_cast<const bf16_t*>(p.w) + wsel * p.w_bs;
  const bf16_t* W2 = DUAL ? reinterpret_cast<const bf16_t*>(p.w2) + wsel * p.w_bs : nullptr;
  const int K = p.K;
  const int kq = (tid & 3) * 8;  // this thread's quarter of a k-step
  const bf16_t* asrc[2];
  const bf16_t* wsrc[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int row = (tid >> 2) + 64 * u;
    const int m = r0 + row < rend ? r0 + row : r0;
    asrc[u] = A + (int64_t)(p.a_rows ? p.a_rows[m] : m) * p.lda;
    const int n = min(n0 + (DUAL ? (row & 63) : row), p.N - 1);
    wsrc[u] = ((DUAL && row >= 64) ? W2 : W) + (int64_t)n * p.ldw;
  }
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Step {
    uint4 a[2], w[2];
  };
  auto fetch = [&](Step& x, int k0) {   // (past K: a clamped address)
    const int k = k0 + kq, kk = min(k, K - 8);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      x.a[u] = ld16(asrc[u] + kk);
      x.w[u] = ld16(wsrc[u] + kk);
    }
  };
  auto stage = [&](const Step& x, int buf, int k0) {
    const bool in = k0 + kq < K;   // a zero A piece zeroes the product
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = (tid >> 2) + 64 * u;
      *reinterpret_cast<uint4*>(&As[buf][row][kq]) = in ? x.a[u] : make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(&Ws[buf][row][kq]) = x.w[u];
    }
  };
  auto compute = [&](int buf) {
    bf16x8 af[4], wf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) af[i] = as_bf16x8(*reinterpret_cast<const uint4*>(&As[buf][wm * 64 + i * 16 + lr][8 * lg]));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int wrow = DUAL ? (j >> 1) * 64 + wn * 32 + (j & 1) * 16 + lr : wn * 64 + j * 16 + lr;
      wf[j] = as_bf16x8(*reinterpret_cast<const uint4*>(&Ws[buf][wrow][8 * lg]));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma16(af[i], wf[j], acc[i][j]);
  };
  // A buffer is rewritten one step later, after the barrier that every wave reaches only when it has read it (the barriers wait for
  // LDS traffic only).
  Step xa;
  fetch(xa, 0);
  if constexpr (AHEAD == 2) {
    // k-step k0 from LDS; x: what was asked for step k0 + LKS, two steps ago, goes to the other buffer, then asks for the step
    // after the next
    auto step = [&](Step& x, int buf, int k0) {
      compute(buf);
      stage(x, buf ^ 1, k0 + LKS);
      fetch(x, k0 + 3 * LKS);
      lds_barrier();
    };
    Step xb;
    fetch(xb, LKS);
    stage(xa, 0, 0);
    fetch(xa, 2 * LKS);
    lds_barrier();
    int k0 = 0;
    for (; k0 + LKS < K; k0 += 2 * LKS) {
      step(xb, 0, k0);
      step(xa, 1, k0 + LKS);
    }
    if (k0 < K) step(xb, 0, k0);
  } else {
    stage(xa, 0, 0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += LKS) {
      const bool more = k0 + LKS < K;
      if (more) fetch(xa, k0 + LKS);
      compute(buf);
      if (more) stage(xa, buf ^ 1, k0 + LKS);
      __syncthreads();
      buf ^= 1;
    }
  }
  lds_store<DUAL, OUT>(p, acc, smem, b, r0, rend, n0);
}

// The same block tile from operands brought by LDS-DMA, for K of whole 64-k stages: both matrices are rows of k, so both lie in LDS as x does
// in the prompt GEMMs (lds_rows.h), and the loop is theirs (gemm_prompt.h): fragments of a k-step read during the MFMAs of the one before,
// one barrier per stage between its two k-steps, accumulators in AGPRs. By way of registers a thread brought 64 B of a row at a time, which
// keeps the CU's address path busy four times as long as whole 128-B lines.
template <int DUAL, int NS, int OUT>
__global__ __launch_bounds__(256, NS == 2 ? 2 : 1) void gemm_any_dma_kernel(AnyGemmArgs p) {
  constexpr int WN = DUAL ? 64 : 128, STAGE = 32 * 1024, PPW = 8, AB = 16 * 1024;  // W tiles, then A tiles (16 rows x 64 k: 2 KiB each)
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  int grp, r0, rend;
  if (!locate_tile(p, blockIdx.y, grp, r0, rend, LM)) return;
  const int64_t b = blockIdx.z;
  const int64_t wsel = (p.group_off != nullptr) ? grp : b;
  const int n0 = blockIdx.x * WN;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv & 1, wn = wv >> 1;
  const bf16_t* A = reinterpret_cast<const bf16_t*>(p.a) + b * p.a_bs;
  const bf16_t* W = reinterpret_cast<const bf16_t*>(p.w) + wsel * p.w_bs;
  const bf16_t* W2 = DUAL ? reinterpret_cast<const bf16_t*>(p.w2) + wsel * p.w_bs : nullptr;
  const int nk = p.K >> 6;
  const bf16_t* src[PPW];   // pieces of this wave: two tiles of W, two of A, two halves each
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tile = 2 * wv + (i >> 1), row = tile * 16 + 8 * (i & 1) + (l >> 3), col = x_piece_col(i & 1, l);
    const int n = min(n0 + (DUAL ? (row & 63) : row), p.N - 1);
    src[i] = ((DUAL && row >= 64) ? W2 : W) + (int64_t)n * p.ldw + col;
    const int m = r0 + row < rend ? r0 + row : r0;
    src[4 + i] = A + (int64_t)(p.a_rows ? p.a_rows[m] : m) * p.lda + col;
  }
  const uint32_t lds0 = lds_addr_of(dsm) + (uint32_t)wv * 4096u;
  auto issue = [&](int i, int st, int buf) {
    glds16(src[i] + (size_t)st * 64, lds0 + (uint32_t)(buf * STAGE + (i >> 2) * AB + (i & 3) * 1024));
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));  // (written here, well before the first mfma_acc)
    }
  uint4 af[2][4], wf[2][4];
  const int xo[2] = {x_frag_off(0, l), x_frag_off(1, l)};
  // fragment read rd, in the order in which a phase needs them: A tile 0, W tiles, the other A tiles
  auto read_frag = [&](int rd, int ks, const char* sb) {
    if (rd == 0 || rd > 4) {
      const int i = rd == 0 ? 0 : rd - 4;
      af[ks][i] = *reinterpret_cast<const uint4*>(sb + AB + (wm * 4 + i) * 2048 + xo[ks]);
    } else {
      const int j = rd - 1;
      wf[ks][j] = *reinterpret_cast<const uint4*>(sb + (DUAL ? (j >> 1) * 4 + wn * 2 + (j & 1) : wn * 4 + j) * 2048 + xo[ks]);
    }
  };
  // the MFMAs of k-step ks, between them the reads of the other k-step (from sb) and, if `dma`, the pieces of stage st
  auto phase = [&](auto ksc, const char* sb, auto dmac, int st, int buf) {
    constexpr int ks = decltype(ksc)::value, dma = decltype(dmac)::value;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i < 2) {
#pragma unroll
        for (int u = 0; u < 4; ++u) read_frag(4 * i + u, ks ^ 1, sb);
      }
      if constexpr (dma) {
        issue(2 * i, st, buf);
        issue(2 * i + 1, st, buf);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) mfma_acc(acc[i][j], af[ks][i], wf[ks][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
#pragma unroll
  for (int s0 = 0; s0 < NS; ++s0)
#pragma unroll
    for (int i = 0; i < PPW; ++i) issue(i, s0 < nk ? s0 : nk - 1, s0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * PPW) : "memory");
#pragma unroll
  for (int rd = 0; rd < 8; ++rd) read_frag(rd, 0, dsm);
  int buf = 0;
  for (int t = 0; t < nk; ++t) {
    const char* sb = dsm + buf * STAGE;
    const int nb = buf + 1 == NS ? 0 : buf + 1;
    phase(C0{}, sb, C0{}, 0, 0);
    // this stage is read (its second k-step is in registers), the next one has landed: both for every wave
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * PPW) : "memory");
    phase(C1{}, dsm + nb * STAGE, C1{}, t + NS < nk ? t + NS : nk - 1, buf);   // past the end: clamped duplicates, never used
    buf = nb;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15\n\ts_barrier" ::: "memory");  // the trailing duplicates, of every wave
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[i][j]));
  lds_store<DUAL, OUT>(p, acc, reinterpret_cast<bf16_t*>(dsm), b, r0, rend, n0);
}

template <int DUAL, int NS, int OUT>
void launch_any_dma(const AnyGemmArgs& p, dim3 grid, hipStream_t st) {
  auto kern = gemm_any_dma_kernel<DUAL, NS, OUT>;
  static bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, NS * 32 * 1024) == hipSuccess;
  (void)attr;
  hipLaunchKernelGGL(kern, grid, dim3(256), NS * 32 * 1024, st, p);
}

template <typename T>
__device__ __forceinline__ float ldf(const T* q);
template <>
__device__ __forceinline__ float ldf<float>(const float* q) { return *q; }
template <>
__device__ __forceinline__ float ldf<bf16_t>(const bf16_t* q) { return bf2f(*q); }

constexpr int BK = 16;

template <typename T, int DUAL>
__global__ __launch_bounds__(256) void gemm_any_fma_kernel(AnyGemmArgs p) {
  __shared__ float As[BK][BM + 4];
  __shared__ float Ws[BK][BN + 4];
  __shared__ float Us[DUAL ? BK : 1][BN + 4];
  int grp, r0, rend;
  if (!locate_tile(p, blockIdx.y, grp, r0, rend)) return;
  const int64_t b = blockIdx.z;
  const int64_t wsel = (p.group_off != nullptr) ? grp : b;
  const int n0 = blockIdx.x * BN;
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const T* A = reinterpret_cast<const T*>(p.a) + b * p.a_bs;
  const T* W = reinterpret_cast<const T*>(p.w) + wsel * p.w_bs;
  const T* W2 = DUAL ? reinterpret_cast<const T*>(p.w2) + wsel * p.w_bs : nullptr;
  // loader: row tid >> 2 of the tile, 4 consecutive k from (tid & 3) * 4
  const int lrow = tid >> 2, lk = (tid & 3) * 4;
  const int am = r0 + lrow;
  const bool aok = am < rend;
  const T* ap = A + (int64_t)(aok ? (p.a_rows ? p.a_rows[am] : am) : 0) * p.lda;
  const int wn_ = n0 + lrow;
  const bool wok = wn_ < p.N;
  const T* wp = W + (int64_t)(wok ? wn_ : 0) * p.ldw;
  const T* up = DUAL ? W2 + (int64_t)(wok ? wn_ : 0) * p.ldw : nullptr;
  float acc[4][4], acc2[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) { acc[i][j] = 0.f; acc2[i][j] = 0.f; }
  for (int k0 = 0; k0 < p.K; k0 += BK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + lk + e;
      const bool kin = k < p.K;
      As[lk + e][lrow] = (aok && kin) ? ldf<T>(ap + k) : 0.f;
      Ws[lk + e][lrow] = (wok && kin) ? ldf<T>(wp + k) : 0.f;
      if (DUAL) Us[lk + e][lrow] = (wok && kin) ? ldf<T>(up + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      float av[4], wv[4], uv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        wv[j] = Ws[k][tx * 4 + j];
        uv[j] = DUAL ? Us[k][tx * 4 + j] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
          if (DUAL) acc2[i][j] = fmaf(av[i], uv[j], acc2[i][j]);
        }
    }
    __syncthreads();
  }
  with_act<DUAL>(p, [&](auto act) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = r0 + ty * 4 + i;
      if (m >= rend) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + tx * 4 + j;
        if (n >= p.N) continue;
        const float bias = p.bias ? p.bias[n] : 0.f;
        store_out(p, b, m, n, act_val<decltype(act)::value>(p, acc[i][j] + bias, DUAL ? acc2[i][j] : 0.f));
      }
    }
  });
}

// "1": large products through the LDS-tiled kernel (default); "0": the direct-fragment kernels only
bool lds_tiles() {
  static const bool v = [] {
    const char* e = getenv("VGATE_GEMM_ANY_LDS");
    return e == nullptr || e[0] != '0';
  }();
  return v;
}

int cu_count() {
  static const int n = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev);
    return v > 0 ? v : 256;
  }();
  return n;
}

bool simple_only() {
  static const bool v = [] {
    const char* e = getenv("VGATE_GEMM_ANY_FMA");
    return e != nullptr && e[0] == '1';
  }();
  return v;
}

}  // namespace

void launch_gemm_any(const AnyGemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.N <= 0 || g.batch <= 0) return;
  const int mt = (g.M + BM - 1) / BM + (g.group_off ? g.groups : 0);
  const dim3 grid((g.N + BN - 1) / BN, mt, g.batch), block(256);
  const bool dual = g.w2 != nullptr;
  if (g.in_f32) {
    if (dual) hipLaunchKernelGGL((gemm_any_fma_kernel<float, 1>), grid, block, 0, st, g);
    else hipLaunchKernelGGL((gemm_any_fma_kernel<float, 0>), grid, block, 0, st, g);
  } else if (simple_only()) {
    if (dual) hipLaunchKernelGGL((gemm_any_fma_kernel<bf16_t, 1>), grid, block, 0, st, g);
    else hipLaunchKernelGGL((gemm_any_fma_kernel<bf16_t, 0>), grid, block, 0, st, g);
  } else {
    auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    const bool al = g.K >= 8 && g.K % 8 == 0 && g.lda % 8 == 0 && g.ldw % 8 == 0 && g.a_bs % 8 == 0 &&
                    g.w_bs % 8 == 0 && a16(g.a) && a16(g.w) && (!dual || a16(g.w2));
    // Few rows, or few 64 x 64 tiles, leave the chip idle behind chains of loads: 16 columns and a quarter of K per wave there. us, the
    // tiles' kernels / this form: 64 x 1024 at 32 rows 12.4, 6.1; 128 x 512 of 12 products at 64 rows 12.4, 6.9, at 192 (72 tiles) 12.5, 8.3, at
    // 384 (144) 12.7, 15; 256 x 1024 at 2048 (128) 19.7, 16.0. Of broad products below 1024 rows, which run as 64 x 128 tiles, up to
    // 256: 2048 x 1024 at 384 rows (192) 29.7, 20.6, at 512 (256) 29.8, 25.6; from 1024 rows the LDS tiles are ahead of that. Experts: 8 of
    // 1024 x 2048 pairs with 32 rows each 45, 27; above the line 32 of 1536 x 1024 with 8 (864 tiles) 22, 25.
    const bool broad = g.N >= 512 && g.M >= 256;
    const int64_t tiles = (int64_t)grid.x * mt * g.batch;
    if (al && (g.group_off ? g.M <= 512 && tiles < 768 : g.M <= 64 || tiles <= (!broad ? 128 : (g.M < 1024 ? 256 : 64)))) {
      const dim3 gr((g.N + 15) / 16, mt, g.batch);
      // A workgroup of 16 rows where all of them together are no more than the CUs and a wave's k is a chain of several loads, which
      // then are all under way (us, 64 rows / 16: 8 x 1024 at 32 rows 4.7, 3.6, at 2048 8.3, 3.8; 16 x 1536 at 512 11.4, 6.0; 128 x 768 at 300
      // 7.8, 4.1; 1024 x 512 at 64, two passes in one, 6.4, 4.1). With one pass of K = 512 there is little to gain (128 x 512 at 32
      // rows 3.9, 4.0, at 8 3.3, 3.7). Half as many loads under way where their last round would lie past K by half (128 x 1536 at 16 rows
      // by 64 5.5, by 16 with four 6.2).
      const dim3 gn(gr.x, (g.M + 15) / 16, g.batch);
      if (!g.group_off && g.K > (g.M > 32 ? 256 : 512) && (int64_t)gn.x * gn.y * gn.z <= cu_count()) {
        auto even = [&](int k) { return (g.K + 2 * k - 1) / (2 * k) * 2 == (g.K + k - 1) / k; };   // rounds of 2 k: none of them half empty
        auto kern = dual ? (even(256) ? gemm_any_rows_kernel<1, 2, 16> : gemm_any_rows_kernel<1, 1, 16>)
                         : (even(512) ? gemm_any_rows_kernel<0, 4, 16> : gemm_any_rows_kernel<0, 2, 16>);
        hipLaunchKernelGGL(kern, gn, block, 0, st, g);
        return;
      }
      const bool deep = g.M <= 8 && g.K > 512;
      auto kern = dual ? (deep ? gemm_any_rows_kernel<1, 2, BM> : gemm_any_rows_kernel<1, 1, BM>)
                       : (deep ? gemm_any_rows_kernel<0, 4, BM> : gemm_any_rows_kernel<0, 1, BM>);
      hipLaunchKernelGGL(kern, gr, block, 0, st, g);
      return;
    }
    // enough 64 x 128 tiles to fill the chip; experts with few rows each take tiles whose waves split K (32 of 512 x 512 with 24 rows
    // each 12.5 us, as wide tiles 19.1) until the LDS tiles come in (64 of 1024 x 1024 with 16 each 31.6 us, as LDS tiles 27.1)
    const bool wide = al && broad && (!g.group_off || g.M > (g.M >= 1024 ? 15 : 32) * g.groups);
    const dim3 gridw((g.N + 127) / 128, mt, g.batch);
    // enough 128-row tiles; also where whole 128-column tiles of many products fill half the chip (us at 2048 rows: 12 of
    // 128 x 512 27.9 -> 15.8, 8 of 256 x 128 14.1 -> 7.3, 2 of 128 x 256 stay at 9; with gates, which come
    // through LDS in whole pieces, from 192 tiles on: 12 of 128 x 512 30.8 -> 23.7, 8 of 128 x 256 15.3, as wide tiles 18.3)
    const int mt128 = (g.M + LM - 1) / LM + (g.group_off ? g.groups : 0);
    const bool gates = g.gate == nullptr || g.g_cs == 0 || (g.g_cs == 1 && !g.gate_f32 && g.ldg % 8 == 0 && g.g_bs % 8 == 0 && a16(g.gate));
    const bool vec = !g.out_f32 && gates && !(dual && g.gate != nullptr) && g.N % 8 == 0 && g.ldo % 8 == 0 && g.o_bs % 8 == 0 && a16(g.out);
    const bool heads = al && !dual && !g.group_off && (g.gate == nullptr || vec) && g.N % 128 == 0 &&
                       (int64_t)(g.N / 128) * mt128 * g.batch >= (g.gate != nullptr ? 192 : 128);
    if ((wide || heads) && g.M >= 1024 && lds_tiles()) {
      AnyGemmArgs v = g;
      v.vec_out = vec;
      const dim3 grid2((g.N + (dual ? 63 : 127)) / (dual ? 64 : 128), mt128, g.batch);
      const bool one = !dual && g.K <= 256 && (int64_t)grid2.x * grid2.y * grid2.z > 512;
      const bool gated = vec && g.gate != nullptr;
      const bool f32 = g.out_f32 && !dual && g.gate == nullptr && g.N % 4 == 0 && g.ldo % 4 == 0 && g.o_bs % 4 == 0 && a16(g.out);
      // By LDS-DMA from four stages of k on (us, through registers -> by DMA: K = 64 of 3072 columns 9.5, 9.6; 12 products of 512 x 128 at 2048 rows
      // 12.9, 15.2, 16 of them 15.4, 18.8; 4096 x 256 at 1024 8.6 -> 8.3, 12 of 128 x 512 11.2, 11.3): two stages
      // in LDS and two workgroups to a CU, or four stages where there is one at most
      // (two / four: 1024 x 4096 at 2048 rows, 128 workgroups, 47.6 -> 43.3 / 33.6; 8 experts of 1024 x 2048 with 150 rows each, 144, 28.5 -> 25.7 / 21.6,
      // with 500, 320, 45.8 -> 33.2 / 42.2; pairs of 2048 x 1024 with 500, 64.8 -> 61.6 / 73.6). Workgroups past an expert's rows exit and do
      // not count, but the host knows only about how many those are: in 110 drawn products four stages were ahead by 5 to 25 % wherever up to a
      // workgroup per CU had rows (32 experts of 768 x 2944 with 46 rows each, 264, 192 of them with rows, registers 48.7, 52.3 / 39.3; 32 of 896 x 1600 with 38
      // 30.7, 33.1 / 24.6; 8 of 1792 x 1024 with 178 19.7, 21.4 / 18.5) and behind by 10 to 25 % right above that (8 of 1344 x 2944 with 379, 264 with rows,
      // 74.4, 58.4 / 73.5), so they are taken up to eleven twelfths of the CUs, where one estimate of the 110 was too low. Through registers a CU holds three workgroups: with more than two to a CU that wins over short K
      // (4224 x 256 with gates at 1985 rows, 528, 25.8, 32.7; 4536 x 320 28.5, 35.0; 5440 x 512 at 3324 51.0, 55.7; 5760 x 960 at 2124 51.1, 55.2; without
      // gates 2712 x 320 at 3958, fp32, 682, 20.5, 22.4, and even at 1024 x 512 of 12; 32 experts of 3072 x 576 with 38 rows each, 768, 24.7, 28.2, pairs of
      // 2176 x 640 with 51, 1088, 41.0, 45.7, of 3072 x 640 with 112 31.1, 34.0). What bounds the many is the operands' way through L2, 25 B a clock and CU.
      const int64_t blocks = (int64_t)grid2.x * grid2.y * grid2.z, cus = cu_count();
      const int64_t busy = g.group_off ? (int64_t)grid2.x * std::max(g.groups, mt128 - (g.groups + 1) / 2) : blocks;   // (experts: about so many have rows)
      if (g.K % 64 == 0 && g.K >= 256 && (busy <= 2 * cus || g.K > (gated ? 1024 : g.group_off ? 640 : 512))) {
        const bool few = blocks <= cus || (g.group_off && 12 * busy <= 11 * cus);
        auto by_dma = [&](auto du, auto out) {
          constexpr int DU = decltype(du)::value, O = decltype(out)::value;
          if (few) launch_any_dma<DU, 4, O>(v, grid2, st);
          else launch_any_dma<DU, 2, O>(v, grid2, st);
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        if (dual) by_dma(I1{}, std::integral_constant<int, OUT_PLAIN>{});
        else if (gated) by_dma(I0{}, std::integral_constant<int, OUT_GATED>{});
        else if (f32) by_dma(I0{}, std::integral_constant<int, OUT_F32>{});
        else by_dma(I0{}, std::integral_constant<int, OUT_PLAIN>{});
        return;
      }
      auto kern = dual ? gemm_any_lds_kernel<1, 2, OUT_PLAIN>
                       : (gated ? gemm_any_lds_kernel<0, 2, OUT_GATED>
                                : (f32 ? gemm_any_lds_kernel<0, 2, OUT_F32>
                                       : (one ? gemm_any_lds_kernel<0, 1, OUT_PLAIN> : gemm_any_lds_kernel<0, 2, OUT_PLAIN>)));
      hipLaunchKernelGGL(kern, grid2, block, 0, st, v);
    } else if (dual && wide) hipLaunchKernelGGL((gemm_any_mfma_kernel<1, true, 4>), gridw, block, 0, st, g);
    else if (wide) hipLaunchKernelGGL((gemm_any_mfma_kernel<0, true, 4>), gridw, block, 0, st, g);
    else if (dual && al) hipLaunchKernelGGL((gemm_any_mfma_kernel<1, true, 2>), grid, block, 0, st, g);
    else if (dual) hipLaunchKernelGGL((gemm_any_mfma_kernel<1, false, 2>), grid, block, 0, st, g);
    else if (al) hipLaunchKernelGGL((gemm_any_mfma_kernel<0, true, 2>), grid, block, 0, st, g);
    else hipLaunchKernelGGL((gemm_any_mfma_kernel<0, false, 2>), grid, block, 0, st, g);
  }
}

}  // namespace vgate
