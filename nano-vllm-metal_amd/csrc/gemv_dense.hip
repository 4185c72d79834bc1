// Dense W4A16 products of few rows (one expert): out[M, R] = x . dequant(W)^T
// for decode batches of the attention and MLP projections
// (layers/linear.py:92-126), and the gate/up pair of the dense MLP with SwiGLU
// (models/qwen3.py:176-184, silu op by op as layers/activation.py:21-24).
//
// Bound: latency.  A projection's weights (4.5 to 7 MB) are 1 to 1.5 us of
// HBM time, so a call is its dependent round trips.  The unit-list GEMV
// (gemv.hip) builds a chunk table, waits for the activations of each 16-row
// chunk, keeps at most 64 groups of a reduction in its wavefronts' registers
// (longer ones ran on the prefill GEMM) and reads the weights again for every
// chunk.  Here:
//  * a block owns 16 weight rows and 16 rows of x, and there is no prologue:
//    its NW wavefronts split the reduction in runs of whole 128-wide pairs of
//    groups, and each issues the weights, scales, biases and activations of
//    its first RING pairs at once (one round trip, for a reduction of up to
//    128 NW RING all there is);
//  * the activations come in whole 256-byte row segments and reach MFMA
//    operand order through the wavefront's own LDS (loaded in operand order,
//    16 bytes of 16 rows an instruction, 16 rows took 9.0 us at 2048 ->
//    5120 where one took 6.2; this way 6.7 and 6.5);
//  * the wavefronts' partial sums meet in LDS once, summed in order.
// The arithmetic is gemv.hip's: codes as the exact 16-bit floats M + q, the
// group scale applied to float32 sums, then the bias terms (b - M s) times
// the groups' sums of x, four groups a float32 MFMA.  (Each group's sum goes
// through lane swaps and adds: an MFMA that read a dot instruction's result
// right behind it got a stale operand, and the compiler leaves no wait
// there.)
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace nvm {

namespace {

// RING: pairs in flight per wavefront, and pairs between two applications of
// the bias terms.
template <int DT, bool DUAL, int NW, int RING, bool G128>
__global__ __launch_bounds__(64 * NW) void gemv_dense_kernel(const GroupedArgs a) {
  using A = Act<DT>;
  constexpr int NM = DUAL ? 2 : 1;
  constexpr int NB = (RING + 1) / 2;  // bias MFMAs of RING pairs (four groups each)
  constexpr int XP = 272;  // LDS bytes of a row's pair (256 + 16: rows 4 banks apart)
  __shared__ float s_red[NW][NM][4][64];
  __shared__ __attribute__((aligned(16))) uint8_t s_x[NW][16 * XP];

  hoist_args(a.act, a.act_ld, a.act_rows, a.w0, a.s0, a.b0, a.w1, a.s1, a.b1, a.R, a.K, a.out,
             a.out_ld);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, G = lane >> 4;
  const int M = (int)a.act_rows, R = a.R, KW = a.K >> 3, GPR = a.K / (G128 ? 128 : 64);
  const int r0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
  const int np = a.K >> 7, ppw = (np + NW - 1) / NW;
  const int p0 = wv * ppw, p1 = min(np, p0 + ppw);

  rsrc_t wr[NM], sr[NM], br[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    wr[m] = make_rsrc(m ? a.w1 : a.w0, (uint32_t)R * KW * 4);
    sr[m] = make_rsrc(m ? a.s1 : a.s0, (uint32_t)R * GPR * 2);
    br[m] = make_rsrc(m ? a.b1 : a.b0, (uint32_t)R * GPR * 2);
  }
  const rsrc_t xr = make_rsrc(a.act, (uint32_t)(a.act_rows * a.act_ld * 2));
  const int wo = (r0 + col) * KW * 4 + 16 * G;
  const int so = (r0 + col) * GPR * 2;
  // activation load j: rows 4j + lane / 16 of a chunk, 16 bytes at
  // 16 (lane % 16) of the pair
  int xo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = m0 + 4 * j + G;
    xo[j] = row < M ? (int)((int64_t)row * a.act_ld * 2) + 16 * col : kMaskedOffset;
  }

  struct Pair {
    u32x4 w[NM], x[4];
    uint32_t s[NM], b[NM];  // both groups' values (one group of 128: its value)
  };
  auto issue = [&](Pair &q, int ps) {
    if (ps >= p1) return;  // uniform
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      q.w[m] = bload16(wr[m], wo, 64 * ps);
      if constexpr (G128) {
        q.s[m] = bload2(sr[m], so, 2 * ps);
        q.b[m] = bload2(br[m], so, 2 * ps);
      } else {
        q.s[m] = bload4(sr[m], so, 4 * ps);
        q.b[m] = bload4(br[m], so, 4 * ps);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) q.x[j] = bload16(xr, xo[j], 256 * ps);
  };
  f32x4 o[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) o[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t nib_mask = sgpr_const(0x000F000Fu << A::kCodeShift);
  const uint32_t magic = vgpr_const(A::kMagic2);
  float xb[NB], bb[NB][NM];
  auto compute = [&](const Pair &q, int d) {
    // into MFMA operand order through the wavefront's own LDS: step st of the
    // pair covers codes 64(st/2) + 32(G%2) + 16(G/2) + 8(st%2) + 0..7 of row
    // `col` in lane group G, as the weights after swap_pairs
    uint8_t *const xs = s_x[wv];
#pragma unroll
    for (int j = 0; j < 4; ++j) *(u32x4 *)(xs + (4 * j + G) * XP + 16 * col) = q.x[j];
    wave_lds_sync();
    u32x4 xa[4];
#pragma unroll
    for (int st = 0; st < 4; ++st)
      xa[st] = *(const u32x4 *)(xs + col * XP + 64 * (G & 1) + 32 * (G >> 1) + 128 * (st >> 1) +
                                16 * (st & 1));
    wave_lds_sync();
    float ps[2];  // the two groups' sums of x over row `col`, in every lane of it
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      ps[g] = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ps[g] = A::dot2(xa[2 * g + j][i], A::kOne2, ps[g]);
        xa[2 * g + j] = pair_order(xa[2 * g + j]);
      }
      ps[g] += __shfl_xor(ps[g], 16);
      ps[g] += __shfl_xor(ps[g], 32);
    }
    // bias operands: lane (c, G) holds group 4 (d / 2) + G of the RING pairs
    const bool mine = (G >> 1) == (d & 1);
    if (mine) xb[d >> 1] = (G & 1) ? ps[1] : ps[0];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const u32x4 w = swap_pairs(q.w[m]);
      u32x4 bop[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) bop[j] = nibble_pairs_v<A::kCodeShift>(w[j], nib_mask, magic);
      float bp[2];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const float s = (g && !G128) ? A::hi(q.s[m]) : A::lo(q.s[m]);
        const float b = (g && !G128) ? A::hi(q.b[m]) : A::lo(q.b[m]);
        bp[g] = fmaf(-A::kMagic, s, b);
        f32x4 acc = A::mfma16(xa[2 * g], bop[2 * g], f32x4{0.f, 0.f, 0.f, 0.f});
        acc = A::mfma16(xa[2 * g + 1], bop[2 * g + 1], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[m][v] = fmaf(s, acc[v], o[m][v]);
      }
      if (mine) bb[d >> 1][m] = (G & 1) ? bp[1] : bp[0];
    }
  };

  Pair ring[RING];
#pragma unroll
  for (int d = 0; d < RING; ++d) issue(ring[d], p0 + d);
  for (int p = p0; p < p1; p += RING) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      xb[b] = 0.f;
#pragma unroll
      for (int m = 0; m < NM; ++m) bb[b][m] = 0.f;
    }
#pragma unroll
    for (int d = 0; d < RING; ++d) {
      if (p + d < p1) {  // uniform
        compute(ring[d], d);
        issue(ring[d], p + d + RING);
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int m = 0; m < NM; ++m)
        o[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(xb[b], bb[b][m], o[m], 0, 0, 0);
  }
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int v = 0; v < 4; ++v) s_red[wv][m][v][lane] = o[m][v];
  __syncthreads();
  // output (row, column): C row 4G + v is register v of lane column + 16 G
  const int rows = min(16, M - m0);
  if (tid < rows * 16) {
    const int row = tid >> 4, cc = tid & 15;
    const int v = row & 3, pl = cc + 16 * (row >> 2);
    float sum[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      float acc = s_red[0][m][v][pl];
#pragma unroll
      for (int w = 1; w < NW; ++w) acc += s_red[w][m][v][pl];
      sum[m] = acc;
    }
    uint16_t r;
    if constexpr (DUAL)
      r = A::from_f32(silu_act<DT>(round_act<DT>(sum[0])) * round_act<DT>(sum[NM - 1]));
    else
      r = A::from_f32(sum[0]);
    a.out[(int64_t)(m0 + row) * a.out_ld + r0 + cc] = r;
  }
}

template <int DT, bool DUAL, int NW, int RING>
hipError_t launch_n(const GroupedArgs &a, hipStream_t st) {
  const dim3 grid((unsigned)(a.R / 16), (unsigned)((a.act_rows + 15) / 16));
  if (a.gs == 128)
    hipLaunchKernelGGL((gemv_dense_kernel<DT, DUAL, NW, RING, true>), grid, dim3(64 * NW), 0, st,
                       a);
  else
    hipLaunchKernelGGL((gemv_dense_kernel<DT, DUAL, NW, RING, false>), grid, dim3(64 * NW), 0, st,
                       a);
  return hipGetLastError();
}

// Reductions that the unit-list GEMV splits into eight slices (K 2048, 4096)
// are split alike, two or four pairs a wavefront, and sum in its order: a
// row's result is the same bit for bit from either kernel, for the row counts
// that either of them takes (the GEMM beyond them rounds the weights to fp16).
// (4096 -> 2048 at 16 rows: 7.2 us; sixteen wavefronts of two pairs took 6.7,
// in another order.)  Longer ones take sixteen wavefronts, the gate/up pair
// eight (its partial sums fill twice the LDS).
template <int DT>
hipError_t launch_t(bool dual, const GroupedArgs &a, hipStream_t st) {
  if (dual)
    return a.K <= 2048 ? launch_n<DT, true, 8, 2>(a, st) : launch_n<DT, true, 8, 4>(a, st);
  if (a.K <= 2048) return launch_n<DT, false, 8, 2>(a, st);
  if (a.K <= 4096) return launch_n<DT, false, 8, 4>(a, st);
  return launch_n<DT, false, 16, 3>(a, st);
}

}  // namespace

// The line is drawn on the number of blocks a CU, each of which reads its
// weights and 16 rows of x anew, against the unit-list GEMV (us a call, that
// GEMV / this kernel, bf16, groups of 64, weights rotated past the last-level
// cache; fp16 and groups of 128 alike).  That GEMV runs 1, 2, 4 or 8 chunks
// of 16 rows well and other counts unevenly.
//  * K below 2048, 2.5 blocks: 1536 -> 10240, 1 row 8.0 / 7.4; 1024 -> 5120,
//    17 rows 7.6 / 5.7.
//  * K 2048, two blocks: 2048 -> 8192, 1 row 7.1 / 7.1, 16 rows 7.9 / 7.4; 2048
//    -> 4096, 32 rows 7.3 / 6.7; beyond it 2048 -> 10240, 1 row 7.8 / 9.2, and
//    2048 -> 5120, 17 rows 8.7 / 9.0.  2.5 blocks for other chunk counts: 2048
//    -> 3072, 33 rows 9.3 / 8.5; 2048 -> 1024, 145 rows 10.5 / 8.5.
//  * K up to 3072, 1.5 blocks: 2560 -> 6144, 1 row 9.3 / 9.4, 16 rows 11.0 /
//    10.0; 2560 -> 9216 11.2 / 13.1.
//  * K up to 4096, one block (the longer ring leaves registers for one): 4096
//    -> 4096, 1 row 8.8 / 7.8, 4096 -> 2048, 32 rows 10.2 / 7.4; beyond it 4096
//    -> 5120, 1 row 11.1 / 13.3, 3072 -> 6144 8.5 / 10.8.  1.5 blocks for other
//    chunk counts: 4096 -> 2048, 33 rows 15.3 / 12.5; 3072 -> 1024, 81 rows
//    11.8 / 9.9.
// The gate/up pair has the same lines: 2048 -> 6144, 1 row 9.6 / 10.1, 16 rows
// 10.6 / 10.3, 17 rows (3 blocks) 12.1 / 13.4; 2048 -> 10240 12.0 / 13.5; 4096
// -> 4096 16.3 / 11.3, 4096 -> 6144 19.5 / 20.6.
// Where that GEMV does not hold the reduction (K 5120, 6144, 8192) the
// alternative is the GEMM, whose few blocks run every k-step in sequence
// (gemm_mid.hip): 6144 -> 2048, 128 rows 46.6 / 31.1, 160 rows 46.5 / 38.1, 200
// rows 47 / 51.5; 5120 -> 20480, 16 rows 46.1 / 42.0: five blocks there, four
// for the pair (5120 -> 2048, 128 rows 42.6 / 44.3, fp16 41.1 / 37.0).
bool gemv_dense_supports(bool dual, int64_t M, int K, int R) {
  if (M < 1 || M > 4096 || K % 128 || K > 8192 || R % 16) return false;
  const int64_t chunks = (M + 15) / 16, blocks = chunks * (R / 16), cu = cu_count();
  if (!gemv_supports(K)) return blocks <= (dual ? 4 : 5) * cu;
  const bool pow2 = (chunks & (chunks - 1)) == 0;
  if (K <= 2048) return 2 * blocks <= (K == 2048 && pow2 ? 4 : 5) * cu;
  return 2 * blocks <= (K >= 3072 && pow2 ? 2 : 3) * cu;
}

hipError_t launch_gemv_dense(int dtype, bool dual, const GroupedArgs &a, hipStream_t st) {
  return dtype == DT_BF16 ? launch_t<DT_BF16>(dual, a, st) : launch_t<DT_F16>(dual, a, st);
}

}  // namespace nvm
