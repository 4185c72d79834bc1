// Grouped W4A16 expert products of mid-sized batches (up to some 48 routed
// rows per expert, and dense products whose 128-row grid would not fill the
// chip): the operands and arithmetic of gemm.hip's kernels, bit for bit, on
// m-tiles of 32 or 64 routed rows.
//
// Bound: the weight stream and each block's fixed latencies.  At 10 rows per
// expert the 128-row kernels read every expert's weights for a tile that is
// mostly padding: accumulators for 128 rows leave registers for two blocks a
// CU and a k-step pair of weights in flight, the grid ran in two rounds, and
// the epilogue evaluated SwiGLU for 128 rows.  With one 32-row block the
// kernel takes 156 registers, three blocks a CU (a whole gate/up grid of the
// 30B-A3B shape at once); with two, 220.  The freed registers hold four
// k-steps of the wavefront's own packed weights and four of the block's
// activations, all requested three to four k-steps ahead, the activations
// staged through two LDS buffers.  (Eight k-steps of weights spilled and
// measured slower: loads return in order, so the weights in flight are those
// issued since the next k-step's activations.)  Gate/up and down of 150
// tokens at the 30B-A3B shape together: 131 us on the 128-row kernels, 98
// here.
#include <stdlib.h>

#include <type_traits>

#include "common.h"
#include "gemm_common.h"
#include "internal.h"

namespace nvm {

namespace {

constexpr int MWROWS = 256;       // weight rows per tile (gate/up: 128 of each matrix)
constexpr int MA_PITCH = 144;     // bytes per staged activation row (128 + 16)
constexpr int MW_PITCH = 72;      // scale/bias window rows, as gemm.hip
constexpr int MW_WAVE = 32 * MW_PITCH;
constexpr int kARing = 4;         // k-steps of activations in registers
constexpr int kWRing = 4;         // k-steps of weights

// KB: k-steps between two barriers (2 KB activation stages)
constexpr int stage_lds(int NI, int KB) { return 2 * KB * 32 * NI * MA_PITCH + 4 * MW_WAVE; }
template <bool DUAL>
constexpr int mid_lds(int NI, int KB) {
  const int out = 32 * NI * (2 * (DUAL ? MWROWS / 2 : MWROWS) + 16);
  return out > stage_lds(NI, KB) ? out : stage_lds(NI, KB);
}

// (nothing moves across: the rings' loads stay in the k-step that issues them)
__device__ __forceinline__ void step_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// NI: 32-row blocks of routed rows per tile.
template <int DT, bool DUAL, bool AH, bool G128, int NI, int KB>
__global__ __launch_bounds__(256, NI == 1 ? 3 : 2) void gemm_mid_kernel(const GroupedArgs a,
                                                                       int n_tiles) {
  using A = Act<DT>;
  constexpr int MBM = 32 * NI;  // routed rows per tile
  constexpr int MA_STAGE = MBM * MA_PITCH;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int s_arow[MBM];
  __shared__ int s_orow[MBM];
  // the m-tile prefix and the expert offsets, in the staging LDS until the
  // tile's rows are known
  int *const s_tiles = (int *)smem;
  int *const s_offs = s_tiles + kMaxExperts + 1;
  static_assert(2 * (kMaxExperts + 1) * 4 <= stage_lds(NI, KB), "m-tile list exceeds the staging LDS");

  hoist_args(a.act, a.act_ld, a.act_rows, a.a_map, a.a_div, a.offsets, a.w0, a.s0, a.b0, a.w1,
             a.s1, a.b1, a.R, a.K, a.E, a.out, a.o_map, a.out_ld, n_tiles);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;

  auto offs = [&](int i) { return a.offsets ? a.offsets[i] : (i == 0 ? 0 : (int)a.act_rows); };
  if (wv == 0) {
    int carry = 0;
    for (int c0 = 0; c0 < a.E; c0 += 64) {
      const int e = c0 + lane;
      const int o0 = e < a.E ? offs(e) : 0, o1 = e < a.E ? offs(e + 1) : 0;
      const int tv = e < a.E ? (o1 - o0 + MBM - 1) / MBM : 0;
      int inc = tv;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
      }
      if (e < a.E) {
        s_tiles[e] = carry + inc - tv;
        s_offs[e + 1] = o1;
        if (e == 0) s_offs[0] = o0;
      }
      carry += __shfl(inc, 63);
    }
    if (lane == 0) s_tiles[a.E] = carry;
  }
  __syncthreads();
  // XCD-aware tile order (as gemm.hip)
  const int total = s_tiles[a.E] * n_tiles;
  const int per_xcd = (total + 7) >> 3;
  const int local = blockIdx.x >> 3;
  if (local >= per_xcd) return;
  const int t = (blockIdx.x & 7) * per_xcd + local;
  if (t >= total) return;
  const int mt = t / n_tiles, nt = t - mt * n_tiles;
  int lo = 0, hi = a.E - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_tiles[mid] <= mt)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int e = lo;
  const int m0 = s_offs[e] + (mt - s_tiles[e]) * MBM;
  const int mcnt = min(MBM, s_offs[e + 1] - m0);
  const int R = a.R, KW = a.K >> 3, GPR = a.K / (G128 ? 128 : 64);
  const int n0 = nt * (DUAL ? MWROWS / 2 : MWROWS);
  if (tid < MBM) {
    const int slot = m0 + tid;
    s_arow[tid] = tid < mcnt ? (a.a_map ? a.a_map[slot] / a.a_div : slot) : -1;
    s_orow[tid] = tid < mcnt ? (a.o_map ? a.o_map[slot] : slot) : -1;
  }
  __syncthreads();

  const int KSG = a.K >> 6;
  const rsrc_t ra = make_rsrc(a.act, (uint32_t)(a.act_rows * a.act_ld * 2));
  const int64_t eoff = (int64_t)e * R;
  const rsrc_t rw0 = make_rsrc(a.w0 + eoff * KW, (uint32_t)R * KW * 4);
  const rsrc_t rw1 = make_rsrc((DUAL ? a.w1 : a.w0) + eoff * KW, (uint32_t)R * KW * 4);
  const rsrc_t rs0 = make_rsrc(a.s0 + eoff * GPR, (uint32_t)R * GPR * 2);
  const rsrc_t rb0 = make_rsrc(a.b0 + eoff * GPR, (uint32_t)R * GPR * 2);
  const rsrc_t rs1 = make_rsrc((DUAL ? a.s1 : a.s0) + eoff * GPR, (uint32_t)R * GPR * 2);
  const rsrc_t rb1 = make_rsrc((DUAL ? a.b1 : a.b0) + eoff * GPR, (uint32_t)R * GPR * 2);

  // activations: thread loads rows (tid >> 3) + 32c, 16-byte chunk tid & 7
  int a_voff[NI];
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int ar = s_arow[(tid >> 3) + 32 * c];
    a_voff[c] = ar >= 0 ? (int)(((int64_t)ar * a.act_ld) * 2) + 16 * (tid & 7) : kMaskedOffset;
  }
  // the lane's two weight rows (sub 0/1)
  int srow[2], b_voff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int grow = DUAL ? n0 + 32 * wv + l32 : n0 + 64 * wv + 32 * s + l32;
    srow[s] = grow < R ? grow * GPR * 2 : kMaskedOffset;
    b_voff[s] = grow < R ? grow * KW * 4 + 16 * h : kMaskedOffset;
  }
  const int nk = a.K / 64;  // a multiple of 4
  u32x4 xa[kARing][NI];     // slot ks % 4: activations of k-step ks
  u32x4 wq[kWRing][2];      // slot ks % kWRing: the lane's packed words of k-step ks
  // (k-steps past the end read zeros through masked offsets: every step makes
  // the same loads, so the wait counts hold on every path)
  auto issue_a = [&](u32x4 (&q)[NI], int ks) {
    const bool ok = ks < nk;
    const int so = ok ? ks * 128 : 0;
#pragma unroll
    for (int c = 0; c < NI; ++c) q[c] = bload16(ra, ok ? a_voff[c] : kMaskedOffset, so);
  };
  // k-steps ks, ks + 1 (ks even): 64 bytes of each row, back to back
  auto issue_b = [&](u32x4 (&q0)[2], u32x4 (&q1)[2], int ks) {
    const bool ok = ks < nk;
    const int so = ok ? ks * 32 : 0;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int vo = ok ? b_voff[s] : kMaskedOffset;
      q0[s] = bload16(s ? rw1 : rw0, vo, so);
      q1[s] = bload16(s ? rw1 : rw0, vo, so + 32);
    }
  };
  // scale/bias windows of eight groups (as gemm.hip: GPR a multiple of 4)
  u32x2 wcur[4];
  auto issue_w = [&](int wi) {
    const int gh = 8 * wi + 4 * h;
    const int so = 16 * wi;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const rsrc_t r = t2 ? (s ? rb1 : rb0) : (s ? rs1 : rs0);
        wcur[2 * s + t2] = bload8(r, gh < GPR ? srow[s] + 8 * h : kMaskedOffset, so);
      }
  };
  uint8_t *const w_lds = smem + 2 * KB * MA_STAGE + wv * MW_WAVE + l32 * MW_PITCH;
  auto new_window = [&](int wi) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      auto val = [&](const u32x2 &w) {
        const uint32_t d = (i & 2) ? w.y : w.x;
        return sb_h<DT>((i & 1) ? d >> 16 : d & 0xFFFFu);
      };
      *(u32x2 *)(w_lds + 8 * (4 * h + i)) =
          u32x2{val(wcur[0]) | (val(wcur[1]) << 16), val(wcur[2]) | (val(wcur[3]) << 16)};
    }
    issue_w(wi + 1);
  };
  uint32_t sc[2], bi[2];
  auto take_sb = [&](int g) {  // group g of the window
    const u32x2 v = *(const u32x2 *)(w_lds + 8 * g);
    sc[0] = perm_b32(v.x, v.x, 0x01000100u);
    bi[0] = perm_b32(v.x, v.x, 0x03020302u);
    sc[1] = perm_b32(v.y, v.y, 0x01000100u);
    bi[1] = perm_b32(v.y, v.y, 0x03020302u);
  };
  auto store = [&](const u32x4 (&q)[NI], int buf) {
    uint8_t *As = smem + buf * MA_STAGE;
#pragma unroll
    for (int c = 0; c < NI; ++c)
      *(u32x4 *)(As + ((tid >> 3) + 32 * c) * MA_PITCH + 16 * (tid & 7)) =
          AH ? q[c] : act_to_h<DT>(q[c]);
  };

  f32x16 acc[2][NI];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[s][i][r] = 0.f;
  const DeqConst dk = deq_const();
  auto compute = [&](int buf, const u32x4 (&bw)[2], auto NA) {
    constexpr int na = decltype(NA)::value;
    const uint8_t *As = smem + buf * MA_STAGE;
    auto load_a = [&](int c, u32x4 (&af)[NI]) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (i < na) af[i] = *(const u32x4 *)(As + (32 * i + l32) * MA_PITCH + 16 * (4 * h + c));
    };
    auto deq = [&](int c, u32x4 (&bf)[2]) {
#pragma unroll
      for (int s = 0; s < 2; ++s) bf[s] = dequant8_h(bw[s][c], sc[s], bi[s], dk);
    };
    u32x4 af[NI], bf[2];
    load_a(0, af);
    deq(0, bf);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      u32x4 afn[NI], bfn[2];
      if (c < 3) {
        load_a(c + 1, afn);
        deq(c + 1, bfn);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < NI; ++i)
          if (i < na) acc[s][i] = mfma32_h(bf[s], af[i], acc[s][i]);
      if (c < 3) {
#pragma unroll
        for (int i = 0; i < NI; ++i) af[i] = afn[i];
        bf[0] = bfn[0];
        bf[1] = bfn[1];
      }
    }
  };

  // k-step ks computes LDS buffer ks % (2 KB); its activations' register slot
  // (stored before the last barrier) takes those of ks + 4, its weights'
  // slot, after the pair's second step, those of kWRing k-steps on
  auto k_loop = [&](auto NA) {
    auto trip = [&](int ks0, auto N) {
#pragma unroll
      for (int j = 0; j < decltype(N)::value; ++j) {
        const int ks = ks0 + j;
        if (j % KB == 0) {
#pragma unroll
          for (int d = 0; d < KB; ++d) issue_a(xa[(j + d) % kARing], ks + d + kARing);
          step_fence();
        }
        if (j == 0 && (!G128 || (ks0 & 8) == 0)) new_window(ks0 >> (G128 ? 4 : 3));
        take_sb(G128 ? ((ks0 & 8) + j) >> 1 : j);
        compute(j % (2 * KB), wq[j % kWRing], NA);
        if (j & 1) issue_b(wq[(j - 1) % kWRing], wq[j % kWRing], ks - 1 + kWRing);
        if (j % KB == KB - 1) {
          step_fence();
#pragma unroll
          for (int d = 1; d <= KB; ++d) store(xa[(j + d) % kARing], (j + d) % (2 * KB));
          __syncthreads();
        }
      }
    };
    int ks0 = 0;
    for (; ks0 + 8 <= nk; ks0 += 8) trip(ks0, std::integral_constant<int, 8>{});
    if (ks0 < nk) trip(ks0, std::integral_constant<int, 4>{});
  };
  // The k-loop of a tile whose fp16 activations carry group shifts (values
  // beyond 2^15: rare), one k-step at a time without the rings: before each
  // k-step a row's sums go from the units of the previous group's shift to
  // those of its own (2^(old - new), exact), at the end back to units of one.
  auto shifted_loop = [&]() {
    int cs[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) cs[i] = 0;
    auto scale_rows = [&](int i, int nsh) {
      const float f = pow2f(cs[i] - nsh);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[s][i][q] *= f;
      cs[i] = nsh;
    };
    for (int ks = 0; ks < nk; ++ks) {
      u32x4 x1[NI], w1[2];
      issue_a(x1, ks);
#pragma unroll
      for (int s = 0; s < 2; ++s) w1[s] = bload16(s ? rw1 : rw0, b_voff[s], ks * 32);
      store(x1, 0);
      const int g = ks >> (G128 ? 1 : 0);
      if ((g & 7) == 0 && (!G128 || !(ks & 1))) new_window(g >> 3);
      take_sb(g & 7);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = s_arow[32 * i + l32];
        scale_rows(i, r >= 0 ? (int)a.act_sh[(int64_t)r * KSG + ks] : cs[i]);
      }
      compute(0, w1, std::integral_constant<int, NI>{});
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) scale_rows(i, 0);
  };
  issue_w(0);
  issue_a(xa[0], 0);
  step_fence();
  issue_b(wq[0], wq[1], 0);
  issue_a(xa[1], 1);
  issue_a(xa[2], 2);
  step_fence();
  issue_b(wq[2], wq[3], 2);
  issue_a(xa[3], 3);
  step_fence();
  // fp16 copies stored with group shifts (as gemm.hip)
  bool shifted = false;
  if constexpr (AH && DT == DT_BF16) {
    uint32_t any = 0;
    if (a.act_sh) {
      const int W = KSG >> 2;  // (KSG a multiple of 4)
      for (int j = tid; j < MBM * W; j += 256) {
        const int r = s_arow[j / W];
        if (r >= 0) any |= *(const uint32_t *)(a.act_sh + (int64_t)r * KSG + 4 * (j % W));
      }
    }
    shifted = __syncthreads_or(any != 0);
  }
  if (shifted) {
    shifted_loop();
  } else {
#pragma unroll
    for (int d = 0; d < KB; ++d) store(xa[d], d);
    __syncthreads();
    if (NI > 1 && mcnt > 32)
      k_loop(std::integral_constant<int, NI>{});
    else
      k_loop(std::integral_constant<int, 1>{});
  }

  // Epilogue through LDS (as gemm.hip); the last step's barrier is past the
  // last use of the stages
  constexpr int OCOLS = DUAL ? MWROWS / 2 : MWROWS;
  constexpr int O_PITCH = 2 * OCOLS + 16;
  uint8_t *Os = smem;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (32 * i >= mcnt) break;  // uniform: no routed row in this block
    uint8_t *orow = Os + (32 * i + l32) * O_PITCH;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (DUAL) {
        uint32_t o[2];
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          float g0 = acc[0][i][4 * q + j], g1 = acc[0][i][4 * q + j + 1];
          float u0 = acc[1][i][4 * q + j], u1 = acc[1][i][4 * q + j + 1];
          round_act2<DT>(g0, g1);
          round_act2<DT>(u0, u1);
          o[j >> 1] = swiglu_act2<DT>(g0, g1, u0, u1);
        }
        *(u32x2 *)(orow + 2 * (32 * wv + 8 * q + 4 * h)) = u32x2{o[0], o[1]};
      } else {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          *(u32x2 *)(orow + 2 * (64 * wv + 32 * s + 8 * q + 4 * h)) =
              u32x2{A::pack2(acc[s][i][4 * q], acc[s][i][4 * q + 1]),
                    A::pack2(acc[s][i][4 * q + 2], acc[s][i][4 * q + 3])};
      }
    }
  }
  __syncthreads();
  constexpr int CPR = OCOLS / 8;
  const int c = tid % CPR, col = n0 + 8 * c;
  const bool vec = (a.out_ld & 7) == 0 && ((uintptr_t)a.out & 15) == 0 && col + 8 <= R;
  for (int r = tid / CPR; r < mcnt; r += 256 / CPR) {
    u32x4 v = *(const u32x4 *)(Os + r * O_PITCH + 16 * c);
    if constexpr (DUAL && DT == DT_BF16) {
      if (a.out_h) {
        const int sh = f16_shift_of(max8_lanes(bf16_absmax_bits(v)));
        v = bf16_to_f16_pairs(v, sh);
        if ((c & 7) == 0 && a.out_sh && col < R)
          a.out_sh[(int64_t)s_orow[r] * (R >> 6) + (col >> 6)] = (uint8_t)sh;
      }
    }
    uint16_t *op = a.out + (int64_t)s_orow[r] * a.out_ld + col;
    if (vec) {
      *(u32x4 *)op = v;
    } else {
#pragma unroll
      for (int e2 = 0; e2 < 8; ++e2)
        if (col + e2 < R) op[e2] = (uint16_t)(v[e2 >> 1] >> (16 * (e2 & 1)));
    }
  }
}

template <int DT, bool DUAL, bool AH, int NI, int KB>
hipError_t launch_n(const GroupedArgs &a, int64_t pairs, hipStream_t st) {
  constexpr int cols = DUAL ? MWROWS / 2 : MWROWS;
  const int n_tiles = (a.R + cols - 1) / cols;
  const int64_t max_m_tiles = pairs / (32 * NI) + a.E;
  const unsigned grid = (unsigned)(8 * ((max_m_tiles * n_tiles + 7) / 8));
  if (a.gs == 128)
    hipLaunchKernelGGL((gemm_mid_kernel<DT, DUAL, AH, true, NI, KB>), dim3(grid), dim3(256),
                       mid_lds<DUAL>(NI, KB), st, a, n_tiles);
  else
    hipLaunchKernelGGL((gemm_mid_kernel<DT, DUAL, AH, false, NI, KB>), dim3(grid), dim3(256),
                       mid_lds<DUAL>(NI, KB), st, a, n_tiles);
  return hipGetLastError();
}

// Two k-steps a barrier where a CU holds one block (dense products: 4096 ->
// 2048 at 1500 rows 42.8 -> 41.4 us) or three (32-row tiles: 0.5 % of a
// layer); with two co-resident blocks, which cover each other's barriers, one
// (700 tokens at hidden 4096: 493 against 500 us).
template <int DT, bool DUAL, bool AH>
hipError_t launch_t(int ni, const GroupedArgs &a, int64_t pairs, hipStream_t st) {
  if (ni == 1) return launch_n<DT, DUAL, AH, 1, 2>(a, pairs, st);
  if constexpr (!AH) {
    if (!a.offsets) return launch_n<DT, DUAL, AH, 2, 2>(a, pairs, st);
  }
  return launch_n<DT, DUAL, AH, 2, 1>(a, pairs, st);
}

}  // namespace

// Expert products: by the routed rows per expert.  Layer at hidden 2048 with
// one / two blocks a tile / the 128-row kernels (bf16, us): 150 tokens (9 rows
// an expert) 126 / 132 / 159, 256 (16) 130 / 135 / 163, 384 (24) 149 / 142 /
// 161, 700 (44) 191 / 172 / 178, 1000 (62) - / 211 / 202; hidden 4096: 700
// tokens 655 / 489 / 523, 1000 - / 617 / 584.  Skewed routing (the first
// experts at 10 to 16 times the mean) leaves the line where it is: the layer
// against the 128-row design, 150 tokens 136 / 184, 512 170 / 218, 767 198 /
// 225; hidden 4096, 700 tokens 560 / 610.
// Dense products: by the grid.  A block runs the whole reduction, so the time
// goes in rounds of one block a CU (fp16, groups of 128, weights rotated past
// the caches, one / two blocks a tile / 128-row kernels, in brackets the
// blocks): 4096 -> 2048 at 600 rows 32 / 39 / 67, 1000 rows (256, 128, 64) 36 /
// 40 / 67, 1500 rows (376, 192, 96) 50 / 41 / 68, 2500 rows (632, 320, 160) 74 /
// 66 / 68; 2048 -> 5120 at 1500 rows (940, 480, 240) 58 / 47 / 44.  A second
// round of up to a quarter of the CUs pays with groups of 128, with groups of
// 64 up to a reduction of 4096: two blocks / 128-row kernels, groups of 128,
// 6144 -> 2048 at 2100 rows (bf16) 93.6 / 97.3, 8192 -> 4096 at 1250 (fp16)
// 129 / 133; groups of 64 (bf16), 4096 -> 2048 at 2500 69.3 / 69.7, 5120 ->
// 5120 at 800 88.3 / 85.5, 8192 -> 4096 at 1250 136 / 130.
// NVM_GEMM_NODMA=1 takes the register-staged 128-row kernel instead.
int gemm_mid_blocks(bool dual, const GroupedArgs &a, int64_t pairs) {
  const char *v = getenv("NVM_GEMM_NODMA");
  if ((v && v[0] == '1') || a.K % 256 || a.K % (4 * a.gs)) return 0;
  if (a.offsets) return pairs <= 20 * a.E ? 1 : pairs <= 48 * a.E ? 2 : 0;
  const int cols = dual ? MWROWS / 2 : MWROWS;
  const int64_t nt = (a.R + cols - 1) / cols, cu = cu_count();
  if ((pairs + 31) / 32 * nt <= cu) return 1;
  const int quarters = a.gs == 64 && a.K > 4096 ? 4 : 5;
  return 4 * ((pairs + 63) / 64 * nt) <= quarters * cu ? 2 : 0;
}

hipError_t launch_gemm_mid(int dtype, bool dual, int blocks, const GroupedArgs &a, int64_t pairs,
                           hipStream_t st) {
  if (dtype != DT_BF16)
    return dual ? launch_t<DT_F16, true, false>(blocks, a, pairs, st)
                : launch_t<DT_F16, false, false>(blocks, a, pairs, st);
  if (a.act_h)
    return dual ? launch_t<DT_BF16, true, true>(blocks, a, pairs, st)
                : launch_t<DT_BF16, false, true>(blocks, a, pairs, st);
  return dual ? launch_t<DT_BF16, true, false>(blocks, a, pairs, st)
              : launch_t<DT_BF16, false, false>(blocks, a, pairs, st);
}

}  // namespace nvm
