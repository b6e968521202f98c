// dK/dV pass at head dims of 128 and 256, bf16/f16 MFMA, gfx950: every 32 keys are held by two waves.
//
// The pass keeps K, V, dK and dV of a wave's 32 keys in registers. From D = 128 on that leaves one wave
// per SIMD (395 VGPRs at D = 128) and at D = 256 not even that (384 of 512 VGPRs in operands and
// accumulators alone, 400 spilled), so the score, exponential and gradient products of a chunk ran
// one after another on each SIMD. Here an 8-wave workgroup owns 128 keys of one stream: waves 0-3
// (the score side) hold K and dV of 32 keys each, waves 4-7 (the gradient side) V and dK of the same
// keys, so two waves share a SIMD and one's products run under the other's exponentials:
//   score side, chunk i:         S = Q K^T, P = exp2(S*scale2 - LSE), dV^T += dO^T P, P -> LDS (fp32)
//   gradient side, chunk i - 1:  dP = dO V^T - Delta, dS = P dP (P <- LDS), dK^T += Q^T dS
// The gradient side works one 32-query chunk behind, so one barrier per chunk orders everything: the
// P tile (two buffers) and the Q / dO chunks (three: one per side, one being loaded by direct
// global -> LDS loads). P crosses in fp32 in the accumulator's own lane layout, so results are
// those of a wave that keeps P in registers.
//
// Bound by the LDS and the matrix cores together: at D = 256 a chunk reads 256 KiB of fragments per
// CU (~1000-2000 cycles) beside 2048 MFMA cycles per SIMD. Measured against the one-wave form
// (kernel time, MI355X): D = 256, B2 H8 N2048, packed documents, 400-495 -> 109 us; D = 128, B2 H16
// N4096, 158 -> 138 us; D = 128 f16, B3 H10 N3062, 87 -> 77 us. At D = 64 the one-wave form holds two
// waves per SIMD by itself and is faster (88 against 96 us at B4 H16 N4096), so it keeps that.
#include "attn_tiles.hpp"

namespace sps {

constexpr int kSplitThreads = 512;
constexpr int kStages = 3;

template <int D, class E>
__global__ __launch_bounds__(kSplitThreads) void attn_bwd_dkdv_split_kernel(const AttnArgs a) {
  // The conflict-free swizzle at D = 128; at D = 256 its second address per fragment would spill.
  using DT = DmaTile<D, D == 128, kSplitThreads>;
  constexpr int TE = DT::ELEMS;
  constexpr int DC = D / 32;
  // At D = 256 the last three stationary fragments are read from LDS: with all 16 in registers the
  // compiler spilled two, and a spill reload waits (vmcnt counts in order) for the chunk loads issued
  // before it, which made every chunk's loads synchronous (137 against 109 us).
  constexpr int kLdsFrags = D == 256 ? 3 : 0, kRegFrags = D / 16 - kLdsFrags;
  // One array per stage, named by compile-time indices, so a stage's reads do not wait for the
  // direct loads filling another.
  __shared__ __attribute__((aligned(16))) uint16_t sQ0[TE], sQ1[TE], sQ2[TE];
  __shared__ __attribute__((aligned(16))) uint16_t sO0[TE], sO1[TE], sO2[TE];
  // -LSE of the chunk's query rows in [0, kBlock), their -Delta in [kBlock, 2 kBlock).
  __shared__ __attribute__((aligned(16))) float sS0[2 * kBlock], sS1[2 * kBlock], sS2[2 * kBlock];
  __shared__ __attribute__((aligned(16))) float sP[2][kWaves][kBlock * kBlock];
  __shared__ __attribute__((aligned(16))) uint16_t sF[kSplitThreads / 64][kLdsFrags ? kLdsFrags : 1][64 * 8];
  __shared__ int s_span[2 * kWaves];
  auto tQ = [&](int s) -> uint16_t* { return s == 0 ? sQ0 : s == 1 ? sQ1 : sQ2; };
  auto tO = [&](int s) -> uint16_t* { return s == 0 ? sO0 : s == 1 ? sO1 : sO2; };
  auto tS = [&](int s) -> float* { return s == 0 ? sS0 : s == 1 ? sS1 : sS2; };

  const MaskSpec m = a.m;
  const int tid = threadIdx.x, lane = tid & 63, wave8 = wave_uniform(tid >> 6);
  const int wave = wave8 & (kWaves - 1);   // which 32 keys of the tile
  const bool score_side = wave8 < kWaves;  // S, P, dV (else dP, dS, dK)
  const int g = lane >> 5, c32 = lane & 31;
  int b, h;
  TilePlan tp;
  k_workgroup(a, b, h, tp);
  const RowView row = row_view(a, b, tp.mono);
  KState st;
  int run_end;
  const bool planned = k_begin(a, tp, row, s_span, st, run_end, wave);
  const int kp = st.kp;
  const bool kvalid = st.kvalid;
  const int nc = st.nc;
  const bool exact = row.mono;
  const int64_t dk_doc = (!exact && kvalid) ? load_doc(a, b, kp) : 0;

  const BufRsrc q_src = head_rsrc<D>(a.q + b * a.sq.b + h * a.sq.h, a.sq.n, m.N);
  const BufRsrc o_src = head_rsrc<D>(a.dO + b * a.sdo.b + h * a.sdo.h, a.sdo.n, m.N);
  const BufRsrc seed_src = make_rsrc(a.seeds + ((int64_t)b * a.H + h) * 2 * m.N, (uint32_t)(2 * m.N * 4));

  // The wave's stationary fragments: K (score side) or V, lane: key c32, d = 16c + 8g ...
  // Lanes without a key read row 0: their scores are all masked and their columns never stored.
  u32x4_t kv[kRegFrags];
  {
    const uint16_t* krow = score_side ? a.k + b * a.sk.b + h * a.sk.h + (int64_t)kp * a.sk.n
                                      : a.v + b * a.sv.b + h * a.sv.h + (int64_t)kp * a.sv.n;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      const u32x4_t x = *reinterpret_cast<const u32x4_t*>(krow + 16 * c + 8 * g);
      if (c < kRegFrags)
        kv[c] = x;
      else
        lds_write_b128(&sF[wave8][c - kRegFrags][lane * 8], x);
    }
  }

  const uint32_t q_blk = (uint32_t)(kBlock * a.sq.n * 2), o_blk = (uint32_t)(kBlock * a.sdo.n * 2);
  const uint32_t q_c0 = (uint32_t)((int64_t)st.c0 * kBlock * a.sq.n * 2);
  const uint32_t o_c0 = (uint32_t)((int64_t)st.c0 * kBlock * a.sdo.n * 2);
  // Each pass of the workgroup's loads covers 512 / CPR rows, a multiple of the swizzle's period, so
  // a thread's pieces differ by a wave-uniform offset and one VGPR per tensor holds them all.
  constexpr int kRowsPerPass = kSplitThreads / DT::CPR;
  static_assert(kRowsPerPass % 16 == 0, "the swizzle repeats every 16 rows (8 for the register-lean one)");
  const uint32_t q_off = DT::sources(tid, (uint32_t)(a.sq.n * 2)).o[0];
  const uint32_t o_off = DT::sources(tid, (uint32_t)(a.sdo.n * 2)).o[0];
  auto issue = [&](int i, int s) {
#pragma unroll
    for (int p = 0; p < DT::PASSES; ++p) {
      const int at = (p * kSplitThreads + wave8 * 64) * 8;
      const uint32_t row = (uint32_t)(p * kRowsPerPass);
      lds_dma_b128(q_src, tQ(s) + at, (q_c0 + (uint32_t)i * q_blk + row * (uint32_t)(a.sq.n * 2)) + q_off);
      lds_dma_b128(o_src, tO(s) + at, (o_c0 + (uint32_t)i * o_blk + row * (uint32_t)(a.sdo.n * 2)) + o_off);
    }
    if (wave8 == 0)
      lds_dma_b32(seed_src, tS(s), (uint32_t)(((lane >> 5) * m.N + imin((st.c0 + i) * kBlock + c32, m.N - 1)) * 4));
  };

  auto kv_frag = [&](int c) {
    return c < kRegFrags ? kv[c] : lds_read_b128(&sF[wave8][c - kRegFrags][lane * 8]);
  };
  f32x16_t acc[DC];
#pragma unroll
  for (int dc = 0; dc < DC; ++dc) acc[dc] = f32x16_t{};

  auto run = [&](auto exact_tag) {
    constexpr bool EXACT = decltype(exact_tag)::value;
    if (nc > 0) issue(0, 0);
    if (planned) k_lanes(m, run_end, st);
    const float scale2 = a.scale2;
    const BlockMask bm = k_block_mask(st, EXACT);
    auto cls_of = [&](int i) { return classify_block(st.w, (st.c0 + i) * kBlock, EXACT); };
    // Products of a 32 x 32 weight tile (packed pairs w) with the rows of `tile`: acc += tile^T w.
    auto accumulate = [&](const uint16_t* tile, const uint32_t* w) {
#pragma unroll
      for (int dc = 0; dc < DC; ++dc) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
          const u32x4_t f = {w[4 * kh], w[4 * kh + 1], w[4 * kh + 2], w[4 * kh + 3]};
          acc[dc] = E::mfma(DT::frag_tr(tile, 16 * kh, dc, lane), f, acc[dc]);
        }
      }
    };
    auto score_block = [&](int i, int s, bool full) {
      const uint16_t* q = tQ(s);
      f32x16_t sc = f32x16_t{};
#pragma unroll
      for (int c = 0; c < D / 16; ++c) sc = E::mfma(lds_read_b128(q + DT::frag(c32, g, c)), kv_frag(c), sc);
      const float* seed = tS(s);
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4_t l4 = *reinterpret_cast<const SPS_LDS f32x4_t*>((const SPS_LDS float*)(seed + 8 * i4 + 4 * g));
#pragma unroll
        for (int t = 0; t < 4; ++t) sc[4 * i4 + t] = __builtin_fmaf(sc[4 * i4 + t], scale2, l4[t]);
      }
      const int qc = (st.c0 + i) * kBlock;
      if (!full)
        mask_partial<EXACT>(sc, st.r, st.w, qc, g,
                            [&] { return ks_exact_bits<D == 256 ? 2 : 16>(a, b, kp, st.r.hi, qc, g, dk_doc); });
      float* p_out = sP[i & 1][wave];
      uint32_t pk[8];
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        f32x4_t p;
#pragma unroll
        for (int t = 0; t < 4; ++t) p[t] = fast_exp2(sc[4 * i4 + t]);
        *reinterpret_cast<SPS_LDS f32x4_t*>((SPS_LDS float*)(p_out + (i4 * 64 + lane) * 4)) = p;
        pk[2 * i4] = E::pack2(p[0], p[1]);
        pk[2 * i4 + 1] = E::pack2(p[2], p[3]);
      }
      accumulate(tO(s), pk);
    };
    auto grad_block = [&](int i, int s) {
      const uint16_t* o = tO(s);
      const float* seed = tS(s);
      f32x16_t dp;
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4_t d4 =
            *reinterpret_cast<const SPS_LDS f32x4_t*>((const SPS_LDS float*)(seed + kBlock + 8 * i4 + 4 * g));
#pragma unroll
        for (int t = 0; t < 4; ++t) dp[4 * i4 + t] = d4[t];
      }
#pragma unroll
      for (int c = 0; c < D / 16; ++c) dp = E::mfma(lds_read_b128(o + DT::frag(c32, g, c)), kv_frag(c), dp);
      const float* p_in = sP[i & 1][wave];
      uint32_t ds[8];
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4_t p = *reinterpret_cast<const SPS_LDS f32x4_t*>((const SPS_LDS float*)(p_in + (i4 * 64 + lane) * 4));
        ds[2 * i4] = E::pack2(p[0] * dp[4 * i4], p[1] * dp[4 * i4 + 1]);
        ds[2 * i4 + 1] = E::pack2(p[2] * dp[4 * i4 + 2], p[3] * dp[4 * i4 + 3]);
      }
      accumulate(tQ(s), ds);
    };
    vmem_wait_all();
    __syncthreads();
    // The two sides run separate loops with the same barriers.
    auto loop = [&](auto side_tag) {
      constexpr bool SCORE = decltype(side_tag)::value;
      for (int i0 = 0; i0 <= nc; i0 += kStages) {
#pragma unroll
        for (int u = 0; u < kStages; ++u) {
          const int i = i0 + u;  // chunk of the score side; the gradient side is one behind
          if (i <= nc) {
            if (i + 1 < nc) issue(i + 1, (u + 1) % kStages);  // the stage chunk i - 2 has left
            const int j = SCORE ? i : i - 1;
            if (j >= 0 && j < nc) {
              const int cls = j < 128 ? mask_class(bm, j) : cls_of(j);
              if (cls != TILE_SKIP) {
                if constexpr (SCORE)
                  score_block(j, u, cls == TILE_FULL);
                else
                  grad_block(j, (u + kStages - 1) % kStages);
              }
            }
            vmem_wait_all();
            lds_only_barrier();
          }
        }
      }
    };
    if (score_side)
      loop(std::true_type{});
    else
      loop(std::false_type{});
  };
  if (exact)
    run(std::true_type{});
  else
    run(std::false_type{});

  // Outputs: dV from the score side, dK (times sm_scale) from the gradient side.
  const float sc = score_side ? 1.f : a.sm_scale;
  auto piece = [&](int dc, int ii) {
    return u32x2_t{E::pack2(acc[dc][4 * ii] * sc, acc[dc][4 * ii + 1] * sc),
                   E::pack2(acc[dc][4 * ii + 2] * sc, acc[dc][4 * ii + 3] * sc)};
  };
  uint16_t* out = score_side ? a.dv : a.dk;
  const Strides3 so = score_side ? a.sdv : a.sdk;
  if (rows16_ok(a.dk, a.sdk) && rows16_ok(a.dv, a.sdv)) {
    const int t0 = st.first + wave * kBlock;
    const int p0 = stream_pos(m, st.stream, t0);
    const int nrows = imin(kBlock, stream_len(m.family, m.N, st.stream, m.P) - t0);
    const int kstep = m.family == FAMILY_FULL ? 1 : 2;
    // 32 rows of 128 columns at a time (8 KiB) through an idle tile (waves 6 and 7 at D = 128: the P buffers).
    constexpr int kCols = 128, kPart = kBlock * kCols;
    uint16_t* tile;
    if constexpr (D == 256)
      tile = (wave8 >> 1) == 0 ? sQ0 : (wave8 >> 1) == 1 ? sQ1 : (wave8 >> 1) == 2 ? sQ2 : sO0;
    else
      tile = wave8 == 0 ? sQ0 : wave8 == 1 ? sQ1 : wave8 == 2 ? sQ2 : wave8 == 3 ? sO0 : wave8 == 4 ? sO1
           : wave8 == 5 ? sO2 : wave8 == 6 ? reinterpret_cast<uint16_t*>(sP[0]) : reinterpret_cast<uint16_t*>(sP[1]);
    if constexpr (D == 256) tile += (wave8 & 1) * kPart;
#pragma unroll
    for (int part = 0; part < D / kCols; ++part)
      store_rows_via_lds<kCols>(tile, lane, out + b * so.b + h * so.h + (int64_t)p0 * so.n + part * kCols, kstep * so.n,
                                nrows, [&](int dc, int ii) { return piece(part * (kCols / 32) + dc, ii); });
  } else if (kvalid) {
    uint16_t* orow = out + b * so.b + h * so.h + (int64_t)kp * so.n;
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) *reinterpret_cast<u32x2_t*>(orow + 32 * dc + 8 * ii + 4 * g) = piece(dc, ii);
    }
  }
}

hipError_t launch_attn_bwd_dkdv_split(const AttnArgs& a, int D, int is_f16, int64_t nblocks, hipStream_t stream) {
  const dim3 grid((unsigned)nblocks), block(kSplitThreads);
  if (D == 128) {
    if (is_f16)
      hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<128, ElemF16>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<128, ElemBF16>), grid, block, 0, stream, a);
  } else {
    if (is_f16)
      hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<256, ElemF16>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((attn_bwd_dkdv_split_kernel<256, ElemBF16>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace sps
