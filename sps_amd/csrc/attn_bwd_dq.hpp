// The dQ pass of the backward attention (see attn_bwd.hip for the two passes).
#pragma once
#include "attn_tiles.hpp"

namespace sps {

// Groups of blocks whose loads are in flight while a group is computed (run_groups).
constexpr int kLook = 1;

// Blocks per barrier (LDS budget: up to D = 128 both passes run 2 workgroups per CU, so four 32-row
// blocks of two tensors, double-buffered, fit; fewer barriers per block than pairs). At D = 256 a
// block is 16 KiB, so groups of two (128 KiB of tiles, one workgroup per CU).
template <int D>
constexpr int bwd_group() { return D >= 256 ? 2 : 4; }

// One waves-per-SIMD floor per head dim: 2 at D <= 64; above, the MFMA accumulators of D-wide rows
// need the registers of one wave per SIMD.
template <int D>
constexpr int bwd_waves() { return D <= 64 ? 2 : 1; }

// The dQ pass in groups of two blocks (32 KiB of tiles at D = 64, 64 KiB at D = 128), so the LDS holds
// as many workgroups as the registers: three waves per SIMD at D = 64 (168 VGPRs; dQ -4 % at C3, -6 %
// at C2 against four-block groups at 2 waves per SIMD). D = 128 has two forms, picked by dq_two_waves():
// four-block groups at one wave per SIMD (345 VGPRs), and two-block groups at two (256 VGPRs, 28 spilled). Both
// need the iterative ILP schedule of attn_bwd.hip, spills and all: under the default scheduler the two-wave form
// spills none, but a workgroup that ends up alone on its CU then takes ~30 % longer than the one-wave form, which
// small grids and layouts with one long document are made of (MI355X, dQ, one wave / two waves with ILP
// / two without: C4 118.5 / 107.2 / 120.3 us, B2 H16 N2048 dense causal 72.7 / 69.9 / 78.0, B4 H16 N4096
// 227 / 190 / 191).
template <int D>
constexpr int dq_waves() { return D == 64 ? 3 : bwd_waves<D>(); }
template <int D, int WAVES>
constexpr int dq_group() { return D == 64 || (D == 128 && WAVES == 2) ? 2 : bwd_group<D>(); }

// The wave index, wave-uniform at D = 64 (so every LDS address derived from it, the direct-to-LDS
// loads' M0 values among them, is computed in scalar registers instead of VGPRs that the 3-wave dQ
// pass would have to spill).
template <int D>
__device__ __forceinline__ int wave_index() {
  return D == 64 ? wave_uniform((int)threadIdx.x >> 6) : (int)threadIdx.x >> 6;
}

// The wave's own 32-row tile of a [2][NG][32 * D] staging array (an idle buffer at the end of the
// kernel): every layout holds at least kWaves of them.
template <int NG, int TE>
__device__ __forceinline__ uint16_t* wave_tile(uint16_t (&arr)[2][NG][TE], int wave) {
  static_assert(2 * NG >= kWaves, "one tile per wave");
  return &arr[0][0][0] + wave * TE;
}

template <int D, class E, int WAVES = dq_waves<D>()>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES, 8))) void attn_bwd_dq_kernel(const AttnArgs a) {
  using G = TileGeom<D>;
  constexpr int NG = dq_group<D, WAVES>();
  // Head dims of 64 and more stage K / V blocks by direct global -> LDS loads into dense swizzled
  // tiles (frees the staging VGPRs: -7 % at D = 128, -2 % of the C3 step at D = 64 under the
  // iterative ILP schedule); smaller ones through registers into padded tiles.
  constexpr bool kDma = D >= 64;
  // The conflict-free swizzle costs a few address VGPRs: at D = 64 (3 waves per SIMD) and D = 256
  // they would spill, so those keep the register-lean one.
  using DT = DmaTile<kDma ? D : 64, D == 128>;
  constexpr int TE = kDma ? DT::ELEMS : G::ELEMS;
  __shared__ __attribute__((aligned(16))) uint16_t sK[2][NG][TE];  // [buffer][block of the group]
  __shared__ __attribute__((aligned(16))) uint16_t sV[2][NG][TE];
  __shared__ int s_span[4 * kWaves];

  const MaskSpec m = a.m;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index<D>();
  const int g = lane >> 5, c32 = lane & 31;
  int b, h;
  TilePlan tp;
  q_workgroup(a, b, h, tp);
  const RowView row = row_view(a, b, tp.mono);
  const int qp = tp.tile * kTile + wave * kBlock + c32;
  const bool qvalid = qp < m.N;
  const int qsafe = qvalid ? qp : 0;
  QState st;
  int run_start;
  const bool planned = q_begin(a, tp, row, qp, s_span, st, run_start);
  const QPlan& plan = st.plan;
  const int nb = plan.count();
  const bool exact = row.mono;
  const int64_t dq_doc = (!exact && qvalid) ? load_doc(a, b, qp) : 0;

  const BufRsrc k_src = head_rsrc<D>(a.k + b * a.sk.b + h * a.sk.h, a.sk.n, m.N);
  const BufRsrc v_src = head_rsrc<D>(a.v + b * a.sv.b + h * a.sv.h, a.sv.n, m.N);
  const int step = m.family == FAMILY_FULL ? 1 : 2;  // positions between consecutive stream rows
  const auto k_off = TileRegs<D>::offsets(tid, (uint32_t)(step * a.sk.n * 2));
  const auto v_off = TileRegs<D>::offsets(tid, (uint32_t)(step * a.sv.n * 2));

  // Q, dO and O fragments (B operands; lane: query c32, d = 16c + 8g .. +7) and the LSE, loaded
  // raw here; everything computed from them waits until the first group's loads are issued too.
  u32x4_t qf[D / 16], dof[D / 16], of[D / 16];
  const int64_t rowid = ((int64_t)b * a.H + h) * m.N + qsafe;
  {
    const uint16_t* qrow = a.q + b * a.sq.b + h * a.sq.h + (int64_t)qsafe * a.sq.n;
    const uint16_t* dorow = a.dO + b * a.sdo.b + h * a.sdo.h + (int64_t)qsafe * a.sdo.n;
    const uint16_t* orow = a.o + b * a.so.b + h * a.so.h + (int64_t)qsafe * a.so.n;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      u32x4_t z = {0u, 0u, 0u, 0u};
      qf[c] = qvalid ? *reinterpret_cast<const u32x4_t*>(qrow + 16 * c + 8 * g) : z;
      dof[c] = qvalid ? *reinterpret_cast<const u32x4_t*>(dorow + 16 * c + 8 * g) : z;
      of[c] = qvalid ? *reinterpret_cast<const u32x4_t*>(orow + 16 * c + 8 * g) : z;
    }
  }
  const float lse_raw = qvalid ? a.lse[rowid] : 0.f;

  if constexpr (!kDma) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
#pragma unroll
      for (int y = 0; y < NG; ++y) {
        zero_pad_cols<D>(sK[x][y], tid);
        zero_pad_cols<D>(sV[x][y], tid);
      }
    }
  }

  // Byte offset of block i's first row: i * (bytes per block) + a per-stream constant (modulo 2^32).
  const uint32_t k_blk = (uint32_t)(kBlock * step * a.sk.n * 2), v_blk = (uint32_t)(kBlock * step * a.sv.n * 2);
  const int c0 = stream_pos(m, plan.stream0, kBlock * plan.b0);
  const int c1 = m.family == FAMILY_FULL ? 0 : stream_pos(m, STREAM_TEMPORARY, kBlock * plan.b1) - kBlock * step * plan.n0;
  const uint32_t k_c0 = (uint32_t)(c0 * a.sk.n * 2), k_c1 = (uint32_t)(c1 * a.sk.n * 2);
  const uint32_t v_c0 = (uint32_t)(c0 * a.sv.n * 2), v_c1 = (uint32_t)(c1 * a.sv.n * 2);

  // Register staging (head dims below 64).
  TileRegs<D> rk[kLook][NG], rv[kLook][NG];
  auto issue_regs = [&](int j, int slot) {
#pragma unroll
    for (int y = 0; y < NG; ++y) {
      const int i = NG * j + y;
      if (i < nb) {
        const bool s0 = i < plan.n0;
        rk[slot][y].load(k_src, (uint32_t)i * k_blk + (s0 ? k_c0 : k_c1), k_off, tid);
        rv[slot][y].load(v_src, (uint32_t)i * v_blk + (s0 ? v_c0 : v_c1), v_off, tid);
      }
    }
  };
  auto put_regs = [&](int slot, int buf) {
#pragma unroll
    for (int y = 0; y < NG; ++y) {
      rk[slot][y].store(sK[buf][y], tid);
      rv[slot][y].store(sV[buf][y], tid);
    }
  };
  // LDS-DMA staging (head dims of 64 and more).
  const auto k_dma = DT::sources(tid, (uint32_t)(step * a.sk.n * 2));
  const auto v_dma = DT::sources(tid, (uint32_t)(step * a.sv.n * 2));
  auto issue_dma = [&](int j, int buf) {
#pragma unroll
    for (int y = 0; y < NG; ++y) {
      const int i = NG * j + y;
      if (i < nb) {
        const bool s0 = i < plan.n0;
        DT::load(k_src, (uint32_t)i * k_blk + (s0 ? k_c0 : k_c1), k_dma, sK[buf][y], wave);
        DT::load(v_src, (uint32_t)i * v_blk + (s0 ? v_c0 : v_c1), v_dma, sV[buf][y], wave);
      }
    }
  };
  // Fragment reads of a staged key block.
  auto row_frag = [&](const uint16_t* tile, int c) {
    if constexpr (kDma)
      return lds_read_b128(tile + DT::frag(c32, g, c));
    else
      return lds_read_b128(tile + c32 * G::RS + 16 * c + 8 * g);
  };
  auto tr_frag = [&](const uint16_t* tile, int kh, int dc) {
    if constexpr (kDma)
      return DT::frag_tr(tile, 16 * kh, dc, lane);
    else
      return lds_frag_tr(tile, G::RS, 16 * kh, 32 * dc, lane);
  };
  // With LDS-DMA staging the first group's loads cost no registers: they go out now, with the Q /
  // dO / O fragment loads below, ahead of the lanes' setup.
  if constexpr (kDma) issue_dma(0, 0);

  f32x16_t acc[G::DC];
#pragma unroll
  for (int dc = 0; dc < G::DC; ++dc) acc[dc] = f32x16_t{};

  if (planned) q_lanes(m, qp, run_start, st);

  // Delta = rowsum(O * dO) of the lane's query, stored for the dK/dV pass: one v_dot2 per packed pair
  // (two exact products and the fp32 accumulation in one instruction), two independent partial sums.
  float delta;
  {
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
#pragma unroll
      for (int j = 0; j < 4; ++j) part[j & 1] = E::dot2(of[c][j], dof[c][j], part[j & 1]);
    }
    delta = half_sum(part[0] + part[1]);
  }
  const float lse = lse_raw == -INFINITY ? 0.f : lse_raw;  // a query with no visible key: every score is masked to -inf
  if (qvalid && g == 0) {
    // Seeds of the dK/dV pass for this query: -LSE and -Delta.
    float* seed = a.seeds + ((int64_t)b * a.H + h) * 2 * m.N + qp;
    seed[0] = -lse;
    seed[m.N] = -delta;
  }

  // The dP tile starts from -Delta, so it comes out of the MFMAs as dP - Delta and dS = P * dP' is one
  // VALU operation per element; the S tile is scaled in fp32 (one FMA per score forms
  // S * scale2 - LSE), never by rounding a scaled Q to the input type.
  const float scale2 = a.scale2, neg_lse = -lse;
  const f32x16_t c_dp = f32x16_t{} - delta;

  auto run = [&](auto exact_tag) {
    constexpr bool EXACT = decltype(exact_tag)::value;
    auto cls_of = [&](int i) {
      return classify_block(i < plan.n0 ? st.w0 : st.w1, plan.first(i), EXACT);
    };
    const BlockMask bm = q_block_mask(st, EXACT);
    auto body = [&](int j, int buf) {
      int act2, full2;
      group_codes<NG>(bm, NG * j, nb, cls_of, act2, full2);
#pragma unroll
      for (int y = 0; y < NG; ++y) {
        const int i = NG * j + y;
        const bool s0 = i < plan.n0;
        const int t0 = plan.first(i);
        const WaveSpan ws = s0 ? st.w0 : st.w1;
        const Interval lr = s0 ? st.r0 : st.r1;
        if ((act2 >> y) & 1) {
          const uint16_t* tK = sK[buf][y];
          const uint16_t* tV = sV[buf][y];
          f32x16_t sc = f32x16_t{}, dp = c_dp;
#pragma unroll
          for (int c = 0; c < D / 16; ++c) {
            sc = E::mfma(row_frag(tK, c), qf[c], sc);
            dp = E::mfma(row_frag(tV, c), dof[c], dp);
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) sc[e] = __builtin_fmaf(sc[e], scale2, neg_lse);
          if (!((full2 >> y) & 1))
            mask_partial<EXACT>(sc, lr, ws, t0, g,
                                [&] { return qs_exact_bits<D == 128 && WAVES == 2 ? 2 : 16>(a, b, lr, plan.stream(i), t0, g, dq_doc); });
          uint32_t dsk[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float p0 = fast_exp2(sc[2 * e]);
            const float p1 = fast_exp2(sc[2 * e + 1]);
            dsk[e] = E::pack2(p0 * dp[2 * e], p1 * dp[2 * e + 1]);
          }
#pragma unroll
          for (int dc = 0; dc < G::DC; ++dc) {
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
              const u32x4_t df = {dsk[4 * kh], dsk[4 * kh + 1], dsk[4 * kh + 2], dsk[4 * kh + 3]};
              acc[dc] = E::mfma(tr_frag(tK, kh, dc), df, acc[dc]);
            }
          }
        }
      }
    };
    if constexpr (kDma)
      run_groups_dma<NG, true>(nb, issue_dma, body);
    else
      run_groups<kLook, NG>(nb, issue_regs, put_regs, body);
  };
  if (exact)
    run(std::true_type{});
  else
    run(std::false_type{});

  uint16_t* orow = a.dq + b * a.sdq.b + h * a.sdq.h + (int64_t)qsafe * a.sdq.n;
  const float sc = a.sm_scale;
  auto piece = [&](int dc, int ii) {
    return u32x2_t{E::pack2(acc[dc][4 * ii] * sc, acc[dc][4 * ii + 1] * sc),
                   E::pack2(acc[dc][4 * ii + 2] * sc, acc[dc][4 * ii + 3] * sc)};
  };
  // Head dims of 64 and more with 16-byte aligned rows: dQ goes through the wave's idle LDS tile so
  // every global store writes whole rows.
  bool staged = false;
  if constexpr (D >= 64) {
    if (rows16_ok(a.dq, a.sdq)) {
      const int q0 = tp.tile * kTile + wave * kBlock;
      store_rows_via_lds<D>(wave_tile(sK, wave), lane, a.dq + b * a.sdq.b + h * a.sdq.h + (int64_t)q0 * a.sdq.n,
                            a.sdq.n, imin(kBlock, m.N - q0), piece);
      staged = true;
    }
  }
  if (qvalid && !staged) {
#pragma unroll
    for (int dc = 0; dc < G::DC; ++dc) {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int d0 = 32 * dc + 8 * ii + 4 * g;
        if (d0 < D) *reinterpret_cast<u32x2_t*>(orow + d0) = piece(dc, ii);
      }
    }
  }
}

}  // namespace sps
