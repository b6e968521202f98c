// Backward attention, bf16/f16 MFMA, gfx950. Two deterministic passes, no atomics, as in the
// reference (_sps_bwd_dq_kernel / _sps_bwd_dkdv_kernel, triton_sps_flash_attention.py:272-488;
// reverse twins triton_reverse_sps_flash_attention.py:370-599; full triton_full_flash_attention.py:301-460):
//
//  1. dQ pass (query-stationary, the forward's plan and classification). Its prologue computes
//     Delta = rowsum(O * dO) for its own queries and stores it for pass 2 (this replaces the
//     reference's separate _attn_bwd_preprocess launch). Per 32-key block:
//       S^T = K Q^T, dP^T = V dO^T (K, V rows from LDS; Q, dO in registers),
//       P = exp2(S*scale2 - LSE) (one fp32 FMA per score, as the reference scales its fp32 scores:
//       triton_sps_flash_attention.py:471), dS = P (dP - Delta)   (lane-local LSE and Delta),
//       dQ^T += K^T dS^T  (K^T fragments via ds_read_b64_tr_b16).
//  2. dK/dV pass (key-stationary; head dims up to 64, attn_bwd_split.hip has the larger ones). A
//     workgroup owns 128 keys of one stream (natural, persistent or temporary), each wave 32 of them
//     held in registers; it walks the 32-query chunks of the union of its lanes' query intervals
//     (persistent keys: diagonal to document end; temporary keys: the w-token window):
//       S = Q K^T, dP = dO V^T (Q, dO rows from LDS; K, V in registers),
//       P = exp2(S*scale2 - LSE) (fp32 FMA per score, triton_sps_flash_attention.py:361),
//       dV^T += dO^T P, dK^T += Q^T dS (dO^T, Q^T fragments via ds_read_b64_tr_b16).
// Both passes consume their tiles in groups of four 32-row blocks (one barrier per group) through
// the run_groups pipeline: buffer loads one group ahead into registers, double-buffered LDS; with
// documents the first group's loads leave right after the workgroup's plan is read. dK and dQ are
// scaled by sm_scale at the end, as in the reference.
#include "attn_bwd_dq.hpp"

namespace sps {

// Register-staged query chunk y of a dK/dV group (head dims below 64): Q and dO rows, plus (in wave
// y only) the chunk's -LSE (lanes 0-31) or -Delta (lanes 32-63) of query row lane % 32.
template <int D>
struct ChunkRegs {
  TileRegs<D> q, o;
  uint32_t seed;  // raw bits
};

template <int D, class E>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(bwd_waves<D>(), 8))) void attn_bwd_dkdv_kernel(const AttnArgs a) {
  using G = TileGeom<D>;
  constexpr int NG = bwd_group<D>();
  // Head dims of 64 and more stage Q / dO chunks and their seeds by direct global -> LDS loads into
  // dense swizzled tiles; smaller ones through registers into padded tiles.
  constexpr bool kDma = D >= 64;
  using DT = DmaTile<64>;
  constexpr bool kSkew = D == 64 && NG == 4;
  constexpr int kSkewMaxChunks = 16;
  constexpr int TE = kDma ? DT::ELEMS : G::ELEMS;
  __shared__ __attribute__((aligned(16))) uint16_t sQ[2][NG][TE];  // [buffer][chunk of the group]
  __shared__ __attribute__((aligned(16))) uint16_t sDO[2][NG][TE];
  // -LSE of the chunk's query rows in [0, kBlock), their -Delta in [kBlock, 2 kBlock).
  __shared__ __attribute__((aligned(16))) float sSeed[2][NG][2 * kBlock];
  __shared__ int s_span[2 * kWaves];
  __shared__ int s_steps[kWaves];

  const MaskSpec m = a.m;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index<D>();
  const int g = lane >> 5, c32 = lane & 31;
  int b, h;
  TilePlan tp;
  k_workgroup(a, b, h, tp);
  const RowView row = row_view(a, b, tp.mono);
  KState st;
  int run_end;
  const bool planned = k_begin(a, tp, row, s_span, st, run_end, tid >> 6);
  const int kp = st.kp;
  const bool kvalid = st.kvalid;
  const int nc = st.nc;
  const bool exact = row.mono;
  const int64_t dk_doc = (!exact && kvalid) ? load_doc(a, b, kp) : 0;
  // Skewed schedule: wave w's keys start 2w chunks after the tile's first key, and a temporary-stream
  // key with a short window sees only a few chunks, so waves sharing one 4-chunk group would each be
  // busy in about half of it. Instead, at step s wave w takes chunk 2w + s: the eight staged chunks
  // (both buffers, as one ring of slots) always hold chunks s .. s + 7, every wave has a block at
  // each step, and one chunk enters the ring per step.
  const bool skew = kSkew && st.stream == STREAM_TEMPORARY && nc > 0 && nc <= kSkewMaxChunks &&
                    (stream_pos(m, st.stream, st.first) >> 5) == st.c0;

  const BufRsrc q_src = head_rsrc<D>(a.q + b * a.sq.b + h * a.sq.h, a.sq.n, m.N);
  const BufRsrc o_src = head_rsrc<D>(a.dO + b * a.sdo.b + h * a.sdo.h, a.sdo.n, m.N);
  // Seeds of this (row, head): -LSE of every query, then -Delta of every query (written by the dQ pass).
  const BufRsrc seed_src = make_rsrc(a.seeds + ((int64_t)b * a.H + h) * 2 * m.N, (uint32_t)(2 * m.N * 4));

  // K and V fragments: B operands of S = Q K^T and dP = dO V^T (lane: key c32, d = 16c + 8g ..).
  u32x4_t kf[D / 16], vf[D / 16];
  {
    const uint16_t* krow = a.k + b * a.sk.b + h * a.sk.h + (int64_t)kp * a.sk.n;
    const uint16_t* vrow = a.v + b * a.sv.b + h * a.sv.h + (int64_t)kp * a.sv.n;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      u32x4_t z = {0u, 0u, 0u, 0u};
      kf[c] = kvalid ? *reinterpret_cast<const u32x4_t*>(krow + 16 * c + 8 * g) : z;
      vf[c] = kvalid ? *reinterpret_cast<const u32x4_t*>(vrow + 16 * c + 8 * g) : z;
    }
  }
  if constexpr (!kDma) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
#pragma unroll
      for (int y = 0; y < NG; ++y) {
        zero_pad_cols<D>(sQ[x][y], tid);
        zero_pad_cols<D>(sDO[x][y], tid);
      }
    }
  }

  // Byte offset of chunk i's first row: i * (bytes per chunk) + the first chunk's offset.
  const uint32_t q_blk = (uint32_t)(kBlock * a.sq.n * 2), o_blk = (uint32_t)(kBlock * a.sdo.n * 2);
  const uint32_t q_c0 = (uint32_t)((int64_t)st.c0 * kBlock * a.sq.n * 2);
  const uint32_t o_c0 = (uint32_t)((int64_t)st.c0 * kBlock * a.sdo.n * 2);
  // Byte offset, within the seed buffer, of the seed lane `lane` stages for chunk i (wave y of the
  // group stages chunk y's): -LSE for lanes 0-31, -Delta for lanes 32-63, of query row lane % 32.
  auto seed_off = [&](int i) {
    return (uint32_t)(((lane >> 5) * m.N + imin((st.c0 + i) * kBlock + c32, m.N - 1)) * 4);
  };

  // Register staging (head dims below 64).
  ChunkRegs<D> rc[kLook][NG];
  const auto q_off = TileRegs<D>::offsets(tid, (uint32_t)(a.sq.n * 2));
  const auto o_off = TileRegs<D>::offsets(tid, (uint32_t)(a.sdo.n * 2));
  auto issue_regs = [&](int j, int slot) {
#pragma unroll
    for (int y = 0; y < NG; ++y) {
      const int i = NG * j + y;
      if (i < nc) {
        rc[slot][y].q.load(q_src, q_c0 + (uint32_t)i * q_blk, q_off, tid);
        rc[slot][y].o.load(o_src, o_c0 + (uint32_t)i * o_blk, o_off, tid);
        if (wave == y % kWaves) rc[slot][y].seed = __builtin_amdgcn_raw_buffer_load_b32(seed_src, seed_off(i), 0, 0);
      }
    }
  };
  auto put_regs = [&](int slot, int buf) {
#pragma unroll
    for (int y = 0; y < NG; ++y) {
      rc[slot][y].q.store(sQ[buf][y], tid);
      rc[slot][y].o.store(sDO[buf][y], tid);
      if (wave == y % kWaves) sSeed[buf][y][lane] = __builtin_bit_cast(float, rc[slot][y].seed);
    }
  };
  // LDS-DMA staging (head dims of 64 and more).
  const auto q_dma = DT::sources(tid, (uint32_t)(a.sq.n * 2));
  const auto o_dma = DT::sources(tid, (uint32_t)(a.sdo.n * 2));
  auto issue_dma = [&](int j, int buf) {
#pragma unroll
    for (int y = 0; y < NG; ++y) {
      const int i = NG * j + y;
      if (i < nc) {
        DT::load(q_src, q_c0 + (uint32_t)i * q_blk, q_dma, sQ[buf][y], wave);
        DT::load(o_src, o_c0 + (uint32_t)i * o_blk, o_dma, sDO[buf][y], wave);
        if (wave == y % kWaves) lds_dma_b32(seed_src, sSeed[buf][y], seed_off(i));
      }
    }
  };
  // Fragment reads of a staged chunk tile.
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

  f32x16_t dk[G::DC], dv[G::DC];
#pragma unroll
  for (int dc = 0; dc < G::DC; ++dc) {
    dk[dc] = f32x16_t{};
    dv[dc] = f32x16_t{};
  }

  auto run = [&](auto exact_tag) {
    constexpr bool EXACT = decltype(exact_tag)::value;
    // The first group's loads go out with the lanes' run ends and the K/V fragments; what depends
    // on those waits below, for all of them at once.
    if constexpr (kDma)
      issue_dma(0, 0);
    else
      issue_regs(0, 0);
    if constexpr (kSkew)
      if (skew) issue_dma(1, 1);
    if (planned) k_lanes(m, run_end, st);
    // The dP tile starts from the -Delta seeds of its query rows, so it comes out of the MFMAs as
    // dP - Delta and dS = P * dP' is one VALU operation per element; the S tile is scaled in fp32 by
    // one FMA per score with the -LSE seeds (S * scale2 - LSE), never by rounding a scaled K.
    const float scale2 = a.scale2;
    auto cls_of = [&](int i) { return classify_block(st.w, (st.c0 + i) * kBlock, EXACT); };
    const BlockMask bm = k_block_mask(st, EXACT);
    // S and dP tiles of block y of the group (the dP tile starts from its rows' -Delta seeds).
    auto sdp = [&](const uint16_t* tQ, const uint16_t* tDO, const float* seed, f32x16_t& sc, f32x16_t& dp) {
      sc = f32x16_t{};
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        // Query rows 8*i4 + 4g + {0..3} of this chunk.
        const f32x4_t d4 = *reinterpret_cast<const SPS_LDS f32x4_t*>(
            (const SPS_LDS float*)(seed + kBlock + 8 * i4 + 4 * g));
#pragma unroll
        for (int t = 0; t < 4; ++t) dp[4 * i4 + t] = d4[t];
      }
#pragma unroll
      for (int c = 0; c < D / 16; ++c) {
        sc = E::mfma(row_frag(tQ, c), kf[c], sc);
        dp = E::mfma(row_frag(tDO, c), vf[c], dp);
      }
    };
    // Block y's S tile in fp32 (S * scale2 - LSE, the -LSE seeds read here), masked when partial.
    auto scores = [&](const float* seed, int qc, bool full, f32x16_t& sc) {
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4_t l4 = *reinterpret_cast<const SPS_LDS f32x4_t*>(
            (const SPS_LDS float*)(seed + 8 * i4 + 4 * g));
#pragma unroll
        for (int t = 0; t < 4; ++t) sc[4 * i4 + t] = __builtin_fmaf(sc[4 * i4 + t], scale2, l4[t]);
      }
      if (!full)
        mask_partial<EXACT>(sc, st.r, st.w, qc, g, [&] { return ks_exact_bits(a, b, kp, st.r.hi, qc, g, dk_doc); });
    };
    // P and dS of block y, then the dV and dK products.
    auto grads = [&](const uint16_t* tQ, const uint16_t* tDO, const f32x16_t& sc, const f32x16_t& dp) {
      uint32_t pk[8], dsk[8];
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        float p[4], ds[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int e = 4 * i4 + t;
          p[t] = fast_exp2(sc[e]);
          ds[t] = p[t] * dp[e];
        }
        pk[2 * i4] = E::pack2(p[0], p[1]);
        pk[2 * i4 + 1] = E::pack2(p[2], p[3]);
        dsk[2 * i4] = E::pack2(ds[0], ds[1]);
        dsk[2 * i4 + 1] = E::pack2(ds[2], ds[3]);
      }
#pragma unroll
      for (int dc = 0; dc < G::DC; ++dc) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
          const u32x4_t pf = {pk[4 * kh], pk[4 * kh + 1], pk[4 * kh + 2], pk[4 * kh + 3]};
          const u32x4_t df = {dsk[4 * kh], dsk[4 * kh + 1], dsk[4 * kh + 2], dsk[4 * kh + 3]};
          dv[dc] = E::mfma(tr_frag(tDO, kh, dc), pf, dv[dc]);
          dk[dc] = E::mfma(tr_frag(tQ, kh, dc), df, dk[dc]);
        }
      }
    };
    auto block = [&](const uint16_t* tQ, const uint16_t* tDO, const float* seed, int qc, bool full) {
      f32x16_t sc, dp;
      sdp(tQ, tDO, seed, sc, dp);
      scores(seed, qc, full, sc);
      grads(tQ, tDO, sc, dp);
    };
    auto body = [&](int j, int buf) {
      int act2, full2;
      group_codes<NG>(bm, NG * j, nc, cls_of, act2, full2);
#pragma unroll
      for (int y = 0; y < NG; ++y) {
        if ((act2 >> y) & 1) block(sQ[buf][y], sDO[buf][y], sSeed[buf][y], (st.c0 + NG * j + y) * kBlock, (full2 >> y) & 1);
      }
    };
    if constexpr (kSkew) {
      if (skew) {
        // Chunk c sits in slot c % 8 = (buffer, chunk of the group) (c % 8 / 4, c % 4). Chunks 0-7
        // were loaded by direct LDS loads before the lanes' setup; chunk s + 8 goes through
        // registers during step s and is written at the start of step s + 1 into the slot of chunk
        // s, which every wave has finished with by then (its last reader, wave 0, took it at step s).
        uint16_t* const ringQ = &sQ[0][0][0];
        uint16_t* const ringO = &sDO[0][0][0];
        float* const ringS = &sSeed[0][0][0];
        const uint64_t act = bm.act0, full = bm.full0;  // nc <= 16: every chunk's bit is in word 0
        // Steps: until every wave has reached its last active chunk.
        if (lane == 0) s_steps[wave] = (act ? 63 - __builtin_clzll(act) : -1) - 2 * wave + 1;
        vmem_wait_all();
        __syncthreads();
        int steps = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) steps = imax(steps, s_steps[w]);
        steps = wave_uniform(steps);
        u32x4_t rq = {0u, 0u, 0u, 0u}, ro = {0u, 0u, 0u, 0u};
        uint32_t rs = 0u;
        for (int sp = 0; sp < steps; ++sp) {
          if (sp > 0) {
            const int c = sp + 7;
            if (c < nc) {
              const int sl = c & 7;
              lds_write_b128(ringQ + sl * TE + tid * 8, rq);
              lds_write_b128(ringO + sl * TE + tid * 8, ro);
              if (wave == (c & 3)) ringS[sl * 2 * kBlock + lane] = __builtin_bit_cast(float, rs);
            }
          }
          {
            const int c = sp + 8;
            if (c < nc) {
              rq = buf_load_b128(q_src, q_c0 + (uint32_t)c * q_blk + q_dma.o[0]);
              ro = buf_load_b128(o_src, o_c0 + (uint32_t)c * o_blk + o_dma.o[0]);
              if (wave == (c & 3)) rs = __builtin_amdgcn_raw_buffer_load_b32(seed_src, seed_off(c), 0, 0);
            }
          }
          const int i = 2 * wave + sp;
          if (i < nc && ((act >> i) & 1ull)) {
            const int sl = i & 7;
            block(ringQ + sl * TE, ringO + sl * TE, ringS + sl * 2 * kBlock, (st.c0 + i) * kBlock, (full >> i) & 1ull);
          }
          lds_barrier();
        }
        return;
      }
    }
    if constexpr (kDma)
      run_groups_dma<NG, true>(nc, issue_dma, body);
    else
      run_groups<kLook, NG, true>(nc, issue_regs, put_regs, body);
  };
  if (exact)
    run(std::true_type{});
  else
    run(std::false_type{});

  const float sc = a.sm_scale;
  // Pieces of the lane's key row: d = 32 dc + 8 ii + 4 g .. +3 of dK (scaled by sm_scale) and dV.
  auto piece_k = [&](int dc, int ii) {
    return u32x2_t{E::pack2(dk[dc][4 * ii] * sc, dk[dc][4 * ii + 1] * sc),
                   E::pack2(dk[dc][4 * ii + 2] * sc, dk[dc][4 * ii + 3] * sc)};
  };
  auto piece_v = [&](int dc, int ii) {
    return u32x2_t{E::pack2(dv[dc][4 * ii], dv[dc][4 * ii + 1]), E::pack2(dv[dc][4 * ii + 2], dv[dc][4 * ii + 3])};
  };
  // With dense tiles and 16-byte aligned output rows the wave's 32 rows go through its own part of
  // the (now idle) first staging buffer, so every global store writes whole rows (dK/dV -4.6 % at C3).
  bool staged = false;
  if constexpr (kDma) {
    if (rows16_ok(a.dk, a.sdk) && rows16_ok(a.dv, a.sdv)) {
      // The wave's keys are consecutive indices of one stream: rows `step` positions apart.
      const int t0 = st.first + wave * kBlock;
      const int p0 = stream_pos(m, st.stream, t0);
      const int nrows = imin(kBlock, stream_len(m.family, m.N, st.stream, m.P) - t0);
      const int kstep = m.family == FAMILY_FULL ? 1 : 2;
      store_rows_via_lds<D>(wave_tile(sQ, wave), lane, a.dk + b * a.sdk.b + h * a.sdk.h + (int64_t)p0 * a.sdk.n,
                            kstep * a.sdk.n, nrows, piece_k);
      store_rows_via_lds<D>(wave_tile(sDO, wave), lane, a.dv + b * a.sdv.b + h * a.sdv.h + (int64_t)p0 * a.sdv.n,
                            kstep * a.sdv.n, nrows, piece_v);
      staged = true;
    }
  }
  if (!staged && kvalid) {
    uint16_t* dkrow = a.dk + b * a.sdk.b + h * a.sdk.h + (int64_t)kp * a.sdk.n;
    uint16_t* dvrow = a.dv + b * a.sdv.b + h * a.sdv.h + (int64_t)kp * a.sdv.n;
#pragma unroll
    for (int dc = 0; dc < G::DC; ++dc) {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int d0 = 32 * dc + 8 * ii + 4 * g;
        if (d0 < D) {
          *reinterpret_cast<u32x2_t*>(dkrow + d0) = piece_k(dc, ii);
          *reinterpret_cast<u32x2_t*>(dvrow + d0) = piece_v(dc, ii);
        }
      }
    }
  }
}

// Writes the visibility mask exactly as the key-stationary dK/dV kernel evaluates it.
__global__ __launch_bounds__(256) void mask_dump_kv_kernel(const AttnArgs a) {
  __shared__ int s_span[2 * kWaves];
  const MaskSpec m = a.m;
  const int tid = threadIdx.x, lane = tid & 63;
  const int g = lane >> 5;
  int b, h;
  TilePlan tp;
  k_workgroup(a, b, h, tp);
  const RowView row = row_view(a, b, tp.mono);
  KState st;
  int run_end;
  if (k_begin(a, tp, row, s_span, st, run_end, tid >> 6)) k_lanes(m, run_end, st);
  const bool exact = row.mono;
  const int64_t dk_doc = (!exact && st.kvalid) ? load_doc(a, b, st.kp) : 0;
  const BlockMask bm = k_block_mask(st, exact);
  for (int i = 0; i < st.nc; ++i) {
    const int qc = (st.c0 + i) * kBlock;
    const int cls = i < 128 ? mask_class(bm, i) : classify_block(st.w, qc, exact);
    if (cls == TILE_SKIP || !st.kvalid) continue;
    uint32_t bits = 0xffffu;
    if (cls == TILE_PARTIAL) {
      f32x16_t z = {};
      auto exact_bits = [&] { return ks_exact_bits(a, b, st.kp, st.r.hi, qc, g, dk_doc); };
      if (exact)
        mask_partial<true>(z, st.r, st.w, qc, g, exact_bits);
      else
        mask_partial<false>(z, st.r, st.w, qc, g, exact_bits);
      bits = 0;
      for (int e = 0; e < 16; ++e) bits |= (uint32_t)(z[e] == 0.f) << e;
    }
    for (int e = 0; e < 16; ++e) {
      const int qp = qc + acc_row(e, g);
      if (((bits >> e) & 1u) && qp < m.N) a.mask_out[((int64_t)b * m.N + qp) * m.N + st.kp] = 1;
    }
  }
}

template <int D, class E>
static hipError_t launch_bwd_t(const AttnArgs& a, int passes, hipStream_t stream) {
  const int64_t nq = (int64_t)q_tiles(a.m.N) * a.B * a.H;
  const int64_t nk = (int64_t)k_tiles(a.m.family, a.m.N, a.m.P) * a.B * a.H;
  if ((passes & kBwdDq) && nq > 0) {
    const dim3 grid((unsigned)nq), block(256);
    if (D == 128 && dq_two_waves(a.m, nq))
      hipLaunchKernelGGL((attn_bwd_dq_kernel<D, E, D == 128 ? 2 : dq_waves<D>()>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((attn_bwd_dq_kernel<D, E>), grid, block, 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if ((passes & kBwdDkdv) && nk > 0) {
    // From D = 128 on a wave cannot hold K, V, dK and dV of 32 keys beside another wave: two share them.
    if constexpr (D >= 128) {
      return launch_attn_bwd_dkdv_split(a, D, std::is_same<E, ElemF16>::value, nk, stream);
    } else {
      hipLaunchKernelGGL((attn_bwd_dkdv_kernel<D, E>), dim3((unsigned)nk), dim3(256), 0, stream, a);
      return hipGetLastError();
    }
  }
  return hipSuccess;
}

hipError_t launch_attn_bwd(const AttnArgs& a, int D, int is_f16, int passes, hipStream_t stream) {
#define SPS_BWD_CASE(DD)                                                                                  \
  case DD:                                                                                                \
    return is_f16 ? launch_bwd_t<DD, ElemF16>(a, passes, stream) : launch_bwd_t<DD, ElemBF16>(a, passes, stream);
  switch (D) {
    SPS_BWD_CASE(16)
    SPS_BWD_CASE(32)
    SPS_BWD_CASE(64)
    SPS_BWD_CASE(128)
    SPS_BWD_CASE(256)
    default:
      return hipErrorInvalidValue;
  }
#undef SPS_BWD_CASE
}

hipError_t launch_mask_dump_q(const AttnArgs& a, hipStream_t stream);

hipError_t launch_mask_dump(const AttnArgs& a, int schedule, hipStream_t stream) {
  if (schedule == 0) return launch_mask_dump_q(a, stream);
  const int n = k_tiles(a.m.family, a.m.N, a.m.P) * a.B * a.H;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(mask_dump_kv_kernel, dim3(n), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace sps
