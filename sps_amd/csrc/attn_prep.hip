// Row-layout prepass of the attention kernels (one workgroup per batch row).
//
// From a row's document ids it writes, for every position, the first and last position of the
// maximal run of equal ids containing it, and whether the row's ids are non-decreasing. In a
// non-decreasing row every document is one run, so the attention kernels turn the document mask
// into interval bounds (see attn_sched.hpp). A row with decreasing steps is recorded as one run
// covering the row (start 0, end N - 1) and the kernels compare ids pair by pair there.
//
// It also writes the work plan of every query tile and key tile (the 32-row blocks covering the
// union of the tile's lanes' visible intervals, per stream: exactly what the kernels would derive
// from the run bounds, in closed form from the tile's first and last rows) in decreasing order of block count, so the heaviest workgroups are
// dispatched first and each workgroup starts its first tile loads after reading one plan. The order
// only affects speed: it is always a permutation of the tiles.
#include <type_traits>

#include "attn_kernels.hpp"

namespace sps {

constexpr int kPrepThreads = 1024;
constexpr int kMaxSortTiles = 2048;  // rows with more tiles keep the closed-form order

// Exclusive scans of the per-thread chunk summaries, both in one pass so their latencies overlap:
// a max-scan of `up` in thread order and a min-scan of `down` in reverse thread order. Inside each
// wave: DPP shifts within the 16-lane rows (no LDS round trips), then the rows' totals from one lane
// each; across the waves: their totals through LDS, read back as vectors (two barriers in all).
constexpr int kPrepWaves = kPrepThreads / 64;
static_assert(kPrepWaves == 16, "the wave totals are read back as four int4 vectors");

template <int CTRL>
__device__ __forceinline__ int dpp_shift(int x, int id) {
  // Lanes whose source lane lies outside the shift's range get `id`.
  return __builtin_amdgcn_update_dpp(id, x, CTRL, 0xF, 0xF, false);
}

__device__ void block_exclusive_scans(int* s_up, int* s_down, int up, int down, int up_identity, int down_identity,
                                      int& up_ex, int& down_ex) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row = lane >> 4;
  const int iu = up_identity, id = down_identity;
  // Inclusive max-scan upward (row_shr 1, 2, 4, 8) and min-scan downward (row_shl 1, 2, 4, 8) per row.
  int u = up, d = down;
  u = imax(u, dpp_shift<0x111>(u, iu));
  d = imin(d, dpp_shift<0x101>(d, id));
  u = imax(u, dpp_shift<0x112>(u, iu));
  d = imin(d, dpp_shift<0x102>(d, id));
  u = imax(u, dpp_shift<0x114>(u, iu));
  d = imin(d, dpp_shift<0x104>(d, id));
  u = imax(u, dpp_shift<0x118>(u, iu));
  d = imin(d, dpp_shift<0x108>(d, id));
  // Across the rows: row r adds the totals of rows below it (up) / above it (down).
  const int t0 = __builtin_amdgcn_readlane(u, 15), t1 = __builtin_amdgcn_readlane(u, 31);
  const int t2 = __builtin_amdgcn_readlane(u, 47), t3 = __builtin_amdgcn_readlane(u, 63);
  const int p1 = t0, p2 = imax(t0, t1), p3 = imax(p2, t2);
  u = imax(u, row == 0 ? iu : row == 1 ? p1 : row == 2 ? p2 : p3);
  const int b0 = __builtin_amdgcn_readlane(d, 0), b1 = __builtin_amdgcn_readlane(d, 16);
  const int b2 = __builtin_amdgcn_readlane(d, 32), b3 = __builtin_amdgcn_readlane(d, 48);
  const int s2 = b3, s1 = imin(b2, b3), s0 = imin(b1, s1);
  d = imin(d, row == 3 ? id : row == 2 ? s2 : row == 1 ? s1 : s0);
  if (lane == 0) {
    s_up[wave] = imax(p3, t3);
    s_down[wave] = imin(b0, s0);
  }
  // The lane's exclusive value inside the wave: its neighbour's inclusive one (wave_shr / wave_shl 1).
  const int eu = dpp_shift<0x138>(u, iu), ed = dpp_shift<0x130>(d, id);
  __syncthreads();
  int cu = iu, cd = id;
#pragma unroll
  for (int k = 0; k < kPrepWaves / 4; ++k) {
    const int4 vu = reinterpret_cast<const int4*>(s_up)[k], vd = reinterpret_cast<const int4*>(s_down)[k];
    const int w = 4 * k;
    cu = imax(cu, w + 0 < wave ? vu.x : iu);
    cu = imax(cu, w + 1 < wave ? vu.y : iu);
    cu = imax(cu, w + 2 < wave ? vu.z : iu);
    cu = imax(cu, w + 3 < wave ? vu.w : iu);
    cd = imin(cd, w + 0 > wave ? vd.x : id);
    cd = imin(cd, w + 1 > wave ? vd.y : id);
    cd = imin(cd, w + 2 > wave ? vd.z : id);
    cd = imin(cd, w + 3 > wave ? vd.w : id);
  }
  __syncthreads();  // the wave totals may be overwritten by a later scan
  up_ex = imax(cu, eu);
  down_ex = imin(cd, ed);
}

// Minimum / maximum over each group of 8 consecutive lanes (all lanes active), held by every lane
// of the group: quad swaps, then the half-row mirror.
template <class Op>
__device__ __forceinline__ int group8_reduce(int x, Op op) {
  x = op(x, __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false));   // quad_perm [1, 0, 3, 2]
  x = op(x, __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false));   // quad_perm [2, 3, 0, 1]
  return op(x, __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false));  // row_half_mirror
}
__device__ __forceinline__ int group8_min(int x) { return group8_reduce(x, [](int u, int v) { return imin(u, v); }); }
__device__ __forceinline__ int group8_max(int x) { return group8_reduce(x, [](int u, int v) { return imax(u, v); }); }

// Ranks `n` <= kMaxSortTiles tiles by decreasing cost (ties: lower index first) and calls
// emit(rank, tile) for each, with threads [first, first + count) of the workgroup (rank sort; the
// cost reads are batched so their LDS latencies overlap).
template <class Emit>
__device__ void sort_tiles(const int* cost, int n, int first, int count, Emit emit) {
  const int tid = threadIdx.x - first;
  if (tid < 0 || tid >= count) return;
  for (int t = tid; t < n; t += count) {
    const int c = cost[t];
    int r = 0, j = 0;
    for (; j + 8 <= n; j += 8) {
      int x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = cost[j + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) r += (x[u] > c) || (x[u] == c && j + u < t);
    }
    for (; j < n; ++j) r += (cost[j] > c) || (cost[j] == c && j < t);
    emit(r, t);
  }
}

// One workgroup a row: bound by the instructions and latencies of its phases on one CU, not by bytes.
// kRegIds is therefore no larger than the row needs (MI355X: N = 2048 with 8 ids a thread 7.0-8.1 us,
// with 2 5.0-6.2; N = 4096 with 8 9.5, with 4 8.0).
// kRegIds: ids per thread held in registers; rows of up to kPrepThreads * kRegIds positions keep their
// ids there and their runs in LDS.
template <int kRegIds>
__global__ __launch_bounds__(kPrepThreads) void row_layout_kernel(const AttnArgs a) {
  constexpr int kLdsRow = kPrepThreads * kRegIds;
  __shared__ __attribute__((aligned(16))) int s_scan[kPrepThreads];
  __shared__ int s_cost[kMaxSortTiles], s_cost_k[kMaxSortTiles];
  __shared__ int s_qplan[kMaxSortTiles][4], s_kplan[kMaxSortTiles][2];
  __shared__ int s_nonmono;
  __shared__ __attribute__((aligned(16))) uint16_t s_start[kLdsRow], s_end[kLdsRow];
  const MaskSpec m = a.m;
  const int b = blockIdx.x, tid = threadIdx.x, N = m.N;
  int* start = a.run_start + (int64_t)b * N;
  int* end = a.run_end + (int64_t)b * N;
  // Rows that fit give each thread kRegIds consecutive positions, longer ones an even share.
  const bool in_regs = N <= kLdsRow;
  const int C = in_regs ? kRegIds : (N + kPrepThreads - 1) / kPrepThreads;
  const int p0 = imin(tid * C, N), p1 = imin(p0 + C, N);
  if (tid == 0) s_nonmono = 0;

  int last = -1, first = N;
  bool dec = false;
  int64_t d[kRegIds];
  bool flag[kRegIds];
  if (in_regs) {
    // Common case: every id of this thread's chunk (and its predecessor) loaded once, together, in
    // 16-byte pieces where the chunk is whole, else one by one with positions clamped into the row (values
    // past the chunk are never used). The pieces start at an id, wherever it lies: rows of odd lengths are not
    // 16-byte aligned, and global loads need 4 bytes only.
    int64_t before = 0;
    auto load_all = [&](auto* ids) {
      using T = std::remove_cv_t<std::remove_pointer_t<decltype(ids)>>;
      ids += (int64_t)b * a.docs_sb;
      constexpr int kBytes = kRegIds * (int)sizeof(T), kVec = kBytes < 16 ? kBytes : 16;
      typedef T vec_t __attribute__((ext_vector_type(kVec / (int)sizeof(T)), aligned(sizeof(T))));
      const int64_t bv = ids[imax(imin(p0, N) - 1, 0)];
      if (p0 + kRegIds <= N) {
        vec_t x[kBytes / kVec];
#pragma unroll
        for (int v = 0; v < kBytes / kVec; ++v) x[v] = reinterpret_cast<const vec_t*>(ids + p0)[v];
#pragma unroll
        for (int j = 0; j < kRegIds; ++j) d[j] = x[j * (int)sizeof(T) / kVec][j % (kVec / (int)sizeof(T))];
      } else {
#pragma unroll
        for (int j = 0; j < kRegIds; ++j) d[j] = ids[imin(p0 + j, N - 1)];
      }
      before = (p0 > 0 && p0 < N) ? bv : 0;
    };
    if (a.docs_i64)
      load_all(reinterpret_cast<const int64_t*>(a.docs));
    else
      load_all(reinterpret_cast<const int32_t*>(a.docs));
#pragma unroll
    for (int j = 0; j < kRegIds; ++j) {
      const int p = p0 + j;
      const int64_t prev = j == 0 ? before : d[j - 1];
      flag[j] = p < p1 && (p == 0 || d[j] != prev);
      dec |= p < p1 && p > 0 && d[j] < prev;
      if (flag[j]) {
        last = p;
        first = imin(first, p);
      }
    }
  } else {
    int64_t prev = p0 > 0 ? load_doc(a, b, p0 - 1) : 0;
    for (int p = p0; p < p1; ++p) {
      const int64_t x = load_doc(a, b, p);
      if (p == 0 || x != prev) {
        last = p;
        first = imin(first, p);
      }
      dec |= (p > 0 && x < prev);
      prev = x;
    }
  }
  __syncthreads();
  if (dec) atomicOr(&s_nonmono, 1);
  int carry_start, carry_next;
  block_exclusive_scans(s_scan, s_scan + kPrepWaves, last, first, -1, N, carry_start, carry_next);
  const bool mono = s_nonmono == 0;

  int cs[kRegIds], ce[kRegIds];  // run bounds of the thread's positions (rows that fit)
  if (in_regs) {
    int cur = carry_start, nxt = carry_next;
#pragma unroll
    for (int j = 0; j < kRegIds; ++j) {
      if (flag[j]) cur = p0 + j;
      cs[j] = mono ? cur : 0;
    }
#pragma unroll
    for (int j = kRegIds - 1; j >= 0; --j) {
      ce[j] = mono ? nxt - 1 : N - 1;
      if (flag[j]) nxt = p0 + j;
    }
    // Into LDS for the plans, two positions a word (a partial chunk's rest lies inside the arrays); the
    // global arrays follow once the plans can start.
#pragma unroll
    for (int j = 0; j < kRegIds; j += 2) {
      reinterpret_cast<uint32_t*>(s_start)[(tid * kRegIds + j) / 2] = (uint32_t)(cs[j] & 0xffff) | (uint32_t)cs[j + 1] << 16;
      reinterpret_cast<uint32_t*>(s_end)[(tid * kRegIds + j) / 2] = (uint32_t)(ce[j] & 0xffff) | (uint32_t)ce[j + 1] << 16;
    }
  } else if (mono) {
    int cur = carry_start;
    int64_t prev = p0 > 0 ? load_doc(a, b, p0 - 1) : 0;
    for (int p = p0; p < p1; ++p) {
      const int64_t x = load_doc(a, b, p);
      if (p == 0 || x != prev) cur = p;
      start[p] = cur;
      prev = x;
    }
    int nxt = carry_next;
    for (int p = p1 - 1; p >= p0; --p) {
      end[p] = nxt - 1;
      if (p == 0 || load_doc(a, b, p) != load_doc(a, b, p - 1)) nxt = p;
    }
  } else {
    for (int p = p0; p < p1; ++p) {
      start[p] = 0;
      end[p] = N - 1;
    }
  }
  if (tid == 0) a.row_mono[b] = mono ? 1 : 0;
  if (in_regs) {
    lds_barrier();  // the plans read only LDS
    // The global arrays; the stores drain while the plans below are computed. Rows the store width divides: the
    // thread's own positions, 4 (2) a store. Others: consecutive positions of the wave from LDS, since 4-byte stores
    // of own positions touch a line each (with the ids' loads in pieces, prepass and a one-head forward, B4, N = 7001:
    // 38.4 -> 31.3 us with int32 ids, 37.0 -> 31.4 with int64).
    constexpr int kStore = kRegIds < 4 ? kRegIds : 4;
    typedef int store_t __attribute__((ext_vector_type(kStore)));
    if ((N & (kStore - 1)) == 0) {
      if (p0 < N) {
#pragma unroll
        for (int j = 0; j < kRegIds; j += kStore) {
          if (p0 + j >= N) continue;
          store_t vs, ve;
#pragma unroll
          for (int u = 0; u < kStore; ++u) {
            vs[u] = cs[j + u];
            ve[u] = ce[j + u];
          }
          *reinterpret_cast<store_t*>(start + p0 + j) = vs;
          *reinterpret_cast<store_t*>(end + p0 + j) = ve;
        }
      }
    } else {
      for (int p = tid; p < N; p += kPrepThreads) {
        start[p] = s_start[p];
        end[p] = s_end[p];
      }
    }
  } else {
    __syncthreads();  // start/end of the whole row are visible to every thread below
  }
  // Rows that fit read their run bounds from LDS (16 bits: positions < kLdsRow <= 8192).
  const bool lds_ok = in_regs;

  // Query-tile and key-tile plans, then both sorts. Rows with more than
  // kMaxSortTiles tiles keep the closed-form order (query tiles last to first, key tiles first to
  // last) and write their plans directly.
  const int nqt = q_tiles(N);
  const int nkt = k_tiles(m.family, N, m.P);
  const bool sort_q = nqt <= kMaxSortTiles, sort_k = nkt <= kMaxSortTiles;
  TilePlan* qplan = a.q_plan + (int64_t)b * nqt;
  TilePlan* kplan = a.k_plan + (int64_t)b * nkt;
  const int mono_flag = mono ? 1 : 0;
  // One 8-lane group per tile, one lane per row of the tile's first and last kTileEnds rows (the
  // rows q_tile_union / k_tile_union take), the group's intervals combined by three DPP steps:
  // query tiles on waves 0-7, key tiles on waves 8-15 (no wave runs both paths), 64 tiles per pass.
  // The run bounds come from LDS or from global memory in two separate copies of the loop: with a
  // global read anywhere in it, the loads' waits (vmcnt counts stores too) would also wait for the
  // run-bound stores above.
  static_assert(2 * kTileEnds == 8, "one lane of an 8-lane group per end row");
  const bool key_half = tid >= kPrepThreads / 2;
  const int lt = tid & (kPrepThreads / 2 - 1), grp = lt >> 3, row8 = lt & 7;
  auto plans = [&](auto st_of, auto en_of) {
    const int n = key_half ? nkt : nqt;
    for (int t0 = 0; t0 < n; t0 += kPrepThreads / 16) {
      const int t = t0 + grp;
      if (!key_half) {
        Interval i0 = {kEmptyLo, kEmptyHi}, i1 = i0;
        const int q = t < n ? q_tile_row(m, t, row8) : -1;
        if (q >= 0) query_intervals(m, q, st_of(q), i0, i1);
        const Interval u0 = {group8_min(i0.lo), group8_max(i0.hi)}, u1 = {group8_min(i1.lo), group8_max(i1.hi)};
        if (t < n && row8 == 0) {
          int b0, n0, b1, n1;
          cover_blocks(u0.lo, u0.hi, b0, n0);
          cover_blocks(u1.lo, u1.hi, b1, n1);
          if (sort_q) {
            s_cost[t] = n0 + n1;
            s_qplan[t][0] = b0;
            s_qplan[t][1] = n0;
            s_qplan[t][2] = b1;
            s_qplan[t][3] = n1;
          } else {
            qplan[nqt - 1 - t] = TilePlan{t, mono_flag, b0, n0, b1, n1, 0, 0};
          }
        }
      } else {
        Interval r = {kEmptyLo, kEmptyHi};
        int stream = STREAM_NATURAL;
        const int kp = t < n ? k_tile_row(m, t, row8, stream) : -1;
        if (kp >= 0) {
          const int last = key_last_query(m, stream, kp, en_of(kp));
          if (last >= kp) r = Interval{kp, last};
        }
        const Interval k = {group8_min(r.lo), group8_max(r.hi)};
        if (t < n && row8 == 0) {
          int c0, nc;
          cover_blocks(k.lo, k.hi, c0, nc);
          if (sort_k) {
            s_cost_k[t] = nc;
            s_kplan[t][0] = c0;
            s_kplan[t][1] = nc;
          } else {
            kplan[t] = TilePlan{t, mono_flag, c0, nc, 0, 0, 0, 0};
          }
        }
      }
    }
  };
  if (lds_ok)
    plans([&](int q) { return (int)s_start[q]; }, [&](int k) { return (int)s_end[k]; });
  else
    plans([&](int q) { return start[q]; }, [&](int k) { return end[k]; });
  lds_barrier();  // the plans and costs are in LDS; the run-bound stores above keep draining
  if (sort_q)
    sort_tiles(s_cost, nqt, 0, kPrepThreads / 2, [&](int r, int t) {
      qplan[r] = TilePlan{t, mono_flag, s_qplan[t][0], s_qplan[t][1], s_qplan[t][2], s_qplan[t][3], 0, 0};
    });
  if (sort_k)
    sort_tiles(s_cost_k, nkt, kPrepThreads / 2, kPrepThreads / 2, [&](int r, int t) {
      kplan[r] = TilePlan{t, mono_flag, s_kplan[t][0], s_kplan[t][1], 0, 0, 0, 0};
    });
}

hipError_t launch_row_layout(const AttnArgs& a, hipStream_t stream) {
  if (a.B == 0 || a.m.N == 0 || !a.m.has_docs) return hipSuccess;
  const dim3 grid(a.B), block(kPrepThreads);
  if (a.m.N <= 2 * kPrepThreads)
    hipLaunchKernelGGL(row_layout_kernel<2>, grid, block, 0, stream, a);
  else if (a.m.N <= 4 * kPrepThreads)
    hipLaunchKernelGGL(row_layout_kernel<4>, grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL(row_layout_kernel<8>, grid, block, 0, stream, a);
  return hipGetLastError();
}

}  // namespace sps
