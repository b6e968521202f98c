// Prefill -> decode state: after a prompt's batched prefill, the current document's K/V rows of one
// layer go into the decode caches (retained buffer: every token of the document; ring: its last
// window_tokens tokens), one launch for the whole batch instead of a per-row host loop.
//
// Reference: _materialize_prefill_layer_state (reverse_sps/inference.py:568-613). Per sequence b,
// doc = the token positions t with current_doc_mask[b, t] set, in increasing order (n = |doc|;
// rows with n == 0 are left untouched):
//   retained K/V[b, :, j, :] = K/V[b, 2 doc[j] + retained_slot, :, :]  (j < n), ret_len[b, :] = n
//   ring (window_tokens > 0): w = min(n, window_tokens), ring K/V[b, :, i, :] =
//     K/V[b, 2 doc[n - w + i] + window_slot, :, :] (i < w), ring_len[b] = w, ring_pos[b] = 0,
// with the rows converted to the cache dtype (round to nearest even).
//
// kPfSplit workgroups per (head, sequence): each compacts the mask row into an LDS list of positions (a
// shuffle scan gives each set position its rank; rows of up to kPfChunk tokens in one pass, whose total
// is the document's length, longer ones chunk by chunk after a count), then copies every kPfSplit-th
// group of rows with groups of D/8 threads moving 16-byte pieces, so a long document is copied by many
// workgroups at once. HBM-bound with latency around it: 16 sequences x 12 heads of ~768 tokens, D = 64
// (75 MB read and written) 22.0 -> 18.3 us on MI355X with all of a thread's loads ahead of its stores,
// the ring in a loop of its own (fewer live strides) and one pass over the mask.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cdna4.hpp"
#include "decode_kernels.hpp"

namespace sps {

namespace {

constexpr int kPfThreads = 256;
constexpr int kPfChunk = 2048;  // positions compacted per pass
constexpr int kPfSplit = 8;     // workgroups per (head, sequence)
constexpr int kPfRows = 2;      // rows of K and V a thread has in flight (4 measured 67 us, 2 18.3)

// Eight elements of a row as loaded: 16 bytes of 16-bit ones (lo), 32 of fp32.
struct Piece {
  u32x4_t lo, hi;
};

template <bool IN32>
__device__ __forceinline__ Piece load_piece(const void* p, int64_t i) {
  Piece r;
  r.hi = u32x4_t{0u, 0u, 0u, 0u};
  if constexpr (IN32) {
    r.lo = *reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p) + i);
    r.hi = *reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p) + i + 4);
  } else {
    r.lo = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(p) + i);
  }
  return r;
}

// Stores a piece of in_dtype as dtype (round to nearest even; bits unchanged where the types agree).
__device__ __forceinline__ void store_piece(void* p, int64_t i, int dtype, const Piece& in, int in_dtype) {
  if (dtype == in_dtype) {
    if (dtype == 2) {
      *reinterpret_cast<u32x4_t*>(static_cast<float*>(p) + i) = in.lo;
      *reinterpret_cast<u32x4_t*>(static_cast<float*>(p) + i + 4) = in.hi;
    } else {
      *reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(p) + i) = in.lo;
    }
    return;
  }
  float x[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = in.lo[e], hi = in.hi[e];
    if (in_dtype == 2) {
      x[e] = __builtin_bit_cast(float, lo);
      x[4 + e] = __builtin_bit_cast(float, hi);
    } else {
      x[2 * e] = in_dtype == 1 ? ElemF16::to_f32((uint16_t)(lo & 0xffffu)) : ElemBF16::to_f32((uint16_t)(lo & 0xffffu));
      x[2 * e + 1] = in_dtype == 1 ? ElemF16::to_f32((uint16_t)(lo >> 16)) : ElemBF16::to_f32((uint16_t)(lo >> 16));
    }
  }
  if (dtype == 2) {
    f32x4_t u, v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] = x[e];
      v[e] = x[4 + e];
    }
    *reinterpret_cast<f32x4_t*>(static_cast<float*>(p) + i) = u;
    *reinterpret_cast<f32x4_t*>(static_cast<float*>(p) + i + 4) = v;
  } else {
    u32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = dtype == 1 ? ElemF16::pack2(x[2 * e], x[2 * e + 1]) : ElemBF16::pack2(x[2 * e], x[2 * e + 1]);
    *reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(p) + i) = o;
  }
}

// Exclusive prefix sum over the workgroup's threads (shuffle scan per wave, wave totals in LDS).
__device__ int block_exclusive_sum(int x, int* s_tot, int& total) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int v = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(v, o);
    if (lane >= o) v += y;
  }
  if (lane == 63) s_tot[wave] = v;
  __syncthreads();
  int carry = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kPfThreads / 64; ++w) {
    const int t = s_tot[w];
    carry += w < wave ? t : 0;
    total += t;
  }
  __syncthreads();
  return carry + v - x;
}

}  // namespace

// IN32: fp32 input rows.
template <bool IN32>
__global__ __launch_bounds__(kPfThreads) void prefill_state_kernel(const PrefillStateArgs a) {
  __shared__ int s_pos[kPfChunk];
  __shared__ int s_tot[kPfThreads / 64];
  const int h = blockIdx.x, b = blockIdx.y, split = blockIdx.z, tid = threadIdx.x;
  const uint8_t* mrow = a.mask + (int64_t)b * a.mask_sb;

  const int pieces = a.D / 8;
  const int rows_per_pass = kPfThreads / pieces;
  const int r_in = tid / pieces, piece = tid - r_in * pieces;

  // The set positions of chunk [c0, c0 + span) into s_pos in order; returns how many there are.
  auto compact = [&](int c0, int span) {
    const int per = (span + kPfThreads - 1) / kPfThreads;  // contiguous positions per thread
    const int p0 = c0 + tid * per, p1 = p0 + per < c0 + span ? p0 + per : c0 + span;
    uint32_t set = 0;  // per <= kPfChunk / kPfThreads positions, all loaded together
#pragma unroll
    for (int u = 0; u < kPfChunk / kPfThreads; ++u) set |= (uint32_t)(p0 + u < p1 && mrow[p0 + u] != 0) << u;
    int total;
    int rank = block_exclusive_sum(__builtin_popcount(set), s_tot, total);
    for (; set; set &= set - 1) s_pos[rank++] = p0 + __builtin_ctz(set);
    __syncthreads();
    return total;
  };
  // Copies K and V rows of the positions s_pos[r0 .. r1) (parity `slot` of each token) to cache rows
  // `first`, first + 1, ...: kPfRows rows a thread at a time, every load before the first store (a load
  // behind a store, which might be to the same memory, would wait for the row before it).
  auto copy_rows = [&](int r0, int r1, int slot, void* dk, int64_t dk0, int64_t dk_st, void* dv, int64_t dv0,
                       int64_t dv_st, int first) {
    if (r_in >= rows_per_pass) return;
    const int step = rows_per_pass * kPfSplit;
    const int64_t k0 = b * a.k_sb + h * a.k_sh + slot * a.k_sn + 8 * piece;
    const int64_t v0 = b * a.v_sb + h * a.v_sh + slot * a.v_sn + 8 * piece;
    for (int r = r0 + r_in + split * rows_per_pass; r < r1; r += kPfRows * step) {
      Piece k[kPfRows], v[kPfRows];
#pragma unroll
      for (int u = 0; u < kPfRows; ++u) {
        const int64_t t2 = 2 * (int64_t)s_pos[r + u * step < r1 ? r + u * step : r];
        k[u] = load_piece<IN32>(a.k, k0 + t2 * a.k_sn);
        v[u] = load_piece<IN32>(a.v, v0 + t2 * a.v_sn);
      }
#pragma unroll
      for (int u = 0; u < kPfRows; ++u) {
        if (r + u * step >= r1) continue;
        const int64_t j = first + (r + u * step - r0);
        store_piece(dk, dk0 + j * dk_st + 8 * piece, a.kv_dtype, k[u], a.in_dtype);
        store_piece(dv, dv0 + j * dv_st + 8 * piece, a.kv_dtype, v[u], a.in_dtype);
      }
    }
  };
  // The rows of the `count` positions in s_pos, the first of rank `base` in the document: all to the
  // retained cache, the last w of the document's n to the ring too.
  auto copy_both = [&](int base, int count, int first_w) {
    const int kept = base < a.ret_storage ? (count < a.ret_storage - base ? count : a.ret_storage - base) : 0;
    copy_rows(0, kept, a.retained_slot, a.ret_k, b * a.tk_sb + h * a.tk_sh, a.tk_st, a.ret_v,
              b * a.tv_sb + h * a.tv_sh, a.tv_st, base);
    if (a.window > 0) {
      const int from = first_w > base ? first_w - base : 0;
      const int room = first_w + a.ring_storage - base;  // ring rows are i = rank - first_w < ring_storage
      copy_rows(from, count < room ? count : room, a.window_slot, a.ring_k, b * a.rk_sb + h * a.rk_sh, a.rk_st,
                a.ring_v, b * a.rv_sb + h * a.rv_sh, a.rv_st, base + from - first_w);
    }
  };

  int n, w = 0;
  if (a.T <= kPfChunk) {
    n = compact(0, a.T);
    if (n == 0) return;  // untouched, as in the reference (uniform over the workgroup)
    w = a.window > 0 ? (n < a.window ? n : a.window) : 0;
    copy_both(0, n, n - w);
  } else {
    // Longer rows: the document's length first, then chunk by chunk.
    int cnt = 0;
    for (int t = tid; t < a.T; t += kPfThreads) cnt += mrow[t] != 0;
    block_exclusive_sum(cnt, s_tot, n);
    if (n == 0) return;
    w = a.window > 0 ? (n < a.window ? n : a.window) : 0;
    int base = 0;  // ranks before this chunk
    for (int c0 = 0; c0 < a.T; c0 += kPfChunk) {
      const int count = compact(c0, (a.T - c0) < kPfChunk ? (a.T - c0) : kPfChunk);
      copy_both(base, count, n - w);
      base += count;
      __syncthreads();  // s_pos is rewritten by the next chunk
    }
  }
  if (tid == 0 && split == 0) {
    const int64_t nl = n < a.ret_storage ? n : a.ret_storage;
    const int64_t off = b * a.ret_len_sb + h * a.ret_len_sh;
    if (a.len_i64) reinterpret_cast<int64_t*>(a.ret_len)[off] = nl;
    else reinterpret_cast<int*>(a.ret_len)[off] = (int)nl;
    if (a.window > 0 && h == 0) {
      if (a.len_i64) {
        reinterpret_cast<int64_t*>(a.ring_len)[b * a.ring_len_sb] = w;
        reinterpret_cast<int64_t*>(a.ring_pos)[b * a.ring_pos_sb] = 0;
      } else {
        reinterpret_cast<int*>(a.ring_len)[b * a.ring_len_sb] = w;
        reinterpret_cast<int*>(a.ring_pos)[b * a.ring_pos_sb] = 0;
      }
    }
  }
}

hipError_t launch_prefill_state(const PrefillStateArgs& a, hipStream_t stream) {
  if (a.B == 0 || a.H == 0 || a.T == 0) return hipSuccess;
  const dim3 grid(a.H, a.B, kPfSplit);
  if (a.in_dtype == 2)
    hipLaunchKernelGGL(prefill_state_kernel<true>, grid, dim3(kPfThreads), 0, stream, a);
  else
    hipLaunchKernelGGL(prefill_state_kernel<false>, grid, dim3(kPfThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace sps
