// Internal helpers shared by the gfx950 KV-cache kernels: error reporting,
// dtype traits, 16-bit vector types for the MFMA builtins, wave primitives.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "../../include/nslg_kv.h"

namespace nslg {

// ---- error reporting (thread-local text, integer status) -------------------
void set_error(const char* fmt, ...);
int fail(int code, const char* fmt, ...);
int check_launch(const char* what);

inline int elem_bytes(int dtype) {
  switch (dtype) {
    case NSLG_F16: return 2;
    case NSLG_BF16: return 2;
    case NSLG_F32: return 4;
    default: return 0;
  }
}

inline hipStream_t as_stream(nslg_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// ---- vector types -------------------------------------------------------------
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// 16-bit element tags. Kernels move raw 16-bit words and only reinterpret them
// at the MFMA / conversion boundary.
struct F16 {
  static constexpr int kDtype = NSLG_F16;
  __device__ static inline float to_f32(unsigned short u) {
    return (float)__builtin_bit_cast(_Float16, u);
  }
  __device__ static inline unsigned short from_f32(float x) {
    return __builtin_bit_cast(unsigned short, (_Float16)x);
  }
  // D[16x16] += A[16x32] * B[32x16]   (8 elements per lane per operand)
  __device__ static inline f32x4 mma_k32(u16x8 a, u16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  // D[16x16] += A[16x16] * B[16x16]   (4 elements per lane per operand)
  __device__ static inline f32x4 mma_k16(u16x4 a, u16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                                 __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
  }
};

struct BF16 {
  static constexpr int kDtype = NSLG_BF16;
  __device__ static inline float to_f32(unsigned short u) {
    return __builtin_bit_cast(float, (unsigned int)u << 16);
  }
  __device__ static inline unsigned short from_f32(float x) {
    return __builtin_bit_cast(unsigned short, (__bf16)x);
  }
  __device__ static inline f32x4 mma_k32(u16x8 a, u16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ static inline f32x4 mma_k16(u16x4 a, u16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a),
                                                     __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
  }
};

// ---- wave helpers ---------------------------------------------------------------
__device__ inline float wave_xor_max(float x, int mask) {
  return fmaxf(x, __shfl_xor(x, mask, 64));
}
__device__ inline float wave_xor_sum(float x, int mask) {
  return x + __shfl_xor(x, mask, 64);
}

// Reductions over the four 16-lane rows of a wave (lanes l, l^16, l^32, l^48) with
// gfx950's row-swap permutes: v_permlane16_swap(x, x) leaves rows {0,0,2,2} in one
// result and {1,1,3,3} in the other, v_permlane32_swap(x, x) rows {0,1,0,1} and
// {2,3,2,3}. VALU only: no LDS instruction, no wait on the LDS counter.
__device__ inline float rows_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ inline float rows_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Sum over the wave's lanes.
__device__ inline int wave_sum_i32(int x) {
  x += __builtin_amdgcn_mov_dpp(x, 0x128, 0xf, 0xf, false);  // row_ror:8
  x += __builtin_amdgcn_mov_dpp(x, 0x124, 0xf, 0xf, false);  // row_ror:4
  x += __builtin_amdgcn_mov_dpp(x, 0x122, 0xf, 0xf, false);  // row_ror:2
  x += __builtin_amdgcn_mov_dpp(x, 0x121, 0xf, 0xf, false);  // row_ror:1
  const auto a = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
  x = (int)(a[0] + a[1]);
  const auto c = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
  return (int)(c[0] + c[1]);
}

// Largest value of the wave's lanes.
__device__ inline int wave_max_i32(int x) {
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0x128, 0xf, 0xf, false));  // row_ror:8
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0x124, 0xf, 0xf, false));  // row_ror:4
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0x122, 0xf, 0xf, false));  // row_ror:2
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0x121, 0xf, 0xf, false));  // row_ror:1
  const auto a = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
  x = max((int)a[0], (int)a[1]);
  const auto c = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
  return max((int)c[0], (int)c[1]);
}

__device__ inline float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ---- rotary embedding, the eager expression's arithmetic -------------------------
// out[d] = rnd(rnd(x[d] * c) + rnd(rot[d] * s)) in the storage type T, with c and s
// the table values rounded to T and rot = cat(-x[D/2:], x[:D/2]). A 16-bit times
// 16-bit product is exact in fp32 and the sum is done in fp32, as the eager ops do,
// so results match them bit for bit.
template <typename T>
__device__ inline unsigned short rope_elem(float x, float c, float r, float s) {
  float a = T::to_f32(T::from_f32(x * c));
  float b = T::to_f32(T::from_f32(r * s));
  // Both products stay rounded on their own: without this the compiler narrows the
  // ops to 16 bits and fuses one product into the add (v_fma_f16 / v_fma_mix),
  // which rounds once where the eager ops round twice.
  asm volatile("" : "+v"(a), "+v"(b));
  return T::from_f32(a + b);
}

__device__ inline void load8f(const float* p, float (&f)[8]) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p);
  const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[e] = a[e];
    f[4 + e] = b[e];
  }
}

// Rotates the 8 elements at d0 .. d0 + 7 of one head (lo: d0 < D/2, whose partners
// are at d0 + D/2; else partners at d0 - D/2) at table rows crow / srow: x holds the
// elements, y their partners.
template <typename T, typename V8>
__device__ inline V8 rope8(V8 x, V8 y, const float* crow, const float* srow, int d0, bool lo) {
  float c[8], sn[8];
  load8f(crow + d0, c);
  load8f(srow + d0, sn);
  V8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float xe = T::to_f32(x[e]);
    const float ye = T::to_f32(y[e]);
    const float ce = T::to_f32(T::from_f32(c[e]));
    const float se = T::to_f32(T::from_f32(sn[e]));
    o[e] = lo ? rope_elem<T>(xe, ce, -ye, se) : rope_elem<T>(xe, ce, ye, se);
  }
  return o;
}

// ---- streaming (non-temporal) vector accesses -----------------------------------
// Pool pages written by the append / zero / copy kernels are not read again by the
// writing kernel: stored with the non-temporal hint they go out to HBM instead of
// lingering as dirty lines in the memory-side cache, where the next decode, which
// streams the whole pool, would pay for writing them back (measured: a decode right
// after ~300 MB of ordinary stores into the pool, 590 us instead of 470 us).
template <typename V>
__device__ inline void stream_store(V* p, V v) {
  __builtin_nontemporal_store(v, p);
}

// ---- row tiles of a ragged prefill batch, longest first --------------------------
// Sequence b's n_b new tokens x G query heads are cut into tiles of `rows` query rows;
// later tiles see more keys (causal). Slot g of a launch is one tile, in an order that
// leaves short tiles for the end:
//   near-uniform batches (the chunks of a batch of prompts): in rounds, round r taking
//     each sequence's r-th tile from the end;
//   others: the sequences in batch order, so that neighbouring workgroups read one
//     sequence's keys, each one's tiles from the end.
// Measured with one layer's call, tiles from the front before: 8 prompts of 300 to 2000
// tokens 216 -> 206 us (D = 256 273 -> 233), 4 of 517 to 1463 at D = 64 76.8 -> 68.4, 16
// suffixes over a shared prefix 481 -> 477 (all tiles by their keys: 505; sequences by
// their tokens: 493). Every wave finds its tile by itself, the lanes holding the
// sequences.
struct PrefillSeq {
  int b, tile, q0, n_new, len;  // sequence, row tile, first ragged row, new tokens, tokens in all
};

__device__ inline bool locate_row_tile(const int32_t* qo, const int32_t* indptr, const int32_t* last_len, int page_size,
                                       int batch, int G, int rows, int g, PrefillSeq& out) {
  const int lane = threadIdx.x & 63;
  int k = g;
  for (int s0 = 0; s0 < batch; s0 += 64) {
    const int s = s0 + lane;
    int q0 = 0, n = 0, len = 0;
    if (s < batch) {
      q0 = qo[s];
      n = max(qo[s + 1] - q0, 0);
      const int np = indptr[s + 1] - indptr[s];
      int lpl = last_len[s];
      lpl = lpl < 1 ? 1 : (lpl > page_size ? page_size : lpl);
      len = np > 0 ? (np - 1) * page_size + lpl : 0;
    }
    const int nt = (n * G + rows - 1) / rows;
    const int total = __builtin_amdgcn_readfirstlane(wave_sum_i32(nt));
    if (k >= total) {
      k -= total;
      continue;
    }
    int tile, src;
    const int nt0 = __builtin_amdgcn_readfirstlane(nt);
    if (batch <= 64 && __ballot(lane < batch && nt != nt0) == 0) {  // one number of tiles
      src = k % batch;
      tile = nt0 - 1 - k / batch;
    } else if (batch <= 64 && 4 * batch * __builtin_amdgcn_readfirstlane(wave_max_i32(nt)) <= 5 * total) {
      int r = 0;
      unsigned long long m = __ballot(nt > 0);
      while (k >= __popcll(m)) {
        k -= __popcll(m);
        m = __ballot(nt > ++r);
      }
      const int idx = __popcll(m & ((1ull << lane) - 1));
      src = __ffsll((long long)__ballot(nt > r && idx == k)) - 1;
      tile = nt - 1 - r;
    } else {
      int incl = nt;
      if (batch <= 32) {  // a few lane reads are over sooner than the six rounds through LDS
        for (int i = 0; i < batch - 1; ++i) incl += lane > i ? __builtin_amdgcn_readlane(nt, i) : 0;
      } else {
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int y = __shfl_up(incl, off, 64);
          if (lane >= off) incl += y;
        }
      }
      src = __ffsll((long long)__ballot(k >= incl - nt && k < incl)) - 1;
      tile = incl - 1 - k;
    }
    out.b = s0 + src;
    out.tile = __builtin_amdgcn_readlane(tile, src);
    out.q0 = __builtin_amdgcn_readlane(q0, src);
    out.n_new = __builtin_amdgcn_readlane(n, src);
    out.len = __builtin_amdgcn_readlane(len, src);
    return true;
  }
  return false;
}

// ---- padded output grids of the prefill entries ----------------------------------
// A wave's share of a padded grid of batch x width rows (row_bytes each, a multiple of
// 16, 16-byte aligned): of rows first, first + step, ..., those that hold no new token
// are set to zero. Sequence b's n_b = qo[b + 1] - qo[b] tokens sit at rows q_rows[qo[b]]
// .. + n_b - 1, contiguous and inside its block of `width` rows (the forward's padded
// layout). Every wave of the launch takes a share: the pads are up to half of the
// output, and one workgroup per sequence took longer to zero them (2.5 MB for 156 rows
// of 16 KB, 100 us) than the others to attend (prompts of 128 to 284 tokens, 30 us).
inline __device__ void zero_pad_rows(const int32_t* qo, const int32_t* q_rows, int width, int batch, void* out,
                                     int64_t out_row_bytes, int row_bytes, int first, int step) {
  const int lane = threadIdx.x & 63;
  const int rows = batch * width;  // < 2^31 (checked by the host)
  const u32x4 z = {0u, 0u, 0u, 0u};
  for (int64_t at_row = __builtin_amdgcn_readfirstlane(first); at_row < rows; at_row += step) {
    const int r = (int)at_row, b = r / width, c = r - b * width;
    const int q0 = qo[b], n = qo[b + 1] - q0;
    if (n > 0) {
      const int64_t at = (int64_t)q_rows[q0] - (int64_t)b * width;
      const int64_t lo = at < 0 ? 0 : at;
      if (c >= lo && c < lo + n) continue;  // a token's row
    }
    char* row = static_cast<char*>(out) + (int64_t)r * out_row_bytes;
    for (int i = 16 * lane; i < row_bytes; i += 1024) *reinterpret_cast<u32x4*>(row + i) = z;
  }
}

// ---- fp32 attention (attn_f32.hip), shared by the decode and prefill entries ----
struct AttnF32Args {
  int32_t dtype = NSLG_F32;    // element type of q, the pools and out (fp32 only)
  const float* q;
  int64_t q_stride;            // elements between query tokens
  const int32_t* qo_indptr;    // [B+1] new-token offsets; null: one token per sequence
  const int32_t* q_rows = nullptr;  // null, or row of q / out of each new token (a padded grid)
  int32_t grid_width = 0;           // rows per sequence of that grid (q_rows set)
  const float* k_pool;         // one layer, [P, ps, Hkv, D]
  const float* v_pool;
  int64_t num_pages;
  int32_t page_size;
  const int32_t* indptr;
  const int32_t* indices;
  const int32_t* last_len;
  int32_t batch;
  int32_t num_qo_heads;
  int32_t num_kv_heads;
  int32_t group;
  float scale;                 // softmax scale, natural-exponent units
  float* out;
  int64_t out_stride;
  int64_t total_q;             // query tokens (batch for decode)
  // decode: the step's new rows (null: none), sequence b's token L_b - 1, written into
  // the pool by the call; strides in elements between batch rows
  const float* k_new = nullptr;
  const float* v_new = nullptr;
  int64_t k_new_stride = 0;
  int64_t v_new_stride = 0;
  int32_t splits;              // runs of keys per row tile (1: no partials)
  void* workspace = nullptr;   // splits > 1: attention_f32_workspace bytes
  // set by attention_f32
  uint64_t* ws_tag = nullptr;  // splits > 1: the workspace's first word, set to 0 (see ws_tag in paged_prefill.hip)
  float* part_o = nullptr;     // [splits, total_q, Hq, D] partial outputs
  float* part_ml = nullptr;    // [splits, total_q, Hq, 2] running max and sum
};
// Launch on stream s (decode if qo_indptr is null, else prefill).
int attention_f32(const AttnF32Args& a, int32_t head_dim, hipStream_t s);
// Runs of keys for a decode batch of at most total_tokens keys in all, for a prefill of
// total_q rows with that workspace, and the workspace they need.
int attention_f32_decode_splits(int64_t batch, int32_t num_kv_heads, int64_t total_tokens);
int attention_f32_prefill_splits(int64_t total_q, int32_t num_qo_heads, size_t workspace_bytes, int32_t head_dim);
size_t attention_f32_workspace(int64_t total_q, int32_t num_qo_heads, int32_t head_dim, int splits);

}  // namespace nslg
