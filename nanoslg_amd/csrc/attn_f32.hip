// Paged attention of fp32 caches on the fp32 matrix instructions, for gfx950 (the
// contiguous backend of an fp32 model, kv_cache.py:227-322, whose attention is torch
// SDPA in the model's dtype). Products, sums and softmax are fp32 throughout.
//
// Query rows are packed GQA-style, row = token * G + g, so one K/V load serves all G
// query heads of a KV head. Both kernels hand 16 rows and 16 keys at a time to one wave
// (v_mfma_f32_16x16x4_f32; lane = 16 gq + r):
//   S^T[key x row] = K Q^T. The contraction's order is free, so step (i, e) takes d =
//     16 i + 4 gq + e: a lane's operands are then whole float4s of its key's (A) and its
//     row's (B) elements at 16 i + 4 gq, and S leaves keys 4 gq + j of row r in a lane.
//   online softmax per row in natural exponents: 4 values per lane, then across gq.
//   O^T[d x row] += V^T P^T. Step j takes keys 4 gq + j: B is exactly the S layout, A
//     the lane's float4s of token 4 gq + j at d = 64 c + 4 r (whole 256-byte pieces of a
//     row per load); output tile (c, e) holds d = 64 c + 4 x + e at its row x.
//
// decode_f32_kernel: one token per sequence. A workgroup takes one (sequence, KV head,
//   run of keys); its waves take the run's 16-key tiles in turn straight from memory, the
//   next tile's loads in flight during the present one's products, and combine through
//   LDS. The step's new K/V row is written by the wave that reads it. 16 matrix columns
//   for G rows leaves them partly empty, but a tile's 2 x D / 4 products (2048 cycles of
//   a SIMD at D = 128) pass at 3x the memory rate. One CU draws ~2x its share of the
//   memory rate, so small batches are cut down to 64 keys a workgroup: 4 waves, one tile
//   each. Measured at 32/8 heads x 128, with the merge, against the VALU kernel before:
//   one sequence of 512 tokens 70 -> 9.5 us, of 4000 98 -> 13 (of 5 us merge), 8 of 4000
//   149 -> 49 (5.4 TB/s).
// prefill_f32_kernel: 64 rows (4 waves x 16) of one (sequence, KV head), K/V tiles staged
//   in LDS once for all four. Bound by the matrix instructions (a tile of 32 keys is 4096
//   cycles of a SIMD; two waves on it take ~10000 for both): 8 x 512 tokens over 512 keys
//   1808 -> 500 us (103 of the 153 TFLOP/s that a large fp32 product reaches), one of 512
//   from zero 145 -> 59, 64 over 4000 631 -> 63; 8 tokens, all latency, 8.9 and 9.3.
// Both cut their keys into runs where there are too few workgroups; the runs' rows are
// combined by merge_f32_kernel.
//
// Causality is bottom-right aligned: token t of a sequence with L keys and n new
// tokens sees keys j <= L - n + t (FlashInfer's causal prefill with a KV prefix,
// kv_cache.py:627-632, and the contiguous path's mask, kv_cache.py:218-220).
#include "nslg_common.h"

#include <math.h>

namespace nslg {
namespace {

constexpr int kMaxSplitsF = 64;
constexpr int kRowsP = 64;               // query rows per prefill workgroup, 16 per wave
constexpr int kRunP = 128;               // prefill: keys per run are a multiple of this

constexpr int kWavesD = 4;               // decode: waves per workgroup, a 16-key tile each at a time
constexpr int kRunD = 16 * kWavesD;      // decode: keys per run are a multiple of this

// Row of q / out holding new token t (-1: a grid row out of range, not read or written).
__device__ inline int64_t f32_grid_row(const AttnF32Args& p, int t) {
  if (!p.q_rows) return t;
  const int64_t r = p.q_rows[t];
  return r >= 0 && r < (int64_t)p.batch * p.grid_width ? r : -1;
}

__device__ inline int kv_len_f32(const AttnF32Args& p, int s) {
  const int np = p.indptr[s + 1] - p.indptr[s];
  if (np <= 0) return 0;
  int lpl = p.last_len[s];
  lpl = lpl < 1 ? 1 : (lpl > p.page_size ? p.page_size : lpl);
  return (np - 1) * p.page_size + lpl;
}

__device__ inline f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Online softmax state of a wave's 16 rows: the running max of row r in all its lanes
// (gq = 0..3), the lane's own share of the row's sum, O^T as NT = D / 16 output tiles.
template <int D>
struct RowsF32 {
  static constexpr int NT = D / 16;
  float m, l;
  f32x4 o[NT];

  __device__ void clear() {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // scores of kTiles 16-key tiles (scaled, masked with -inf) -> probabilities in place
  template <int kTiles>
  __device__ void softmax(f32x4 (&s)[kTiles]) {
    float t = -INFINITY;
#pragma unroll
    for (int k = 0; k < kTiles; ++k) t = fmaxf(t, fmaxf(fmaxf(s[k][0], s[k][1]), fmaxf(s[k][2], s[k][3])));
    t = rows_max(t);
    if (__ballot(t > m)) {
      const float m_new = fmaxf(m, t);
      const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
      l *= alpha;
#pragma unroll
      for (int n = 0; n < NT; ++n) o[n] *= alpha;
      m = m_new;
    }
#pragma unroll
    for (int k = 0; k < kTiles; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[k][j] = s[k][j] == -INFINITY ? 0.f : expf(s[k][j] - m);
        l += s[k][j];
      }
  }
};

// Query operands of the wave's row r (zeros past the rows): float4 at 16 i + 4 gq.
template <int D>
__device__ inline void load_q_f32(const float* row, bool ok, int gq, f32x4 (&q)[D / 16]) {
#pragma unroll
  for (int i = 0; i < D / 16; ++i)
    q[i] = ok ? *reinterpret_cast<const f32x4*>(row + 16 * i + 4 * gq) : f32x4{0.f, 0.f, 0.f, 0.f};
}

// S^T of one tile: two chains, so that a product need not wait for the one before it.
template <int D>
__device__ inline f32x4 scores_f32(const f32x4 (&k)[D / 16], const f32x4 (&q)[D / 16]) {
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    a = mfma_f32(k[i][0], q[i][0], a);
    b = mfma_f32(k[i][1], q[i][1], b);
    a = mfma_f32(k[i][2], q[i][2], a);
    b = mfma_f32(k[i][3], q[i][3], b);
  }
  return a + b;
}

// A run's rows: out (one run per call) or the partials of run `split`.
template <int D>
__device__ inline void store_piece(const AttnF32Args& p, int64_t prow, int64_t orow, int split, int64_t rows, int d,
                                   f32x4 v) {
  if (p.splits > 1)
    *reinterpret_cast<f32x4*>(p.part_o + (split * rows + prow) * D + d) = v;
  else if (orow >= 0)
    *reinterpret_cast<f32x4*>(p.out + orow * p.out_stride + (prow % p.num_qo_heads) * D + d) = v;
}

// ---- decode ---------------------------------------------------------------------------

template <int D>
struct TileF32 {
  f32x4 k[D / 16];      // key r at 16 i + 4 gq
  f32x4 v[4][D / 64];   // token 4 gq + j at 64 c + 4 r
};

template <int D>
__global__ void __launch_bounds__(64 * kWavesD) decode_f32_kernel(AttnF32Args p) {
  constexpr int W = kWavesD;
  constexpr int NT = D / 16;
  constexpr int kPitch = D + 4;
  __shared__ __attribute__((aligned(16))) float o_lds[W][16 * kPitch];
  __shared__ float ml_lds[W][16][2];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, gq = lane >> 4;
  const int h = blockIdx.x % p.num_kv_heads;
  const int b = blockIdx.x / p.num_kv_heads;
  const int split = blockIdx.y;
  const int G = p.group, ps = p.page_size;
  const int L = kv_len_f32(p, b);
  const int piece = ((L + p.splits - 1) / p.splits + kRunD - 1) / kRunD * kRunD;
  const int kv_begin = min(L, split * piece);
  const int kv_end = min(L, kv_begin + piece);
  if (p.ws_tag && blockIdx.x == 0 && split == 0 && threadIdx.x == 0) *p.ws_tag = 0;
  const int64_t rows = (int64_t)p.batch * p.num_qo_heads;
  const int64_t prow0 = (int64_t)b * p.num_qo_heads + h * G;
  if (kv_begin >= kv_end && p.splits > 1) {  // uniform: no key, no share in the merge
    if ((int)threadIdx.x < G) *reinterpret_cast<float2*>(p.part_ml + (split * rows + prow0 + threadIdx.x) * 2) = float2{-INFINITY, 0.f};
    return;
  }
  const int32_t* idx = p.indices + p.indptr[b];
  const int64_t row_elems = (int64_t)p.num_kv_heads * D;
  const int n_tiles = (kv_end - kv_begin + 15) / 16;

  f32x4 q[NT];
  load_q_f32<D>(p.q + b * p.q_stride + (int64_t)(h * G + r) * D, r < G, gq, q);

  // The step's new row: token L - 1, written by the wave whose tile holds it (and which
  // then reads it back: a wave's loads follow its own stores), not at all for a page id
  // outside the pool.
  if (p.k_new && kv_end == L && n_tiles > 0 && (n_tiles - 1) % W == wave) {
    const int pid = idx[(L - 1) / ps];
    if (pid >= 0 && (int64_t)pid < p.num_pages) {
      const int64_t off = ((int64_t)pid * ps + (L - 1) % ps) * row_elems + (int64_t)h * D;
      const float* ks = p.k_new + b * p.k_new_stride + (int64_t)h * D;
      const float* vs = p.v_new + b * p.v_new_stride + (int64_t)h * D;
#pragma unroll
      for (int c = 0; c < D / 64; ++c) {
        const_cast<float*>(p.k_pool)[off + 64 * c + lane] = ks[64 * c + lane];
        const_cast<float*>(p.v_pool)[off + 64 * c + lane] = vs[64 * c + lane];
      }
    }
  }

  // Tile t of the run: keys kv_begin + 16 t + 0..15, those past the run repeat its last
  // (a tile past the run reads one row). A tile inside one page (all of them where pages
  // are whole slots or multiples of 16 tokens) takes one page id for the wave. The loads
  // are issued on every path, so that the waits count exactly and a tile's products wait
  // for its own loads only, not for the next tile's.
  const int last = kv_end - 1;
  auto page_of = [&](int t) { return idx[min(kv_begin + 16 * t, last) / ps]; };
  auto load = [&](int t, int pid0, TileF32<D>& x) {
    const int k0 = min(kv_begin + 16 * t, last);
    const int left = min(15, last - k0);
    const int s0 = k0 % ps;
    int64_t krow, vrow[4];
    if (s0 + left < ps) {
      const int64_t base = (int64_t)(pid0 < 0 || (int64_t)pid0 >= p.num_pages ? 0 : pid0) * ps + s0;
      krow = base + min(r, left);
#pragma unroll
      for (int j = 0; j < 4; ++j) vrow[j] = base + min(4 * gq + j, left);
    } else {
      auto row = [&](int key) {
        int pid = idx[key / ps];
        pid = pid < 0 || (int64_t)pid >= p.num_pages ? 0 : pid;
        return (int64_t)pid * ps + key % ps;
      };
      krow = row(k0 + min(r, left));
#pragma unroll
      for (int j = 0; j < 4; ++j) vrow[j] = row(k0 + min(4 * gq + j, left));
    }
    const float* kr = p.k_pool + krow * row_elems + (int64_t)h * D + 4 * gq;
#pragma unroll
    for (int i = 0; i < NT; ++i) x.k[i] = *reinterpret_cast<const f32x4*>(kr + 16 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float* vr = p.v_pool + vrow[j] * row_elems + (int64_t)h * D + 4 * r;
#pragma unroll
      for (int c = 0; c < D / 64; ++c) x.v[j][c] = *reinterpret_cast<const f32x4*>(vr + 64 * c);
    }
  };
  RowsF32<D> st;
  st.clear();
  auto compute = [&](int t, const TileF32<D>& x) {
    f32x4 s[1] = {scores_f32<D>(x.k, q)};
#pragma unroll
    for (int j = 0; j < 4; ++j) s[0][j] = kv_begin + 16 * t + 4 * gq + j < kv_end ? s[0][j] * p.scale : -INFINITY;
    st.template softmax<1>(s);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int n = 0; n < NT; ++n) st.o[n] = mfma_f32(x.v[j][n >> 2][n & 3], s[0][j], st.o[n]);
  };

  if (wave < n_tiles) {
    TileF32<D> x0, x1;
    load(wave, page_of(wave), x0);
    if (n_tiles <= W) compute(wave, x0);
    int pid = page_of(wave + W);
    for (int t = wave; n_tiles > W && t < n_tiles; t += 2 * W) {
      load(t + W, pid, x1);
      pid = page_of(t + 2 * W);
      compute(t, x0);
      load(t + 2 * W, pid, x0);
      pid = page_of(t + 3 * W);
      if (t + W < n_tiles) compute(t + W, x1);
    }
  }

  // combine the waves: every row's max and sum, then O scaled to the common max
  const float l = rows_sum(st.l);
  if (gq == 0) {
    ml_lds[wave][r][0] = st.m;
    ml_lds[wave][r][1] = l;
  }
  if (r < G) {
#pragma unroll
    for (int c = 0; c < D / 64; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(&o_lds[wave][r * kPitch + 64 * c + 4 * (4 * gq + j)]) =
            f32x4{st.o[4 * c][j], st.o[4 * c + 1][j], st.o[4 * c + 2][j], st.o[4 * c + 3][j]};
  }
  __syncthreads();
  for (int e = threadIdx.x; e < G * (D / 4); e += 64 * W) {
    const int row = e / (D / 4), d = 4 * (e % (D / 4));
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) m = fmaxf(m, ml_lds[w][row][0]);
    float sum = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float lw = ml_lds[w][row][1];
      const float f = lw == 0.f ? 0.f : expf(ml_lds[w][row][0] - m);  // 0: a wave without keys
      const f32x4 ow = *reinterpret_cast<const f32x4*>(&o_lds[w][row * kPitch + d]);
      sum = fmaf(f, lw, sum);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(f, ow[i], acc[i]);
    }
    if (p.splits == 1) {
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] *= inv;
    } else if (d == 0) {
      *reinterpret_cast<float2*>(p.part_ml + (split * rows + prow0 + row) * 2) = float2{m, sum};
    }
    store_piece<D>(p, prow0 + row, b, split, rows, d, acc);
  }
}

// ---- prefill --------------------------------------------------------------------------

template <int D, int kGroups>
__global__ void __launch_bounds__(256 * kGroups) prefill_f32_kernel(AttnF32Args p) {
  constexpr int NT = D / 16;
  constexpr int kWaveKeys = D == 256 ? 16 : 32;  // keys per wave and tile
  constexpr int kKeys = kGroups * kWaveKeys;     // keys per LDS tile
  constexpr int kThreads = 256 * kGroups;
  // +4 floats: the 16-byte operand reads of 8 lanes fall on distinct banks
  constexpr int kPitch = D + 4;
  constexpr int kVecs = D / 4;                          // float4s per row
  constexpr int kPer = kKeys * kVecs / kThreads;        // float4s of K per thread and tile
  __shared__ __attribute__((aligned(16))) float kv_lds[2 * kKeys * kPitch];
  __shared__ float2 ml_lds[kGroups == 2 ? 256 : 1];
  float* k_lds = kv_lds;
  float* v_lds = kv_lds + kKeys * kPitch;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);   // rows 16 wave .. + 15 of the tile
  const int group_keys = kWaveKeys * __builtin_amdgcn_readfirstlane(tid >> 8);  // the wave's keys of an LDS tile
  const int r = lane & 15, gq = lane >> 4;
  // work item: the tile's slot (longest first, empty ones last), then (run, KV head) in turn
  if (p.q_rows)
    zero_pad_rows(p.qo_indptr, p.q_rows, p.grid_width, p.batch, p.out, p.out_stride * 4, p.num_qo_heads * D * 4,
                  blockIdx.x * (kThreads / 64) + (tid >> 6), gridDim.x * (kThreads / 64));
  if (p.ws_tag && blockIdx.x == 0 && tid == 0) *p.ws_tag = 0;
  const int runs = p.num_kv_heads * p.splits;
  const int run = blockIdx.x % runs;
  const int split = run / p.num_kv_heads, h = run - split * p.num_kv_heads;  // a head's runs on one XCD
  PrefillSeq sq;
  if (!locate_row_tile(p.qo_indptr, p.indptr, p.last_len, p.page_size, p.batch, p.group, kRowsP, blockIdx.x / runs, sq))
    return;  // uniform over the workgroup
  const int b = sq.b, tile = sq.tile, q0 = sq.q0, n_new = sq.n_new, L = sq.len;
  const int G = p.group, ps = p.page_size;
  const int start = L - n_new > 0 ? L - n_new : 0;
  const int nrows = n_new * G;
  const int last_row = min(tile * kRowsP + kRowsP, nrows) - 1;
  const int kv_all = min(L, start + last_row / G + 1);
  const int piece = ((kv_all + p.splits - 1) / p.splits + kRunP - 1) / kRunP * kRunP;
  const int kv_begin = min(kv_all, split * piece);
  const int kv_end = min(kv_all, kv_begin + piece);
  const int64_t rows = p.total_q * p.num_qo_heads;
  // the lane's row: 16 rows per wave, row r of them in the lanes of column r
  const int row = tile * kRowsP + 16 * wave + r;
  const bool row_ok = row < nrows && q0 + row / G < p.total_q;
  const int t_row = row_ok ? row / G : 0;
  const int64_t prow = (int64_t)(q0 + t_row) * p.num_qo_heads + h * G + (row_ok ? row % G : 0);
  if (kv_begin >= kv_end && p.splits > 1) {  // uniform: no key, no share in the merge
    if (row_ok && gq == 0) *reinterpret_cast<float2*>(p.part_ml + (split * rows + prow) * 2) = float2{-INFINITY, 0.f};
    return;
  }
  const int pos = start + t_row;  // the row sees keys <= pos
  // keys below wave_end are seen by some row of the wave, those up to wave_all by all
  const int w_last = min(tile * kRowsP + 16 * wave + 16, nrows) - 1;
  const int wave_end = tile * kRowsP + 16 * wave < nrows ? min(kv_end, start + w_last / G + 1) : 0;
  const int wave_all = min(kv_end, start + (tile * kRowsP + 16 * wave) / G + 1);
  const int64_t orow = row_ok ? f32_grid_row(p, q0 + t_row) : -1;
  const int32_t* idx = p.indices + p.indptr[b];
  const int64_t row_elems = (int64_t)p.num_kv_heads * D;

  f32x4 q[NT];
  load_q_f32<D>(p.q + (orow >= 0 ? orow : 0) * p.q_stride + (int64_t)(h * G + (row_ok ? row % G : 0)) * D, orow >= 0,
                gq, q);

  // Thread tid moves float4 tid % kVecs of keys tid / kVecs + (kThreads / kVecs) i of a
  // tile: page ids a tile ahead of the rows, rows a tile ahead of their products. A tile
  // inside one page (whole slots, pages of many tokens) takes one division and one page
  // id for all its keys.
  const int f_c = 4 * (tid % kVecs), f_key = tid / kVecs;
  constexpr int kStep = kThreads / kVecs;
  const int last = kv_end - 1;
  int pid[kPer];
  f32x4 kreg[kPer], vreg[kPer];
  auto one_page = [&](int key0) { return min(key0, last) % ps + min(kKeys - 1, max(last - key0, 0)) < ps; };  // uniform
  auto fetch_pages = [&](int key0) {
    if (one_page(key0)) {
      const int page = idx[min(key0, last) / ps];
#pragma unroll
      for (int i = 0; i < kPer; ++i) pid[i] = page;
    } else {
#pragma unroll
      for (int i = 0; i < kPer; ++i) pid[i] = idx[min(key0 + f_key + kStep * i, last) / ps];
    }
  };
  auto fetch_rows = [&](int key0) {
    int slot[kPer];
    if (one_page(key0)) {
      const int slot0 = key0 % ps;
#pragma unroll
      for (int i = 0; i < kPer; ++i) slot[i] = slot0 + min(f_key + kStep * i, last - key0);
    } else {
#pragma unroll
      for (int i = 0; i < kPer; ++i) slot[i] = min(key0 + f_key + kStep * i, last) % ps;
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int64_t page = pid[i] < 0 || (int64_t)pid[i] >= p.num_pages ? 0 : pid[i];
      const int64_t off = (page * ps + slot[i]) * row_elems + (int64_t)h * D + f_c;
      kreg[i] = *reinterpret_cast<const f32x4*>(p.k_pool + off);
      vreg[i] = *reinterpret_cast<const f32x4*>(p.v_pool + off);
    }
  };

  RowsF32<D> st;
  st.clear();
  if (kv_begin < kv_end) {
    fetch_pages(kv_begin);
    fetch_rows(kv_begin);
    if (kv_begin + kKeys < kv_end) fetch_pages(kv_begin + kKeys);
  }
  // Q is waited for here: pending at the loop's entry, its wait would sit in the loop and
  // hold for the next tile's rows too, every tile.
#pragma unroll
  for (int i = 0; i < NT; ++i) asm volatile("" : "+v"(q[i]));
  for (int key0 = kv_begin; key0 < kv_end; key0 += kKeys) {
    __syncthreads();  // the tile before is read
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int key = f_key + kStep * i;
      *reinterpret_cast<f32x4*>(&k_lds[key * kPitch + f_c]) = kreg[i];
      *reinterpret_cast<f32x4*>(&v_lds[key * kPitch + f_c]) = vreg[i];
    }
    __syncthreads();
    if (key0 + kKeys < kv_end) {
      fetch_rows(key0 + kKeys);
      fetch_pages(key0 + 2 * kKeys);
    }
    const int wkey0 = key0 + group_keys;
    if (wkey0 >= wave_end) continue;  // uniform over the wave
    f32x4 s[kWaveKeys / 16];
    // the wave's last tile may need one of its two 16-key halves only (16 tokens 11.0 ->
    // 9.7 us, prompts of 300 to 600 111 -> 92 with the longest tiles first)
    auto seen = [&](int k) { return k == 0 || wkey0 + 16 * k < wave_end; };  // uniform over the wave
#pragma unroll
    for (int k = 0; k < kWaveKeys / 16; ++k) {
      s[k] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (!seen(k)) break;
      f32x4 kt[NT];
#pragma unroll
      for (int i = 0; i < NT; ++i)
        kt[i] = *reinterpret_cast<const f32x4*>(&k_lds[(group_keys + 16 * k + r) * kPitch + 16 * i + 4 * gq]);
      s[k] = scores_f32<D>(kt, q) * p.scale;
    }
    if (wkey0 + kWaveKeys > wave_all) {
#pragma unroll
      for (int k = 0; k < kWaveKeys / 16; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int key = wkey0 + 16 * k + 4 * gq + j;
          if (!(key < kv_end && key <= pos)) s[k][j] = -INFINITY;
        }
    }
    st.template softmax<kWaveKeys / 16>(s);
#pragma unroll
    for (int k = 0; k < kWaveKeys / 16; ++k) {
      if (!seen(k)) break;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < D / 64; ++c) {
          const f32x4 v =
              *reinterpret_cast<const f32x4*>(&v_lds[(group_keys + 16 * k + 4 * gq + j) * kPitch + 64 * c + 4 * r]);
#pragma unroll
          for (int e = 0; e < 4; ++e) st.o[4 * c + e] = mfma_f32(v[e], s[k][j], st.o[4 * c + e]);
        }
    }
  }

  float l = rows_sum(st.l);
  if constexpr (kGroups == 2) {
    // the second group's rows to the first, lane to lane, through the tiles' LDS
    __syncthreads();
    f32x4* o_buf = reinterpret_cast<f32x4*>(kv_lds) + 64 * NT * wave + lane;
    if (group_keys) {
#pragma unroll
      for (int n = 0; n < NT; ++n) o_buf[64 * n] = st.o[n];
      ml_lds[64 * wave + lane] = float2{st.m, l};
    }
    __syncthreads();
    if (group_keys) return;
    const float2 ml = ml_lds[64 * wave + lane];
    const float m = fmaxf(st.m, ml.x);
    const float f0 = l == 0.f ? 0.f : expf(st.m - m);  // 0: no key of the group seen
    const float f1 = ml.y == 0.f ? 0.f : expf(ml.x - m);
    l = fmaf(f0, l, f1 * ml.y);
    st.m = m;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const f32x4 o1 = o_buf[64 * n];
#pragma unroll
      for (int e = 0; e < 4; ++e) st.o[n][e] = fmaf(f0, st.o[n][e], f1 * o1[e]);
    }
  }
  if (!row_ok) return;
  float f = 1.f;
  if (p.splits == 1)
    f = l > 0.f ? 1.f / l : 0.f;
  else if (gq == 0)
    *reinterpret_cast<float2*>(p.part_ml + (split * rows + prow) * 2) = float2{st.m, l};
#pragma unroll
  for (int c = 0; c < D / 64; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      store_piece<D>(p, prow, orow, split, rows, 64 * c + 4 * (4 * gq + j),
                     f32x4{st.o[4 * c][j] * f, st.o[4 * c + 1][j] * f, st.o[4 * c + 2][j] * f, st.o[4 * c + 3][j] * f});
}

// Log-sum-exp merge of the runs of each (query token, query head) row: D / 4 lanes per
// row, one float4 each, and kParts such groups of lanes, 16 runs each (one after the
// other, 63 runs took 9.7 us). A run without a key of the row has sum 0 and is passed
// over (its rows may be unwritten); one whose scores are all NaN has max -inf and sum NaN,
// and its weight is NaN.
template <int D, int kParts>
__global__ void __launch_bounds__(kParts * (D / 4) < 256 ? 256 : kParts * (D / 4)) merge_f32_kernel(AttnF32Args p) {
  constexpr int kLanes = D / 4;
  constexpr int kRows = kParts * kLanes < 256 ? 256 / (kParts * kLanes) : 1;  // rows per workgroup
  __shared__ f32x4 acc_lds[kParts > 1 ? kRows * (kParts - 1) * kLanes : 1];
  const int64_t rows = p.total_q * p.num_qo_heads;
  const int part = threadIdx.x / kLanes % kParts;
  const int wg_row = threadIdx.x / (kLanes * kParts);
  const int64_t row0 = (int64_t)blockIdx.x * kRows + wg_row;
  const int64_t prow = row0 < rows ? row0 : rows - 1;  // (rows past the last repeat it, unwritten)
  const int t = (int)(prow / p.num_qo_heads);
  // (max, sum) of run 16 i + lane % 16 in each 16-lane group
  const int sl = threadIdx.x & 15;
  float2 ml[kParts];
#pragma unroll
  for (int i = 0; i < kParts; ++i) {
    const int s = min(16 * i + sl, p.splits - 1);
    ml[i] = *reinterpret_cast<const float2*>(p.part_ml + (s * rows + prow) * 2);
    if (16 * i + sl >= p.splits) ml[i] = float2{-INFINITY, 0.f};
  }
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < kParts; ++i) m = fmaxf(m, ml[i].x);
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 16));
  float f = -1.f, l = 0.f;  // the weight of the part's run sl (-1: no key); the row's sum
#pragma unroll
  for (int i = 0; i < kParts; ++i) {
    if (ml[i].y == 0.f) continue;
    const float w = ml[i].y != ml[i].y ? ml[i].y : expf(ml[i].x - m);
    if (i == part) f = w;
    l = fmaf(w, ml[i].y, l);
  }
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) l += __shfl_xor(l, off, 16);
  const int d = 4 * (threadIdx.x % kLanes);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int s_end = min(p.splits, 16 * part + 16);
  for (int s0 = 16 * part; s0 < s_end; s0 += 8) {
    f32x4 o[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      o[u] = *reinterpret_cast<const f32x4*>(p.part_o + (min(s0 + u, s_end - 1) * rows + prow) * D + d);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float fs = s0 + u < s_end ? __shfl(f, (s0 + u) & 15, 16) : -1.f;
      if (fs < 0.f) continue;  // a run without keys left no rows
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(fs, o[u][e], acc[e]);
    }
  }
  if constexpr (kParts > 1) {
    f32x4* mine = acc_lds + wg_row * (kParts - 1) * kLanes + threadIdx.x % kLanes;
    if (part) mine[(part - 1) * kLanes] = acc;
    __syncthreads();
    if (part) return;
#pragma unroll
    for (int i = 0; i < kParts - 1; ++i) acc += mine[i * kLanes];
  }
  if (row0 >= rows) return;
  // (a row of no sequence has no runs: past the last's, or before the first's in a batch
  // that is part of a larger one)
  if (p.qo_indptr && (t < p.qo_indptr[0] || t >= p.qo_indptr[p.batch])) return;
  const int64_t orow = f32_grid_row(p, t);
  if (orow < 0) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  *reinterpret_cast<f32x4*>(p.out + orow * p.out_stride + (prow - (int64_t)t * p.num_qo_heads) * D + d) =
      f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
}

template <int D, int kParts>
void launch_merge_f32(const AttnF32Args& p, hipStream_t s) {
  constexpr int kThreads = kParts * (D / 4) < 256 ? 256 : kParts * (D / 4);
  constexpr int kRows = kThreads / (kParts * (D / 4));
  const int64_t rows = p.total_q * p.num_qo_heads;
  merge_f32_kernel<D, kParts><<<dim3((unsigned)((rows + kRows - 1) / kRows)), kThreads, 0, s>>>(p);
}

template <int D>
int launch_f32(const AttnF32Args& p, dim3 grid, hipStream_t s) {
  if (p.qo_indptr) {
    // Two groups of waves on each row tile, half of an LDS tile's keys each, where one group
    // leaves SIMDs idle: fresh prompts of few tiles (4 x 128 tokens 25.5 -> 24.0 us, 4 x
    // 100..512 47.6 -> 42.4; D = 64, 4 x 512, 105 -> 84). Not for calls of many workgroups
    // (8 x 512 over 512: 542 us, with two groups 646), calls cut into runs (512 from zero, in
    // a call given a workspace, 57.3 and 63.5), nor a few short tiles (16 tokens 10.9 and 12.5).
    if (p.splits == 1 && grid.x > 32 && grid.x <= (D == 64 ? 2048u : 1024u))
      prefill_f32_kernel<D, 2><<<grid, 512, 0, s>>>(p);
    else
      prefill_f32_kernel<D, 1><<<grid, 256, 0, s>>>(p);
  } else {
    decode_f32_kernel<D><<<grid, 64 * kWavesD, 0, s>>>(p);
  }
  const int rc = check_launch("attention_f32");
  if (rc || p.splits == 1) return rc;
  if (p.splits > 16)
    launch_merge_f32<D, 4>(p, s);
  else
    launch_merge_f32<D, 1>(p, s);
  return check_launch("attention_f32_merge");
}

}  // namespace

int attention_f32_decode_splits(int64_t batch, int32_t num_kv_heads, int64_t total_tokens) {
  if (batch <= 0 || num_kv_heads <= 0) return 1;
  const int64_t by_keys = total_tokens / batch / kRunD;
  const int64_t by_wgs = 512 / (batch * num_kv_heads);
  const int64_t s = by_keys < by_wgs ? by_keys : by_wgs;
  return (int)(s < 1 ? 1 : (s > kMaxSplitsF ? kMaxSplitsF : s));
}

int attention_f32_prefill_splits(int64_t total_q, int32_t num_qo_heads, size_t workspace_bytes, int32_t head_dim) {
  const int64_t rows = total_q * num_qo_heads;
  if (rows <= 0) return 1;
  int64_t s = 512 / ((rows + kRowsP - 1) / kRowsP);
  s = s > kMaxSplitsF ? kMaxSplitsF : s;
  while (s > 1 && attention_f32_workspace(total_q, num_qo_heads, head_dim, (int)s) > workspace_bytes) --s;
  return (int)(s < 1 ? 1 : s);
}

size_t attention_f32_workspace(int64_t total_q, int32_t num_qo_heads, int32_t head_dim, int splits) {
  if (splits <= 1) return 256;
  return (size_t)total_q * num_qo_heads * splits * (head_dim + 2) * sizeof(float) + 512;
}

int attention_f32(const AttnF32Args& a, int32_t head_dim, hipStream_t s) {
  if (a.group > 16) return fail(NSLG_EUNSUPPORTED, "attention_f32: GQA group %d", a.group);
  if (a.dtype != NSLG_F32)
    return fail(NSLG_EUNSUPPORTED, "attention_f32: dtype %d (16-bit pools run on the MFMA kernels)", a.dtype);
  // 16-byte rows: the kernels' vector accesses and the pad-row zeroing (16-byte stores)
  if (((uintptr_t)a.q | (uintptr_t)a.k_pool | (uintptr_t)a.v_pool | (uintptr_t)a.out) & 15 ||
      (a.q_stride * 4) % 16 || (a.out_stride * 4) % 16)
    return fail(NSLG_EINVAL, "attention_f32: q/pool/out must be 16-byte aligned with row strides of 16 bytes");
  if (a.num_pages * (int64_t)a.page_size >= ((int64_t)1 << 31))
    return fail(NSLG_EUNSUPPORTED, "attention_f32: pool has >= 2^31 token slots");
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return fail(NSLG_EUNSUPPORTED, "attention_f32: head_dim %d (64, 128 or 256)", head_dim);
  if (a.splits < 1 || a.splits > kMaxSplitsF) return fail(NSLG_EINVAL, "attention_f32: %d splits", a.splits);
  if (a.splits > 1 && !a.workspace) return fail(NSLG_EWORKSPACE, "attention_f32: no workspace");
  if (a.q_rows && (!a.qo_indptr || a.grid_width < 1))
    return fail(NSLG_EINVAL, "attention_f32: a padded grid needs ragged rows and a width");
  AttnF32Args p = a;
  if (a.splits > 1) {  // the first word, part_o [splits, rows, D], part_ml [splits, rows, 2]
    p.ws_tag = (uint64_t*)(((uintptr_t)a.workspace + 255) / 256 * 256);
    p.part_o = (float*)(p.ws_tag + 32);
    p.part_ml = p.part_o + a.total_q * a.num_qo_heads * a.splits * head_dim;
  }
  dim3 grid;
  if (a.qo_indptr) {
    // row-tile slots: an upper bound over the batch (every sequence may end in a partial tile)
    const int64_t tiles = (a.total_q * a.group + kRowsP - 1) / kRowsP + a.batch;
    const int64_t wgs = tiles * a.num_kv_heads * a.splits;
    if (wgs > 0x7fffffff / 8) return fail(NSLG_EUNSUPPORTED, "attention_f32: too many rows");
    grid = dim3((unsigned)wgs);
  } else {
    const int64_t wgs = (int64_t)a.batch * a.num_kv_heads;
    if (wgs > 0x7fffffff) return fail(NSLG_EUNSUPPORTED, "attention_f32: too many rows");
    grid = dim3((unsigned)wgs, (unsigned)a.splits);
  }
  if (a.splits > 1 && a.total_q * a.num_qo_heads >= 0x7fffffff)
    return fail(NSLG_EUNSUPPORTED, "attention_f32: too many rows");
  switch (head_dim) {
    case 64: return launch_f32<64>(p, grid, s);
    case 128: return launch_f32<128>(p, grid, s);
    default: return launch_f32<256>(p, grid, s);
  }
}

}  // namespace nslg
