// Windowed causal attention over a paged cache whose scores are soft-capped and carry a logarithmic distance
// penalty, with key and value heads of different sizes, and the preparation of its operands.
//
//   s_ij = scale (q_i . k_j);   s <- cap tanh(s / cap)  (cap > 0);   s <- s - r1_h ln(1 + r2_h (i - j))  (r1 given)
//   o_i  = sum_j softmax_j(s_ij) v_j     over  max(0, i - window + 1) <= j <= i   (window 0: every earlier key)
//
// Two further options: `chunk` > 0 lets row i see only the keys of its own chunk, floor(i / chunk) chunk <= j <= i
// (chunks are counted from position 0 of the request); `sink` [heads] adds exp(sink_h) to the softmax's denominator,
// a term without key or value.  `wide_norm_store` prepares the operands of an attention whose q and k are RMS-normed
// over the whole projection (all heads at once) and whose values may be mixed with another layer's.
//
// q head h reads kv head h / (nq / nkv).  Keys lie in pages [page, nkv, slot, Dk], values d-major
// [page, nkv, Dv, slot].  Scores, the cap, the penalty, probabilities and sums are 32-bit.
//
// `qkv_norm_store`: per-head RMS norm of q and k (one weight of Dk for all heads, eps inside the root), the
// query temperature q <- q (1 + coef ln(floor((p + 1) / every) + 1)) at position p, and the write of k and v
// into the request's pages.  `attn_softcap_simt`: one wave a (row, q head), keys in tiles of 64 aligned to
// the absolute key index and walked in ascending order, so that a row's arithmetic depends on its position
// and window only: the true 32-bit path, and the plain counterpart of the matrix-core kernel below.
#include "common.h"

namespace arle {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kCapMaxD = 1024;   // the widest head: a latent attention's keys are its latent and its rotated part together

// One wave a (row, head of q, k or v).  T: the element type of q, k, v and the pages; the loads of a head are typed and
// unconditional (an element past the head's size reads the head's last one and is dropped).
template <typename T>
__global__ __launch_bounds__(kWave) void qkv_norm_store_kernel(
    T* __restrict__ q, long long q_stride, const T* __restrict__ k, long long k_stride, const T* __restrict__ v,
    long long v_stride, const void* __restrict__ q_weight, const void* __restrict__ k_weight, int w_dtype, float eps,
    float temp_coef, int temp_every, const int* __restrict__ positions, const int* __restrict__ slot_of_token,
    const int* __restrict__ block_table, int table_stride, T* __restrict__ k_pages, T* __restrict__ v_pages, int nq,
    int nkv, int Dk, int Dv, int page_size) {
  const int64_t t = blockIdx.x;
  const int y = blockIdx.y, lane = threadIdx.x;
  const int pos = positions[t];
  if (y < nq + nkv) {
    const bool is_q = y < nq;
    const int g = is_q ? y : y - nq;
    const T* src = is_q ? q + t * q_stride + g * Dk : k + t * k_stride + g * Dk;
    const void* weight = is_q ? q_weight : k_weight;
    float x[kCapMaxD / kWave], w[kCapMaxD / kWave];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < kCapMaxD / kWave; ++j) {
      const int d = lane + j * kWave;
      if (j * kWave < Dk) {
        x[j] = to_float(src[min(d, Dk - 1)]);
        w[j] = weight ? load_as_float(weight, w_dtype, min(d, Dk - 1)) : 1.0f;
        if (d < Dk) ss = fmaf(x[j], x[j], ss);
      }
    }
    float f = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(Dk) + eps);
    T* dst;
    if (is_q) {
      if (temp_coef != 0.f) f *= 1.0f + temp_coef * logf(static_cast<float>((pos + 1) / temp_every + 1));
      dst = q + t * q_stride + g * Dk;
    } else {
      const int page = block_table[static_cast<int64_t>(slot_of_token[t]) * table_stride + pos / page_size];
      dst = k_pages + ((static_cast<int64_t>(page) * nkv + g) * page_size + pos % page_size) * Dk;
    }
#pragma unroll
    for (int j = 0; j < kCapMaxD / kWave; ++j) {
      const int d = lane + j * kWave;
      if (j * kWave < Dk && d < Dk) dst[d] = from_float<T>(x[j] * f * w[j]);
    }
    return;
  }
  const int page = block_table[static_cast<int64_t>(slot_of_token[t]) * table_stride + pos / page_size];
  const int g = y - nq - nkv;
  T* dst = v_pages + (static_cast<int64_t>(page) * nkv + g) * Dv * page_size + pos % page_size;
  for (int d = lane; d < Dv; d += kWave) dst[static_cast<int64_t>(d) * page_size] = v[t * v_stride + g * Dv + d];
}

// The same for steps of many rows, bfloat16 heads of 8 LPH elements (Dk = Dv), everything on the 16-byte grid: LPH lanes a
// head, eight elements a lane and access, kStoreHeads heads a lane so that the norm's weight and the position are read once
// for all of them.  Sixteen consecutive positions of a request that fill a page's slots are turned through LDS and leave as
// 16-byte pieces of a column; one element at a time (2-byte stores 32 bytes apart) is what the kernel above spends its time
// on.  MI355X, 2,048 rows of 32 + 8 + 8 heads of 128: 12.2 us, the
// 50 MB at 4.1 TB/s; the kernel above 40.
constexpr int kStoreHeads = 4;
constexpr int kStoreManyRows = 96;   // rows of a step from which on this form is taken: kernel above / this one at 64 rows 5.2 / 5.6 us, 96 5.8 / 5.7, 128 6.3 / 5.7, 256 8.6 / 6.2

template <int LPH>
__global__ __launch_bounds__(256) void qkv_norm_store_rows_kernel(
    uint16_t* __restrict__ q, long long q_stride, const uint16_t* __restrict__ k, long long k_stride,
    const uint16_t* __restrict__ v, long long v_stride, const void* __restrict__ q_weight, const void* __restrict__ k_weight,
    int w_dtype, float eps, float temp_coef, int temp_every, const int* __restrict__ positions,
    const int* __restrict__ slot_of_token, const int* __restrict__ block_table, int table_stride,
    uint16_t* __restrict__ k_pages, uint16_t* __restrict__ v_pages, int tokens, int nq, int nkv, int page_size) {
  constexpr int D = 8 * LPH;
  constexpr int kRows = 256 / LPH;      // rows of a workgroup
  constexpr int kPitch = D + 8;         // LDS row of the value tile, in elements
  __shared__ __align__(16) uint16_t tile[kRows * kPitch];
  const int tl = threadIdx.x / LPH, d0 = (threadIdx.x % LPH) * 8;
  const int row0 = blockIdx.x * kRows, t = row0 + tl;
  const bool valid = t < tokens;
  const int64_t src_row = min(t, tokens - 1);
  // blockIdx.y: groups of kStoreHeads q heads, then groups of k heads, then the v heads one by one
  const int q_groups = (nq + kStoreHeads - 1) / kStoreHeads, k_groups = (nkv + kStoreHeads - 1) / kStoreHeads;
  const int y = blockIdx.y;
  const int pos = positions[src_row];
  if (y >= q_groups + k_groups) {
    const int g = y - q_groups - k_groups;
    const u32x4_t raw = *reinterpret_cast<const u32x4_t*>(v + src_row * v_stride + g * D + d0);
    const int slot = slot_of_token[src_row];
    bool run = false;
    if constexpr (kRows >= 16) {
      const int first_pos = positions[row0], first_slot = slot_of_token[row0];
      run = __syncthreads_and(valid && pos == first_pos + tl && slot == first_slot && first_pos % 16 == 0 && page_size % 16 == 0) != 0;
      if (run) {
        *reinterpret_cast<u32x4_t*>(&tile[tl * kPitch + d0]) = raw;
        __syncthreads();
        constexpr int kPieces = kRows / 8;      // 16-byte pieces of eight slots of a column
        const int d = threadIdx.x / kPieces, first = (threadIdx.x % kPieces) * 8;
        static_assert(256 / kPieces == D, "a thread a piece");
        u32x4_t piece;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          piece[e] = static_cast<uint32_t>(tile[(first + 2 * e) * kPitch + d]) |
                     (static_cast<uint32_t>(tile[(first + 2 * e + 1) * kPitch + d]) << 16);
        const int p = first_pos + first;
        const int page = block_table[static_cast<int64_t>(first_slot) * table_stride + p / page_size];
        *reinterpret_cast<u32x4_t*>(v_pages + ((static_cast<int64_t>(page) * nkv + g) * D + d) * page_size + p % page_size) = piece;
      }
    }
    if (!run && valid) {
      const int page = block_table[static_cast<int64_t>(slot) * table_stride + pos / page_size];
      uint16_t* dst = v_pages + ((static_cast<int64_t>(page) * nkv + g) * D + d0) * page_size + pos % page_size;
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[static_cast<int64_t>(e) * page_size] = static_cast<uint16_t>(raw[e / 2] >> (16 * (e & 1)));
    }
    return;
  }
  const bool is_q = y < q_groups;
  const int count = is_q ? nq : nkv, first = (is_q ? y : y - q_groups) * kStoreHeads;
  const uint16_t* src = is_q ? q + src_row * q_stride + d0 : k + src_row * k_stride + d0;
  u32x4_t raw[kStoreHeads];
#pragma unroll
  for (int h = 0; h < kStoreHeads; ++h) raw[h] = *reinterpret_cast<const u32x4_t*>(src + min(first + h, count - 1) * D);
  const void* weight = is_q ? q_weight : k_weight;
  float w[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = weight ? load_as_float(weight, w_dtype, d0 + e) : 1.0f;
  const float temp = is_q && temp_coef != 0.f ? 1.0f + temp_coef * logf(static_cast<float>((pos + 1) / temp_every + 1)) : 1.0f;
  uint16_t* dst = q + src_row * q_stride + d0;
  int64_t head_step = D;
  if (!is_q) {
    const int page = block_table[static_cast<int64_t>(slot_of_token[src_row]) * table_stride + pos / page_size];
    head_step = static_cast<int64_t>(page_size) * D;
    dst = k_pages + static_cast<int64_t>(page) * nkv * head_step + (pos % page_size) * D + d0;
  }
#pragma unroll
  for (int h = 0; h < kStoreHeads; ++h) {
    float x[8], ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[2 * e] = __uint_as_float(raw[h][e] << 16);
      x[2 * e + 1] = __uint_as_float(raw[h][e] & 0xffff0000u);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
    ss = lanes_sum<LPH>(ss);
    const float f = 1.0f / sqrtf(ss / static_cast<float>(D) + eps) * temp;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = x[e] * f * w[e];
    if (valid && first + h < count)
      *reinterpret_cast<u32x4_t*>(dst + (first + h) * head_step) =
          u32x4_t{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]), pack_bf16x2(x[6], x[7])};
  }
}

template <typename T>
__global__ __launch_bounds__(kWave) void attn_softcap_simt_kernel(
    const T* __restrict__ q, int64_t q_stride, T* __restrict__ out, int64_t o_stride, const T* __restrict__ k_pages,
    const T* __restrict__ v_pages, const int* __restrict__ block_table, int table_stride,
    const int* __restrict__ positions, const int* __restrict__ slot_of_token, int nq, int nkv, int Dk, int Dv,
    int page_size, float scale, float cap, const void* __restrict__ r1, const void* __restrict__ r2, int r_dtype,
    int window, int chunk, const void* __restrict__ sink, int sink_dtype, int keep_first, float out_scale) {
  extern __shared__ float qs[];  // [Dk]
  const int t = blockIdx.x;
  const int h = blockIdx.y;
  const int lane = threadIdx.x;
  const int kvh = h / (nq / nkv);
  const int pos = positions[t];
  const int* table = block_table + static_cast<int64_t>(slot_of_token[t]) * table_stride;
  const float pen1 = r1 ? load_as_float(r1, r_dtype, h) : 0.f;
  const float pen2 = r1 ? load_as_float(r2, r_dtype, h) : 0.f;
  const float inv_cap = cap > 0.f ? 1.0f / cap : 0.f;

  const T* qr = q + static_cast<int64_t>(t) * q_stride + h * Dk;
  for (int d = lane; d < Dk; d += kWave) qs[d] = to_float(qr[d]);
  __syncthreads();

  int first = window > 0 ? max(0, pos - window + 1) : 0;
  // the first `kept` keys of the request stay visible when the window has passed them (the chunk rule still holds)
  const int chunk_first = chunk > 0 ? pos / chunk * chunk : 0;
  first = max(first, chunk_first);
  const int kept = min(keep_first, first);              // keys [chunk_first, kept) and [first, pos] are seen
  const bool head_part = kept > chunk_first;
  const int64_t k_page = static_cast<int64_t>(nkv) * page_size * Dk, v_page = static_cast<int64_t>(nkv) * page_size * Dv;
  const int64_t k_head = static_cast<int64_t>(kvh) * page_size * Dk, v_head = static_cast<int64_t>(kvh) * page_size * Dv;

  float m = -INFINITY, l = 0.f;
  float acc[kCapMaxD / kWave];
#pragma unroll
  for (int i = 0; i < kCapMaxD / kWave; ++i) acc[i] = 0.f;

  for (int tile = head_part ? chunk_first / kWave : first / kWave; tile * kWave <= pos; ++tile) {
    if (head_part && tile * kWave >= kept && (tile + 1) * kWave <= first) {   // a tile between the two parts
      tile = first / kWave - 1;
      continue;
    }
    const int c = tile * kWave + lane;
    const bool valid = c <= pos && (c >= first || (head_part && c >= chunk_first && c < kept));
    float s = -INFINITY;
    if (valid) {
      const int page = table[c / page_size];
      const T* kr = k_pages + page * k_page + k_head + static_cast<int64_t>(c % page_size) * Dk;
      float dot = 0.f;
      for (int d = 0; d < Dk; ++d) dot = fmaf(qs[d], to_float(kr[d]), dot);
      s = dot * scale;
      if (cap > 0.f) s = cap * tanhf(s * inv_cap);
      if (r1) s -= pen1 * log1pf(pen2 * static_cast<float>(pos - c));
    }
    const float m_new = fmaxf(m, wave_max(s));  // the tile holds at least one visible key
    const float alpha = expf(m - m_new);        // 0 on the first tile (m = -inf)
    const float p = valid ? expf(s - m_new) : 0.f;
    l = l * alpha + wave_sum(p);
#pragma unroll
    for (int i = 0; i < kCapMaxD / kWave; ++i) acc[i] *= alpha;

    const int j_lo = max((head_part ? chunk_first : first) - tile * kWave, 0);
    const int j_hi = min(pos - tile * kWave, kWave - 1);
    for (int j = j_lo; j <= j_hi; ++j) {
      const float pj = __shfl(p, j, kWave);
      const int cj = tile * kWave + j;
      if (cj < first && cj >= kept) continue;   // between the parts: a page that may have been given back
      const int page = table[cj / page_size];
      const T* vr = v_pages + page * v_page + v_head + (cj % page_size);  // [d][slot in page]
#pragma unroll
      for (int i = 0; i < kCapMaxD / kWave; ++i) {
        const int d = lane + i * kWave;
        if (d < Dv) acc[i] = fmaf(pj, to_float(vr[static_cast<int64_t>(d) * page_size]), acc[i]);
      }
    }
    m = m_new;
  }

  T* o = out + static_cast<int64_t>(t) * o_stride + h * Dv;
  float keep = 1.0f;
  if (sink) {  // one more term in the denominator, with no value behind it
    const float sk = load_as_float(sink, sink_dtype, h);
    const float m_all = fmaxf(m, sk);
    keep = expf(m - m_all);
    l = l * keep + expf(sk - m_all);
  }
  const float inv_l = keep / l * out_scale;
#pragma unroll
  for (int i = 0; i < kCapMaxD / kWave; ++i) {
    const int d = lane + i * kWave;
    if (d < Dv) o[d] = from_float<T>(acc[i] * inv_l);
  }
}

// Operands of an attention that norms q and k over the whole projection.  One workgroup a (row, one of q, k, v):
//   q <- q / rms(q) * wq  in place over all nq * Dk entries (wq null: q stays as it is);
//   k likewise over all nkv * Dk entries, into the pages;
//   v <- (1 - lambda) v + lambda v_first (v_first given), into the pages (d-major).
// lambda is one number in memory, so that a captured launch reads the checkpoint's value.
constexpr int kWideThreads = 256;
template <typename T>
__global__ __launch_bounds__(kWideThreads) void wide_norm_store_kernel(
    T* __restrict__ q, long long q_stride, const T* __restrict__ k, long long k_stride, const T* __restrict__ v,
    long long v_stride, const T* __restrict__ v_first, long long vf_stride, const void* __restrict__ q_weight,
    const void* __restrict__ k_weight, int w_dtype, const void* __restrict__ lambda, int lambda_dtype, float eps,
    const int* __restrict__ positions, const int* __restrict__ slot_of_token, const int* __restrict__ block_table,
    int table_stride, T* __restrict__ k_pages, T* __restrict__ v_pages, int nq, int nkv, int Dk, int Dv, int page_size,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, int rot, int halves) {
  extern __shared__ float staged[];   // [max(nq, nkv) * Dk] with a rotation, else nothing
  __shared__ float lds[kWideThreads / kWave];
  const int64_t t = blockIdx.x;
  const int what = blockIdx.y;
  const int pos = positions[t];
  // With a rotation the normed row waits in LDS, so that an entry's partner is read as it was before anything is
  // written: entry d < rot of a head turns with entry d ^ 1 (or, with `halves`, d +- rot / 2) by the angle of its pair.
  const int half = rot / 2;
  const float* cs = rot ? cos_t + static_cast<int64_t>(pos) * half : nullptr;
  const float* sn = rot ? sin_t + static_cast<int64_t>(pos) * half : nullptr;
  auto turned = [&](const float* head, int d) {
    const int partner = halves ? (d < half ? d + half : d - half) : (d ^ 1);
    const int pair = halves ? (d < half ? d : d - half) : d / 2;
    const bool second = halves ? d >= half : (d & 1);
    const float c = cs[pair], sv = sn[pair];
    return second ? fmaf(head[d], c, head[partner] * sv) : fmaf(head[d], c, -head[partner] * sv);
  };
  auto stage = [&](const T* row, int width, const void* weight) {   // the row, normed where it has a weight, into LDS
    float ss = 0.f;
    for (int i = threadIdx.x; i < width; i += kWideThreads) {
      const float x = to_float(row[i]);
      staged[i] = x;
      ss = fmaf(x, x, ss);
    }
    const float total = block_sum<kWideThreads / kWave>(ss, lds);   // (its barriers also order the writes above)
    if (weight) {
      const float inv = 1.0f / sqrtf(total / static_cast<float>(width) + eps);
      for (int i = threadIdx.x; i < width; i += kWideThreads) staged[i] = staged[i] * inv * load_as_float(weight, w_dtype, i);
    }
    __syncthreads();
  };
  if (what == 0) {
    if (!q_weight && !rot) return;
    const int width = nq * Dk;
    T* row = q + t * q_stride;
    if (rot) {
      stage(row, width, q_weight);
      for (int i = threadIdx.x; i < width; i += kWideThreads) {
        const int d = i % Dk;
        row[i] = from_float<T>(d < rot ? turned(staged + (i - d), d) : staged[i]);
      }
      return;
    }
    float ss = 0.f;
    for (int i = threadIdx.x; i < width; i += kWideThreads) {
      const float x = to_float(row[i]);
      ss = fmaf(x, x, ss);
    }
    const float inv = 1.0f / sqrtf(block_sum<kWideThreads / kWave>(ss, lds) / static_cast<float>(width) + eps);
    for (int i = threadIdx.x; i < width; i += kWideThreads)
      row[i] = from_float<T>(to_float(row[i]) * inv * load_as_float(q_weight, w_dtype, i));
    return;
  }
  const int64_t page = block_table[static_cast<int64_t>(slot_of_token[t]) * table_stride + pos / page_size];
  const int in_page = pos % page_size;
  if (what == 1) {
    const int width = nkv * Dk;
    const T* row = k + t * k_stride;
    if (rot) {
      stage(row, width, k_weight);
      for (int i = threadIdx.x; i < width; i += kWideThreads) {
        const int g = i / Dk, d = i % Dk;
        k_pages[((page * nkv + g) * page_size + in_page) * Dk + d] =
            from_float<T>(d < rot ? turned(staged + (i - d), d) : staged[i]);
      }
      return;
    }
    float inv = 1.0f;
    if (k_weight) {
      float ss = 0.f;
      for (int i = threadIdx.x; i < width; i += kWideThreads) {
        const float x = to_float(row[i]);
        ss = fmaf(x, x, ss);
      }
      inv = 1.0f / sqrtf(block_sum<kWideThreads / kWave>(ss, lds) / static_cast<float>(width) + eps);
    }
    for (int i = threadIdx.x; i < width; i += kWideThreads) {
      const int g = i / Dk, d = i % Dk;
      const float x = to_float(row[i]);
      k_pages[((page * nkv + g) * page_size + in_page) * Dk + d] =
          k_weight ? from_float<T>(x * inv * load_as_float(k_weight, w_dtype, i)) : row[i];
    }
    return;
  }
  const int width = nkv * Dv;
  const float lam = v_first ? load_as_float(lambda, lambda_dtype, 0) : 0.f;
  for (int i = threadIdx.x; i < width; i += kWideThreads) {
    const int g = i / Dv, d = i % Dv;
    T x = v[t * v_stride + i];
    if (v_first) x = from_float<T>((1.0f - lam) * to_float(x) + lam * to_float(v_first[t * vf_stride + i]));
    v_pages[((page * nkv + g) * Dv + d) * page_size + in_page] = x;
  }
}

}  // namespace arle

using namespace arle;

// q [T, nq*Dk] is normed and scaled in place; k [T, nkv*Dk] and v [T, nkv*Dv] go to the pages (nkv 0: a layer
// that reads another layer's pages and only prepares q).  q_weight, k_weight: [Dk] or null.
extern "C" int arle_qkv_norm_store(void* q, long long q_stride, const void* k, long long k_stride, const void* v,
                                   long long v_stride, int dtype, const void* q_weight, const void* k_weight,
                                   int w_dtype, float eps, float temp_coef, int temp_every, const int* positions,
                                   const int* slot_of_token, const int* block_table, int table_stride, void* k_pages,
                                   void* v_pages, int tokens, int nq, int nkv, int Dk, int Dv, int page_size,
                                   void* stream) {
  if (tokens == 0) return 0;
  if (Dk > kCapMaxD || Dk < 1 || nq + 2 * nkv > 65535 || (temp_coef != 0.f && temp_every < 1))
    return static_cast<int>(hipErrorInvalidValue);
  const dim3 grid(tokens, nq + 2 * nkv);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto on_grid = [](const void* p, long long stride) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 8 == 0; };
  if (dtype == kBF16 && tokens >= kStoreManyRows && (Dk == 64 || Dk == 128 || Dk == 256) && on_grid(q, q_stride) &&
      (nkv == 0 || (Dv == Dk && on_grid(k, k_stride) && on_grid(v, v_stride) && on_grid(k_pages, 0) && on_grid(v_pages, 0)))) {
    auto u16 = [](const void* p) { return static_cast<uint16_t*>(const_cast<void*>(p)); };
    const int lanes = Dk / 8, rows = 256 / lanes;
    const dim3 groups((tokens + rows - 1) / rows, (nq + kStoreHeads - 1) / kStoreHeads + (nkv + kStoreHeads - 1) / kStoreHeads + nkv);
#define ARLE_STORE_ROWS(LPH)                                                                                               \
  qkv_norm_store_rows_kernel<LPH><<<groups, 256, 0, s>>>(u16(q), q_stride, u16(k), k_stride, u16(v), v_stride, q_weight,    \
                                                         k_weight, w_dtype, eps, temp_coef, temp_every, positions,         \
                                                         slot_of_token, block_table, table_stride, u16(k_pages),           \
                                                         u16(v_pages), tokens, nq, nkv, page_size)
    if (Dk == 64) ARLE_STORE_ROWS(8); else if (Dk == 128) ARLE_STORE_ROWS(16); else ARLE_STORE_ROWS(32);
#undef ARLE_STORE_ROWS
    return launch_status();
  }
  if (dtype == kF32) {
    qkv_norm_store_kernel<float><<<grid, kWave, 0, s>>>(
        static_cast<float*>(q), q_stride, static_cast<const float*>(k), k_stride, static_cast<const float*>(v), v_stride,
        q_weight, k_weight, w_dtype, eps, temp_coef, temp_every, positions, slot_of_token, block_table, table_stride,
        static_cast<float*>(k_pages), static_cast<float*>(v_pages), nq, nkv, Dk, Dv, page_size);
  } else {
    qkv_norm_store_kernel<bf16><<<grid, kWave, 0, s>>>(
        static_cast<bf16*>(q), q_stride, static_cast<const bf16*>(k), k_stride, static_cast<const bf16*>(v), v_stride,
        q_weight, k_weight, w_dtype, eps, temp_coef, temp_every, positions, slot_of_token, block_table, table_stride,
        static_cast<bf16*>(k_pages), static_cast<bf16*>(v_pages), nq, nkv, Dk, Dv, page_size);
  }
  return launch_status();
}

// q [T, nq*Dk], out [T, nq*Dv] of `dtype`, as the pages.  cap 0: no soft cap.  r1, r2: [nq] or null.
extern "C" int arle_attn_softcap_simt(const void* q, long long q_stride, void* out, long long o_stride,
                                      const void* k_pages, const void* v_pages, int dtype, const int* block_table,
                                      int table_stride, const int* positions, const int* slot_of_token, int tokens,
                                      int nq, int nkv, int Dk, int Dv, int page_size, float scale, float cap,
                                      const void* r1, const void* r2, int r_dtype, int window, int chunk,
                                      const void* sink, int sink_dtype, int keep_first, float out_scale,
                                      void* stream) {
  if (tokens == 0) return 0;
  if (Dk > kCapMaxD || Dv > kCapMaxD || nkv < 1 || nq % nkv != 0 || nq > 65535 || window < 0 || chunk < 0 ||
      keep_first < 0 || (keep_first > 0 && window == 0))
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid(tokens, nq);
  const size_t lds = static_cast<size_t>(Dk) * sizeof(float);
  if (dtype == kF32) {
    attn_softcap_simt_kernel<float><<<grid, kWave, lds, s>>>(
        static_cast<const float*>(q), q_stride, static_cast<float*>(out), o_stride, static_cast<const float*>(k_pages),
        static_cast<const float*>(v_pages), block_table, table_stride, positions, slot_of_token, nq, nkv, Dk, Dv,
        page_size, scale, cap, r1, r2, r_dtype, window, chunk, sink, sink_dtype, keep_first,
        out_scale);
  } else {
    attn_softcap_simt_kernel<bf16><<<grid, kWave, lds, s>>>(
        static_cast<const bf16*>(q), q_stride, static_cast<bf16*>(out), o_stride, static_cast<const bf16*>(k_pages),
        static_cast<const bf16*>(v_pages), block_table, table_stride, positions, slot_of_token, nq, nkv, Dk, Dv,
        page_size, scale, cap, r1, r2, r_dtype, window, chunk, sink, sink_dtype, keep_first,
        out_scale);
  }
  return launch_status();
}

// q [T, nq*Dk] is normed in place over the whole row (q_weight [nq*Dk] or null); k [T, nkv*Dk] is normed likewise
// (k_weight [nkv*Dk] or null) and goes to the pages; v [T, nkv*Dv], mixed with v_first by *lambda where v_first is
// given, goes to the pages.  rot > 0: behind the norm the first `rot` entries of every head of q and k turn by the
// angles of float32 tables cos, sin [positions, rot / 2]; halves != 0 pairs entry i with i + rot / 2, else 2i with 2i + 1.
extern "C" int arle_wide_norm_store(void* q, long long q_stride, const void* k, long long k_stride, const void* v,
                                    long long v_stride, const void* v_first, long long vf_stride, int dtype,
                                    const void* q_weight, const void* k_weight, int w_dtype, const void* lambda,
                                    int lambda_dtype, float eps, const int* positions, const int* slot_of_token,
                                    const int* block_table, int table_stride, void* k_pages, void* v_pages, int tokens,
                                    int nq, int nkv, int Dk, int Dv, int page_size, const float* cos_t,
                                    const float* sin_t, int rot, int halves, void* stream) {
  if (tokens == 0) return 0;
  if (nq < 1 || nkv < 1 || Dk < 1 || Dv < 1 || page_size < 1 || (v_first && !lambda) || rot < 0 || rot > Dk || rot % 2 ||
      (rot && (!cos_t || !sin_t)))
    return static_cast<int>(hipErrorInvalidValue);
  const dim3 grid(tokens, 3);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t staged_bytes = rot ? static_cast<size_t>(nq > nkv ? nq : nkv) * Dk * sizeof(float) : 0;
  if (staged_bytes > 64 * 1024) return static_cast<int>(hipErrorInvalidValue);
  static OnceADevice asked;
  if (staged_bytes > 48 * 1024)
    if (const int e = ask_lds(asked, 64 * 1024, {reinterpret_cast<const void*>(&wide_norm_store_kernel<float>),
                                                 reinterpret_cast<const void*>(&wide_norm_store_kernel<bf16>)}))
      return e;
  if (dtype == kF32) {
    wide_norm_store_kernel<float><<<grid, kWideThreads, staged_bytes, s>>>(
        static_cast<float*>(q), q_stride, static_cast<const float*>(k), k_stride, static_cast<const float*>(v), v_stride,
        static_cast<const float*>(v_first), vf_stride, q_weight, k_weight, w_dtype, lambda, lambda_dtype, eps, positions,
        slot_of_token, block_table, table_stride, static_cast<float*>(k_pages), static_cast<float*>(v_pages), nq, nkv, Dk,
        Dv, page_size, cos_t, sin_t, rot, halves);
  } else {
    wide_norm_store_kernel<bf16><<<grid, kWideThreads, staged_bytes, s>>>(
        static_cast<bf16*>(q), q_stride, static_cast<const bf16*>(k), k_stride, static_cast<const bf16*>(v), v_stride,
        static_cast<const bf16*>(v_first), vf_stride, q_weight, k_weight, w_dtype, lambda, lambda_dtype, eps, positions,
        slot_of_token, block_table, table_stride, static_cast<bf16*>(k_pages), static_cast<bf16*>(v_pages), nq, nkv, Dk,
        Dv, page_size, cos_t, sin_t, rot, halves);
  }
  return launch_status();
}

// ---- matrix-core kernel (bfloat16) ------------------------------------------------------------
// One wave a work item of queries that share a kv head: sixteen or 32 consecutive rows of one request for one
// q head (prompt portions), or one decoded row for the up to sixteen q heads of a kv head.  The scores are
// computed transposed, S^T[key][query] = K . Q^T with `v_mfma_f32_16x16x32_bf16`, of a tile of 32 keys in two halves:
// row r of half h is key 8 (r / 4) + 4 h + r % 4, so that a lane holds, for its query (lane % 16), the keys 8g..8g+7
// (g = lane / 16): the cap, the penalty, the mask and the running softmax are per-lane arithmetic plus two lane
// exchanges, and the eight probabilities of a lane are, as they lie, the B operand of the second product
// O^T += V^T . P^T with one 16-byte load from the d-major value pages on the V side.  Sixteen keys in a row are slots of
// one page (page sizes are multiples of 16).  Pages that a window has passed (entry -1) and slots beyond the newest key are never visible;
// their keys are masked by a select and their values replaced by zeros, so that stale bits cannot reach a sum.
namespace arle {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

struct CapArgs {
  const bf16* q; long long q_stride;
  bf16* out; long long o_stride;
  const bf16* k_pages; const bf16* v_pages;
  const int* block_table; int table_stride;
  const int* seg_row0; const int* seg_slot; const int* seg_start;
  int segments, nq, nkv, Dk, Dv, page_size;
  float scale, cap;
  const void* r1; const void* r2; int r_dtype;
  int window;
  int chunk;                          // 0: none; else a row sees only the keys of its own chunk of so many positions
  const void* sink; int sink_dtype;   // [nq] or null: exp(sink_h) joins the softmax's denominator
  int merge_floats;   // floats of dynamic LDS in front of the page ids
  int keep_first;     // with a window: the request's first so many keys stay visible behind it (0: none)
  float out_scale;    // a factor on the output, in 32 bits
};

}  // namespace arle
#include "attention_softcap_portions.h"
namespace arle {

// KC: chunks of 32 of the key size held (Dk <= 32 KC); VC: chunks of 16 of the value size (Dv <= 16 VC).
// HEADS: a work item is one row (a segment of one row) and the q heads of a kv head, and the WAVES waves of the
// workgroup take its tiles of keys in turn and add their sums through LDS; else an item is 16 QB rows of one q head,
// and the waves of a workgroup are WAVES q heads of one kv head on the same rows, so that they fetch the same tiles.
//
// What bounds portions: every wave fetches its tiles by itself, 16 KB for 32 keys of 128, through its compute unit's
// cache, and a score costs three quarter-rate instructions (two exponentials and a reciprocal).  So two blocks of sixteen
// rows share a tile (QB 2, where there are waves enough), values come in pieces of 16 bytes, keys of the next tile are
// fetched while this one's probabilities are made and values while its scores are, masks are worked out in the tiles at
// the ends only, sums are rescaled only where a maximum moved, and the lanes' sums meet once at the end.  A layer of 2,048
// rows, 32 q heads and 8 kv heads of 128, window 1,024: 173 us before, 89 now (184 and 110 between the other kernels of a
// prompt; the masks that each block of sixteen rows has of its own are 4 and 8 of these; at heads of 128 most of these now go to
// the kernel of attention_softcap_portions.h); 256 rows 25 -> 16; eight decoded
// rows behind 2,048 keys 21 -> 17.  (Portions of heads up to 128 are held to the registers of two waves a SIMD.)
template <int KC, int VC, bool HEADS, int WAVES, int QB>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(!HEADS && KC <= 4 && VC <= 8 ? 2 : 1)))
void attn_softcap_mfma_kernel(const CapArgs a) {
  extern __shared__ float merge_lds[];   // HEADS: [WAVES][n_vc][64 lanes][4], then m [WAVES][16], l [WAVES][16]; then page ids
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, n = lane % 16, g = lane / 16;
  const int group = a.nq / a.nkv;
  int seg, head, kvh, first_row, last_row, row[QB];
  bool live[QB];
  if (HEADS) {
    // a kv head with more than sixteen q heads is taken by several workgroups, sixteen q heads each
    const int parts = (group + 15) / 16, part = blockIdx.y % parts;
    seg = blockIdx.x;
    kvh = blockIdx.y / parts;
    row[0] = first_row = last_row = a.seg_row0[seg];
    head = kvh * group + min(16 * part + n, group - 1);
    live[0] = 16 * part + n < group;
  } else {
    // Workgroups go to the chip's eight dies in turn (the launch order is blockIdx.x fastest), and every die has a
    // level-two cache of its own: with the head groups a multiple of eight, die i takes the head groups i, i + 8, ...
    // with all their row blocks, so that it keeps the keys and values of its own kv heads and not everybody's.
    int bx = blockIdx.x, by = blockIdx.y;
    if (gridDim.y % 8 == 0) {
      const unsigned linear = blockIdx.y * gridDim.x + blockIdx.x, die = linear % 8, within = linear / 8;
      by = die + 8 * (within / gridDim.x);
      bx = within % gridDim.x;
    }
    // the bx-th block of rows, counted through the segments
    int left = bx, found = -1;
    for (int s = 0; s < a.segments; ++s) {
      const int blocks = (a.seg_row0[s + 1] - a.seg_row0[s] + 16 * QB - 1) / (16 * QB);
      if (left < blocks) {
        found = s;
        break;
      }
      left -= blocks;
    }
    if (found < 0) return;
    seg = found;
    head = by * WAVES + wave;
    kvh = head / group;
    const int end = a.seg_row0[seg + 1];
    first_row = a.seg_row0[seg] + left * (16 * QB);
    last_row = min(first_row + 16 * QB - 1, end - 1);
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      live[b] = first_row + 16 * b + n < end;
      row[b] = min(first_row + 16 * b + n, end - 1);
    }
  }
  const int seg_first = a.seg_row0[seg];
  const int start = a.seg_start[seg];
  // keys that any query of the item sees: from the first row's window to the last row's own position
  const int pos_lo = start + (first_row - seg_first);
  const int pos_hi = start + (last_row - seg_first);
  auto first_seen = [&](int p) {
    int lo = a.window > 0 ? max(0, p - a.window + 1) : 0;
    if (a.chunk > 0) lo = max(lo, p / a.chunk * a.chunk);
    return lo;
  };
  const int key_lo = first_seen(pos_lo);
  const int all_lo = first_seen(pos_hi);   // every row sees the keys from here to pos_lo
  // The request's first `keep` keys stay visible to rows whose window has passed them.  Their tiles of 32 keys that
  // lie wholly in front of the first tile of the windows are `head_tiles` tiles of their own, walked first; the walk
  // counts tiles through both parts (`walk` 0 .. walk_last), and `tile_of` gives the tile of keys behind a count.
  const int keep = a.keep_first;
  const int head_tiles = min((keep + 31) / 32, key_lo / 32);
  const int main_first = key_lo / 32;
  auto tile_of = [&](int walk) { return walk < head_tiles ? walk : walk - head_tiles + main_first; };
  // Scores are kept in units of ln 2, so that every exponential is one of base 2.
  constexpr float kLog2e = 1.4426950408889634f;
  const float sink = a.sink ? load_as_float(a.sink, a.sink_dtype, head) * kLog2e : -INFINITY;
  const int* table = a.block_table + static_cast<int64_t>(a.seg_slot[seg]) * a.table_stride;
  const float pen1 = a.r1 ? load_as_float(a.r1, a.r_dtype, head) : 0.f;
  const float pen2 = a.r1 ? load_as_float(a.r2, a.r_dtype, head) : 0.f;
  // cap tanh(x / cap) = cap - 2 cap / (1 + exp(2 x / cap)), x = scale * product
  const float to_exp = a.cap > 0.f ? 2.0f * kLog2e * a.scale / a.cap : 0.f, cap2 = a.cap * kLog2e, scale2 = a.scale * kLog2e;
  const int n_kc = (a.Dk + 31) / 32, n_vc = a.Dv / 16;

  // Q^T operand: for chunk c, Q[row][32 c + 8 g .. + 7]
  bf16x8_t qreg[QB][KC];
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    const bf16* qr = a.q + static_cast<int64_t>(row[b]) * a.q_stride + head * a.Dk;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const u32x4_t raw = *reinterpret_cast<const u32x4_t*>(qr + min(32 * c + 8 * g, a.Dk - 8));
      qreg[b][c] = __builtin_bit_cast(bf16x8_t, 32 * c + 8 * g < a.Dk ? raw : u32x4_t{0, 0, 0, 0});
    }
  }
  f32x4_t acc[QB][VC];
  float m_run[QB], l_run[QB];   // a row's largest score so far (the same in its four lanes), and this lane's part of its sum
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    m_run[b] = -INFINITY;
    l_run[b] = 0.f;
#pragma unroll
    for (int c = 0; c < VC; ++c) acc[b][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  const int64_t k_page = static_cast<int64_t>(a.nkv) * a.page_size * a.Dk, v_page = static_cast<int64_t>(a.nkv) * a.page_size * a.Dv;
  const int64_t k_head = static_cast<int64_t>(kvh) * a.page_size * a.Dk, v_head = static_cast<int64_t>(kvh) * a.page_size * a.Dv;
  const int tile_step = HEADS ? WAVES : 1;
  const int tile_first = HEADS ? wave : 0;                                   // counts of the walk
  const int tile_last = head_tiles + pos_hi / 32 - main_first, last_entry = a.table_stride - 1;

  // The ids of the pages that the item sees are put into LDS once: a tile's loads then follow no load of a page id,
  // and the reads of LDS are counted apart from the loads from memory, so they disturb no wait for those.
  const int page_first = (key_lo / 32 * 32) / a.page_size;   // the page of the first tile's first key, which may lie in front of key_lo's
  // (the ids of the head tiles' pages, the request's first ones, lie in front of them)
  const int head_pages = head_tiles > 0 ? (head_tiles * 32 + a.page_size - 1) / a.page_size : 0;
  int* head_lds = reinterpret_cast<int*>(merge_lds) + a.merge_floats;
  int* page_lds = head_lds + head_pages;
  for (int i = threadIdx.x; i < head_pages; i += WAVES * kWave) head_lds[i] = table[min(i, last_entry)];
  for (int i = threadIdx.x; i <= (pos_hi / 32 * 32 + 31) / a.page_size - page_first; i += WAVES * kWave)
    page_lds[i] = table[min(page_first + i, last_entry)];
  __syncthreads();
  // A tile past the last is the last one again, fetched and dropped.  No load stands under a condition (one would make
  // every later wait a wait for all loads in flight): a piece past the head's size is the head's last piece again, zeroed
  // or left unused afterwards.
  // the page (clamped) and the slot in it of key key0 + 16 * high, high given a lane
  auto place = [&](int at, bool high, int64_t& page, int& in_page) {
    const int key0 = tile_of(at) * 32;
    const int p0 = key0 / a.page_size, p1 = (key0 + 16) / a.page_size;
    const int p = high ? p1 : p0;
    in_page = (high ? key0 + 16 - p1 * a.page_size : key0 - p0 * a.page_size);
    page = max(at < head_tiles ? head_lds[p] : page_lds[max(p - page_first, 0)], 0);
  };
  // Row r of half h of a tile is key 8 (r / 4) + 4 h + r % 4: a lane's scores 4 g .. 4 g + 3 of both halves are then the
  // keys 8 g .. 8 g + 7, which the value pages hold in one piece of 16 bytes.
  auto load_keys = [&](int walk, u32x4_t (&kraw)[2][KC]) {
    int64_t page;
    int in_page;
    place(min(walk, tile_last), n >= 8, page, in_page);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bf16* kr = a.k_pages + page * k_page + k_head +
                       static_cast<int64_t>(in_page + 8 * (n / 4 % 2) + 4 * half + n % 4) * a.Dk;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const u32x4_t raw = *reinterpret_cast<const u32x4_t*>(kr + min(32 * c + 8 * g, a.Dk - 8));
        kraw[half][c] = 32 * c + 8 * g < a.Dk ? raw : u32x4_t{0, 0, 0, 0};
      }
    }
  };
  auto load_values = [&](int walk, u32x4_t (&vraw)[VC]) {
    int64_t page;
    int in_page;
    place(min(walk, tile_last), g >= 2, page, in_page);
    const bf16* vp = a.v_pages + page * v_page + v_head + in_page + 8 * (g % 2);
#pragma unroll
    for (int c = 0; c < VC; ++c)
      vraw[c] = *reinterpret_cast<const u32x4_t*>(vp + static_cast<int64_t>(min(16 * c + n, a.Dv - 1)) * a.page_size);
  };

  // the scores of a tile, capped, penalised and masked: s[b][4 half + i] is key 8 g + 4 half + i of it
  auto score = [&](int walk, const u32x4_t (&kraw)[2][KC], float (&s)[QB][8]) {
    const int key0 = tile_of(walk) * 32 + 8 * g;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        // S^T half tile: A = K[the half's sixteen keys][32 c + 8 g ..], B = Q^T
        f32x4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c)
          if (c < n_kc) z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kraw[half][c]), qreg[b][c], z, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[b][4 * half + i] = z[i];
      }
    }
    const bool whole = key0 - 8 * g >= all_lo && key0 - 8 * g + 31 <= pos_lo;   // every row sees every key
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      if (a.cap > 0.f) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          s[b][i] = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(s[b][i] * to_exp)), cap2);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) s[b][i] *= scale2;
      }
      const int pos = start + (row[b] - seg_first);
      if (a.r1) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          s[b][i] -= pen1 * __builtin_amdgcn_logf(1.0f + pen2 * static_cast<float>(pos - key0 - i));
      }
      if (!whole) {
        const int my_lo = first_seen(pos);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          s[b][i] = ((key0 + i >= my_lo || key0 + i < keep) && key0 + i <= pos) ? s[b][i] : -INFINITY;
      }
    }
  };
  // the running maximum and sums, and O^T += V^T . P^T
  auto gather = [&](int walk, float (&s)[QB][8], const u32x4_t (&vraw)[VC]) {
    const int key0 = tile_of(walk) * 32 + 8 * g;
    bf16x8_t pop[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float m_new = m_run[b];
#pragma unroll
      for (int i = 0; i < 8; ++i) m_new = fmaxf(m_new, s[b][i]);
      const LanePair near = across16(m_new), far = across32(fmaxf(near.lo, near.hi));
      m_new = fmaxf(far.lo, far.hi);
      // a query whose window begins behind this tile has seen nothing yet: keep its sums at zero without 0 * inf
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      if (__any(m_new != m_run[b])) {   // later tiles seldom hold a larger score for any of the rows
        const float alpha = __builtin_amdgcn_exp2f(m_run[b] - m_safe);
        l_run[b] *= alpha;
#pragma unroll
        for (int c = 0; c < VC; ++c) {
          acc[b][c][0] *= alpha; acc[b][c][1] *= alpha; acc[b][c][2] *= alpha; acc[b][c][3] *= alpha;
        }
        m_run[b] = m_new;
      }
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(s[b][i] - m_safe);
      l_run[b] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
      u32x4_t pb;
      pb[0] = pack_bf16x2(p[0], p[1]);
      pb[1] = pack_bf16x2(p[2], p[3]);
      pb[2] = pack_bf16x2(p[4], p[5]);
      pb[3] = pack_bf16x2(p[6], p[7]);
      pop[b] = __builtin_bit_cast(bf16x8_t, pb);
    }
    // In the tiles at the ends, which of this lane's eight key slots hold keys that a block of sixteen rows sees (those
    // between its first row's first and its last row's last key, and the kept first ones): the values of the others enter
    // its sums as zeros, so that what is in a slot never written, or a NaN that only the other block sees, stays out of them.
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const int lo = b == 0 ? key_lo : first_seen(pos_lo + 16 * b), hi = QB == 1 ? pos_hi : min(pos_lo + 16 * b + 15, pos_hi);
      const bool edge = key0 - 8 * g < lo || key0 - 8 * g + 31 > hi;
      u32x4_t seen = {~0u, ~0u, ~0u, ~0u};
      if (edge) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int key = key0 + j;
          if ((key < lo && key >= keep) || key > hi) seen[j / 2] &= (j % 2) ? 0x0000ffffu : 0xffff0000u;
        }
      }
#pragma unroll
      for (int c = 0; c < VC; ++c) {
        if (c < n_vc) {
          u32x4_t vr = vraw[c];
          if (edge) vr &= seen;
          acc[b][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vr), pop[b], acc[b][c], 0, 0, 0);
        }
      }
    }
  };

  // (with keys of more than 128 and values of more than 128 a second set of tile registers no longer fits a wave's
  // registers: a decoded row behind 1,024 keys of 256 took 144 us with it)
  float sc[QB][8];
  if (HEADS && 2 * KC + VC <= 24) {
    // a decoded row's waves are few and each walks a chain of tiles: the next tile's loads fly while this one is worked
    u32x4_t k_even[2][KC], v_even[VC], k_odd[2][KC], v_odd[VC];
    if (tile_first <= tile_last) {
      load_keys(tile_first, k_even);
      load_values(tile_first, v_even);
    }
    for (int tile = tile_first; tile <= tile_last; tile += 2 * tile_step) {
      load_keys(tile + tile_step, k_odd);
      load_values(tile + tile_step, v_odd);
      score(tile, k_even, sc);
      gather(tile, sc, v_even);
      if (tile + tile_step > tile_last) break;
      load_keys(tile + 2 * tile_step, k_even);
      load_values(tile + 2 * tile_step, v_even);
      score(tile + tile_step, k_odd, sc);
      gather(tile + tile_step, sc, v_odd);
    }
  } else if (tile_first <= tile_last) {
    // the keys' registers are free once the scores are there, the values' once they are added: each then takes the next
    // tile's, which fly while the other half of the work is done
    u32x4_t k_now[2][KC], v_now[VC];
    load_keys(tile_first, k_now);
    load_values(tile_first, v_now);
    for (int tile = tile_first; tile <= tile_last; tile += tile_step) {
      score(tile, k_now, sc);
      load_keys(tile + tile_step, k_now);
      gather(tile, sc, v_now);
      load_values(tile + tile_step, v_now);
    }
  }
  // Shuffles, and not the moves of the loop: those want pairs of registers side by side, and for this one sum the loop's registers
  // were laid out anew and went to memory (portions of 32 rows a wave, 160 of them: 2,048 rows of heads of 128 with a sink 562 us
  // a layer, 91 so; decoded rows of heads of 256, 8 behind 2,048, 269 and 118).
#pragma unroll
  for (int b = 0; b < QB; ++b) {   // a row's sum: its four lanes' parts
    l_run[b] += __shfl_xor(l_run[b], 16, kWave);
    l_run[b] += __shfl_xor(l_run[b], 32, kWave);
  }

  if (HEADS && WAVES > 1) {
    // the waves' sums meet in LDS; wave w then finishes the chunks w, w + WAVES, ... of the value size
    f32x4_t* part = reinterpret_cast<f32x4_t*>(merge_lds);
    float* part_m = merge_lds + WAVES * n_vc * kWave * 4;
    float* part_l = part_m + WAVES * 16;
#pragma unroll
    for (int c = 0; c < VC; ++c)
      if (c < n_vc) part[(wave * n_vc + c) * kWave + lane] = acc[0][c];
    if (g == 0) {
      part_m[wave * 16 + n] = m_run[0];
      part_l[wave * 16 + n] = l_run[0];
    }
    __syncthreads();
    float m_all = sink;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) m_all = fmaxf(m_all, part_m[w * 16 + n]);
    float l_all = a.sink ? __builtin_amdgcn_exp2f(sink - m_all) : 0.f, f[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      f[w] = __builtin_amdgcn_exp2f(part_m[w * 16 + n] - m_all);
      l_all += part_l[w * 16 + n] * f[w];
    }
    if (!live[0]) return;
    const float inv_l = a.out_scale / l_all;
    bf16* orow = a.out + static_cast<int64_t>(row[0]) * a.o_stride + head * a.Dv;
    for (int c = wave; c < n_vc; c += WAVES) {
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const f32x4_t t = part[(w * n_vc + c) * kWave + lane];
        o[0] += t[0] * f[w]; o[1] += t[1] * f[w]; o[2] += t[2] * f[w]; o[3] += t[3] * f[w];
      }
      u32x2_t packed;
      packed[0] = pack_bf16x2(o[0] * inv_l, o[1] * inv_l);
      packed[1] = pack_bf16x2(o[2] * inv_l, o[3] * inv_l);
      *reinterpret_cast<u32x2_t*>(orow + 16 * c + 4 * g) = packed;
    }
    return;
  }
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    if (!live[b]) continue;
    float inv_l = a.out_scale / l_run[b];
    if (a.sink) {
      const float m_all = fmaxf(m_run[b], sink), kept = __builtin_amdgcn_exp2f(m_run[b] - m_all);
      inv_l = kept / (l_run[b] * kept + __builtin_amdgcn_exp2f(sink - m_all)) * a.out_scale;
    }
    bf16* orow = a.out + static_cast<int64_t>(row[b]) * a.o_stride + head * a.Dv;
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      if (c < n_vc) {
        u32x2_t packed;
        packed[0] = pack_bf16x2(acc[b][c][0] * inv_l, acc[b][c][1] * inv_l);
        packed[1] = pack_bf16x2(acc[b][c][2] * inv_l, acc[b][c][3] * inv_l);
        *reinterpret_cast<u32x2_t*>(orow + 16 * c + 4 * g) = packed;
      }
    }
  }
}

// Waves of 32 rows from which a prompt portion takes them rather than waves of 16: with fewer, more waves fill the chip
// better than fewer loads help (32 q heads of 128, window 1,024, 16 against 32 rows a wave: 640 rows, 672 such waves, 36
// and 45 us; 1,024 rows, 1,056 waves, 62 and 64; 1,150 rows 72 and 73; 1,250 rows 81 and 74; four portions of 300 rows 33
// and 32; 2,048 rows 136 and 89).
constexpr long long kCapTwoBlocks = 1024;
// From how many workgroups of 128 rows on (tokens times the q heads of a kv head; every segment ends one) heads of 128 go to the
// kernel whose waves share their tiles (attention_softcap_portions.h): with fewer, one-wave items spread over more of the chip.  32 q heads over 8
// kv heads, window 1,024, cap and penalty, this kernel / that one, us: 100 rows 11.5 / 13.1, 400 rows (112 of them) 22.7 / 23.2, 512 behind 3,000
// (136) 52.1 / 53.9, 300 beside eight decoded rows (144) 50 / 43, 640 (168) 36.9 / 31.0, 1,024 72 / 44, 2,048 110 / 66, 4,096 195 / 120.
// The same line for 32 q heads over 16 and 4 kv heads, 64 and 16 over 8, no window, no penalty and no cap: 0.97 to 1.00 of
// the time one step below it, 0.48 to 0.87 from there on.
constexpr long long kCapPortions = 144;
// Steps of short segments leave most rows of their workgroups empty, which costs more than shared tiles give while there are
// few keys to share: with two q heads a kv head (of which one-wave items hold as many as that kernel's waves) up to 224 keys
// where a workgroup has 64 rows and less, with more up to 96 keys where it has 80 and less (96 and 224 end classes of contexts that
// captured steps are told apart by).  This kernel / that one, us: 20 prompts of
// 16 tokens 10.2 / 11.5 (18.0 / 18.6 behind 200), 100 of 20 35.4 / 39.1, and over 16 kv heads 40 of 30 15.9 / 22.1, behind 100 28 / 35, behind 400 55 /
// 54, 100 of 8 30 / 44, 67 / 75 behind 200, 110 / 105 behind 400.  Decoded rows beside a portion, as good as empty workgroups all,
// gain by their keys: 32 of them behind 1,000 beside 20 tokens 81 / 47.
inline bool cap_portions_pay(long long tokens, int segments, int max_qlen, int max_keys, int group, int nkv) {
  const long long longest = (static_cast<long long>(max_qlen) * group + kCpRows - 1) / kCpRows;
  const long long most = tokens * group / kCpRows + segments, each = longest * segments;
  const long long blocks = most < each ? most : each;   // no fewer than there are
  if (blocks * nkv < kCapPortions) return false;
  const int few_keys = group == 2 ? 224 : 96;
  const bool empty = tokens * group <= (group == 2 ? 64 : 80) * blocks;
  return max_keys == 0 || max_keys > few_keys || !empty;
}
constexpr int kCapSplitWaves = 8;   // waves that share the keys of a decoded row
constexpr int kCapLdsMost = 160 * 1024;   // LDS of a gfx950 compute unit: no workgroup can ask for more

// What a workgroup may ask for on this device (never more than kCapLdsMost), asked once.
inline int cap_lds_limit() {
  static int limit = 0;
  if (limit == 0) {
    int dev = 0, value = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&value, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && value > 0)
      limit = value < kCapLdsMost ? value : kCapLdsMost;
    else
      limit = 64 * 1024;
  }
  return limit;
}

}  // namespace arle

// Bytes of LDS that a workgroup of the matrix-core kernel may use on this device (the return value, not an error code).
extern "C" int arle_attn_softcap_lds_limit() { return cap_lds_limit(); }

// Whether portions of heads of 128 of a step of these sizes go to the kernel whose waves share their tiles, as far as sizes decide it.
extern "C" int arle_attn_softcap_shares_tiles(int tokens, int segments, int max_qlen, int max_keys, int nq, int nkv) {
  return nkv > 0 && cap_portions_pay(tokens, segments, max_qlen, max_keys, nq / nkv, nkv);
}

// bfloat16 only.  Dk a multiple of 8 up to 256, Dv a multiple of 16 up to 256, page_size a multiple of 16, rows of
// q and out 16-byte aligned (strides multiples of 8).  heads_mode: every segment is one row.
// tokens: rows of all segments; max_qlen: rows of the longest one.  max_keys: the longest context with its rows, 0 where the caller
// does not know it (a choice between kernels only).
extern "C" int arle_attn_softcap_mfma(const void* q, long long q_stride, void* out, long long o_stride,
                                      const void* k_pages, const void* v_pages, const int* block_table,
                                      int table_stride, const int* seg_row0, const int* seg_slot, const int* seg_start,
                                      int segments, int tokens, int max_qlen, int max_keys, int heads_mode, int nq, int nkv, int Dk, int Dv,
                                      int page_size, float scale, float cap, const void* r1, const void* r2,
                                      int r_dtype, int window, int chunk, const void* sink, int sink_dtype,
                                      int keep_first, float out_scale, void* stream) {
  if (segments == 0) return 0;
  // (kept first keys go with a window alone: under the chunk rule a row's chunk would have to hold them)
  if (Dk % 8 || Dk > 256 || Dv % 16 || Dv > 256 || page_size % 16 || nkv < 1 || nq % nkv || nq > 65535 ||
      window < 0 || chunk < 0 || keep_first < 0 || (keep_first > 0 && (window == 0 || chunk > 0)))
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const CapArgs a{static_cast<const bf16*>(q), q_stride, static_cast<bf16*>(out), o_stride,
                  static_cast<const bf16*>(k_pages), static_cast<const bf16*>(v_pages), block_table, table_stride,
                  seg_row0, seg_slot, seg_start, segments, nq, nkv, Dk, Dv, page_size, scale, cap, r1, r2, r_dtype, window,
                  chunk, sink, sink_dtype, heads_mode ? kCapSplitWaves * ((Dv / 16) * kWave * 4 + 32) : 0, keep_first,
                  out_scale};
  // pages an item can see: its rows' windows (or everything the block table maps) and the tiles' rounding to 32 keys;
  // nothing of a step's lengths, so that a captured launch holds for every later step of its shape
  const long long mapped = static_cast<long long>(table_stride) * page_size;
  const int span = window > 0 && chunk > 0 ? (window < chunk ? window : chunk) : (window > 0 ? window : chunk);
  const long long keys_seen = (span > 0 && span + 16 < mapped ? span + 16 : mapped) + 64;
  const size_t page_bytes = (static_cast<size_t>(keys_seen) / page_size + 2 + (keep_first + 31) / page_size + 2) * sizeof(int);
  if (page_bytes > 48 * 1024) return static_cast<int>(hipErrorInvalidValue);
  const int size = (Dk + 1) / 2 > Dv ? (Dk + 1) / 2 : Dv;   // Dk counts half: a chunk of keys is 32 wide, of values 16
  const int group = nq / nkv;
  const int head_waves = group % 4 == 0 ? 4 : (group % 2 == 0 ? 2 : 1);   // q heads of one kv head that share a workgroup
  const size_t merge_bytes = static_cast<size_t>(kCapSplitWaves) * ((Dv / 16) * kWave * 4 + 32) * sizeof(float) + page_bytes;
  if (heads_mode && merge_bytes > static_cast<size_t>(cap_lds_limit())) return static_cast<int>(hipErrorInvalidValue);
  const int row_blocks = tokens / 16 + segments;                    // no fewer than the sixteen-row blocks of all segments
  const int wide_blocks = (row_blocks - segments) / 2 + segments;   // as row_blocks, of 32 rows
  const bool two = Dk <= 128 && Dv <= 128 && static_cast<long long>(wide_blocks) * nq >= kCapTwoBlocks &&
                   page_bytes + 2 * sizeof(int) <= 48 * 1024;
  if (!heads_mode && cap_portions_take(a) && cap_portions_pay(tokens, segments, max_qlen, max_keys, group, nkv)) {
    const int blocks = static_cast<int>(static_cast<long long>(tokens) * group / kCpRows) + segments;   // no fewer than there are
    if (r1 == nullptr) return launch_cap_portions<0>(a, blocks, s);
    return group == kCpTableGroup && window > 0 && window <= kCpTableMax ? launch_cap_portions<1>(a, blocks, s) : launch_cap_portions<2>(a, blocks, s);
  }
#define ARLE_CAP_ROWS(KC, VC, QB, BLOCKS, BYTES)                                                                   \
  do {                                                                                                             \
    constexpr int kQb = KC <= 4 && VC <= 8 ? QB : 1;                                                               \
    if (head_waves == 4)                                                                                           \
      attn_softcap_mfma_kernel<KC, VC, false, 4, kQb><<<dim3(BLOCKS, nq / 4), 4 * kWave, BYTES, s>>>(a);           \
    else if (head_waves == 2)                                                                                      \
      attn_softcap_mfma_kernel<KC, VC, false, 2, kQb><<<dim3(BLOCKS, nq / 2), 2 * kWave, BYTES, s>>>(a);           \
    else                                                                                                           \
      attn_softcap_mfma_kernel<KC, VC, false, 1, kQb><<<dim3(BLOCKS, nq), kWave, BYTES, s>>>(a);                   \
  } while (0)
#define ARLE_CAP(KC, VC)                                                                                           \
  do {                                                                                                             \
    if (heads_mode) {                                                                                              \
      static OnceADevice asked;                                                                                    \
      if (merge_bytes > 48 * 1024) {                                                                               \
        const int most = kCapSplitWaves * (VC * kWave * 4 + 32) * 4 + 48 * 1024;                                   \
        if (const int e = ask_lds(asked, most < cap_lds_limit() ? most : cap_lds_limit(),                          \
                                  {reinterpret_cast<const void*>(&attn_softcap_mfma_kernel<KC, VC, true, kCapSplitWaves, 1>)})) \
          return e;                                                                                                \
      }                                                                                                            \
      attn_softcap_mfma_kernel<KC, VC, true, kCapSplitWaves, 1>                                                    \
          <<<dim3(segments, nkv * ((group + 15) / 16)), kCapSplitWaves * kWave, merge_bytes, s>>>(a);                                    \
    }                                                                                                              \
    else if (two)                                                                                                  \
      ARLE_CAP_ROWS(KC, VC, 2, wide_blocks, page_bytes + 2 * sizeof(int));                                         \
    else                                                                                                           \
      ARLE_CAP_ROWS(KC, VC, 1, row_blocks, page_bytes);                                                            \
  } while (0)
  if (size <= 64) {
    ARLE_CAP(4, 4);
  } else if (Dk <= 128 && Dv <= 128) {
    ARLE_CAP(4, 8);
  } else if (size <= 128) {
    ARLE_CAP(8, 8);
  } else if (Dv <= 192) {
    ARLE_CAP(8, 12);
  } else {
    ARLE_CAP(8, 16);
  }
#undef ARLE_CAP
#undef ARLE_CAP_ROWS
  return launch_status();
}
