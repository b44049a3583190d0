// The mLSTM matrix memory (see mlstm.hip for the recurrence) over chunks of 64 rows, for prompt portions: a chunk's rows meet
// each other in matrix products and the state moves once a chunk.  With b_t the sum of the chunk's log forget gates up to
// row t, e_s = i_s - b_s and m_0 the running maximum in front of the chunk,
//
//   M_t = max(m_0, max_(s<=t) e_s),  m_t = b_t + M_t
//   numerator_t = sum_(s<=t) exp(e_s - M_t) (q_t . k_s) v_s + exp(m_0 - M_t) S_0^T q_t     (n_t . q_t alike, with 1 for v_s)
//   S_end = exp(m_0 + b_end - m_end) S_0 + sum_s exp(e_s + b_end - m_end) k_s v_s^T          (n_end alike)
//
// Everything is 32-bit: the products run on the float32 matrix instructions (157 TFLOP/s, a chunk and head of 128 x 128 is
// 6 MFLOP), so operands, weights and state keep what the token-by-token kernels keep.  The sums b are made in 64 bits and
// e, M and b travel as pairs of floats: an exponent is the difference of two of them, and a chunk's b may be a thousand
// times the difference that counts.
//
//   mlstm_chunk_gates   a wave a (chunk, head): gates, b, e and the running maximum of e by scans over the lanes
//   mlstm_chunk_carry   a workgroup a (request, head, 32 columns of Dv) walks the request's chunks with its part of S in
//                       accumulators, leaves S_0, n_0 and m_0 of every chunk; the next chunk's k and v are fetched meanwhile
//   mlstm_chunk_sums,   the same for longer requests in two kernels without a chain of products: see there
//   mlstm_chunk_scan
//   mlstm_chunk_out     a workgroup a (chunk, head): scores, weights, both products, the denominator, the head norm, the
//                       norm weight and the output gate
//
// Measured on MI355X, 2,048 rows, 20 heads, D = Dv = 128, us a layer: 5 + 47 + 50 (5 + 91 + 50 with the walk) where the
// token-by-token kernels take 125 (gates) + 708 (memory) + 18 (output); the error of a layer's output against 64 bits is the same (2e-7 to 6e-6 either way).
// A NaN or an infinity in a row's v spoils that row and the later ones, as token by token (where an infinity meets a
// state's column with both signs).  The second product would carry it to the chunk's earlier rows too, as a weight of zero
// times it: it takes zeros for such values, and the rows from the first one on are made NaN behind it.
#include "chunks.h"
#include "common.h"

#include <type_traits>

namespace arle {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct ChunkRow {   // of a row and head: each value is hi + lo
  float e_hi, e_lo, top_hi, top_lo, b_hi, b_lo;   // e; max_(s<=t) e_s inside the chunk; b
};
struct ChunkEnd {   // of a chunk and head
  double b, top;    // b of the last row, the largest e
};

__device__ __forceinline__ float log_sigmoid(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

__device__ __forceinline__ void split_double(double v, float& hi, float& lo) {
  hi = static_cast<float>(v);
  lo = v == -INFINITY ? 0.f : static_cast<float>(v - static_cast<double>(hi));
}

struct MlstmChunkArgs {
  const float* q;
  const float* k;
  const float* v;
  const float* gate;
  int64_t row_stride;      // of q, k, v and gate, in elements
  const float* gates;
  int64_t gates_stride;
  const float* bias_i;
  const float* bias_f;
  float cap, q_scale, eps;
  float* s_state;
  float* n_state;
  float* m_state;
  const int* seg_row0;
  const int* seg_slot;
  int segments, items, H, D, Dv;
  ChunkRow* rows;          // [items][H][64]
  ChunkEnd* ends;          // [items][H]
  float* s0;               // [items][H][D][Dv]
  float* n0;               // [items][H][D]
  float* m0;               // [items][H][2]: in front of the chunk, behind it
  const void* weight;
  int w_dtype;
  void* out;
  int out_dtype;
};

__global__ __launch_bounds__(kWave) void mlstm_chunk_gates_kernel(const MlstmChunkArgs a) {
  const int item = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const ChunkAt c = find_chunk(a.seg_row0, a.segments, item);
  if (c.rows == 0) return;
  const int64_t t = c.row0 + min(lane, c.rows - 1);
  const float inv_cap = 1.0f / a.cap;
  const float it = a.cap * tanhf((a.gates[t * a.gates_stride + h] + a.bias_i[h]) * inv_cap);
  const float ft = log_sigmoid(a.cap * tanhf((a.gates[t * a.gates_stride + a.H + h] + a.bias_f[h]) * inv_cap));
  const bool live = lane < c.rows;
  double b = live ? static_cast<double>(ft) : 0.0;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double below = __shfl_up(b, off, kWave);
    if (lane >= off) b += below;
  }
  const double e = live ? static_cast<double>(it) - b : -INFINITY;
  double top = e;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double below = __shfl_up(top, off, kWave);
    if (lane >= off) top = fmax(top, below);
  }
  ChunkRow r;
  split_double(e, r.e_hi, r.e_lo);
  split_double(top, r.top_hi, r.top_lo);
  split_double(b, r.b_hi, r.b_lo);
  const int64_t at = static_cast<int64_t>(item) * a.H + h;
  a.rows[at * kChunkRows + lane] = r;
  if (lane == kWave - 1) a.ends[at] = ChunkEnd{b, top};
}

// A wave a tile of 32 rows of S (d) x 32 columns; nothing is shared between the waves but what the L1 holds.  Bound by the
// chain of chunks: 2.7 us each, of which the products are 0.9 (operands through LDS by 16-byte loads instead, with the
// barriers that takes: 4.2 us).
template <int KD>
__global__ __launch_bounds__(KD* kWave) void mlstm_chunk_carry_kernel(const MlstmChunkArgs a) {
  __shared__ float weights[KD][kChunkRows];
  constexpr int D = 32 * KD;
  const int seg = blockIdx.x, h = blockIdx.y, z = blockIdx.z;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, i = lane & 31, half = lane >> 5;
  const int Dv = a.Dv, H = a.H;
  const int row0 = a.seg_row0[seg], rows = a.seg_row0[seg + 1] - row0;
  if (rows <= 0) return;
  int item = 0;
  for (int s = 0; s < seg; ++s) item += (a.seg_row0[s + 1] - a.seg_row0[s] + kChunkRows - 1) / kChunkRows;
  const int chunks = (rows + kChunkRows - 1) / kChunkRows;
  const int64_t slot = a.seg_slot[seg];
  float* s_state = a.s_state + ((slot * H + h) * D + 32 * wave) * Dv + 32 * z;
  float* n_state = a.n_state + (slot * H + h) * D + 32 * wave;
  auto d_of = [&](int r) { return 8 * (r / 4) + 4 * half + r % 4; };    // the row of the tile that register r holds

  f32x16 S;
#pragma unroll
  for (int r = 0; r < 16; ++r) S[r] = s_state[static_cast<int64_t>(d_of(r)) * Dv + i];
  float n = n_state[i];
  float m = a.m_state[slot * H + h];

  // what a chunk brings; step j takes its rows j (lower half of the lanes) and j + 32 (upper half)
  struct Brought {
    float k[32], v[32];
    ChunkEnd end;
    float2 e;        // e of row `lane`, as a pair
  };
  const float* kp = a.k + static_cast<int64_t>(h) * D + 32 * wave + i;
  const float* vp = a.v + static_cast<int64_t>(h) * Dv + 32 * z + i;
  auto fetch = [&](int c, Brought& to) {
    const int64_t at = static_cast<int64_t>(item + c) * H + h;
    to.end = a.ends[at];
    to.e = *reinterpret_cast<const float2*>(a.rows + at * kChunkRows + lane);
    const int64_t first = (row0 + c * kChunkRows) * a.row_stride;
    const float* kc = kp + first;
    const float* vc = vp + first;
    const int last = rows - 1 - c * kChunkRows;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int64_t t = min(j + 32 * half, last) * a.row_stride;     // rows past the chunk's end weigh nothing
      to.k[j] = kc[t];
      to.v[j] = vc[t];
    }
  };
  auto walk = [&](int c, Brought& now, Brought& next) {
    const int64_t at = static_cast<int64_t>(item + c) * H + h;
    float* s0 = a.s0 + (at * D + 32 * wave) * Dv + 32 * z;
#pragma unroll
    for (int r = 0; r < 16; ++r) s0[static_cast<int64_t>(d_of(r)) * Dv + i] = S[r];
    const double b = now.end.b;
    const float m_end = static_cast<float>(b + fmax(static_cast<double>(m), now.end.top));
    const float keep = expf(static_cast<float>(static_cast<double>(m) + b - static_cast<double>(m_end)));
    // rows that are not there have e = -inf and weigh 0
    weights[wave][lane] = expf(static_cast<float>(static_cast<double>(now.e.x) + static_cast<double>(now.e.y) + b -
                                                  static_cast<double>(m_end)));
    if (z == 0) {
      if (half == 0) a.n0[at * D + 32 * wave + i] = n;
      if (tid == 0) {
        a.m0[at * 2] = m;
        a.m0[at * 2 + 1] = m_end;
      }
    }
    m = m_end;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float n_sum = 0.f;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const float w = weights[wave][j + 32 * half];
      n_sum = fmaf(w, now.k[j], n_sum);
      now.v[j] *= w;
    }
    if (c + 1 < chunks) fetch(c + 1, next);
#pragma unroll
    for (int r = 0; r < 16; ++r) S[r] *= keep;
#pragma unroll
    for (int j = 0; j < 32; ++j) S = __builtin_amdgcn_mfma_f32_32x32x2f32(now.k[j], now.v[j], S, 0, 0, 0);
    n_sum += __shfl_xor(n_sum, 32, kWave);
    n = fmaf(n, keep, n_sum);
    __builtin_amdgcn_wave_barrier();
  };
  Brought even, odd;
  fetch(0, even);
  for (int c = 0; c < chunks; c += 2) {
    walk(c, even, odd);
    if (c + 1 < chunks) walk(c + 1, odd, even);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) s_state[static_cast<int64_t>(d_of(r)) * Dv + i] = S[r];
  if (z == 0 && half == 0) n_state[i] = n;      // m goes back in the last kernel: other workgroups of the head may still read it here
}

// The same walk for requests of several chunks, in two kernels: the chunks' own sums side by side, then the states in front
// of them.  With top_c the largest e of chunk c, U_c = sum_s exp(e_s - top_c) k_s v_s^T needs nothing of the chunks before it,
// and S_(c+1) = exp(m_c + b_c - m_(c+1)) S_c + exp(top_c + b_c - m_(c+1)) U_c is element by element.
//
// The sums: a workgroup a (chunk, head), a wave 32 rows (d) of U, 32 columns after another.  The products of a chunk and head
// are 2 MFLOP; what bounds it is the fetch of k and v, and U on its way out.
template <int KD>
__global__ __launch_bounds__(KD* kWave) void mlstm_chunk_sums_kernel(const MlstmChunkArgs a) {
  constexpr int D = 32 * KD;
  __shared__ float weights[KD][kChunkRows];
  const int item = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, i = lane & 31, half = lane >> 5;
  const ChunkAt c = find_chunk(a.seg_row0, a.segments, item);
  if (c.rows == 0) return;                    // the whole workgroup
  const int Dv = a.Dv, H = a.H;
  const int64_t at = static_cast<int64_t>(item) * H + h;
  // rows that are not there have e = -inf and weigh 0
  const float2 e = *reinterpret_cast<const float2*>(a.rows + at * kChunkRows + lane);
  const double top = a.ends[at].top;
  const float* kp = a.k + static_cast<int64_t>(h) * D + 32 * wave + i;
  const float* vp = a.v + static_cast<int64_t>(h) * Dv + i;
  float k[32], v[2][32];
  auto row = [&](int j) { return static_cast<int64_t>(c.row0 + min(j + 32 * half, c.rows - 1)) * a.row_stride; };
#pragma unroll
  for (int j = 0; j < 32; ++j) k[j] = kp[row(j)];
#pragma unroll
  for (int j = 0; j < 32; ++j) v[0][j] = vp[row(j)];
  weights[wave][lane] = expf(static_cast<float>(static_cast<double>(e.x) + static_cast<double>(e.y) - top));
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float n_sum = 0.f;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    k[j] *= weights[wave][j + 32 * half];
    n_sum += k[j];
  }
  n_sum += __shfl_xor(n_sum, 32, kWave);
  if (half == 0) a.n0[at * D + 32 * wave + i] = n_sum;
  float* u = a.s0 + (at * D + 32 * wave) * Dv + i;
#pragma unroll
  for (int z = 0; z < 4; ++z) {
    if (32 * z < Dv) {
      if (32 * z + 32 < Dv) {
#pragma unroll
        for (int j = 0; j < 32; ++j) v[(z + 1) & 1][j] = vp[row(j) + 32 * z + 32];
      }
      f32x16 U;
#pragma unroll
      for (int r = 0; r < 16; ++r) U[r] = 0.f;
#pragma unroll
      for (int j = 0; j < 32; ++j) U = __builtin_amdgcn_mfma_f32_32x32x2f32(k[j], v[z & 1][j], U, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; ++r) u[static_cast<int64_t>(8 * (r / 4) + 4 * half + r % 4) * Dv + 32 * z] = U[r];
    }
  }
}

// The states: a thread four elements of a (request, head)'s S through all its chunks, whose sums it fetches kScanAhead chunks
// ahead and whose places take S_0 (the last blockIdx.z: n, an element a thread).  Bound by reading U and writing S_0, 84 MB
// a layer at 2,048 rows of 20 heads.
constexpr int kScanThreads = 256, kScanAhead = 8;
// Sums and scan take the walk's place for requests of kSumsMinRows and more, unless the walk keeps the matrix cores busy: a wave of
// it is a chain of products, so it is its waves for every SIMD of the chip (1,024) that decide, and requests of unequal length leave
// it with a tail.  MI355X, all kernels of a layer, us, walk / sums and scan, by the walk's waves:
//   320 (20 heads of 128, one request) 256 rows 37.8 / 39.5, 384 43.3 / 42.7, 512 49.5 / 44.6, 1,024 81 / 64, 2,048 134 / 92; 128 (8 heads
//     of 128) 384 rows 40.0 / 36.3, 2,048 120 / 65; 512 (4 heads of 128, eight requests) 384 rows 45.3 / 44.7, 1,024 92 / 80, 2,048
//     150 / 123; 512 (8 heads of 64, 16) 384 rows 53.1 / 55.1, 512 70.6 / 69.8, 1,024 117 / 111
//   640 (20 heads, two) 384 rows 54.3 / 59.4, 512 60.0 / 62.4, 640 67.3 / 66.2, 2,048 168 / 154
//   1,024 (8 heads of 128, eight) 384 rows 56.6 / 65.7, 1,024 113 / 123, 2,048 223 / 254; (8 heads of 64, 32) 384 rows 78.9 / 89.9
//   1,280 (20 heads, four), the walk's second turn mostly empty: 384 rows 83.2 / 78.7, 512 94.3 / 89.2, 2,048 323 / 307; 1,536 (8 heads,
//     12) 600 rows 126 / 121
//   2,048 and more: (8 heads, 16) 384 rows 91.8 / 101.8, 1,024 221 / 250; (20 heads, 16) 1,024 rows 535 / 589
//   unequal requests, 20 heads: 4,631 rows in 16 up to 681 248 / 206, 3,584 in 8 up to 798 185 / 154, 2,471 in 4 up to 883 139 / 118,
//     7,505 in 16 up to 584 316 / 315, 3,765 in 3 up to 1,380 137 / 145; 8 heads: 4,100 in 8 up to 700 81 / 88, 4,631 in 16 112 / 95
constexpr int kSumsMinRows = 384, kSumsMinRowsFuller = 640, kWalkWaves = 1024;

static bool sums_preferred(long long tokens, long long segments, long long longest, int H, int D, int Dv) {
  if (longest < kSumsMinRows) return false;
  if (4 * tokens <= 3 * segments * longest) return true;      // far from equal
  const long long waves = segments * H * (Dv / 32) * (D / 32), turns = (waves + kWalkWaves - 1) / kWalkWaves;
  if (turns > 1) return 4 * waves <= 3 * turns * kWalkWaves;
  return waves <= kWalkWaves / 2 || (waves <= kWalkWaves * 5 / 8 && longest >= kSumsMinRowsFuller);
}

__global__ __launch_bounds__(kScanThreads) void mlstm_chunk_scan_kernel(const MlstmChunkArgs a, int D) {
  const int seg = blockIdx.x, h = blockIdx.y, z = blockIdx.z, tid = threadIdx.x;
  const int Dv = a.Dv, H = a.H;
  const int row0 = a.seg_row0[seg], rows = a.seg_row0[seg + 1] - row0;
  if (rows <= 0) return;
  int item = 0;
  for (int s = 0; s < seg; ++s) item += (a.seg_row0[s + 1] - a.seg_row0[s] + kChunkRows - 1) / kChunkRows;
  const int chunks = (rows + kChunkRows - 1) / kChunkRows;
  const int64_t slot = a.seg_slot[seg], first = static_cast<int64_t>(item) * H + h;
  float m = a.m_state[slot * H + h];      // it goes back in the last kernel: other workgroups of the head may still read it here
  auto walk = [&](auto* state, auto* sums, int64_t a_chunk, bool tells, auto scaled) {
    using T = std::remove_reference_t<decltype(*state)>;
    T S = *state, ahead[kScanAhead];
    ChunkEnd ends[kScanAhead];
#pragma unroll
    for (int j = 0; j < kScanAhead; ++j) {
      const int c = min(j, chunks - 1);
      ahead[j] = sums[c * a_chunk];
      ends[j] = a.ends[first + static_cast<int64_t>(c) * H];
    }
    for (int c0 = 0; c0 < chunks; c0 += kScanAhead) {
#pragma unroll
      for (int j = 0; j < kScanAhead; ++j) {
        const int c = c0 + j;
        if (c < chunks) {
          const T u = ahead[j];
          const ChunkEnd end = ends[j];
          // (nothing past the last chunk: the places in front of this one hold S_0 by now, not sums)
          if (const int next = c + kScanAhead; next < chunks) {
            ahead[j] = sums[next * a_chunk];
            ends[j] = a.ends[first + static_cast<int64_t>(next) * H];
          }
          const float m_end = static_cast<float>(end.b + fmax(static_cast<double>(m), end.top));
          const float keep = expf(static_cast<float>(static_cast<double>(m) + end.b - static_cast<double>(m_end)));
          const float take = expf(static_cast<float>(end.top + end.b - static_cast<double>(m_end)));
          sums[c * a_chunk] = S;
          if (tells) {
            const int64_t at = first + static_cast<int64_t>(c) * H;
            a.m0[at * 2] = m;
            a.m0[at * 2 + 1] = m_end;
          }
          S = scaled(S, keep, u, take);
          m = m_end;
        }
      }
    }
    *state = S;
  };
  if (z + 1 < static_cast<int>(gridDim.z)) {
    const int e = z * kScanThreads + tid;
    if (e >= D * Dv / 4) return;
    walk(reinterpret_cast<float4*>(a.s_state + (slot * H + h) * D * Dv) + e, reinterpret_cast<float4*>(a.s0 + first * D * Dv) + e,
         static_cast<int64_t>(H) * D * Dv / 4, z == 0 && tid == 0, [](float4 S, float keep, float4 u, float take) {
           return float4{fmaf(S.x, keep, u.x * take), fmaf(S.y, keep, u.y * take), fmaf(S.z, keep, u.z * take), fmaf(S.w, keep, u.w * take)};
         });
  } else if (tid < D) {
    walk(a.n_state + (slot * H + h) * D + tid, a.n0 + first * D + tid, static_cast<int64_t>(H) * D, false,
         [](float S, float keep, float u, float take) { return fmaf(S, keep, u * take); });
  }
}

constexpr int kOutWaves = 4;

// What bounds it: a chunk is 195 KB of loads, then 240 float32 matrix instructions a wave, then its rows' ends, with barriers
// between, so other workgroups of the compute unit have to fill the waits: three fit (k through LDS in halves of its columns, v and
// the gate fetched when the registers of what came before are free; two before, with 69 KB of LDS and 244 registers), and a
// prompt of 2,048 rows and 20 heads, 660 of them, is one turn of the chip instead of one and a third.  No load stands behind a
// wait that it does not need, the weight comes once through LDS.  65.9 -> 50.5 us a layer at that size.
template <int KD>
__global__ __launch_bounds__(kOutWaves* kWave, 3) void mlstm_chunk_out_kernel(const MlstmChunkArgs a) {
  constexpr int D = 32 * KD;
  constexpr int kQPitch = D + 2;              // a pitch of 2 modulo 64: the 32 rows and two columns of an operand meet 64 banks
  constexpr int kPPitch = kChunkRows + 2;
  constexpr int kOPitch = 128 + 2;
  constexpr int kQFloats = kChunkRows * (kQPitch > kOPitch ? kQPitch : kOPitch);   // q, later the outputs
  constexpr int kKPitch = D / 2 + 2;
  constexpr int kKFloats = kChunkRows * (kKPitch > kPPitch ? kKPitch : kPPitch);   // half of k's columns, then the other, later the weighted scores
  __shared__ __align__(16) float q_lds[kQFloats];
  __shared__ __align__(16) float k_lds[kKFloats];
  __shared__ __align__(16) float w_lds[128];   // the norm's weight
  __shared__ float n_lds[D], inter[kChunkRows], inv_den[kChunkRows];
  __shared__ ChunkRow row_lds[kChunkRows];
  const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid % kWave, wave = tid / kWave, i = lane & 31, half = lane >> 5;
  const ChunkAt c = find_chunk(a.seg_row0, a.segments, item);
  if (c.rows == 0) return;                    // the whole workgroup
  const int Dv = a.Dv, H = a.H;
  const int64_t at = static_cast<int64_t>(item) * H + h;
  const float m0 = a.m0[at * 2];
  const bool has_cols = 32 * wave < Dv;       // the wave's 32 columns of Dv

  float4 kh[2][KD];
#pragma unroll
  for (int x = 0; x < 2 * KD; ++x) {
    const int e = tid + (x % KD) * (kOutWaves * kWave), r = e / (D / 8), d = (e % (D / 8)) * 4 + (x / KD) * (D / 2);
    kh[x / KD][x % KD] = ld4<float>(a.k + (c.row0 + min(r, c.rows - 1)) * a.row_stride + static_cast<int64_t>(h) * D + d);
  }
  float4 qh[2 * KD];
#pragma unroll
  for (int x = 0; x < 2 * KD; ++x) {
    const int e = tid + x * (kOutWaves * kWave), r = e / (D / 4), d = (e % (D / 4)) * 4;
    qh[x] = ld4<float>(a.q + (c.row0 + min(r, c.rows - 1)) * a.row_stride + static_cast<int64_t>(h) * D + d);
  }
  // (loads without a condition around them: one under a condition is waited for on the spot)
  const float n_mine = a.n0[at * D + min(tid, D - 1)];
  const ChunkRow row_mine = a.rows[at * kChunkRows + tid % kChunkRows];
  const float w_mine = load_as_float(a.weight, a.w_dtype, static_cast<int64_t>(h) * Dv + min(tid, Dv - 1));
  auto put_keys = [&](const float4 (&from)[KD]) {
#pragma unroll
    for (int x = 0; x < KD; ++x) {
      const int e = tid + x * (kOutWaves * kWave);
      float* kd = k_lds + e / (D / 8) * kKPitch + (e % (D / 8)) * 4;
      *reinterpret_cast<float2*>(kd) = float2{from[x].x, from[x].y};
      *reinterpret_cast<float2*>(kd + 2) = float2{from[x].z, from[x].w};
    }
  };
#pragma unroll
  for (int x = 0; x < 2 * KD; ++x) {
    const int e = tid + x * (kOutWaves * kWave);
    const float4 qv = qh[x];
    float* qd = q_lds + e / (D / 4) * kQPitch + (e % (D / 4)) * 4;
    *reinterpret_cast<float2*>(qd) = float2{qv.x * a.q_scale, qv.y * a.q_scale};
    *reinterpret_cast<float2*>(qd + 2) = float2{qv.z * a.q_scale, qv.w * a.q_scale};
  }
  put_keys(kh[0]);
  if (tid < Dv) w_lds[tid] = w_mine;
  if (tid < D) n_lds[tid] = n_mine;
  if (tid < kChunkRows) {
    const ChunkRow r = row_mine;
    ChunkRow kept = r;
    // M_t = max(m_0, top_t), as a pair
    if (!(r.top_hi > m0 || (r.top_hi == m0 && r.top_lo > 0.f))) kept.top_hi = m0, kept.top_lo = 0.f;
    row_lds[tid] = kept;
    inter[tid] = expf((m0 - kept.top_hi) - kept.top_lo);
  }
  __builtin_amdgcn_sched_barrier(0);
  // the wave's operands of the state leave for their registers, to be there behind the scores
  float s0[D / 2];
  {
    const float* sp = a.s0 + at * D * Dv + (has_cols ? 32 * wave : 0) + i + half * Dv;
#pragma unroll
    for (int j = 0; j < D / 2; ++j) s0[j] = sp[static_cast<int64_t>(2 * j) * Dv];
  }
  __syncthreads();

  // scores of the wave's quadrant: rows 32 rt .., keys 32 ct ..; nothing of the upper right one is seen
  const int rt = wave >> 1, ct = wave & 1;
  f32x16 p;
#pragma unroll
  for (int r = 0; r < 16; ++r) p[r] = 0.f;
  const bool seen = !(rt == 0 && ct == 1);
  const float* qa = q_lds + (32 * rt + i) * kQPitch + half;
  const float* kb = k_lds + (32 * ct + i) * kKPitch + half;
  if (seen) {
#pragma unroll 8
    for (int j = 0; j < D / 4; ++j) p = __builtin_amdgcn_mfma_f32_32x32x2f32(qa[2 * j], kb[2 * j], p, 0, 0, 0);
  }
  __syncthreads();   // the first half of k has been read
  put_keys(kh[1]);
  __syncthreads();
  if (seen) {
#pragma unroll 8
    for (int j = 0; j < D / 4; ++j) p = __builtin_amdgcn_mfma_f32_32x32x2f32(qa[D / 2 + 2 * j], kb[2 * j], p, 0, 0, 0);
    const ChunkRow key = row_lds[32 * ct + i];
    const int s = 32 * ct + i;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int t = 32 * rt + 8 * (r / 4) + 4 * half + r % 4;
      const float w = expf((key.e_hi - row_lds[t].top_hi) + (key.e_lo - row_lds[t].top_lo));
      p[r] = s <= t ? p[r] * w : 0.f;
    }
  }
  // four threads a row from here on: q . n_0 now
  const int my_row = tid >> 2, part = tid & 3;
  const int64_t my_t = c.row0 + min(my_row, c.rows - 1);
  float qn = 0.f;
#pragma unroll 8
  for (int d = part; d < D; d += 4) qn = fmaf(q_lds[my_row * kQPitch + d], n_lds[d], qn);
  // the wave's operands of v, to be there behind the state's product (and neither their addresses nor the check of their values earlier:
  // there are no registers for them)
  float vr[32];
  __builtin_amdgcn_sched_barrier(0);
  {
    const float* vp = a.v + (c.row0 + half) * a.row_stride + static_cast<int64_t>(h) * Dv + (has_cols ? 32 * wave : 0) + i;
    const int most = c.rows - 1 - half;      // -1 in the second half of a chunk of one row: the row in front again
#pragma unroll
    for (int j = 0; j < 32; ++j) vr[j] = vp[min(2 * j, most) * a.row_stride];
  }
  __syncthreads();   // k has been read
#pragma unroll
  for (int r = 0; r < 16; ++r) k_lds[(32 * rt + 8 * (r / 4) + 4 * half + r % 4) * kPPitch + 32 * ct + i] = p[r];
  __syncthreads();
  {
    float nq = qn * inter[my_row];
#pragma unroll
    for (int s = part; s < kChunkRows; s += 4) nq += k_lds[my_row * kPPitch + s];
    nq += __shfl_xor(nq, 1, kWave);
    nq += __shfl_xor(nq, 2, kWave);
    if (part == 0) {
      const ChunkRow r = row_lds[my_row];
      const float m_t = (r.top_hi + r.b_hi) + (r.top_lo + r.b_lo);
      inv_den[my_row] = 1.0f / (fmaxf(fabsf(nq), expf(-m_t)) + 1e-6f);
    }
  }

  f32x16 acc[2];
  if (has_cols) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    }
    const float* q0 = q_lds + i * kQPitch + half;
#pragma unroll
    for (int j = 0; j < D / 2; ++j) {
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(q0[2 * j], s0[j], acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(q0[32 * kQPitch + 2 * j], s0[j], acc[1], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][r] *= inter[32 * t + 8 * (r / 4) + 4 * half + r % 4];
    __builtin_amdgcn_sched_barrier(0);
    const float* p0 = k_lds + i * kPPitch + half;
    float check = 0.f;        // NaN as soon as a value is no finite number
#pragma unroll
    for (int j = 0; j < 32; ++j) check = fmaf(vr[j], 0.f, check);
    int spoilt = kChunkRows;  // the first row of this column that holds such a value
    if (__any(check != 0.f)) {
#pragma unroll
      for (int j = 31; j >= 0; --j)
        if (!__builtin_isfinite(vr[j])) spoilt = 2 * j, vr[j] = 0.f;
      if (spoilt < kChunkRows) spoilt += half;
      spoilt = min(spoilt, __shfl_xor(spoilt, 32, kWave));
    }
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      if (j < 16) acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(p0[2 * j], vr[j], acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(p0[32 * kPPitch + 2 * j], vr[j], acc[1], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * t + 8 * (r / 4) + 4 * half + r % 4 >= spoilt) acc[t][r] = __builtin_nanf("");
  }
  // the output gate's columns 16 x + 4 part .. + 3 leave for registers that the state and v are done with
  float4 gate[8];
  const float* gp = a.gate + my_t * a.row_stride + static_cast<int64_t>(h) * Dv;
#pragma unroll
  for (int x = 0; x < 8; ++x) gate[x] = ld4<float>(gp + min(16 * x + 4 * part, Dv - 4));
  __syncthreads();   // q has been read
  if (has_cols) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * t + 8 * (r / 4) + 4 * half + r % 4;
        q_lds[row * kOPitch + 32 * wave + i] = acc[t][r] * inv_den[row];
      }
  }
  __syncthreads();
  // head norm, weight and output gate
  {
    float4 o[8];
    float ss = 0.f;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int col = 16 * x + 4 * part;
      const float2 lo = *reinterpret_cast<const float2*>(q_lds + my_row * kOPitch + col);
      const float2 hi = *reinterpret_cast<const float2*>(q_lds + my_row * kOPitch + col + 2);
      o[x] = float4{lo.x, lo.y, hi.x, hi.y};
      if (col < Dv) ss = fmaf(o[x].x, o[x].x, fmaf(o[x].y, o[x].y, fmaf(o[x].z, o[x].z, fmaf(o[x].w, o[x].w, ss))));
    }
    ss += __shfl_xor(ss, 1, kWave);
    ss += __shfl_xor(ss, 2, kWave);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(Dv) + a.eps);
    if (my_row < c.rows) {
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int col = 16 * x + 4 * part;
        if (col >= Dv) continue;
        const int64_t w_at = static_cast<int64_t>(h) * Dv + col;
        const float4 w4 = *reinterpret_cast<const float4*>(w_lds + col);
        const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
        const float ov[4] = {o[x].x, o[x].y, o[x].z, o[x].w}, gv[4] = {gate[x].x, gate[x].y, gate[x].z, gate[x].w};
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = ov[e] * inv * wv[e] / (1.0f + expf(-gv[e]));
        const int64_t to = my_t * H * Dv + w_at;
        if (a.out_dtype == kF32)
          st4<float>(static_cast<float*>(a.out) + to, float4{y[0], y[1], y[2], y[3]});
        else
          st4<bf16>(static_cast<bf16*>(a.out) + to, float4{y[0], y[1], y[2], y[3]});
      }
    }
  }
  // the request's last chunk: its running maximum goes back
  if (tid == 0 && c.row0 + c.rows == a.seg_row0[c.seg + 1]) a.m_state[static_cast<int64_t>(a.seg_slot[c.seg]) * H + h] = a.m0[at * 2 + 1];
}

template <int KD>
int launch_chunks(const MlstmChunkArgs& a, bool sums, hipStream_t s) {
  mlstm_chunk_gates_kernel<<<dim3(a.items, a.H), kWave, 0, s>>>(a);
  if (sums) {
    constexpr int D = 32 * KD;
    mlstm_chunk_sums_kernel<KD><<<dim3(a.items, a.H), KD * kWave, 0, s>>>(a);
    mlstm_chunk_scan_kernel<<<dim3(a.segments, a.H, (D * a.Dv / 4 + kScanThreads - 1) / kScanThreads + 1), kScanThreads, 0, s>>>(a, D);
  } else {
    mlstm_chunk_carry_kernel<KD><<<dim3(a.segments, a.H, a.Dv / 32), KD * kWave, 0, s>>>(a);
  }
  mlstm_chunk_out_kernel<KD><<<dim3(a.items, a.H), kOutWaves * kWave, 0, s>>>(a);
  return launch_status();
}

}  // namespace arle

using namespace arle;

// bytes of workspace of arle_mlstm_chunks: rows, ends, S_0, n_0 and m_0 of `items` chunks
extern "C" long long arle_mlstm_chunks_bytes(int items, int H, int D, int Dv) {
  const long long pairs = static_cast<long long>(items) * H;
  return pairs * (kChunkRows * static_cast<long long>(sizeof(ChunkRow)) + static_cast<long long>(sizeof(ChunkEnd)) +
                  4LL * (static_cast<long long>(D) * Dv + D + 2)) + 64;
}

// q, k, v, gate float32 [T, H*D or H*Dv] with rows row_stride apart (16-byte aligned), gates float32 [T, 2H] (input gates of
// the heads, then forget gates), states as arle_mlstm_scan.  items: chunks of 64 rows that the segments may have
// together (at least sum ceil(rows / 64)).  workspace: arle_mlstm_chunks_bytes, 16-byte aligned.  out [T, H*Dv]: the head
// norm's output times weight [H*Dv] and sigmoid(gate).  D and Dv multiples of 32 up to 128.
extern "C" int arle_mlstm_chunks(const float* q, const float* k, const float* v, const float* gate, long long row_stride,
                                 const float* gates, long long gates_stride, const float* bias_i, const float* bias_f, float cap,
                                 float* s_state, float* n_state, float* m_state, const int* seg_row0, const int* seg_slot,
                                 int segments, int items, int tokens, int longest, int H, int D, int Dv, void* workspace, const void* weight, int w_dtype,
                                 void* out, int out_dtype, float eps, void* stream) {
  if (segments == 0 || items == 0) return 0;
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (D < 32 || D > 128 || D % 32 != 0 || Dv < 32 || Dv > 128 || Dv % 32 != 0 || H < 1 || H > 65535 || row_stride % 4 != 0 ||
      !aligned(q) || !aligned(k) || !aligned(v) || !aligned(gate) || !aligned(out) || !aligned(workspace) || workspace == nullptr)
    return static_cast<int>(hipErrorInvalidValue);
  MlstmChunkArgs a{q, k, v, gate, row_stride, gates, gates_stride, bias_i, bias_f, cap, 1.0f / sqrtf(static_cast<float>(D)), eps,
                   s_state, n_state, m_state, seg_row0, seg_slot, segments, items, H, D, Dv,
                   nullptr, nullptr, nullptr, nullptr, nullptr, weight, w_dtype, out, out_dtype};
  const int64_t pairs = static_cast<int64_t>(items) * H;
  unsigned char* at = static_cast<unsigned char*>(workspace);
  a.ends = reinterpret_cast<ChunkEnd*>(at), at += pairs * sizeof(ChunkEnd);
  a.s0 = reinterpret_cast<float*>(at), at += pairs * D * Dv * 4;
  a.n0 = reinterpret_cast<float*>(at), at += pairs * D * 4;
  a.rows = reinterpret_cast<ChunkRow*>(at), at += pairs * kChunkRows * sizeof(ChunkRow);
  a.m0 = reinterpret_cast<float*>(at);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool sums = aligned(s_state) && sums_preferred(tokens, segments, longest, H, D, Dv);      // the states' kernel reads four elements at a time
  switch (D / 32) {
    case 1: return launch_chunks<1>(a, sums, s);
    case 2: return launch_chunks<2>(a, sums, s);
    case 3: return launch_chunks<3>(a, sums, s);
    default: return launch_chunks<4>(a, sums, s);
  }
}
