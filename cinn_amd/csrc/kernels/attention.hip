// Attention in one kernel for gfx950: O = softmax(scale Q K^T) V per head, fp16 / bf16 / fp32, scores and probabilities
// never in memory.
//
// As separate calls the scores went through memory twice in the element type, split heads were transposed before and
// merged after, and a key cache was copied to append one token.  Here each operand is read where it lies ([b][h][t][d],
// [b][t][h][d], or one part of packed projections [b][t][parts][h][d]; keys and values in two pieces, a cache and what
// is appended to it), and scores, probabilities' sums and the result stay fp32 in registers.
//
// Many queries (attention_kernel): a wavefront owns 32 queries and walks tiles of keys that the block stages in LDS, one
// tile ahead.  The products are taken transposed, S^T = K Q^T and O^T = V^T P^T, so that a lane holds scores of one query
// only: the row maximum and sum are chains of its own registers plus one exchange with the other half of the wavefront,
// rescaling O is one multiplier per lane, and the 32x32 result of the first product is, as it lies in registers, the B
// operand of the second (the key order inside an MFMA is free as long as V's fragments agree).  16-bit V fragments come
// from [key][d] rows by ds_read_b64_tr_b16.
//
// One or a few queries (attention_row_kernel): bound by one read of keys and values.  A block takes one query of one
// head; groups of lanes stream whole key and value rows, four at a time, each with its own running maximum, and meet
// once at the end.
//
// Measured, us, the calls this replaces -> here: fp16 [8][12] heads x 512 queries x 512 keys x 64: products, softmax and
// four transposes 79 -> 19 (340 TFLOP/s; bound by the softmax's vector instructions between the products,
// with three wavefronts per SIMD to cover them); one query against 511 + 1 keys 38 -> 7.  fp32 96 heads x 512 x 512 x
// 64: 77, half of the matrix rate.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>

#include "cinn_hip_runtime.h"
#include "kernels/flex_tile.h"
#include "runtime/hip_check.h"

namespace {

using cinn_hip_kernels::flex::bf16x8;
using cinn_hip_kernels::flex::f16x8;
using cinn_hip_kernels::flex::f32x16;
using cinn_hip_kernels::flex::f32x4;
using cinn_hip_kernels::flex::LoadAny;
using cinn_hip_kernels::flex::s16x4;
using cinn_hip_kernels::flex::u32x4;

// [b][h][t][d] in any order of the first three: d is contiguous
struct Rows {
  const void* base;
  int64_t batch, head, row;  // strides in elements
};

struct AttentionParams {
  Rows q, k[2], v[2], o;
  int heads, bh, tq, t1, t2, d;
  int q_tiles;
  float scale;
};

template <typename T>
__device__ __forceinline__ const char* HeadOf(const Rows& r, int b, int h) {
  return static_cast<const char*>(r.base) + (b * r.batch + h * r.head) * (int64_t)sizeof(T);
}

// exp(|scale| (s - m)); the scale's sign has gone into the query (a scale of 0 too: there the query is zero and the
// factor 1, since 0 * -inf of a maximum not yet found or of a masked key is no number).  Full accuracy for fp32; v_exp_f32 (2^-22 or so) of one
// fused multiply-add where the result is rounded to 16 bits anyway.  -inf for m (no finite score so far) must not make
// -inf - -inf of scores.
template <typename T>
struct Exp {
  float c;
  __device__ __forceinline__ explicit Exp(float scale) : c(scale == 0.0f ? 1.0f : fabsf(scale) * 1.4426950408889634f) {}
  __device__ __forceinline__ float Base(float m) const { return m == -__builtin_inff() ? 0.0f : m * c; }
  __device__ __forceinline__ float operator()(float s, float base) const { return __builtin_amdgcn_exp2f(__builtin_fmaf(s, c, -base)); }
};
template <>
struct Exp<float> {
  float c;
  __device__ __forceinline__ explicit Exp(float scale) : c(scale == 0.0f ? 1.0f : fabsf(scale)) {}
  __device__ __forceinline__ float Base(float m) const { return m == -__builtin_inff() ? 0.0f : m; }
  __device__ __forceinline__ float operator()(float s, float base) const { return expf((s - base) * c); }
};

// a chunk of the query, negated where the scale is negative, zero where it is zero
template <typename T>
__device__ __forceinline__ u32x4 Signed(u32x4 v, float scale) {
  if (scale == 0.0f) return u32x4{0, 0, 0, 0};
  return scale < 0.0f ? v ^ (sizeof(T) == 4 ? 0x80000000u : 0x80008000u) : v;
}

template <typename T>
struct Mma;
template <>
struct Mma<_Float16> {
  typedef f16x8 vec8;
  static __device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(vec8, a), __builtin_bit_cast(vec8, b), c, 0, 0, 0);
  }
};
template <>
struct Mma<__bf16> {
  typedef bf16x8 vec8;
  static __device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vec8, a), __builtin_bit_cast(vec8, b), c, 0, 0, 0);
  }
};
template <>
struct Mma<float> {  // four MFMAs of two k each: element e of the lane's chunk is k = e of its half of the wavefront
  static __device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], y[e], c, 0, 0, 0);
    return c;
  }
};

// One tile of keys or values on its way to LDS: [KT][PITCH bytes], rows beyond the keys and chunks beyond d are zero.
template <typename T, int KT, int NC, int THREADS, int PITCH>
struct Stage {
  static constexpr int N = (KT * NC + THREADS - 1) / THREADS;
  const char *first, *second;  // the rows of the two pieces
  int64_t row1, row2;          // and their strides in bytes
  unsigned off[N];             // this thread's chunks in a tile of the first piece
  bool near;                   // they fit
  u32x4 r[N];

  __device__ __forceinline__ Stage(const Rows& a, const Rows& b, int batch, int head, int tid)
      : first(HeadOf<T>(a, batch, head)), second(HeadOf<T>(b, batch, head)), row1(a.row * sizeof(T)), row2(b.row * sizeof(T)) {
#pragma unroll
    for (int i = 0; i < N; ++i) off[i] = (unsigned)((tid + i * THREADS) / NC * row1 + (tid + i * THREADS) % NC * 16);
    near = row1 < (1 << 30) / KT;
  }
  __device__ __forceinline__ void Load(int key0, int t1, int total, int chunks, int tid) {
    if (key0 + KT <= t1 && chunks == NC && KT * NC % THREADS == 0 && near) {
      const char* tile = first + key0 * row1;
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] = LoadAny<T>(tile + off[i]);
      return;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int at = tid + i * THREADS, key = key0 + at / NC, c = at % NC;
      r[i] = u32x4{0, 0, 0, 0};
      if (key < total && c < chunks && (KT * NC % THREADS == 0 || at < KT * NC))
        r[i] = LoadAny<T>((key < t1 ? first + key * row1 : second + (key - t1) * row2) + c * 16);
    }
  }
  __device__ __forceinline__ void Store(char* tile, int tid) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int at = tid + i * THREADS;
      if (KT * NC % THREADS == 0 || at < KT * NC) *reinterpret_cast<u32x4*>(tile + at / NC * PITCH + at % NC * 16) = r[i];
    }
  }
};

constexpr int kKeyGroups = 2;

// D: d rounded up to an instance; WQ x 32 queries per block, groups of wavefronts that take the tiles' keys in turn
template <typename T, int D, int WQ>
__global__ void __launch_bounds__(64 * WQ * kKeyGroups, 2)
attention_kernel(AttentionParams p) {
  constexpr int KG      = kKeyGroups;
  constexpr bool F32    = sizeof(T) == 4;
  constexpr int THREADS = 64 * WQ * KG;
  constexpr int KT      = 32 * KG;                  // keys per tile
  constexpr int NC      = D * (int)sizeof(T) / 16;  // 16-byte chunks per row
  constexpr int DT      = (D + 31) / 32;            // 32-row results of O^T
  // K rows are read 16 bytes per lane, rows over lanes: an odd number of 16-byte chunks.  V rows: the four rows of a
  // transposing read, 64 bytes each, fall into different quarters of the banks; single floats: rows four apart do.
  constexpr int K_PITCH = NC * 16 + 16;
  constexpr int V_PITCH = F32 ? DT * 128 + 32 : (DT * 64) % 128 == 64 ? DT * 64 : DT * 64 + 64;
  constexpr int V_AT    = KT * K_PITCH;
  constexpr int STAGE   = V_AT + KT * V_PITCH;
  constexpr int MEET    = (KG - 1) * WQ * 64 * (DT * 16 + 2) * 4;  // what the other groups hand to the first
  __shared__ __attribute__((aligned(256))) char lds[2 * STAGE > MEET ? 2 * STAGE : MEET];

  // the query tiles of a head share keys and values: every XCD gets a contiguous run of (head, tile)
  const int blocks = gridDim.x, bid = blockIdx.x, xcd = bid & 7;
  const int id = xcd * (blocks >> 3) + min(xcd, blocks & 7) + (bid >> 3);
  const int bh = id / p.q_tiles, b = bh / p.heads, h = bh % p.heads;
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / WQ, wq = wave % WQ;
  const int query = (id % p.q_tiles * WQ + wq) * 32 + (lane & 31);
  const int chunks = p.d * (int)sizeof(T) / 16, total = p.t1 + p.t2;

  Stage<T, KT, NC, THREADS, K_PITCH> sk(p.k[0], p.k[1], b, h, tid);
  Stage<T, KT, NC, THREADS, V_PITCH> sv(p.v[0], p.v[1], b, h, tid);
  sk.Load(0, p.t1, total, chunks, tid);
  sv.Load(0, p.t1, total, chunks, tid);

  u32x4 q[NC / 2];  // chunks 2 i + half of the query's row
  const char* q_row = HeadOf<T>(p.q, b, h) + min(query, p.tq - 1) * p.q.row * (int64_t)sizeof(T);
#pragma unroll
  for (int i = 0; i < NC / 2; ++i) {
    q[i] = u32x4{0, 0, 0, 0};
    if (2 * i + half < chunks) q[i] = Signed<T>(LoadAny<T>(q_row + (2 * i + half) * 16), p.scale);
  }

  const Exp<T> ex(p.scale);
  float m = -__builtin_inff(), l = 0.0f;  // l: of this lane's keys only
  f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
  sk.Store(lds, tid);
  sv.Store(lds + V_AT, tid);
  __syncthreads();

  const int tiles = (total + KT - 1) / KT;
#pragma unroll 1
  for (int kt = 0; kt < tiles; ++kt) {
    const char* cur = lds + (kt & 1) * STAGE;
    if (kt + 1 < tiles) {
      sk.Load((kt + 1) * KT, p.t1, total, chunks, tid);
      sv.Load((kt + 1) * KT, p.t1, total, chunks, tid);
    }
    const int left = total - kt * KT - kg * 32;  // keys of this group's 32
    if (left > 0) {
      f32x16 s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.0f;
      const char* row = cur + (kg * 32 + (lane & 31)) * K_PITCH + half * 16;
#pragma unroll
      for (int i = 0; i < NC / 2; ++i) s = Mma<T>::mma(*reinterpret_cast<const u32x4*>(row + i * 32), q[i], s);
      // register r is key 8 (r / 4) + 4 half + r % 4
      if (left < 32) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + 4 * half + (r & 3) >= left) s[r] = -__builtin_inff();
      }
      float top = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) top = fmaxf(top, s[r]);
      top = fmaxf(m, fmaxf(top, __shfl_xor(top, 32)));
      // What has been summed is rescaled only when a maximum has grown by more than a factor of 2^8 (fp32, whose exponent
      // is natural: e^8): probabilities up to 256 (2981) lose nothing in either type, and after the first tiles few maxima
      // grow that much.
      if (__ballot((top - m) * ex.c > 8.0f)) {
        const float keep = ex(m, ex.Base(top));
        l *= keep;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= keep;
        m = top;
      }
      const float base = ex.Base(m);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = ex(s[r], base);
        l += s[r];
      }
      const char* v_tile = cur + V_AT + kg * 32 * V_PITCH;
      if constexpr (F32) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = 8 * (r >> 2) + 4 * half + (r & 3);
            const float v = *reinterpret_cast<const float*>(v_tile + key * V_PITCH + (t * 32 + (lane & 31)) * 4);
            o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, s[r], o[t], 0, 0, 0);
          }
      } else {
        typedef T vec8 __attribute__((ext_vector_type(8)));
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          vec8 pr;
#pragma unroll
          for (int e = 0; e < 8; ++e) pr[e] = (T)s[8 * g + e];
#pragma unroll
          for (int t = 0; t < DT; ++t) {
            // four keys x sixteen d per group of 16 lanes, transposed on the way
            s16x4 part[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const char* at = v_tile + (16 * g + 8 * u + 4 * half + ((lane & 15) >> 2)) * V_PITCH +
                               (32 * t + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
              part[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)at);
            }
            o[t] = Mma<T>::mma(__builtin_bit_cast(u32x4, __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7)),
                               __builtin_bit_cast(u32x4, pr), o[t]);
          }
        }
      }
    }
    if (kt + 1 < tiles) {
      char* next = lds + ((kt + 1) & 1) * STAGE;
      sk.Store(next, tid);
      sv.Store(next + V_AT, tid);
      __syncthreads();
    }
  }

  // the groups hold the same queries in the same registers: [register][lane] per wavefront
  constexpr int REGS = DT * 16 + 2;
  __syncthreads();
  float* meet = reinterpret_cast<float*>(lds);
  if (kg > 0) {
    float* mine = meet + ((kg - 1) * WQ + wq) * REGS * 64 + lane;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(t * 16 + r) * 64] = o[t][r];
    mine[(REGS - 2) * 64] = m;
    mine[(REGS - 1) * 64] = l;
  }
  __syncthreads();
  if (kg > 0) return;
#pragma unroll
  for (int g = 1; g < KG; ++g) {
    const float* other = meet + ((g - 1) * WQ + wq) * REGS * 64 + lane;
    const float m2 = other[(REGS - 2) * 64], top = fmaxf(m, m2), base = ex.Base(top);
    const float keep = ex(m, base), add = ex(m2, base);
    l = l * keep + other[(REGS - 1) * 64] * add;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[t][r] = o[t][r] * keep + other[(t * 16 + r) * 64] * add;
    m = top;
  }
  if (query >= p.tq) return;
  // both halves of the wavefront hold this query; their shuffle partner has the same query and does not leave early
  const float inv = 1.0f / (l + __shfl_xor(l, 32));
  char* out = const_cast<char*>(HeadOf<T>(p.o, b, h)) + query * p.o.row * (int64_t)sizeof(T);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = t * 32 + 8 * i + 4 * half;
      T four[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) four[e] = (T)(o[t][4 * i + e] * inv);
      if (d < p.d) __builtin_memcpy(out + d * sizeof(T), four, sizeof(four));
    }
}

// LPK lanes hold a key's row, one chunk each.  Dynamic LDS: per wavefront a row of sums, its maximum and its total.
template <typename T, int LPK>
__global__ void __launch_bounds__(1024)
attention_row_kernel(AttentionParams p) {
  constexpr int E = 16 / (int)sizeof(T), U = 4, G = 64 / LPK;
  typedef T chunk_t __attribute__((ext_vector_type(E)));
  extern __shared__ float shared[];
  const int bh = blockIdx.x / p.tq, b = bh / p.heads, h = bh % p.heads;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  const int c = lane % LPK, group = wave * G + lane / LPK, groups = waves * G;
  const int chunks = p.d / E, total = p.t1 + p.t2;
  const bool live = c < chunks;

  const char *k1 = HeadOf<T>(p.k[0], b, h), *k2 = HeadOf<T>(p.k[1], b, h);
  const char *v1 = HeadOf<T>(p.v[0], b, h), *v2 = HeadOf<T>(p.v[1], b, h);
  float q[E];
  {
    chunk_t raw = {0};
    if (live)
      raw = __builtin_bit_cast(chunk_t, Signed<T>(LoadAny<T>(HeadOf<T>(p.q, b, h) + (blockIdx.x % p.tq) * p.q.row * (int64_t)sizeof(T) + c * 16), p.scale));
#pragma unroll
    for (int e = 0; e < E; ++e) q[e] = (float)raw[e];
  }
  const Exp<T> ex(p.scale);
  float m = -__builtin_inff(), l = 0.0f, o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = 0.0f;
#pragma unroll 1
  for (int key0 = group; key0 < total; key0 += groups * U) {
    u32x4 kr[U], vr[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = key0 + u * groups;
      kr[u] = vr[u] = u32x4{0, 0, 0, 0};
      if (key < total && live) {
        const bool cached = key < p.t1;
        kr[u] = LoadAny<T>((cached ? k1 + key * p.k[0].row * (int64_t)sizeof(T) : k2 + (key - p.t1) * p.k[1].row * (int64_t)sizeof(T)) + c * 16);
        vr[u] = LoadAny<T>((cached ? v1 + key * p.v[0].row * (int64_t)sizeof(T) : v2 + (key - p.t1) * p.v[1].row * (int64_t)sizeof(T)) + c * 16);
      }
    }
    float s[U], top = m;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const chunk_t k = __builtin_bit_cast(chunk_t, kr[u]);
      s[u] = 0.0f;
#pragma unroll
      for (int e = 0; e < E; ++e) s[u] = __builtin_fmaf(q[e], (float)k[e], s[u]);
#pragma unroll
      for (int x = 1; x < LPK; x *= 2) s[u] += __shfl_xor(s[u], x);
      if (key0 + u * groups >= total) s[u] = -__builtin_inff();
      top  = fmaxf(top, s[u]);
    }
    const float base = ex.Base(top), keep = ex(m, base);
    m = top;
    l *= keep;
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] *= keep;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const chunk_t v  = __builtin_bit_cast(chunk_t, vr[u]);
      const float prob = ex(s[u], base);
      l += prob;
#pragma unroll
      for (int e = 0; e < E; ++e) o[e] = __builtin_fmaf(prob, (float)v[e], o[e]);
    }
  }
  // the groups of a wavefront, then the wavefronts
  float top = m;
#pragma unroll
  for (int x = LPK; x < 64; x *= 2) top = fmaxf(top, __shfl_xor(top, x));
  const float keep = ex(m, ex.Base(top));
  l *= keep;
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] *= keep;
#pragma unroll
  for (int x = LPK; x < 64; x *= 2) {
    l += __shfl_xor(l, x);
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] += __shfl_xor(o[e], x);
  }
  const int pitch = p.d + 2;
  if (lane < LPK && live) {
    float* mine = shared + wave * pitch;
#pragma unroll
    for (int e = 0; e < E; ++e) mine[c * E + e] = o[e];
    if (c == 0) mine[p.d] = top, mine[p.d + 1] = l;
  }
  __syncthreads();
  for (int e = tid; e < p.d; e += blockDim.x) {
    float all = -__builtin_inff(), sum = 0.0f, norm = 0.0f;
    for (int w = 0; w < waves; ++w) all = fmaxf(all, shared[w * pitch + p.d]);
    const float base = ex.Base(all);
    for (int w = 0; w < waves; ++w) {
      const float f = ex(shared[w * pitch + p.d], base);
      sum  = __builtin_fmaf(f, shared[w * pitch + e], sum);
      norm = __builtin_fmaf(f, shared[w * pitch + p.d + 1], norm);
    }
    T* out = reinterpret_cast<T*>(const_cast<char*>(HeadOf<T>(p.o, b, h))) + (blockIdx.x % p.tq) * p.o.row;
    out[e] = (T)(sum / norm);
  }
}

// Queries per head up to which the row kernel is taken (every query reads all keys): a tile of the other kernel computes
// 32 queries whatever their number.  us for 1 | 2 | 3 | 4 queries of d = 64 and on tiles: fp32 96 heads x 512 keys 8.6 | 11.9
// | 18.0 | 18.6 and 29, 96 x 2048 23 | 34 | 55 | 60 and 102; fp16 12 x 512 6.2 | 6.3 | 6.4 | 6.4 and 10.3, 96 x 512 6.5 | 6.6
// | 10.9 | 14.7 and 10.3, 96 x 2048 13 | 19 | 32 | 34 and 29.  The line is drawn by queries alone: with several heads per CU
// tiles are ahead from two queries on (512 heads x 512 keys, fp16 16 | 28 | 38 | 49 and 15, fp32 23 | 42 | 59 | 80 and 35).
constexpr int kRowQueries = 4;

template <typename T, int LPK>
void LaunchRows(const AttentionParams& p, hipStream_t stream) {
  // four keys per lane group and pass, so long as there are keys for another wavefront
  const int per_wave = 4 * (64 / LPK);
  const int waves    = std::max(1, std::min(16, (p.t1 + p.t2 + per_wave - 1) / per_wave));
  hipLaunchKernelGGL((attention_row_kernel<T, LPK>), dim3((unsigned)p.bh * p.tq), dim3(64 * waves), waves * (p.d + 2) * sizeof(float),
                     stream, p);
}

template <typename T, int D, int WQ>
void LaunchBlocks(AttentionParams p, hipStream_t stream) {
  p.q_tiles = (p.tq + 32 * WQ - 1) / (32 * WQ);
  hipLaunchKernelGGL((attention_kernel<T, D, WQ>), dim3((unsigned)(p.bh * p.q_tiles)), dim3(64 * WQ * kKeyGroups), 0, stream, p);
}

// Wavefronts of queries per block: more share a staged tile, fewer divide the work more evenly over 256 CUs.  Blocks per
// CU times a block's work, staging counted as half a wavefront.  us with 1 | 2 | 4, d = 64, the choice in brackets: fp16 96
// heads x 512 queries x 512 keys 26.7 | [17.7] | 24.1, 192 x 96 x 512 13.6 | 12.8 | [12.7], 12 x 1024 x 1024 20.2 | [17.0] |
// 20.3; fp32 96 x 200 x 512 61 | 47 | [46], 96 x 512 x 512 92 | [71] | 90, 512 x 64 x 512 67 | [51] | 89.  Within 4% of the
// best of the three in 24 shapes of 12 to 512 heads and 33 to 1024 queries.
template <typename T, int D>
void LaunchTiles(const AttentionParams& p, hipStream_t stream) {
  auto cost = [&](int wq) {
    const int64_t blocks = (int64_t)p.bh * ((p.tq + 32 * wq - 1) / (32 * wq));
    return (blocks + 255) / 256 * (2 * wq + 1);
  };
  if (cost(4) <= cost(2) && cost(4) <= cost(1)) {
    LaunchBlocks<T, D, 4>(p, stream);
  } else if (cost(2) <= cost(1)) {
    LaunchBlocks<T, D, 2>(p, stream);
  } else {
    LaunchBlocks<T, D, 1>(p, stream);
  }
}

template <typename T>
void Launch(const AttentionParams& p, hipStream_t stream) {
  if (p.tq <= kRowQueries) {
    const int chunks = p.d * (int)sizeof(T) / 16;
    if (chunks <= 4) {
      LaunchRows<T, 4>(p, stream);
    } else if (chunks <= 8) {
      LaunchRows<T, 8>(p, stream);
    } else if (chunks <= 16) {
      LaunchRows<T, 16>(p, stream);
    } else {
      LaunchRows<T, 32>(p, stream);
    }
  } else if (p.d <= 32) {
    LaunchTiles<T, 32>(p, stream);
  } else if (p.d <= 48) {
    LaunchTiles<T, 48>(p, stream);
  } else if (p.d <= 64) {
    LaunchTiles<T, 64>(p, stream);
  } else if (p.d <= 80) {
    LaunchTiles<T, 80>(p, stream);
  } else if (p.d <= 96) {
    LaunchTiles<T, 96>(p, stream);
  } else {
    LaunchTiles<T, 128>(p, stream);
  }
}

cinn_buffer_t* BufferArg(void* v_args, int index) {
  auto* args = static_cast<cinn_pod_value_t*>(v_args);
  CINN_RT_CHECK(args[index].type_code_ == CINN_POD_BUFFER_P, "attention: argument %d is not a buffer", index);
  auto* b = static_cast<cinn_buffer_t*>(args[index].value_.v_handle);
  CINN_RT_CHECK(b && b->memory, "attention: argument %d has no device memory", index);
  return b;
}

}  // namespace

extern "C" void cinn_call_hip_attention(void* v_args, int num_args, float scale, int batch, int heads, int queries, int keys,
                                        int appended, int d, int operands, int layouts, int parts, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(batch >= 0 && heads >= 0 && queries >= 0 && appended >= 0, "attention: negative extent");
  CINN_RT_CHECK(keys > 0 && d > 0 && d <= 128 && parts >= 1, "attention: %d keys, %d elements per row (at most 128), %d parts", keys, d,
                parts);
  if ((int64_t)batch * heads * queries == 0) return;
  const cinn_buffer_t* out = BufferArg(v_args, num_args - 1);
  const bool f32 = out->type.code == cinn_type_float && out->type.bits == 32;
  const bool f16 = out->type.code == cinn_type_float && out->type.bits == 16;
  CINN_RT_CHECK(f32 || f16 || (out->type.code == cinn_type_bfloat && out->type.bits == 16), "attention: fp16 / bf16 / fp32 only");
  CINN_RT_CHECK(d % (f32 ? 4 : 8) == 0, "attention: rows of %d elements are no whole number of 16-byte chunks", d);
  AttentionParams p;
  p.heads = heads, p.bh = batch * heads, p.tq = queries, p.t1 = keys, p.t2 = appended, p.d = d, p.q_tiles = 0, p.scale = scale;
  const int64_t row = (int64_t)heads * d;
  CINN_RT_CHECK((int64_t)batch * row * std::max<int64_t>(queries, (int64_t)keys + appended) * parts < INT_MAX,
                "attention: tensor too large for 32-bit offsets");
  auto operand = [&](int i, int extent, const cinn_buffer_t* buffer) {
    CINN_RT_CHECK(buffer->type.code == out->type.code && buffer->type.bits == out->type.bits, "attention: operands of different types");
    const int layout = (layouts >> (4 * i)) & 15;
    if (layout == 0) return Rows{buffer->memory, row * extent, (int64_t)d * extent, d};
    if (layout == 1) return Rows{buffer->memory, row * extent, d, row};
    CINN_RT_CHECK(layout - 2 < parts, "attention: part %d of %d", layout - 2, parts);
    return Rows{buffer->memory + (layout - 2) * row * (f32 ? 4 : 2), row * extent * parts, d, row * parts};
  };
  auto input = [&](int i, int extent) {
    const int at = (operands >> (4 * i)) & 15;
    CINN_RT_CHECK(at < num_args - 1, "attention: operand %d is argument %d of %d", i, at, num_args);
    return operand(i, extent, BufferArg(v_args, at));
  };
  p.q    = input(0, queries);
  p.k[0] = input(1, keys);
  p.v[0] = input(3, keys);
  p.k[1] = appended > 0 ? input(2, appended) : p.k[0];
  p.v[1] = appended > 0 ? input(4, appended) : p.v[0];
  p.o    = operand(5, queries, out);
  auto s = static_cast<hipStream_t>(stream);
  if (f32) {
    Launch<float>(p, s);
  } else if (f16) {
    Launch<_Float16>(p, s);
  } else {
    Launch<__bf16>(p, s);
  }
  CINN_HIP_CALL(hipGetLastError());
}
