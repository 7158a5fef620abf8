// Tile-op kernels for gfx950 on [rows, cols] tensors in HBM: the reduction
// of frisk.reduce / frisk.reduce_tensor, the element-converting copy of
// frisk.copy (and of arith.truncf / arith.extf before a tile_store) and
// frisk.fill.  All three are HBM-bound; each moves its bytes once.
//
// Reduction order.  The reference fixes one association for sums, the
// canonical_fiber_tree_v1 (lib/Dialect/Frisk/Analysis/
// ReductionLayoutProof.cpp:108-140, op contract include/Dialect/Frisk/IR/
// FriskLayoutOps.td:17-30): the inputs of one output, in order, are combined
// pairwise, adjacent nodes first, and an odd last node is carried up to the
// next level.  That tree is the complete binary tree over the index padded
// to a power of two with an identity element (-0.0 for sum: x + -0.0 == x
// for every x, +0.0 included; -inf for max; +inf for min), so one level of
// the tree is a pairwise combine along one bit of the reduced index.  The
// kernels put the low index bits on the elements of a 16-byte vector, the
// next ones on lanes and the high ones on registers or on a binary counter
// over chunks, and evaluate the levels in order: the result is bit-exact
// with the sequential definition whatever the split.  Here the inputs are
// ordered by their logical index along the reduced axis (the leaf order of
// any layout whose owners walk that axis in ascending carrier order).
//
// Arithmetic.  Sums are rounded to the element type after every addition:
// an f32 addition of two f16 (bf16) values rounded to f16 (bf16) is the
// correctly rounded f16 (bf16) sum, since f32 carries at least 2p + 2 bits.
// max / min propagate NaN and order -0.0 below +0.0 (arith.maximumf /
// minimumf), so their result is always one of the inputs.  NaN results are
// quiet NaNs with an unspecified payload.

#include "common.h"
#include "kernels.h"

namespace frisk {

namespace tile {

constexpr int kThreads = 256;

// ---- combine -------------------------------------------------------------
template <Elt E> __device__ __forceinline__ float round_to(float x);
template <> __device__ __forceinline__ float round_to<Elt::F32>(float x) { return x; }
template <> __device__ __forceinline__ float round_to<Elt::F16>(float x) {
  return (float)(_Float16)x;
}
template <> __device__ __forceinline__ float round_to<Elt::BF16>(float x) {
  return bf16_bits_to_f32(f32_to_bf16_bits(x));
}

template <int KIND> __device__ __forceinline__ float identity();
template <> __device__ __forceinline__ float identity<kReduceSum>() { return -0.0f; }
template <> __device__ __forceinline__ float identity<kReduceMax>() { return -__builtin_inff(); }
template <> __device__ __forceinline__ float identity<kReduceMin>() { return __builtin_inff(); }

// Symmetric in its operands (bitwise, NaN payloads aside), so a lane
// exchange can evaluate one tree node on both partners.  max / min are one
// v_maximum3_f32 / v_minimum3_f32 for up to two combines (written out in
// compares and selects they made an 8192x16384 max along axis 0 a third
// slower than its sum: 125 us against 97), and associative, so their order is
// free.
template <Elt E, int KIND>
__device__ __forceinline__ float combine(float a, float b) {
  if constexpr (KIND == kReduceSum) return round_to<E>(a + b);
  else if constexpr (KIND == kReduceMax) return __builtin_elementwise_maximum(a, b);
  else return __builtin_elementwise_minimum(a, b);
}

// Binary counter over a sequence of complete, equally sized subtrees of NV
// outputs: after push(k, x) for k = 0..n-1, level l holds the block of 2^l
// subtrees for every set bit l of n, and finish(n) combines them from the
// smallest (rightmost) block up, which is the canonical tree over the
// sequence.  k is the same in every lane, so a push takes a branch per merge,
// two on average.  max / min keep one running value.
template <Elt E, int KIND, int L, int NV>
struct Counter {
  static constexpr bool kTree = KIND == kReduceSum;
  float lvl[kTree ? L : 1][NV];
  __device__ __forceinline__ void push(uint32_t k, float (&x)[NV]) {
    if constexpr (kTree) {
      merge<0>(__builtin_amdgcn_readfirstlane(k), x);
    } else {
#pragma unroll
      for (int j = 0; j < NV; ++j) lvl[0][j] = k ? combine<E, KIND>(lvl[0][j], x[j]) : x[j];
    }
  }
  template <int l>
  __device__ __forceinline__ void merge(uint32_t k, float (&x)[NV]) {
    if constexpr (l < L) {
      if ((k >> l) & 1u) {
#pragma unroll
        for (int j = 0; j < NV; ++j) x[j] = combine<E, KIND>(lvl[l][j], x[j]);
        merge<l + 1>(k, x);
      } else {
#pragma unroll
        for (int j = 0; j < NV; ++j) lvl[l][j] = x[j];
      }
    }
  }
  __device__ __forceinline__ float finish(uint32_t n, int j) const {
    if constexpr (!kTree) return n ? lvl[0][j] : identity<KIND>();
    float t = identity<KIND>();
    bool have = false;
#pragma unroll
    for (int l = 0; l < (kTree ? L : 1); ++l) {
      if ((n >> l) & 1u) {
        t = have ? combine<E, KIND>(lvl[l][j], t) : lvl[l][j];
        have = true;
      }
    }
    return t;
  }
};

// Vectors at any (element) alignment: a global load or store takes any
// address (32768x4095 bf16 rows, loaded by element before: 222 -> 78 us).
// Reductions load them past the caches, each byte being read once: f32
// 32768x4096 along axis 1 91 -> 82 us, 8192x16384 along axis 0 103 -> 93.
typedef f32x4 f32x4_any __attribute__((aligned(1)));
typedef i32x4 i32x4_any __attribute__((aligned(1)));
typedef i32x2 i32x2_any __attribute__((aligned(1)));

template <Elt E> __device__ __forceinline__ float load_elt(const void* p, int64_t i) {
  return load_as_f32<E>(p, i);
}

// The pairwise tree over V consecutive elements starting at column c (the
// lowest log2(V) levels); columns at or past `cols` are the identity.
template <Elt E, int KIND, int V>
__device__ __forceinline__ float slot_tree(const void* row, int64_t c, int64_t cols) {
  float x[V];
  if (c + V <= cols) {
    if constexpr (E == Elt::F32) {
      static_assert(V == 4, "f32 slot");
            const f32x4 v = __builtin_nontemporal_load((const f32x4_any*)((const float*)row + c));
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = v[i];
    } else {
      static_assert(V == 8, "16-bit slot");
            const i32x4 v = __builtin_nontemporal_load((const i32x4_any*)((const uint16_t*)row + c));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t w = (uint32_t)v[i];
        if constexpr (E == Elt::BF16) {
          x[2 * i] = bf16_bits_to_f32((uint16_t)(w & 0xffffu));
          x[2 * i + 1] = bf16_bits_to_f32((uint16_t)(w >> 16));
        } else {
          x[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu));
          x[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < V; ++i) x[i] = c + i < cols ? load_elt<E>(row, c + i) : identity<KIND>();
  }
#pragma unroll
  for (int w = 1; w < V; w <<= 1)
#pragma unroll
    for (int i = 0; i < V; i += 2 * w) x[i] = combine<E, KIND>(x[i], x[i + w]);
  return x[0];
}

}  // namespace tile

// ---- axis 1: reduce along the contiguous dimension ---------------------------
// A row is split into chunks of S = LPR * R * V columns.  Within a chunk,
// column c = k S + (r LPR + lane) V + e: vector elements e are the lowest
// index bits, then the LPR lanes of the row's lane group, then the R
// registers.  Loads are coalesced across lanes for each r.  Chunk roots
// (complete subtrees of S columns, the last one padded) go through a binary
// counter.  A wave holds 64 / LPR rows; or, of few long rows, WPR waves share
// one (each an aligned run of chunks_per_wave chunks, a power of two; the
// runs' roots combine pairwise through LDS): with a wave per row 128x28653 f32
// ran on 128 waves (109 -> 6.7 us; 384x14080 58.8 -> 6.8).
template <Elt E, int KIND, int R, int WPR>
__global__ __launch_bounds__(WPR > 4 ? 64 * WPR : tile::kThreads) void reduce_rows_kernel(
    const void* __restrict__ src, int64_t ld, int64_t rows, int64_t cols, void* __restrict__ dst,
    int64_t dst_stride, int clear, int lpr_log2, uint32_t chunks, uint32_t chunks_per_wave) {
  using namespace tile;
  constexpr int V = 16 / EltInfo<E>::bytes;
  __shared__ float part[WPR > 1 ? WPR : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lpr = 1 << lpr_log2;
  const int lr = lane & (lpr - 1);
  const int64_t row = WPR > 1 ? (int64_t)blockIdx.x
                              : ((int64_t)blockIdx.x * (kThreads / 64) + wave) * (64 >> lpr_log2) +
                                    (lane >> lpr_log2);
  const bool live = row < rows;
  const char* rp = (const char*)src + (live ? row : 0) * ld * EltInfo<E>::bytes;
  const int64_t span = live ? cols : 0;  // dead rows load nothing
  const int64_t S = (int64_t)lpr * R * V;
  const uint32_t k0 = WPR > 1 ? min(chunks, wave * chunks_per_wave) : 0;
  const uint32_t n = WPR > 1 ? min(chunks, k0 + chunks_per_wave) - k0 : chunks;

  Counter<E, KIND, 24, 1> ctr;
  // Every lane runs the same trip count: the lane exchanges need the whole
  // wave.
  for (uint32_t k = 0; k < n; ++k) {
    float v[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      v[r] = slot_tree<E, KIND, V>(rp, (int64_t)(k0 + k) * S + ((int64_t)r * lpr + lr) * V, span);
    for (int j = 0; j < lpr_log2; ++j) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = combine<E, KIND>(v[r], __shfl_xor(v[r], 1 << j, 64));
    }
#pragma unroll
    for (int w = 1; w < R; w <<= 1)
#pragma unroll
      for (int r = 0; r < R; r += 2 * w) v[r] = combine<E, KIND>(v[r], v[r + w]);
    float x[1] = {v[0]};
    ctr.push(k, x);
  }
  float res = ctr.finish(n, 0);
  if constexpr (WPR > 1) {
    if (lane == 0) part[wave] = res;
    __syncthreads();
    float t[WPR];
#pragma unroll
    for (int w = 0; w < WPR; ++w) t[w] = part[w];
#pragma unroll
    for (int s = 1; s < WPR; s <<= 1)
#pragma unroll
      for (int w = 0; w < WPR; w += 2 * s) t[w] = combine<E, KIND>(t[w], t[w + s]);
    res = t[0];
  }
  if (live && (WPR > 1 ? threadIdx.x == 0 : lr == 0)) {
    if (!clear) res = combine<E, KIND>(load_as_f32<E>(dst, row * dst_stride), res);
    store_from_f32<E>(dst, row * dst_stride, res);
  }
}

// ---- axis 0: reduce across rows -------------------------------------------------
// A workgroup of T threads owns 2^cvb_log2 slots of 4 adjacent columns and the
// rows of block blockIdx.y, or with TOP all `blocks` blocks one after another;
// in a block its T >> cvb_log2 row groups each take an aligned run of 2^b_log2
// (>= 8) rows.  A thread walks its run eight rows at a time: the eight-row
// subtree is built in registers and pushed into a binary counter of LV levels.
// The groups' roots (complete subtrees; an empty run is the identity) are
// combined in LDS by the pairwise tree over the groups.  The block's root goes
// to dst, or, in the first of two passes, to partial[block][column] as f32
// (the second pass is the same kernel over the partials, LOAD f32, with the
// combines of E), or, with TOP, into a binary counter of TOP levels in LDS.
template <Elt E, Elt LOAD, int KIND, int T, int LV, int TOP>
__global__ __launch_bounds__(T, T > 256 || LV <= 6 ? 4 : 1) void reduce_cols_kernel(
    const void* __restrict__ src, int64_t ld, int64_t rows, int64_t cols, void* __restrict__ dst,
    int64_t dst_stride, int clear, int cvb_log2, int b_log2, int blocks, float* __restrict__ partial) {
  using namespace tile;
  constexpr int kEsz = EltInfo<LOAD>::bytes;
  __shared__ float part[T * 4];
  __shared__ float top[TOP > 0 ? TOP * 256 : 1];
  const int tid = threadIdx.x;
  const int cvb = 1 << cvb_log2;
  const int cs = tid & (cvb - 1), g = tid >> cvb_log2;
  const int groups = T >> cvb_log2;
  const int64_t c0 = ((int64_t)blockIdx.x * cvb + cs) * 4;
  const bool full = c0 + 4 <= cols;

  for (int k = 0; k < (TOP > 0 ? blocks : 1); ++k) {
    const int64_t r0 = ((int64_t)(blockIdx.y + k) * groups + g) << b_log2;
    const int64_t r1 = min(rows, r0 + ((int64_t)1 << b_log2));
    Counter<E, KIND, LV, 4> ctr;
    uint32_t n8 = 0;
    for (int64_t i0 = r0; i0 < r1; i0 += 8, ++n8) {
      float x[8][4];
      const char* rp = (const char*)src + (i0 * ld + c0) * kEsz;
      if (full && i0 + 8 <= r1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const char* p = rp + i * ld * kEsz;
          if constexpr (LOAD == Elt::F32) {
            const f32x4 v = __builtin_nontemporal_load((const f32x4_any*)p);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[i][j] = v[j];
          } else {
            const i32x2 v = __builtin_nontemporal_load((const i32x2_any*)p);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const uint16_t h = (uint16_t)((uint32_t)v[j >> 1] >> (16 * (j & 1)));
              x[i][j] = LOAD == Elt::BF16 ? bf16_bits_to_f32(h) : (float)__builtin_bit_cast(_Float16, h);
            }
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            x[i][j] = i0 + i < r1 && c0 + j < cols ? load_as_f32<LOAD>(rp + i * ld * kEsz, j)
                                                   : identity<KIND>();
      }
      float t[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int w = 1; w < 8; w <<= 1)
#pragma unroll
          for (int i = 0; i < 8; i += 2 * w) x[i][j] = combine<E, KIND>(x[i][j], x[i + w][j]);
        t[j] = x[0][j];
      }
      ctr.push(n8, t);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) part[(g * cvb + cs) * 4 + j] = ctr.finish(n8, j);
    __syncthreads();
    // The pairwise tree over the row groups, one level at a time across the
    // workgroup: at level w group g (a multiple of 2w) takes in group g + w.
    for (int w = 1; w < groups; w <<= 1) {
      if ((g & (2 * w - 1)) == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          part[(g * cvb + cs) * 4 + j] = combine<E, KIND>(part[(g * cvb + cs) * 4 + j],
                                                          part[((g + w) * cvb + cs) * 4 + j]);
      }
      __syncthreads();
    }
    // (Only the thread of its columns touches an entry of `top`, and part of
    // group 0.)
    if (TOP > 0 && g == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float x = part[cs * 4 + j];
        int l = 0;
        for (; (k >> l) & 1; ++l) x = combine<E, KIND>(top[l * 256 + cs * 4 + j], x);
        top[l * 256 + cs * 4 + j] = x;
      }
    }
  }
  if (g == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t c = c0 + j;
      if (c < cols) {
        float res = part[cs * 4 + j];
        if constexpr (TOP > 0) {  // from the smallest (rightmost) set of blocks up
          int l = __builtin_ctz(blocks);
          res = top[l * 256 + cs * 4 + j];
          for (++l; blocks >> l; ++l)
            if ((blocks >> l) & 1) res = combine<E, KIND>(top[l * 256 + cs * 4 + j], res);
        }
        if (partial) {
          partial[(int64_t)blockIdx.y * cols + c] = res;
        } else {
          if (!clear) res = combine<E, KIND>(load_as_f32<E>(dst, c * dst_stride), res);
          store_from_f32<E>(dst, c * dst_stride, res);
        }
      }
    }
  }
}

// ---- any axis, permuted leaf order ------------------------------------------------
// The tree over 2^nb leaves in which leaf position p holds reduced index
// sum_j bit_j(p) << order[j] (the fiber order of a distributed layout whose
// reduced-axis bits sit on single carrier bits, sorted by carrier).  One
// thread per output walks the positions in order through a binary counter;
// threads of a wave take consecutive outputs.  Used for tile-sized
// reductions whose fibers are not in ascending index order.
struct LeafOrder {
  uint8_t bit[32];
};

template <Elt E, int KIND>
__global__ __launch_bounds__(tile::kThreads) void reduce_perm_kernel(
    const void* __restrict__ src, int64_t ld, int64_t outputs, int axis, int nb, LeafOrder order,
    void* __restrict__ dst, int64_t dst_stride, int clear) {
  using namespace tile;
  const int64_t o = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (o >= outputs) return;
  Counter<E, KIND, 32, 1> ctr;
  const uint32_t n = 1u << nb;
  for (uint32_t p = 0; p < n; ++p) {
    int64_t idx = 0;
    for (int j = 0; j < nb; ++j) idx |= (int64_t)((p >> j) & 1u) << order.bit[j];
    const int64_t off = axis == 1 ? o * ld + idx : idx * ld + o;
    float x[1] = {load_as_f32<E>(src, off)};
    ctr.push(p, x);
  }
  float res = ctr.finish(n, 0);
  if (!clear) res = combine<E, KIND>(load_as_f32<E>(dst, o * dst_stride), res);
  store_from_f32<E>(dst, o * dst_stride, res);
}

// ---- copy with element conversion ------------------------------------------------
namespace tile {

// f32 -> OCP e4m3fn, round to nearest even; magnitudes that round past 448
// (above 464) and NaN become NaN (S.1111.111): the format has no infinity.
__device__ __forceinline__ uint8_t f32_to_e4m3_bits(float f) {
  const uint8_t s = (__builtin_bit_cast(uint32_t, f) >> 24) & 0x80u;
  const float a = __builtin_fabsf(f);
  if (!(a <= 464.0f)) return s | 0x7fu;  // NaN, +-inf, overflow
  if (a < 0.015625f) {                   // below 2^-6: multiples of 2^-9
    return s | (uint8_t)__builtin_rintf(a * 512.0f);  // 8 -> 0x08, the least normal
  }
  int e;
  const float m = __builtin_frexpf(a, &e);  // a = m 2^e, m in [0.5, 1)
  int q = (int)__builtin_rintf((m * 2.0f - 1.0f) * 8.0f);
  int ef = e - 1 + 7;
  if (q == 8) {
    q = 0;
    ++ef;
  }
  return s | (uint8_t)((ef << 3) | q);
}

template <Elt D> __device__ __forceinline__ void put(void* p, int64_t i, float v);
template <> __device__ __forceinline__ void put<Elt::F32>(void* p, int64_t i, float v) {
  ((float*)p)[i] = v;
}
template <> __device__ __forceinline__ void put<Elt::F16>(void* p, int64_t i, float v) {
  ((_Float16*)p)[i] = (_Float16)v;
}
template <> __device__ __forceinline__ void put<Elt::BF16>(void* p, int64_t i, float v) {
  ((uint16_t*)p)[i] = f32_to_bf16_bits(v);
}
template <> __device__ __forceinline__ void put<Elt::E4M3>(void* p, int64_t i, float v) {
  ((uint8_t*)p)[i] = f32_to_e4m3_bits(v);
}

// Eight elements as raw bits, for vector loads and stores of 8 * esize bytes.
template <int BYTES> struct Raw8;
template <> struct Raw8<1> { using T = i32x2; };
template <> struct Raw8<2> { using T = i32x4; };
template <> struct Raw8<4> { using T = i32x8; };
template <> struct Raw8<8> { using T = i32x16; };

template <Elt E> __device__ __forceinline__ float elt_of(const void* raw, int i) {
  return load_as_f32<E>(raw, i);
}

template <Elt D> __device__ __forceinline__ void convert8(const float* x, void* raw) {
#pragma unroll
  for (int i = 0; i < 8; ++i) put<D>(raw, i, x[i]);
}

constexpr int kSlots = 4;  // 8-element slots per thread

}  // namespace tile

// Slot s of row r holds columns [8 s, 8 s + 8).  A thread works on kSlots of
// them, its loads first and its stores after, so that kSlots loads are in
// flight.  WIDE: thread t of block x takes slots (x kSlots + u) 256 + t, u <
// kSlots, of rows y, y + gridDim.y, ...  Short rows share a workgroup instead,
// 2^tpr_log2 threads each, spt slots a thread: with a workgroup per row a
// [30000, 136] copy kept 17 of 256 threads busy (23.3 -> 6.7 us).
// load(u, r, c) and store(u, r, c) are called for every slot inside.
// (The tails of conversions are loops neither unrolled nor vectorised: those
// took registers, 93 against 68 for fp8 -> bf16, and waves: 16384x8192 91 -> 75
// us.)
template <bool WIDE, typename Load, typename Store>
__device__ __forceinline__ void each_slot(int64_t rows, int64_t cols, int tpr_log2, int spt,
                                          Load load, Store store) {
  using namespace tile;
  if constexpr (WIDE) {
    for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) {
#pragma unroll
      for (int u = 0; u < kSlots; ++u) {
        const int64_t c = ((int64_t)(blockIdx.x * kSlots + u) * kThreads + threadIdx.x) * 8;
        if (c < cols) load(u, r, c);
      }
#pragma unroll
      for (int u = 0; u < kSlots; ++u) {
        const int64_t c = ((int64_t)(blockIdx.x * kSlots + u) * kThreads + threadIdx.x) * 8;
        if (c < cols) store(u, r, c);
      }
    }
  } else {
    const int rpp = kThreads >> tpr_log2;  // rows per pass of the workgroup
    const int64_t c = (int64_t)(threadIdx.x & ((1 << tpr_log2) - 1)) * 8;
    if (c >= cols) return;
    const int sub = threadIdx.x >> tpr_log2;
    for (int64_t r0 = (int64_t)blockIdx.x * rpp * spt; r0 < rows;
         r0 += (int64_t)gridDim.x * rpp * spt) {
      const int64_t end = min(rows, r0 + (int64_t)rpp * spt);
#pragma unroll
      for (int u = 0; u < kSlots; ++u)
        if (r0 + u * rpp + sub < end) load(u, r0 + u * rpp + sub, c);
#pragma unroll
      for (int u = 0; u < kSlots; ++u)
        if (r0 + u * rpp + sub < end) store(u, r0 + u * rpp + sub, c);
    }
  }
}

// Eight elements at any element alignment.
namespace tile {
template <typename Raw> __device__ __forceinline__ Raw load_any(const void* p) {
  typedef Raw Any __attribute__((aligned(1)));
  return *(const Any*)p;
}
template <typename Raw> __device__ __forceinline__ void store_any(void* p, const Raw& v) {
  typedef Raw Any __attribute__((aligned(1)));
  *(Any*)p = v;
}
// A converted output: past the caches when a lane's eight elements are at most
// 16 bytes, whole lines per wave (us: 16384x8192 bf16 -> f16 96.1 -> 92.9, f32 ->
// bf16 144 -> 140; as two halves of 32 bytes f32 188 -> 326).  Copies of one
// type are faster through them (bf16 200000x256 46 -> 36, 2000x16384 26.5 ->
// 24.9, fp8 16384x8192 46 -> 43), short rows of bytes apart (fp8 200000x300 47
// through them, 37).
template <typename Raw> __device__ __forceinline__ void store_stream(void* p, const Raw& v) {
  typedef Raw Any __attribute__((aligned(1)));
  if constexpr (sizeof(Raw) <= 16) __builtin_nontemporal_store(v, (Any*)p);
  else *(Any*)p = v;
}
}  // namespace tile

template <Elt S, Elt D, bool WIDE>
__global__ __launch_bounds__(tile::kThreads) void copy_convert_kernel(
    const void* __restrict__ src, int64_t ld_src, void* __restrict__ dst, int64_t ld_dst,
    int64_t rows, int64_t cols, int tpr_log2, int spt) {
  using namespace tile;
  constexpr int kSe = EltInfo<S>::bytes, kDe = EltInfo<D>::bytes;
  using SRaw = typename Raw8<kSe>::T;
  using DRaw = typename Raw8<kDe>::T;
  SRaw in[kSlots];
  each_slot<WIDE>(
      rows, cols, tpr_log2, spt,
      [&](int u, int64_t r, int64_t c) {
        if (c + 8 <= cols) in[u] = load_any<SRaw>((const char*)src + (r * ld_src + c) * kSe);
      },
      [&](int u, int64_t r, int64_t c) {
        if (c + 8 <= cols) {
          float x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = elt_of<S>(&in[u], i);
          DRaw out;
          convert8<D>(x, &out);
          store_stream<DRaw>((char*)dst + (r * ld_dst + c) * kDe, out);
        } else {
#pragma clang loop vectorize(disable) unroll(disable)
          for (; c < cols; ++c) put<D>(dst, r * ld_dst + c, load_as_f32<S>(src, r * ld_src + c));
        }
      });
}

// An unsigned word of BYTES bytes.
template <int BYTES>
using WordOf = typename std::conditional<
    BYTES == 1, uint8_t,
    typename std::conditional<BYTES == 2, uint16_t,
                              typename std::conditional<BYTES == 4, uint32_t, uint64_t>::type>::type>::type;

// Same-type copy of BYTES-wide elements (any dtype).
template <int BYTES, bool WIDE>
__global__ __launch_bounds__(tile::kThreads) void copy_raw_kernel(
    const void* __restrict__ src, int64_t ld_src, void* __restrict__ dst, int64_t ld_dst,
    int64_t rows, int64_t cols, int tpr_log2, int spt) {
  using namespace tile;
  using Raw = typename Raw8<BYTES>::T;
  using Word = WordOf<BYTES>;
  const Word* sp = (const Word*)src;
  Word* dp = (Word*)dst;
  Raw in[kSlots];
  each_slot<WIDE>(
      rows, cols, tpr_log2, spt,
      [&](int u, int64_t r, int64_t c) {
        if (c + 8 <= cols) in[u] = load_any<Raw>(sp + r * ld_src + c);
      },
      [&](int u, int64_t r, int64_t c) {
        if (c + 8 <= cols) {
          if constexpr (BYTES == 1 && !WIDE) store_stream<Raw>(dp + r * ld_dst + c, in[u]);
          else store_any<Raw>(dp + r * ld_dst + c, in[u]);
        } else if constexpr (BYTES == 8) {  // (as a loop 100 registers, so 75)
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (c + i < cols) dp[r * ld_dst + c + i] = sp[r * ld_src + c + i];
        } else {
          for (; c < cols; ++c) dp[r * ld_dst + c] = sp[r * ld_src + c];
        }
      });
}

// Fill with a BYTES-wide bit pattern.
template <int BYTES, bool WIDE>
__global__ __launch_bounds__(tile::kThreads) void fill_kernel(void* __restrict__ dst, int64_t ld,
                                                              int64_t rows, int64_t cols,
                                                              uint64_t bits, int tpr_log2, int spt) {
  using namespace tile;
  using Raw = typename Raw8<BYTES>::T;
  using Word = WordOf<BYTES>;
  Word* dp = (Word*)dst;
  Raw pat;
  Word* pw = (Word*)&pat;
#pragma unroll
  for (int i = 0; i < 8; ++i) pw[i] = (Word)bits;
  each_slot<WIDE>(
      rows, cols, tpr_log2, spt, [](int, int64_t, int64_t) {},
      [&](int, int64_t r, int64_t c) {
        if (c + 8 <= cols) store_any<Raw>(dp + r * ld + c, pat);
        else
          for (; c < cols; ++c) dp[r * ld + c] = (Word)bits;
      });
}

// ---- launchers ------------------------------------------------------------------------

namespace {

int ilog2(int64_t x) {
  int l = 0;
  while (((int64_t)1 << l) < x) ++l;
  return l;
}

}  // namespace

ColsSplit cols_split(int64_t rows, int64_t cols) {
  // About 1024 workgroups of 256 threads: four fit a CU's registers.  (Swept
  // on 8192 x 16384 f32 with the kernel before this one: 2048 and 512 were
  // slower; strips of 64 or 128 columns, whose 16 or 8 row groups keep each
  // thread on a long run of rows, the fastest.)
  ColsSplit sp;
  const int64_t slots = (cols + 3) / 4;
  sp.sps_log2 = ilog2(slots) < 5 ? ilog2(slots) : 5;
  const int g_log2 = 8 - sp.sps_log2;  // log2 of the row groups
  sp.strips = (slots + ((int64_t)1 << sp.sps_log2) - 1) >> sp.sps_log2;
  const int64_t want_blocks = sp.strips >= 1024 ? 1 : 1024 / sp.strips;
  sp.b_log2 = ilog2((rows + want_blocks - 1) / want_blocks);
  if (sp.b_log2 < 3 + g_log2) sp.b_log2 = 3 + g_log2;
  if (sp.b_log2 > 12 + g_log2) sp.b_log2 = 12 + g_log2;
  sp.blocks = (rows + ((int64_t)1 << sp.b_log2) - 1) >> sp.b_log2;
  return sp;
}

namespace {

// One pass over `rows` rows of src (of a.cols columns) into a.dst
// (plan::cols_pass).  T 256: at most 256 * 2^8 rows of a sum's few partials.
template <Elt E, Elt LOAD, int KIND, int T>
hipError_t cols_pass(const void* src, int64_t ld, int64_t rows, const ReduceArgs& a, hipStream_t s) {
  const plan::ColsPass p = plan::cols_pass(rows, a.cols, KIND == kReduceSum, T);
#define FRISK_COLS(THREADS, LV, TOP)                                                                \
  hipLaunchKernelGGL((reduce_cols_kernel<E, LOAD, KIND, THREADS, LV, TOP>), dim3((unsigned)p.strips), \
                     dim3(THREADS), 0, s, src, ld, rows, a.cols, a.dst, a.dst_stride, a.clear,      \
                     p.cvb_log2, p.b_log2, p.blocks, (float*)nullptr)
  // A run of 2^b_log2 rows is 2^(b_log2 - 3) pushes, which fill up to
  // b_log2 - 2 levels; rows < 2^23 in blocks of at least 2^12 fill 12.
  if constexpr (KIND == kReduceSum && T > 256) {
    if (p.blocks > 1) FRISK_COLS(T, 6, 12);
    else if (p.b_log2 > 8) FRISK_COLS(256, 22, 0);
    else FRISK_COLS(T, 6, 0);
  } else {
    if (KIND == kReduceSum && p.b_log2 > 8) return hipErrorInvalidValue;  // no such call
    FRISK_COLS(T, 6, 0);
  }
#undef FRISK_COLS
  return hipGetLastError();
}

template <Elt E, int KIND>
hipError_t reduce_typed(const ReduceArgs& a, hipStream_t s) {
  constexpr int kEsz = EltInfo<E>::bytes;
  if (a.order_bits > 0) {
    LeafOrder ord;
    for (int j = 0; j < 32; ++j) ord.bit[j] = j < a.order_bits ? a.order[j] : 0;
    const int64_t outputs = a.axis == 1 ? a.rows : a.cols;
    const dim3 grid((unsigned)((outputs + tile::kThreads - 1) / tile::kThreads));
    hipLaunchKernelGGL((reduce_perm_kernel<E, KIND>), grid, dim3(tile::kThreads), 0, s, a.src,
                       a.ld, outputs, a.axis, a.order_bits, ord, a.dst, a.dst_stride, a.clear);
    return hipGetLastError();
  }
  if (a.axis == 1) {
    constexpr int V = 16 / kEsz;
    const int64_t slots = (a.cols + V - 1) / V;
    const int pl = ilog2(slots);  // log2 of the padded slot count
    const int lpr_log2 = pl < 6 ? pl : 6;
    // Waves per row: enough for 2048 waves (8 per CU) as long as a row has 64
    // slots for each.
    int wpr_log2 = 0;
    while (wpr_log2 < 4 && (a.rows << wpr_log2) < 2048 && pl - 6 > wpr_log2 + 1) wpr_log2 += 2;
    const int left = pl - 6 - wpr_log2;
    const int r_log2 = left > 3 ? 3 : left > 0 ? left : 0;
    const int64_t S = ((int64_t)1 << (lpr_log2 + r_log2)) * V;
    const uint32_t chunks = (uint32_t)((a.cols + S - 1) / S);
    const uint32_t per_wave = 1u << ilog2((chunks + (1u << wpr_log2) - 1) >> wpr_log2);
    const int64_t rows_per_block = (int64_t)(tile::kThreads / 64) << (6 - lpr_log2);
    const dim3 grid((unsigned)(wpr_log2 ? a.rows : (a.rows + rows_per_block - 1) / rows_per_block));
#define FRISK_ROWS(R, W)                                                                       \
  hipLaunchKernelGGL((reduce_rows_kernel<E, KIND, R, W>), grid,                                \
                     dim3(W > 4 ? 64 * W : tile::kThreads), 0, s, a.src, a.ld, a.rows, a.cols, \
                     a.dst, a.dst_stride, a.clear, lpr_log2, chunks, per_wave)
#define FRISK_ROWS_R(W)             \
  switch (r_log2) {                 \
    case 0: FRISK_ROWS(1, W); break; \
    case 1: FRISK_ROWS(2, W); break; \
    case 2: FRISK_ROWS(4, W); break; \
    default: FRISK_ROWS(8, W);       \
  }
    if (wpr_log2 == 0) FRISK_ROWS_R(1)
    else if (wpr_log2 == 2) FRISK_ROWS_R(4)
    else FRISK_ROWS_R(16)
#undef FRISK_ROWS_R
#undef FRISK_ROWS
    return hipGetLastError();
  }
  // Two passes where plan::cols_two_pass asks for a workspace and the call has
  // one; under 256 rows one pass of 256 threads a strip (f32 max of
  // 112x15874 with 1024 threads, most of them without rows: 23.6 us, now 4.7).
  if (a.rows < 256) return cols_pass<E, E, KIND, 256>(a.src, a.ld, a.rows, a, s);
  if (!a.workspace) return cols_pass<E, E, KIND, 1024>(a.src, a.ld, a.rows, a, s);
  const ColsSplit sp = cols_split(a.rows, a.cols);
  const int run_log2 = sp.b_log2 - (8 - sp.sps_log2);  // rows a group: at most 2^12, 10 levels
#define FRISK_BLOCKS(LV)                                                                             \
  hipLaunchKernelGGL((reduce_cols_kernel<E, E, KIND, 256, LV, 0>), dim3(sp.strips, sp.blocks), dim3(256), \
                     0, s, a.src, a.ld, a.rows, a.cols, a.dst, a.dst_stride, a.clear, sp.sps_log2,    \
                     run_log2, 1, (float*)a.workspace)
  if (KIND != kReduceSum || run_log2 <= 8) FRISK_BLOCKS(6);
  else FRISK_BLOCKS(10);
#undef FRISK_BLOCKS
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return cols_pass<E, Elt::F32, KIND, 256>(a.workspace, a.cols, sp.blocks, a, s);
}

template <Elt E>
hipError_t reduce_kind(const ReduceArgs& a, hipStream_t s) {
  switch (a.kind) {
    case kReduceSum: return reduce_typed<E, kReduceSum>(a, s);
    case kReduceMax: return reduce_typed<E, kReduceMax>(a, s);
    case kReduceMin: return reduce_typed<E, kReduceMin>(a, s);
    default: return hipErrorInvalidValue;
  }
}

// Grid, threads per row and slots per thread of each_slot.
struct SlotGrid {
  dim3 grid;
  int tpr_log2, spt;
};
// Rows of up to most_slots slots share workgroups, and a thread takes as many
// slots as leave fill_blocks workgroups: two per CU for conversions (four slots
// whatever the rows: bf16 -> fp8 500x512 5.8 us, now 3.1), one for copies
// (4000x1024 4.7 us, 5.2 with two), any for fills, which wait for no load.
SlotGrid slot_grid(int64_t rows, int64_t cols, int most_slots, int fill_blocks) {
  const int64_t slots = (cols + 7) / 8;
  if (slots > most_slots) {
    const int64_t per_block = (int64_t)tile::kThreads * tile::kSlots * 8;
    return SlotGrid{dim3((unsigned)((cols + per_block - 1) / per_block),
                         (unsigned)(rows < 65535 ? rows : 65535)), -1, tile::kSlots};
  }
  const int tpr_log2 = ilog2(slots);
  const int64_t rpp = tile::kThreads >> tpr_log2;
  int spt = tile::kSlots;
  while (spt > 1 && rows < fill_blocks * rpp * spt) spt /= 2;
  const int64_t blocks = (rows + rpp * spt - 1) / (rpp * spt);
  return SlotGrid{dim3((unsigned)(blocks < (1 << 20) ? blocks : 1 << 20)), tpr_log2, spt};
}

template <Elt S, Elt D>
hipError_t copy_typed(const CopyArgs& a, hipStream_t s) {
  // Slots of 32 bytes: 65536x1024 f32 -> bf16 81 us shared, 69 a row each.
  const bool words = EltInfo<S>::bytes == 4 || EltInfo<D>::bytes == 4;
  const SlotGrid g = slot_grid(a.rows, a.cols, words ? 64 : 128, 512);
  auto kern = g.tpr_log2 < 0 ? copy_convert_kernel<S, D, true> : copy_convert_kernel<S, D, false>;
  hipLaunchKernelGGL(kern, g.grid, dim3(tile::kThreads), 0, s, a.src, a.ld_src,
                     a.dst, a.ld_dst, a.rows, a.cols, g.tpr_log2, g.spt);
  return hipGetLastError();
}

template <Elt S>
hipError_t copy_from(const CopyArgs& a, hipStream_t s) {
  switch (a.dst_t) {
    case Elt::F32: return copy_typed<S, Elt::F32>(a, s);
    case Elt::F16: return copy_typed<S, Elt::F16>(a, s);
    case Elt::BF16: return copy_typed<S, Elt::BF16>(a, s);
    case Elt::E4M3: return copy_typed<S, Elt::E4M3>(a, s);
    default: return hipErrorInvalidValue;
  }
}

template <int BYTES>
hipError_t copy_raw(const CopyArgs& a, hipStream_t s) {
  const SlotGrid g = slot_grid(a.rows, a.cols, BYTES >= 4 ? 64 : 128, 256);
  auto kern = g.tpr_log2 < 0 ? copy_raw_kernel<BYTES, true> : copy_raw_kernel<BYTES, false>;
  hipLaunchKernelGGL(kern, g.grid, dim3(tile::kThreads), 0, s, a.src, a.ld_src,
                     a.dst, a.ld_dst, a.rows, a.cols, g.tpr_log2, g.spt);
  return hipGetLastError();
}

template <int BYTES>
hipError_t fill_bytes(const FillArgs& a, hipStream_t s) {
  const SlotGrid g = slot_grid(a.rows, a.cols, BYTES == 8 ? 64 : 128, 0);
  auto kern = g.tpr_log2 < 0 ? fill_kernel<BYTES, true> : fill_kernel<BYTES, false>;
  hipLaunchKernelGGL(kern, g.grid, dim3(tile::kThreads), 0, s, a.dst, a.ld, a.rows,
                     a.cols, a.bits, g.tpr_log2, g.spt);
  return hipGetLastError();
}

}  // namespace

hipError_t tile_reduce(const ReduceArgs& a, hipStream_t s) {
  switch (a.dtype) {
    case Elt::F32: return reduce_kind<Elt::F32>(a, s);
    case Elt::F16: return reduce_kind<Elt::F16>(a, s);
    case Elt::BF16: return reduce_kind<Elt::BF16>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t tile_copy(const CopyArgs& a, hipStream_t s) {
  if (a.src_t == a.dst_t) {
    switch (a.esize) {
      case 1: return copy_raw<1>(a, s);
      case 2: return copy_raw<2>(a, s);
      case 4: return copy_raw<4>(a, s);
      case 8: return copy_raw<8>(a, s);
      default: return hipErrorInvalidValue;
    }
  }
  switch (a.src_t) {
    case Elt::F32: return copy_from<Elt::F32>(a, s);
    case Elt::F16: return copy_from<Elt::F16>(a, s);
    case Elt::BF16: return copy_from<Elt::BF16>(a, s);
    case Elt::E4M3: return copy_from<Elt::E4M3>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t tile_fill(const FillArgs& a, hipStream_t s) {
  switch (a.esize) {
    case 1: return fill_bytes<1>(a, s);
    case 2: return fill_bytes<2>(a, s);
    case 4: return fill_bytes<4>(a, s);
    case 8: return fill_bytes<8>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace frisk
