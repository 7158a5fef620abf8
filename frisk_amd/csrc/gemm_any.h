// MFMA GEMM for operands of any alignment on gfx950: the route of every
// request the LDS-DMA kernels (gemm_w4.h, gemm_128.h, gemm_skinny.hip) do not
// take, that is element-aligned bases, row pitches that are not multiples of
// 16 bytes, a K that ends inside a 16-byte piece, an odd pitch of C, or an
// operand that reaches past 2^31 bytes.
//
// Semantics: frisk.gemm (include/Dialect/Frisk/IR/FriskOps.td:252-292),
// C = op(A).op(B) when clear_accum, else C += op(A).op(B).
//
//  * One BT x BT output tile per 256-thread workgroup (4 waves, 2x2, each a
//    quarter of it as accumulators of the 32x32 MFMA), BT 128 or 64, K in
//    stages of 128 bytes of LDS: the operand tiles, LDS swizzles and fragment
//    reads of gemm_tile.h.  What bounds a stage is LDS traffic and its waits:
//    1.1 us for a 128 tile alone on its CU (1111x3333x1777 f16, 28 stages in
//    34 us), 0.8 in many rounds of two per CU (3824x8704x2225), 0.3 to 0.4
//    for a 64 tile.  BT and the K slices follow from the rounds of tiles over
//    the CUs (plan::any_plan).
//  * LDS-DMA needs aligned pieces, so a stage goes through registers: each
//    lane loads 16 bytes from an element-aligned address (a global load takes
//    any alignment) and writes them where the DMA would have put them, halfway
//    through the MFMAs of the stage before, into the other of two LDS slots:
//    one barrier per stage.  D stages of loads are in flight (64 tiles, three,
//    whose stages are short: 1589 x 256 x 13953 fp8 95 -> 75 us against one).
//  * Against the fp32 FMA kernel that took these requests before (us, all
//    from its 64x64 tiles): 1111x3333x1777 f16 410 -> 36, 3824x8704x2225
//    bf16 2770 -> 205, 2203x5760x4705 int8 3381 -> 111, 2x210x13418 bf16
//    1861 -> 13.
//  * Loads never leave the operand: an address is held back to the last 16
//    bytes of the matrix, and the stages near the end of K (fix_from) shift
//    the register right by the bytes it was held back and clear the bytes
//    past K.  Rows and columns past the edge are not loaded; what their
//    registers hold feeds outputs that are never stored.
//  * Addresses are 64-bit per lane, so pitches have no limit.
//
// gemm_any_a*b*.hip instantiate one layout each.
#pragma once

#include "common.h"
#include "gemm_common.h"
#include "gemm_tile.h"
#include "kernels.h"

namespace frisk {

namespace gany {

constexpr int kRow = 128;  // bytes of K per row per stage in LDS
// LDS of a BT x BT tile: the stage buffers, or the epilogue's staging (each
// wave 32 rows of BT / 2 + 4 32-bit values).
constexpr int lds_bytes(int bt) {
  const int stages = 2 * 2 * bt * kRow, epi = 4 * 32 * (bt / 2 + 4) * 4;
  return stages > epi ? stages : epi;
}

// Pieces at any address.
typedef i32x4 i32x4_any __attribute__((aligned(1)));
typedef uint64_t u64_any __attribute__((aligned(1)));

// v without its lowest `drop` bytes (0..15), then only the lowest `keep`
// bytes of that (none if not positive).  Selects only, no branches: the loads
// in flight around it stay counted.
__device__ __forceinline__ i32x4 shift_mask(i32x4 v, int drop, int keep) {
  const bool b3 = drop & 8, b2 = drop & 4;
  const uint32_t s0 = b3 ? v[2] : v[0], s1 = b3 ? v[3] : v[1], s2 = b3 ? 0 : v[2], s3 = b3 ? 0 : v[3];
  const uint32_t t0 = b2 ? s1 : s0, t1 = b2 ? s2 : s1, t2 = b2 ? s3 : s2, t3 = b2 ? 0 : s3;
  auto mask = [&](int k) {  // the lowest k bytes of a word
    return k >= 4 ? ~0u : k <= 0 ? 0u : (1u << (8 * (k & 3))) - 1;
  };
  return i32x4{(int)(__builtin_amdgcn_alignbyte(t1, t0, drop & 3) & mask(keep)),
               (int)(__builtin_amdgcn_alignbyte(t2, t1, drop & 3) & mask(keep - 4)),
               (int)(__builtin_amdgcn_alignbyte(t3, t2, drop & 3) & mask(keep - 8)),
               (int)(__builtin_amdgcn_alignbyte(0, t3, drop & 3) & mask(keep - 12))};
}

// Calls f(std::integral_constant<int, i>) for i = I .. N-1 while it returns
// true.
template <int I, int N, typename F>
__device__ __forceinline__ void static_while(F&& f) {
  if constexpr (I < N) {
    if (f(std::integral_constant<int, I>{})) static_while<I + 1, N>(f);
  }
}

// Eight e4m3 values as f16 (exact: f16 holds every e4m3 value).
__device__ __forceinline__ i32x4 e4m3x8_to_f16(int lo, int hi) {
  i32x4 r;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int w = j ? hi : lo;
    r[2 * j] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false));
    r[2 * j + 1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true));
  }
  return r;
}

// The type a stage holds in LDS.  fp8 becomes f16 on the way: the fp8 MFMAs
// (32x32x64_f8f6f4 and 32x32x16_fp8_fp8 alike) align their products before
// adding them and lose bits an f32 sum keeps (f32 output, 5x7x9: 2.8e-5 of
// the row's largest value).
template <Elt IN> constexpr Elt kLdsType = IN == Elt::E4M3 ? Elt::F16 : IN;

// One operand of the workgroup's tile: four pieces per lane and stage, each
// 16 bytes of LDS (from 16 bytes of memory, or 8 of fp8).
template <Elt IN, bool MN, int BT, int D>
struct Loader {
  using T = OpTile<kLdsType<IN>, MN, BT, kRow>;
  static constexpr int kEsz = EltInfo<IN>::bytes;
  static constexpr int kPiece = 16 / T::kEsz * kEsz;      // bytes of memory per piece
  static constexpr int kStage = kRow / T::kEsz * kEsz;    // bytes of K per stage
  static constexpr int kN = BT * kRow / 1024 / 4;         // 1 KiB blocks of LDS per wave
  const char* p[kN];   // stage 0's piece
  int lim[kN];         // K (bytes, or k rows when MN) left at it
  const char* last;    // last address a load may take
  int64_t adv;         // bytes per stage
  bool tiny;           // a matrix smaller than a piece: byte loads
  const char* end;
  i32x4 v[D][kN];      // D stages in flight, stage kt in v[kt % D]

  // X: the matrix; extent: its M or N; [k0, k0 + kb): this slice's bytes of K
  // of kb_all.
  __device__ __forceinline__ void init(const char* X, int extent, int row0, int64_t k0, int kb,
                                       int64_t kb_all, int64_t ld_b, int wave, int lane) {
    end = MN ? X + (kb_all / kEsz - 1) * ld_b + (int64_t)extent * kEsz
             : X + (int64_t)(extent - 1) * ld_b + kb_all;
    tiny = end - X < kPiece;
    last = end - kPiece;
    adv = MN ? (int64_t)T::kKS * ld_b : kStage;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int r = (kN * wave + i) * T::kRowsPerBlock + lane / T::kChunks;
      const int c = (lane % T::kChunks) ^ T::swz(r);
      if constexpr (MN) {
        const int col = min(row0 + c * (16 / T::kEsz), extent - 1);
        p[i] = X + (k0 / kEsz + r) * ld_b + (int64_t)col * kEsz;
        lim[i] = kb / kEsz - r;
      } else {
        p[i] = X + (int64_t)min(row0 + r, extent - 1) * ld_b + k0 + c * kPiece;
        lim[i] = kb - c * kPiece;
      }
    }
  }
  // First stage whose pieces may reach past K or past the matrix.
  __device__ static __forceinline__ int fix_from(int kb) {
    // K-major: the stage that holds the end of K.  MN-major: a piece of k-row
    // r starts inside the row and is at most 15 bytes too long, so it leaves
    // the matrix only in its last 16 k-rows.
    return MN ? max(kb / kEsz - 16, 0) / T::kKS : kb / kStage;
  }
  // The pieces of stage kt.
  template <int BUF>
  __device__ __forceinline__ void load(int kt) {
    const int64_t off = kt * adv;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const char* q = p[i] + off < last ? p[i] + off : last;
      if constexpr (kPiece == 16) {
        v[BUF][i] = *(const i32x4_any*)q;
      } else {
        const i32x2 x = __builtin_bit_cast(i32x2, *(const u64_any*)q);
        v[BUF][i][0] = x[0];
        v[BUF][i][1] = x[1];
      }
    }
  }
  // Stage 0 of a matrix smaller than a piece, which has no other.
  __device__ __forceinline__ void load_tiny() {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      uint64_t lo = 0, hi = 0;
#pragma unroll 1
      for (int b = 0; b < kPiece; ++b)
        if (p[i] + b < end) {
          const uint64_t x = (uint64_t)*(const uint8_t*)(p[i] + b) << (8 * (b & 7));
          if (b < 8) lo |= x;
          else hi |= x;
        }
      v[0][i] = i32x4{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
    }
  }
  // Writes the loaded stage kt to LDS; FIX: a stage from fix_from on.
  template <int BUF, bool FIX>
  __device__ __forceinline__ void store(char* lds, int wave, int lane, int kt) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      i32x4 w = v[BUF][i];
      if constexpr (FIX) {
        const int64_t back = tiny ? 0 : p[i] + kt * adv - last;
        const int keep = MN ? (kt * T::kKS < lim[i] ? kPiece : 0) : lim[i] - kt * kStage;
        w = shift_mask(w, back <= 0 ? 0 : back < kPiece - 1 ? (int)back : kPiece - 1, keep);
      }
      if constexpr (IN == Elt::E4M3) w = e4m3x8_to_f16(w[0], w[1]);
      *(i32x4*)(lds + (kN * wave + i) * 1024 + lane * 16) = w;
    }
  }
};

// Stores n (1..8) consecutive outputs at an element-aligned C[idx ..].
template <Elt OUT, typename AccS>
__device__ __forceinline__ void store_any(void* c, int64_t idx, const AccS* v, int n,
                                          bool accumulate, float scale) {
  if (n >= 8 && !accumulate) {
    if constexpr (EltInfo<OUT>::bytes == 2) {
      i32x4 r;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r[i] = (int)pack_f32x2<OUT>(v[2 * i] * scale, v[2 * i + 1] * scale);
      *(i32x4_any*)((uint16_t*)c + idx) = r;
    } else {
      i32x4 lo, hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (OUT == Elt::I32) {
          lo[i] = (int)v[i];
          hi[i] = (int)v[4 + i];
        } else {
          lo[i] = __builtin_bit_cast(int, (float)v[i] * scale);
          hi[i] = __builtin_bit_cast(int, (float)v[4 + i] * scale);
        }
      }
      *(i32x4_any*)((int32_t*)c + idx) = lo;
      *(i32x4_any*)((int32_t*)c + idx + 4) = hi;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < n) store_n<OUT>(c, idx + e, v + e, 1, accumulate, scale);
  }
}

}  // namespace gany

// Split-K: blockIdx.y is a slice of kb_slice bytes of K (a multiple of the
// stage), whose 32-bit partial tile goes c_slice_bytes further in C.
template <Elt IN, Elt OUT, bool AM, bool BM, int BT, int D, int MINW>
__global__ __launch_bounds__(256, MINW) void gemm_any_kernel(
    const char* __restrict__ A, const char* __restrict__ B, void* __restrict__ C, int M, int N,
    int64_t Kb, int64_t lda_b, int64_t ldb_b, int64_t ldc, float scale, int accumulate,
    int kb_slice, int64_t c_slice_bytes) {
#if defined(__HIP_DEVICE_COMPILE__)
  using namespace gany;
  using LA = Loader<IN, AM, BT, D>;
  using LB = Loader<IN, BM, BT, D>;
  using TA = typename LA::T;
  using TB = typename LB::T;
  using Op = Mfma32<kLdsType<IN>>;
  using Acc = typename Op::Acc;
  using AccS = typename std::conditional<IN == Elt::I8, int32_t, float>::type;
  constexpr int kHalf = BT / 2;  // rows and columns of a wave
  constexpr int TM = kHalf / 32, TN = kHalf / 32;
  constexpr int kSteps = kRow / Op::kBytes;
  constexpr int kTileBytes = BT * kRow, kSlotBytes = 2 * kTileBytes;
  __shared__ __attribute__((aligned(1024))) char smem[lds_bytes(BT)];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, half = lane >> 5;
  const int tiles_m = (M + BT - 1) / BT, tiles_n = (N + BT - 1) / BT;
  int tm, tn;
  tile_of_block<4>(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
  const int row0 = tm * BT, col0 = tn * BT;
  const int64_t k0 = (int64_t)blockIdx.y * kb_slice;
  const int kb = (int)min(Kb - k0, (int64_t)kb_slice);
  C = (char*)C + (int64_t)blockIdx.y * c_slice_bytes;

  LA la;
  LB lb;
  la.init(A, M, row0, k0, kb, Kb, lda_b, wave, lane);
  lb.init(B, N, col0, k0, kb, Kb, ldb_b, wave, lane);

  typename TA::Frag fa[TA::kSharedFrag ? 1 : TM];
  typename TB::Frag fb[TB::kSharedFrag ? 1 : TN];
#pragma unroll
  for (int t = 0; t < (TA::kSharedFrag ? 1 : TM); ++t) fa[t] = TA::frag(wm * kHalf + t * 32, lane);
#pragma unroll
  for (int t = 0; t < (TB::kSharedFrag ? 1 : TN); ++t) fb[t] = TB::frag(wn * kHalf + t * 32, lane);
  using Frag = Frags<TM, TN, TA::kLaneChunks>;
  auto load_frags = [&](const char* base, int s, Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TM; ++t)
      TA::read(base, fa[TA::kSharedFrag ? 0 : t], s, f.a[t], TA::tile_off(t * 32));
#pragma unroll
    for (int t = 0; t < TN; ++t)
      TB::read(base + kTileBytes, fb[TB::kSharedFrag ? 0 : t], s, f.b[t], TB::tile_off(t * 32));
  };
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Acc{};

  const int nk = (kb + LA::kStage - 1) / LA::kStage;
  // Writes stage kt, loaded in buffer `d`, to its slot; FIX: a stage from
  // fix_from on.
  auto put = [&](int kt, auto d, auto fix) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(d)::value;
    constexpr bool kFix = decltype(fix)::value;
    char* base = smem + (kt & 1) * kSlotBytes;
    la.template store<kBuf, kFix>(base, wave, lane, kt);
    lb.template store<kBuf, kFix>(base + kTileBytes, wave, lane, kt);
  };
  // Loads past the last stage repeat it: no condition around loads in flight.
  auto load = [&](int kt, auto d) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(d)::value;
    la.template load<kBuf>(min(kt, nk - 1));
    lb.template load<kBuf>(min(kt, nk - 1));
  };
  auto publish = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  // Multiplies stage kt; halfway `mid` writes stage kt + 1 to the other slot,
  // which every wave stopped reading at the barrier before.
  auto multiply = [&](int kt, auto&& mid) __attribute__((always_inline)) {
    const char* base = smem + (kt & 1) * kSlotBytes;
    Frag fr[kSteps];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) load_frags(base, s, fr[s]);
    static_for<0, kSteps>([&](auto sc) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Op::run(fr[s].a[i], fr[s].b[j], acc[i][j]);
      if constexpr (s == kSteps / 2 - 1) {
        __builtin_amdgcn_sched_barrier(0);
        mid();
      }
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  using Zero = std::integral_constant<int, 0>;
  if (la.tiny || lb.tiny) {
    if (la.tiny) la.load_tiny();
    else la.template load<0>(0);
    if (lb.tiny) lb.load_tiny();
    else lb.template load<0>(0);
    put(0, Zero{}, std::true_type{});
    publish();
  } else {
    static_for<0, D>([&](auto d) __attribute__((always_inline)) { load(decltype(d)::value, d); });
    put(0, Zero{}, std::true_type{});
    load(D, Zero{});
    publish();
    // Stage kt, with stage kt + 1 written from buffer d and the buffer loaded
    // again.
    auto step = [&](int kt, auto d, auto fix) __attribute__((always_inline)) {
      multiply(kt, [&]() __attribute__((always_inline)) {
        put(kt + 1, d, fix);
        load(kt + 1 + D, d);
      });
      publish();
    };
    // Groups of D steps to plain stages, then the rest, at most D + 1 steps
    // (the last two stages may need fixing).
    const int n_main = max(min(LA::fix_from(kb), LB::fix_from(kb)) - 1, 0) / D * D;
    int kt = 0;
    for (; kt < n_main; kt += D)
      static_for<0, D>([&](auto r) __attribute__((always_inline)) {
        constexpr int kR = decltype(r)::value;
        step(kt + kR, std::integral_constant<int, (kR + 1) % D>{}, std::false_type{});
      });
    static_while<0, D + 1>([&](auto r) __attribute__((always_inline)) {
      constexpr int kR = decltype(r)::value;
      if (kt + kR + 1 >= nk) return false;
      step(kt + kR, std::integral_constant<int, (kR + 1) % D>{}, std::true_type{});
      return true;
    });
  }
  multiply(nk - 1, []() __attribute__((always_inline)) {});
  __syncthreads();

  // Epilogue: each wave stages 32 rows of its tile at a time, then a lane
  // stores 8 consecutive columns.  The accumulator holds
  // D[8*(r/4) + 4*(lane/32) + r%4][lane%32] in element r.
  constexpr int kPitch = kHalf + 4, kGroups = kHalf / 8;
  AccS* out = (AccS*)(smem + wave * (32 * kPitch * 4));
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        out[(8 * (r >> 2) + 4 * half + (r & 3)) * kPitch + j * 32 + l32] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kGroups / 2; ++it) {
      const int q = it * 64 + lane, rr = q / kGroups, g = q % kGroups;
      const int gr = row0 + wm * kHalf + i * 32 + rr, gc = col0 + wn * kHalf + g * 8;
      if (gr < M && gc < N) {
        AccS v[8];
        *(i32x4*)&v[0] = *(const i32x4*)&out[rr * kPitch + g * 8];
        *(i32x4*)&v[4] = *(const i32x4*)&out[rr * kPitch + g * 8 + 4];
        store_any<OUT>(C, (int64_t)gr * ldc + gc, v, N - gc, accumulate != 0, scale);
      }
    }
    __syncthreads();
  }
#endif  // __HIP_DEVICE_COMPILE__
}

template <Elt IN, Elt OUT, bool AM, bool BM, int BT, int D, int MINW>
static hipError_t launch_any(const GemmArgs& g, int slices, int64_t kb_slice, void* ws,
                             hipStream_t stream) {
  constexpr int kEsz = EltInfo<IN>::bytes;
  const int64_t tiles = ((g.m + BT - 1) / BT) * ((g.n + BT - 1) / BT);
  const int64_t pitch = plan::any_partial_pitch(g.n);
  const bool split = slices > 1;
  hipLaunchKernelGGL((gemm_any_kernel<IN, OUT, AM, BM, BT, D, MINW>),
                     dim3((unsigned)tiles, (unsigned)slices), dim3(256), 0, stream,
                     (const char*)g.a, (const char*)g.b, split ? ws : g.c, (int)g.m, (int)g.n,
                     g.k * kEsz, g.lda * kEsz, g.ldb * kEsz, split ? pitch : g.ldc,
                     split ? 1.0f : g.scale, split ? 0 : g.accumulate, (int)kb_slice,
                     split ? g.m * pitch * 4 : (int64_t)0);
  return hipGetLastError();
}

#define FRISK_PAIR(i, o) (((int)(i) << 8) | (int)(o))

// The tile and slices of plan::any_plan; `slices` > 1: 32-bit partials (f32,
// int8: i32) to ws, summed by gemm_splitk_sum.
template <bool AM, bool BM>
hipError_t gemm_any_layout(const GemmArgs& g, const plan::SplitPlan& p, void* ws, hipStream_t s) {
  const Elt out = p.slices > 1 ? (g.in == Elt::I8 ? Elt::I32 : Elt::F32) : g.out;
  switch (FRISK_PAIR(g.in, out)) {
#define FRISK_ANY(I, O)                                                                    \
  case FRISK_PAIR(Elt::I, Elt::O):                                                         \
    return p.big ? launch_any<Elt::I, Elt::O, AM, BM, 128, 1, 2>(g, p.slices, p.kb_slice, ws, s) \
                 : launch_any<Elt::I, Elt::O, AM, BM, 64, 3, 3>(g, p.slices, p.kb_slice, ws, s);
    FRISK_ANY(BF16, BF16)
    FRISK_ANY(BF16, F32)
    FRISK_ANY(F16, F16)
    FRISK_ANY(F16, F32)
    FRISK_ANY(E4M3, BF16)
    FRISK_ANY(E4M3, F16)
    FRISK_ANY(E4M3, F32)
    FRISK_ANY(I8, I32)
    FRISK_ANY(F32, F32)
#undef FRISK_ANY
    default: return hipErrorInvalidValue;
  }
}

#undef FRISK_PAIR

}  // namespace frisk
