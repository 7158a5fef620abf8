// Attention forward for few queries (seq_q <= 32: decode steps) and enough keys
// (plan::attn_few) on gfx950: one workgroup per (batch, head) and key split, whose waves share one tile
// of 32 queries and divide the keys.
//
// attn.h gives every wave queries of its own and walks the keys together, one
// block of loads ahead, so a decode step with one query keeps 32 KiB of a
// workgroup in flight behind two barriers per 64 keys (b4 h32 s4096 d128: 81
// us for 268 MB).  Here a wave owns whole key blocks (64 keys, every NW-th):
// its K and V tiles in its own LDS, no barrier in the loop, 128 KiB of loads
// in flight per CU.  What bounds it is HBM; the arithmetic (31 of 32 query
// columns are padding at seq_q 1) takes a fifth of the time a block's bytes
// take.
//
// The arithmetic of a block is attn.h's: S^T = K.Q^T on 32x32x16 MFMAs,
// online softmax in the exp2 domain with a lazily moving row maximum, P
// rounded to the input type for O^T += V^T.P^T, the row sum over the rounded
// P.  At the end the waves' (m, l, O) combine through LDS in wave order, and
// with key splits (few heads) the splits' combine in a second launch, in
// split order: the same inputs give the same bits.
#pragma once

#include "attn.h"

namespace frisk {

namespace fewq {

constexpr int kMaxQ = plan::kFewQ;

// Waves per workgroup: K and V tiles of all waves take 96 to 128 KiB of LDS.
template <int D> constexpr int kWaves = plan::few_waves(D);

template <int D> constexpr int lds_bytes() {
  const int tiles = kWaves<D> * AttnGeom<D>::kBuf;
  const int epi = kWaves<D> * (kMaxQ * (AttnGeom<D>::kDP + 4) + 2 * kMaxQ) * 4;
  return tiles > epi ? tiles : epi;
}

// The rows of one (batch, head) and split in the workspace: O (f32, not yet
// divided by l), then m and l.
struct Part {
  float* o;   // [batch * heads][splits][seq_q][D]
  float* ml;  // [batch * heads][splits][seq_q][2]
  int splits;
};

// Natural-log row log-sum-exp from the exp2-domain maximum and the row sum.
__device__ __forceinline__ float lse_of(float m, float l) {
  return l > 0.0f ? (m + __log2f(l)) * kLn2 : -__builtin_inff();
}

}  // namespace fewq

template <Elt T, Elt OUT, int D, bool CAUSAL, bool KT>
__global__ __launch_bounds__(64 * fewq::kWaves<D>) void attn_fewq_kernel(
    const char* __restrict__ Q, const char* __restrict__ K, const char* __restrict__ V,
    char* __restrict__ O, float* __restrict__ LSE, int heads, int seq_q, int seq_k,
    int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss,
    int64_t v_sb, int64_t v_sh, int64_t v_ss, int64_t o_sb, int64_t o_sh, int64_t o_ss,
    float scale_log2, int blocks_per_split, fewq::Part part) {
#if defined(__HIP_DEVICE_COMPILE__)
  using Mf = AttnMfma<T>;
  using G = AttnGeom<D>;
  constexpr int NW = fewq::kWaves<D>, kMaxQ = fewq::kMaxQ;
  constexpr int kKI = G::kKTile / 1024, kVI = G::kVTile / 1024;  // DMA loads per tile
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int bh = blockIdx.x, split = blockIdx.y;
  const int b = bh / heads, h = bh % heads;
  const int diag = seq_k - seq_q;  // key j is visible to query i iff j <= i + diag
  const char* qh = Q + (b * q_sb + h * q_sh) * 2;
  const char* kh = K + (b * k_sb + h * k_sh) * 2;
  const char* vh = V + (b * v_sb + h * v_sh) * 2;
  char* ks = smem + wave * G::kBuf;

  // Q fragments, as attn.h loads them.
  i32x4 qf[G::kKSteps];
  {
    const char* row = qh + (int64_t)min(l32, seq_q - 1) * q_ss * 2;
#pragma unroll
    for (int ds = 0; ds < G::kKSteps; ++ds) {
      if constexpr (KT) {
        const i32x2 lo = *(const i32x2*)(row + ds * 32 + half * 8);
        const i32x2 hi = *(const i32x2*)(row + ds * 32 + 16 + half * 8);
        qf[ds] = i32x4{lo[0], lo[1], hi[0], hi[1]};
      } else {
        qf[ds] = *(const i32x4*)(row + ds * 32 + half * 16);
      }
    }
  }

  // K and V tiles of one key block by LDS-DMA (1 KiB per instruction) into
  // this wave's LDS, swizzled as in attn.h.  Rows past seq_k and the V
  // padding dims read zeros (offsets past the buffer range).
  const __amdgpu_buffer_rsrc_t rsk = __builtin_amdgcn_make_buffer_rsrc(
      (void*)kh, (short)0,
      (int)min(KT ? (int64_t)(D - 1) * k_ss * 2 + (int64_t)seq_k * 2
                  : (int64_t)(seq_k - 1) * k_ss * 2 + D * 2,
               (int64_t)0x7fffffff),
      0x00020000);
  const __amdgpu_buffer_rsrc_t rsv = __builtin_amdgcn_make_buffer_rsrc(
      (void*)vh, (short)0, (int)min((int64_t)(seq_k - 1) * v_ss * 2 + D * 2, (int64_t)0x7fffffff),
      0x00020000);
  uint32_t k_off[kKI], v_off[kVI];
  int k_row[kKI], v_row[kVI];
#pragma unroll
  for (int i = 0; i < kKI; ++i) {
    if constexpr (KT) {
      const int r = i * 8 + lane / 8, c = (lane % 8) ^ G::swz_kt(r);
      k_row[i] = c * 8;
      k_off[i] = (uint32_t)(r * k_ss * 2) + (c << 4);
    } else {
      const int r = i * (1024 / G::kRB) + lane / G::kKC, c = (lane % G::kKC) ^ G::swz_k(r);
      k_row[i] = r;
      k_off[i] = (uint32_t)(r * k_ss * 2) + (c << 4);
    }
  }
#pragma unroll
  for (int i = 0; i < kVI; ++i) {
    const int r = i * (1024 / G::kRV) + lane / G::kVC, c = (lane % G::kVC) ^ G::swz_v(r);
    v_row[i] = c * 8 < D ? r : 1 << 30;
    v_off[i] = (uint32_t)(r * v_ss * 2) + (c << 4);
  }
  auto issue_k = [&](int kb) FRISK_INLINE {
    const uint32_t base = (uint32_t)(KT ? (int64_t)kb * kBN * 2 : (int64_t)kb * kBN * k_ss * 2);
#pragma unroll
    for (int i = 0; i < kKI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsk, (lds_ptr_t)(ks + i * 1024), 16,
          kb * kBN + k_row[i] < seq_k ? base + k_off[i] : 0x80000000u, 0, 0, 0);
  };
  auto issue_v = [&](int kb) FRISK_INLINE {
    const uint32_t base = (uint32_t)((int64_t)kb * kBN * v_ss * 2);
#pragma unroll
    for (int i = 0; i < kVI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsv, (lds_ptr_t)(ks + G::kKTile + i * 1024), 16,
          kb * kBN + v_row[i] < seq_k ? base + v_off[i] : 0x80000000u, 0, 0, 0);
  };

  // Lane offsets of the transposing reads of V^T (and K^T), as in attn.h.
  int vt_off[G::kDT], kt_off[2];
  {
    const int g = lane >> 4, hh = g >> 1, dg = g & 1, e = (lane >> 2) & 3, q = lane & 3;
#pragma unroll
    for (int dt = 0; dt < G::kDT; ++dt) {
      const int chunk = (4 * dt + 2 * dg + (q >> 1)) ^ G::swz_v(4 * hh + e);
      vt_off[dt] = G::kKTile + (4 * hh + e) * G::kRV + (chunk << 4) + 8 * (q & 1);
    }
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const int chunk = (4 * kt + 2 * dg + (q >> 1)) ^ G::swz_kt(4 * hh + e);
      kt_off[kt] = (4 * hh + e) * 128 + (chunk << 4) + 8 * (q & 1);
    }
  }
  auto read_tr = [&](const char* p, int pitch) FRISK_INLINE {
    const i32x2 a = __builtin_bit_cast(i32x2, lds_read_tr16(p));
    const i32x2 c = __builtin_bit_cast(i32x2, lds_read_tr16(p + 8 * pitch));
    return i32x4{a[0], a[1], c[0], c[1]};
  };

  f32x16 o[G::kDT];
#pragma unroll
  for (int dt = 0; dt < G::kDT; ++dt) o[dt] = f32x16{};
  float m = -__builtin_inff(), l = 0.0f;

  const int nkb = (seq_k + kBN - 1) / kBN;
  const int kb_end = min(nkb, (split + 1) * blocks_per_split);
  // Blocks from n_plain on hold keys some query does not see.
  const int n_plain = CAUSAL ? min(seq_k, max(0, diag + 1)) / kBN : seq_k / kBN;
  int kb = split * blocks_per_split + wave;
  if (kb < kb_end) {
    issue_k(kb);
    issue_v(kb);
  }
  // Drain the scalar loads of kernel arguments used after the loop.
  __builtin_amdgcn_s_waitcnt(0xC07F);
  for (; kb < kb_end; kb += NW) {
    const bool more = kb + NW < kb_end;
    // K landed (V's loads may still be in flight); S^T = K.Q^T.
    __builtin_amdgcn_s_waitcnt((kVI & 15) | ((kVI >> 4) << 14) | (7 << 4) | (15 << 8));
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int ds = 0; ds < G::kKSteps; ++ds)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const int r = kt * 32 + l32;
        const i32x4 kf = KT ? read_tr(ks + kt_off[kt] + ds * 16 * 128, 128)
                            : *(const i32x4*)(ks + r * G::kRB + (((2 * ds + half) ^ G::swz_k(r)) << 4));
        s[kt] = Mf::run(kf, qf[ds], s[kt]);
      }
    // Every K fragment has been read: the next block's K may land.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    if (more) issue_k(kb + NW);
    __builtin_amdgcn_sched_barrier(0);

    if (kb >= n_plain) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kb * kBN + kt * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
          if (key >= seq_k || (CAUSAL && key > l32 + diag)) s[kt][r] = -__builtin_inff();
        }
    }
    float mraw = -__builtin_inff();
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mraw = fmaxf(mraw, s[kt][r]);
    const float mb = pair_reduce(mraw, true) * scale_log2;
    const bool move = mb > m + kRescaleSlack;
    if (__builtin_amdgcn_ballot_w64(move)) {
      const float alpha = move ? __builtin_amdgcn_exp2f(m - mb) : 1.0f;
      m = move ? mb : m;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < G::kDT; ++dt) o[dt] *= alpha;
    }
    // A row with every key masked so far keeps m = -inf: p = 0, not NaN.
    const float nm = m == -__builtin_inff() ? 0.0f : -m;
    i32x4 pf[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int kt = kk >> 1, r0 = 8 * (kk & 1);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r0 + 2 * e], scale_log2, nm));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r0 + 2 * e + 1], scale_log2, nm));
        const uint32_t w = Mf::pack(p0, p1);
        l = Mf::dot2_ones(w, l);
        pf[kk][e] = (int)w;
      }
    }
    // V landed (only the next block's K may be in flight); O^T += V^T.P^T.
    __builtin_amdgcn_sched_barrier(0);
    if (more) __builtin_amdgcn_s_waitcnt((kKI & 15) | ((kKI >> 4) << 14) | (7 << 4) | (15 << 8));
    else FRISK_WAIT_VMCNT0();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int dt = 0; dt < G::kDT; ++dt)
        o[dt] = Mf::run(read_tr(ks + vt_off[dt] + kk * 16 * G::kRV, G::kRV), pf[kk], o[dt]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    if (more) issue_v(kb + NW);
    __builtin_amdgcn_sched_barrier(0);
  }
  l = pair_reduce(l, false);  // both lane halves of the row

  // Combine the waves: O_w as rows of D floats (padded), then m and l.
  __syncthreads();
  constexpr int kPitch = G::kDP + 4;
  float* po = (float*)smem;
  float* pm = po + NW * kMaxQ * kPitch;
  if (l32 < seq_q) {
    float* row = po + (wave * kMaxQ + l32) * kPitch;
#pragma unroll
    for (int dt = 0; dt < G::kDT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(f32x4*)(row + dt * 32 + 8 * g + 4 * half) =
            f32x4{o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2], o[dt][4 * g + 3]};
    if (half == 0) {
      pm[(wave * kMaxQ + l32) * 2] = m;
      pm[(wave * kMaxQ + l32) * 2 + 1] = l;
    }
  }
  __syncthreads();
  constexpr int kOB = EltInfo<OUT>::bytes;
  char* oh = O + (b * o_sb + h * o_sh) * kOB;
  for (int idx = tid; idx < seq_q * (D / 4); idx += 64 * NW) {
    const int q = idx / (D / 4), d = idx % (D / 4) * 4;
    float M = -__builtin_inff();
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, pm[(w * kMaxQ + q) * 2]);
    const float nM = M == -__builtin_inff() ? 0.0f : -M;
    float L = 0.0f;
    f32x4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = __builtin_amdgcn_exp2f(pm[(w * kMaxQ + q) * 2] + nM);
      L += a * pm[(w * kMaxQ + q) * 2 + 1];
      acc += a * *(const f32x4*)(po + (w * kMaxQ + q) * kPitch + d);
    }
    if (part.splits > 1) {
      const int64_t row = ((int64_t)bh * part.splits + split) * seq_q + q;
      *(f32x4*)(part.o + row * D + d) = acc;
      if (d == 0) {
        part.ml[row * 2] = M;
        part.ml[row * 2 + 1] = L;
      }
      continue;
    }
    acc *= L > 0.0f ? 1.0f / L : 0.0f;
    if constexpr (OUT == Elt::F32) {
      *(f32x4*)(oh + ((int64_t)q * o_ss + d) * 4) = acc;
    } else {
      *(i32x2*)(oh + ((int64_t)q * o_ss + d) * 2) =
          i32x2{(int)Mf::pack(acc[0], acc[1]), (int)Mf::pack(acc[2], acc[3])};
    }
    if (LSE && d == 0) LSE[(int64_t)bh * seq_q + q] = fewq::lse_of(M, L);
  }
#endif  // __HIP_DEVICE_COMPILE__
}

// The key splits of each row combined: one lane per 4 dims of a row.
template <Elt T, Elt OUT, int D>
__global__ __launch_bounds__(256) void attn_fewq_sum_kernel(fewq::Part part, char* __restrict__ O,
                                                            float* __restrict__ LSE, int heads,
                                                            int seq_q, int64_t rows, int64_t o_sb,
                                                            int64_t o_sh, int64_t o_ss) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t r = idx / (D / 4);
  if (r >= rows) return;
  const int d = (int)(idx % (D / 4)) * 4;
  const int64_t bh = r / seq_q;
  const int q = (int)(r % seq_q), b = (int)(bh / heads), h = (int)(bh % heads);
  const int64_t row0 = bh * part.splits * seq_q + q;
  float M = -__builtin_inff();
  for (int s = 0; s < part.splits; ++s) M = fmaxf(M, part.ml[(row0 + (int64_t)s * seq_q) * 2]);
  const float nM = M == -__builtin_inff() ? 0.0f : -M;
  float L = 0.0f;
  f32x4 acc = {0, 0, 0, 0};
  for (int s = 0; s < part.splits; ++s) {
    const int64_t row = row0 + (int64_t)s * seq_q;
    const float a = __builtin_amdgcn_exp2f(part.ml[row * 2] + nM);
    L += a * part.ml[row * 2 + 1];
    acc += a * *(const f32x4*)(part.o + row * D + d);
  }
  acc *= L > 0.0f ? 1.0f / L : 0.0f;
  const int64_t at = b * o_sb + h * o_sh + q * o_ss + d;
  if constexpr (OUT == Elt::F32) {
    *(f32x4*)(O + at * 4) = acc;
  } else {
    *(i32x2*)(O + at * 2) = i32x2{(int)AttnMfma<T>::pack(acc[0], acc[1]),
                                  (int)AttnMfma<T>::pack(acc[2], acc[3])};
  }
  if (LSE && d == 0) LSE[r] = fewq::lse_of(M, L);
}

template <Elt T, Elt OUT, int D, bool CAUSAL, bool KT>
static hipError_t launch_fewq(const AttnArgs& a, hipStream_t stream) {
  auto kern = attn_fewq_kernel<T, OUT, D, CAUSAL, KT>;
  constexpr int lds = fewq::lds_bytes<D>();
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return attr;
  const int64_t bh = a.batch * a.heads;
  const int nkb = (int)((a.seq_k + kBN - 1) / kBN);
  const int splits = a.workspace ? plan::attn_splits(bh, a.seq_q, a.seq_k, D, device_cus()) : 1;
  const int per = (nkb + splits - 1) / splits;
  fewq::Part part{nullptr, nullptr, splits};
  if (splits > 1) {
    part.o = (float*)a.workspace;
    part.ml = part.o + bh * splits * a.seq_q * D;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)bh, (unsigned)splits), dim3(64 * fewq::kWaves<D>), lds,
                     stream, (const char*)a.q, (const char*)a.k, (const char*)a.v, (char*)a.o, a.lse,
                     (int)a.heads, (int)a.seq_q, (int)a.seq_k, a.q_sb, a.q_sh, a.q_ss, a.k_sb, a.k_sh,
                     a.k_ss, a.v_sb, a.v_sh, a.v_ss, a.o_sb, a.o_sh, a.o_ss, a.sm_scale * kLog2e, per,
                     part);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits <= 1) return e;
  const int64_t rows = bh * a.seq_q;
  hipLaunchKernelGGL((attn_fewq_sum_kernel<T, OUT, D>), dim3((unsigned)((rows * (D / 4) + 255) / 256)),
                     dim3(256), 0, stream, part, (char*)a.o, a.lse, (int)a.heads, (int)a.seq_q, rows,
                     a.o_sb, a.o_sh, a.o_ss);
  return hipGetLastError();
}

}  // namespace frisk
