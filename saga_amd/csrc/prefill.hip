// Prefill attention with separate key-head and value-head counts.
//
// The reference's prefill is torch SDPA on keys and values expanded to the
// query heads: key head h / (q_h / k_h), value head h / (q_h / v_h)
// (attention/attention.py:13-53, repeat_kv).  This kernel computes
//   out[b, q, h, :] = softmax_k(scale * q_h . k + mask) . v
// with that head map, over the caches as they lie, without expanding them.
//
// One block of NW waves owns 32 * NW queries of one (batch, query head), 32
// per wave (one 32-column MFMA operand).  Keys are visited in tiles of 64 that
// the block stages in two LDS buffers:
//  * scores are computed transposed, S^T = K . Q^T (v_mfma_f32_32x32x16, A =
//    32 key rows from LDS, B = the wave's queries held in registers), so a
//    lane holds 32 scores of one query per tile and its running max and sum
//    need one cross-lane step (v_permlane32_swap).  The K rows of a 32-key
//    chunk are stored permuted in LDS (pf_krow), which leaves every lane with
//    8 consecutive keys per 16-key step: exactly the B operand of
//  * O^T = V^T . P^T, whose A operand (8 consecutive keys of one value dim)
//    is read with the transposing LDS load (ds_read_b64_tr_b16: each lane of a
//    16-lane group gets 4 keys of its dim) from V tiles stored as they lie;
//  * online softmax in base 2: per lane partial sums, reduced across the
//    two lanes of a query only at the end; the running max is moved
//    (and O rescaled) only when a score exceeds it by 2^8, and the causal /
//    length masks are applied only to the tiles that cross them.
//
// A wave's tile is a matrix phase (O += V P of the tile before, then S of this
// one: 32 MFMAs at d 128, 1024 cycles) and a vector phase (staging, softmax:
// about 130 VALU instructions, 32 of them exponentials, 900 cycles).  With 8
// waves (two per SIMD) the block's halves run opposite phases, kept so by a
// barrier per phase, so that one wave's MFMAs hide the other's softmax; with 4
// waves (one per SIMD) two blocks share a CU and drift apart by themselves.
// Blocks are ordered heaviest first (causal: the last query blocks see the
// most keys) and, within one query block, by head: blocks in flight together
// share the key / value head.
#include <type_traits>

#include "common.cuh"
#include "kernels.h"

namespace saga {
namespace {

constexpr int kPfBN = 64;  // keys per tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kPfRescale = 8.0f;  // log2 headroom of the running max

// How the mask reaches a wave: none, one byte or one 16-bit float per element
// with a unit key stride (8 elements per load), or any other (f32 with a unit
// key stride 4 elements per load, other strides one).  Every form is loaded one
// tile ahead, and tiles without a visible key are skipped.  (kPfAny with its
// loads inside the softmax and no tile skipped, 4 x 15 heads, d 64, 1021 causal
// tokens: f32 mask 209 us, booleans of another stride 203; now 57 and 43.)
enum PfMask { kPfNone, kPfBool, kPfHalf, kPfAny };

template <int D, int NW, int KS>
struct PfShape {
  static constexpr int THREADS = 64 * NW;
  static constexpr int QW = NW / KS;                    // waves over the queries
  static constexpr int BM = 32 * QW;                    // queries per block
  static constexpr int BNS = kPfBN * KS;                // keys per stage: a tile for each of the KS wave groups
  static constexpr int NDC = D / 8;                     // 16-byte chunks per row
  static constexpr int RPP = THREADS / NDC;             // rows staged per pass
  static constexpr int KPT = BNS / RPP;                 // rows per thread in a stage
  static constexpr int NJ = D / 16;                     // MFMA k-steps over d
  static constexpr int NDT = D / 32;                    // 32-dim output tiles
  static constexpr int KROW = D / 2 + 4;                // K row stride in dwords: 32 rows cover all banks
  static constexpr int VROW = D / 2 + 16;               // V row stride: 4 rows of 64 bytes cover all banks
  static constexpr int KSZ = BNS * KROW, VSZ = BNS * VROW;  // one buffer
};

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int DT>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
  if constexpr (DT == SAGA_DTYPE_BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

// LDS row of tile-local key k.  The 32x32 result puts row 8 (r / 4) + 4 hi + r
// % 4 into register r of lane half hi: key 16 e + 8 hi + j must be register
// 8 e + j.
__device__ __forceinline__ int pf_krow(int k) {
  return (k & ~15) + ((k >> 2) & 1) * 8 + ((k >> 3) & 1) * 4 + (k & 3);
}

__device__ __forceinline__ u32x4 lds16(const uint32_t* p) { return *reinterpret_cast<const u32x4*>(p); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 4 consecutive keys of one dim: lane i of a 16-lane group passes the address
// of key i / 4, dims 4 (i % 4) .. + 3 of a 4 x 16 block and gets dim i.
__device__ __forceinline__ u32x2 lds_tr(const uint32_t* p) {
  return __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 reinterpret_cast<lds_s16x4*>((__attribute__((address_space(3))) void*)const_cast<uint32_t*>(p))));
}

// Two floats -> two 16-bit elements, round to nearest even
// (v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const f32x2 v = {a, b};
  if constexpr (DT == SAGA_DTYPE_BF16) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
  }
}

// The other lane half's value of the same query.
__device__ __forceinline__ float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int DT, int D, int NW, int KS, int MASK>
__global__ __launch_bounds__(64 * NW, 2) void prefill_attn_kernel(PrefillParams p) {
  using S = PfShape<D, NW, KS>;
  using E = Elt<DT>;
  __shared__ __attribute__((aligned(16))) uint32_t ks[2 * S::KSZ];
  __shared__ __attribute__((aligned(16))) uint32_t vs[2 * S::VSZ];

  // the wave index through readfirstlane: every per-wave condition below is
  // then a scalar branch, not an exec-masked region issued by every wave
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, c = lane & 31;
  const int nhb = p.q_h * p.b;
  const int id = blockIdx.x;
  const int mb = p.nmb - 1 - id / nhb;
  const int h = (id % nhb) % p.q_h, bi = (id % nhb) / p.q_h;
  const int kh = h / (p.q_h / p.k_h), vh = h / (p.q_h / p.v_h);
  const int grp = KS > 1 ? wave / S::QW : 0;  // the wave's tile of each stage
  const int q0 = mb * S::BM, q0w = q0 + 32 * (KS > 1 ? wave % S::QW : wave);
  const int q = q0w + c;  // the lane's query

  // keys the block needs: key <= q + causal_off for its last query
  int kend = p.Lk;
  if (p.causal) kend = min(kend, min(q0 + S::BM, p.Lq) + p.causal_off);
  kend = max(kend, 0);
  const int ntiles = (kend + S::BNS - 1) / S::BNS;  // stages
  // stages in which any query of the wave may see a key of its tile
  int kmine = q0w < p.Lq ? kend : 0;
  if (p.causal) kmine = min(kmine, q0w + 32 + p.causal_off);
  const int nmine = max(kmine - kPfBN * grp + S::BNS - 1, 0) / S::BNS;

  const char* kb = p.k + (bi * p.k_sb + static_cast<int64_t>(kh) * p.k_sh) * E::kBytes;
  const char* vb = p.v + (bi * p.v_sb + static_cast<int64_t>(vh) * p.v_sh) * E::kBytes;

  // the wave's queries as B fragments: lane (hi, c) holds query q, dims 16 j + 8 hi ..
  u32x4 qf[S::NJ];
  {
    const char* qr = p.q + (bi * p.q_sb + static_cast<int64_t>(h) * p.q_sh + static_cast<int64_t>(min(q, p.Lq - 1)) *
                            p.q_sl) * E::kBytes;
#pragma unroll
    for (int j = 0; j < S::NJ; ++j)
      qf[j] = q < p.Lq ? ld16(qr + (16 * j + 8 * hi) * E::kBytes) : u32x4{0u, 0u, 0u, 0u};
  }

  // staging: stage s is the K rows of keys BNS s .. and the V rows of stage s -
  // 1 (read by the same matrix phase), in buffer s & 1.  Thread (chunk lc, row
  // lr) holds rows lr + i * RPP, dims 8 lc ..
  const int lc = tid % S::NDC, lr = tid / S::NDC;
  u32x4 kr[S::KPT], vr[S::KPT];
  const int64_t krow = p.k_sl * E::kBytes, vrow = p.v_sl * E::kBytes;
  const int kst = pf_krow(lr) * S::KROW + 4 * lc;  // and kstep dwords per RPP (16, 32 or 64) rows
  constexpr int kstep = S::RPP * S::KROW;
  static_assert(S::RPP % 16 == 0, "pf_krow permutes within 16 rows");
  // Rows outside the cache repeat its first or last row (rows at or past Lk get
  // weight 0 from the length mask and zero values from zero_tail) and stages past
  // the last are loaded but never read, so that no load sits under a branch (900 cycles a stage); scalar
  // bases and one 32-bit offset per lane keep 64-bit address arithmetic off the
  // vector unit (20 % of the whole kernel when each load did its own).
  const bool near = krow < (1 << 23) && vrow < (1 << 23);  // a stage's offsets fit 32 bits
  const uint32_t koffs = lr * static_cast<uint32_t>(krow) + 8 * lc * E::kBytes;
  const uint32_t voffs = lr * static_cast<uint32_t>(vrow) + 8 * lc * E::kBytes;
  auto load_rows = [&](const char* base, int64_t row_bytes, int r0, u32x4* dst) {
    const int s0 = max(min(r0, p.Lk - 1), 0);
    if (near) {
      const char* sb = base + s0 * row_bytes;
#pragma unroll
      for (int i = 0; i < S::KPT; ++i)
        dst[i] = ld16(sb + (static_cast<uint32_t>(min(lr + i * S::RPP, p.Lk - 1 - s0)) * static_cast<uint32_t>(row_bytes) +
                            8u * lc * E::kBytes));
    } else {
#pragma unroll
      for (int i = 0; i < S::KPT; ++i)
        dst[i] = ld16(base + min(s0 + lr + i * S::RPP, p.Lk - 1) * row_bytes + 8 * lc * E::kBytes);
    }
  };
  auto load_stage = [&](int st) {
    load_rows(kb, krow, st * S::BNS, kr);
    load_rows(vb, vrow, (st - 1) * S::BNS, vr);
  };
  // V rows at or past Lk are copies of the last row: their weight is 0, but 0 *
  // inf is NaN, so zeros are staged in their place.  One stage has such rows
  // beside others, and load_stage_full never loads it.  (Tested ahead of the
  // matrix phase: a branch between its MFMAs and the staging keeps them apart.)
  const int tail = p.Lk % S::BNS ? p.Lk / S::BNS + 1 : -1;
  auto zero_tail = [&](int st) {
    if (st != tail) return;
#pragma unroll
    for (int i = 0; i < S::KPT; ++i)
      if ((st - 1) * S::BNS + lr + i * S::RPP >= p.Lk) vr[i] = u32x4{0u, 0u, 0u, 0u};
  };
  // the next stage of a run of stages whose K rows lie below Lk, near
  const char* kcur = kb + 3 * S::BNS * krow + koffs;
  const char* vcur = vb + 2 * S::BNS * vrow + voffs;
  auto load_stage_full = [&]() {
#pragma unroll
    for (int i = 0; i < S::KPT; ++i) {
      kr[i] = ld16(kcur + i * S::RPP * krow);
      vr[i] = ld16(vcur + i * S::RPP * vrow);
    }
    kcur += S::BNS * krow;
    vcur += S::BNS * vrow;
  };
  auto write_stage = [&](int st) {
    uint32_t* kd = ks + (st & 1) * S::KSZ;
    uint32_t* vd = vs + (st & 1) * S::VSZ;
#pragma unroll
    for (int i = 0; i < S::KPT; ++i) {
      *reinterpret_cast<u32x4*>(kd + kst + i * kstep) = kr[i];
      *reinterpret_cast<u32x4*>(vd + (lr + i * S::RPP) * S::VROW + 4 * lc) = vr[i];
    }
  };

  // the mask of one tile, 8 elements per 16-key step: loaded one tile ahead
  // (kPfAny: an element's bits per register)
  typedef typename std::conditional<MASK == kPfHalf, u32x4, u32x2>::type MaskVec;
  constexpr int kMaskEs = MASK == kPfHalf ? 2 : 1;
  MaskVec mk[4];
  uint32_t ma[32];
  const char* mrow = nullptr;
  const int64_t mrow_at = bi * p.m_sb + static_cast<int64_t>(h) * p.m_sh + static_cast<int64_t>(min(q, p.Lq - 1)) * p.m_sq;
  if constexpr (MASK == kPfBool || MASK == kPfHalf) mrow = static_cast<const char*>(p.mask) + mrow_at * kMaskEs;
  auto load_any = [&](auto* row, int k0) {
    const bool whole = k0 + kPfBN <= p.Lk;
    if (whole && p.m_sk == 1 && sizeof(*row) == 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) __builtin_memcpy(ma + 8 * e, row + k0 + 16 * e + 8 * hi, 32);
    } else {  // past Lk: its last element
      const int last = p.Lk - 1;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int key = k0 + 16 * (i >> 3) + 8 * hi + (i & 7);
        ma[i] = row[min(key, last) * p.m_sk];
      }
    }
  };
  auto load_mask = [&](int it) {
    if constexpr (MASK == kPfAny) {
      if (it >= nmine) return;
      const int k0 = it * S::BNS + kPfBN * grp;
      if (p.mask_dt == SAGA_DTYPE_BOOL) load_any(static_cast<const uint8_t*>(p.mask) + mrow_at, k0);
      else if (p.mask_dt == SAGA_DTYPE_F32) load_any(static_cast<const uint32_t*>(p.mask) + mrow_at, k0);
      else load_any(static_cast<const uint16_t*>(p.mask) + mrow_at, k0);
    } else if constexpr (MASK == kPfBool || MASK == kPfHalf) {
      if (it >= nmine) return;
      const int k0 = it * S::BNS + kPfBN * grp;
      if (k0 + kPfBN <= p.Lk) {
#pragma unroll
        for (int e = 0; e < 4; ++e) __builtin_memcpy(&mk[e], mrow + (k0 + 16 * e + 8 * hi) * static_cast<int64_t>(kMaskEs), sizeof(MaskVec));
      } else {  // the last, partial tile: element by element, none past Lk
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t w[sizeof(MaskVec) / 4] = {};
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int key = k0 + 16 * e + 8 * hi + j;
            if (key < p.Lk) {
              const uint32_t v = kMaskEs == 2 ? *reinterpret_cast<const uint16_t*>(mrow + 2 * static_cast<int64_t>(key))
                                              : *reinterpret_cast<const uint8_t*>(mrow + key);
              w[j * kMaskEs / 4] |= v << (8 * (j * kMaskEs % 4));
            }
          }
          __builtin_memcpy(&mk[e], w, sizeof(MaskVec));
        }
      }
    }
  };

  f32x16 o[S::NDT];
#pragma unroll
  for (int dt = 0; dt < S::NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  f32x16 sc[2];   // S^T: chunk ch, register 8 e + j <-> key k0 + 32 ch + 16 e + 8 hi + j
  u32x4 pf[4];    // P^T: B fragment of 16-key step e
  float mrun = kNegInf, lsum = 0.f;
  const float sl2 = p.scale * kLog2e;  // > 0 (checked by the host)
  const float inv_scale = 1.0f / p.scale;
  bool mixed = false;  // the mask hides or moves part of the tile (wave-uniform)

  // 16-bit float x * inv_scale is -inf: the element hides its key whatever the score
  auto half_val = [&](uint32_t bits) {
    return p.mask_dt == SAGA_DTYPE_BF16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(static_cast<uint16_t>(bits));
  };

  // the bits of a float mask element (kPfAny) as a float
  auto any_val = [&](uint32_t bits) {
    return p.mask_dt == SAGA_DTYPE_F32 ? __uint_as_float(bits) : half_val(bits);
  };

  // whether the mask leaves the wave a key of the tile whose mask is in mk (ma)
  auto mask_visible = [&]() {
    if constexpr (MASK == kPfBool) {
      const u32x2 any = mk[0] | mk[1] | mk[2] | mk[3];
      uint32_t bad = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= (mk[e].x ^ 0x01010101u) | (mk[e].y ^ 0x01010101u);
      mixed = __any(bad != 0u);
      return __any((any.x | any.y) != 0u) != 0;
    } else if constexpr (MASK == kPfHalf) {
      bool some = false;
      uint32_t bad = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          bad |= mk[e][w];
          some |= half_val(mk[e][w] & 0xffffu) * inv_scale != kNegInf;
          some |= half_val(mk[e][w] >> 16) * inv_scale != kNegInf;
        }
      }
      mixed = __any(bad != 0u);
      return __any(some) != 0;
    } else if constexpr (MASK == kPfAny) {
      bool some = false, bad = false;
      if (p.mask_dt == SAGA_DTYPE_BOOL) {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          some |= ma[i] != 0u;
          bad |= ma[i] == 0u;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          some |= any_val(ma[i]) * inv_scale != kNegInf;
          bad |= ma[i] != 0u;
        }
      }
      mixed = __any(bad);
      return __any(some) != 0;
    } else {
      return true;
    }
  };

  // the matrix phase reads stage st: V tile st - 1 (O += V P) and K tile st
  // (S = K Q^T)
  const int g16 = lane >> 4, i16 = lane & 15;
  const int voff = kPfBN * grp * S::VROW + (8 * (g16 >> 1) + (i16 >> 2)) * S::VROW + 8 * (g16 & 1) + 2 * (i16 & 3);
  const int koff = (kPfBN * grp + c) * S::KROW + 4 * hi;
  auto pv = [&](int st) {
    const uint32_t* vp = vs + (st & 1) * S::VSZ + voff;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int dt = 0; dt < S::NDT; ++dt) {
        const u32x2 x = lds_tr(vp + 16 * e * S::VROW + 16 * dt), y = lds_tr(vp + (16 * e + 4) * S::VROW + 16 * dt);
        o[dt] = mfma32<DT>(u32x4{x.x, x.y, y.x, y.y}, pf[e], o[dt]);
      }
  };
  auto qk = [&](int st) {
    const uint32_t* kd = ks + (st & 1) * S::KSZ + koff;
#pragma unroll
    for (int ch = 0; ch < 2; ++ch)
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[ch][r] = 0.f;
#pragma unroll
    for (int j = 0; j < S::NJ; ++j)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) sc[ch] = mfma32<DT>(lds16(kd + 32 * ch * S::KROW + 8 * j), qf[j], sc[ch]);
  };
  // The whole matrix phase as one block of MFMAs (32 at d 128), stage st + 2
  // full: LDS reads PRE fragments ahead of their MFMA (right before it, each
  // fragment's LDS latency, over 100 cycles against 32 of an MFMA, is in the
  // open); the staging of st + 1 and the loads of st + 2 between the MFMAs
  // (issued together in the vector phase they held it for 1300 cycles).  LDS
  // writes do not pass LDS reads in the schedule: ahead of them where a thread
  // stages 4 rows of d 128 (4001 tokens, KS 2: 88 -> 73 us), else behind them
  // (32768 tokens, 8 waves: 3.18 -> 2.89 ms; d 64, 4001 tokens: 60 -> 50 us).
  auto pv_qk_stage = [&](int st) {
    constexpr int PRE = 4;
    constexpr int NV = 4 * S::NDT, NK = 2 * S::NJ, NM = NV + NK;
    constexpr bool kFirst = D == 128 && S::KPT == 4;
    constexpr int GAP = kFirst ? NM / (2 * S::KPT) : NM / (4 * S::KPT);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kFirst) {
      write_stage(st + 1);
      load_stage_full();
      __builtin_amdgcn_sched_group_barrier(0x200, 2 * S::KPT, 0);
    }
    pv(st);
    qk(st);
    if constexpr (!kFirst) {
      write_stage(st + 1);
      load_stage_full();
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * PRE, 0);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      if (m + PRE < NV) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      else if (m + PRE < NM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (kFirst ? m % GAP == 0 : m % GAP == GAP - 1) {
        if (!kFirst && m < NM / 2) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        else __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // softmax of tile it: scores sc -> P fragments pf
  auto softmax = [&](int it) {
    const int k0 = it * S::BNS + kPfBN * grp;
    if (mixed) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float v = sc[e >> 1][8 * (e & 1) + j];
          if constexpr (MASK == kPfBool) {
            const uint32_t w = j < 4 ? mk[e].x : mk[e].y;
            if (!((w >> (8 * (j & 3))) & 0xffu)) v = kNegInf;
          } else if constexpr (MASK == kPfHalf) {
            v += half_val((mk[e][j >> 1] >> (16 * (j & 1))) & 0xffffu) * inv_scale;
          } else if constexpr (MASK == kPfAny) {
            if (p.mask_dt == SAGA_DTYPE_BOOL) v = ma[8 * e + j] ? v : kNegInf;
            else v += any_val(ma[8 * e + j]) * inv_scale;
          }
          sc[e >> 1][8 * (e & 1) + j] = v;
        }
    }
    // the wave's diagonal and the last, partial tile
    if ((p.causal && k0 + kPfBN - 1 > q0w + p.causal_off) || k0 + kPfBN > p.Lk) {
      const int last = p.causal ? min(p.Lk - 1, q + p.causal_off) : p.Lk - 1;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k0 + 16 * e + 8 * hi + j > last) sc[e >> 1][8 * (e & 1) + j] = kNegInf;
    }
    // v_maximum3_f32: no NaN quieting of the MFMA results ahead of each max (a
    // NaN score makes its query NaN either way)
    float mx = __builtin_elementwise_maximum(sc[0][0], sc[1][0]);
#pragma unroll
    for (int r = 1; r < 16; ++r)
      mx = __builtin_elementwise_maximum(mx, __builtin_elementwise_maximum(sc[0][r], sc[1][r]));
    mx = half_max(mx) * sl2;  // base-2 units (scale > 0 keeps the max)
    // lazy rescale: the reference max moves only when a score exceeds it
    // by more than 2^8, so p <= 256 and most tiles skip the O rescale
    const bool grow = mx > mrun + kPfRescale;
    if (__any(grow)) {
      asm volatile("" ::: "memory");  // a real branch: not flattened into every tile
      const float alpha = grow ? __builtin_amdgcn_exp2f(mrun - mx) : 1.0f;
      mrun = grow ? mx : mrun;
      lsum *= alpha;
#pragma unroll
      for (int dt = 0; dt < S::NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    const float msub = mrun == kNegInf ? 0.f : mrun;
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float pv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pv[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[e >> 1][8 * (e & 1) + j], sl2, -msub));
        ps[j & 1] += pv[j];
      }
      pf[e] = u32x4{pack2<DT>(pv[0], pv[1]), pack2<DT>(pv[2], pv[3]), pack2<DT>(pv[4], pv[5]), pack2<DT>(pv[6], pv[7])};
    }
    lsum += ps[0] + ps[1];
  };

  if (ntiles > 0) {
    constexpr bool kPing = NW == 8;
    const bool second = kPing && wave >= NW / 2;  // (KS == 2: the second group)
    load_stage(0);
    load_mask(0);
    write_stage(0);
    load_stage(1);
    lds_sync();
    if (second) lds_sync();  // the second half runs one phase behind the first; a barrier ends every phase
    bool vis = nmine > 0 && mask_visible();
    zero_tail(1);
    if (vis) qk(0);
    write_stage(1);
    load_stage(2);
    if constexpr (kPing) lds_sync();
    int it = 0;
    if constexpr (MASK == kPfNone) {
      const int nfull = near ? min(nmine - 1, p.Lk / S::BNS - 3) : 0;
      for (; it < nfull; ++it) {
        softmax(it);
        lds_sync();
        pv_qk_stage(it + 1);
        if constexpr (kPing) lds_sync();
      }
    }
    for (; it < nmine; ++it) {
      if (vis) softmax(it);
      load_mask(it + 1);
      lds_sync();
      zero_tail(it + 2);
      if (vis) pv(it + 1);
      const bool next = it + 1 < nmine && mask_visible();
      if (next) qk(it + 1);
      write_stage(it + 2);
      load_stage(it + 3);
      vis = next;
      if constexpr (kPing) lds_sync();
    }
    for (; it < ntiles; ++it) {  // keys only the block's later waves see
      lds_sync();
      zero_tail(it + 2);
      write_stage(it + 2);
      load_stage(it + 3);
      if constexpr (kPing) lds_sync();
    }
    if (kPing && !second) lds_sync();
    if constexpr (KS == 2) {
      // the second group's (max, sum, O) of the same queries join the first's
      float* mg = reinterpret_cast<float*>(ks) + (wave % S::QW) * (2 + 16 * S::NDT) * 64 + lane;
      static_assert(S::QW * (2 + 16 * S::NDT) * 64 <= 2 * S::KSZ, "the merge buffer is the K buffers");
      if (grp == 1) {
        mg[0] = mrun;
        mg[64] = lsum;
#pragma unroll
        for (int dt = 0; dt < S::NDT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) mg[(2 + 16 * dt + r) * 64] = o[dt][r];
      }
      lds_sync();
      if (grp == 1) return;
      const float m1 = mg[0], m = fmaxf(mrun, m1);
      const float a0 = mrun == kNegInf ? 0.f : __builtin_amdgcn_exp2f(mrun - m);
      const float a1 = m1 == kNegInf ? 0.f : __builtin_amdgcn_exp2f(m1 - m);
      lsum = lsum * a0 + mg[64] * a1;
#pragma unroll
      for (int dt = 0; dt < S::NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = o[dt][r] * a0 + mg[(2 + 16 * dt + r) * 64] * a1;
    }
  }

  // out[b, q, h, 32 dt + 8 g + 4 hi + r] = O^T[d][q] / l; a query with no visible key gets 0
  const float l = half_sum(lsum);
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  if (q >= p.Lq) return;
  char* orow = static_cast<char*>(p.out) +
               (bi * p.o_sb + static_cast<int64_t>(q) * p.o_sq + static_cast<int64_t>(h) * p.o_sh) * E::kBytes;
#pragma unroll
  for (int dt = 0; dt < S::NDT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      *reinterpret_cast<u32x2*>(orow + (32 * dt + 8 * g + 4 * hi) * E::kBytes) =
          u32x2{pack2<DT>(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv), pack2<DT>(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv)};
    }
}

template <int DT, int D>
void launch_prefill_shape(const PrefillParams& p, dim3 grid, hipStream_t st) {
  const PrefillShape sh = p.shape;
  if (!p.mask) {
    if (sh.nw == 4) hipLaunchKernelGGL((prefill_attn_kernel<DT, D, 4, 1, kPfNone>), grid, dim3(256), 0, st, p);
    else if (sh.ks == 2) hipLaunchKernelGGL((prefill_attn_kernel<DT, D, 8, 2, kPfNone>), grid, dim3(512), 0, st, p);
    else if constexpr (D == 128)
      hipLaunchKernelGGL((prefill_attn_kernel<DT, D, 8, 1, kPfNone>), grid, dim3(512), 0, st, p);
  } else if (p.m_sk == 1 && p.mask_dt == SAGA_DTYPE_BOOL) {
    hipLaunchKernelGGL((prefill_attn_kernel<DT, D, 4, 1, kPfBool>), grid, dim3(256), 0, st, p);
  } else if (p.m_sk == 1 && (p.mask_dt == SAGA_DTYPE_BF16 || p.mask_dt == SAGA_DTYPE_F16)) {
    hipLaunchKernelGGL((prefill_attn_kernel<DT, D, 4, 1, kPfHalf>), grid, dim3(256), 0, st, p);
  } else {
    hipLaunchKernelGGL((prefill_attn_kernel<DT, D, 4, 1, kPfAny>), grid, dim3(256), 0, st, p);
  }
}

template <int DT>
hipError_t launch_prefill_typed(int d, const PrefillParams& p, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(p.nmb) * static_cast<unsigned>(p.q_h * p.b));
  if (grid.x == 0) return hipSuccess;
  if (d == 128) launch_prefill_shape<DT, 128>(p, grid, st);
  else launch_prefill_shape<DT, 64>(p, grid, st);
  return hipGetLastError();
}

}  // namespace

// Waves per block and key split, by the keys that the last query can see.  A
// launch of at most one block of 256 queries per CU is bound by its longest
// chain of tiles: the block's waves split the keys (4 waves over 128 queries,
// two tiles per stage; 4001 tokens of 12 heads, d 128: 73 us against 95 with 4
// unsplit waves and 101 with 8), unless that takes a second round of blocks
// for a short chain (8 x 512 tokens: 27 against 22 us), or the chain is so
// short that its start and the merge count for more (12 heads, d 128, split
// against 4 waves: 64 tokens 8.4 and 6.1 us, 256 12.5 and 11.5, 384 14.8 and
// 13.9, 512 16.5 and 16.3, 700 18.0 and 18.6; d 64, 15 heads: 64 6.2 and 4.8, 320
// 8.9 and 8.7, 384 9.8 and 10.2).  Larger launches: 8 waves from 8192 keys at d 128 (32768
// tokens: 2.9 ms against 3.2 with 4), else 4 (d 64, 32768 tokens: 2.14 against
// 2.19 ms).  Masked: always 4 (2999 tokens, boolean mask: 125 us against 143
// split and 171 with 8; now 94), whose waves skip the tiles that the mask hides.
// One masked query per row runs b * q_h such blocks, a wave each with work (12
// heads, d 128, 4096 keys: batch 1 101 us, batch 32 112); a split was not built.
PrefillShape prefill_shape(int64_t b, int64_t q_h, int64_t Lq, int64_t keys, int d, bool masked) {
  constexpr int64_t kCUs = 256;
  if (masked) return {4, 1};
  const int64_t units = b * q_h;
  if ((Lq + 255) / 256 * units <= kCUs) {
    if (keys > (d == 128 ? 384 : 320) && ((Lq + 127) / 128 * units <= kCUs || keys >= 1536)) return {8, 2};
    return {4, 1};
  }
  return d == 128 && keys >= 8192 ? PrefillShape{8, 1} : PrefillShape{4, 1};
}

int64_t prefill_query_blocks(const PrefillShape& sh, int64_t Lq) {
  const int64_t bm = 32 * sh.nw / sh.ks;
  return (Lq + bm - 1) / bm;
}

hipError_t launch_prefill_attention(int dtype, int d, const PrefillParams& p, hipStream_t st) {
  if (dtype == SAGA_DTYPE_BF16) return launch_prefill_typed<SAGA_DTYPE_BF16>(d, p, st);
  return launch_prefill_typed<SAGA_DTYPE_F16>(d, p, st);
}

}  // namespace saga
