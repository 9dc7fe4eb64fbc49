// Dense decode attention, split-L (flash-decoding), one pass over K and V.
//
// Replaces full_einsum_forward (attention/attention.py:64-85) for l_q == 1:
// it serves the layers exempt from Atop-N, SAGA with full attention and the
// dense-GQA comparator.  Kernel 1 gives a block one (batch, key head) unit
// and one split of the positions; its four waves step through
// sub-chunks of 16 positions, each with one burst of loads (the K rows and
// the V rows of up to two value heads):
//   * QK on MFMA exactly as the score kernel (K rows -> A fragments, the
//     g <= 16 query heads of the unit -> B fragment),
//   * online softmax per head (running max / sum, rescale factor alpha),
//   * P (fp32) through wave-private LDS, then P . V on the VALU in fp32, one
//     V row per wave load (d / 64 dims per lane); heads read value head
//     h / (q_h / v_h), so a unit may touch several value heads (SAGA: 1 key
//     head, 2 value heads).
// Waves merge in LDS; with several splits each writes a (max, sum, o[d])
// partial per head and kernel 2 (one block per head) merges them.
//
// 16-bit caches whose units hold whole value heads (1, 2 or, at d 64, 5 of
// them) take dense_mfma_kernel instead: both products on MFMA, see there.  These
// are the units of the decoder's shapes; it is built and measured for no other
// count (3, 4, 8; 5 at d 128), which stay here.
#include <type_traits>

#include "common.cuh"
#include "kernels.h"

namespace saga {

constexpr int kDenseSubDefault = 16;  // positions per wave step (MFMA tiles of 16)

// Wave-local LDS ordering: the P and alpha buffers of a wave are private to it.
__device__ __forceinline__ void dense_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One V row per wave load: lane l holds dims [l*DL, l*DL + DL), DL = D / 64.
template <int DT, int DL>
struct VLane {
  static constexpr int BYTES = DL * Elt<DT>::kBytes;  // 2, 4 or 8
  using Raw = typename std::conditional<BYTES == 8, u32x2, typename std::conditional<BYTES == 4, uint32_t, uint16_t>::type>::type;
  __device__ static Raw load(const char* p) { return *reinterpret_cast<const Raw*>(p); }
  __device__ static void unpack(const Raw& r, float* f) {
    if constexpr (DT == SAGA_DTYPE_F32) {
      if constexpr (DL == 2) {
        f[0] = __uint_as_float(r.x);
        f[1] = __uint_as_float(r.y);
      } else {
        f[0] = __uint_as_float(r);
      }
    } else if constexpr (DL == 2) {
      f[0] = Elt<DT>::to_f32(r & 0xffffu);
      f[1] = Elt<DT>::to_f32(r >> 16);
    } else {
      f[0] = Elt<DT>::to_f32(r);
    }
  }
};

template <int DT, int D, int kDenseSub>
__global__ void __launch_bounds__(256) dense_split_kernel(DenseParams p) {
  using E = Elt<DT>;
  constexpr int E16 = E::kPer16B;
  constexpr int NLOAD = D / (4 * E16);
  constexpr int DL = D / kWave;  // dims per lane in the P . V phase
  using VL = VLane<DT, DL>;
  __shared__ float Ps[4][16][kDenseSub];  // per wave: P[head][position]
  __shared__ float Al[4][16];
  __shared__ float Wm[4][16], Wl[4][16];
  __shared__ float Wo[4][16][D];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int col = lane & 15, s = lane >> 4;
  const int split = blockIdx.x % p.nsplit;
  const int unit = blockIdx.x / p.nsplit;
  const int bi = unit / p.k_h, kh = unit - bi * p.k_h;
  const int g = p.g;
  const int g_v = p.q_h / p.v_h;
  int Leff = p.L;
  if (p.kv_len) Leff = min(Leff, max(p.kv_len[bi], 0));
  const bool hvalid = col < g;
  const int h0 = kh * g;
  const int h = h0 + (hvalid ? col : 0);

  u32x4 qf[NLOAD];
  const char* qrow = p.q + (bi * p.q_sb + static_cast<int64_t>(h) * p.q_sh) * E::kBytes;
#pragma unroll
  for (int j = 0; j < NLOAD; ++j)
    qf[j] = hvalid ? ld16(qrow + (j * 4 * E16 + s * E16) * E::kBytes) : u32x4{0u, 0u, 0u, 0u};
  const char* kbase = p.k + (bi * p.k_sb + static_cast<int64_t>(kh) * p.k_sh) * E::kBytes;

  const int vh_first = h0 / g_v, vh_last = (h0 + g - 1) / g_v;
  const int64_t vrow = p.v_sl * E::kBytes;
  const char* vlane = p.v + (bi * p.v_sb + static_cast<int64_t>(lane) * DL) * E::kBytes;

  float acc[16][DL];
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int d = 0; d < DL; ++d) acc[i][d] = 0.f;
  float m_run = kNegInf, l_run = 0.f;  // for head `col` (replicated over s)

  const int beg = split * p.split_len;
  const int end = min(beg + p.split_len, Leff);
  const int n_iter = end > beg ? (end - beg + 4 * kDenseSub - 1) / (4 * kDenseSub) : 0;
  for (int it = 0; it < n_iter; ++it) {
    const int c0 = beg + (it * 4 + w) * kDenseSub;
    const bool active = c0 < end;
    // V rows of the unit's first two value heads ride in the K load burst
    typename VL::Raw v0[kDenseSub], v1[kDenseSub];
    if (active) {
      constexpr int NT = kDenseSub / 16;
      u32x4 kf[NT][NLOAD];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int pos = min(c0 + 16 * t + col, p.L - 1);
        const char* krow = kbase + static_cast<int64_t>(pos) * p.k_sl * E::kBytes;
#pragma unroll
        for (int j = 0; j < NLOAD; ++j) kf[t][j] = ld16(krow + (j * 4 * E16 + s * E16) * E::kBytes);
      }
      const char* vb0 = vlane + static_cast<int64_t>(vh_first) * p.v_sh * E::kBytes;
#pragma unroll
      for (int i = 0; i < kDenseSub; ++i) v0[i] = VL::load(vb0 + static_cast<int64_t>(min(c0 + i, p.L - 1)) * vrow);
      if (vh_last > vh_first) {
        const char* vb1 = vlane + static_cast<int64_t>(vh_first + 1) * p.v_sh * E::kBytes;
#pragma unroll
        for (int i = 0; i < kDenseSub; ++i) v1[i] = VL::load(vb1 + static_cast<int64_t>(min(c0 + i, p.L - 1)) * vrow);
      }
      __builtin_amdgcn_sched_barrier(0);  // the K and V burst stays in flight together
      float x[NT][4];
      float mt = kNegInf;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NLOAD; ++j) a = mfma_16b<DT>(kf[t][j], qf[j], a);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int pos = c0 + 16 * t + 4 * s + r;
          float v = a[r] * p.scale;
          if (p.mask) {
            const int mp = min(pos, p.L - 1);
            v = v + load_as_f32(p.mask, p.mask_dt, bi * p.m_sb + static_cast<int64_t>(h) * p.m_sh +
                                                       static_cast<int64_t>(mp) * p.m_sl);
          }
          if (pos >= end) v = kNegInf;
          x[t][r] = v;
          mt = fmaxf(mt, v);
        }
      }
      mt = fmaxf(mt, __shfl_xor(mt, 16));
      mt = fmaxf(mt, __shfl_xor(mt, 32));
      const float m_new = fmaxf(m_run, mt);
      const float alpha = (m_run == kNegInf) ? (m_new == kNegInf ? 1.f : 0.f) : __expf(m_run - m_new);
      float ps = 0.f;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        f32x4 e4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e = m_new == kNegInf ? 0.f : __expf(x[t][r] - m_new);
          ps += e;
          e4[r] = e;
        }
        *reinterpret_cast<f32x4*>(&Ps[w][col][16 * t + 4 * s]) = e4;
      }
      ps += __shfl_xor(ps, 16);
      ps += __shfl_xor(ps, 32);
      l_run = l_run * alpha + ps;
      m_run = m_new;
      if (s == 0) Al[w][col] = alpha;
    }
    dense_wave_sync();  // this wave's P and alpha (waves advance independently)
    if (active) {
      {
        const f32x4* a4 = reinterpret_cast<const f32x4*>(&Al[w][0]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 a = a4[q];
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < DL; ++d) acc[4 * q + e][d] *= a[e];
        }
      }
      for (int vh = vh_first; vh <= vh_last; ++vh) {
        const int u = vh - vh_first;
        float vf[kDenseSub][DL];
        if (u == 1) {
#pragma unroll
          for (int i = 0; i < kDenseSub; ++i) VL::unpack(v1[i], vf[i]);
        } else {
          if (u >= 2) {  // further value heads: a load burst of their own
            const char* vb = vlane + static_cast<int64_t>(vh) * p.v_sh * E::kBytes;
#pragma unroll
            for (int i = 0; i < kDenseSub; ++i) v0[i] = VL::load(vb + static_cast<int64_t>(min(c0 + i, p.L - 1)) * vrow);
          }
#pragma unroll
          for (int i = 0; i < kDenseSub; ++i) VL::unpack(v0[i], vf[i]);
        }
        const int hb = max(vh * g_v, h0) - h0, he = min((vh + 1) * g_v, h0 + g) - h0;  // unit-local heads
#pragma unroll
        for (int hh = 0; hh < 16; ++hh) {
          if (hh >= hb && hh < he) {
            const f32x4* p4 = reinterpret_cast<const f32x4*>(&Ps[w][hh][0]);
#pragma unroll
            for (int i4 = 0; i4 < kDenseSub / 4; ++i4) {
              const f32x4 pw = p4[i4];
#pragma unroll
              for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int d = 0; d < DL; ++d) acc[hh][d] += pw[k] * vf[4 * i4 + k][d];
            }
          }
        }
      }
    }
    dense_wave_sync();  // P is rewritten by this wave's next step
  }

  if (s == 0) {
    Wm[w][col] = m_run;
    Wl[w][col] = l_run;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int d = 0; d < DL; ++d) Wo[w][i][lane * DL + d] = acc[i][d];
  __syncthreads();

  // merge the four waves: the split's partial, or the output when nsplit == 1
  float* part = p.part + (static_cast<int64_t>(unit) * p.nsplit + split) * g * (2 + D);
  for (int e = tid; e < g * D; e += 256) {
    const int hh = e / D, dd = e - hh * D;
    float M = kNegInf;
#pragma unroll
    for (int q = 0; q < 4; ++q) M = fmaxf(M, Wm[q][hh]);
    float l = 0.f, o = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float f = Wm[q][hh] == kNegInf ? 0.f : __expf(Wm[q][hh] - M);
      l += Wl[q][hh] * f;
      o += Wo[q][hh][dd] * f;
    }
    if (p.nsplit == 1) {
      store_from_f32(p.out, p.out_dt, bi * p.o_sb + static_cast<int64_t>(h0 + hh) * p.o_sh + dd, o / l);
    } else {
      part[hh * (2 + D) + 2 + dd] = o;
      if (dd == 0) {
        part[hh * (2 + D)] = M;
        part[hh * (2 + D) + 1] = l;
      }
    }
  }
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// Two floats rounded to two 16-bit values, and what the rounding left over.
template <int DT>
__device__ __forceinline__ uint32_t split2(float& a, float& b) {
  const f32x2 v = {a, b};
  uint32_t w;
  if constexpr (DT == SAGA_DTYPE_BF16) w = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  else w = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
  a -= Elt<DT>::to_f32(w & 0xffffu);
  b -= Elt<DT>::to_f32(w >> 16);
  return w;
}

// The infinite and NaN values of 8, or all the others; 0 elsewhere.
template <int DT>
__device__ __forceinline__ u32x4 dense_pick(u32x4 v, bool special) {
  constexpr uint32_t kInf = DT == SAGA_DTYPE_BF16 ? 0x7f80u : 0x7c00u;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = ((v[e] & 0x7fffu) >= kInf) == special ? 0xffffu : 0u;
    const uint32_t hi = (((v[e] >> 16) & 0x7fffu) >= kInf) == special ? 0xffff0000u : 0u;
    v[e] &= lo | hi;
  }
  return v;
}

__device__ __forceinline__ u32x2 lds_tr16(const uint32_t* p) {
  return __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 reinterpret_cast<lds_s16x4*>((__attribute__((address_space(3))) void*)const_cast<uint32_t*>(p))));
}

template <int D, int NV>
struct DenseMfma {
  static constexpr int VROW = D / 2 + 16;          // V row stride in dwords
  static constexpr int VSZ = 32 * VROW;            // one value head's 32 rows
  static constexpr int WROW = D + 4;               // merge row stride in floats
  static constexpr int MERGE = 4 * 16 * (WROW + 2);
  static constexpr int LDS = 4 * NV * VSZ > MERGE ? 4 * NV * VSZ : MERGE;  // dwords (2 heads of d 128: half the CU's)
};

// Kernel 1 for 16-bit caches, units of NV whole value heads.  A wave step is
// 32 positions: K fragments straight from memory (the rows of the two 16-row
// tiles taken as key 8 (i / 4) + 4 t + i % 4, so that a lane's 8 scores are 8
// consecutive keys of its head: the B operand of the second product), V rows
// through wave-private LDS, read transposed (ds_read_b64_tr_b16: 4 keys of
// one dim) as the A operand of O^T += V^T P^T.  P stays 32 bits: it is split
// exactly into 16-bit terms, an MFMA each: three of bf16 (24 bits).  f16 ends
// at 2^-24, so P is held times 2^15, where three terms are exact for weights
// from 2^-16 on, and a step with smaller ones adds terms in smaller units
// until nothing is left of them.  A head's output column only takes its own
// value head's sums.
//
// Bound by the K + V stream, so the registers of a step's loads are emptied
// (QK, LDS write) and refilled with the next step's before its softmax and
// second product: the stream does not wait for either.  The VALU kernel
// above spends 12 FMAs per value element and head group and loads value heads
// past the second in a dependent burst.  Both kernels of a call, 20 calls in one
// captured graph (on data that the last-level cache partly keeps): 8 x 33024
// positions, 12 / 2 / 2 heads, d 128: 63.0 -> 47.4 us; 4 x 33024, 12 / 1 / 2
// heads: 35.0 -> 26.6; d 64, 4 x 33024: 15 / 1 / 5 heads 41.5 -> 33.0, 15 / 5 / 5
// heads 62.1 -> 36.8; 4 x 4096, 15 / 1 / 5 heads: 13.0 -> 10.3 (latency: one block
// per CU, two launches).  f16 the same within 4 %, and up to a third more where
// logits 30 nats apart need further terms.
template <int DT, int D, int NV>
__global__ void __launch_bounds__(256, 2) dense_mfma_kernel(DenseParams p) {
  using S = DenseMfma<D, NV>;
  constexpr int NLOAD = D / 32;       // K fragments per row and lane
  constexpr int RPL = 512 / D;        // V rows per wave load (16 bytes per lane)
  constexpr int NVL = 32 / RPL;       // loads per value head and step
  constexpr int NDT = D / 16;
  constexpr uint16_t kInf16 = DT == SAGA_DTYPE_BF16 ? 0x7f80 : 0x7c00;
  constexpr bool kF16 = DT == SAGA_DTYPE_F16;
  constexpr float kTop = 32768.f;  // f16: P and o are held times this
  __shared__ __attribute__((aligned(16))) uint32_t lds[S::LDS];

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, s = lane >> 4;
  const int split = blockIdx.x % p.nsplit;
  const int unit = blockIdx.x / p.nsplit;
  const int bi = unit / p.k_h, kh = unit - bi * p.k_h;
  const int g = p.g, g_v = p.q_h / p.v_h;
  int Leff = p.L;
  if (p.kv_len) Leff = min(Leff, max(p.kv_len[bi], 0));
  const bool hvalid = col < g;
  const int h0 = kh * g;
  const int h = h0 + (hvalid ? col : 0);
  const int vh0 = h0 / g_v;

  u32x4 qf[NLOAD];
  const char* qrow = p.q + (bi * p.q_sb + static_cast<int64_t>(h) * p.q_sh) * 2;
#pragma unroll
  for (int j = 0; j < NLOAD; ++j) qf[j] = hvalid ? ld16(qrow + (32 * j + 8 * s) * 2) : u32x4{0u, 0u, 0u, 0u};
  const char* kbase = p.k + (bi * p.k_sb + static_cast<int64_t>(kh) * p.k_sh) * 2 + 16 * s;
  const int vlc = lane % (D / 8), vlr = lane / (D / 8);  // V chunk and row of a load
  const char* vbase = p.v + (bi * p.v_sb + static_cast<int64_t>(vh0) * p.v_sh) * 2 + 16 * vlc;
  const int krow = 8 * (col >> 2) + (col & 3);

  const int beg = split * p.split_len;
  const int end = min(beg + p.split_len, Leff);
  const int nstep = end > beg ? (end - beg + 31) / 32 : 0;

  // rows past the range repeat its last one (their weight is 0)
  u32x4 kf[2][NLOAD], vr[NV][NVL];
  auto load_step = [&](int c0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const char* kr = kbase + static_cast<int64_t>(min(c0 + krow + 4 * t, end - 1)) * p.k_sl * 2;
#pragma unroll
      for (int j = 0; j < NLOAD; ++j) kf[t][j] = ld16(kr + 64 * j);
    }
#pragma unroll
    for (int i = 0; i < NVL; ++i) {
      const char* vp = vbase + static_cast<int64_t>(min(c0 + vlr + i * RPL, end - 1)) * p.v_sl * 2;
#pragma unroll
      for (int u = 0; u < NV; ++u) vr[u][i] = ld16(vp + u * p.v_sh * 2);
    }
  };

  uint32_t* vt = lds + w * NV * S::VSZ;
  const uint32_t* vtr = vt + (8 * s + (col >> 2)) * S::VROW + 2 * (col & 3);
  f32x4 o[NV][NDT];
#pragma unroll
  for (int u = 0; u < NV; ++u)
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[u][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegInf, l_run = 0.f;  // for head `col` (replicated over s)

  if (w < nstep) load_step(beg + 32 * w);
  for (int it = w; it < nstep; it += 4) {
    const int c0 = beg + 32 * it;
    float x[8];  // positions c0 + 8 s + i
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NLOAD; ++j) a = mfma_16b<DT>(kf[t][j], qf[j], a);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[4 * t + r] = a[r];
    }
    if (c0 + 32 > end) {  // repeated rows: their weight is 0, and 0 * inf is not
#pragma unroll
      for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int i = 0; i < NVL; ++i)
          if (c0 + vlr + i * RPL >= end) vr[u][i] = u32x4{0u, 0u, 0u, 0u};
    }
    // An infinite or NaN value must not meet a zero or negative term of a split
    // weight: such values (checked on the whole step's magnitude bits) are
    // taken out here and added below
    u16x2 big = {0, 0};
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int i = 0; i < NVL; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          big = __builtin_elementwise_max(big, __builtin_bit_cast(u16x2, vr[u][i][e] & 0x7fff7fffu));
    const bool special = __any(big.x >= kInf16 || big.y >= kInf16);
    if (special) {
#pragma unroll
      for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int i = 0; i < NVL; ++i) vr[u][i] = dense_pick<DT>(vr[u][i], false);
    }
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int i = 0; i < NVL; ++i)
        *reinterpret_cast<u32x4*>(vt + u * S::VSZ + (vlr + i * RPL) * S::VROW + 4 * vlc) = vr[u][i];
    dense_wave_sync();
    if (it + 4 < nstep) load_step(c0 + 128);
    __builtin_amdgcn_sched_barrier(0);  // the next step's loads are in flight from here

    float mt = kNegInf;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int pos = c0 + 8 * s + i;
      float v = x[i] * p.scale;
      if (p.mask) {
        v = v + load_as_f32(p.mask, p.mask_dt, bi * p.m_sb + static_cast<int64_t>(h) * p.m_sh +
                                                   static_cast<int64_t>(min(pos, p.L - 1)) * p.m_sl);
      }
      if (pos >= end) v = kNegInf;
      x[i] = v;
      mt = fmaxf(mt, v);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 16));
    mt = fmaxf(mt, __shfl_xor(mt, 32));
    const float m_new = fmaxf(m_run, mt);
    const float alpha = (m_run == kNegInf) ? (m_new == kNegInf ? 1.f : 0.f) : __expf(m_run - m_new);
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = m_new == kNegInf ? 0.f : __expf(x[i] - m_new);
      ps += x[i];
    }
    ps += __shfl_xor(ps, 16);
    ps += __shfl_xor(ps, 32);
    l_run = l_run * alpha + ps;
    m_run = m_new;
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) o[u][dt] *= alpha;
    u32x4 some;  // 1 where the weight is above 0
    constexpr uint32_t kOne = DT == SAGA_DTYPE_BF16 ? 0x3f80u : 0x3c00u;
#pragma unroll
    for (int i = 0; i < 4; ++i) some[i] = (x[2 * i] > 0.f ? kOne : 0u) | (x[2 * i + 1] > 0.f ? kOne << 16 : 0u);
    if constexpr (kF16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= kTop;
    }
    u32x4 pf[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) pf[k][i] = split2<DT>(x[2 * i], x[2 * i + 1]);
    auto v_frag = [&](int u, int dt) {
      const uint32_t* a = vtr + u * S::VSZ + 8 * dt;
      const u32x2 lo = lds_tr16(a), hi = lds_tr16(a + 4 * S::VROW);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const u32x4 vf = v_frag(u, dt);
#pragma unroll
        for (int k = 0; k < 3; ++k) o[u][dt] = mfma_16b<DT>(vf, pf[k], o[u][dt]);
      }
    if constexpr (kF16) {
      // what f16 terms in the first unit leave of weights below 2^-16, at most 2^-25: in a unit 2^40 times smaller, and
      // then in steps of 2^12 (8 terms reach the last bit of the smallest float)
      float unit = 1.f;
#pragma unroll 1  // a peeled pass spills
      for (int k = 0; k < 8; ++k) {
        uint32_t left = 0u;
#pragma unroll
        for (int i = 0; i < 8; ++i) left |= __float_as_uint(x[i]);
        if (!__any((left & 0x7fffffffu) != 0u)) break;
        const float up = k == 0 ? 0x1p40f : 0x1p12f;
        unit *= k == 0 ? 0x1p-40f : 0x1p-12f;
        u32x4 pt;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[2 * i] *= up;
          x[2 * i + 1] *= up;
          pt[i] = split2<DT>(x[2 * i], x[2 * i + 1]);
        }
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const f32x4 t = mfma_16b<DT>(v_frag(u, dt), pt, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int e = 0; e < 4; ++e) o[u][dt][e] = __builtin_fmaf(t[e], unit, o[u][dt][e]);
          }
      }
    }
    if (special) {  // weight > 0: inf, -inf or NaN; weight 0: NaN
      dense_wave_sync();
      for (int i = 0; i < NVL; ++i) {
        const int pos = c0 + vlr + i * RPL;
        const char* vp = vbase + static_cast<int64_t>(min(pos, end - 1)) * p.v_sl * 2;
        for (int u = 0; u < NV; ++u)
          *reinterpret_cast<u32x4*>(vt + u * S::VSZ + (vlr + i * RPL) * S::VROW + 4 * vlc) =
              pos < end ? dense_pick<DT>(ld16(vp + u * p.v_sh * 2), true) : u32x4{0u, 0u, 0u, 0u};
      }
      dense_wave_sync();
#pragma unroll
      for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[u][dt] = mfma_16b<DT>(v_frag(u, dt), some, o[u][dt]);
    }
    dense_wave_sync();  // the LDS rows are rewritten by this wave's next step
  }

  __syncthreads();  // every wave is done with the V rows
  float* Wo = reinterpret_cast<float*>(lds);
  float (*Wm)[16] = reinterpret_cast<float (*)[16]>(Wo + 4 * 16 * S::WROW);
  float (*Wl)[16] = Wm + 4;
  if (s == 0) {
    Wm[w][col] = m_run;
    Wl[w][col] = l_run;
  }
  const int u_mine = h / g_v - vh0;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    f32x4 a = o[0][dt];
#pragma unroll
    for (int u = 1; u < NV; ++u) a = u_mine == u ? o[u][dt] : a;
    if constexpr (kF16) a *= 1.f / kTop;
    *reinterpret_cast<f32x4*>(Wo + (w * 16 + col) * S::WROW + 16 * dt + 4 * s) = a;
  }
  __syncthreads();

  // merge the four waves: the split's partial, or the output when nsplit == 1
  float* part = p.part + (static_cast<int64_t>(unit) * p.nsplit + split) * g * (2 + D);
  for (int e = tid; e < g * D; e += 256) {
    const int hh = e / D, dd = e - hh * D;
    float M = kNegInf;
#pragma unroll
    for (int q = 0; q < 4; ++q) M = fmaxf(M, Wm[q][hh]);
    float l = 0.f, a = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float f = Wm[q][hh] == kNegInf ? 0.f : __expf(Wm[q][hh] - M);
      l += Wl[q][hh] * f;
      a += Wo[(q * 16 + hh) * S::WROW + dd] * f;
    }
    if (p.nsplit == 1) {
      store_from_f32(p.out, p.out_dt, bi * p.o_sb + static_cast<int64_t>(h0 + hh) * p.o_sh + dd, a / l);
    } else {
      part[hh * (2 + D) + 2 + dd] = a;
      if (dd == 0) {
        part[hh * (2 + D)] = M;
        part[hh * (2 + D) + 1] = l;
      }
    }
  }
}

// Merge the split partials of one (batch, head): block of D threads.
// Kernel 2: one block per head, kMergeGroups x D threads: thread (grp, i)
// sums dim i of the splits grp, grp + kMergeGroups, ... (all of its loads in
// one burst for up to kMergeGroups x kMergeBurst splits), then the groups
// are added in LDS in a fixed order.
constexpr int kMergeGroups = 8;
constexpr int kMergeBurst = 8;

template <int D>
__global__ void __launch_bounds__(kMergeGroups * D) dense_merge_kernel(DenseParams p) {
  constexpr int NT = kMergeGroups * D;
  __shared__ float fm[1024];
  __shared__ float red[NT / kWave];
  __shared__ float og[kMergeGroups][D];
  const int unit = blockIdx.x / p.g, hh = blockIdx.x - unit * p.g;
  const int bi = unit / p.k_h, kh = unit - bi * p.k_h;
  const int tid = threadIdx.x, grp = tid / D, i = tid - grp * D;
  const int64_t stride = static_cast<int64_t>(p.g) * (2 + D);  // between splits
  const float* base = p.part + static_cast<int64_t>(unit) * p.nsplit * stride + hh * (2 + D);
  // (max, sum) of every split, then the common max
  float mloc = kNegInf;
  for (int q = tid; q < p.nsplit; q += NT) {
    const float m = base[q * stride];
    fm[q] = m;
    mloc = fmaxf(mloc, m);
  }
  const float M = block_max<NT / kWave>(mloc, red);
  float lloc = 0.f;
  for (int q = tid; q < p.nsplit; q += NT) {
    const float f = fm[q] == kNegInf ? 0.f : __expf(fm[q] - M);
    lloc += base[q * stride + 1] * f;
    fm[q] = f;
  }
  const float l = block_sum<NT / kWave>(lloc, red);  // orders the fm writes too
  // dim i of this group's splits: independent loads, kMergeBurst in flight
  float o = 0.f;
  for (int q0 = grp; q0 < p.nsplit; q0 += kMergeGroups * kMergeBurst) {
    float ov[kMergeBurst];
#pragma unroll
    for (int u = 0; u < kMergeBurst; ++u) {
      const int q = q0 + u * kMergeGroups;
      ov[u] = q < p.nsplit ? base[q * stride + 2 + i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kMergeBurst; ++u) {
      const int q = q0 + u * kMergeGroups;
      if (q < p.nsplit) o += ov[u] * fm[q];
    }
  }
  og[grp][i] = o;
  __syncthreads();
  if (grp == 0) {
    float t = og[0][i];
#pragma unroll
    for (int g2 = 1; g2 < kMergeGroups; ++g2) t += og[g2][i];
    store_from_f32(p.out, p.out_dt, bi * p.o_sb + static_cast<int64_t>(kh * p.g + hh) * p.o_sh + i, t / l);
  }
}

// Value heads of a unit if every one lies wholly in it (or it in one), else 0.
static int dense_unit_value_heads(const DenseParams& p) {
  const int g_v = p.q_h / p.v_h;
  if (g_v % p.g == 0) return 1;
  return p.g % g_v == 0 ? p.g / g_v : 0;
}

template <int DT, int D>
static void launch_dense_split(const DenseParams& p, dim3 grid, hipStream_t st) {
  if constexpr (DT != SAGA_DTYPE_F32) {
    const int nv = dense_unit_value_heads(p);
    bool done = true;
    if (nv == 1) {
      hipLaunchKernelGGL((dense_mfma_kernel<DT, D, 1>), grid, dim3(256), 0, st, p);
    } else if (nv == 2) {
      hipLaunchKernelGGL((dense_mfma_kernel<DT, D, 2>), grid, dim3(256), 0, st, p);
    } else {
      done = D == 64 && nv == 5;
      if constexpr (D == 64) {
        if (nv == 5) hipLaunchKernelGGL((dense_mfma_kernel<DT, D, 5>), grid, dim3(256), 0, st, p);
      }
    }
    if (done) return;
  }
  hipLaunchKernelGGL((dense_split_kernel<DT, D, kDenseSubDefault>), grid, dim3(256), 0, st, p);
}

template <int DT>
static hipError_t launch_dense_typed(int d, const DenseParams& p, hipStream_t st) {
  const unsigned blocks = static_cast<unsigned>(p.b * p.k_h * p.nsplit);
  const unsigned heads = static_cast<unsigned>(p.b * p.k_h * p.g);
  if (d == 128) {
    launch_dense_split<DT, 128>(p, dim3(blocks), st);
    if (p.nsplit > 1)
      hipLaunchKernelGGL((dense_merge_kernel<128>), dim3(heads), dim3(kMergeGroups * 128), 0, st, p);
  } else {
    launch_dense_split<DT, 64>(p, dim3(blocks), st);
    if (p.nsplit > 1)
      hipLaunchKernelGGL((dense_merge_kernel<64>), dim3(heads), dim3(kMergeGroups * 64), 0, st, p);
  }
  return hipGetLastError();
}

hipError_t launch_dense_decode(int dtype, int d, const DenseParams& p, hipStream_t st) {
  if (dtype == SAGA_DTYPE_BF16) return launch_dense_typed<SAGA_DTYPE_BF16>(d, p, st);
  if (dtype == SAGA_DTYPE_F16) return launch_dense_typed<SAGA_DTYPE_F16>(d, p, st);
  return launch_dense_typed<SAGA_DTYPE_F32>(d, p, st);
}

}  // namespace saga
