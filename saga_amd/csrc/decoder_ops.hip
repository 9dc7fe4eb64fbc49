// Decode-step kernels around the attention path (one launch each):
//   * rope_kv_append: the new tokens' q/k/v from the fused projection, RoPE on
//     q and k, k/v written into the separate key-head / value-head caches
//     (replaces apply_rotary_pos_emb + StaticLayer.update's index_copy_,
//     transformers models/qwen2/modeling_qwen2.py:211-214 and
//     cache_utils.py:455-487, with the caches laid out as speedup.py:119-139);
//   * rmsnorm: y = w * x / sqrt(mean(x^2) + eps) per row (Qwen2RMSNorm);
//   * silu_mul: act = silu(gate) * up over a fused [gate | up] projection;
//   * unpack: packed decode weights back to row-major for a prompt's GEMMs.
// All arithmetic in fp32, one rounding to the storage dtype.
#include "common.cuh"
#include "kernels.h"

namespace saga {

// 8 values of a 16-bit type in one 16-byte vector, from fp32.
template <int DT>
__device__ __forceinline__ u32x4 pack16(const float (&f)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = DT == SAGA_DTYPE_BF16 ? f32_to_bf16_bits(f[2 * i]) : f32_to_f16_bits(f[2 * i]);
    const uint32_t hi = DT == SAGA_DTYPE_BF16 ? f32_to_bf16_bits(f[2 * i + 1]) : f32_to_f16_bits(f[2 * i + 1]);
    w[i] = lo | (hi << 16);
  }
  return u32x4{w[0], w[1], w[2], w[3]};
}

// A prompt's rotation + append, 16-bit types with 16-byte aligned rows (the
// kernel below takes every other call, and few tokens).  A block computes the
// cos / sin of its tokens (1 or 2) once, in LDS, and applies them to all of
// their heads in 16-byte vectors: bound by the bytes of the projection (read
// once, written once).  One 64-lane block per (token, head) recomputed the
// same powf and sincosf for every head and moved 2 bytes per lane: 4001 tokens
// of 15 heads, d 128 (31 MB) 23.4 us, here 9.2.
template <int DT>
__global__ void __launch_bounds__(256) rope_kv_append_vec_kernel(RopeParams p, int tokens) {
  extern __shared__ float rot[];  // [tokens][2][d / 2]: cos, sin
  const int half = p.d / 2, nh = half / 8, nv = p.d / 8;
  const int t0 = blockIdx.x * tokens, nt = min(tokens, p.N - t0);
  for (int e = threadIdx.x; e < nt * half; e += 256) {
    const int t = e / half, i = e - t * half;
    float cs, sn;
    rope_cos_sin(p.pos[t0 + t], i, p.d, p.theta, cs, sn);
    rot[2 * t * half + i] = cs;
    rot[(2 * t + 1) * half + i] = sn;
  }
  __syncthreads();
  const int nrot = (p.n_q + p.n_k) * nh;    // rotated vector pairs per token
  const int per = nrot + p.n_v * nv;        // + copied v vectors
  const float nan = __builtin_nanf("");
  for (int e = threadIdx.x; e < nt * per; e += 256) {
    const int t = e / per, w = e - t * per, n = t0 + t;
    const int pos = p.pos[n];
    const int b = p.batch ? p.batch[n] : n;
    const bool ok = pos >= 0 && pos < p.Lmax && b >= 0 && b < p.B;
    const uint16_t* row = static_cast<const uint16_t*>(p.qkv) + static_cast<int64_t>(n) * p.qkv_ld;
    if (w < nrot) {
      const int hh = w / nh, i = 8 * (w - hh * nh);
      float x1[8], x2[8], y1[8], y2[8];
      unpack16<DT>(ld16(row + hh * p.d + i), x1);
      unpack16<DT>(ld16(row + hh * p.d + i + half), x2);
      const float* cs = rot + 2 * t * half + i;
      const float* sn = cs + half;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        y1[j] = x1[j] * cs[j] - x2[j] * sn[j];
        y2[j] = x2[j] * cs[j] + x1[j] * sn[j];
      }
      uint16_t* dst = nullptr;
      if (hh < p.n_q) {
        dst = static_cast<uint16_t*>(p.q_out) + static_cast<int64_t>(n) * p.q_sn + static_cast<int64_t>(hh) * p.q_sh;
        if (!ok) {
#pragma unroll
          for (int j = 0; j < 8; ++j) y1[j] = y2[j] = nan;
        }
      } else if (ok) {
        dst = static_cast<uint16_t*>(p.k_cache) + b * p.k_sb + static_cast<int64_t>(hh - p.n_q) * p.k_sh +
              static_cast<int64_t>(pos) * p.k_sl;
      }
      if (dst) {
        *reinterpret_cast<u32x4*>(dst + i) = pack16<DT>(y1);
        *reinterpret_cast<u32x4*>(dst + i + half) = pack16<DT>(y2);
      }
    } else if (ok) {
      const int c = w - nrot, vh = c / nv, i = 8 * (c - vh * nv);
      uint16_t* dst = static_cast<uint16_t*>(p.v_cache) + b * p.v_sb + static_cast<int64_t>(vh) * p.v_sh +
                      static_cast<int64_t>(pos) * p.v_sl;
      *reinterpret_cast<u32x4*>(dst + i) = ld16(row + (p.n_q + p.n_k + vh) * p.d + i);
    }
  }
}

// One 64-lane block per (token n, head hh); heads are ordered q, k, v as in
// the fused projection row.  q and k heads rotate pairs (i, i + d/2), v heads
// are copied.  Any dtype, alignment and even d.
__global__ void __launch_bounds__(64) rope_kv_append_kernel(RopeParams p) {
  const int n = blockIdx.x, hh = blockIdx.y;
  const int half = p.d / 2;
  const int pos = p.pos[n];
  const int b = p.batch ? p.batch[n] : n;
  const bool ok = pos >= 0 && pos < p.Lmax && b >= 0 && b < p.B;
  const int64_t base = static_cast<int64_t>(n) * p.qkv_ld + static_cast<int64_t>(hh) * p.d;
  if (hh < p.n_q + p.n_k) {
    for (int i = threadIdx.x; i < half; i += 64) {
      float cs, sn;
      rope_cos_sin(pos, i, p.d, p.theta, cs, sn);
      const float x1 = load_as_f32(p.qkv, p.dt, base + i);
      const float x2 = load_as_f32(p.qkv, p.dt, base + i + half);
      const float y1 = x1 * cs - x2 * sn;
      const float y2 = x2 * cs + x1 * sn;
      if (hh < p.n_q) {
        const int64_t qo = static_cast<int64_t>(n) * p.q_sn + static_cast<int64_t>(hh) * p.q_sh;
        store_from_f32(p.q_out, p.dt, qo + i, ok ? y1 : __builtin_nanf(""));
        store_from_f32(p.q_out, p.dt, qo + i + half, ok ? y2 : __builtin_nanf(""));
      } else if (ok) {
        const int kh = hh - p.n_q;
        const int64_t ko = b * p.k_sb + static_cast<int64_t>(kh) * p.k_sh + static_cast<int64_t>(pos) * p.k_sl;
        store_from_f32(p.k_cache, p.dt, ko + i, y1);
        store_from_f32(p.k_cache, p.dt, ko + i + half, y2);
      }
    }
  } else if (ok) {
    const int vh = hh - p.n_q - p.n_k;
    const int64_t vo = b * p.v_sb + static_cast<int64_t>(vh) * p.v_sh + static_cast<int64_t>(pos) * p.v_sl;
    for (int i = threadIdx.x; i < p.d; i += 64) store_from_f32(p.v_cache, p.dt, vo + i, load_as_f32(p.qkv, p.dt, base + i));
  }
}

// 16-byte rows: a 16-bit type, vectors of 8 in each rotated half, every
// stride a multiple of 8 elements.
static bool rope_vec(const RopeParams& p) {
  const int64_t st = p.qkv_ld | p.q_sn | p.q_sh | p.k_sb | p.k_sh | p.k_sl | p.v_sb | p.v_sh | p.v_sl;
  const uintptr_t a = reinterpret_cast<uintptr_t>(p.qkv) | reinterpret_cast<uintptr_t>(p.q_out) |
                      reinterpret_cast<uintptr_t>(p.k_cache) | reinterpret_cast<uintptr_t>(p.v_cache);
  return p.dt != SAGA_DTYPE_F32 && p.d % 16 == 0 && p.d <= 1024 && st % 8 == 0 && a % 16 == 0;
}

hipError_t launch_rope_kv_append(const RopeParams& p, hipStream_t st) {
  // Measured (us; heads q + k + v): element form, 1, 2, 4 tokens per block.  15 heads, d 128: 64 tokens 3.0, 3.5, 3.8,
  // 4.9; 128 3.4, 3.5, 3.8, 4.9; 256 4.0, 3.6, 3.9, 5.0; 1024 7.7, 4.2, 4.7, 5.4; 2048 12.8, 6.2, 5.8, 6.5; 4001 23.4,
  // 10.6, 9.2, 9.3.  21 heads, d 64: 128 3.4, 3.4, 3.6, 4.7; 4001 28.7, 8.4, 7.9, 7.6.  (The element form's blocks are
  // its tokens times heads; at 2^25 tokens a launch of 2 per block ends.)
  const int64_t blocks = static_cast<int64_t>(p.N) * (p.n_q + p.n_k + p.n_v);
  if (rope_vec(p) && blocks >= 3072 && p.N < (1 << 25)) {
    const int tokens = p.N < 1536 ? 1 : 2;
    const dim3 grid((p.N + tokens - 1) / tokens);
    const size_t lds = sizeof(float) * tokens * p.d;
    if (p.dt == SAGA_DTYPE_BF16)
      hipLaunchKernelGGL((rope_kv_append_vec_kernel<SAGA_DTYPE_BF16>), grid, dim3(256), lds, st, p, tokens);
    else
      hipLaunchKernelGGL((rope_kv_append_vec_kernel<SAGA_DTYPE_F16>), grid, dim3(256), lds, st, p, tokens);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(rope_kv_append_kernel, dim3(p.N, p.n_q + p.n_k + p.n_v), dim3(64), 0, st, p);
  return hipGetLastError();
}

// The rotations of a decode step's token rows, computed once per step for
// every layer's fused q/k/v projection (the same rope_cos_sin as the kernels
// that compute them in place: identical values).
__global__ void __launch_bounds__(256) rope_table_kernel(const int32_t* pos, int N, int d, float theta,
                                                         float* table) {
  const int half = d / 2;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= N * half) return;
  const int n = t / half, i = t - n * half;
  float cs, sn;
  rope_cos_sin(pos[n], i, d, theta, cs, sn);
  *reinterpret_cast<f32x2*>(table + 2 * static_cast<int64_t>(t)) = f32x2{cs, sn};
}

hipError_t launch_rope_table(const int32_t* pos, int N, int d, float theta, float* table, hipStream_t st) {
  const int total = N * (d / 2);
  hipLaunchKernelGGL(rope_table_kernel, dim3((total + 255) / 256), dim3(256), 0, st, pos, N, d, theta, table);
  return hipGetLastError();
}

// The opening of a decode step, one block per token row b: x[b] =
// embed[tokens[b]] (16-byte chunks when rows allow, else element by element,
// exact for every float dtype; a token id outside [0, V) writes a NaN row)
// and, with a table, the row's rotations as rope_table_kernel computes them.
__global__ void __launch_bounds__(256) embed_rope_kernel(EmbedParams p) {
  const int b = blockIdx.x, tid = threadIdx.x;
  const int64_t tok = p.tokens[b];
  const bool ok = tok >= 0 && tok < p.V;
  if (ok && p.vec) {
    const int64_t es = p.dt == SAGA_DTYPE_F32 ? 4 : 2;
    const char* src = static_cast<const char*>(p.embed) + tok * p.e_ld * es;
    char* dst = static_cast<char*>(p.x) + static_cast<int64_t>(b) * p.x_ld * es;
    const int chunks = static_cast<int>(p.H * es / 16);
    for (int c = tid; c < chunks; c += 256) *reinterpret_cast<u32x4*>(dst + 16 * c) = ld16(src + 16 * c);
  } else {
    for (int i = tid; i < p.H; i += 256)
      store_from_f32(p.x, p.dt, static_cast<int64_t>(b) * p.x_ld + i,
                     ok ? load_as_f32(p.embed, p.dt, tok * p.e_ld + i) : __builtin_nanf(""));
  }
  if (p.table) {
    const int half = p.d / 2;
    const int pos = p.pos[b];
    for (int i = tid; i < half; i += 256) {
      float cs, sn;
      rope_cos_sin(pos, i, p.d, p.theta, cs, sn);
      *reinterpret_cast<f32x2*>(p.table + 2 * (static_cast<int64_t>(b) * half + i)) = f32x2{cs, sn};
    }
  }
}

hipError_t launch_embed_rope(const EmbedParams& p, hipStream_t st) {
  hipLaunchKernelGGL(embed_rope_kernel, dim3(p.B), dim3(256), 0, st, p);
  return hipGetLastError();
}

// The close of a decode step: every row's position and cache length + 1.
__global__ void __launch_bounds__(256) advance_kernel(int32_t* pos, int32_t* kv_len, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  if (pos) pos[i] += 1;
  if (kv_len) kv_len[i] += 1;
}

hipError_t launch_advance(int32_t* pos, int32_t* kv_len, int n, hipStream_t st) {
  hipLaunchKernelGGL(advance_kernel, dim3((n + 255) / 256), dim3(256), 0, st, pos, kv_len, n);
  return hipGetLastError();
}

// Rows of a 16-bit type with 16-byte aligned strides and H <= 64 * 8 *
// kNormVecs: one wave per row, the row held in registers between the sum of
// squares and the scaling, so it is read once, 16 bytes per lane (4001 rows
// of 1536 bf16, 25 MB: 16.5 us with one block per row and 2 bytes per lane,
// here 7.3).
constexpr int kNormVecs = 16;

template <int DT, int NV>
__global__ void __launch_bounds__(256) rmsnorm_vec_kernel(RowParams p) {
  const int lane = threadIdx.x & 63, n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= p.N) return;
  const int nvec = p.H / 8;
  const uint16_t* x = static_cast<const uint16_t*>(p.x) + static_cast<int64_t>(n) * p.x_ld;
  u32x4 v[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = lane + 64 * j;
    v[j] = c < nvec ? ld16(x + 8 * c) : u32x4{0u, 0u, 0u, 0u};
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    float f[8];
    unpack16<DT>(v[j], f);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += f[i] * f[i];
  }
  ss = wave_sum(ss);
  const float r = rsqrtf(ss / static_cast<float>(p.H) + p.eps);
  uint16_t* y = static_cast<uint16_t*>(p.y) + static_cast<int64_t>(n) * p.y_ld;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = lane + 64 * j;
    if (c < nvec) {
      float f[8], w[8];
      unpack16<DT>(v[j], f);
      unpack16<DT>(ld16(static_cast<const uint16_t*>(p.w) + 8 * c), w);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = w[i] * (f[i] * r);
      *reinterpret_cast<u32x4*>(y + 8 * c) = pack16<DT>(f);
    }
  }
}

__global__ void __launch_bounds__(256) rmsnorm_kernel(RowParams p) {
  __shared__ float red[4];
  const int n = blockIdx.x;
  const int64_t xi = static_cast<int64_t>(n) * p.x_ld;
  float ss = 0.f;
  for (int i = threadIdx.x; i < p.H; i += 256) {
    const float v = load_as_f32(p.x, p.dt, xi + i);
    ss += v * v;
  }
  ss = block_sum<4>(ss, red);
  const float r = rsqrtf(ss / static_cast<float>(p.H) + p.eps);
  const int64_t yi = static_cast<int64_t>(n) * p.y_ld;
  for (int i = threadIdx.x; i < p.H; i += 256) {
    const float v = load_as_f32(p.x, p.dt, xi + i);
    store_from_f32(p.y, p.dt, yi + i, load_as_f32(p.w, p.dt, i) * (v * r));
  }
}

// 16-byte vectors of a 16-bit type in every row of x, y (and w, when given).
static bool row_vec(const RowParams& p) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.y) |
                      reinterpret_cast<uintptr_t>(p.w);
  return p.dt != SAGA_DTYPE_F32 && p.H % 8 == 0 && (p.x_ld | p.y_ld) % 8 == 0 && a % 16 == 0;
}

template <int DT>
static void launch_rmsnorm_vec(const RowParams& p, hipStream_t st) {
  const dim3 grid((p.N + 3) / 4);
  const int nv = (p.H / 8 + 63) / 64;
  if (nv <= 4) hipLaunchKernelGGL((rmsnorm_vec_kernel<DT, 4>), grid, dim3(256), 0, st, p);
  else if (nv <= 8) hipLaunchKernelGGL((rmsnorm_vec_kernel<DT, 8>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((rmsnorm_vec_kernel<DT, kNormVecs>), grid, dim3(256), 0, st, p);
}

hipError_t launch_rmsnorm(const RowParams& p, hipStream_t st) {
  if (row_vec(p) && p.H <= 64 * 8 * kNormVecs) {
    if (p.dt == SAGA_DTYPE_BF16) launch_rmsnorm_vec<SAGA_DTYPE_BF16>(p, st);
    else launch_rmsnorm_vec<SAGA_DTYPE_F16>(p, st);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(p.N), dim3(256), 0, st, p);
  return hipGetLastError();
}

// 16-bit rows with 16-byte aligned strides: 8 outputs per thread, each wave
// reading 1 KB of gates and 1 KB of ups in a row.  Bound by HBM (3 H values
// per token): 4001 x 8960 bf16, 215 MB, 38 us (5.6 TB/s); one element per
// thread and 2 bytes per lane took 112.
template <int DT>
__global__ void __launch_bounds__(256) silu_mul_vec_kernel(RowParams p) {
  const uint32_t nvec = p.H / 8;
  const uint32_t e = blockIdx.x * 256 + threadIdx.x;  // below 2^32: the launch sees to it
  const int64_t n = e / nvec;
  if (n >= p.N) return;
  const int i = 8 * static_cast<int>(e % nvec);
  const uint16_t* x = static_cast<const uint16_t*>(p.x) + n * p.x_ld + i;
  const u32x4 gv = ld16(x), uv = ld16(x + p.H);
  float g[8], u[8];
  unpack16<DT>(gv, g);
  unpack16<DT>(uv, u);
#pragma unroll
  for (int j = 0; j < 8; ++j) g[j] = g[j] / (1.0f + expf(-g[j])) * u[j];
  *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.y) + n * p.y_ld + i) = pack16<DT>(g);
}

// y[n, i] = silu(x[n, i]) * x[n, H + i]; H = width of the output row.
__global__ void __launch_bounds__(256) silu_mul_kernel(RowParams p) {
  const int n = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.H) return;
  const int64_t xi = static_cast<int64_t>(n) * p.x_ld;
  const float g = load_as_f32(p.x, p.dt, xi + i);
  const float u = load_as_f32(p.x, p.dt, xi + p.H + i);
  store_from_f32(p.y, p.dt, static_cast<int64_t>(n) * p.y_ld + i, g / (1.0f + expf(-g)) * u);
}

hipError_t launch_silu_mul(const RowParams& p, hipStream_t st) {
  // Vectors from 600000 outputs on: below, 8 serial SiLUs per thread take longer than the memory (64 x 8960: 2.9 us
  // in either form, 8 x 8960 2.6 against 2.2, 512 x 512 2.7 against 2.3; 256 x 2560 2.9 against 3.0, 128 x 8960 3.4
  // against 3.7).  A launch holds less than 2^32 threads in x, which the element form divides over y.
  const int64_t outputs = static_cast<int64_t>(p.N) * p.H, blocks = (outputs / 8 + 255) / 256;
  if (row_vec(p) && outputs >= 600000 && blocks < (1LL << 24)) {
    const dim3 grid(static_cast<unsigned>(blocks));
    if (p.dt == SAGA_DTYPE_BF16)
      hipLaunchKernelGGL((silu_mul_vec_kernel<SAGA_DTYPE_BF16>), grid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((silu_mul_vec_kernel<SAGA_DTYPE_F16>), grid, dim3(256), 0, st, p);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(silu_mul_kernel, dim3((p.H + 255) / 256, p.N), dim3(256), 0, st, p);
  return hipGetLastError();
}

// Packed decode weights (16-row or 8-row tiles, layouts in saga_amd.h) to
// row-major, several weights in one launch: a block moves one tile of rows
// by 16 KB / rows of columns, 16 bytes per lane, its four loads in flight
// together, the writes of a wave 1 KB of one row.  Rows of a rotated head of
// head_rows rows go from rotary-pair order [0, d/2, 1, d/2 + 1, ...] to
// natural order on the way.  Bound by HBM (each weight read and written
// once): the q/k/v, o and down weights of a 1.5B layer, 76 MB moved, in 16.4 us
// (4.7 TB/s).  As torch permutes (and, in place of the row order, a reordering
// pass over the prompt's q/k/v rows) they and gate/up took 190 us at 4001 tokens.
__global__ void __launch_bounds__(256) unpack_kernel(UnpackParams p) {
  int it = 0;
  while (it + 1 < p.n && static_cast<int>(blockIdx.x) >= p.item[it + 1].block0) ++it;
  const UnpackParams::Item& w = p.item[it];
  const int rows = w.tile_rows;                 // 16 or 8
  const int cw = rows == 16 ? 64 : 128;         // 16-byte chunks of a row per block
  const int nchunk = w.K / 8, nc = (nchunk + cw - 1) / cw;
  const int blk = blockIdx.x - w.block0;
  const int tile = blk / nc, q = (blk - tile * nc) * cw + threadIdx.x % cw;
  if (q >= nchunk) return;
  const int r0 = threadIdx.x / cw, dr = 256 / cw;
  u32x4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = r0 + u * dr;
    // 16-row tiles: fragment q / 4 of 32 columns; 8-row tiles: fragment q / 8
    // of 64, its second 32 columns in fragment rows 8-15
    const int64_t frag = rows == 16 ? static_cast<int64_t>(tile) * (w.K / 32) + q / 4
                                    : static_cast<int64_t>(tile) * (w.K / 64) + q / 8;
    const int fr = rows == 16 ? r : 8 * ((q >> 2) & 1) + r;
    v[u] = ld16(static_cast<const uint16_t*>(w.src) + frag * 512 + fr * 32 + 8 * (q & 3));
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int n = tile * rows + r0 + u * dr;
    int dst = n;
    if (w.head_rows > 0) {
      const int h = n / w.head_rows, j = n - h * w.head_rows;
      if (h < w.rot_heads) dst = h * w.head_rows + (j & 1) * (w.head_rows / 2) + j / 2;
    }
    *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(w.dst) + static_cast<int64_t>(dst) * w.dst_ld + 8 * q) = v[u];
  }
}

hipError_t launch_unpack(UnpackParams& p, hipStream_t st) {
  int64_t blocks = 0;
  for (int i = 0; i < p.n; ++i) {
    const int cw = p.item[i].tile_rows == 16 ? 64 : 128;
    p.item[i].block0 = static_cast<int>(blocks);
    blocks += static_cast<int64_t>(p.item[i].N / p.item[i].tile_rows) * ((p.item[i].K / 8 + cw - 1) / cw);
    if (blocks >= (1LL << 31)) return hipErrorInvalidValue;
  }
  if (blocks) hipLaunchKernelGGL(unpack_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, p);
  return hipGetLastError();
}

}  // namespace saga
