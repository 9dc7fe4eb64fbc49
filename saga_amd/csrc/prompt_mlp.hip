// Gate/up projection of a prompt with its activation:
// y[t, j] = silu(g) * u, (g, u) = rows 2j, 2j + 1 of x[t, :] . W[n, :], W packed
// [N/16][K/32][16][32] as the decode step keeps it (pack_gemv_weight).
//
// Bound by the matrix cores.  A block computes 32 MF tokens x 64 NF rows of W
// in 8 waves (2 along the tokens, 4 along the rows).  A packed tile is an MFMA A
// fragment already, so W goes from memory to registers, 1 KB per load, D
// k steps (of 64) ahead; x goes through LDS in fragment order, double-buffered,
// its 16-byte units XOR-placed so that neither the row-wise writes nor the
// fragment reads meet in a bank.  gate and up meet in one lane, so the
// [T, N] projection never exists in memory and W is not unpacked first.
// Against unpacking W, the library GEMM and silu_mul (one box, us): N 17920,
// K 1536: 4001 tokens 239 -> 198 (1.11 PFLOP/s), 8192 451 -> 381, 1500
// 107 -> 84, 700 65 -> 40, 128 41 -> 19; N 5120, K 960: 4001 73 -> 49, 512
// 39 -> 13.
#include <algorithm>

#include "common.cuh"
#include "kernels.h"

namespace saga {
namespace {

constexpr int kMlpThreads = 512;
constexpr int kMlpStep = 64;  // k per step
constexpr int kXcds = 8;
constexpr int64_t kCus = 256;
constexpr int kMlpGroup = 8;  // token tiles that share a sweep over W (their x and the W tiles stay in an XCD's L2)

// LDS of a block: two x buffers, or the output rows (TN / 2 values, padded).
template <int MF, int NF>
constexpr int mlp_lds() {
  constexpr int x = 2 * 32 * MF * kMlpStep * 2, out = 32 * MF * (64 * NF + 16);
  return x > out ? x : out;
}

// Tokens from t0, W rows from n0.
template <int MF, int NF, int D>
__device__ __forceinline__ void mlp_block(const PromptMlpParams& p, int t0, int n0, char* lds) {
  constexpr int TM = 32 * MF, TN = 64 * NF;
  constexpr int NX = TM / 64;                // 16-byte units of x per thread and step
  constexpr int kLoads = NX + 2 * NF;        // global loads per step
  constexpr int XBYTES = TM * kMlpStep * 2;  // one x buffer
  constexpr int OROW = TN + 16;              // bytes of an output row in LDS
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, s = lane >> 4;
  const int wm = w & 1, wn = w >> 1;

  const int ksteps = p.K / kMlpStep;

  // x: unit i of the thread is k chunk c (8 values) of token row r
  const char* xsrc[NX];
  int xdst[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int u = i * kMlpThreads + tid, r = u >> 3, c = u & 7;
    xsrc[i] = static_cast<const char*>(p.x) + (static_cast<int64_t>(min(t0 + r, p.T - 1)) * p.x_ld + 8 * c) * 2;
    xdst[i] = ((r >> 4) * 2 + (c >> 2)) * 1024 + ((c & 3) * 16 + ((r & 15) ^ c)) * 16;
  }
  const char* wsrc[NF];
  const int wtiles = p.N / 16;
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    const int wt = min(n0 / 16 + wn * NF + j, wtiles - 1);
    wsrc[j] = static_cast<const char*>(p.w) + static_cast<int64_t>(wt) * ksteps * 2048 + col * 64 + s * 16;
  }
  int xread[2];  // this lane's unit in the fragment of k half h
#pragma unroll
  for (int h = 0; h < 2; ++h) xread[h] = (wm * MF * 2 + h) * 1024 + (s * 16 + (col ^ (4 * h + s))) * 16;

  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Loads run D steps ahead of their use, in a ring of D + 1 register stages.
  constexpr int R = D + 1, F = 2 * MF;
  u32x4 xs[R][NX], wf[R][2 * NF];
  auto load_x = [&](int k, int i, u32x4 (&x)[NX]) { x[i] = ld16(xsrc[i] + k * 128); };
  auto load_w = [&](int k, int i, u32x4 (&f)[2 * NF]) { f[i] = ld16(wsrc[i % NF] + k * 2048 + (i / NF) * 1024); };
  auto store_x = [&](int buf, const u32x4 (&x)[NX]) {
#pragma unroll
    for (int i = 0; i < NX; ++i) *reinterpret_cast<u32x4*>(lds + buf * XBYTES + xdst[i]) = x[i];
  };
  // One step.  Fragment f of x (k half f / MF) is read kAhead fragments ahead
  // of its NF products, and one global load goes between the products of each
  // fragment: issued at once they fill the CU's address queue (16 cycles a
  // load, 96 loads) and every wave waits there with its products undone.  The
  // step's own x is in LDS; the next step's goes into the other buffer last
  // (read by every wave before this step's barrier).
  // 4001 tokens, 17920 x 1536: loads at the step's start 250 us, spread 209
  // (both with five whole rounds of blocks); then 190 with 4 fragments ahead,
  // 188 with 3 (no more than boxes differ), 203 with 6 (spills), 226 without
  // the scheduling fences between the fragments.
  constexpr int kAhead = 4;
  auto step = [&](int k, int st) {
    lds_sync();
    const int kn = min(k + D, ksteps - 1), sn = (st + D) % R;
    const char* xb = lds + (k & 1) * XBYTES;
    u32x4 xf[F];
#pragma unroll
    for (int f = 0; f < kAhead; ++f) xf[f] = *reinterpret_cast<const u32x4*>(xb + xread[f / MF] + (f % MF) * 2048);
#pragma unroll
    for (int f = 0; f < F; ++f) {
#pragma unroll
      for (int q = f * kLoads / F; q < (f + 1) * kLoads / F; ++q) {
        if (q < NX) load_x(kn, q, xs[sn]);
        else load_w(kn, q - NX, wf[sn]);
      }
#pragma unroll
      for (int j = 0; j < NF; ++j)
        acc[f % MF][j] = mfma_16b<SAGA_DTYPE_BF16>(wf[st][(f / MF) * NF + j], xf[f], acc[f % MF][j]);
      const int g = f + kAhead;
      if (g < F) xf[g] = *reinterpret_cast<const u32x4*>(xb + xread[g / MF] + (g % MF) * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
    store_x((k + 1) & 1, xs[(st + 1) % R]);
  };

#pragma unroll
  for (int d = 0; d < D; ++d) {
#pragma unroll
    for (int i = 0; i < NX; ++i) load_x(min(d, ksteps - 1), i, xs[d]);
#pragma unroll
    for (int i = 0; i < 2 * NF; ++i) load_w(min(d, ksteps - 1), i, wf[d]);
  }
  store_x(0, xs[0]);
  for (int k0 = 0; k0 < ksteps; k0 += R) {
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (k0 + i < ksteps) step(k0 + i, i);
  }

  // lane (col, s): token col of fragment i, rows 4s .. 4s + 3 = two (gate, up)
  // pairs; through LDS into rows of 16-byte stores
  lds_sync();
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      float o[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float g = acc[i][j][2 * q], u = acc[i][j][2 * q + 1];
        // The hardware's reciprocal flushes results below 2^-126 (gates from -87.3
        // down to -88.7, where exp overflows): taken in 2^-32 units.  With the
        // hardware's exp the activation is within 8e-6 of exact before its
        // rounding to bf16; expf and a division cost 10 % of the kernel (4001
        // tokens, 17920 x 1536: 201 -> 220 us).
        o[q] = g * (__builtin_amdgcn_rcpf((1.0f + __expf(-g)) * 0x1p-32f) * 0x1p-32f) * u;
      }
      const uint32_t bits = f32_to_bf16_bits(o[0]) | (static_cast<uint32_t>(f32_to_bf16_bits(o[1])) << 16);
      *reinterpret_cast<uint32_t*>(lds + (16 * (wm * MF + i) + col) * OROW + (wn * NF + j) * 16 + s * 4) = bits;
    }
  lds_sync();
  constexpr int UPR = TN / 16;  // 16-byte units (W tiles) per output row
#pragma unroll 4
  for (int u = tid; u < TM * UPR; u += kMlpThreads) {
    const int r = u / UPR, c = u - r * UPR;
    if (t0 + r < p.T && n0 / 16 + c < wtiles) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * OROW + c * 16);
      *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.y) + static_cast<int64_t>(t0 + r) * p.y_ld + n0 / 2 + 8 * c) = v;
    }
  }
}

// Position of block b of n in the tile list: blocks go to the XCDs round
// robin, XCD i takes the i-th contiguous part.
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int xcd = b % kXcds, rem = n % kXcds;
  return xcd * (n / kXcds) + min(xcd, rem) + b / kXcds;
}

// Token and W tile of entry i of the list (groups of kMlpGroup token tiles, W
// tiles within).
__device__ __forceinline__ void list_tile(const PromptMlpParams& p, int i, int& mt, int& nt) {
  const int gsize = kMlpGroup * p.ntiles;
  const int grp = i / gsize, in = i - grp * gsize;
  const int gm = min(kMlpGroup, p.mtiles - grp * kMlpGroup);
  nt = in / gm;
  mt = grp * kMlpGroup + in - nt * gm;
}

// One block per tile of the list for the first p.whole tiles, then (NF even)
// two blocks per tile, one half of its W rows each: the last round's tiles
// when they would leave half the CUs idle.
template <int MF, int NF, int D>
__global__ void __launch_bounds__(kMlpThreads, 2) prompt_mlp_kernel(PromptMlpParams p) {
  __shared__ __attribute__((aligned(16))) char lds[mlp_lds<MF, NF>()];
  const int b = blockIdx.x;
  int mt, nt;
  if constexpr (NF == 4) {
    if (b >= p.whole) {
      const int h = xcd_tile(b - p.whole, gridDim.x - p.whole);
      list_tile(p, p.whole + h / 2, mt, nt);
      const int n0 = nt * 64 * NF + (h & 1) * 32 * NF;
      if (n0 < p.N) mlp_block<MF, NF / 2, D>(p, mt * 32 * MF, n0, lds);
      return;
    }
  }
  list_tile(p, xcd_tile(b, p.whole), mt, nt);
  mlp_block<MF, NF, D>(p, mt * 32 * MF, nt * 64 * NF, lds);
}

template <int MF, int NF, int D>
hipError_t launch_shape(PromptMlpParams p, bool halves, hipStream_t st) {
  p.mtiles = (p.T + 32 * MF - 1) / (32 * MF);
  p.ntiles = (p.N + 64 * NF - 1) / (64 * NF);
  const int total = p.mtiles * p.ntiles;
  p.whole = halves ? total / kCus * kCus : total;
  hipLaunchKernelGGL((prompt_mlp_kernel<MF, NF, D>), dim3(static_cast<unsigned>(2 * total - p.whole)),
                     dim3(kMlpThreads), 0, st, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_prompt_mlp(const PromptMlpParams& p, hipStream_t st) {
  // The block shape of the least estimated time, rounds of one block per CU
  // times a block's time.  At K = 1536 a block of 256 x 256 takes 36 us, of
  // 256 x 128 25, of 128 x 128 (loads three steps ahead, in the registers
  // that its products leave) 18.5: ratios 8, 5.6 and 4.1.  64-token blocks
  // took as long as 128-token ones; 128 x 256 31 us.
  // After a whole round of 256 x 256 blocks a rest of at most half a round
  // goes as 256 x 128 blocks (N 17920: 1000 tokens, 280 tiles, 77 -> 66 us;
  // 4001, 1120 tiles, 212 -> 198).
  auto tiles = [&](int tm, int tn) { return static_cast<int64_t>((p.T + tm - 1) / tm) * ((p.N + tn - 1) / tn); };
  auto rounds = [&](int64_t n) { return (n + kCus - 1) / kCus; };
  const int64_t n84 = tiles(256, 256), rest = n84 % kCus;
  const bool halves = n84 > kCus && rest > 0 && 2 * rest <= kCus;
  const int64_t c84 = halves ? 80 * (n84 / kCus) + 56 : 80 * rounds(n84);
  const int64_t c82 = 56 * rounds(tiles(256, 128)), c42 = 41 * rounds(tiles(128, 128));
  if (c42 <= c82 && c42 <= c84) return launch_shape<4, 2, 3>(p, false, st);
  if (c82 < c84) return launch_shape<8, 2, 1>(p, false, st);
  return launch_shape<8, 4, 1>(p, halves, st);
}

}  // namespace saga
