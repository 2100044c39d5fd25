// Coordinate-MLP passes for networks whose layers fit a tile of rows in LDS
// (at most MLP_PASS_MAX features a layer): the forward and backward sweeps of
// a tile of samples in one workgroup, the weight gradients of all layers in
// one launch, their sums with Adam in a third.
//
// Layouts.  An MFMA operand of 16 rows (or columns) x 32 values of k is a
// fragment: 64 lanes x 8 BF16, lane l holding row l % 16 and k = 8 (l / 16)
// .. + 7, 1 KB in memory.  Weights, activations and gradients are kept in
// memory as fragments, so that every load and store of a wavefront is one
// contiguous KB:
//   WT[l]: fragments [n block][k step] of B(k, n) = W(k, n) (forward);
//   Wb[l]: fragments [k block][n step] of W's transpose (input gradients);
//   H[l], dZ[l]: fragments [32 samples][feature block], k the samples (the
//     operands of the weight gradients);
//   Z[l]: the FP32 accumulator blocks [16 samples][16 features], 64 lanes x 4;
//     a hidden layer's dZ takes its place (dz_block).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mlp_dev.hpp"

namespace glh {
namespace mlp {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ inline uint32_t pack2(float a, float b)
{
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

__device__ inline uint64_t mix64(uint64_t z)
{
  z += 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}

// The tile in LDS: feature f of the 16 MB samples at row f, its 16-sample
// chunks permuted by tile_swizzle(f) so that the transposing reads (4
// consecutive features x 16 samples per 16 lanes) and the writes of 4
// samples per lane both touch every bank equally.
template <int MB>
__device__ inline int tile_swizzle(int f)
{
  return MB == 8   ? (f & 3) | ((f >> 1) & 4)
         : MB == 4 ? ((f >> 1) & 1) | ((f >> 2) & 2)
                   : (f >> 3) & 1;
}
template <int MB>
__device__ inline int tile_at(int f, int chunk)
{
  return f * (MB * 16) + ((chunk ^ tile_swizzle<MB>(f)) * 16);
}

// a fragment of the tile: samples of one chunk, k = 32 consecutive features,
// as two transposing reads of 4 features (the swizzle is the same for both)
template <int MB>
__device__ inline bf16x8 tile_frag(const uint16_t *p)
{
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(p + 4 * MB * 16));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The weight fragments of a wavefront's NB column blocks, PD steps of k in
// flight: start() issues the first ones (before the previous layer's
// epilogue, so their latency is behind it), run() multiplies.
template <int MB, int NB, int PD>
struct Weights {
  bf16x8 b[PD][NB];
  const uint16_t *bp;
  int kst, ksteps;  // steps stored per block, steps used
  __device__ inline void load(int u, int ks)
  {
#pragma unroll
    for (int i = 0; i < NB; ++i)
      b[u][i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(bp + (size_t)(i * kst + ks) * 512));
  }
  __device__ inline void start(const bf16 *W, int w, int lane, int stored, int used)
  {
    kst = stored;
    ksteps = used;
    bp = reinterpret_cast<const uint16_t *>(W) + (size_t)w * NB * stored * 512 + lane * 8;
#pragma unroll
    for (int u = 0; u < PD; ++u)
      if (u < ksteps) load(u, u);
  }
  // acc[i][j] = tile (samples of chunk j) x column block i
  __device__ inline void run(f32x4 (&acc)[NB][MB], const uint16_t *tile, int lane)
  {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < MB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint16_t *ap[MB];
#pragma unroll
    for (int j = 0; j < MB; ++j)
      ap[j] = tile + tile_at<MB>(8 * (lane >> 4) + ((lane & 15) >> 2), j) + (lane & 3) * 4;
    for (int k0 = 0; k0 < ksteps; k0 += PD) {
#pragma unroll
      for (int u = 0; u < PD; ++u) {
        if (k0 + u >= ksteps) break;
#pragma unroll
        for (int j = 0; j < MB; ++j) {
          const bf16x8 a = tile_frag<MB>(ap[j] + (k0 + u) * (32 * MB * 16));
#pragma unroll
          for (int i = 0; i < NB; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[u][i], acc[i][j], 0, 0, 0);
        }
        if (k0 + u + PD < ksteps) load(u, k0 + u + PD);
      }
    }
  }
};

// SiLU(z) = z / (1 + exp(-z)) and sigma(z) = 1 / (1 + exp(-z)): the quotient
// as a product with the hardware reciprocal and one residual correction, 8
// instructions with the sum (sigma 6) where the general division takes 11.
// The reciprocal is that of a quarter of the divisor, so that it is never
// denormal.  SiLU takes the quarter back from the reciprocal, not from the
// quotient: the quotient of a quarter overflows from z = FLT_MAX / 4 on, and
// its residual makes that a NaN.  Over all 2^32 values of z SiLU has the
// division's bits, sigma except where it is denormal (then one unit off in
// 34043 cases).
__device__ inline float silu(float z)
{
  const float e = expf(-z), d = 1.f + e, y = 0.25f * __builtin_amdgcn_rcpf(fmaf(e, 0.25f, 0.25f)), x = z * y;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, x, z), y, x), d, z);
}
__device__ inline float sigma(float z)
{
  const float d = fmaf(expf(-z), 0.25f, 0.25f), y = __builtin_amdgcn_rcpf(d);
  return 0.25f * __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, y, 1.f), y, y), d, 1.f);
}

// Fragment blocks before the 32 samples sb of a hidden layer's dZ, nfb blocks
// each.  They lie in the layer's Z, twice as large, of which a tile has read
// its rows when it writes them: in the first half of its 32 samples' part for
// even sb, the second for odd, so that they meet every memory channel.
__device__ inline size_t dz_block(int sb, int nfb) { return (size_t)(2 * sb + (sb & 1)) * nfb; }

// the tile's nfb feature blocks to memory as fragments of 32 samples (INZ: a
// hidden layer's dZ, at dz_block)
template <int MB, bool INZ = false>
__device__ inline void store_tile(const uint16_t *tile, int nfb, int row0, uint16_t *__restrict__ dst, int w, int lane)
{
  const int g = lane >> 4;
  for (int q = w; q < nfb * (MB / 2); q += 4) {
    const int sb = q / nfb, fb = q - sb * nfb;
    const uint4 v =
        *reinterpret_cast<const uint4 *>(tile + tile_at<MB>(fb * 16 + (lane & 15), 2 * sb + (g >> 1)) + 8 * (g & 1));
    const size_t block = INZ ? dz_block(row0 / 32 + sb, nfb) : (size_t)(row0 / 32 + sb) * nfb;
    // past the caches, which keep Z for the backward sweep
    __builtin_nontemporal_store(__builtin_bit_cast(f32x4, v),
                                reinterpret_cast<f32x4 *>(dst + (block + fb) * 512 + lane * 8));
  }
}

// The forward sweep of a tile of 16 MB samples (GRAD: then the loss, dY and
// the backward sweep).  The tile's activations stay in LDS from layer to
// layer, each overwriting the last, so a layer reads nothing but its weights
// (131 KB at width 256, from L2) and writes only what the gradient needs; a
// wavefront holds 64 NB / 4 columns of all 16 MB rows, so the weights go
// straight to its registers and LDS carries the activations only.  Inference
// is bound by the SiLU's instructions (25 per value, of which exp 13: 63 of
// 109 us at 65536 rows, the vector unit busy 68% of the time and longer by
// its exp and reciprocal, matrix cores 17%; 237 us as one product a layer);
// the gradient by those (vector unit 52%) and the 1.08 GB of Z, H and dZ
// (264 us, 4.1 TB/s, against 445 for the same sweeps as products).
template <int MB, int NB, bool GRAD>
__global__ __launch_bounds__(256, 2) void k_mlp_pass(PassArgs A)
{
  __shared__ __attribute__((aligned(16))) uint16_t tile[MLP_PASS_MAX * MB * 16];
  __shared__ long long src[MB * 16];
  __shared__ float red[4];
  constexpr int W = 64 * NB, MBO = MB >= 4 ? MB / 4 : 1, PD = MB >= 4 ? 2 : 8;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int row0 = blockIdx.x * (MB * 16);
  const int nbo = (A.n_out + 31) / 32 * 2;  // output column blocks, whole k steps of the backward product
  Weights<MB, NB, PD> wt;
  wt.start(A.WT[0], w, lane, 2 * A.F / 32, 2 * A.F / 32);
  // source rows: the batch's own, or drawn from the data by (seed, step, row)
  if (t < MB * 16) {
    const int s = row0 + t;
    long long q = s < A.n_real ? s : -1;
    if (GRAD && A.n_data > 0 && q >= 0) {
      const uint64_t h = mix64(A.seed ^ mix64(((uint64_t)(uint32_t)(A.step[0] + 1) << 32) | (uint32_t)s));
      q = (long long)(h % (uint64_t)A.n_data);
    }
    src[t] = q;
  }
  __syncthreads();
  // Fourier features: a thread keeps one sample and walks the frequencies
  // (one frequency per wavefront when the tile has 64 rows or more)
  {
    const int s = t % (MB * 16);
    const long long q = src[s];
    float x[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) x[d] = q >= 0 ? A.X[(size_t)q * 6 + d] : 0.f;
    for (int j = t / (MB * 16); j < A.F; j += 256 / (MB * 16)) {
      const int ju = MB >= 4 ? __builtin_amdgcn_readfirstlane(j) : j;
      float a = 0.f;
#pragma unroll
      for (int d = 0; d < 6; ++d) a += x[d] * A.Bf[d * A.F + ju];
      const float ang = 6.283185307179586f * a;
      float sn, cs;
      sincosf(ang, &sn, &cs);
      const uint32_t v = pack2(q >= 0 ? sn : 0.f, q >= 0 ? cs : 0.f);
      tile[tile_at<MB>(ju, s >> 4) + (s & 15)] = (uint16_t)v;
      tile[tile_at<MB>(A.F + ju, s >> 4) + (s & 15)] = (uint16_t)(v >> 16);
    }
  }
  __syncthreads();
  if (GRAD) store_tile<MB>(tile, A.F / 8, row0, reinterpret_cast<uint16_t *>(A.H[0]), w, lane);
  f32x4 acc[NB][MB];
  uint2 hp[NB][MB];
  float bias[NB];
  const auto load_bias = [&](int l) {
#pragma unroll
    for (int i = 0; i < NB; ++i) bias[i] = A.P[A.boff[l] + (w * NB + i) * 16 + r];
  };
  // the packed results take the tile's place
  const auto put = [&] {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < MB; ++j)
        *reinterpret_cast<uint2 *>(tile + tile_at<MB>((w * NB + i) * 16 + r, j) + 4 * g) = hp[i][j];
    __syncthreads();
  };
  // accumulator block (i, j) of the wavefront in Z
  const auto zat = [&](int i, int j) {
    return ((size_t)(row0 / 16 + j) * (W / 16) + (w * NB + i)) * 256 + lane * 4;
  };
  for (int l = 0; l < A.depth; ++l) {
    load_bias(l);
    wt.run(acc, tile, lane);
    if (l + 1 < A.depth) wt.start(A.WT[l + 1], w, lane, W / 32, W / 32);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
#pragma unroll
      for (int j = 0; j < MB; ++j) {
        const f32x4 z = acc[i][j] + bias[i];
        if (GRAD) *reinterpret_cast<f32x4 *>(A.Z[l] + zat(i, j)) = z;
        hp[i][j] = uint2{pack2(silu(z[0]), silu(z[1])), pack2(silu(z[2]), silu(z[3]))};
      }
    }
    put();
    if (GRAD) store_tile<MB>(tile, W / 16, row0, reinterpret_cast<uint16_t *>(A.H[l + 1]), w, lane);
  }
  // output layer: wavefront w takes the sample blocks w MBO .. + MBO - 1
  const bool own = w * MBO < MB;
  f32x4 out[4][MBO];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MBO; ++j) out[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (own) {
    const uint16_t *bp = reinterpret_cast<const uint16_t *>(A.WT[A.depth]) + lane * 8;
    const uint16_t *ap[MBO];
#pragma unroll
    for (int j = 0; j < MBO; ++j) ap[j] = tile + tile_at<MB>(8 * g + (r >> 2), w * MBO + j) + (lane & 3) * 4;
    // several steps' weights in flight
    constexpr int OD = W / 32 % 4 ? 2 : 4;
    for (int k0 = 0; k0 < W / 32; k0 += OD) {
      bf16x8 b[OD][4];
#pragma unroll
      for (int u = 0; u < OD; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i < nbo)
            b[u][i] =
                __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(bp + (size_t)(i * (W / 32) + k0 + u) * 512));
#pragma unroll
      for (int u = 0; u < OD; ++u)
#pragma unroll
        for (int j = 0; j < MBO; ++j) {
          const bf16x8 a = tile_frag<MB>(ap[j] + (k0 + u) * (32 * MB * 16));
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (i < nbo) out[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[u][i], out[i][j], 0, 0, 0);
        }
    }
  }
  if (!GRAD) {
    if (own)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = i * 16 + r;
        if (n >= A.n_out) continue;
        const float bias = A.P[A.boff[A.depth] + n];
#pragma unroll
        for (int j = 0; j < MBO; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int s = row0 + (w * MBO + j) * 16 + 4 * g + q;
            if (s < A.n_real) A.Y[(size_t)s * A.n_out + n] = out[i][j][q] + bias;
          }
      }
    return;
  }
  // mean-squared error: dY = bf16(2 (Y - T) / (n_real n_out)), 0 in the
  // padding, and the workgroup's part of the sum of squares
  float e2 = 0.f;
  __syncthreads();
  if (own)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= nbo) continue;
      const int n = i * 16 + r;
      const float bias = n < A.n_out ? A.P[A.boff[A.depth] + n] : 0.f;
#pragma unroll
      for (int j = 0; j < MBO; ++j) {
        float gr[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const long long s = src[(w * MBO + j) * 16 + 4 * g + q];
          gr[q] = 0.f;
          if (s >= 0 && n < A.n_out) {
            const float d = out[i][j][q] + bias - A.T[(size_t)s * A.n_out + n];
            e2 += d * d;
            gr[q] = 2.f * d / ((float)A.n_real * (float)A.n_out);
          }
        }
        *reinterpret_cast<uint2 *>(tile + tile_at<MB>(n, w * MBO + j) + 4 * g) =
            uint2{pack2(gr[0], gr[1]), pack2(gr[2], gr[3])};
      }
    }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) e2 += __shfl_xor(e2, o);
  if (lane == 0) red[w] = e2;
  __syncthreads();
  if (t == 0) A.lpart[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
  store_tile<MB>(tile, nbo, row0, reinterpret_cast<uint16_t *>(A.dZ[A.depth]), w, lane);
  // dZ of layer l - 1 = (dZ_l W_l^T) SiLU'(Z of layer l - 1)
  wt.start(A.Wb[A.depth], w, lane, MLP_OUTP / 32, nbo / 2);
  for (int l = A.depth; l >= 1; --l) {
    // Z of the first column blocks is on its way during the product
    constexpr int ZD = MB >= 8 ? 2 : NB;
    f32x4 z[ZD][MB];
    const auto loadz = [&](int i) {
#pragma unroll
      for (int j = 0; j < MB; ++j) z[i % ZD][j] = *reinterpret_cast<const f32x4 *>(A.Z[l - 1] + zat(i, j));
    };
    if (MB < 8)
#pragma unroll
      for (int i = 0; i < NB; ++i) loadz(i);
    wt.run(acc, tile, lane);
    if (MB >= 8) loadz(0);
    if (l > 1) wt.start(A.Wb[l - 1], w, lane, W / 32, W / 32);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (MB >= 8) {
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < NB) loadz(i + 1);
      }
#pragma unroll
      for (int j = 0; j < MB; ++j) {
        const f32x4 zz = z[i % ZD][j];
        float o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float sg = sigma(zz[q]);
          o[q] = acc[i][j][q] * sg * (1.f + zz[q] * (1.f - sg));
        }
        hp[i][j] = uint2{pack2(o[0], o[1]), pack2(o[2], o[3])};
      }
    }
    put();
    store_tile<MB, true>(tile, W / 16, row0, reinterpret_cast<uint16_t *>(A.dZ[l - 1]), w, lane);
  }
}

// dW_l = H_l^T dZ_l and the column sums of dZ_l over split z's samples, all
// layers in one launch: workgroup = (split, layer, tile of 2 TB x 2 TB
// blocks), wavefront = TB x TB blocks.  Both operands are stored as
// fragments, so a step of 32 samples is 4 TB contiguous KB: R steps ahead in
// registers, one in LDS.  Bound by reading H and dZ (0.36 GB) and writing the
// splits' partials (77 MB) at 65536 rows: 108 us, 4 TB/s, against 240 us for
// the products that transposed their operands in registers.
template <int TB, int R>
__global__ __launch_bounds__(256, TB == 4 ? 2 : 4) void k_mlp_wgrad(WgradArgs A)
{
  __shared__ __attribute__((aligned(16))) uint16_t fr[2][4 * TB][512];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  // splits over the XCDs, the tiles of one split (which share its samples) on one
  int z, q;
  const int tiles = A.tile0[A.n_layers];
  if (A.splits % 8 == 0) {
    const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
    z = x + 8 * (k / tiles);
    q = k % tiles;
  } else {
    z = blockIdx.x / tiles;
    q = blockIdx.x % tiles;
  }
  if (A.step && blockIdx.x == 0 && t == 0) A.step[0] += 1;
  int l = 0;
  while (l + 1 < A.n_layers && q >= A.tile0[l + 1]) ++l;
  q -= A.tile0[l];
  const int nA = A.nA[l], nB = A.nB[l], tB = (nB + 2 * TB - 1) / (2 * TB);
  const int a0 = q / tB * (2 * TB), b0 = q % tB * (2 * TB);
  const int k0 = z * A.per, k1 = k0 + A.per < A.ksteps ? k0 + A.per : A.ksteps;
  const uint16_t *H = reinterpret_cast<const uint16_t *>(A.H[l]);
  const uint16_t *dZ = reinterpret_cast<const uint16_t *>(A.dZ[l]);
  // the wavefront's TB fragments of a step: A's blocks (w = 0, 1) or B's
  const bool isB = w >= 2;
  const int f0 = (isB ? b0 : a0) + (w & 1) * TB, nf = isB ? nB : nA;
  const bool inz = isB && l + 1 < A.n_layers;
  const uint16_t *src = (isB ? dZ : H) + (size_t)f0 * 512 + lane * 8;
  uint4 x[R][TB];
  const auto load = [&](int u, int k) {
#pragma unroll
    for (int i = 0; i < TB; ++i)
      if (f0 + i < nf && k < k1) x[u][i] = *reinterpret_cast<const uint4 *>(src + ((inz ? dz_block(k, nf) : (size_t)k * nf) + i) * 512);
  };
  const auto stage = [&](int u, int b) {
#pragma unroll
    for (int i = 0; i < TB; ++i) *reinterpret_cast<uint4 *>(&fr[b][w * TB + i][lane * 8]) = x[u][i];
  };
  const int wm = w >> 1, wn = w & 1;
  const bool act = a0 + wm * TB < nA && b0 + wn * TB < nB;
  // the column sums of a block: the wavefronts holding it share its columns
  const int rows = (nA + TB - 1) / TB, parts = rows < TB ? rows : TB, part = a0 / TB + wm;
  const bool sums = act && part < parts;
  f32x4 acc[TB][TB];
  float cs[TB][4];  // [block][step mod 4]
#pragma unroll
  for (int i = 0; i < TB; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) cs[i][j] = 0.f;
#pragma unroll
    for (int j = 0; j < TB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const auto step = [&](int b) {
    if (!act) return;
    bf16x8 va[TB], vb[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      va[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(&fr[b][wm * TB + i][lane * 8]));
      vb[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(&fr[b][(2 + wn) * TB + i][lane * 8]));
    }
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int j = 0; j < TB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[i], vb[j], acc[i][j], 0, 0, 0);
    if (sums)
#pragma unroll
      for (int j = 0; j < TB; ++j)
        if (j % parts == part) {
          float v = cs[j][0];
#pragma unroll
          for (int e = 0; e < 8; ++e) v += (float)vb[j][e];
          cs[j][0] = cs[j][1];
          cs[j][1] = cs[j][2];
          cs[j][2] = cs[j][3];
          cs[j][3] = v;
        }
  };
#pragma unroll
  for (int u = 0; u < R; ++u)
#pragma unroll
    for (int i = 0; i < TB; ++i) x[u][i] = uint4{0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < R; ++u) load(u, k0 + u);
  stage(0, 0);
  load(0, k0 + R);
  __syncthreads();
  for (int k = k0; k < k1; k += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      if (k + u >= k1) break;
      step(u & 1);
      stage((u + 1) % R, (u + 1) & 1);
      load((u + 1) % R, k + u + 1 + R);
      __syncthreads();
    }
  }
  if (!act) return;
  float *P = A.part + A.poff[l] + (size_t)z * nA * nB * 256;
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      const int a = a0 + wm * TB + i, b = b0 + wn * TB + j;
      if (a < nA && b < nB) *reinterpret_cast<f32x4 *>(P + ((size_t)a * nB + b) * 256 + lane * 4) = acc[i][j];
    }
  if (!sums) return;
  // lane (column, g) of step k holds rows 32 k + 8 g ..: the 16 row groups
  // 4 (k mod 4) + g in order
  const int turn = (k1 - k0) & 3;
#pragma unroll
  for (int j = 0; j < TB; ++j)
    if (j % parts == part) {
      float s = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int o = (c - turn) & 3;
        const float v = o == 0 ? cs[j][0] : o == 1 ? cs[j][1] : o == 2 ? cs[j][2] : cs[j][3];
#pragma unroll
        for (int g = 0; g < 4; ++g) s += __shfl(v, (lane & 15) + 16 * g);
      }
      const int b = b0 + wn * TB + j;
      if (b < nB && lane < 16) A.cpart[A.coff[l] + (size_t)z * nB * 16 + b * 16 + lane] = s;
    }
}

constexpr int ET = 256;

// offset of B(k, n) in the fragments of a K-deep operand
__device__ inline size_t frag_at(int k, int n, int K)
{
  return ((size_t)(n / 16) * (K / 32) + k / 32) * 512 + (((k % 32) / 8) * 16 + n % 16) * 8 + k % 8;
}

struct Adam {
  float lr, b1, b2, eps, c1, c2;
};
__device__ inline float adam_step(const Adam &C, float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
                                  long long i, float gi)
{
  const float mi = C.b1 * m[i] + (1.f - C.b1) * gi, vi = C.b2 * v[i] + (1.f - C.b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / C.c1, vh = vi / C.c2;
  const float pn = p[i] - C.lr * mh / (sqrtf(vh) + C.eps);
  p[i] = pn;
  return pn;
}

// The splits' partials summed in order, a thread per four consecutive k of a
// weight column (one lane's accumulators) or per bias; then the flat gradient
// G, or (ADAM) the parameter update with the BF16 copies of the new weights.
// The last workgroup sums the loss.
template <bool ADAM>
__global__ __launch_bounds__(ET) void k_mlp_update(UpdateArgs A)
{
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ float sh[ET];
    float s = 0.f;
    for (int i = threadIdx.x; i < A.n_lpart; i += ET) s += A.lpart[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int st = ET / 2; st > 0; st >>= 1) {
      if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) A.loss[0] = sh[0];
    return;
  }
  const int u = blockIdx.x * ET + threadIdx.x;
  if (u >= A.unit0[A.n_layers]) return;
  int l = 0;
  while (l + 1 < A.n_layers && u >= A.unit0[l + 1]) ++l;
  const int q = u - A.unit0[l], nA = A.nA[l], nB = A.nB[l], N = A.N[l];
  Adam C{A.lr, A.b1, A.b2, A.eps, 0.f, 0.f};
  if (ADAM) {
    const int ts = A.step[0];
    C.c1 = 1.f - powf(A.b1, (float)ts);
    C.c2 = 1.f - powf(A.b2, (float)ts);
  }
  if (q >= nA * nB * 64) {
    const int n = q - nA * nB * 64;
    const float *src = A.cpart + A.coff[l] + n;
    float s = 0.f;
    for (int z = 0; z < A.splits; ++z) s += src[(size_t)z * nB * 16];
    const long long i = A.boff[l] + n;
    if (ADAM) adam_step(C, A.P, A.m, A.v, i, s);
    else A.G[i] = s;
    return;
  }
  const float *src = A.part + A.poff[l] + (size_t)q * 4;
  const size_t stride = (size_t)nA * nB * 256;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  int z = 0;
  for (; z + 16 <= A.splits; z += 16) {
    f32x4 v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = *reinterpret_cast<const f32x4 *>(src + (z + e) * stride);
#pragma unroll
    for (int e = 0; e < 16; ++e) s += v[e];
  }
  for (; z < A.splits; ++z) s += *reinterpret_cast<const f32x4 *>(src + z * stride);
  const int lane = q & 63, blk = q >> 6;
  const int n = (blk % nB) * 16 + (lane & 15), k = (blk / nB) * 16 + (lane >> 4) * 4;
  if (n >= N) return;
  const long long i = A.woff[l] + (long long)k * N + n;
  if (!ADAM) {
#pragma unroll
    for (int e = 0; e < 4; ++e) A.G[i + (long long)e * N] = s[e];
    return;
  }
  float p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = adam_step(C, A.P, A.m, A.v, i + (long long)e * N, s[e]);
  const uint2 h = {pack2(p[0], p[1]), pack2(p[2], p[3])};
  *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(A.WT[l]) + frag_at(k, n, nA * 16)) = h;
  uint16_t *wb = reinterpret_cast<uint16_t *>(A.Wb[l]);
  wb[frag_at(n, k, A.Np[l])] = (uint16_t)h.x;
  wb[frag_at(n, k + 1, A.Np[l])] = (uint16_t)(h.x >> 16);
  wb[frag_at(n, k + 2, A.Np[l])] = (uint16_t)h.y;
  wb[frag_at(n, k + 3, A.Np[l])] = (uint16_t)(h.y >> 16);
}

// both fragment copies of a K x N FP32 weight, zeros beyond N
__global__ __launch_bounds__(ET) void k_pack_frag(int K, int N, int Np, const float *__restrict__ W,
                                                  bf16 *__restrict__ Wb, bf16 *__restrict__ WT)
{
  const int i = blockIdx.x * ET + threadIdx.x;
  if (i >= K * Np) return;
  const int k = i / Np, n = i % Np;
  const uint16_t h = (uint16_t)pack2(n < N ? W[(size_t)k * N + n] : 0.f, 0.f);
  reinterpret_cast<uint16_t *>(WT)[frag_at(k, n, K)] = h;
  reinterpret_cast<uint16_t *>(Wb)[frag_at(n, k, Np)] = h;
}

template <int MB, bool GRAD>
void launch_pass(const PassArgs &A, int nb, hipStream_t s)
{
  const dim3 grid((nb + MB * 16 - 1) / (MB * 16));
  if constexpr (MB == 8) {
    hipLaunchKernelGGL((k_mlp_pass<MB, 4, GRAD>), grid, dim3(256), 0, s, A);
  } else {
    switch (A.width / 64) {
      case 1: hipLaunchKernelGGL((k_mlp_pass<MB, 1, GRAD>), grid, dim3(256), 0, s, A); break;
      case 2: hipLaunchKernelGGL((k_mlp_pass<MB, 2, GRAD>), grid, dim3(256), 0, s, A); break;
      case 3: hipLaunchKernelGGL((k_mlp_pass<MB, 3, GRAD>), grid, dim3(256), 0, s, A); break;
      default: hipLaunchKernelGGL((k_mlp_pass<MB, 4, GRAD>), grid, dim3(256), 0, s, A); break;
    }
  }
}

}  // namespace

// Small tiles while they leave more workgroups than CUs (32 rows up to 16384:
// gradient of 14000 rows 75 us against 94 with 64 rows, of 19000 rows 126
// against 118).  128 rows, at width 256, where the training batches lie: two
// workgroups a CU are 65536 rows, and half the reads of the weights shorten
// the gradient from 7/8 of that on.  us with 64 and with 128 rows: gradient
// of 45000 rows 230 / 233, 49152 238 / 243, 57344 262 / 252, 65536 281 / 273;
// past 65536 a second round of 128-row tiles is mostly empty (73728 rows
// 352 / 387, 98304 402 / 420), and inference, which waits for no Z, is a
// little faster with 64 rows at every size (57344 rows 98 / 104, 65536
// 100 / 104).
int pass_rows(int n, int width) { return n >= 57344 && width == 256 ? 128 : n >= 16384 ? 64 : 32; }

hipError_t pass(const PassArgs &A, bool grad, hipStream_t s)
{
  if (A.width < 64 || A.width % 64 || A.width > MLP_PASS_MAX || 2 * A.F % 64 || 2 * A.F > MLP_PASS_MAX ||
      A.depth < 1 || A.depth + 1 > MLP_MAX_LAYERS || A.n_out < 1 || A.n_out > MLP_OUTP || A.n_real < 1)
    return hipErrorInvalidValue;
  // a gradient's rows are whole steps of the weight gradients
  const int nb = grad ? A.n_rows : A.n_real;
  switch (pass_rows(A.n_real, A.width)) {
    case 128: grad ? launch_pass<8, true>(A, nb, s) : launch_pass<8, false>(A, nb, s); break;
    case 64: grad ? launch_pass<4, true>(A, nb, s) : launch_pass<4, false>(A, nb, s); break;
    default: grad ? launch_pass<2, true>(A, nb, s) : launch_pass<2, false>(A, nb, s); break;
  }
  return hipGetLastError();
}

hipError_t wgrad(const WgradArgs &args, hipStream_t s)
{
  WgradArgs A = args;
  if (A.n_layers < 1 || A.n_layers > MLP_MAX_LAYERS || A.splits < 1 || A.per < 1 ||
      (long long)A.splits * A.per < A.ksteps)
    return hipErrorInvalidValue;
  const auto tiles = [&](int tb) {
    int n = 0;
    for (int l = 0; l < A.n_layers; ++l) {
      A.tile0[l] = n;
      n += ((A.nA[l] + 2 * tb - 1) / (2 * tb)) * ((A.nB[l] + 2 * tb - 1) / (2 * tb));
    }
    A.tile0[A.n_layers] = n;
    return (unsigned)(n * A.splits);
  };
  // large tiles read the operands half as often; with fewer than two
  // workgroups per CU a step's latency counts instead (2 splits of 703 steps:
  // 0.80 ms with large tiles two steps ahead, 0.2 ms with small ones)
  unsigned g = tiles(4);
  if (g >= 512) {
    hipLaunchKernelGGL((k_mlp_wgrad<4, 4>), dim3(g), dim3(256), 0, s, A);
  } else {
    g = tiles(2);
    hipLaunchKernelGGL((k_mlp_wgrad<2, 8>), dim3(g), dim3(256), 0, s, A);
  }
  return hipGetLastError();
}

hipError_t update(const UpdateArgs &A, bool adam, hipStream_t s)
{
  if (A.n_layers < 1 || A.n_layers > MLP_MAX_LAYERS) return hipErrorInvalidValue;
  const dim3 grid((A.unit0[A.n_layers] + ET - 1) / ET + 1);
  if (adam) hipLaunchKernelGGL(k_mlp_update<true>, grid, dim3(ET), 0, s, A);
  else hipLaunchKernelGGL(k_mlp_update<false>, grid, dim3(ET), 0, s, A);
  return hipGetLastError();
}

hipError_t pack_frag(int K, int N, int Np, const float *W, bf16 *Wb, bf16 *WT, hipStream_t s)
{
  hipLaunchKernelGGL(k_pack_frag, dim3((K * Np + ET - 1) / ET), dim3(ET), 0, s, K, N, Np, W, Wb, WT);
  return hipGetLastError();
}

}  // namespace mlp
}  // namespace glh
