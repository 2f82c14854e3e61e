// Learned warm start: a 3-D U-Net that predicts lambda0 from the cell-type
// mask, R and the inflow profile, trained on the device.
//
// Network (levels L, base channels c0, c_l = c0 * 2^l):
//   encoder l:  conv3(cin_l -> c_l) ReLU, conv3(c_l -> c_l) ReLU  [skip l]
//               2x2x2 average pool to level l+1            (l < L-1)
//   decoder l:  nearest 2x upsample of level l+1, concat [skip_l, up],
//               conv3(c_l + c_{l+1} -> c_l) ReLU, conv3(c_l -> c_l) ReLU
//   head:       conv1(c_0 -> 1)
// Layout: activations channels-last [voxel][channel] in BF16, voxels x
// fastest.  3x3x3 convolutions are implicit GEMMs on MFMA
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation): rows = voxels, columns =
// output channels, K = 27 taps x input channels.  The data gradient is the
// same kernel with tap-flipped, transposed weights; the weight gradient is an
// MFMA GEMM reducing over voxels, transposed on the matrix cores (split over
// work-groups, FP32 atomics).
// FP32 master weights, Adam.
#include <chrono>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <new>
#include <random>
#include <vector>

#include "qesmc_internal.h"

hipError_t qesmc_launch_divergence(qesmc_ctx *x, int layout, int alpha1);

namespace qesmc {
namespace unet {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;  // storage of one BF16 value

__device__ inline bf16_t f2bf(float f)
{
  const unsigned u = __float_as_uint(f);
  const unsigned even = u + (0x7fffu + ((u >> 16) & 1u));             // round to nearest even
  const unsigned keep = u | ((u & 0xffffu) ? 0x400000u : 0u);  // infinity, and NaN made quiet
  return (bf16_t)(((u & 0x7f800000u) == 0x7f800000u ? keep : even) >> 16);
}
__device__ inline float bf2f(bf16_t h) { return __uint_as_float(((unsigned)h) << 16); }

// Element e of eight BF16 values in a register quad.
__device__ inline float bf_at(const uint4 &t, int e)
{
  const unsigned w = e < 2 ? t.x : e < 4 ? t.y : e < 6 ? t.z : t.w;
  return __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
}

__device__ inline bf16x8 as_bf16x8(uint4 u) { return __builtin_bit_cast(bf16x8, u); }

// ---------------------------------------------------------------------------
// 3x3x3 convolution, forward (also the data gradient)
// ---------------------------------------------------------------------------
struct ConvFwdArgs {
  const bf16_t *x;      // input [V][ldx], channels [0, cin)
  int ldx, cin, ktot;   // ktot = 27 * cin
  int cout;
  const bf16_t *w;      // packed weights (k_pack_w)
  int kp;               // of a row of them (ConvKind::rows)
  const float *bias;    // [cout] or null
  bf16_t *y;            // output [V][ldy]
  int ldy;
  int dx, dy, dz;
  int relu;
};

// Taps and channels in one sequence k = tap*cin + c, 32 at a time, both
// operands gathered from L2: for channel counts that are neither one chunk
// nor a multiple of 32, on volumes of few bricks (ConvKind::rows).
// A wave computes MT tiles of 16 voxels x NT tiles of 16 output channels.
// MFMA operand layout (16x16x32): lane l holds A[l%16][8*(l/16)+0..7],
// B[8*(l/16)+0..7][l%16]; the result D[4*(l/16)+i][l%16].
template <int NT, int MT>
__global__ __launch_bounds__(256) void k_conv_fwd(ConvFwdArgs a)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long V = (long long)a.dx * a.dy * a.dz;
  const long long mbase = ((long long)blockIdx.x * 4 + wave) * (16 * MT);
  if (mbase >= V) return;
  const int r = lane & 15, oct = lane >> 4;
  const int nb = blockIdx.y * NT;  // first output tile of this launch row
  int vx[MT], vy[MT], vz[MT];
  bool vin[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    long long m = mbase + 16 * t + r;
    vin[t] = m < V;
    if (!vin[t]) m = 0;
    vx[t] = (int)(m % a.dx);
    vy[t] = (int)((m / a.dx) % a.dy);
    vz[t] = (int)(m / ((long long)a.dx * a.dy));
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  int tap = 0, c = 8 * oct;
  while (c >= a.cin) {
    c -= a.cin;
    ++tap;
  }
  const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
  for (int kc = 0; kc < a.kp; kc += 32) {
    const int koct = kc + 8 * oct;
    const bool kvalid = koct < a.ktot;
    const int ox = tap % 3 - 1, oy = (tap / 3) % 3 - 1, oz = tap / 9 - 1;
    bf16x8 av[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int nx = vx[t] + ox, ny = vy[t] + oy, nz = vz[t] + oz;
      const bool ok = kvalid && vin[t] && nx >= 0 && nx < a.dx && ny >= 0 && ny < a.dy && nz >= 0 && nz < a.dz;
      const long long nv = ((long long)nz * a.dy + ny) * a.dx + nx;
      av[t] = as_bf16x8(ok ? *reinterpret_cast<const uint4 *>(a.x + nv * a.ldx + c) : zero4);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const bf16x8 bv = as_bf16x8(*reinterpret_cast<const uint4 *>(a.w + (long long)(16 * (nb + n) + r) * a.kp + koct));
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t], bv, acc[t][n], 0, 0, 0);
    }
    c += 32;
    while (c >= a.cin) {
      c -= a.cin;
      ++tap;
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int col = 16 * (nb + n) + r;
      const float b = a.bias ? a.bias[col] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long long m = mbase + 16 * t + 4 * oct + i;
        if (m >= V) continue;
        float v = acc[t][n][i] + b;
        if (a.relu) v = v > 0.f ? v : 0.f;
        as_global(a.y)[m * a.ldy + col] = f2bf(v);
      }
    }
}

// ---------------------------------------------------------------------------
// 3x3x3 convolution, forward, from bricks in LDS
//
// A work-group of four waves owns a brick of 16 x SY x SZ voxels: SY * SZ tiles
// of 16 voxels along x.  It stages the brick and a halo of one voxel (zero
// outside the volume), and every matrix operand is one 16-byte LDS read per
// lane at a fixed offset from the lane's voxel.  The weights are the A operand
// (rows are output channels) and the voxels the B operand, so a lane ends
// with four consecutive channels of one voxel, an 8-byte store, and the
// weights, stored in lane order, come in 1 KB loads.
//
// The order of a voxel's products is part of the result (activations are
// rounded to BF16).  Two orders, by the volume (conv_kind):
//   k_conv_chunks  chunks of CH = 16 channels (8 for the input) outermost, within
//                  them 16-channel taps two by two (8-channel taps four by four)
//   k_conv_whole   taps outermost, within them 32 channels at a time; all
//                  channels are staged
//
// Within a voxel's 16-byte octets the octet index is XORed with bits of x, so
// that the 16 lanes of an LDS phase (16 consecutive x, one octet) hit all
// banks once.
//
// Bound: LDS, one 1 KB read per product (8 cycles of the CU's LDS where the
// product takes 4 of its matrix cores), and the staging before it.  All
// convolutions of a forward pass of 4 levels at 128x128x64 take 366 us, and took 972
// with bricks of 8x8x4 whose reads hit half the banks, weights read by
// output row (64 cache lines a load) and results stored two bytes at a
// time, and, below 1024 of them, both operands gathered from L2 for each
// product.  16 -> 16 channels at 128x128x64: 100 -> 34 us; 48 -> 16: 190 -> 80;
// its gradient, 16 -> 48: 197 -> 84; 192 -> 64 at 32x32x16: 145 -> 30.
// Operands in flight need the order of the code kept (sched_barrier): left to
// itself the compiler reads each just before its product, 46 us instead of 34.
// ---------------------------------------------------------------------------
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

enum class ConvKind { chunks8, chunks16, whole, rows };

constexpr int kBrickX = 16, kHaloX = kBrickX + 2;
constexpr int kXcdsU = 8;  // work-groups are dealt to the XCDs in turn

// The order of products for cin input channels on a volume, and so the kernel
// and the weights' layout.  (One chunk, or one tap group, is the same in either order.)
__host__ __device__ inline ConvKind conv_kind(int cin, int dx, int dy, int dz)
{
  if (cin == 8) return ConvKind::chunks8;
  if (cin == 16) return ConvKind::chunks16;
  const long long bricks = (long long)((dx + 7) / 8) * ((dy + 7) / 8) * ((dz + 3) / 4);
  if (bricks >= 1024) return ConvKind::chunks16;
  return cin % 32 == 0 ? ConvKind::whole : ConvKind::rows;
}

// BF16 values of the packed weights
__host__ __device__ inline long long packed_weights(ConvKind k, int cin, int cout)
{
  switch (k) {
  case ConvKind::chunks8: return (long long)(cout / 16) * 7 * 512;
  case ConvKind::chunks16: return (long long)(cout / 16) * (cin / 16) * 14 * 512;
  case ConvKind::whole: return (long long)(cout / 16) * 27 * (cin / 32) * 512;
  default: return (long long)cout * ((27 * cin + 31) / 32 * 32);
  }
}

// brick b of the XCD-ordered grid: x fastest, then y, then z; false past the end
template <int SY, int SZ>
__device__ __forceinline__ bool brick_origin(const ConvFwdArgs &a, int *x0, int *y0, int *z0)
{
  const unsigned nbx = (unsigned)(a.dx + kBrickX - 1) / kBrickX, nby = (unsigned)(a.dy + SY - 1) / SY,
                 nbz = (unsigned)(a.dz + SZ - 1) / SZ;
  const unsigned per = gridDim.x / kXcdsU, b = blockIdx.x % kXcdsU * per + blockIdx.x / kXcdsU;
  const unsigned row = b / nbx, layer = row / nby;
  if (layer >= nbz) return false;
  *x0 = (int)(b - row * nbx) * kBrickX;
  *y0 = (int)(row - layer * nby) * SY;
  *z0 = (int)layer * SZ;
  return true;
}

__device__ __forceinline__ uint2 pack_out(const f32x4 &acc, const float *b, int relu)
{
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = acc[i] + b[i];
    if (relu) v[i] = v[i] > 0.f ? v[i] : 0.f;
  }
  return make_uint2((unsigned)f2bf(v[0]) | ((unsigned)f2bf(v[1]) << 16),
                    (unsigned)f2bf(v[2]) | ((unsigned)f2bf(v[3]) << 16));
}

// SY = 8, SZ = 4: a wave takes one z and its 8 rows, with the chunk's 14 (7)
// weight fragments in registers and seven voxel operands in flight.  grid.y
// splits the output channels.  WIDE: the brick's planes pass 31 bits of offset.
template <int CH, bool WIDE>
__global__ __launch_bounds__(256, 3) void k_conv_chunks(ConvFwdArgs a)
{
  constexpr int SY = 8, SZ = 4, HY = SY + 2, HZ = SZ + 2, HV = kHaloX * HY * HZ;
  constexpr int OPT = CH / 8;               // octets per voxel
  constexpr int TPM = 4 / OPT;              // taps per product
  constexpr int NG = (27 + TPM - 1) / TPM;  // products per chunk
  constexpr int NE = (HV * OPT + 255) / 256, AHEAD = 7;
  typedef typename std::conditional<WIDE, unsigned long long, unsigned>::type off_t;
  constexpr off_t kNowhere = (off_t)~0ull;
  __shared__ __attribute__((aligned(16))) uint4v lds[NE * 256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, oct = lane >> 4;
  int x0, y0, z0;
  if (!brick_origin<SY, SZ>(a, &x0, &y0, &z0)) return;
  const uint4v zero4 = {0u, 0u, 0u, 0u};
  auto slot = [](int voxel, int x, int h) { return OPT == 1 ? voxel : 2 * voxel + (h ^ ((x >> 3) & 1)); };
  // the octets this thread stages: offset from the halo's first voxel (nowhere: 0)
  const char *base = reinterpret_cast<const char *>(a.x) +
                     ((((long long)z0 - 1) * a.dy + y0 - 1) * a.dx + x0 - 1) * a.ldx * 2;
  off_t off[NE];
  int put[NE];
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int e = q * 256 + (int)threadIdx.x, hv = e / OPT, h = e % OPT;
    const int x = hv % kHaloX, row = hv / kHaloX, y = row % HY, z = row / HY;
    const int gx = x0 + x - 1, gy = y0 + y - 1, gz = z0 + z - 1;
    const bool in = e < HV * OPT && gx >= 0 && gx < a.dx && gy >= 0 && gy < a.dy && gz >= 0 && gz < a.dz;
    off[q] = in ? (((off_t)z * (off_t)a.dy + (off_t)y) * (off_t)a.dx + (off_t)x) * (off_t)(2 * a.ldx) + (off_t)(16 * h)
                : kNowhere;
    put[q] = slot(hv, x, h);
  }
  // this lane's octet of each product, for the wave's first row
  unsigned at[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int tap = g * TPM + oct / OPT < 27 ? g * TPM + oct / OPT : 0;  // (the 28th has zero weights)
    const int x = r + tap % 3;
    at[g] = (unsigned)slot(((wave + tap / 9) * HY + tap / 3 % 3) * kHaloX + x, x, oct % OPT);
  }
  const bool live27 = oct / OPT + (NG - 1) * TPM < 27;
  const int nchunk = a.cin / CH, nper = a.cin == CH ? a.cout / 16 / (int)gridDim.y : 1;
#pragma unroll 1
  for (int nn = 0; nn < nper; ++nn) {
    const int n = (int)blockIdx.y * nper + nn;
    f32x4 acc[SY];
#pragma unroll
    for (int t = 0; t < SY; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c = 0; c < nchunk; ++c) {
      if (nn == 0) {
        uint4v v[NE];
        const char *from = base + 2 * CH * c;
        if constexpr (WIDE) {
#pragma unroll
          for (int q = 0; q < NE; ++q)
            v[q] = off[q] == kNowhere ? zero4 : *reinterpret_cast<const uint4v *>(from + off[q]);
        } else {
          const __amdgpu_buffer_rsrc_t rs =
              __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(from), 0, 0x7fffffff, 0x00027000);
#pragma unroll
          for (int q = 0; q < NE; ++q) v[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, off[q], 0, 0);
        }
        if (c > 0) __syncthreads();  // the previous chunk's readers are done
#pragma unroll
        for (int q = 0; q < NE; ++q) lds[put[q]] = v[q];
      }
      const bf16_t *wl = a.w + ((long long)n * nchunk + c) * (NG * 512) + lane * 8;
      bf16x8 W[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) W[g] = *reinterpret_cast<const bf16x8 *>(wl + g * 512);
      if (nn == 0) __syncthreads();
      uint4v f[AHEAD];
#pragma unroll
      for (int q = 0; q < AHEAD; ++q) f[q] = lds[at[q % NG] + (unsigned)(q / NG * kHaloX * OPT)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < SY; ++t)
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          const int q = t * NG + g, next = q + AHEAD;
          uint4v o = f[q % AHEAD];
          if (g == NG - 1) o = live27 ? o : zero4;
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[g], __builtin_bit_cast(bf16x8, o), acc[t], 0, 0, 0);
          if (next < SY * NG) f[q % AHEAD] = lds[at[next % NG] + (unsigned)(next / NG * kHaloX * OPT)];
          __builtin_amdgcn_sched_barrier(0);  // or every read would move down to its use
        }
    }
    // lane holds channels 16 n + 4 oct + 0..3 of voxel x0 + r
    const int col = 16 * n + 4 * oct, gx = x0 + r, gz = z0 + wave;
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.bias) {
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = a.bias[col + i];
    }
    if (gx < a.dx && gz < a.dz) {
#pragma unroll
      for (int t = 0; t < SY; ++t)
        if (y0 + t < a.dy)
          *reinterpret_cast<uint2 *>(a.y + (((long long)gz * a.dy + y0 + t) * a.dx + gx) * a.ldy + col) =
              pack_out(acc[t], b, a.relu);
    }
  }
}

// The waves split into WN over the output channels and 4 / WN over the tiles,
// MT tiles each; grid.y takes further channels.  Weights are read nine products
// ahead; LDS holds the whole brick, cin channels a voxel.
template <int SY, int SZ, int WN>
__global__ __launch_bounds__(256, 2) void k_conv_whole(ConvFwdArgs a)
{
  constexpr int HY = SY + 2, HZ = SZ + 2, HV = kHaloX * HY * HZ, WM = 4 / WN, MT = SY * SZ / WM;
  static_assert(SY * SZ % WM == 0, "");
  constexpr int PF = 9;  // divides the 27 cin / 32 products
  extern __shared__ __attribute__((aligned(16))) uint4 whole_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, oct = lane >> 4;
  int x0, y0, z0;
  if (!brick_origin<SY, SZ>(a, &x0, &y0, &z0)) return;
  const int m = a.cin / 32, so = a.cin / 8;  // products per tap, octets per voxel
  // octets move within groups of `grp`, the power of two in so up to 16
  const int grp = (so & -so) < 16 ? (so & -so) : 16, sh = grp == 4 ? 2 : grp == 8 ? 1 : 0;
  auto swizzle = [&](int s, int x) { return (s & ~(grp - 1)) | ((s ^ (x >> sh)) & (grp - 1)); };
  const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
  const int n = (int)blockIdx.y * WN + wave % WN, mw = wave / WN;
  const bf16_t *wl = a.w + (long long)n * (27 * m) * 512 + lane * 8;
  bf16x8 W[PF];
#pragma unroll
  for (int u = 0; u < PF; ++u) W[u] = *reinterpret_cast<const bf16x8 *>(wl + u * 512);
  for (int e0 = 0; e0 < HV * so; e0 += 256 * 4) {
    uint4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = e0 + q * 256 + (int)threadIdx.x, hv = (int)((unsigned)e / (unsigned)so), s = e - hv * so;
      const int x = hv % kHaloX, row = hv / kHaloX, y = row % HY, z = row / HY;
      const int gx = x0 + x - 1, gy = y0 + y - 1, gz = z0 + z - 1;
      v[q] = zero4;
      if (hv < HV && gx >= 0 && gx < a.dx && gy >= 0 && gy < a.dy && gz >= 0 && gz < a.dz)
        v[q] = *reinterpret_cast<const uint4 *>(a.x + (((long long)gz * a.dy + gy) * a.dx + gx) * a.ldx + 8 * s);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = e0 + q * 256 + (int)threadIdx.x, hv = (int)((unsigned)e / (unsigned)so), s = e - hv * so;
      if (hv < HV) whole_lds[hv * so + swizzle(s, hv % kHaloX)] = v[q];
    }
  }
  __syncthreads();
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int tile[MT];  // the tiles' first halo row (uniform)
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int q = mw * MT + t;
    tile[t] = (q / SY * HY + q % SY) * kHaloX * so;
  }
  const int steps = 27 * m;
  // the next product's 32 channels, x shift, and rows (z, y) passed
  int c = 0, ox = 0, rows = 0, oy = 0;
  uint4 f[2][MT];
  auto read = [&](uint4 *v) {
    const int x = r + ox;
    const int at = (rows * kHaloX + x) * so + swizzle(4 * c + oct, x);
#pragma unroll
    for (int t = 0; t < MT; ++t) v[t] = whole_lds[at + tile[t]];
    if (++c == m) {
      c = 0;
      if (++ox == 3) {
        ox = 0;
        ++rows;
        if (++oy == 3) {
          oy = 0;
          rows += HY - 3;
        }
      }
    }
  };
  read(f[0]);
  // by twos, so that the operands in flight keep their registers
  for (int base = 0; base < steps; base += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      if (base + u + 1 < steps) read(f[(u + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);  // or the reads would move down to their use
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[u], as_bf16x8(f[u & 1][t]), acc[t], 0, 0, 0);
      const int next = base + u + PF < steps ? base + u + PF : steps - 1;
      W[u] = *reinterpret_cast<const bf16x8 *>(wl + (long long)next * 512);
    }
    // PF is odd: the operand read last is where the next round looks for it
#pragma unroll
    for (int t = 0; t < MT; ++t) f[0][t] = f[PF & 1][t];
  }
  const int col = 16 * n + 4 * oct, gx = x0 + r;
  float b[4] = {0.f, 0.f, 0.f, 0.f};
  if (a.bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = a.bias[col + i];
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int q = mw * MT + t, gy = y0 + q % SY, gz = z0 + q / SY;
    if (gx < a.dx && gy < a.dy && gz < a.dz)
      *reinterpret_cast<uint2 *>(a.y + (((long long)gz * a.dy + gy) * a.dx + gx) * a.ldy + col) = pack_out(acc[t], b, a.relu);
  }
}

// ---------------------------------------------------------------------------
// 3x3x3 convolution, weight gradient: dW[n][tap][c] += sum_v g[v][n] * X[v+off(tap)][c]
//
// An MFMA GEMM that reduces over voxels, so each lane needs several voxels of
// one channel, while memory holds several channels of one voxel.  The 16 x 16
// tiles are transposed on the matrix cores: a product with the identity
// leaves D[voxel 4*(l/16)+i][channel l%16] in lane l, exactly (the other
// terms are zeros), whose upper halves are the operand.
//
// A wave owns 16 input by 16 output channels (27 accumulator tiles) and a
// strip: 32 voxels along x, one z, a range of y.  Per row of X it transposes
// the row at the three x shifts and the three new rows of g (z-1, z, z+1 of
// row y+1; rows y-1 and y are kept), then runs 27 products of K = 32
// voxels.  The next row's loads are in flight meanwhile.  The four waves of a
// work-group take strips of one channel pair and add up in LDS, so that there
// is one atomic per work-group and weight.
//
// Per row 27 products and 12 transposes against 12 loads of 512 bytes: at
// 128x128x64 with 48 -> 16 channels 2110 us before (a lane gathered its voxels
// with eight 2-byte loads per operand, and one atomic per wave and weight),
// 99 us now.
// ---------------------------------------------------------------------------
struct ConvWgradArgs {
  const bf16_t *x;      // [V][ldx], channels [0, cin); ldx a multiple of 8
  int ldx, cin, ktot;
  const bf16_t *g;      // gradient w.r.t. the pre-activation output [V][ldg]; ldg a multiple of 8
  int ldg;
  float *dw;            // [cout][ktot]
  int dx, dy, dz;
  int ctiles;           // 16-channel tiles of the input
  int ylen;             // rows of X per strip
};

typedef short short4v __attribute__((ext_vector_type(4)));

// The transpose of a 16 x 16 tile: lane l gives voxel l%16, channels 4*(l/16)..+3
// (raw), and gets voxels 4*(l/16)..+3 of channel l%16.
__device__ __forceinline__ uint2 transpose16(uint2 raw, short4v ident)
{
  const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4v, raw), ident,
                                                            f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  uint2 r;
  r.x = __builtin_amdgcn_perm(__float_as_uint(d[1]), __float_as_uint(d[0]), 0x07060302u);
  r.y = __builtin_amdgcn_perm(__float_as_uint(d[3]), __float_as_uint(d[2]), 0x07060302u);
  return r;
}

// One channel's operand: voxels x..x+3 and x+16..x+19 of a row of dx, moved
// by `shift`; 0 outside it or without `in`.
__device__ __forceinline__ bf16x8 gather16(const bf16_t *v, int ld, bool in, long long row, int x, int shift, int dx)
{
  unsigned w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int at = x + 16 * (e >> 2) + (e & 3), from = at + shift;
    const unsigned h = in && at < dx && from >= 0 && from < dx ? v[(row + from) * ld] : 0u;
    w[e >> 1] |= h << (16 * (e & 1));
  }
  return as_bf16x8(make_uint4(w[0], w[1], w[2], w[3]));
}

__global__ __launch_bounds__(256, 2) void k_conv_wgrad(ConvWgradArgs a)
{
  __shared__ float sum[27 * 256];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, oct = lane >> 4;
  const int c0 = 16 * ((int)blockIdx.y % a.ctiles), n0 = 16 * ((int)blockIdx.y / a.ctiles);
  const int nxt = (a.dx + 31) / 32, nys = (a.dy + a.ylen - 1) / a.ylen;
  const int strips = nxt * nys * a.dz;
  const int cch = c0 + 4 * oct;          // this lane's four input channels
  const bool cin_ok = cch < a.cin;       // cin is 8 or a multiple of 16
  short4v ident;
#pragma unroll
  for (int i = 0; i < 4; ++i) ident[i] = 4 * oct + i == r ? (short)0x3f80 : (short)0;
  f32x4 acc[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint2 zero2 = make_uint2(0u, 0u);

  for (int strip = (int)blockIdx.x * 4 + wave; strip < strips; strip += (int)gridDim.x * 4) {
    const int xt = strip % nxt, ys = strip / nxt % nys, z = strip / (nxt * nys);
    const int x0 = 32 * xt, y0 = ys * a.ylen, y1 = y0 + a.ylen < a.dy ? y0 + a.ylen : a.dy;
    // a row's 2 x 16 voxels of X at the three shifts / of g; 0 outside the volume
    auto load_x = [&](int y, uint2 (*v)[2]) {
      const bf16_t *row = a.x + ((long long)z * a.dy + y) * a.dx * a.ldx + cch;
#pragma unroll
      for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int x = x0 + 16 * h + r + s - 1;
          v[s][h] = y < y1 && cin_ok && x >= 0 && x < a.dx ? *reinterpret_cast<const uint2 *>(row + (long long)x * a.ldx)
                                                           : zero2;
        }
    };
    auto load_g = [&](int y, uint2 (*v)[2]) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int zz = z + q - 1;
        const bool in = y >= 0 && y < a.dy && zz >= 0 && zz < a.dz;
        const bf16_t *row = a.g + ((long long)zz * a.dy + y) * a.dx * a.ldg + n0 + 4 * oct;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int x = x0 + 16 * h + r;
          v[q][h] = in && x < a.dx ? *reinterpret_cast<const uint2 *>(row + (long long)x * a.ldg) : zero2;
        }
      }
    };
    auto operand = [&](const uint2 *v) {
      const uint2 lo = transpose16(v[0], ident), hi = transpose16(v[1], ident);
      return as_bf16x8(make_uint4(lo.x, lo.y, hi.x, hi.y));
    };
    bf16x8 G[3][3];  // g rows y-1, y, y+1 (first index), z-1, z, z+1
    uint2 rx[3][2], rg[3][2];
    load_g(y0 - 1, rg);
#pragma unroll
    for (int q = 0; q < 3; ++q) G[1][q] = operand(rg[q]);
    load_g(y0, rg);
#pragma unroll
    for (int q = 0; q < 3; ++q) G[2][q] = operand(rg[q]);
    load_g(y0 + 1, rg);
    load_x(y0, rx);
    for (int y = y0; y < y1; ++y) {
      bf16x8 X[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        G[0][q] = G[1][q];
        G[1][q] = G[2][q];
        G[2][q] = operand(rg[q]);
        X[q] = operand(rx[q]);
      }
      load_g(y + 2, rg);
      load_x(y + 1, rx);
      // X row (y, z) meets g row (y - oy, z - oz) at tap (ox, oy, oz)
#pragma unroll
      for (int oz = -1; oz <= 1; ++oz)
#pragma unroll
        for (int oy = -1; oy <= 1; ++oy)
#pragma unroll
          for (int ox = -1; ox <= 1; ++ox) {
            const int t = (oz + 1) * 9 + (oy + 1) * 3 + ox + 1;
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(G[1 - oy][1 - oz], X[ox + 1], acc[t], 0, 0, 0);
          }
    }
  }
  // An infinity or a NaN makes the identity product's other terms NaN: it would
  // reach all 16 channels of its tile.  Any in a strip has left a NaN in the
  // wave's sums; the wave then takes its strips again with operands gathered a
  // channel at a time (the same voxels in the same order), and with the products that
  // a gradient at the border has with the zeros beyond it, which are then NaN.
  // probe: 0, or NaN where any sum is not finite.
  float probe = 0.f;
#pragma unroll
  for (int t = 0; t < 27; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) probe += 0.f * acc[t][i];
  if (__builtin_amdgcn_ballot_w64(!(probe == 0.f)) != 0) {
    // three taps at a time, so that little is held besides the sums
#pragma unroll
    for (int oz = -1; oz <= 1; ++oz)
#pragma unroll
      for (int oy = -1; oy <= 1; ++oy) {
        f32x4 *const three = acc + (oz + 1) * 9 + (oy + 1) * 3;
        three[0] = three[1] = three[2] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int strip = (int)blockIdx.x * 4 + wave; strip < strips; strip += (int)gridDim.x * 4) {
          const int xt = strip % nxt, ys = strip / nxt % nys, z = strip / (nxt * nys);
          const int x0 = 32 * xt, y0 = ys * a.ylen, y1 = y0 + a.ylen < a.dy ? y0 + a.ylen : a.dy;
          // the strip's rows of X, and the rows of zeros beside them where it lies at the border
          const int za = z == 0 ? -1 : z, zb = z == a.dz - 1 ? a.dz : z;
          const int ya = y0 == 0 ? -1 : y0, yb = y1 == a.dy ? a.dy : y1 - 1;
#pragma unroll 1
          for (int row = 0; row < (zb - za + 1) * (yb - ya + 1); ++row) {
            const int zz = za + row / (yb - ya + 1), yy = ya + row % (yb - ya + 1);
            const int gz = zz - oz, gy = yy - oy;
            if (gz < 0 || gz >= a.dz || gy < 0 || gy >= a.dy) continue;
            const bool in = zz >= 0 && zz < a.dz && yy >= 0 && yy < a.dy && c0 + r < a.cin;
            const bf16x8 G = gather16(a.g + n0 + r, a.ldg, true, ((long long)gz * a.dy + gy) * a.dx, x0 + 4 * oct, 0, a.dx);
#pragma unroll
            for (int ox = -1; ox <= 1; ++ox) {
              const bf16x8 X = gather16(a.x + c0 + r, a.ldx, in, ((long long)zz * a.dy + yy) * a.dx, x0 + 4 * oct, ox, a.dx);
              three[ox + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(G, X, three[ox + 1], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
      }
  }
  // lane holds D[n0 + 4*oct + i][c0 + r] of every tap
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int t = 0; t < 27; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float *p = sum + t * 256 + (4 * oct + i) * 16 + r;
          *p = w == 0 ? acc[t][i] : *p + acc[t][i];
        }
    }
    __syncthreads();
  }
  const int c = c0 + (threadIdx.x & 15);
  if (c < a.cin)
    for (int t = 0; t < 27; ++t)
      atomicAdd(a.dw + (long long)(n0 + (threadIdx.x >> 4)) * a.ktot + t * a.cin + c, sum[t * 256 + threadIdx.x]);
}

// Backward of bias and ReLU, in place: g <- g where y > 0, else 0, and
// db[c] += sum of it.  With gpool (the gradient of the 2x2x2 average pool's
// output, [V/8][ch]) g first takes its eighth.  Eight channels (16 bytes) per
// thread, so one pass over g and y: at 128x128x64 with 16 channels 47 us (27
// without gpool), against 59 + 43 + 69 (30 + 63) in kernels of one element a
// thread.
__global__ __launch_bounds__(256) void k_relu_bias_bwd(bf16_t *g, int ldg, const bf16_t *y, int ldy, int ch,
                                                       long long V, const bf16_t *gpool, int dx, int dy, float *db)
{
  const int groups = ch >> 3, per = 256 / groups;  // ch is 16, 32, 64 or 128
  const int c8 = 8 * ((int)threadIdx.x % groups);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (long long v = (long long)blockIdx.x * per + threadIdx.x / groups; v < V; v += (long long)gridDim.x * per) {
    uint4 t = *reinterpret_cast<const uint4 *>(g + v * ldg + c8);
    const uint4 m = *reinterpret_cast<const uint4 *>(y + v * ldy + c8);
    uint4 pl = make_uint4(0u, 0u, 0u, 0u);
    if (gpool) {
      const unsigned vv = (unsigned)v;
      const unsigned x = vv % (unsigned)dx, yy = vv / (unsigned)dx % (unsigned)dy, z = vv / ((unsigned)dx * (unsigned)dy);
      const unsigned vp = ((z >> 1) * ((unsigned)dy >> 1) + (yy >> 1)) * ((unsigned)dx >> 1) + (x >> 1);
      pl = *reinterpret_cast<const uint4 *>(gpool + (size_t)vp * ch + c8);
    }
    unsigned o[4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float f = bf_at(t, e);
      if (gpool) f = bf2f(f2bf(f + 0.125f * bf_at(pl, e)));
      f = bf_at(m, e) > 0.f ? f : 0.f;
      s[e] += f;
      const unsigned h = __float_as_uint(f) >> 16;  // f is a BF16 value
      o[e >> 1] = (e & 1) ? o[e >> 1] | (h << 16) : h;
    }
    *reinterpret_cast<uint4 *>(g + v * ldg + c8) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  __shared__ float red[256 * 9];
#pragma unroll
  for (int e = 0; e < 8; ++e) red[threadIdx.x * 9 + e] = s[e];
  __syncthreads();
  if ((int)threadIdx.x < ch) {
    float t = 0.f;
    for (int q = 0; q < per; ++q) t += red[(q * groups + (int)threadIdx.x / 8) * 9 + (threadIdx.x & 7)];
    atomicAdd(db + threadIdx.x, t);
  }
}

// 2x2x2 average pool: out[V/8][ldo] <- in[V][ldi] (channels [ioff, ioff+ch))
__global__ __launch_bounds__(256) void k_pool_fwd(const bf16_t *in, int ldi, int ioff, bf16_t *out, int ldo, int ch,
                                                  int odx, int ody, int odz)
{
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long Vo = (long long)odx * ody * odz;
  if (q >= Vo * ch) return;
  const long long vo = q / ch;
  const int c = (int)(q - vo * ch);
  const int x = (int)(vo % odx), y = (int)((vo / odx) % ody), z = (int)(vo / ((long long)odx * ody));
  const int idx = 2 * odx, idy = 2 * ody;
  float s = 0.f;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const long long vi = ((long long)(2 * z + (b >> 2)) * idy + (2 * y + ((b >> 1) & 1))) * idx + 2 * x + (b & 1);
    s += bf2f(in[vi * ldi + ioff + c]);
  }
  out[vo * ldo + c] = f2bf(s * 0.125f);
}

// nearest 2x upsample: out[V][ldo] (channels [ooff, ooff+ch)) <- in[V/8][ldi]
__global__ __launch_bounds__(256) void k_up_fwd(const bf16_t *in, int ldi, bf16_t *out, int ldo, int ooff, int ch,
                                                int dx, int dy, int dz)
{
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long V = (long long)dx * dy * dz;
  if (q >= V * ch) return;
  const long long v = q / ch;
  const int c = (int)(q - v * ch);
  const int x = (int)(v % dx), y = (int)((v / dx) % dy), z = (int)(v / ((long long)dx * dy));
  const long long vp = ((long long)(z >> 1) * (dy >> 1) + (y >> 1)) * (dx >> 1) + (x >> 1);
  out[v * ldo + ooff + c] = in[vp * ldi + c];
}

// gin[parent] = sum of gout over its 8 children, eight channels per thread
__global__ __launch_bounds__(256) void k_up_bwd(const bf16_t *gout, int ldo, int ooff, bf16_t *gin, int ldi, int ch,
                                                int pdx, int pdy, int pdz)
{
  const unsigned g = (unsigned)ch >> 3;
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long Vp = (long long)pdx * pdy * pdz;
  if (q >= Vp * g) return;
  const long long vp = q / g;
  const int c8 = 8 * (int)(q - vp * g);
  const int x = (int)(vp % pdx), y = (int)((vp / pdx) % pdy), z = (int)(vp / ((long long)pdx * pdy));
  const int dx = 2 * pdx, dy = 2 * pdy;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const long long v = ((long long)(2 * z + (b >> 2)) * dy + (2 * y + ((b >> 1) & 1))) * dx + 2 * x + (b & 1);
    const uint4 t = *reinterpret_cast<const uint4 *>(gout + v * ldo + ooff + c8);
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] += bf_at(t, e);
  }
  unsigned o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (unsigned)f2bf(s[2 * e]) | ((unsigned)f2bf(s[2 * e + 1]) << 16);
  *reinterpret_cast<uint4 *>(gin + vp * ldi + c8) = make_uint4(o[0], o[1], o[2], o[3]);
}

// The forward data-movement steps with 8 channels (16 bytes) per thread
// and 32-bit index math, for channel counts, strides and offsets that are
// multiples of 8 and V * ch / 8 < 2^32 (the host checks): same arithmetic in
// the same order per channel, so the same results.
__global__ __launch_bounds__(256) void k_pool_fwd8(const bf16_t *in, int ldi, int ioff, bf16_t *out, int ldo, int ch,
                                                   int odx, int ody, int odz)
{
  const unsigned g = (unsigned)ch >> 3;
  const unsigned q = blockIdx.x * 256u + threadIdx.x;
  if (q >= (unsigned)odx * ody * odz * g) return;
  const unsigned vo = q / g;
  const unsigned c8 = (q - vo * g) * 8u;
  const unsigned x = vo % odx, y = (vo / odx) % ody, z = vo / ((unsigned)odx * ody);
  const unsigned idx = 2u * odx, idy = 2u * ody;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const unsigned vi = ((2u * z + (b >> 2)) * idy + (2u * y + ((b >> 1) & 1))) * idx + 2u * x + (b & 1);
    const uint4 t = *reinterpret_cast<const uint4 *>(in + (size_t)vi * ldi + ioff + c8);
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] += bf_at(t, e);
  }
  unsigned o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = (unsigned)f2bf(s[2 * e] * 0.125f) | ((unsigned)f2bf(s[2 * e + 1] * 0.125f) << 16);
  *reinterpret_cast<uint4 *>(out + (size_t)vo * ldo + c8) = make_uint4(o[0], o[1], o[2], o[3]);
}

__global__ __launch_bounds__(256) void k_up_fwd8(const bf16_t *in, int ldi, bf16_t *out, int ldo, int ooff, int ch,
                                                 int dx, int dy, int dz)
{
  const unsigned g = (unsigned)ch >> 3;
  const unsigned q = blockIdx.x * 256u + threadIdx.x;
  if (q >= (unsigned)dx * dy * dz * g) return;
  const unsigned v = q / g;
  const unsigned c8 = (q - v * g) * 8u;
  const unsigned x = v % dx, y = (v / dx) % dy, z = v / ((unsigned)dx * dy);
  const unsigned vp = ((z >> 1) * ((unsigned)dy >> 1) + (y >> 1)) * ((unsigned)dx >> 1) + (x >> 1);
  *reinterpret_cast<uint4 *>(out + (size_t)v * ldo + ooff + c8) =
      *reinterpret_cast<const uint4 *>(in + (size_t)vp * ldi + c8);
}

__global__ __launch_bounds__(256) void k_head_fwd8(const bf16_t *x, int ldx, int ch, const float *w, float *y,
                                                   long long V)
{
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  if (v >= V) return;
  float s = w[ch];
  for (int c8 = 0; c8 < ch; c8 += 8) {
    const uint4 t = *reinterpret_cast<const uint4 *>(x + v * ldx + c8);
#pragma unroll
    for (int e = 0; e < 8; ++e) s += w[c8 + e] * bf_at(t, e);
  }
  y[v] = s;
}

// head: y[v] = sum_c W[c] x[v][c] + b
__global__ __launch_bounds__(256) void k_head_fwd(const bf16_t *x, int ldx, int ch, const float *w, float *y,
                                                  long long V)
{
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  if (v >= V) return;
  float s = w[ch];
  for (int c = 0; c < ch; ++c) s += w[c] * bf2f(x[v * ldx + c]);
  y[v] = s;
}

// head backward: gx[v][c] = gy[v] W[c]; dW[c] += sum gy x; db += sum gy.
// Eight channels per thread, a work-group sums many voxels before its one
// atomic per weight (878 us at 128x128x64 with a tree reduction in LDS per
// channel and 256 voxels, 25 us now).
__global__ __launch_bounds__(256) void k_head_bwd(const bf16_t *x, int ldx, int ch, const float *w, const float *gy,
                                                  bf16_t *gx, float *dw, long long V)
{
  const int groups = ch >> 3, per = 256 / groups;
  const int c8 = 8 * ((int)threadIdx.x % groups);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, sg = 0.f, wr[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) wr[e] = w[c8 + e];
  for (long long v = (long long)blockIdx.x * per + threadIdx.x / groups; v < V; v += (long long)gridDim.x * per) {
    const float g = gy[v];
    const uint4 t = *reinterpret_cast<const uint4 *>(x + v * ldx + c8);
    unsigned o[4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e] += g * bf_at(t, e);
      const unsigned h = f2bf(g * wr[e]);
      o[e >> 1] = (e & 1) ? o[e >> 1] | (h << 16) : h;
    }
    sg += g;
    *reinterpret_cast<uint4 *>(gx + v * ldx + c8) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  __shared__ float red[256 * 9];
#pragma unroll
  for (int e = 0; e < 8; ++e) red[threadIdx.x * 9 + e] = s[e];
  red[threadIdx.x * 9 + 8] = sg;
  __syncthreads();
  if ((int)threadIdx.x <= ch) {
    // thread ch sums the gradient itself, from the first channel group
    const int grp = (int)threadIdx.x < ch ? (int)threadIdx.x / 8 : 0, e = (int)threadIdx.x < ch ? (int)threadIdx.x & 7 : 8;
    float t = 0.f;
    for (int q = 0; q < per; ++q) t += red[(q * groups + grp) * 9 + e];
    atomicAdd(dw + threadIdx.x, t);
  }
}

// MSE loss over the volume: gy = 2 (y - t) / V, loss += (y - t)^2 / V
__global__ __launch_bounds__(256) void k_mse(const float *y, const float *t, float inv_scale, float *gy, long long V,
                                             float *loss)
{
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  float e = 0.f;
  if (v < V) {
    const float d = y[v] - t[v] * inv_scale;
    gy[v] = 2.f * d / (float)V;
    e = d * d / (float)V;
  }
  __shared__ float red[256];
  red[threadIdx.x] = e;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Block-mean loss term.  The error e = y - t (k_mse leaves gy = 2 e / V) is
// averaged over blocks of S^3 voxels; loss += weight * mean_b(ebar_b^2) and
// gy += weight * 2 ebar_b / (NB * S^3) for every voxel of block b.  Smooth
// errors (which SOR removes slowest) are penalised by (1 + weight), errors
// that change sign within a block by about 1.  One work-group per block.
__global__ __launch_bounds__(256) void k_block_err(const float *gy, float half_v, int dx, int dy, int S,
                                                   float w_over_nb, float *eblk, float *loss)
{
  const int nbx = dx / S, nby = dy / S;
  const int b = blockIdx.x;
  const int bx = b % nbx, by = (b / nbx) % nby, bz = b / (nbx * nby);
  const int n = S * S * S;
  float acc = 0.f;
  for (int q = threadIdx.x; q < n; q += 256) {
    const int x = q % S, y = (q / S) % S, z = q / (S * S);
    const long long v = ((long long)(bz * S + z) * dy + (by * S + y)) * dx + (bx * S + x);
    acc += gy[v] * half_v;
  }
  __shared__ float red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float m = red[0] / (float)n;
    eblk[b] = m;
    if (loss) atomicAdd(loss, w_over_nb * m * m);
  }
}

__global__ __launch_bounds__(256) void k_block_grad(float *gy, const float *eblk, int dx, int dy, int dz, int S,
                                                    float coef)
{
  const long long V = (long long)dx * dy * dz;
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  if (v >= V) return;
  const int x = (int)(v % dx), y = (int)((v / dx) % dy), z = (int)(v / ((long long)dx * dy));
  const int b = ((z / S) * (dy / S) + (y / S)) * (dx / S) + x / S;
  gy[v] += coef * eblk[b];
}

// acc += sum of t^2
__global__ __launch_bounds__(256) void k_sumsq(const float *t, long long n, double *acc)
{
  double s = 0.0;
  for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += (long long)gridDim.x * 256)
    s += (double)t[q] * t[q];
  __shared__ double red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(acc, red[0]);
}

__global__ __launch_bounds__(256) void k_adam(float *p, const float *g, float *m, float *v, long long n, float lr,
                                              float b1, float b2, float eps, float c1, float c2)
{
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const float gq = g[q];
  const float mq = b1 * m[q] + (1.f - b1) * gq;
  const float vq = b2 * v[q] + (1.f - b2) * gq * gq;
  m[q] = mq;
  v[q] = vq;
  p[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

// BF16 weights from the FP32 master W[cout][27*cin], as the convolution's lanes
// read them: [16 outputs][chunk][product][lane][8] (chunks), [16 outputs]
// [product][lane][8] (whole) or [cout][kp], kp = 27 cin rounded up to 32 (rows).
// The data gradient is the same convolution with the taps reversed and the
// channels exchanged, W'[c][26 - tap][n]; its weights follow in wd (null: none).
__global__ __launch_bounds__(256) void k_pack_w(const float *W, int cin, int cout, int kind, int kind_d, bf16_t *wt,
                                                bf16_t *wd)
{
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long nt = packed_weights((ConvKind)kind, cin, cout);
  const long long nd = wd ? packed_weights((ConvKind)kind_d, cout, cin) : 0;
  if (q >= nt + nd) return;
  const bool grad = q >= nt;
  const ConvKind k = (ConvKind)(grad ? kind_d : kind);
  const long long p = grad ? q - nt : q;
  const int ci = grad ? cout : cin;  // channels summed over
  int n, tap, c;
  if (k == ConvKind::rows) {
    const int kp = (27 * ci + 31) / 32 * 32;
    n = (int)(p / kp);
    const int kk = (int)(p - (long long)n * kp);
    tap = kk / ci;
    c = kk - tap * ci;
  } else {
    const int j = (int)(p & 7), lane = (int)(p >> 3) & 63, oct = lane >> 4;
    const int f = (int)(p >> 9);
    if (k == ConvKind::whole) {
      const int m = ci / 32, step = f % (27 * m);
      n = f / (27 * m);
      tap = step / m;
      c = 32 * (step - tap * m) + 8 * oct + j;
    } else {
      const int opt = k == ConvKind::chunks8 ? 1 : 2, tpm = 4 / opt, ng = (27 + tpm - 1) / tpm;
      const int g = f % ng, nchunk = ci / (8 * opt), chunk = f / ng % nchunk;
      n = f / ng / nchunk;
      tap = g * tpm + oct / opt;
      c = 8 * opt * chunk + 8 * (oct % opt) + j;
    }
    n = 16 * n + (lane & 15);
  }
  bf16_t val = 0;
  if (tap < 27)
    val = f2bf(grad ? W[(long long)c * 27 * cin + (26 - tap) * cin + n] : W[(long long)n * 27 * cin + tap * cin + c]);
  (grad ? wd : wt)[p] = val;
}

// fp32 host volume -> BF16 device volume, eight values per thread (n is a
// multiple of eight): 20 -> 8 us for 8.4 M values
__global__ __launch_bounds__(256) void k_f2bf(const float *src, bf16_t *dst, long long n)
{
  const long long q = 8 * ((long long)blockIdx.x * 256 + threadIdx.x);
  if (q >= n) return;
  const float4 a = *reinterpret_cast<const float4 *>(src + q), b = *reinterpret_cast<const float4 *>(src + q + 4);
  *reinterpret_cast<uint4 *>(dst + q) =
      make_uint4((unsigned)f2bf(a.x) | ((unsigned)f2bf(a.y) << 16), (unsigned)f2bf(a.z) | ((unsigned)f2bf(a.w) << 16),
                 (unsigned)f2bf(b.x) | ((unsigned)f2bf(b.y) << 16), (unsigned)f2bf(b.z) | ((unsigned)f2bf(b.w) << 16));
}

// Per-problem scales: s = rms(R) over updated cells, u = max inflow speed of
// the boundary column (0,0).  sc[0] = s, sc[1] = u.
__global__ __launch_bounds__(256) void k_scales(Dims d, const float *R, const float *u0, const float *v0,
                                                double *acc, float *sc, int stage)
{
  if (stage == 0) {
    const int W = d.NX - 2, H = d.NY - 2;
    const long long n = (long long)W * H * (d.NZ - 2);
    double s = 0.0;
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += (long long)gridDim.x * 256) {
      const long long k = q / ((long long)W * H);
      const long long rem = q - k * W * H;
      const long long j = rem / W, i = rem - j * W;
      const float r = R[(i + 1) + (j + 1) * d.sy + (k + 1) * d.sz];
      s += (double)r * r;
    }
    __shared__ double red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int t = 128; t > 0; t >>= 1) {
      if (threadIdx.x < t) red[threadIdx.x] += red[threadIdx.x + t];
      __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(acc, red[0]);
  } else if (blockIdx.x == 0 && threadIdx.x == 0) {
    const long long n = (long long)(d.NX - 2) * (d.NY - 2) * (d.NZ - 2);
    double ms = n > 0 ? acc[0] / (double)n : 0.0;
    float s = (float)sqrt(ms);
    sc[0] = s > 1e-30f ? s : 1.f;
    float um = 0.f;
    for (int k = 0; k < d.nz; ++k) {
      const float a = u0[k * d.fz], b = v0[k * d.fz];
      um = fmaxf(um, sqrtf(a * a + b * b));
    }
    sc[1] = um > 1e-30f ? um : 1.f;
  }
}

// Input features of the padded volume (dx, dy, dz): net voxel (x, y, z) is
// cell (x, y, z+1).  ch0 fluid mask, ch1 R/s, ch2-3 inflow (u, v)/speed at
// that height, ch4 normalised height, ch5-7 zero.
__global__ __launch_bounds__(256) void k_features(Dims d, const int *flag, const float *R, const float *u0,
                                                  const float *v0, const float *sc, int ncx, int ncy, int ncz,
                                                  int dx, int dy, int dz, bf16_t *feat)
{
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long V = (long long)dx * dy * dz;
  if (v >= V) return;
  const int x = (int)(v % dx), y = (int)((v / dx) % dy), z = (int)(v / ((long long)dx * dy));
  float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (x < ncx && y < ncy && z < ncz) {
    const int k = z + 1;
    const long long c = x + (long long)y * d.sy + (long long)k * d.sz;
    f[0] = flag[c] == 1 ? 1.f : 0.f;
    f[1] = R[c] / sc[0];
    f[2] = u0[(long long)k * d.fz] / sc[1];
    f[3] = v0[(long long)k * d.fz] / sc[1];
    f[4] = (z + 0.5f) / (float)ncz;
  }
  uint4 u;
  u.x = f2bf(f[0]) | ((unsigned)f2bf(f[1]) << 16);
  u.y = f2bf(f[2]) | ((unsigned)f2bf(f[3]) << 16);
  u.z = f2bf(f[4]) | ((unsigned)f2bf(f[5]) << 16);
  u.w = f2bf(f[6]) | ((unsigned)f2bf(f[7]) << 16);
  *reinterpret_cast<uint4 *>(feat + v * 8) = u;
}

// target[v] = lambda(cell)/s (0 outside the problem)
__global__ __launch_bounds__(256) void k_target(Dims d, const float *lam, const float *sc, int ncx, int ncy, int ncz,
                                                int dx, int dy, int dz, float *tgt)
{
  const long long v = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long V = (long long)dx * dy * dz;
  if (v >= V) return;
  const int x = (int)(v % dx), y = (int)((v / dx) % dy), z = (int)(v / ((long long)dx * dy));
  float t = 0.f;
  if (x < ncx && y < ncy && z < ncz) t = lam[x + (long long)y * d.sy + (long long)(z + 1) * d.sz] / sc[0];
  tgt[v] = t;
}

// lambda0 of the solver from the prediction: updated cells get out*s, every
// other cell 0, then the k = 0 ghost mirrors k = 1.
__global__ __launch_bounds__(256) void k_install(Dims d, const float *out, const float *sc, float tscale, int dx,
                                                 int dy, float *lam)
{
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long n = (long long)d.NX * d.NY * d.NZ;
  if (c >= n) return;
  const int k = (int)(c / d.sz);
  const long long rem = c - (long long)k * d.sz;
  const int j = (int)(rem / d.sy), i = (int)(rem - (long long)j * d.sy);
  const int kk = k == 0 ? 1 : k;  // ghost layer mirrors layer 1
  float val = 0.f;
  if (i >= 1 && i <= d.NX - 2 && j >= 1 && j <= d.NY - 2 && kk >= 1 && kk <= d.NZ - 2 && d.NZ >= 3)
    val = out[((long long)(kk - 1) * dy + j) * dx + i] * tscale * sc[0];
  lam[c] = val;
}

}  // namespace unet
}  // namespace qesmc

using namespace qesmc;
using namespace qesmc::unet;

namespace {

struct Conv {
  int cin, cout, kp, kpd;
  long long woff, boff;  // offsets in the parameter vector
  ConvKind kind, kind_d;  // forward, data gradient
  bf16_t *wt = nullptr, *wd = nullptr;
};

struct Level {
  int dx, dy, dz;
  long long V;
  int c;        // channels of this level
  int ldcat;    // channels of CAT (c + c_{l+1}, or c at the bottom)
  bf16_t *A = nullptr, *CAT = nullptr, *P = nullptr, *E = nullptr, *D = nullptr;
  bf16_t *gA = nullptr, *gCAT = nullptr, *gP = nullptr, *gE = nullptr, *gD = nullptr;
};

inline int round_up(int a, int b) { return (a + b - 1) / b * b; }

}  // namespace

struct qesmc_unet {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev[2] = {};
  int L = 4, c0 = 16;
  int ncx = 0, ncy = 0, ncz = 0;
  int dx = 0, dy = 0, dz = 0;
  std::vector<Conv> enc1, enc2, dec1, dec2;  // per level
  long long head_off = 0, nparams = 0;
  float *p = nullptr, *gp = nullptr, *m1 = nullptr, *m2 = nullptr;
  int adam_t = 0;
  std::vector<Level> lv;
  bf16_t *feat = nullptr;        // scratch input [V0][8]
  float *out = nullptr, *gout = nullptr, *tgt = nullptr, *hostbuf_dev = nullptr;
  float *sc = nullptr;           // scales of the current problem
  double *dacc = nullptr;
  float *loss = nullptr;
  std::vector<bf16_t *> sfeat;   // dataset
  std::vector<float *> stgt;
  double conv_flops = 0.0;       // forward FLOPs of all convolutions
  float tscale = 0.f;            // output unit (0: derive from the samples)
  int loss_block = 0;            // block-mean loss term: block edge (0: off)
  float loss_weight = 0.f;       //   and its weight
  float *eblk = nullptr;         //   block means of the error
};

namespace {

#define UCHK(expr)                                   \
  do {                                               \
    hipError_t _e = (expr);                          \
    if (_e != hipSuccess) return map_err(_e);        \
  } while (0)

int map_err(hipError_t e)
{
  if (e == hipErrorOutOfMemory) return QESMC_ERR_OOM;
  if (e == hipErrorNoDevice || e == hipErrorInvalidDevice) return QESMC_ERR_NO_DEVICE;
  return QESMC_ERR_HIP;
}

template <typename T>
hipError_t dmalloc(T **p, long long n)
{
  *p = nullptr;
  return hipMalloc((void **)p, sizeof(T) * (size_t)(n > 0 ? n : 1));
}

inline dim3 g1(long long n) { return dim3((unsigned)((n + 255) / 256)); }

// the 8-channel data-movement kernels apply: channels, strides and offset in
// whole 16-byte groups, and every index fits 32 bits
inline bool vec8(int ch, int ld_a, int ld_b, int off, long long V)
{
  return ch % 8 == 0 && ld_a % 8 == 0 && ld_b % 8 == 0 && off % 8 == 0 && V * (long long)(ld_a > ld_b ? ld_a : ld_b) < (1LL << 31);
}

template <int SY, int SZ, int WN>
hipError_t launch_whole(hipStream_t s, const ConvFwdArgs &a)
{
  const size_t bytes = 2 * (size_t)kHaloX * (SY + 2) * (SZ + 2) * a.cin;
  const long long bricks =
      (long long)((a.dx + kBrickX - 1) / kBrickX) * ((a.dy + SY - 1) / SY) * ((a.dz + SZ - 1) / SZ);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv_whole<SY, SZ, WN>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_conv_whole<SY, SZ, WN>), dim3((unsigned)((bricks + kXcdsU - 1) / kXcdsU * kXcdsU), (unsigned)(a.cout / 16 / WN)),
                     dim3(256), bytes, s, a);
  return hipGetLastError();
}

template <int WN>
hipError_t launch_whole_size(hipStream_t s, const ConvFwdArgs &a)
{
  // the largest brick that fits the 160 KB of LDS and leaves a work-group per CU
  auto fits = [&](int sy, int sz) {
    const long long bricks =
        (long long)((a.dx + kBrickX - 1) / kBrickX) * ((a.dy + sy - 1) / sy) * ((a.dz + sz - 1) / sz);
    return 2LL * kHaloX * (sy + 2) * (sz + 2) * a.cin <= 160 * 1024 && bricks * (a.cout / 16 / WN) >= 256;
  };
  if constexpr (WN < 4)  // 16 tiles a wave would spill
    if (fits(4, 4)) return launch_whole<4, 4, WN>(s, a);
  if (fits(4, 2)) return launch_whole<4, 2, WN>(s, a);
  if (fits(2, 2)) return launch_whole<2, 2, WN>(s, a);
  return launch_whole<WN == 1 ? 2 : 1, 2, WN>(s, a);
}

hipError_t launch_conv_fwd(hipStream_t s, const ConvFwdArgs &a)
{
  if (a.cout % 16 || a.ldx % 8 || a.ldy % 4) return hipErrorInvalidValue;
  const int NT = a.cout / 16;
  const long long V = (long long)a.dx * a.dy * a.dz;
  auto chunks = [&](auto kern) {
    const long long bricks = (long long)((a.dx + kBrickX - 1) / kBrickX) * ((a.dy + 7) / 8) * ((a.dz + 3) / 4);
    // one chunk: staged once for all outputs where there are bricks enough
    const bool split = a.cin > 16 || bricks < 1024;
    hipLaunchKernelGGL(kern, dim3((unsigned)((bricks + kXcdsU - 1) / kXcdsU * kXcdsU), (unsigned)(split ? NT : 1)),
                       dim3(256), 0, s, a);
    return hipGetLastError();
  };
  // A lane's offset from the halo's first voxel has 31 bits in a buffer load.
  // The halo's last voxel is at most a row of it (kHaloX) beyond six planes, and 32
  // bytes of it are read.
  const bool wide = (6LL * a.dy * a.dx + kHaloX) * 2 * a.ldx + 32 > 0x7fffffffLL;
  switch (conv_kind(a.cin, a.dx, a.dy, a.dz)) {
  case ConvKind::chunks8: return wide ? chunks(k_conv_chunks<8, true>) : chunks(k_conv_chunks<8, false>);
  case ConvKind::chunks16: return wide ? chunks(k_conv_chunks<16, true>) : chunks(k_conv_chunks<16, false>);
  case ConvKind::whole:
    return NT % 4 == 0 ? launch_whole_size<4>(s, a) : NT % 2 == 0 ? launch_whole_size<2>(s, a) : launch_whole_size<1>(s, a);
  default: break;
  }
  auto go = [&](auto kern, int MT, int rows = 1) {
    const long long waves = (V + 16LL * MT - 1) / (16LL * MT);
    hipLaunchKernelGGL(kern, dim3((unsigned)((waves + 3) / 4), (unsigned)rows), dim3(256), 0, s, a);
    return hipGetLastError();
  };
  // up to 4096 waves cover the GPU
  const long long want = 4096, w4 = (V + 63) / 64 * NT, w2 = (V + 31) / 32 * NT;
  return w4 >= want ? go(k_conv_fwd<1, 4>, 4, NT) : w2 >= want ? go(k_conv_fwd<1, 2>, 2, NT) : go(k_conv_fwd<1, 1>, 1, NT);
}

// Work-groups of the weight gradient: two per CU over all channel pairs (its
// registers allow two waves per SIMD), and strips of at least 8 rows of X,
// shorter than the volume only as far as there are work-groups for them.
hipError_t launch_wgrad(hipStream_t s, const ConvWgradArgs &a0, int cout)
{
  ConvWgradArgs a = a0;
  a.ctiles = (a.cin + 15) / 16;
  const int pairs = a.ctiles * (cout / 16);
  const long long columns = (long long)((a.dx + 31) / 32) * a.dz;
  const long long waves = 2048 / pairs > 4 ? 2048 / pairs : 4;
  a.ylen = a.dy;
  while (a.ylen > 8 && columns * ((a.dy + a.ylen - 1) / a.ylen) < waves) a.ylen = (a.ylen + 1) / 2;
  const long long strips = columns * ((a.dy + a.ylen - 1) / a.ylen);
  const long long blocks = (strips < waves ? strips : waves) + 3;
  hipLaunchKernelGGL(k_conv_wgrad, dim3((unsigned)(blocks / 4), (unsigned)pairs), dim3(256), 0, s, a);
  return hipGetLastError();
}

// Work-groups of the kernels that reduce over voxels, eight channels per
// thread: enough to fill the GPU, few enough for their atomics.
inline unsigned reduce_blocks(long long V, int ch)
{
  const long long b = (V * (ch / 8) + 255) / 256;
  return (unsigned)(b < 1024 ? b : 1024);
}

// One conv layer forward: x (ldx, cin) -> y (ldy), bias + ReLU
hipError_t conv_forward(qesmc_unet *u, const Conv &cv, const Level &lv, const bf16_t *x, int ldx, bf16_t *y, int ldy)
{
  ConvFwdArgs a{x, ldx, cv.cin, 27 * cv.cin, cv.cout, cv.wt, cv.kp, u->p + cv.boff, y, ldy, lv.dx, lv.dy, lv.dz, 1};
  return launch_conv_fwd(u->stream, a);
}

// Backward through one conv layer whose ReLU output y (ldy) received the
// gradient g (ldg; masked in place, after gpool's share if given); x is its
// input.  Adds dW, db; if gx is given, writes dL/dx into it (ldgx, cin
// channels at offset 0).
hipError_t conv_backward(qesmc_unet *u, const Conv &cv, const Level &lv, const bf16_t *x, int ldx,
                         const bf16_t *y, int ldy, bf16_t *g, int ldg, const bf16_t *gpool, bf16_t *gx, int ldgx)
{
  hipStream_t s = u->stream;
  const long long V = lv.V;
  hipLaunchKernelGGL(k_relu_bias_bwd, dim3(reduce_blocks(V, cv.cout)), dim3(256), 0, s, g, ldg, y, ldy, cv.cout, V,
                     gpool, lv.dx, lv.dy, u->gp + cv.boff);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ConvWgradArgs wa{x, ldx, cv.cin, 27 * cv.cin, g, ldg, u->gp + cv.woff, lv.dx, lv.dy, lv.dz, 0, 0};
  if ((e = launch_wgrad(s, wa, cv.cout)) != hipSuccess) return e;
  if (gx) {
    ConvFwdArgs a{g, ldg, cv.cout, 27 * cv.cout, cv.cin, cv.wd, cv.kpd, nullptr, gx, ldgx, lv.dx, lv.dy, lv.dz, 0};
    if ((e = launch_conv_fwd(s, a)) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t pack_weights(qesmc_unet *u)
{
  auto pk = [&](Conv &c) {
    const long long n = packed_weights(c.kind, c.cin, c.cout) + (c.wd ? packed_weights(c.kind_d, c.cout, c.cin) : 0);
    hipLaunchKernelGGL(k_pack_w, g1(n), dim3(256), 0, u->stream, u->p + c.woff, c.cin, c.cout, (int)c.kind,
                       (int)c.kind_d, c.wt, c.wd);
  };
  for (int l = 0; l < u->L; ++l) {
    pk(u->enc1[l]);
    pk(u->enc2[l]);
  }
  for (int l = 0; l + 1 < u->L; ++l) {
    pk(u->dec1[l]);
    pk(u->dec2[l]);
  }
  return hipGetLastError();
}

hipError_t forward(qesmc_unet *u, const bf16_t *feat)
{
  hipStream_t s = u->stream;
  hipError_t e;
  const int L = u->L;
  for (int l = 0; l < L; ++l) {
    Level &lv = u->lv[l];
    const bf16_t *in = l == 0 ? feat : lv.P;
    const int ldin = l == 0 ? QESMC_UNET_IN_CHANNELS : u->lv[l - 1].c;
    if ((e = conv_forward(u, u->enc1[l], lv, in, ldin, lv.A, lv.c)) != hipSuccess) return e;
    if ((e = conv_forward(u, u->enc2[l], lv, lv.A, lv.c, lv.CAT, lv.ldcat)) != hipSuccess) return e;
    if (l + 1 < L) {
      Level &nx = u->lv[l + 1];
      if (vec8(lv.c, lv.ldcat, lv.c, 0, nx.V))
        hipLaunchKernelGGL(k_pool_fwd8, g1(nx.V * lv.c / 8), dim3(256), 0, s, lv.CAT, lv.ldcat, 0, nx.P, lv.c, lv.c,
                           nx.dx, nx.dy, nx.dz);
      else
        hipLaunchKernelGGL(k_pool_fwd, g1(nx.V * lv.c), dim3(256), 0, s, lv.CAT, lv.ldcat, 0, nx.P, lv.c, lv.c,
                           nx.dx, nx.dy, nx.dz);
    }
  }
  for (int l = L - 2; l >= 0; --l) {
    Level &lv = u->lv[l];
    Level &dn = u->lv[l + 1];
    const bf16_t *src = (l == L - 2) ? dn.CAT : dn.D;
    const int ldsrc = (l == L - 2) ? dn.ldcat : dn.c;
    if (vec8(dn.c, ldsrc, lv.ldcat, lv.c, lv.V))
      hipLaunchKernelGGL(k_up_fwd8, g1(lv.V * dn.c / 8), dim3(256), 0, s, src, ldsrc, lv.CAT, lv.ldcat, lv.c, dn.c,
                         lv.dx, lv.dy, lv.dz);
    else
      hipLaunchKernelGGL(k_up_fwd, g1(lv.V * dn.c), dim3(256), 0, s, src, ldsrc, lv.CAT, lv.ldcat, lv.c, dn.c, lv.dx,
                         lv.dy, lv.dz);
    if ((e = conv_forward(u, u->dec1[l], lv, lv.CAT, lv.ldcat, lv.E, lv.c)) != hipSuccess) return e;
    if ((e = conv_forward(u, u->dec2[l], lv, lv.E, lv.c, lv.D, lv.c)) != hipSuccess) return e;
  }
  Level &top = u->lv[0];
  if (vec8(top.c, top.c, top.c, 0, top.V))
    hipLaunchKernelGGL(k_head_fwd8, g1(top.V), dim3(256), 0, s, top.D, top.c, top.c, u->p + u->head_off, u->out,
                       top.V);
  else
    hipLaunchKernelGGL(k_head_fwd, g1(top.V), dim3(256), 0, s, top.D, top.c, top.c, u->p + u->head_off, u->out,
                       top.V);
  return hipGetLastError();
}

// gradients of all parameters (added into u->gp, which the caller zeroes)
// from u->gout (dL/d output)
hipError_t backward(qesmc_unet *u, const bf16_t *feat)
{
  hipStream_t s = u->stream;
  hipError_t e;
  const int L = u->L;
  Level &top = u->lv[0];
  hipLaunchKernelGGL(k_head_bwd, dim3(reduce_blocks(top.V, top.c)), dim3(256), 0, s, top.D, top.c, top.c,
                     u->p + u->head_off, u->gout, top.gD, u->gp + u->head_off, top.V);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  for (int l = 0; l + 1 < L; ++l) {
    Level &lv = u->lv[l];
    Level &dn = u->lv[l + 1];
    if ((e = conv_backward(u, u->dec2[l], lv, lv.E, lv.c, lv.D, lv.c, lv.gD, lv.c, nullptr, lv.gE, lv.c)) != hipSuccess)
      return e;
    if ((e = conv_backward(u, u->dec1[l], lv, lv.CAT, lv.ldcat, lv.E, lv.c, lv.gE, lv.c, nullptr, lv.gCAT, lv.ldcat)) !=
        hipSuccess)
      return e;
    bf16_t *gsrc = (l == L - 2) ? dn.gCAT : dn.gD;
    const int ldg = (l == L - 2) ? dn.ldcat : dn.c;
    hipLaunchKernelGGL(k_up_bwd, g1(dn.V * dn.c / 8), dim3(256), 0, s, lv.gCAT, lv.ldcat, lv.c, gsrc, ldg, dn.c, dn.dx,
                       dn.dy, dn.dz);
  }
  for (int l = L - 1; l >= 0; --l) {
    Level &lv = u->lv[l];
    // the encoder output's gradient: the skip's share, plus the pool's from below
    const bf16_t *gpool = l + 1 < L ? u->lv[l + 1].gP : nullptr;
    if ((e = conv_backward(u, u->enc2[l], lv, lv.A, lv.c, lv.CAT, lv.ldcat, lv.gCAT, lv.ldcat, gpool, lv.gA, lv.c)) !=
        hipSuccess)
      return e;
    const bf16_t *in = l == 0 ? feat : lv.P;
    const int ldin = l == 0 ? QESMC_UNET_IN_CHANNELS : u->lv[l - 1].c;
    if ((e = conv_backward(u, u->enc1[l], lv, in, ldin, lv.A, lv.c, lv.gA, lv.c, nullptr, l > 0 ? lv.gP : nullptr,
                           ldin)) != hipSuccess)
      return e;
  }
  return hipSuccess;
}

void free_all(qesmc_unet *u)
{
  auto f = [](auto *&p) {
    if (p) (void)hipFree((void *)p);
    p = nullptr;
  };
  for (auto *v : {&u->enc1, &u->enc2, &u->dec1, &u->dec2})
    for (auto &c : *v) {
      f(c.wt);
      f(c.wd);
    }
  for (auto &l : u->lv) {
    f(l.A), f(l.CAT), f(l.P), f(l.E), f(l.D), f(l.gA), f(l.gCAT), f(l.gP), f(l.gE), f(l.gD);
  }
  f(u->p), f(u->gp), f(u->m1), f(u->m2), f(u->feat), f(u->out), f(u->gout), f(u->tgt), f(u->hostbuf_dev);
  f(u->sc), f(u->dacc), f(u->loss), f(u->eblk);
  for (auto &q : u->sfeat) f(q);
  for (auto &q : u->stgt) f(q);
  u->sfeat.clear();
  u->stgt.clear();
}

// Loss of the current output against target t into u->loss, gradient into
// u->gout: mean squared error plus the optional block-mean term.
hipError_t launch_loss(qesmc_unet *u, const float *t, bool grad)
{
  hipStream_t s = u->stream;
  const long long V0 = (long long)u->dx * u->dy * u->dz;
  hipLaunchKernelGGL(k_mse, g1(V0), dim3(256), 0, s, u->out, t, 1.f / u->tscale, u->gout, V0, u->loss);
  if (u->loss_block > 0 && u->loss_weight > 0.f) {
    const int S = u->loss_block;
    const long long nb = (long long)(u->dx / S) * (u->dy / S) * (u->dz / S);
    hipLaunchKernelGGL(k_block_err, dim3((unsigned)nb), dim3(256), 0, s, u->gout, 0.5f * (float)V0, u->dx, u->dy, S,
                       u->loss_weight / (float)nb, u->eblk, u->loss);
    if (grad)
      hipLaunchKernelGGL(k_block_grad, g1(V0), dim3(256), 0, s, u->gout, u->eblk, u->dx, u->dy, u->dz, S,
                         2.f * u->loss_weight / ((float)nb * (float)(S * S * S)));
  }
  return hipGetLastError();
}

// features + scales of ctx's resident problem into u->feat, u->sc
int problem_features(qesmc_unet *u, qesmc_ctx *x)
{
  if (!x->have_geom || !x->have_inflow) return QESMC_ERR_STATE;
  if (x->d.nx - 1 != u->ncx || x->d.ny - 1 != u->ncy || x->d.nz - 2 != u->ncz) return QESMC_ERR_ARG;
  UCHK(hipStreamSynchronize(x->stream));
  // R on the x-fastest layout, on the solver's stream
  UCHK(qesmc_launch_divergence(x, 0, 1));
  UCHK(hipStreamSynchronize(x->stream));
  hipStream_t s = u->stream;
  UCHK(hipMemsetAsync(u->dacc, 0, sizeof(double), s));
  hipLaunchKernelGGL(k_scales, dim3(512), dim3(256), 0, s, x->d, x->d_R, x->d_u0, x->d_v0, u->dacc, u->sc, 0);
  hipLaunchKernelGGL(k_scales, dim3(1), dim3(64), 0, s, x->d, x->d_R, x->d_u0, x->d_v0, u->dacc, u->sc, 1);
  const long long V = (long long)u->dx * u->dy * u->dz;
  hipLaunchKernelGGL(k_features, g1(V), dim3(256), 0, s, x->d, x->d_flag, x->d_R, x->d_u0, x->d_v0, u->sc, u->ncx,
                     u->ncy, u->ncz, u->dx, u->dy, u->dz, u->feat);
  UCHK(hipGetLastError());
  return QESMC_OK;
}

}  // namespace

extern "C" {

int qesmc_unet_create(qesmc_unet **out, int device, const qesmc_unet_config *cfg)
{
  if (!out || !cfg) return QESMC_ERR_ARG;
  *out = nullptr;
  if (cfg->levels < 2 || cfg->levels > 5 || cfg->base_channels < 16 || cfg->base_channels > 32 ||
      cfg->base_channels % 16 ||
      cfg->base_channels * (1 << (cfg->levels - 1)) > 128 || cfg->ncx < 1 || cfg->ncy < 1 || cfg->ncz < 1)
    return QESMC_ERR_ARG;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n) return QESMC_ERR_NO_DEVICE;
  UCHK(hipSetDevice(device));
  qesmc_unet *u = new (std::nothrow) qesmc_unet();
  if (!u) return QESMC_ERR_OOM;
  u->device = device;
  host_copy_attach(device);
  u->L = cfg->levels;
  u->c0 = cfg->base_channels;
  u->ncx = cfg->ncx;
  u->ncy = cfg->ncy;
  u->ncz = cfg->ncz;
  u->tscale = cfg->target_scale > 0.f ? cfg->target_scale : 0.f;
  const int mult = 1 << (u->L - 1);
  u->dx = round_up(cfg->ncx, mult);
  u->dy = round_up(cfg->ncy, mult);
  u->dz = round_up(cfg->ncz, mult);
  // layers and parameter offsets
  long long off = 0;
  auto mk = [&](int cin, int cout) {
    Conv c;
    c.cin = cin;
    c.cout = cout;
    c.kp = round_up(27 * cin, 32);
    c.kpd = round_up(27 * cout, 32);
    c.woff = off;
    off += 27LL * cin * cout;
    c.boff = off;
    off += cout;
    return c;
  };
  u->lv.resize(u->L);
  for (int l = 0; l < u->L; ++l) {
    const int c = u->c0 << l;
    const int cin = l == 0 ? QESMC_UNET_IN_CHANNELS : (u->c0 << (l - 1));
    u->enc1.push_back(mk(cin, c));
    u->enc2.push_back(mk(c, c));
  }
  u->dec1.resize(u->L - 1);
  u->dec2.resize(u->L - 1);
  for (int l = u->L - 2; l >= 0; --l) {
    const int c = u->c0 << l;
    u->dec1[l] = mk(c + (c << 1), c);
    u->dec2[l] = mk(c, c);
  }
  u->head_off = off;
  off += u->c0 + 1;
  u->nparams = off;

  int rc = QESMC_OK;
  auto fail = [&](hipError_t e) {
    if (e != hipSuccess) rc = map_err(e);
    return e != hipSuccess;
  };
  if (fail(hipStreamCreateWithFlags(&u->stream, hipStreamNonBlocking)) || fail(hipEventCreate(&u->ev[0])) ||
      fail(hipEventCreate(&u->ev[1]))) {
    qesmc_unet_destroy(u);
    return rc;
  }
  bool bad = fail(dmalloc(&u->p, off)) || fail(dmalloc(&u->gp, off)) || fail(dmalloc(&u->m1, off)) ||
             fail(dmalloc(&u->m2, off));
  for (auto *v : {&u->enc1, &u->enc2, &u->dec1, &u->dec2})
    for (size_t l = 0; l < v->size(); ++l) {
      Conv &c = (*v)[l];
      c.kind = conv_kind(c.cin, u->dx >> l, u->dy >> l, u->dz >> l);
      c.kind_d = conv_kind(c.cout, u->dx >> l, u->dy >> l, u->dz >> l);
      bad = bad || fail(dmalloc(&c.wt, packed_weights(c.kind, c.cin, c.cout)));
      if (c.cin % 16 == 0)  // the network's input needs no gradient
        bad = bad || fail(dmalloc(&c.wd, packed_weights(c.kind_d, c.cout, c.cin)));
    }
  double flops = 0.0;
  for (int l = 0; l < u->L && !bad; ++l) {
    Level &lv = u->lv[l];
    lv.dx = u->dx >> l;
    lv.dy = u->dy >> l;
    lv.dz = u->dz >> l;
    lv.V = (long long)lv.dx * lv.dy * lv.dz;
    lv.c = u->c0 << l;
    lv.ldcat = (l + 1 < u->L) ? lv.c + (lv.c << 1) : lv.c;
    const long long V = lv.V;
    bad = fail(dmalloc(&lv.A, V * lv.c)) || fail(dmalloc(&lv.CAT, V * lv.ldcat)) || fail(dmalloc(&lv.E, V * lv.c)) ||
          fail(dmalloc(&lv.D, V * lv.c)) || fail(dmalloc(&lv.gA, V * lv.c)) || fail(dmalloc(&lv.gCAT, V * lv.ldcat)) ||
          fail(dmalloc(&lv.gE, V * lv.c)) || fail(dmalloc(&lv.gD, V * lv.c));
    if (!bad && l > 0) {
      const int cp = u->c0 << (l - 1);
      bad = fail(dmalloc(&lv.P, V * cp)) || fail(dmalloc(&lv.gP, V * cp));
    }
    flops += 2.0 * V * 27.0 * (u->enc1[l].cin * (double)u->enc1[l].cout + u->enc2[l].cin * (double)u->enc2[l].cout);
    if (l + 1 < u->L)
      flops += 2.0 * V * 27.0 * (u->dec1[l].cin * (double)u->dec1[l].cout + u->dec2[l].cin * (double)u->dec2[l].cout);
  }
  u->conv_flops = flops;
  const long long V0 = (long long)u->dx * u->dy * u->dz;
  bad = bad || fail(dmalloc(&u->feat, V0 * QESMC_UNET_IN_CHANNELS)) || fail(dmalloc(&u->out, V0)) ||
        fail(dmalloc(&u->gout, V0)) || fail(dmalloc(&u->tgt, V0)) ||
        fail(dmalloc(&u->hostbuf_dev, V0 * QESMC_UNET_IN_CHANNELS)) || fail(dmalloc(&u->sc, 2)) ||
        fail(dmalloc(&u->dacc, 1)) || fail(dmalloc(&u->loss, 1));
  if (bad) {
    qesmc_unet_destroy(u);
    return rc == QESMC_OK ? QESMC_ERR_OOM : rc;
  }
  // He-normal initialisation of the conv weights, zero biases (host RNG)
  std::vector<float> hp((size_t)off, 0.f);
  std::mt19937_64 rng(cfg->seed);
  auto init = [&](const Conv &c) {
    std::normal_distribution<double> nd(0.0, std::sqrt(2.0 / (27.0 * c.cin)));
    for (long long q = 0; q < 27LL * c.cin * c.cout; ++q) hp[(size_t)(c.woff + q)] = (float)nd(rng);
  };
  for (int l = 0; l < u->L; ++l) {
    init(u->enc1[l]);
    init(u->enc2[l]);
  }
  for (int l = u->L - 2; l >= 0; --l) {
    init(u->dec1[l]);
    init(u->dec2[l]);
  }
  std::normal_distribution<double> nh(0.0, std::sqrt(1.0 / u->c0));
  for (int c = 0; c < u->c0; ++c) hp[(size_t)(u->head_off + c)] = (float)nh(rng);
  rc = qesmc_unet_set_params(u, hp.data(), off);
  if (rc != QESMC_OK) {
    qesmc_unet_destroy(u);
    return rc;
  }
  *out = u;
  return QESMC_OK;
}

int qesmc_unet_destroy(qesmc_unet *u)
{
  if (!u) return QESMC_OK;
  (void)hipSetDevice(u->device);
  if (u->stream) (void)hipStreamSynchronize(u->stream);
  free_all(u);
  for (auto &e : u->ev)
    if (e) (void)hipEventDestroy(e);
  if (u->stream) (void)hipStreamDestroy(u->stream);
  host_copy_detach(u->device);
  delete u;
  return QESMC_OK;
}

int qesmc_unet_num_params(const qesmc_unet *u, long long *count)
{
  if (!u || !count) return QESMC_ERR_ARG;
  *count = u->nparams;
  return QESMC_OK;
}

int qesmc_unet_dims(const qesmc_unet *u, int *dx, int *dy, int *dz)
{
  if (!u || !dx || !dy || !dz) return QESMC_ERR_ARG;
  *dx = u->dx;
  *dy = u->dy;
  *dz = u->dz;
  return QESMC_OK;
}

int qesmc_unet_get_params(qesmc_unet *u, float *host, long long count)
{
  if (!u || !host || count != u->nparams) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  UCHK(hipMemcpyAsync(host, u->p, sizeof(float) * count, hipMemcpyDeviceToHost, u->stream));
  UCHK(hipStreamSynchronize(u->stream));
  return QESMC_OK;
}

int qesmc_unet_set_params(qesmc_unet *u, const float *host, long long count)
{
  if (!u || !host || count != u->nparams) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  UCHK(hipMemcpyAsync(u->p, host, sizeof(float) * count, hipMemcpyHostToDevice, u->stream));
  UCHK(hipMemsetAsync(u->m1, 0, sizeof(float) * count, u->stream));
  UCHK(hipMemsetAsync(u->m2, 0, sizeof(float) * count, u->stream));
  u->adam_t = 0;
  UCHK(pack_weights(u));
  UCHK(hipStreamSynchronize(u->stream));
  return QESMC_OK;
}

int qesmc_unet_forward(qesmc_unet *u, const float *input, float *output)
{
  if (!u || !input || !output) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  const long long V0 = (long long)u->dx * u->dy * u->dz;
  const long long n = V0 * QESMC_UNET_IN_CHANNELS;
  const HostPiece in = host_piece(input, u->hostbuf_dev, sizeof(float) * (size_t)n);
  UCHK(host_copy(u->device, u->stream, &in, 1, true));
  hipLaunchKernelGGL(k_f2bf, g1(n / 8), dim3(256), 0, u->stream, u->hostbuf_dev, u->feat, n);
  UCHK(hipGetLastError());
  UCHK(forward(u, u->feat));
  const HostPiece out = host_piece(output, u->out, sizeof(float) * (size_t)V0);
  UCHK(host_copy(u->device, u->stream, &out, 1, false));
  return QESMC_OK;
}

int qesmc_unet_backward(qesmc_unet *u, const float *grad_output, float *grad_params)
{
  if (!u || !grad_output || !grad_params) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  const long long V0 = (long long)u->dx * u->dy * u->dz;
  const HostPiece in = host_piece(grad_output, u->gout, sizeof(float) * (size_t)V0);
  UCHK(host_copy(u->device, u->stream, &in, 1, true));
  UCHK(hipMemsetAsync(u->gp, 0, sizeof(float) * u->nparams, u->stream));
  UCHK(backward(u, u->feat));
  const HostPiece out = host_piece(grad_params, u->gp, sizeof(float) * (size_t)u->nparams);
  UCHK(host_copy(u->device, u->stream, &out, 1, false));
  return QESMC_OK;
}

int qesmc_unet_add_sample(qesmc_unet *u, qesmc_ctx *x)
{
  if (!u || !x) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  int rc = problem_features(u, x);
  if (rc != QESMC_OK) return rc;
  const long long V0 = (long long)u->dx * u->dy * u->dz;
  bf16_t *f = nullptr;
  float *t = nullptr;
  if (hipMalloc((void **)&f, sizeof(bf16_t) * V0 * QESMC_UNET_IN_CHANNELS) != hipSuccess) return QESMC_ERR_OOM;
  if (hipMalloc((void **)&t, sizeof(float) * V0) != hipSuccess) {
    (void)hipFree(f);
    return QESMC_ERR_OOM;
  }
  UCHK(hipMemcpyAsync(f, u->feat, sizeof(bf16_t) * V0 * QESMC_UNET_IN_CHANNELS, hipMemcpyDeviceToDevice, u->stream));
  hipLaunchKernelGGL(k_target, g1(V0), dim3(256), 0, u->stream, x->d, x->d_lam, u->sc, u->ncx, u->ncy, u->ncz, u->dx,
                     u->dy, u->dz, t);
  UCHK(hipGetLastError());
  UCHK(hipStreamSynchronize(u->stream));
  u->sfeat.push_back(f);
  u->stgt.push_back(t);
  return QESMC_OK;
}

int qesmc_unet_num_samples(const qesmc_unet *u, int *count)
{
  if (!u || !count) return QESMC_ERR_ARG;
  *count = (int)u->sfeat.size();
  return QESMC_OK;
}

int qesmc_unet_clear_samples(qesmc_unet *u)
{
  if (!u) return QESMC_ERR_ARG;
  (void)hipSetDevice(u->device);
  (void)hipStreamSynchronize(u->stream);
  for (auto &q : u->sfeat) (void)hipFree(q);
  for (auto &q : u->stgt) (void)hipFree(q);
  u->sfeat.clear();
  u->stgt.clear();
  return QESMC_OK;
}

int qesmc_unet_train(qesmc_unet *u, int steps, float lr, int first, int last, unsigned long long seed,
                     float *mean_loss, double *ms)
{
  if (!u || steps < 0 || first < 0 || last > (int)u->sfeat.size() || first >= last) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  hipStream_t s = u->stream;
  const long long V0 = (long long)u->dx * u->dy * u->dz;
  if (!(u->tscale > 0.f)) {
    // output unit from the data: RMS of the stored targets lambda / rms(R)
    UCHK(hipMemsetAsync(u->dacc, 0, sizeof(double), s));
    for (size_t q = 0; q < u->stgt.size(); ++q)
      hipLaunchKernelGGL(k_sumsq, dim3(256), dim3(256), 0, s, u->stgt[q], V0, u->dacc);
    double ss = 0.0;
    UCHK(hipMemcpyAsync(&ss, u->dacc, sizeof(double), hipMemcpyDeviceToHost, s));
    UCHK(hipStreamSynchronize(s));
    const double rms = std::sqrt(ss / ((double)V0 * u->stgt.size()));
    u->tscale = rms > 0.0 ? (float)rms : 1.f;
  }
  std::mt19937_64 rng(seed);
  std::uniform_int_distribution<int> pick(first, last - 1);
  UCHK(hipMemsetAsync(u->loss, 0, sizeof(float), s));
  UCHK(hipEventRecord(u->ev[0], s));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int it = 0; it < steps; ++it) {
    const int q = pick(rng);
    UCHK(forward(u, u->sfeat[q]));
    UCHK(launch_loss(u, u->stgt[q], true));
    UCHK(hipMemsetAsync(u->gp, 0, sizeof(float) * u->nparams, s));
    UCHK(backward(u, u->sfeat[q]));
    ++u->adam_t;
    const float c1 = 1.f - std::pow(b1, (float)u->adam_t), c2 = 1.f - std::pow(b2, (float)u->adam_t);
    hipLaunchKernelGGL(k_adam, g1(u->nparams), dim3(256), 0, s, u->p, u->gp, u->m1, u->m2, u->nparams, lr, b1, b2,
                       eps, c1, c2);
    UCHK(pack_weights(u));
  }
  UCHK(hipEventRecord(u->ev[1], s));
  float l = 0.f;
  UCHK(hipMemcpyAsync(&l, u->loss, sizeof(float), hipMemcpyDeviceToHost, s));
  UCHK(hipStreamSynchronize(s));
  if (mean_loss) *mean_loss = steps > 0 ? l / steps : 0.f;
  if (ms) {
    float t = 0.f;
    (void)hipEventElapsedTime(&t, u->ev[0], u->ev[1]);
    *ms = t;
  }
  return QESMC_OK;
}

int qesmc_unet_set_loss(qesmc_unet *u, int block, float weight)
{
  if (!u || block < 0 || !(weight >= 0.f)) return QESMC_ERR_ARG;
  if (block > 0 && ((block & (block - 1)) || u->dx % block || u->dy % block || u->dz % block)) return QESMC_ERR_ARG;
  UCHK(hipSetDevice(u->device));
  if (u->eblk) {
    UCHK(hipStreamSynchronize(u->stream));
    UCHK(hipFree(u->eblk));
    u->eblk = nullptr;
  }
  u->loss_block = weight > 0.f ? block : 0;
  u->loss_weight = u->loss_block ? weight : 0.f;
  if (u->loss_block) {
    const long long nb = (long long)(u->dx / block) * (u->dy / block) * (u->dz / block);
    UCHK(hipMalloc((void **)&u->eblk, sizeof(float) * nb));
  }
  return QESMC_OK;
}

int qesmc_unet_target_scale(const qesmc_unet *u, float *scale)
{
  if (!u || !scale) return QESMC_ERR_ARG;
  *scale = u->tscale;
  return QESMC_OK;
}

int qesmc_unet_eval(qesmc_unet *u, int first, int last, float *mean_loss)
{
  if (!u || !mean_loss || first < 0 || last > (int)u->sfeat.size() || first >= last) return QESMC_ERR_ARG;
  if (!(u->tscale > 0.f)) return QESMC_ERR_STATE;  // no output unit yet: train or configure it
  UCHK(hipSetDevice(u->device));
  hipStream_t s = u->stream;
  UCHK(hipMemsetAsync(u->loss, 0, sizeof(float), s));
  for (int q = first; q < last; ++q) {
    UCHK(forward(u, u->sfeat[q]));
    UCHK(launch_loss(u, u->stgt[q], false));
  }
  float l = 0.f;
  UCHK(hipMemcpyAsync(&l, u->loss, sizeof(float), hipMemcpyDeviceToHost, s));
  UCHK(hipStreamSynchronize(s));
  *mean_loss = l / (last - first);
  return QESMC_OK;
}

int qesmc_unet_predict(qesmc_unet *u, qesmc_ctx *x, double *ms, double *tflops)
{
  if (!u || !x) return QESMC_ERR_ARG;
  if (!(u->tscale > 0.f)) return QESMC_ERR_STATE;
  UCHK(hipSetDevice(u->device));
  UCHK(hipStreamSynchronize(x->stream));
  const auto t0 = std::chrono::steady_clock::now();
  int rc = problem_features(u, x);
  if (rc != QESMC_OK) return rc;
  hipStream_t s = u->stream;
  UCHK(hipEventRecord(u->ev[0], s));
  UCHK(forward(u, u->feat));
  UCHK(hipEventRecord(u->ev[1], s));
  hipLaunchKernelGGL(k_install, g1(x->ncell), dim3(256), 0, s, x->d, u->out, u->sc, u->tscale, u->dx, u->dy,
                     x->d_lam);
  UCHK(hipGetLastError());
  UCHK(hipStreamSynchronize(s));
  const double wall = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  float t = 0.f;
  (void)hipEventElapsedTime(&t, u->ev[0], u->ev[1]);
  if (ms) *ms = wall;
  if (tflops) *tflops = t > 0.f ? u->conv_flops / (t * 1e-3) / 1e12 : 0.0;
  return QESMC_OK;
}

}  // extern "C"
