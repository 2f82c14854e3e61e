// Over-relaxation factor for time to tolerance: an estimate of the Jacobi
// spectral radius of the resident problem and the SOR factor it implies.
//
// Red-black SOR (a consistently ordered iteration) converges fastest at
// omega_opt = 2 / (1 + sqrt(1 - rho_J^2)), rho_J the spectral radius of the
// Jacobi iteration matrix D^-1 C (Young's theorem).  The reference runs at a
// fixed omega = 1.78 (Solver.h:83), which on large domains is far from it:
// with rho_J close to 1 the slowest, domain-scale modes then decay thousands
// of times slower per iteration.  No counterpart in the reference.
//
// The operator.  The cells the sweep relaxes that are fluid (flag not 0 or 2)
// form the active set; everything else holds lambda fixed (the Dirichlet ring
// and top) or is a building cell, which no fluid cell reads (its coefficient
// toward a solid is zero, Wall.cpp:288-340).  On the active set C couples a
// cell to its six neighbours with e..n and, at k = 1, to its own mirror
// image (lambda(i,j,0) = lambda(i,j,1), Solver_CPU_RB.cpp:154-162): a
// diagonal term n.  Weighted by W = dz_k, W C is symmetric (dz_k m_k =
// 2 / (dz_k + dz_k+1) = dz_k+1 n_k+1; the horizontal coefficients are equal
// pairwise among fluid cells), so M = (D W)^-1/2 (W C) (D W)^-1/2 is a
// symmetric matrix similar to D^-1 C, and rho_J = lambda_max(M) (the largest
// eigenvalue; C is non-negative).
//
// The estimate.  Lanczos on M in FP64 from a smooth start (the product of
// the lowest Dirichlet modes in x and y and a vertical half cosine, which is
// close to the dominant eigenvector, so few steps resolve it), dot products
// reduced per work-group and the partials summed in a fixed order, then the
// largest eigenvalue of the tridiagonal Lanczos matrix by bisection on its
// Sturm sequence.  The Ritz value never exceeds lambda_max.
#include <cmath>
#include <utility>
#include <vector>

#include "qesmc_internal.h"

namespace {

using qesmc::Dims;

#define OCHK(expr)                                         \
  do {                                                     \
    hipError_t _e = (expr);                                \
    if (_e != hipSuccess) return qesmc::map_hip_error(_e); \
  } while (0)

constexpr int kDotBlocks = 2048;  // a multiple of kXcds
constexpr int kXcds = 8;

__device__ inline bool active_cell(const Dims &d, int i, int j, int k, int flag)
{
  return i >= 1 && i <= d.NX - 2 && j >= 1 && j <= d.NY - 2 && k >= 1 && k <= d.NZ - 2 && flag != 0 && flag != 2;
}

// The iteration runs in the coordinates y = S^-1 v, S = (D W)^1/2, so that the
// operator needs no square root or division per neighbour: with
// q = W C y, M v = S^-1 q, v.(M v) = q.y and |M v|^2 = q.z for z = q / (D W)
// = S^-1 (M v), and the Lanczos recurrence on v is the same recurrence on y
// (divided through by S).

__device__ __forceinline__ double smooth_start(const Dims &d, int i, int j, int k)
{
  const double pi = 3.14159265358979323846;
  return sin(pi * i / (d.NX - 1)) * sin(pi * j / (d.NY - 1)) * cos(0.5 * pi * (k - 0.5) / (d.NZ - 1.5));
}

constexpr unsigned kInactive = 0x80u, kOpen = 63u;

// y[c] = the smooth start on active cells (the lowest Jacobi mode's shape,
// which in these coordinates is the dominant eigenvector's direction), 0
// elsewhere; yp = z = 0; partial[b] = this block's sum of |v|^2 = y^2 D W.
// Without an encoding of the coefficients inv[c] = 1 / (D_c W_c) on active
// cells and 0 elsewhere; with one (MASKED: split layout, cell (i,j,k) at
// half-index i/2 of row (j,k) of colour (i+j+k)&1) act[c] is the wall mask of
// an active cell and kInactive elsewhere, and layer[8 k ..] = e .. n, dz and
// 1 / (D W) of a cell without walls.
template <bool MASKED>
__global__ __launch_bounds__(256) void k_omega_init(Dims d, const float *__restrict__ e, const float *__restrict__ f,
                                                    const float *__restrict__ g, const float *__restrict__ h,
                                                    const float *__restrict__ m, const float *__restrict__ n,
                                                    const unsigned char *__restrict__ mask0,
                                                    const unsigned char *__restrict__ mask1,
                                                    const unsigned *__restrict__ canon, const int *__restrict__ flag,
                                                    const float *__restrict__ dz, double *__restrict__ inv,
                                                    unsigned char *__restrict__ act, double *__restrict__ layer,
                                                    double *__restrict__ y, double *__restrict__ yp,
                                                    double *__restrict__ z, double *__restrict__ partial)
{
  const long long total = (long long)d.NX * d.NY * d.NZ;
  const long long stride = (long long)gridDim.x * blockDim.x;
  double acc = 0.0;
  for (long long c = blockIdx.x * 256LL + threadIdx.x; c < total; c += stride) {
    const long long row = c / d.NX;
    const int k = (int)(row / d.NY), j = (int)(row - (long long)k * d.NY), i = (int)(c - row * d.NX);
    const bool on = active_cell(d, i, j, k, flag[c]);
    double ic = 0.0, v = 0.0;
    unsigned mk = kInactive;
    if (on) {
      double D;
      if (MASKED) {
        const long long x = row * d.HP + (i >> 1);
        mk = ((i + j + k) & 1) ? mask1[x] : mask0[x];
        D = 0.0;
        for (int a = 0; a < 6; ++a) D += ((mk >> a) & 1u) ? (double)__uint_as_float(canon[a * d.NZ + k]) : 0.0;
      } else {
        D = (double)e[c] + f[c] + g[c] + h[c] + m[c] + n[c];
      }
      ic = 1.0 / (D * (double)dz[k]);
      v = smooth_start(d, i, j, k);
      acc += v * v / ic;
    }
    if (MASKED)
      act[c] = (unsigned char)mk;
    else
      inv[c] = ic;
    y[c] = v;
    yp[c] = 0.0;
    if (!MASKED) z[c] = 0.0;
    if (MASKED && c < d.NZ) {
      double D = 0.0, *l = layer + 8 * c;
      for (int a = 0; a < 6; ++a) {
        l[a] = (double)__uint_as_float(canon[a * d.NZ + c]);
        D += l[a];
      }
      l[6] = (double)dz[c];
      l[7] = 1.0 / (D * l[6]);
    }
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// partial[b], partial[gridDim.x + b] = the work-group's sums
__device__ __forceinline__ void omega_partials(double acc, double acc2, double *__restrict__ partial)
{
  for (int off = 32; off > 0; off >>= 1) {
    acc += __shfl_xor(acc, off, 64);
    acc2 += __shfl_xor(acc2, off, 64);
  }
  __shared__ double red[2][4];
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = acc;
    red[1][threadIdx.x >> 6] = acc2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    partial[gridDim.x + blockIdx.x] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  }
}

// The step's Lanczos coefficients from the partial sums, summed in a fixed
// order by one work-group: hist[2 it] = alpha = w.v, hist[2 it + 1] = beta' =
// sqrt(|w|^2 - alpha^2 - beta^2) (v, u orthonormal, u.w = beta, the previous
// beta'), or 0 when that is not positive (the Krylov space is exhausted; the
// host stops there).  A launch of its own, 5 us: a last work-group that adds
// up in the kernel before needs a fence from each, which took 50 us.
__global__ __launch_bounds__(256) void k_omega_scalars(const double *__restrict__ partial, int count, int it,
                                                       double *__restrict__ hist)
{
  __shared__ double red[2][256];
  double s0 = 0.0, s1 = 0.0;
  for (int q = threadIdx.x; q < count; q += 256) {
    s0 += partial[q];
    s1 += partial[count + q];
  }
  red[0][threadIdx.x] = s0;
  red[1][threadIdx.x] = s1;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      red[0][threadIdx.x] += red[0][threadIdx.x + h];
      red[1][threadIdx.x] += red[1][threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double alpha = red[0][0];
    const double beta = it > 0 ? hist[2 * it - 1] : 0.0;
    const double b2 = red[1][0] - alpha * alpha - beta * beta;
    hist[2 * it] = alpha;
    hist[2 * it + 1] = b2 > 0.0 ? sqrt(b2) : 0.0;
  }
}

// One half of a Lanczos step on a mask-encoded geometry.  NEXT = false: the
// sums of v.(M v) and |M v|^2 of the present vector y, with z = S^-1 M S y of
// each cell used and dropped; NEXT = true: z again, and the next vector
// (z - alpha y - beta yp) / beta' over yp (the host then exchanges the two).
// Recomputing z costs a second read of y where keeping it costs a write and a
// read, and the coefficients come from a byte per cell (the wall mask of an
// active cell, kInactive elsewhere) and the layer's values, which give the
// resident coefficients bit for bit: 34 bytes per cell and step instead of 57, and
// two vectors, which stay in the 256 MB cache where four did not.
//
// A wave marches along k through kc planes of 64 cells of one row j with the
// next plane's loads in flight (its values above and below pass through
// registers); the four waves of a work-group take neighbouring rows, and each
// XCD a contiguous range of work-groups (they go to the XCDs in turn), so that
// neighbouring rows come from its own L2.
//
// At 256x256x96 a step takes 21 + 5 + 29 us (sums, scalars, next vector) and took
// 36 + 5 + 29 with z and 1 / (D W) kept; the next vector moves 160 MB at 5.5 TB/s.
// Tried and not faster: two or three planes in flight (fewer waves fit), the
// x neighbours by a shift across lanes, the wave's planes dealt over the XCDs.
constexpr int kStepMin = 8, kStepMax = 32;  // planes per wave
struct StepGrid {
  int kc, jgroups, nseg, chunks;
  long long blocks;  // a multiple of kXcds
};

inline StepGrid step_grid(const Dims &d)
{
  StepGrid g{kStepMin, (d.NY - 2 + 3) / 4, (d.NX - 2 + 63) / 64, 0, 0};
  // 8 waves per SIMD where there are as many
  const long long columns = (long long)(d.NY - 2) * g.nseg, planes = d.NZ - 2;
  while (g.kc < kStepMax && columns * planes > 8192LL * g.kc) ++g.kc;
  g.chunks = (int)((planes + g.kc - 1) / g.kc);
  g.blocks = ((long long)g.jgroups * g.nseg * g.chunks + kXcds - 1) / kXcds * kXcds;
  return g;
}

template <bool NEXT>
__global__ __launch_bounds__(256) void k_omega_step(Dims d, StepGrid sg, const unsigned char *__restrict__ act,
                                                    const double *__restrict__ layer,
                                                    const double *__restrict__ y, double *__restrict__ yp, int it,
                                                    double *__restrict__ partial, const double *__restrict__ hist)
{
  double alpha = 0.0, beta = 0.0, inb = 0.0;
  if (NEXT) {
    const double nb = hist[2 * it + 1];
    if (!(nb > 0.0)) return;
    alpha = hist[2 * it];
    beta = it > 0 ? hist[2 * it - 1] : 0.0;
    inb = 1.0 / nb;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned tile = blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  const unsigned col = tile / (unsigned)sg.jgroups, chunk = col / (unsigned)sg.nseg;
  const int j = 1 + 4 * (int)(tile - col * sg.jgroups) + wave, i0 = 1 + 64 * (int)(col - chunk * sg.nseg) + lane;
  const int k0 = 1 + sg.kc * (int)chunk;
  const int k1 = k0 + sg.kc < d.NZ - 1 ? k0 + sg.kc : d.NZ - 1;
  double acc = 0.0, acc2 = 0.0;
  if (j <= d.NY - 2 && k0 < k1) {
    const bool in = i0 <= d.NX - 2;
    const int i = in ? i0 : d.NX - 2;  // the lanes beyond the row do the last cell's work and drop it
    long long c = ((long long)k0 * d.NY + j) * d.NX + i;
    struct Plane {
      double up, e, w, n, s, yp;
      unsigned mk;
    };
    auto load = [&](long long q) {  // q in planes 1 .. NZ - 2
      Plane p;
      p.mk = act[q];
      p.up = y[q + d.sz];
      p.e = y[q + 1];
      p.w = y[q - 1];
      p.n = y[q + d.sy];
      p.s = y[q - d.sy];
      p.yp = NEXT ? yp[q] : 0.0;
      return p;
    };
    double below = y[c - d.sz], yc = y[c];
    auto step = [&](const Plane &p, int k) {
      const double *__restrict__ l = layer + 8 * (long long)k;
      double cf[6], ic = l[7];
      const double dzk = l[6];
#pragma unroll
      for (int a = 0; a < 6; ++a) cf[a] = l[a];
      if (p.mk < kOpen) {
#pragma unroll
        for (int a = 0; a < 6; ++a) cf[a] = ((p.mk >> a) & 1u) ? cf[a] : 0.0;
        ic = 1.0 / ((cf[0] + cf[1] + cf[2] + cf[3] + cf[4] + cf[5]) * dzk);
      }
      // y is 0 off the active set, so those neighbours drop out by themselves
      double cy = cf[0] * p.e + cf[1] * p.w + cf[2] * p.n + cf[3] * p.s + cf[4] * p.up;
      cy += cf[5] * (k == 1 ? yc : below);  // the k = 0 mirror
      const double w = dzk * cy, zc = w * ic;
      if (in && p.mk != kInactive) {
        if (NEXT) {
          yp[c] = (zc - alpha * yc - beta * p.yp) * inb;
        } else {
          acc += w * yc;
          acc2 += w * zc;
        }
      }
      below = yc;
      yc = p.up;
      c += d.sz;
    };
    // two planes by name, so that no register is copied while its load is in flight
    Plane p0 = load(c), p1;
    for (int k = k0; k < k1; k += 2) {
      p1 = load(k + 1 < k1 ? c + d.sz : c);
      step(p0, k);
      if (k + 1 == k1) break;
      p0 = load(k + 2 < k1 ? c + d.sz : c);
      step(p1, k + 1);
    }
  }
  if (!NEXT) omega_partials(acc, acc2, partial);
}

// z = S^-1 M S y on active cells and the step's coefficients, for coefficients
// without an encoding, where reading them twice would cost more than keeping z.
// Work-groups take the interior rows (j, k) in turn and their threads the
// row's interior cells; every other cell of z is left as it is (0: the
// buffers start at 0 off the active set and the recurrence keeps them there).
__global__ __launch_bounds__(256) void k_omega_apply(Dims d, const float *__restrict__ e, const float *__restrict__ f,
                                                     const float *__restrict__ g, const float *__restrict__ h,
                                                     const float *__restrict__ m, const float *__restrict__ n,
                                                     const float *__restrict__ dz, const double *__restrict__ inv,
                                                     const double *__restrict__ y, double *__restrict__ z,
                                                     double *__restrict__ partial)
{
  const int ny = d.NY - 2, rows = ny > 0 && d.NZ > 2 ? ny * (d.NZ - 2) : 0;
  // the rows split into one contiguous range per XCD (work-groups go to the
  // XCDs in turn), so the neighbouring rows a work-group reads are in its
  // own XCD's L2
  const int xcd = (int)blockIdx.x % kXcds, per = (int)gridDim.x / kXcds;
  const int span = (rows + kXcds - 1) / kXcds, r0 = xcd * span, r1 = min(rows, r0 + span);
  double acc = 0.0, acc2 = 0.0;
  for (int r = r0 + (int)blockIdx.x / kXcds; r < r1; r += per) {
    const int k = 1 + r / ny, j = 1 + r % ny;
    const long long row = (long long)k * d.NY + j;
    const double dzk = (double)dz[k];
    for (int i = 1 + (int)threadIdx.x; i <= d.NX - 2; i += 256) {
      const long long c = row * d.NX + i;
      const double ic = inv[c];
      if (ic == 0.0) continue;
      const double cf[6] = {e[c], f[c], g[c], h[c], m[c], n[c]};
      // y is 0 off the active set, so those neighbours drop out by themselves
      const double yc = y[c];
      double cy =
          cf[0] * y[c + 1] + cf[1] * y[c - 1] + cf[2] * y[c + d.sy] + cf[3] * y[c - d.sy] + cf[4] * y[c + d.sz];
      cy += cf[5] * ((k == 1) ? yc : y[c - d.sz]);  // the k = 0 mirror
      const double q = dzk * cy;
      const double zc = q * ic;
      z[c] = zc;
      acc += q * yc;
      acc2 += q * zc;
    }
  }
  omega_partials(acc, acc2, partial);
}

// The next Lanczos vector, written over z: z <- (z - alpha y - beta yp) /
// beta' (the host then rotates yp <- y, y <- z), with the coefficients of
// step `it` from hist (nothing when beta' is 0).  Two cells per thread; the
// thread after the last pair takes an odd count's last cell.
__global__ __launch_bounds__(256) void k_omega_next(long long total, int it, const double *__restrict__ hist,
                                                    const double *__restrict__ yp, const double *__restrict__ y,
                                                    double *__restrict__ z)
{
  const double alpha = hist[2 * it], beta = it > 0 ? hist[2 * it - 1] : 0.0, nb = hist[2 * it + 1];
  if (!(nb > 0.0)) return;
  const double inb = 1.0 / nb;
  const long long t = blockIdx.x * 256LL + threadIdx.x, pairs = total / 2;
  if (t < pairs) {
    const double2 a = reinterpret_cast<const double2 *>(z)[t], b = reinterpret_cast<const double2 *>(y)[t],
                  c = reinterpret_cast<const double2 *>(yp)[t];
    reinterpret_cast<double2 *>(z)[t] =
        make_double2((a.x - alpha * b.x - beta * c.x) * inb, (a.y - alpha * b.y - beta * c.y) * inb);
  } else if (t == pairs && (total & 1)) {
    z[total - 1] = (z[total - 1] - alpha * y[total - 1] - beta * yp[total - 1]) * inb;
  }
}

// v *= inv.
__global__ __launch_bounds__(256) void k_omega_scale(long long total, double inv, double *__restrict__ v)
{
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long c = blockIdx.x * 256LL + threadIdx.x; c < total; c += stride) v[c] *= inv;
}

struct Buf {
  void *p = nullptr;
  ~Buf()
  {
    if (p) (void)hipFree(p);
  }
};

// Number of eigenvalues of the symmetric tridiagonal (a, b) below x (Sturm).
int sturm_below(const std::vector<double> &a, const std::vector<double> &b, double x)
{
  int count = 0;
  double q = 1.0;
  for (size_t i = 0; i < a.size(); ++i) {
    const double bb = i ? b[i - 1] * b[i - 1] : 0.0;
    q = (a[i] - x) - (i ? bb / q : 0.0);
    if (q == 0.0) q = -1e-300;
    if (q < 0.0) ++count;
  }
  return count;
}

// Largest eigenvalue of the symmetric tridiagonal (a, b) by bisection.
double tridiag_max_eig(const std::vector<double> &a, const std::vector<double> &b)
{
  double lo = 1e300, hi = -1e300;
  for (size_t i = 0; i < a.size(); ++i) {  // Gershgorin bounds
    const double r = (i ? std::fabs(b[i - 1]) : 0.0) + (i + 1 < a.size() ? std::fabs(b[i]) : 0.0);
    lo = std::fmin(lo, a[i] - r);
    hi = std::fmax(hi, a[i] + r);
  }
  const int n = (int)a.size();
  for (int it = 0; it < 200 && hi - lo > 1e-15 * std::fmax(1.0, std::fabs(hi)); ++it) {
    const double mid = 0.5 * (lo + hi);
    if (sturm_below(a, b, mid) < n) lo = mid;  // some eigenvalue is above mid
    else hi = mid;
  }
  return 0.5 * (lo + hi);
}

}  // namespace

extern "C" {

int qesmc_estimate_omega(qesmc_ctx *x, int steps, double *rho, float *omega)
{
  if (!x || steps < 1 || steps > 100000 || (!rho && !omega)) return QESMC_ERR_ARG;
  if (!x->have_geom) return QESMC_ERR_STATE;
  OCHK(hipSetDevice(x->device));
  const Dims &d = x->d;
  const long long total = x->ncell;
  hipStream_t st = x->stream;
  // the wall-mask encoding built when the geometry was committed, when the
  // coefficients have one
  const bool masked = x->compressible;
  // One allocation: the partial sums, the coefficients of all steps,
  // the layers; y and the previous vector yp, and either the masks or
  // z and inv = 1 / (D W).
  auto lines = [](size_t k) { return (k + 15) / 16 * 16; };  // whole cache lines of doubles
  const StepGrid sg = step_grid(d);
  const int parts = masked && sg.blocks > kDotBlocks ? (int)sg.blocks : kDotBlocks;
  const size_t n = lines((size_t)total), head = lines(2 * (size_t)parts + 2 * (size_t)steps + 8 * (size_t)d.NZ);
  Buf mem;
  OCHK(hipMalloc(&mem.p, sizeof(double) * (head + 2 * n) + (masked ? n : 2 * sizeof(double) * n)));
  double *part = (double *)mem.p, *hist = part + 2 * (size_t)parts, *layer = hist + 2 * (size_t)steps,
         *y = part + head, *yp = y + n, *z = yp + n, *inv = z + n;
  unsigned char *act = (unsigned char *)z;
  const dim3 grid(kDotBlocks), block(256), next_grid((unsigned)((total / 2 + 256) / 256));
  float *const *cf = x->d_coef;
  if (masked)
    hipLaunchKernelGGL(k_omega_init<true>, grid, block, 0, st, d, cf[0], cf[1], cf[2], cf[3], cf[4], cf[5],
                       x->d_mask[0], x->d_mask[1], x->d_canon, x->d_flag, x->d_dz, nullptr, act, layer, y, yp,
                       nullptr, part);
  else
    hipLaunchKernelGGL(k_omega_init<false>, grid, block, 0, st, d, cf[0], cf[1], cf[2], cf[3], cf[4], cf[5], nullptr,
                       nullptr, nullptr, x->d_flag, x->d_dz, inv, nullptr, nullptr, y, yp, z, part);
  OCHK(hipGetLastError());
  // |v|^2 summed on the host in a fixed order, so the estimate is deterministic
  std::vector<double> hp(kDotBlocks);
  OCHK(hipMemcpyAsync(hp.data(), part, sizeof(double) * kDotBlocks, hipMemcpyDeviceToHost, st));
  OCHK(hipStreamSynchronize(st));
  double nrm2 = 0.0;
  for (double v : hp) nrm2 += v;
  if (!(nrm2 > 0.0)) return QESMC_ERR_UNSUPPORTED;  // no active cell
  hipLaunchKernelGGL(k_omega_scale, grid, block, 0, st, total, 1.0 / std::sqrt(nrm2), y);
  OCHK(hipGetLastError());
  // Lanczos with one reduction per step: w = M v gives alpha = w.v and
  // |w|^2 together, the next beta from |w - alpha v - beta u|^2 =
  // |w|^2 - alpha^2 - beta^2.  The coefficients stay on the device; the host
  // reads them every 10 steps to test the largest Ritz value for
  // convergence.
  std::vector<double> hh(2 * (size_t)steps);
  double last = -1.0, r = 0.0;
  for (int it = 0; it < steps; ++it) {
    if (masked)
      hipLaunchKernelGGL(k_omega_step<false>, dim3((unsigned)sg.blocks), block, 0, st, d, sg, (const unsigned char *)act, (const double *)layer,
                         (const double *)y, yp, it, part, (const double *)hist);
    else
      hipLaunchKernelGGL(k_omega_apply, grid, block, 0, st, d, cf[0], cf[1], cf[2], cf[3], cf[4], cf[5], x->d_dz,
                         (const double *)inv, (const double *)y, z, part);
    hipLaunchKernelGGL(k_omega_scalars, dim3(1), block, 0, st, (const double *)part, masked ? (int)sg.blocks : kDotBlocks, it, hist);
    if (masked) {
      hipLaunchKernelGGL(k_omega_step<true>, dim3((unsigned)sg.blocks), block, 0, st, d, sg, (const unsigned char *)act, (const double *)layer,
                         (const double *)y, yp, it, part, (const double *)hist);
      std::swap(y, yp);
    } else {
      hipLaunchKernelGGL(k_omega_next, next_grid, block, 0, st, total, it, (const double *)hist, (const double *)yp,
                         (const double *)y, z);
      double *const old = yp;
      yp = y;
      y = z;
      z = old;
    }
    OCHK(hipGetLastError());
    if ((it + 1) % 10 != 0 && it + 1 != steps) continue;
    OCHK(hipMemcpyAsync(hh.data(), hist, sizeof(double) * 2 * (size_t)(it + 1), hipMemcpyDeviceToHost, st));
    OCHK(hipStreamSynchronize(st));
    // the tridiagonal Lanczos matrix up to the first exhausted step
    std::vector<double> a, b;
    bool done = false;
    for (int q = 0; q <= it; ++q) {
      a.push_back(hh[2 * (size_t)q]);
      if (!(hh[2 * (size_t)q + 1] > 0.0)) {
        done = true;
        break;
      }
      if (q < it) b.push_back(hh[2 * (size_t)q + 1]);
    }
    r = tridiag_max_eig(a, b);
    if (done || std::fabs(r - last) <= 1e-12 || it + 1 == steps) break;
    last = r;
  }
  if (rho) *rho = r;
  if (omega) {
    // Young's optimum, moved back from 2 by a fifth of its distance: past the
    // optimum the slowest modes oscillate at omega - 1 and fp32 rounding noise
    // is amplified, so a small margin costs little and keeps clear of both
    // (measured on 128x128x64 cities: 1.95 fastest, 1.97 slower; on the
    // 1000x1000x150 city 1.99 reached 1e-4 m/s, 1.995 did not)
    const double rr = r < 1.0 ? r : 1.0;
    const double opt = 2.0 / (1.0 + std::sqrt(1.0 - rr * rr));
    *omega = (float)(2.0 - 1.2 * (2.0 - opt));
  }
  return QESMC_OK;
}

}  // extern "C"
