// Red-black SOR with whole iterations in one launch: T iterations (2 T colour
// passes) of a column tile are pipelined along k, on the pair layout with the
// wall-mask stencil (QESMC_PATH_FUSED, and what QESMC_PATH_AUTO runs on a
// wall-mask geometry).
//
// Layout.  The pair layout stores row (j,k) as HP pairs, pair q holding the
// cells i = 2q and 2q+1: x = (k*NY + j)*HP + q, one 8-byte pair of lambda
// and of R and one 2-byte pair of wall masks per index.  A pair holds one red
// and one black cell; which is which alternates with j + k.
//
// A launch reads lambda from one buffer set and writes the other, so no
// work-group reads what another writes.  The result is the reference's
// in-place schedule (src/winds/Solver_CPU_RB.cpp:109-162) exactly: every
// half-sweep sees the other colour as the schedule leaves it, and after each
// iteration lambda(i,j,0) = lambda(i,j,1).
//
// Work decomposition.  A work-group of NW waves owns a tile of 64 half-cells
// (one per lane) by NW*RW rows (RW rows per wave) and a segment of planes, and
// marches up k.  Step p relaxes, for h = 0 .. 2T-1, half-sweep h (red for
// even h) of plane p-h: its z-neighbours are half-sweep h-1's planes p-h+1 (just
// relaxed) and p-h-1, its y-neighbours half-sweep h-1's values of plane p-h,
// relaxed one step earlier, so the rows at the edge of a wave's block are
// exchanged through LDS once per step (one barrier), and the x-neighbour
// outside the pair comes from the adjacent lane (DPP).  Everything else stays
// in registers: a window of planes per row in which each half-sweep replaces
// its colour in place.  The window is a ring whose slots are static because
// the step loop is unrolled over the ring, which also makes every parity
// (j+k) static: tiles start on even rows and segments on odd planes.
// The tiles overlap by a halo that is relaxed redundantly: 2T rows and T
// half-cells on each inner side, 2T planes at each inner segment end.
//
// Per launch a cell moves 4 (lambda) + 4 (R) + 1 (mask) bytes in and 4 out plus
// the halo's re-reads, for T iterations: at T = 2 half of what one iteration
// per launch moves.  omega / (e+f+g+h+m+n) depends only on the layer and
// the 6-bit mask and is tabulated per plane in LDS with the same expression
// (one wave per half-sweep, one mask per lane), and where all masks of a wave's
// rows are open (no wall: most of a city's planes) the six coefficients are
// the layer's wall values themselves, in scalar registers.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "qesmc_march.h"

hipError_t qesmc_launch_fill_u32(qesmc_ctx *x, unsigned *p, long long count, unsigned v);

namespace qesmc {

namespace {

constexpr int kXcds = 8;  // MI355X: 8 XCDs, work-groups dispatched round-robin
constexpr int kMaxSegments = kMarchMaxSegments;
constexpr unsigned kOpenRows = 0xfcfcfcfcu;  // the pairs of two rows without walls

__device__ inline float wave_max(float v)
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// The value of the lane below (FROM = -1) or above (FROM = 1); 0 past the wave's ends.
template <int FROM>
__device__ __forceinline__ float lane_shift(float v)
{
  constexpr int ctrl = FROM < 0 ? 0x138 : 0x130;  // wave_shr:1 / wave_shl:1
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true));
}

// m = max(m, |v|); a NaN never wins, as in the reference's max test.  (fmaxf
// would first canonicalise m, which is never a signalling NaN.)
__device__ __forceinline__ void max_abs(float &m, float v) { asm("v_max_f32 %0, %0, |%1|" : "+v"(m) : "v"(v)); }

// LDS writes of this wave visible to the work-group before the barrier, LDS
// reads after it; global loads and stores in flight are left in flight.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Bit `bit` of a mask word, sign-extended, and the byte from `bit` up (a mask
// times 4: the byte offset of its table entry).
// Written out because the compiler would keep every bit of a mask as a
// condition (a scalar register pair each) or an extended word from one
// half-sweep to the next of the same cell, and spill.
__device__ __forceinline__ unsigned mask_bit(unsigned m, unsigned bit)
{
  unsigned r;
  asm volatile("v_bfe_i32 %0, %1, %2, 1" : "=v"(r) : "v"(m), "n"(bit));
  return r;
}

__device__ __forceinline__ unsigned mask_index(unsigned m, unsigned bit)
{
  unsigned r;
  asm volatile("v_bfe_u32 %0, %1, %2, 8" : "=v"(r) : "v"(m), "n"(bit));
  __builtin_assume(r < 256u);
  return r;
}

// Buffer descriptor over `bytes` bytes at a wave-uniform address: a load or
// store then takes one lane offset and one scalar offset, and what falls past
// the end reads 0 or is dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *p, unsigned bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00027000);
}

typedef unsigned uint2v __attribute__((ext_vector_type(2)));

}  // namespace

// T iterations per launch, NW waves per work-group, RW rows (even) per row
// group, GW lanes per row group (64: a wave is one group; 32: two).
// BATCH: the work-group's problem is taken from A.items (A.which per
// work-group) instead of I.
template <int T, int NW, int RW, int GW, bool BATCH>
__global__ __launch_bounds__(64 * NW, RW == 2 ? 4 : 2) void k_sor_march(MarchItem I, MarchRun A)
{
  constexpr int H = 2 * T;      // half-sweeps
  constexpr int U = 2 * T + 4;  // ring slots (planes p-2T .. p+2 are live); even
  constexpr int NG = NW * (64 / GW);  // row groups
  constexpr int YR = NG * RW;   // rows of the tile
  static_assert(RW % 2 == 0 && NW >= H && (T == 1 || T == 2), "");
  // edge rows of each row group, per half-sweep that reads them: [buffer][h][first / last row][row group and lane]
  __shared__ float edge[2][H][2][NW * 64];
  __shared__ float wd_tab[2][H][64];
  __shared__ __align__(16) unsigned cv_tab[2][H][8];
  __shared__ float wmax[NW][T];
  const int problem = BATCH ? A.which[blockIdx.x] : 0;
  const MarchItem *const ip = BATCH ? A.items + problem : nullptr;
#define QESMC_ITEM(f) (BATCH ? ip->f : I.f)
#define QESMC_ITEM_PTR(f) (BATCH ? (decltype(I.f))as_global(ip->f) : I.f)
  const Dims d = QESMC_ITEM(d);
  unsigned *const err = QESMC_ITEM_PTR(err), *const status = QESMC_ITEM_PTR(status), *const cur = QESMC_ITEM_PTR(cur);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int t = A.t, src = A.src;
  float om[H];
#pragma unroll
  for (int h = 0; h < H; ++h) om[h] = A.om[h];
  if (T == 1 && A.fix) {
    // the last launch ran T iterations but the run ended inside it
    if (!status[kFixGo]) return;
    t = (int)status[kLastT];
    src = (int)(cur[0] ^ 1u);
    om[0] = __uint_as_float(status[kLastOmega]);
    om[1] = __uint_as_float(status[kLastOmega + 1]);
  } else {
    if (t >= A.itermax) return;
  }
  // Each XCD (work-group id % 8) takes a contiguous eighth of the problem's
  // tile range, tiles numbered x fastest, then y, then segment: neighbours that
  // share halos march together on one L2.  Problems follow each other without
  // gaps, so that those of a tile or two go to the XCDs in turn.  With the first
  // work-group of each a multiple of 8 all of them went to one: 512 domains of
  // 10 cells a side 52 us per iteration against 12 (colour passes 16), 256 of
  // 32 cells a side 62 against 35 (colour passes 54).
  const int slot = (int)blockIdx.x - QESMC_ITEM(first), ntiles = QESMC_ITEM(ntiles);
  if (slot >= ntiles) return;
  const int xcd = slot % kXcds, more = ntiles % kXcds;  // the first `more` XCDs have one tile more
  const int tile = xcd * (ntiles / kXcds) + (xcd < more ? xcd : more) + slot / kXcds;
  const int nq = QESMC_ITEM(nq), nyt = QESMC_ITEM(nyt);
  const int tq = tile % nq;
  const int ty = (tile / nq) % nyt;
  const int tz = tile / (nq * nyt);

  // columns: this lane's half-cell, and whether this tile owns it
  const int half = (d.NX + 1) >> 1;
  const int gl = lane & (GW - 1);
  const int q = tq * (GW - 2 * T) + gl;
  const bool lown = q < half && (tq == 0 || gl >= T) && (tq == nq - 1 || gl < GW - T);
  const unsigned qc = (unsigned)(q < half ? q : half - 1);
  const bool col[2] = {q < half && 2 * q >= 1 && 2 * q <= d.NX - 2, 2 * q + 1 <= d.NX - 2};
  // rows of this lane's group
  const int group = (int)threadIdx.x / GW;
  const int jt = ty * (YR - 4 * T);
  const int j0 = jt + group * RW;
  const int jown0 = ty == 0 ? 0 : jt + 2 * T;
  const int jown1 = ty == nyt - 1 ? d.NY : jt + YR - 2 * T;
  bool upd[RW][2], own[RW];
  unsigned voff[RW], moff[RW / 2];  // byte offsets within a plane of lambda and R, of masks
#pragma unroll
  for (int a = 0; a < RW; ++a) {
    const int j = j0 + a;
    const unsigned jc = (unsigned)(j < d.NY ? j : d.NY - 1);
    const bool ru = j >= 1 && j <= d.NY - 2;
    upd[a][0] = ru && col[0];
    upd[a][1] = ru && col[1];
    own[a] = lown && j >= jown0 && j < jown1;
    voff[a] = (jc * (unsigned)d.HP + qc) * 8u;
    if (a % 2 == 0) moff[a / 2] = ((jc / 2u) * (unsigned)d.HP + qc) * 4u;
  }
  // planes: owned [ka, kb); half-sweep h relaxes [lo(h), hi(h)]
  const int ka = QESMC_ITEM(begin[tz]), kb = QESMC_ITEM(begin[tz + 1]);
  const int pfirst = ka - (H - 1) > 0 ? ka - (H - 1) : 0;  // even
  const int plast = kb - 1 + (H - 1);
  const float2 *__restrict__ in = src ? QESMC_ITEM_PTR(set1) : QESMC_ITEM_PTR(set0);
  float2 *__restrict__ out = src ? QESMC_ITEM_PTR(set0) : QESMC_ITEM_PTR(set1);
  const float2 *__restrict__ R = QESMC_ITEM_PTR(R);
  const unsigned *__restrict__ mask = QESMC_ITEM_PTR(mask);
  const unsigned *__restrict__ canon8 = QESMC_ITEM_PTR(canon8);
  const float *__restrict__ sums = QESMC_ITEM_PTR(sums);
  const unsigned plane8 = (unsigned)d.splane * 8u, planem = (unsigned)((d.NY + 1) / 2) * (unsigned)d.HP * 4u;
  // this wave's half-sweep of the tables
  float omw = om[0];
#pragma unroll
  for (int h = 1; h < H; ++h) omw = wave == h ? om[h] : omw;
  auto clampk = [&](int k) -> int { return k < 0 ? 0 : k > d.NZ - 1 ? d.NZ - 1 : k; };

  float W[RW][U][2];   // lambda
  float G[RW][U][2];   // R
  unsigned M[RW / 2][U];    // mask pairs of two rows
  float dm[T][RW];
  bool bad = false;
#pragma unroll
  for (int a = 0; a < RW; ++a)
#pragma unroll
    for (int s = 0; s < U; ++s) {
      W[a][s][0] = W[a][s][1] = G[a][s][0] = G[a][s][1] = 0.f;
      M[a / 2][s] = kOpenRows;
    }
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int a = 0; a < RW; ++a) dm[i][a] = 0.f;

  auto load_lambda = [&](int k, int slot) {
    const __amdgpu_buffer_rsrc_t pl =
        buffer_of(reinterpret_cast<const char *>(in) + (unsigned long long)clampk(k) * plane8, plane8);
#pragma unroll
    for (int a = 0; a < RW; ++a) {
      const uint2v v = __builtin_amdgcn_raw_buffer_load_b64(pl, voff[a], 0, 0);
      W[a][slot][0] = __uint_as_float(v.x);
      W[a][slot][1] = __uint_as_float(v.y);
    }
  };
  auto load_rhs = [&](int k, int slot) {
    const __amdgpu_buffer_rsrc_t pr =
        buffer_of(reinterpret_cast<const char *>(R) + (unsigned long long)clampk(k) * plane8, plane8);
#pragma unroll
    for (int a = 0; a < RW; ++a) {
      const uint2v v = __builtin_amdgcn_raw_buffer_load_b64(pr, voff[a], 0, 0);
      G[a][slot][0] = __uint_as_float(v.x);
      G[a][slot][1] = __uint_as_float(v.y);
    }
  };
  auto load_masks = [&](int k, int slot) {
    const __amdgpu_buffer_rsrc_t pm =
        buffer_of(reinterpret_cast<const char *>(mask) + (unsigned long long)clampk(k) * planem, planem);
#pragma unroll
    for (int a = 0; a < RW / 2; ++a) M[a][slot] = __builtin_amdgcn_raw_buffer_load_b32(pm, moff[a], 0, 0);
  };
  // the wall values of step p's planes and omega / (sum of those a mask
  // selects): wave h for half-sweep h, the sums and values loaded a step
  // ahead (a lane's mask is its number; lanes 0-7 hold the plane's values)
  float tab_sum = 1.f;
  unsigned tab_canon = 0u;
  auto load_tables = [&](int p) {
    if (wave < H) {
      const int k = clampk(p - wave);
      tab_sum = sums[64 * k + lane];
      tab_canon = canon8[8 * k + (lane & 7)];
    }
  };
  auto write_tables = [&](int buf) {
    if (wave < H) {
      wd_tab[buf][wave][lane] = omw / tab_sum;
      if (lane < 8) cv_tab[buf][wave][lane] = tab_canon;
    }
  };
  // the edge rows that step p's half-sweep h reads: plane p-h, the colour
  // it reads, at the component that row's reader needs
  auto write_edges = [&](int s, int buf) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int slot = (s - h + 2 * U) % U;
      const int ofirst = ((s - h + 2 * U) & 1) ^ (h & 1);  // own component of a row with even a
      // my last row is the row above the next group's first row (a = 0), my
      // first row the one below the previous group's last row (a = RW-1, odd)
      edge[buf][h][1][threadIdx.x] = W[RW - 1][slot][ofirst];
      edge[buf][h][0][threadIdx.x] = W[0][slot][ofirst ^ 1];
    }
  };

  load_lambda(pfirst - 1, U - 1);
  load_lambda(pfirst, 0);
  load_lambda(pfirst + 1, 1);
  load_rhs(pfirst, 0);
  load_masks(pfirst, 0);
  load_tables(pfirst);
  int wtop = 0;
  {
    const int nqb = (d.HP + 31) / 32;
    const int *__restrict__ top = QESMC_ITEM_PTR(top);
#pragma unroll
    for (int a = 0; a < RW; a += 2) wtop = max(wtop, top[(j0 + a < d.NY ? j0 + a : d.NY - 1) / 2 * nqb + (int)qc / 32]);
  }
  // the gate is read while those loads are in flight
  if (!(T == 1 && A.fix)) {
    if (!gate_pass_multi(err, t, A.tol, status, lane)) return;  // identical in every wave of the grid
    if (tile == 0 && threadIdx.x == 0) {
      *cur = (unsigned)(src ^ 1);
      status[kLastT] = (unsigned)t;
      status[kLastIters] = (unsigned)T;
      status[kLastOmega] = __float_as_uint(om[0]);
      status[kLastOmega + 1] = __float_as_uint(om[1]);
    }
  }
  // Buildings stand on the ground: below the highest wall of its columns a
  // wave takes every plane as masked, above it none.  (Plane 1's mirror is the
  // masked steps' business: the first ones of a segment at the ground are.)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) wtop = max(wtop, __shfl_xor(wtop, off, 64));
  wtop = __builtin_amdgcn_readfirstlane(wtop);
  write_tables(0);
  write_edges(0, 0);
  lds_barrier();

  // the same lane of the groups above and below
  const int tup = (int)threadIdx.x >= GW ? (int)threadIdx.x - GW : (int)threadIdx.x;
  const int tdn = (int)threadIdx.x < (NG - 1) * GW ? (int)threadIdx.x + GW : (int)threadIdx.x;
  // the steps p0 .. p0+U-1; OPEN: no wall in this wave's rows on the planes they relax
  auto block = [&](int p0, auto is_open) {
    constexpr bool OPEN = decltype(is_open)::value;
#pragma unroll
    for (int s = 0; s < U; ++s) {
      const int p = p0 + s;
      if (p > plast) break;
      const int buf = s & 1;
      load_lambda(p + 2, (s + 2) % U);
      load_rhs(p + 1, (s + 1) % U);
      if (!OPEN) load_masks(p + 1, (s + 1) % U);
      load_tables(p + 1);
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const int k = p - h;
        const int klo = ka - (H - 1 - h) > 1 ? ka - (H - 1 - h) : 1;
        const int khi = kb - 1 + (H - 1 - h) < d.NZ - 2 ? kb - 1 + (H - 1 - h) : d.NZ - 2;
        const bool in_range = k >= klo && k <= khi;  // uniform
        const int sk = (s - h + 2 * U) % U, sup = (sk + 1) % U, sdn = (sk + U - 1) % U;
        const float yabove = edge[buf][h][1][tup], ybelow = edge[buf][h][0][tdn];
        const float omo = 1.0f - om[h];
        const uint4 c03 = *reinterpret_cast<const uint4 *>(&cv_tab[buf][h][0]);
        const uint2 c45 = *reinterpret_cast<const uint2 *>(&cv_tab[buf][h][4]);
        const float wdo = OPEN ? wd_tab[buf][h][63] : 0.f;
#pragma unroll
        for (int a = 0; a < RW; ++a) {
          const int e = (a + s - h + 2 * U) & 1;  // (j + k) & 1
          const int o = e ^ (h & 1);              // the cell relaxed: i = 2q + o
          const float old = W[a][sk][o], xc = W[a][sk][o ^ 1];
          const float xm = o ? xc : lane_shift<-1>(xc);
          const float xp = o ? lane_shift<1>(xc) : xc;
          const float ym = a > 0 ? W[a > 0 ? a - 1 : 0][sk][o] : yabove;
          const float yp = a < RW - 1 ? W[a < RW - 1 ? a + 1 : a][sk][o] : ybelow;
          const float zp = W[a][sup][o], zm = W[a][sdn][o];
          const float r = G[a][sk][o];
          float ec, fc, gc, hc, mc, nc, wd;
          if (OPEN) {
            ec = __uint_as_float(c03.x);
            fc = __uint_as_float(c03.y);
            gc = __uint_as_float(c03.z);
            hc = __uint_as_float(c03.w);
            mc = __uint_as_float(c45.x);
            nc = __uint_as_float(c45.y);
            wd = wdo;
          } else {
            const unsigned m = M[a / 2][sk];
            const unsigned base = 16u * (a & 1) + 8u * o;
            auto coef = [&](unsigned bit, unsigned cb) { return __uint_as_float(cb & mask_bit(m, base + 2u + bit)); };
            ec = coef(0, c03.x);
            fc = coef(1, c03.y);
            gc = coef(2, c03.z);
            hc = coef(3, c03.w);
            mc = coef(4, c45.x);
            nc = coef(5, c45.y);
            wd = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(wd_tab[buf][h]) + mask_index(m, base));
          }
          const float nv = wd * (ec * xp + fc * xm + gc * yp + hc * ym + mc * zp + nc * zm - r) + omo * old;
          const float sel = (upd[a][o] & in_range) ? nv : old;
          W[a][sk][o] = sel;
          max_abs(dm[h >> 1][a], sel - old);
        }
      }
      // after an iteration lambda(i,j,0) = lambda(i,j,1): what the next
      // iteration of plane 1 reads (the first one reads plane 0 as stored)
      if (!OPEN && T > 1 && s == 2 && p == 2) {
#pragma unroll
        for (int a = 0; a < RW; ++a) {
          W[a][0][0] = W[a][1][0];
          W[a][0][1] = W[a][1][1];
        }
      }
      {
        const int k = p - (H - 1), sk = (s - (H - 1) + 2 * U) % U;
        if (k >= ka && k < kb) {
          const __amdgpu_buffer_rsrc_t pl =
              buffer_of(reinterpret_cast<char *>(out) + (unsigned long long)k * plane8, plane8);
#pragma unroll
          for (int a = 0; a < RW; ++a) {
            const float x0 = W[a][sk][0], x1 = W[a][sk][1];
            bad |= own[a] & ((upd[a][0] & !isfinite(x0)) | (upd[a][1] & !isfinite(x1)));
            if (own[a]) {
              uint2v v;
              v.x = __float_as_uint(x0);
              v.y = __float_as_uint(x1);
              __builtin_amdgcn_raw_buffer_store_b64(v, pl, voff[a], 0, 0);
            }
          }
          if (!OPEN && k == 1) {  // the mirror, for the relaxed columns
            const __amdgpu_buffer_rsrc_t p0l = buffer_of(out, plane8);
#pragma unroll
            for (int a = 0; a < RW; ++a) {
#pragma unroll
              for (int o = 0; o < 2; ++o)
                if (own[a] & upd[a][o])
                  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(W[a][sk][o]), p0l, voff[a] + 4u * o, 0, 0);
            }
          }
        }
      }
      write_edges((s + 1) % U, buf ^ 1);
      write_tables(buf ^ 1);
      lds_barrier();
    }
  };
  int p0 = pfirst;
#pragma unroll 1
  for (; p0 <= plast && p0 - (H - 1) <= wtop; p0 += U) block(p0, std::false_type{});
#pragma unroll 1
  for (; p0 <= plast; p0 += U) block(p0, std::true_type{});
  if (bad) atomicMin(status + kBadAt, (unsigned)(t + T - 1));
#pragma unroll
  for (int i = 0; i < T; ++i) {
    float m = 0.f;
#pragma unroll
    for (int a = 0; a < RW; ++a) m = own[a] ? fmaxf(m, dm[i][a]) : m;
    m = wave_max(m);
    if (lane == 0) wmax[wave][i] = m;
  }
  lds_barrier();
  if (threadIdx.x < T) {
    float m = 0.f;
    for (int w = 0; w < NW; ++w) m = fmaxf(m, wmax[w][threadIdx.x]);
    if (m > 0.f)
      atomicMax(err + (long long)(t + 1 + (int)threadIdx.x) * kErrSlots + (blockIdx.x % kErrSlots),
                __float_as_uint(m));
  }
}
#undef QESMC_ITEM
#undef QESMC_ITEM_PTR

// End of a stretch of launches over iterations [.., hi): find the iteration
// the run ended at (rows below lo were scanned before), and if that is inside
// the last launch, order its first iteration to be redone on its own.
// With items, of each of them (one work-group per problem).
__global__ __launch_bounds__(1024) void k_sor_settle(const MarchItem *__restrict__ items, const unsigned *rows, int lo,
                                                     int hi, float tol, unsigned *status)
{
  if (items) {
    rows = items[blockIdx.x].err;
    status = items[blockIdx.x].status;
  }
  __shared__ unsigned first;
  if (threadIdx.x == 0) first = 0xffffffffu;
  __syncthreads();
  // one wave per row, one slot per lane
  for (int t = lo + (int)(threadIdx.x >> 6); t < hi; t += 16) {
    const float v = __uint_as_float(rows[(long long)t * kErrSlots + (threadIdx.x & 63)]);
    const float m = wave_max(v > 0.f ? v : 0.f);
    if ((threadIdx.x & 63) == 0 && !(m > tol)) atomicMin(&first, (unsigned)t);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  unsigned end = status[kEnd];
  if (__uint_as_float(status[kStopExtend]) > 0.f) {
    const unsigned e = status[kStopAt];
    end = e < (unsigned)hi ? e : end;
  } else if (first < end) {
    end = first;
  }
  status[kEnd] = end;
  const unsigned lt = status[kLastT], li = status[kLastIters];
  const bool fix = li > 1u && end > lt && end < lt + li;
  status[kFixGo] = fix ? 1u : 0u;
  if (fix) status[kLastIters] = end - lt;
}

// The wall masks of both colours in the pair layout, two rows (2r, 2r+1) to a
// word: [k][r][q], the even row's pair in the low half, each pair's cell i = 2q
// in its low byte, as mask times 4.  Positions that are not relaxed (the ring, the padding) are
// open.  top[r][q / 32] (zeroed before) is the highest plane with a wall.
__global__ __launch_bounds__(256) void k_pair_masks(Dims d, const unsigned char *__restrict__ m0,
                                                    const unsigned char *__restrict__ m1, unsigned *__restrict__ out,
                                                    int *__restrict__ top)
{
  const int nr = (d.NY + 1) / 2;
  const int plane = nr * d.HP;
  const long long n = (long long)plane * d.NZ;
  const long long stride = (long long)gridDim.x * 256;
  for (long long x = blockIdx.x * 256LL + threadIdx.x; x < n; x += stride) {
    const int k = (int)(x / plane);
    const int rem = (int)(x - (long long)k * plane);
    const int r = rem / d.HP, q = rem - r * d.HP;
    unsigned w = 0;
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int j = 2 * r + y;
      unsigned lo = 63u, hi = 63u;
      if (k >= 1 && k <= d.NZ - 2 && j >= 1 && j <= d.NY - 2) {
        const long long s = (long long)(k * d.NY + j) * d.HP + q;
        const bool odd = (j + k) & 1;
        if (q >= 1 && 2 * q <= d.NX - 2) lo = odd ? m1[s] : m0[s];
        if (2 * q + 1 <= d.NX - 2) hi = odd ? m0[s] : m1[s];
      }
      w |= ((lo << 2) | (hi << 10)) << (16 * y);
    }
    out[x] = w;
    if (w != kOpenRows) atomicMax(top + r * ((d.HP + 31) / 32) + q / 32, k);
  }
}

// The wall values layer-major, canon8[k*8 + a] = canon[a*NZ + k] (words 6 and
// 7 unused), and per layer the sum of those each mask selects, added in the
// order the relaxation adds them.
__global__ __launch_bounds__(64) void k_march_tables(int NZ, const unsigned *__restrict__ canon,
                                                     unsigned *__restrict__ canon8, float *__restrict__ sums)
{
  const int k = blockIdx.x, lane = threadIdx.x;
  float v[6];
#pragma unroll
  for (int a = 0; a < 6; ++a) v[a] = (lane >> a) & 1 ? __uint_as_float(canon[a * NZ + k]) : 0.f;
  sums[64 * k + lane] = v[0] + v[1] + v[2] + v[3] + v[4] + v[5];
  if (lane < 8) canon8[8 * k + lane] = lane < 6 ? canon[lane * NZ + k] : 0u;
}

}  // namespace qesmc

using namespace qesmc;

// words of the highest-wall table of a domain
long long qesmc_march_top_words(const Dims &d) { return (long long)((d.NY + 1) / 2) * ((d.HP + 31) / 32); }

namespace {

// The instantiated shapes for two iterations per launch: waves, lanes per row group (two rows per group).
constexpr int kShapes[][2] = {{4, 32}, {8, 32}, {16, 32}, {16, 64}};
constexpr int kTail = 1;  // the shape of the single-iteration launches
constexpr int kBatchShape = 1;  // and of a batch's, or the one before it
constexpr int kWavesPerCu = 16;  // 128 vector registers each

// Columns of tiles (x tiles, y tiles) of a shape.
void march_columns(const Dims &d, int T, int shape, int *nq, int *nyt)
{
  const int nw = kShapes[shape][0], gw = kShapes[shape][1];
  const int half = (d.NX + 1) / 2, yr = 2 * nw * (64 / gw);
  *nq = half <= gw ? 1 : (half - 2 * T + gw - 2 * T - 1) / (gw - 2 * T);
  *nyt = d.NY <= yr ? 1 : (d.NY - 4 * T + yr - 4 * T - 1) / (yr - 4 * T);
}

// Relative cost of the steps a segment [ka, kb) takes: it fills its pipeline
// over the 2T-1 planes before it (those that exist) and drains over as many
// steps after it.  sum[p]: the cost of the steps below p.
double segment_cost(const std::vector<double> &sum, int T, int ka, int kb)
{
  const int first = ka - (2 * T - 1) > 0 ? ka - (2 * T - 1) : 0;
  return sum[(size_t)(kb + 2 * T - 1)] - sum[(size_t)first];
}

// Cut planes [1, end) into segments that cost at most `limit`, each starting
// on an odd plane and at least `least` planes long: the number of segments, 0
// if they do not fit the table.
int cut_segments(const std::vector<double> &sum, int T, int end, int least, double limit, MarchPlan &m)
{
  int n = 0, ka = 1;
  while (ka < end) {
    if (n == kMaxSegments) return 0;
    int kb = ka + least;
    while (kb < end && segment_cost(sum, T, ka, kb + 2 < end ? kb + 2 : end) <= limit) kb += 2;
    if (kb > end) kb = end;
    m.begin[n++] = (short)ka;
    ka = kb;
  }
  m.begin[n] = (short)end;
  return n;
}

// The cut into at most nseg segments whose dearest is the cheapest.
double balance_segments(const std::vector<double> &sum, int T, int end, int nseg, MarchPlan &m)
{
  const int least = 2 * T;
  double lo = 0.0, hi = segment_cost(sum, T, 1, end);
  m.nseg = cut_segments(sum, T, end, least, hi, m);
  for (int it = 0; it < 14 && nseg > 1; ++it) {
    const double mid = 0.5 * (lo + hi);
    MarchPlan trial = m;
    const int n = cut_segments(sum, T, end, least, mid, trial);
    if (n > 0 && n <= nseg) {
      hi = mid;
      m = trial;
      m.nseg = n;
    } else {
      lo = mid;
    }
  }
  double worst = 0.0;
  for (int q = 0; q < m.nseg; ++q) {
    const double c = segment_cost(sum, T, m.begin[q], m.begin[q + 1]);
    worst = c > worst ? c : worst;
  }
  return worst;
}

// Microseconds of one step with n waves on the CU, and what rows of 32 pairs cost on top.
double step_us(int waves) { return 0.62 + 0.054 * waves; }
double narrow_factor(int gw, bool beyond) { return gw == 64 ? 1.0 : beyond ? 1.15 : 1.04; }
constexpr double kLaunchUs = 4.6;

}  // namespace

// The cost of the steps below p, for all p, from the table of highest walls:
// 1 for an open plane, and 0.32 more for the share of the columns that have a wall there or above.
// In place, so that a run that may not allocate can do it.
void qesmc_march_costs(qesmc_ctx *x)
{
  const size_t NZ = (size_t)x->d.NZ;
  const long long n = qesmc_march_top_words(x->d);
  std::vector<double> &c = x->march_cost;
  std::fill(c.begin(), c.end(), 0.0);
  // first, one place up, the columns whose highest wall is plane k
  for (long long q = 0; q < n; ++q) c[(size_t)x->h_top[q] + 1] += 1.0;
  double above = (double)n, w = 1.0;
  for (size_t k = 0; k + 1 < c.size(); ++k) {
    const double here = c[k + 1];
    if (k < NZ) w = 1.0 + 0.32 * above / (double)n;
    above -= here;
    c[k + 1] = c[k] + w;
  }
}

// The march's shape and segments for the resident domain.  A segment's time is the sum of its steps' and the launch's
// that of the dearest segment.  Measured with 16 waves on a CU: 1.97 us a step
// where every plane has walls (298 vector instructions a wave: the vector ALUs
// are busy throughout), 1.49 us where none has (172; bound by the caches), so
// the segments near the ground are the shorter ones.  Microseconds of an open
// step with n waves on the CU: 0.62 + 0.054 n, and a launch 4.6 besides.
// Rows of 32 pairs touch a fifth more cache lines than rows of 64: 4 % slower
// per step, 15 % where they come from HBM.
// tile_k > 0 sets the planes per segment.
void qesmc_march_choose(qesmc_ctx *x, int tile_k)
{
  const Dims &d = x->d;
  const int end = d.NZ - 1;
  const std::vector<double> &sum = x->march_cost;
  auto uniform = [&](int T, int planes, MarchPlan &m) {
    int seg = planes < 2 * T ? 2 * T : (planes + 1) / 2 * 2;
    while ((end - 1 + seg - 1) / seg > kMaxSegments) seg += 2;
    m.nseg = 0;
    for (int ka = 1; ka < end; ka += seg) m.begin[m.nseg++] = (short)ka;
    m.begin[m.nseg] = (short)end;
  };
  const bool beyond = (double)x->nsplit * 2.0 * (4.0 + 4.0 + 1.0) > 256.0 * (1 << 20);
  for (int T = 2; T >= 1; --T) {
    MarchPlan &plan = x->march[T - 1];
    double best = 1e300;
    const int shapes = (int)(sizeof(kShapes) / sizeof(kShapes[0]));
    for (int c = T == 1 ? kTail : 0; c < (T == 1 ? kTail + 1 : shapes); ++c) {
      MarchPlan m{};
      m.shape = c;
      march_columns(d, T, c, &m.nq, &m.nyt);
      const long long columns = (long long)m.nq * m.nyt;
      const int fit = kWavesPerCu / kShapes[c][0];
      int tried = 0;
      for (int per_cu = 1; per_cu <= 6 * fit; ++per_cu) {
        long long nseg = (long long)per_cu * x->n_cu / columns;
        if (nseg > kMaxSegments) nseg = kMaxSegments;
        if (nseg < 1) nseg = 1;
        if (nseg == tried) continue;
        tried = (int)nseg;
        double worst;
        if (tile_k > 0) {
          uniform(T, tile_k, m);
          worst = segment_cost(sum, T, m.begin[0], m.begin[1]);
        } else {
          worst = balance_segments(sum, T, end, (int)nseg, m);
        }
        const long long per = (columns * m.nseg + x->n_cu - 1) / x->n_cu;
        const int resident = per < fit ? (int)per : fit;
        const double us = kLaunchUs + (double)((per + fit - 1) / fit) * worst * step_us(kShapes[c][0] * resident) *
                                          narrow_factor(kShapes[c][1], beyond);
        if (us < best) {
          best = us;
          plan = m;
        }
        if (tile_k > 0) break;
      }
    }
  }
}

// Whether the domain is a tower on one column of tiles that is too thin to
// march: a plan has at most 127 segments, which then grow with the height.
// March / colour passes in us per iteration: 12x12 cells 1200 high 8.9 / 8.4,
// 2500 12.6 / 10.3, 8000 29 / 16; 20x20 1500 9.7 / 10.1, 2500 12.8 / 12.4,
// 8000 32 / 17; 60x30 2500 16 / 21, 8000 39 / 42.
bool qesmc_march_too_thin(const Dims &d)
{
  int nq, nyt;
  march_columns(d, 2, kBatchShape, &nq, &nyt);
  return nq * nyt == 1 && 5LL * (d.NZ - 700) > 16LL * d.NX * d.NY;
}

hipError_t qesmc_fused_prepare(qesmc_ctx *x)
{
  hipLaunchKernelGGL(k_march_tables, dim3((unsigned)x->d.NZ), dim3(64), 0, x->stream, x->d.NZ, x->d_canon,
                     x->d_canon8, reinterpret_cast<float *>(x->d_canon8 + 8LL * x->d.NZ));
  const long long b = (x->nsplit / 2 + 255) / 256;
  const long long nt = qesmc_march_top_words(x->d);
  hipError_t e = qesmc_launch_fill_u32(x, reinterpret_cast<unsigned *>(x->d_top), nt, 0u);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_pair_masks, dim3((unsigned)(b < 16384 ? b : 16384)), dim3(256), 0, x->stream, x->d,
                     x->d_mask[0], x->d_mask[1], x->d_mask2, x->d_top);
  return hipGetLastError();
}

// The march's view of a problem whose tiles are those of m; first: its first work-group of the launch.
void qesmc_march_item(const qesmc_ctx *x, const MarchPlan &m, int first, MarchItem &a)
{
  const Dims &d = x->d;
  a = MarchItem{};
  a.d = d;
  a.nq = m.nq;
  a.nyt = m.nyt;
  a.ntiles = m.nq * m.nyt * m.nseg;
  a.first = first;
  for (int q = 0; q <= m.nseg; ++q) a.begin[q] = m.begin[q];
  a.set0 = reinterpret_cast<float2 *>(x->d_lc[0]);
  a.set1 = reinterpret_cast<float2 *>(x->d_lc2[0]);
  a.R = reinterpret_cast<const float2 *>(x->d_Rc[0]);
  a.mask = x->d_mask2;
  a.top = x->d_top;
  a.canon8 = x->d_canon8;
  a.sums = reinterpret_cast<const float *>(x->d_canon8 + 8LL * d.NZ);
  a.err = x->d_err;
  a.status = x->d_status;
  a.cur = x->d_cur;
}

namespace {

template <bool BATCH>
hipError_t launch_shape(hipStream_t s, int iters, int shape, int blocks, const MarchItem &item, const MarchRun &run)
{
  const int nw = kShapes[shape][0], gw = kShapes[shape][1];
#define QESMC_MARCH_LAUNCH(T, N, R, G) \
  hipLaunchKernelGGL((k_sor_march<T, N, R, G, BATCH>), dim3((unsigned)blocks), dim3(64 * N), 0, s, item, run)
  if (iters == 1) QESMC_MARCH_LAUNCH(1, 8, 2, 32);
  else if (nw == 4) QESMC_MARCH_LAUNCH(2, 4, 2, 32);
  else if (nw == 8) QESMC_MARCH_LAUNCH(2, 8, 2, 32);
  else if constexpr (BATCH) return hipErrorInvalidValue;
  else if (gw == 32) QESMC_MARCH_LAUNCH(2, 16, 2, 32);
  else QESMC_MARCH_LAUNCH(2, 16, 2, 64);
#undef QESMC_MARCH_LAUNCH
  return hipGetLastError();
}

}  // namespace

// Launch iterations t .. t + iters - 1 (iters 1 or 2), reading buffer set
// src and writing the other; om holds omega of the red and black pass of each.
// With fix, redo what k_sor_settle ordered instead.
hipError_t qesmc_launch_march(qesmc_ctx *x, int t, int iters, int itermax, const float *om, float tol, int src, bool fix)
{
  const Dims &d = x->d;
  if (d.NZ - 2 < 1 || d.NY - 2 < 1) return hipSuccess;
  MarchItem item;
  qesmc_march_item(x, x->march[iters - 1], 0, item);
  MarchRun a{};
  for (int h = 0; h < 2 * iters; ++h) a.om[h] = om[h];
  a.tol = tol;
  a.t = t;
  a.itermax = itermax;
  a.src = src;
  a.fix = fix ? 1 : 0;
  return launch_shape<false>(x->stream, iters, x->march[iters - 1].shape, item.ntiles, item, a);
}

// The run's end over iterations [lo, hi) and, if it falls inside the last
// launch, that launch redone up to it.
hipError_t qesmc_march_settle(qesmc_ctx *x, int lo, int hi, float tol)
{
  hipLaunchKernelGGL(k_sor_settle, dim3(1), dim3(1024), 0, x->stream, nullptr, x->d_err, lo, hi, tol, x->d_status);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const float om[2] = {0.f, 0.f};  // taken from the launch that is redone
  return qesmc_launch_march(x, 0, 1, 1, om, tol, 0, true);
}

// One shape and a cut of every member for launches of T iterations over a
// batch, and the microseconds such a launch is expected to take: in R rounds of
// resident work-groups a launch takes R times its dearest segment, so for
// each R the least segment cost whose tiles fit in R rounds, and the best R.
// (Measured on 4 to 16 cities of 64-256 cells a side, 8 waves: 1.04-1.19 times that,
// the most where the arrays leave the cache.  The smooth total cost over
// the places misleads: 556 tiles on 512 places take two rounds.)  Two work-groups of 8 waves
// per CU fill each other's barriers: at 16 such cities 83 us per iteration against
// 99 and 101 with 16 waves of 32 and 64 lanes a row, so 16 waves are not
// used; 4 waves only where the chip is not full.
int qesmc_march_batch_plan(qesmc_ctx *const *ctxs, int n, int T, std::vector<MarchPlan> &plans, double *expect_us)
{
  double top = 0.0;
  for (int i = 0; i < n; ++i) top = std::max(top, segment_cost(ctxs[i]->march_cost, T, 1, ctxs[i]->d.NZ - 1));
  const int n_cu = ctxs[0]->n_cu;
  std::vector<MarchPlan> trial((size_t)n);
  long long tiles = 0;
  double worst = 0.0;
  auto cut_all = [&](int c, double limit) {
    tiles = 0;
    worst = 0.0;
    for (int i = 0; i < n; ++i) {
      const std::vector<double> &sum = ctxs[i]->march_cost;
      MarchPlan &m = trial[(size_t)i];
      m.shape = c;
      m.nseg = 0;
      if (ctxs[i]->d.NZ < 3 || ctxs[i]->d.NY < 3) continue;  // nothing to relax
      march_columns(ctxs[i]->d, T, c, &m.nq, &m.nyt);
      m.nseg = cut_segments(sum, T, ctxs[i]->d.NZ - 1, 2 * T, limit, m);
      if (m.nseg == 0) return false;
      for (int q = 0; q < m.nseg; ++q) worst = std::max(worst, segment_cost(sum, T, m.begin[q], m.begin[q + 1]));
      tiles += (long long)m.nq * m.nyt * m.nseg;
    }
    return true;
  };
  double best = 1e300;
  int shape = -1;
  for (int c = T == 1 ? kTail : 0; c <= kBatchShape; ++c) {
    const int fit = kWavesPerCu / kShapes[c][0];
    auto us = [&]() {
      const long long per = (tiles + n_cu - 1) / n_cu;
      return kLaunchUs + (double)((per + fit - 1) / fit) * worst * step_us(kShapes[c][0] * (int)(per < fit ? per : fit)) *
                             narrow_factor(kShapes[c][1], false);
    };
    auto take = [&]() {
      if (us() >= best) return;
      best = us();
      plans = trial;
      shape = c;
    };
    if (cut_all(c, top)) take();
    const long long uncut = tiles;
    // R in units of one work-group per CU up to the full chip, then of full chips
    for (int r = 1; r <= (c == kBatchShape ? fit + 5 : fit); ++r) {
      const long long places = (long long)n_cu * (r <= fit ? r : (r - fit + 1) * fit);
      if (places <= uncut) continue;
      double lo = 0.0, hi = top;
      for (int it = 0; it < 10; ++it) {
        const double mid = 0.5 * (lo + hi);
        if (cut_all(c, mid) && tiles <= places) {
          hi = mid;
          take();
        } else {
          lo = mid;
        }
      }
    }
  }
  if (expect_us) *expect_us = best;
  return shape;
}

hipError_t qesmc_launch_march_batch(hipStream_t s, int iters, int shape, int blocks, const MarchRun &run)
{
  return launch_shape<true>(s, iters, shape, blocks, MarchItem{}, run);
}

hipError_t qesmc_march_settle_batch(hipStream_t s, const MarchItem *items, int n, int hi, float tol)
{
  hipLaunchKernelGGL(k_sor_settle, dim3((unsigned)n), dim3(1024), 0, s, items, nullptr, 0, hi, tol, nullptr);
  return hipGetLastError();
}
