// Batched orbital-invariant spin-orbital MP2 over independent instances of
// possibly different sizes (the +/- displaced systems of a finite-difference
// set), one launch per iteration for the whole set.
//
// Per instance k (O_k, V_k, F_k, eps_k, drv_k) the iteration is the Jacobi
// step of the non-canonical MP2 equations (ci_wfn.py:210-212 with the
// driver <ab||ij>, solve_MP2_SO at diagonal F, mp2_wfn.py:64-87):
//   r_ij[a,b] = s drv_ij[a,b] + Y_ij[a,b] - Y_ij[b,a] - Z_ij[a,b] + Z_ji[a,b]
//   Y_ij[a,b] = sum_e x_ij[a,e] Fvv(b,e),   Z_ij[a,b] = sum_m Foo(m,j) x_im[a,b]
//   x_new = x + r / (e_i + e_j - e_a - e_b)
// with Fvv(b,e) = F[O+b][O+e], Foo(m,j) = F[m][j]; an instance with
// transpose_f set uses F^T (the adjoint lambda equations), and s is the
// instance's driver scale, so amplitude and lambda solves share one batch.
// The amplitudes are antisymmetric in (i,j) and in (a,b) and are stored
// packed, x[(i<j)][(a<b)], a quarter of the dense tensor; the residual is
// formed only for i<j, a<b.
//
// Two kernels per step cover every instance.  nc_z_kernel forms
// W_ij[(ab)] = -Z_ij + Z_ji, Z_ij = sum_m Foo(m,j) x_im, for the pairs i<j: a
// workgroup takes one (instance, slab of the (a<b) pairs) with a thread to each
// (i, pair) and joins the two orders in LDS (past O = 47 a wave takes a tile of
// the pairs i<j instead).  ncp_step_kernel then gives a
// workgroup one (instance, pair i<j, tile pair A <= B of the virtual plane): it
// forms Y_ij[a,b] - Y_ij[b,a] over the tile on the FP64 matrix cores with
// K = e staged in 8-wide chunks through LDS (the tile's rows of x_ij expanded
// from the packed row with the antisymmetry signs, and the matching columns
// of Fvv), adds the driver and W, applies the update and writes its partial
// residual norm; per_instance_sum reduces
// those per instance in a fixed order.  All tables live in the workspace, written once
// by apy_mp2_nc_batched_setup, so a sequence of steps can be captured in a
// HIP graph.
#include "common.h"

#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <vector>

namespace {

constexpr int BLK = 256;
constexpr int MT = 32;       // virtual tile edge
#ifndef APY_MP2_MKC
#define APY_MP2_MKC 8
#endif
constexpr int MKC = APY_MP2_MKC;   // e chunk of the Y product (a multiple of 8)
static_assert(MKC % 8 == 0 && MKC <= 32, "e chunk");
constexpr int SBLK = 256;                          // step kernel: 4 waves, 16 x 16 of the 32 x 32 tile each
constexpr int EN_B = 64;     // energy partial sums per instance

struct Item {
  int32_t inst, pij, ta, tb;
};

// The slab of W that a work item forms in LDS: SP pairs (ab) by all (i<j), at most one thread an (i, ab);
// 0: LDS holds fewer than two (O > 47), an item is four WT x WT tiles of pairs (i<j) by 64 pairs (ab) then.
// us a step, slab / tiles:  O=33 V=40, 4 instances 155 / 197   O=46 V=12, 4  130 / 153   O=46 V=40, 2  208 / 236
//                           O=48 V=40, 2           371 / 249   O=48 V=12, 2  119 / 109   O=66 V=40, 2  828 / 404
constexpr int SLAB = 2192;
__host__ __device__ inline int slab_of(int64_t O) {
  const int64_t po = O * (O - 1) / 2;
  if (O < 2 || po > SLAB) return 0;
  const int64_t a = BLK / (O < BLK ? O : BLK), b = SLAB / po;
  return b < 2 ? 0 : (int)(a < b ? a : b);
}
constexpr int WT = 4;
__host__ __device__ inline int64_t wtiles(int64_t O) { const int64_t nt = (O + WT - 1) / WT; return nt * (nt + 1) / 2; }
// pairs (ab) of an item, and items of a span of them
inline int64_t zspan(int64_t O) { return slab_of(O) ? slab_of(O) : 64; }
inline int64_t zrows(int64_t O) { return slab_of(O) ? 1 : (wtiles(O) + BLK / 64 - 1) / (BLK / 64); }

struct ZItem {
  int32_t inst, p0, t0, pad;   // first pair (ab), first tile of pairs (ij)
};

struct Header {
  int64_t n, items, zitems;
  int64_t zitem_off, z_off;   // byte offsets of the W work items and of the W blocks
};

inline size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

__host__ __device__ inline int64_t npair(int64_t N) { return N * (N - 1) / 2; }
__host__ __device__ inline int64_t prow(int64_t p, int64_t N) { return p * (2 * N - p - 1) / 2; }
__host__ __device__ inline int64_t pidx(int64_t p, int64_t q, int64_t N) { return prow(p, N) + q - p - 1; }
inline int64_t ntiles(int64_t V) { return (V + MT - 1) / MT; }

__device__ inline void pdec(int64_t P, int64_t N, int64_t& p, int64_t& q) {
  double b = 2.0 * (double)N - 1.0;
  double disc = b * b - 8.0 * (double)P;
  int64_t pp = (int64_t)((b - sqrt(disc > 0.0 ? disc : 0.0)) * 0.5);
  if (pp < 0) pp = 0;
  if (pp > N - 2) pp = N - 2;
  while (pp > 0 && prow(pp, N) > P) --pp;
  while (pp + 1 <= N - 2 && prow(pp + 1, N) <= P) ++pp;
  p = pp;
  q = P - prow(pp, N) + pp + 1;
}

// Workspace: header, instance table, item table, per-instance item offsets,
// item partial norms, energy partial sums, per-instance offsets of the Z
// blocks, then (at byte offsets the header holds, so the step needs only
// (n, items) on the host) the W work items and the W blocks themselves
// (sum_k Po_k Pv_k complex).
struct WsLayout {
  size_t inst, item, off, part, epart, zoff, zitem, z, total;
};

inline WsLayout layout(int n, int64_t items, int64_t zitems = 0, int64_t zelems = 0) {
  WsLayout L;
  L.inst = al256(sizeof(Header));
  L.item = L.inst + al256((size_t)n * sizeof(apy_mp2_nc_instance));
  L.off = L.item + al256((size_t)items * sizeof(Item));
  L.part = L.off + al256((size_t)(n + 1) * sizeof(int64_t));
  L.epart = L.part + al256((size_t)items * sizeof(double));
  L.zoff = L.epart + al256((size_t)n * EN_B * sizeof(double2));
  L.zitem = L.zoff + al256((size_t)(n + 1) * sizeof(int64_t));
  L.z = L.zitem + al256((size_t)zitems * sizeof(ZItem));
  L.total = L.z + al256((size_t)zelems * sizeof(double2));
  return L;
}

int64_t count_zitems(int n, const apy_mp2_nc_instance* inst, int64_t* zelems) {
  int64_t z = 0, e = 0;
  for (int k = 0; k < n; ++k) {
    if (inst[k].O < 2 || inst[k].V < 2) continue;
    const int64_t Pv = npair(inst[k].V);
    z += (Pv + zspan(inst[k].O) - 1) / zspan(inst[k].O) * zrows(inst[k].O);
    e += npair(inst[k].O) * Pv;
  }
  if (zelems) *zelems = e;
  return z;
}

int64_t count_items(int n, const apy_mp2_nc_instance* inst) {
  int64_t items = 0;
  for (int k = 0; k < n; ++k) {
    const int64_t nt = ntiles(inst[k].V);
    if (inst[k].O >= 2 && inst[k].V >= 2) items += npair(inst[k].O) * (nt * (nt + 1) / 2);
  }
  return items;
}

// acc += a b as four fused multiply-adds (written out: the compiler may not reassociate acc + (ab - cd))
__device__ inline void cfma(double2& acc, double2 a, double2 b) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
}

// F read through the scalar cache: every address is uniform over the workgroup and no kernel of a step
// writes F.
typedef const __attribute__((address_space(4))) double* SF;

// Z_ij[P] = sum_m Foo(m,j) x_im[P] of one (i, P) a thread, JB values of j from j0: x_im from memory, Foo in
// scalar registers, JB complex sums in vector registers.  The vector units do FP64 at the matrix units'
// rate, and this form has no padding: 16 x 16 x 4 blocks spent 2 x 5 of them on the 18 x 18 product of
// O = 18.
template <int JB, bool TF>
__device__ __forceinline__ void z_rows(SF Fr, const double2* __restrict__ x, int O, int n, int64_t Pv, int i, int j0,
                                       int64_t P, double2 (&acc)[JB]) {
#pragma unroll
  for (int j = 0; j < JB; ++j) acc[j] = make_double2(0.0, 0.0);
  int off[JB];                                         // past the end: a sum that is not taken
#pragma unroll
  for (int j = 0; j < JB; ++j) off[j] = 2 * min(j0 + j, O - 1) * n;
  const int ri = (int)prow(i, O) - i - 1;              // pair (i, m), m > i: ri + m; (m, i): prow(m) + i - m - 1
  auto load = [&](int m) {
    const int mm = min(m, O - 1), r = mm > i ? ri + mm : mm < i ? (int)prow(mm, O) + i - mm - 1 : 0;
    return x[(int64_t)r * Pv + P];
  };
  // two x_im ahead: an L2 read takes as long as the sums of two m over the waves of a SIMD
  double2 cur[2] = {load(0), load(1)}, nxt[2];
  for (int m0 = 0; m0 < O; m0 += 2) {
    nxt[0] = load(m0 + 2);
    nxt[1] = load(m0 + 3);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int m = m0 + u;
      if (m >= O) break;
      double2 v = cur[u];
      v.x = m == i ? 0.0 : m < i ? -v.x : v.x;
      v.y = m == i ? 0.0 : m < i ? -v.y : v.y;
      // row m of F_oo from j0 (F^T: its column): the non-transposed row is read on past O, still inside F
      // (m <= O - 1, V >= 2), so that its loads are of four elements each
      const SF Fm = Fr + 2 * (TF ? m : m * n + j0);
#pragma unroll
      for (int j = 0; j < JB; ++j) {
        const int o = TF ? off[j] : 2 * j;
        const double fr = Fm[o], fi = Fm[o + 1];
        acc[j].x = fma(fr, v.x, acc[j].x);
        acc[j].x = fma(-fi, v.y, acc[j].x);
        acc[j].y = fma(fr, v.y, acc[j].y);
        acc[j].y = fma(fi, v.x, acc[j].y);
      }
    }
    cur[0] = nxt[0];
    cur[1] = nxt[1];
  }
}

// W_(i<j)[P] = -Z_ij[P] + Z_ji[P] for the SP pairs (ab) from p0: thread (i, P) forms Z_ij for all j and
// stores the j > i of them to the slab in LDS, then, after a barrier, adds its j < i to the rows that
// thread (j, P) stored; rows past the first pass of threads find every smaller row stored.  With more than
// one block of j (O > JB) both are additions to zeros.  The slab leaves LDS along P.  Kept as one array: as
// Z_ij and Z_ji of every ordered pair this kernel's writes and the step's reads were twice as long.
template <int JB, bool TF>
__device__ __forceinline__ void w_slab(SF Fr, const double2* __restrict__ x, double2* __restrict__ W, double2* slab,
                                       int O, int n, int64_t Pv, int64_t p0, int SP) {
  const int tid = threadIdx.x, rows = BLK / SP, pl = tid % SP, il = tid / SP, Po = (int)npair(O);
  const int64_t P = min(p0 + pl, Pv - 1);
  const bool multi = O > JB;
  if (multi) {
    for (int e = tid; e < Po * SP; e += blockDim.x) slab[e] = make_double2(0.0, 0.0);
    __syncthreads();
  }
  for (int i0 = 0; i0 < O; i0 += rows) {
    const int i = i0 + il;
    const bool own = il < rows && i < O;
    for (int j0 = 0; j0 < O; j0 += JB) {
      double2 acc[JB];
      if (own) {
        z_rows<JB, TF>(Fr, x, O, n, Pv, i, j0, P, acc);
#pragma unroll
        for (int j = 0; j < JB; ++j)
          if (j0 + j > i && j0 + j < O) {
            double2& w = slab[(int)pidx(i, j0 + j, O) * SP + pl];
            w = multi ? make_double2(w.x - acc[j].x, w.y - acc[j].y) : make_double2(-acc[j].x, -acc[j].y);
          }
      }
      __syncthreads();
      if (own) {
#pragma unroll
        for (int j = 0; j < JB; ++j)
          if (j0 + j < i) {
            double2& w = slab[(int)pidx(j0 + j, i, O) * SP + pl];
            w.x += acc[j].x;
            w.y += acc[j].y;
          }
      }
      if (multi) __syncthreads();
    }
  }
  __syncthreads();
  const int np = (int)min((int64_t)SP, Pv - p0);
  for (int e = tid; e < Po * SP; e += blockDim.x) {
    const int r = e / SP, c = e % SP;
    if (c < np) W[r * Pv + p0 + c] = slab[e];
  }
}

// W_(i<j)[P] of a WT x WT tile of pairs (ij) and 64 pairs P a wave: 2 WT rows of x and as many elements of Foo
// (scalar: the tile is the wave's) a value of m for 2 WT^2 complex products, all sums in registers.  Bound by
// the reads of x, each row from L2 once a tile.  One thread an element of W ran on the few workgroups that 256
// pairs P an item left: O=68 V=40, two instances, 111 ms a step, 0.42 ms so.
template <bool TF>
__device__ __forceinline__ void w_tile(SF Fr, const double2* __restrict__ x, double2* __restrict__ W, int O, int n,
                                       int64_t Pv, int64_t P, int t) {
  if (t >= wtiles(O)) return;
  const int nt = (O + WT - 1) / WT;
  int ti = 0;
  while (t >= nt - ti) { t -= nt - ti; ++ti; }
  const int i0 = ti * WT, j0 = (ti + t) * WT;
  const bool in = P < Pv;
  const double2* xp = x + (in ? P : 0);
  double2 acc[WT][WT];
#pragma unroll
  for (int a = 0; a < WT; ++a)
#pragma unroll
    for (int b = 0; b < WT; ++b) acc[a][b] = make_double2(0.0, 0.0);
  // x_pm[P], p past the end: the last row, whose sums are not taken
  auto row = [&](int p, int m) {
    p = min(p, O - 1);
    const int64_t r = p < m ? pidx(p, m, O) : p > m ? pidx(m, p, O) : 0;
    double2 v = xp[r * Pv];
    v.x = p == m ? 0.0 : p > m ? -v.x : v.x;
    v.y = p == m ? 0.0 : p > m ? -v.y : v.y;
    return v;
  };
  auto foo = [&](int m, int p) {
    p = min(p, O - 1);
    const SF f = Fr + 2 * (TF ? (int64_t)p * n + m : (int64_t)m * n + p);
    return make_double2(f[0], f[1]);
  };
  for (int m = 0; m < O; ++m) {
    double2 xi[WT], xj[WT], fi[WT], fj[WT];
#pragma unroll
    for (int a = 0; a < WT; ++a) {
      xi[a] = row(i0 + a, m);
      xj[a] = row(j0 + a, m);
      fi[a] = foo(m, i0 + a);
      fj[a] = foo(m, j0 + a);
      fj[a] = make_double2(-fj[a].x, -fj[a].y);
    }
#pragma unroll
    for (int a = 0; a < WT; ++a)
#pragma unroll
      for (int b = 0; b < WT; ++b) {
        cfma(acc[a][b], fi[a], xj[b]);
        cfma(acc[a][b], fj[b], xi[a]);
      }
  }
  if (!in) return;
#pragma unroll
  for (int a = 0; a < WT; ++a)
#pragma unroll
    for (int b = 0; b < WT; ++b)
      if (i0 + a < j0 + b && j0 + b < O) W[pidx(i0 + a, j0 + b, O) * Pv + P] = acc[a][b];
}

// W_k[(i<j)][(ab)] = sum_m (Foo(m,i) x_jm - Foo(m,j) x_im)[(ab)] for every instance and slice of pairs
// (ab) (grid-stride over the work list, whose length is in the header).
__device__ __forceinline__ void nc_z_phase(char* __restrict__ ws, const apy_mp2_nc_instance* __restrict__ insts,
                                           const int64_t* __restrict__ zoff, int reverse, double2* slab) {
  const Header* hdr = (const Header*)ws;
  const int64_t nz = hdr->zitems;
  const ZItem* zitems = (const ZItem*)(ws + hdr->zitem_off);
  double2* zbase = (double2*)(ws + hdr->z_off);
  for (int64_t w = blockIdx.x; w < nz; w += gridDim.x) {
    const ZItem it = zitems[w];
    const int inst = __builtin_amdgcn_readfirstlane(it.inst);
    const apy_mp2_nc_instance& I = insts[inst];
    const int O = __builtin_amdgcn_readfirstlane((int)I.O), n = O + __builtin_amdgcn_readfirstlane((int)I.V);
    const int64_t Pv = npair(I.V);
    const double2* x = (const double2*)(reverse ? I.x_new : I.x);
    double2* W = zbase + zoff[inst];
    // the pointer of F in scalar registers
    const uint64_t fp = (uint64_t)I.fock;
    const SF Fr = (SF)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)fp) |
                       (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(fp >> 32)) << 32);
    const int SP = slab_of(O);
    if (SP == 0) {                                     // a tile of pairs (ij) a wave
      const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
      if (I.transpose_f) w_tile<true>(Fr, x, W, O, n, Pv, it.p0 + (int64_t)(threadIdx.x & 63), it.t0 + wave);
      else w_tile<false>(Fr, x, W, O, n, Pv, it.p0 + (int64_t)(threadIdx.x & 63), it.t0 + wave);
      continue;
    }
    __syncthreads();                                   // the slab of the previous item is written out
    // the smallest block of j that covers O in as few passes as blocks of 20 do
    const int jb = (O + (O + 19) / 20 - 1) / ((O + 19) / 20);
    auto run = [&](auto c) {
      constexpr int JB = decltype(c)::value;
      if (I.transpose_f) w_slab<JB, true>(Fr, x, W, slab, O, n, Pv, it.p0, SP);
      else w_slab<JB, false>(Fr, x, W, slab, O, n, Pv, it.p0, SP);
    };
    if (jb <= 8) run(std::integral_constant<int, 8>{});
    else if (jb <= 12) run(std::integral_constant<int, 12>{});
    else if (jb <= 16) run(std::integral_constant<int, 16>{});
    else if (jb <= 18) run(std::integral_constant<int, 18>{});
    else run(std::integral_constant<int, 20>{});
  }
}

__global__ __launch_bounds__(BLK, 4) void nc_z_kernel(char* __restrict__ ws, const apy_mp2_nc_instance* __restrict__ insts,
                                                   const int64_t* __restrict__ zoff, int reverse) {
  __shared__ double2 slab[SLAB];
  nc_z_phase(ws, insts, zoff, reverse, slab);
}

// One work item per workgroup of four waves: a 32 x 32 tile of the residual, each wave a 16 x 16
// quarter of it on the FP64 matrix cores.  (64-wide tiles stage half the elements a product, but their
// fewer waves left the reads of the epilogue exposed: a step of the 36-instance set 421 us with four waves
// of 32 x 32, 330 us with eight of 32 x 16, against 322 us for 32-wide tiles.)  Off the diagonal (A < B) both products go into
// one complex accumulator,
//   r[a][b] += sum_e XA[a][e] GB[e][b] - sum_e GA[e][a] XB[b][e],
// as eight v_mfma_f64_16x16x4f64 per block and four values of e (real and imaginary planes; the second
// product with its A operand negated).  On a diagonal tile pair (A == B) the two products are one
// matrix and its transpose, so each wave forms only Y = XA GA over its quarter (four MFMAs per
// four e) and r = Y - Y^T is assembled through LDS.  Quarters past V are skipped.
// MFMA f64 16x16x4 lanes: A[l%16][l/16], B[l/16][l%16], D[l/16 + 4r][l%16].
constexpr int STEP_LDS = 2 * MT * (MKC + 1) + 2 * MKC * (MT + 1) > MT * (MT + 1) ? 2 * MT * (MKC + 1) + 2 * MKC * (MT + 1)
                                                                               : MT * (MT + 1);   // double2

__device__ __forceinline__ void ncp_step_item(int64_t b, const apy_mp2_nc_instance* __restrict__ insts,
                                              const Item* __restrict__ items, int reverse,
                                              const char* __restrict__ ws, const int64_t* __restrict__ zoff,
                                              double* __restrict__ part, double2* sh) {
  __shared__ double red[SBLK];
  auto XA = reinterpret_cast<double2 (*)[MKC + 1]>(sh);
  auto XB = reinterpret_cast<double2 (*)[MKC + 1]>(sh + MT * (MKC + 1));
  auto GA = reinterpret_cast<double2 (*)[MT + 1]>(sh + 2 * MT * (MKC + 1));
  auto GB = reinterpret_cast<double2 (*)[MT + 1]>(sh + 2 * MT * (MKC + 1) + MKC * (MT + 1));
  auto Ysh = reinterpret_cast<double2 (*)[MT + 1]>(sh);    // diagonal tiles, after the products
  __syncthreads();                                   // LDS of the previous item is no longer read
  const Item it = items[b];
  const apy_mp2_nc_instance I = insts[it.inst];
  const int O = (int)I.O, V = (int)I.V, n = O + V;
  const int64_t Pv = npair(V);
  const int transpose_f = I.transpose_f;
  const double s = I.drv_scale;
  const int tid = threadIdx.x, lane = tid & 63, wm = (tid >> 6) & 1, wn = tid >> 7;
  int64_t i, j;
  pdec(it.pij, O, i, j);
  const double2* F = (const double2*)I.fock;
  const double2* row = (const double2*)(reverse ? I.x_new : I.x) + (int64_t)it.pij * Pv;
  double2* xn = (double2*)(reverse ? I.x : I.x_new) + (int64_t)it.pij * Pv;
  const int a0 = it.ta * MT, b0 = it.tb * MT;

  v4d acc_re = (v4d){0, 0, 0, 0}, acc_im = (v4d){0, 0, 0, 0};
  // diagonal tile pair (A == B): XB = XA and GB = GA, so every wave forms only Y = x Fvv^T over its
  // quarter and the residual Y[a][b] - Y[b][a] is assembled through LDS after the products
  const bool diag = it.ta == it.tb;                          // uniform across the workgroup
  // one e chunk of x_ij rows a0.., b0.. and of Fvv columns, fetched into registers while the previous
  // chunk is multiplied (NQ elements of each of the four tiles per thread), then stored to LDS
  constexpr int NQ = MT * MKC / SBLK;
  const int am = a0 + wm * 16, bn = b0 + wn * 16;            // the wave's first row and column
  const bool works = am < V && bn < V;
  // x_ij[p][e] is row[pidx(p, e)] above the diagonal (contiguous along e) and -row[pidx(e, p)] below it
  // (contiguous along p): each tile element is fetched by one of two passes, the upper one with e fastest
  // across the threads and the lower one with p fastest, so that both read along the packed row.  A pass
  // that has no element in the chunk is left out; the addresses step with the chunk.
  double2 sxa_u[NQ], sxa_l[NQ], sxb_u[NQ], sxb_l[NQ], sga[NQ], sgb[NQ];
  int up[NQ];                                          // offset of the upper row (tile A)
  int64_t ga[NQ];                                      // of Fvv(a0 + cc, rr)
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int q = tid + SBLK * k, p = a0 + q / MKC;
    up[k] = p * (2 * V - p - 1) / 2 - p - 1 + q % MKC;
    // GA[rr][cc] = Fvv(a0+cc, e0+rr), Fvv(b, e) = F[O+b][O+e] (F^T: F[O+e][O+b]), read along the contiguous
    // index of F (e, or b for F^T)
    const int rr = transpose_f ? q / MT : q % MKC, cc = transpose_f ? q % MT : q / MKC;
    ga[k] = transpose_f ? (int64_t)(O + rr) * n + O + a0 + cc : (int64_t)(O + a0 + cc) * n + O + rr;
  }
  const int64_t ga_step = transpose_f ? n : 1, gb_off = (int64_t)(b0 - a0) * (transpose_f ? 1 : n);
  auto fetch = [&](int e0) {
    const bool ua = e0 + MKC - 1 > a0, la = a0 + MT - 1 > e0;
    const bool ub = e0 + MKC - 1 > b0, lb = b0 + MT - 1 > e0;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int q = tid + SBLK * k;
      const int r = q / MKC, e = e0 + q % MKC;       // upper pass: XA[r][c] = x_ij[a0+r, e0+c], c fastest
      const int rl = q % MT, el = e0 + q / MT;       // lower pass: r fastest
      const int lrow = el * (2 * V - el - 1) / 2 - el - 1;
      sxa_u[k] = make_double2(0.0, 0.0);
      sxa_l[k] = make_double2(0.0, 0.0);
      if (ua && a0 + r < e && e < V) sxa_u[k] = row[up[k] + e0];
      if (la && a0 + rl > el && a0 + rl < V) sxa_l[k] = row[lrow + a0 + rl];
      const int e2 = e0 + (transpose_f ? q / MT : q % MKC), cc = transpose_f ? q % MT : q / MKC;
      const int64_t go = ga[k] + e0 * ga_step;
      sga[k] = make_double2(0.0, 0.0);
      if (e2 < V && a0 + cc < V) sga[k] = F[go];
      if (!diag) {
        const int pb = b0 + r;
        sxb_u[k] = make_double2(0.0, 0.0);
        sxb_l[k] = make_double2(0.0, 0.0);
        if (ub && pb < e && e < V) sxb_u[k] = row[pb * (2 * V - pb - 1) / 2 + e - pb - 1];
        if (lb && b0 + rl > el && b0 + rl < V) sxb_l[k] = row[lrow + b0 + rl];
        sgb[k] = make_double2(0.0, 0.0);
        if (e2 < V && b0 + cc < V) sgb[k] = F[go + gb_off];
      }
    }
  };
  fetch(0);
  for (int e0 = 0; e0 < V; e0 += MKC) {
    __syncthreads();                                 // the previous chunk is no longer read
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int q = tid + SBLK * k;
      const int r = q / MKC, c = q % MKC, rl = q % MT, cl = q / MT;
      const int e = e0 + c, el = e0 + cl;
      // each element is stored once: by the lower pass where p > e is in range, else by the upper pass
      if (!(a0 + r > e && a0 + r < V)) XA[r][c] = sxa_u[k];
      if (a0 + rl > el && a0 + rl < V) XA[rl][cl] = make_double2(-sxa_l[k].x, -sxa_l[k].y);
      const int rr = transpose_f ? q / MT : q % MKC, cc = transpose_f ? q % MT : q / MKC;
      GA[rr][cc] = sga[k];
      if (!diag) {
        if (!(b0 + r > e && b0 + r < V)) XB[r][c] = sxb_u[k];
        if (b0 + rl > el && b0 + rl < V) XB[rl][cl] = make_double2(-sxb_l[k].x, -sxb_l[k].y);
        GB[rr][cc] = sgb[k];
      }
    }
    __syncthreads();
    if (e0 + MKC < V) fetch(e0 + MKC);               // in flight during the products below
    if (!works) continue;                            // nothing of this wave's quarter is in range
#pragma unroll
    for (int ks = 0; ks < MKC / 4; ++ks) {
      const int kk = ks * 4 + (lane >> 4), ra = wm * 16 + (lane & 15), cb = wn * 16 + (lane & 15);
      const double2 xa = XA[ra][kk], gb = diag ? GA[kk][cb] : GB[kk][cb];   // sum_e x[a,e] Fvv(b,e)
      acc_re = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.x, gb.x, acc_re, 0, 0, 0);
      acc_im = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.x, gb.y, acc_im, 0, 0, 0);
      acc_re = __builtin_amdgcn_mfma_f64_16x16x4f64(-xa.y, gb.y, acc_re, 0, 0, 0);
      acc_im = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.y, gb.x, acc_im, 0, 0, 0);
      if (!diag) {
        const double2 ga2 = GA[kk][ra], xb = XB[cb][kk];   // - sum_e Fvv(a,e) x[b,e]
        acc_re = __builtin_amdgcn_mfma_f64_16x16x4f64(-ga2.x, xb.x, acc_re, 0, 0, 0);
        acc_im = __builtin_amdgcn_mfma_f64_16x16x4f64(-ga2.x, xb.y, acc_im, 0, 0, 0);
        acc_re = __builtin_amdgcn_mfma_f64_16x16x4f64(ga2.y, xb.y, acc_re, 0, 0, 0);
        acc_im = __builtin_amdgcn_mfma_f64_16x16x4f64(-ga2.y, xb.x, acc_im, 0, 0, 0);
      }
    }
  }
  // the epilogue's reads, in flight while a diagonal tile is transposed
  const double* eps = (const double*)I.eps;
  const double2* drv = (const double2*)I.drv + (i * O + j) * (int64_t)V * V;
  // -sum_m Foo(m,j) x_im + sum_m Foo(m,i) x_jm
  const double2* Wp = (const double2*)(ws + ((const Header*)ws)->z_off) + zoff[it.inst] + (int64_t)it.pij * Pv;
  const double eij = eps[i] + eps[j];
  const int bb = bn + (lane & 15);
  double2 dv[4], wv[4], xv[4];
  double ea[4];
  const double ebb = eps[O + min(bb, V - 1)];
#pragma unroll
  for (int r = 0; r < 4; ++r) {                      // past the end or below the diagonal: pair (0, 1)
    const int a = am + (lane >> 4) + 4 * r;
    const bool in = bb < V && a < bb;
    const int pa = in ? a : 0, pb = in ? bb : 1, Pab = pa * (2 * V - pa - 1) / 2 + pb - pa - 1;
    dv[r] = drv[pa * V + pb];
    wv[r] = Wp[Pab];
    xv[r] = row[Pab];
    ea[r] = eps[O + pa];
  }
  if (diag) {
    // every wave holds Y over its quarter of the tile (the lower-left one too): r = Y[a][b] - Y[b][a]
    __syncthreads();                                 // the last chunk's tiles (aliased by Ysh) are read
#pragma unroll
    for (int r = 0; r < 4; ++r)
      Ysh[wm * 16 + (lane >> 4) + 4 * r][wn * 16 + (lane & 15)] = make_double2(acc_re[r], acc_im[r]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double2 yt = Ysh[wn * 16 + (lane & 15)][wm * 16 + (lane >> 4) + 4 * r];
      acc_re[r] -= yt.x;
      acc_im[r] -= yt.y;
    }
  }
  double acc = 0.0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int a = am + (lane >> 4) + 4 * r;
    if (bb >= V || a >= bb) continue;
    const double2 rr = make_double2(s * dv[r].x + acc_re[r] + wv[r].x, s * dv[r].y + acc_im[r] + wv[r].y);
    const double D = eij - ea[r] - ebb;
    xn[a * (2 * V - a - 1) / 2 + bb - a - 1] = make_double2(xv[r].x + rr.x / D, xv[r].y + rr.y / D);
    acc += rr.x * rr.x + rr.y * rr.y;
  }
  red[tid] = acc;
  __syncthreads();
  for (int w = SBLK / 2; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  if (tid == 0) part[b] = red[0];
}

// Five waves a SIMD (94 registers; 98 and four waves without the bound): the waits at the chunks and in the
// epilogue are covered by other workgroups, a solve of 36 instances of O 14-18 V 54-66 3.16 -> 3.07 ms.
__global__ __launch_bounds__(SBLK, 5) void ncp_step_kernel(const apy_mp2_nc_instance* __restrict__ insts,
                                                        const Item* __restrict__ items, int reverse,
                                                        const char* __restrict__ ws, const int64_t* __restrict__ zoff,
                                                        double* __restrict__ part) {
  __shared__ double2 sh[STEP_LDS];
  ncp_step_item(blockIdx.x, insts, items, reverse, ws, zoff, part, sh);
}

// Called by all of a workgroup of at least BLK threads; the first BLK sum.
__device__ __forceinline__ void instance_sum(int64_t k, const int64_t* __restrict__ off,
                                             const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double red[BLK];
  __syncthreads();
  const int64_t b = off[k], e = off[k + 1];
  if (threadIdx.x < BLK) {
    double acc = 0.0;
    for (int64_t q = b + threadIdx.x; q < e; q += BLK) acc += part[q];
    red[threadIdx.x] = acc;
  }
  __syncthreads();
  for (int w = BLK / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[k] = red[0];
}

__global__ __launch_bounds__(BLK) void per_instance_sum(const int64_t* __restrict__ off,
                                                        const double* __restrict__ part, double* __restrict__ out) {
  instance_sum(blockIdx.x, off, part, out);
}

// The whole solve in one cooperative launch: every resident workgroup loops over the W work items,
// the step items and the per-instance sums of an iteration with a grid barrier after each phase, then
// reads the n residual norms and stops when sqrt(max) < tol (the test of MP2NCBatch.solve after every
// step) or after maxit steps.  Each phase is the same per-item code as the three kernels of
// apy_mp2_nc_batched_step, so the iterates are bit-identical to the step-by-step solve.  An odd step
// count leaves the amplitudes in x_new; they are copied back to x before the kernel ends.
__global__ __launch_bounds__(SBLK) void nc_persistent_kernel(char* __restrict__ ws,
                                                             const apy_mp2_nc_instance* __restrict__ insts,
                                                             const Item* __restrict__ items,
                                                             const int64_t* __restrict__ off,
                                                             const int64_t* __restrict__ zoff,
                                                             double* __restrict__ part, double* __restrict__ rnorm,
                                                             int n, int64_t n_items, double tol, int maxit,
                                                             int64_t* __restrict__ iters) {
  cooperative_groups::grid_group grid = cooperative_groups::this_grid();
  __shared__ double2 sh[SLAB > STEP_LDS ? SLAB : STEP_LDS];
  int rev = 0, it = 0;
  while (it < maxit) {
    nc_z_phase(ws, insts, zoff, rev, sh);
    grid.sync();
    for (int64_t b = blockIdx.x; b < n_items; b += gridDim.x) ncp_step_item(b, insts, items, rev, ws, zoff, part, sh);
    grid.sync();
    for (int64_t k = blockIdx.x; k < n; k += gridDim.x) instance_sum(k, off, part, rnorm);
    grid.sync();
    ++it;
    rev ^= 1;
    double mx = 0.0;
    for (int k = 0; k < n; ++k) mx = fmax(mx, rnorm[k]);
    if (sqrt(mx) < tol) break;
  }
  if (rev) {
    for (int k = 0; k < n; ++k) {
      const apy_mp2_nc_instance I = insts[k];
      const int64_t len = npair(I.O) * npair(I.V);
      const double2* src = (const double2*)I.x_new;
      double2* dst = (double2*)I.x;
      for (int64_t e = blockIdx.x * (int64_t)SBLK + threadIdx.x; e < len; e += (int64_t)gridDim.x * SBLK)
        dst[e] = src[e];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *iters = it;
}

// p < q of the packed pair P of N: a float root, off by one at most at these sizes, and a correction.
__device__ inline void pdec_near(int64_t P, int N, int& p, int& q) {
  const float b = 2.0f * (float)N - 1.0f;
  const int64_t d = (int64_t)(2 * N - 1) * (2 * N - 1) - 8 * P;
  int pp = min(max((int)((b - sqrtf((float)(d > 0 ? d : 0))) * 0.5f), 0), N - 2);
  while (pp > 0 && prow(pp, N) > P) --pp;
  while (pp < N - 2 && prow(pp + 1, N) <= P) ++pp;
  p = pp;
  q = (int)(P - prow(pp, N)) + pp + 1;
}

// energy[k] = scale * sum_dense w_k x_k = 4 scale * sum_(i<j, a<b) w_k x_k (w and x
// antisymmetric), in two fixed-order passes: EN_B partial sums per instance
// (blockIdx.y = instance), then one block per instance adds its partials.  A pair index is one float root
// (a division and a double root an element took 90 us for 36 instances of O 14-18 V 54-66, 53 us so).  Rows
// of BLK pairs (ab) and more are cut where half the blocks would have none (45 rows: 13.2 us whole, 15.8 cut); of shorter ones a block takes
// several side by side, a thread keeping its pair (one row a block at a time: O=2 V=200, two instances, 60 us,
// 10 us so; O=68 V=12, four, 62 us, 17 us so).
__global__ __launch_bounds__(BLK) void nc_energy_partial(const apy_mp2_nc_instance* __restrict__ insts, int use_x_new,
                                                         double2* __restrict__ epart) {
  __shared__ double2 red[BLK];
  const apy_mp2_nc_instance I = insts[blockIdx.y];
  const double2* w = (const double2*)I.w;
  const double2* x = (const double2*)(use_x_new ? I.x_new : I.x);
  const int64_t O = I.O, V = I.V, Pv = npair(V), Po = npair(O);
  double2 acc = make_double2(0.0, 0.0);
  if (w && Po > 0 && Pv >= BLK) {
    const int64_t cuts = 2 * Po <= EN_B ? (Pv + BLK - 1) / BLK : 1, len = cuts > 1 ? BLK : Pv;
    for (int64_t u = blockIdx.x; u < Po * cuts; u += EN_B) {
      const int64_t r = u / cuts, p0 = (u - r * cuts) * len;
      int i, j;
      pdec_near(r, (int)O, i, j);
      const double2* wr = w + (i * O + j) * V * V;
      const double2* xr = x + r * Pv;
      for (int64_t P = p0 + threadIdx.x; P < min(p0 + len, Pv); P += BLK) {
        int a, b;
        pdec_near(P, (int)V, a, b);
        cfma(acc, wr[a * V + b], xr[P]);
      }
    }
  } else if (w && Po > 0 && Pv > 0) {
    const int pv = (int)Pv, rows = BLK / pv, row = threadIdx.x / pv, P = threadIdx.x % pv;
    int a, b;
    pdec_near(P, (int)V, a, b);
    for (int64_t r = (int64_t)blockIdx.x * rows + row; row < rows && r < Po; r += (int64_t)EN_B * rows) {
      int i, j;
      pdec_near(r, (int)O, i, j);
      cfma(acc, w[((i * O + j) * V + a) * V + b], x[r * Pv + P]);
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int q = BLK / 2; q > 0; q >>= 1) {
    if ((int)threadIdx.x < q) {
      red[threadIdx.x].x += red[threadIdx.x + q].x;
      red[threadIdx.x].y += red[threadIdx.x + q].y;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) epart[(int64_t)blockIdx.y * EN_B + blockIdx.x] = red[0];
}

__global__ __launch_bounds__(EN_B) void nc_energy_final(const double2* __restrict__ epart, double scale,
                                                       double2* __restrict__ out) {
  __shared__ double2 red[EN_B];
  red[threadIdx.x] = epart[(int64_t)blockIdx.x * EN_B + threadIdx.x];
  __syncthreads();
  for (int q = EN_B / 2; q > 0; q >>= 1) {
    if ((int)threadIdx.x < q) {
      red[threadIdx.x].x += red[threadIdx.x + q].x;
      red[threadIdx.x].y += red[threadIdx.x + q].y;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = make_double2(4.0 * scale * red[0].x, 4.0 * scale * red[0].y);
}

__global__ __launch_bounds__(BLK) void t2_pack_kernel(int64_t O, int64_t V, const double2* __restrict__ dense,
                                                      double2* __restrict__ packed) {
  const int64_t Pv = npair(V), total = npair(O) * Pv;
  for (int64_t t = blockIdx.x * (int64_t)BLK + threadIdx.x; t < total; t += (int64_t)gridDim.x * BLK) {
    int64_t i, j, a, b;
    pdec(t / Pv, O, i, j);
    pdec(t % Pv, V, a, b);
    packed[t] = dense[((i * O + j) * V + a) * V + b];
  }
}

// One workgroup per (pair i<j or diagonal i, 32 x 32 tile pair A <= B of the virtual plane): the packed
// tile is read once and its four images written along b, the transposed two through LDS (an element at a
// time, with its pair index from four divisions, 41 us at O=20 V=120, 92 MB written).
__global__ __launch_bounds__(BLK) void t2_unpack_kernel(int64_t O, int64_t V, int nt, const double2* __restrict__ packed,
                                                        double2* __restrict__ dense) {
  __shared__ double2 T[32][33];
  const int64_t Pv = npair(V), Po = npair(O), ntp = (int64_t)nt * (nt + 1) / 2;
  const int64_t r = blockIdx.x / ntp;
  int t = (int)(blockIdx.x % ntp), ta = 0;
  while (t >= nt - ta) { t -= nt - ta; ++ta; }
  const int64_t a0 = 32 * (int64_t)ta, b0 = 32 * (int64_t)(ta + t);
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const double2 zero = make_double2(0.0, 0.0);
  auto at = [&](int64_t i, int64_t j, int64_t a, int64_t b) -> double2& { return dense[((i * O + j) * V + a) * V + b]; };
  if (r >= Po) {                                        // i == j: zeros
    const int64_t i = r - Po;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t a = a0 + ty + 8 * k, b = b0 + tx, at_ = a0 + tx, bt = b0 + ty + 8 * k;
      if (a < V && b < V) at(i, i, a, b) = zero;
      if (t > 0 && bt < V && at_ < V) at(i, i, bt, at_) = zero;
    }
    return;
  }
  int64_t i, j;
  pdec(r, O, i, j);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t a = a0 + ty + 8 * k, b = b0 + tx;
    double2 v = zero;
    if (b < V && a < b) v = packed[r * Pv + pidx(a, b, V)];
    T[ty + 8 * k][tx] = v;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t a = a0 + ty + 8 * k, b = b0 + tx;     // rows of the tile, b along the lanes
    double2 v = T[ty + 8 * k][tx];
    if (t == 0 && a > b) v = T[tx][ty + 8 * k], v = make_double2(-v.x, -v.y);
    if (a < V && b < V) {
      at(i, j, a, b) = v;
      at(j, i, a, b) = a == b ? zero : make_double2(-v.x, -v.y);
    }
    if (t > 0) {                                         // the mirrored tile, a along the lanes
      const int64_t br = b0 + ty + 8 * k, ac = a0 + tx;
      const double2 u = T[tx][ty + 8 * k];
      if (br < V && ac < V) {
        at(i, j, br, ac) = make_double2(-u.x, -u.y);
        at(j, i, br, ac) = u;
      }
    }
  }
}

}  // namespace

extern "C" {

int64_t apy_t2_packed_length(int64_t O, int64_t V) {
  if (O < 0 || V < 0) return 0;
  return npair(O) * npair(V);
}

int apy_t2_pack(int64_t O, int64_t V, const void* dense, void* packed, void* stream) {
  if (O < 0 || V < 0 || !dense || !packed || dense == packed) return APY_E_ARG;
  const int64_t total = npair(O) * npair(V);
  if (total == 0) return APY_OK;
  t2_pack_kernel<<<apy_grid1d(total, 1 << 20), BLK, 0, (hipStream_t)stream>>>(O, V, (const double2*)dense,
                                                                              (double2*)packed);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

int apy_t2_unpack(int64_t O, int64_t V, const void* packed, void* dense, void* stream) {
  if (O < 0 || V < 0 || !dense || !packed || dense == packed) return APY_E_ARG;
  if (O * V == 0) return APY_OK;
  const int64_t nt = (V + 31) / 32, grid = (npair(O) + O) * (nt * (nt + 1) / 2);
  if (grid > 0x7fffffffLL) return APY_E_ARG;
  t2_unpack_kernel<<<(unsigned)grid, BLK, 0, (hipStream_t)stream>>>(O, V, (int)nt, (const double2*)packed,
                                                                    (double2*)dense);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

size_t apy_mp2_nc_batched_workspace(int n, const apy_mp2_nc_instance* inst) {
  if (n < 1 || !inst) return 0;
  int64_t ze = 0;
  const int64_t zi = count_zitems(n, inst, &ze);
  return layout(n, count_items(n, inst), zi, ze).total;
}

int apy_mp2_nc_batched_setup(int n, const apy_mp2_nc_instance* inst, void* workspace, size_t ws_bytes,
                             int64_t* n_items, void* stream) {
  if (n < 1 || n > 65535 || !inst || !n_items) return APY_E_ARG;
  for (int k = 0; k < n; ++k) {
    const apy_mp2_nc_instance& I = inst[k];
    if (I.O < 1 || I.V < 1 || I.O > 32767 || I.V > 32767 || !I.fock || !I.eps || !I.drv || !I.x || !I.x_new ||
        I.x == I.x_new)
      return APY_E_ARG;
  }
  const int64_t items = count_items(n, inst);
  int64_t zelems = 0;
  const int64_t zitems = count_zitems(n, inst, &zelems);
  if (items < 1 || items > 2147483647 || zitems > 2147483647) return APY_E_ARG;
  const WsLayout L = layout(n, items, zitems, zelems);
  if (!workspace || ws_bytes < L.total) return APY_E_WORKSPACE;
  std::vector<Item> it;
  it.reserve(items);
  std::vector<ZItem> zit;
  zit.reserve(zitems);
  std::vector<int64_t> off(n + 1, 0), zoff(n + 1, 0);
  for (int k = 0; k < n; ++k) {
    off[k] = (int64_t)it.size();
    zoff[k + 1] = zoff[k];
    if (inst[k].O < 2 || inst[k].V < 2) continue;
    const int32_t nt = (int32_t)ntiles(inst[k].V);
    const int64_t Pv = npair(inst[k].V);
    for (int32_t p = 0; p < (int32_t)npair(inst[k].O); ++p)
      for (int32_t ta = 0; ta < nt; ++ta)
        for (int32_t tb = ta; tb < nt; ++tb) it.push_back(Item{k, p, ta, tb});
    for (int64_t p0 = 0; p0 < Pv; p0 += zspan(inst[k].O))
      for (int64_t r = 0; r < zrows(inst[k].O); ++r)
        zit.push_back(ZItem{k, (int32_t)p0, (int32_t)(r * (BLK / 64)), 0});
    zoff[k + 1] = zoff[k] + npair(inst[k].O) * Pv;
  }
  off[n] = (int64_t)it.size();
  Header h{n, items, zitems, (int64_t)L.zitem, (int64_t)L.z};
  char* w = (char*)workspace;
  hipStream_t st = (hipStream_t)stream;
  // pageable sources: each copy returns once the host buffer has been read
  APY_HIP_TRY(hipMemcpyAsync(w, &h, sizeof(h), hipMemcpyHostToDevice, st));
  APY_HIP_TRY(hipMemcpyAsync(w + L.inst, inst, n * sizeof(apy_mp2_nc_instance), hipMemcpyHostToDevice, st));
  APY_HIP_TRY(hipMemcpyAsync(w + L.item, it.data(), items * sizeof(Item), hipMemcpyHostToDevice, st));
  APY_HIP_TRY(hipMemcpyAsync(w + L.off, off.data(), (n + 1) * sizeof(int64_t), hipMemcpyHostToDevice, st));
  APY_HIP_TRY(hipMemcpyAsync(w + L.zoff, zoff.data(), (n + 1) * sizeof(int64_t), hipMemcpyHostToDevice, st));
  if (zitems > 0)
    APY_HIP_TRY(hipMemcpyAsync(w + L.zitem, zit.data(), zitems * sizeof(ZItem), hipMemcpyHostToDevice, st));
  APY_HIP_TRY(hipStreamSynchronize(st));
  *n_items = items;
  return APY_OK;
}

int apy_mp2_nc_batched_step(int n, int64_t n_items, int reverse, void* rnorm, void* workspace, void* stream) {
  if (n < 1 || n > 65535 || n_items < 1 || n_items > 2147483647 || !rnorm || !workspace) return APY_E_ARG;
  const WsLayout L = layout(n, n_items);
  char* w = (char*)workspace;
  hipStream_t st = (hipStream_t)stream;
  double* part = (double*)(w + L.part);
  const auto* insts = (const apy_mp2_nc_instance*)(w + L.inst);
  const int64_t* zoff = (const int64_t*)(w + L.zoff);
  // the W work list is grid-strided over at most 4096 workgroups
  nc_z_kernel<<<(unsigned)std::min<int64_t>(n_items, 4096), BLK, 0, st>>>(w, insts, zoff, reverse);
  APY_LAUNCH_CHECK();
  ncp_step_kernel<<<(unsigned)n_items, SBLK, 0, st>>>(insts, (const Item*)(w + L.item), reverse, w, zoff, part);
  APY_LAUNCH_CHECK();
  per_instance_sum<<<(unsigned)n, BLK, 0, st>>>((const int64_t*)(w + L.off), part, (double*)rnorm);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

int apy_mp2_nc_batched_solve(int n, int64_t n_items, double tol, int maxit, void* rnorm, void* iterations,
                             void* workspace, void* stream) {
  if (n < 1 || n > 65535 || n_items < 1 || n_items > 2147483647 || maxit < 1 || !(tol >= 0.0) || !rnorm ||
      !iterations || !workspace)
    return APY_E_ARG;
  const WsLayout L = layout(n, n_items);
  char* w = (char*)workspace;
  int dev = 0, ncu = 0, per_cu = 0;
  APY_HIP_TRY(hipGetDevice(&dev));
  APY_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  APY_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, nc_persistent_kernel, SBLK, 0));
  if (per_cu < 1 || ncu < 1) return APY_E_HIP;
  // every workgroup resident at once (a cooperative launch refuses a larger grid), and no more of them than the
  // items pay for: a grid barrier takes about 0.08 us a workgroup, three an iteration.  ms a solve at 1 / 2 / 3 a
  // CU: O=10 V=4, 1080 items 0.53 / 0.89 / 1.26; O=10 V=38, 3240 items 1.23 / 1.48 / 1.90; 36 instances of
  // O 14-18 V 54-66, 15000 items 5.89 / 4.62 / 4.70.
  per_cu = std::min(per_cu, n_items > 24 * (int64_t)ncu ? 2 : 1);
  const int64_t grid = std::min<int64_t>((int64_t)per_cu * ncu, n_items);
  const apy_mp2_nc_instance* insts = (const apy_mp2_nc_instance*)(w + L.inst);
  const Item* items = (const Item*)(w + L.item);
  const int64_t* off = (const int64_t*)(w + L.off);
  const int64_t* zoff = (const int64_t*)(w + L.zoff);
  double* part = (double*)(w + L.part);
  double* rn = (double*)rnorm;
  int64_t* it = (int64_t*)iterations;
  void* args[] = {&w, &insts, &items, &off, &zoff, &part, &rn, &n, &n_items, &tol, &maxit, &it};
  APY_HIP_TRY(hipLaunchCooperativeKernel((const void*)nc_persistent_kernel, dim3((unsigned)grid), dim3(SBLK), args, 0,
                                         (hipStream_t)stream));
  return APY_OK;
}

int apy_mp2_nc_batched_energy(int n, int64_t n_items, int use_x_new, double scale, void* energy,
                              void* workspace, void* stream) {
  if (n < 1 || n > 65535 || n_items < 1 || !energy || !workspace) return APY_E_ARG;
  const WsLayout L = layout(n, n_items);
  char* w = (char*)workspace;
  hipStream_t st = (hipStream_t)stream;
  double2* epart = (double2*)(w + L.epart);
  nc_energy_partial<<<dim3(EN_B, (unsigned)n), BLK, 0, st>>>((const apy_mp2_nc_instance*)(w + L.inst), use_x_new,
                                                              epart);
  APY_LAUNCH_CHECK();
  nc_energy_final<<<(unsigned)n, EN_B, 0, st>>>(epart, scale, (double2*)energy);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

}  // extern "C"
