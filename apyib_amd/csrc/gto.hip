// Electron-repulsion integrals over contracted Cartesian Gaussians on the GPU (McMurchie-Davidson),
// the AO integrals psi4's MintsHelper gives the reference (hamiltonian.py:33 ao_eri, analytic_aats.py:94
// mo_tei_deriv1 before its MO transform).  A function is one or two terms sharing a centre and the
// exponents, sum_term sum_p c_term,p x^l y^m z^n exp(-a_p r^2): an s/p basis function is one term, its
// derivative with respect to its centre two (l+1 and l-1).  One workgroup per quartet of shells; every
// primitive quartet is expanded in Hermite Gaussians (E coefficients), the Coulomb integrals R_tuv come
// from the Boys function by the Hermite recursion, and the quartet sum is
//   (ab|cd) = 2 pi^(5/2) / (p q sqrt(p+q)) sum_tuv E^ab_tuv sum_t'u'v' (-1)^(t'+u'+v') E^cd_t'u'v'
//             R_(t+t')(u+u')(v+v')(alpha, P - Q).
#include "common.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace {

constexpr int LF = APY_GTO_MAXL;          // largest angular momentum of one term along all axes together
constexpr int LQ = 3 * 2 + LF;            // largest total of a quartet: three d functions and one f term
constexpr int NE = 2 * LF + 1;            // E_t^{ij}, t <= i + j
constexpr int NRB = 64;                   // (Lx+1)(Ly+1)(Lz+1) <= 64 for Lx+Ly+Lz <= 9

// F_n(T), n = 0..nmax, by the series e^-T sum_k (2T)^k / ((2n+1)(2n+3)...(2n+2k+1)) for the top order and
// downward recursion F_n = (2T F_{n+1} + e^-T) / (2n+1) (all terms positive: no cancellation).
__device__ void boys_series(int nmax, double T, double* F) {
  double term = 1.0 / (2 * nmax + 1), sum = term;
  for (int k = 1; k < 400; ++k) {
    term *= 2.0 * T / (2 * nmax + 2 * k + 1);
    sum += term;
    if (term < 1e-17 * sum) break;
  }
  const double e = exp(-T);
  F[nmax] = e * sum;
  for (int n = nmax - 1; n >= 0; --n) F[n] = (2.0 * T * F[n + 1] + e) / (2 * n + 1);
}

// F_n(T_k), T_k = k / BOYS_DENS below BOYS_TMAX, orders 0..BOYS_NORD-1: filled once per device by
// boys_table_kernel (boys_series at every grid point), read by boys_fn.
constexpr int BOYS_NORD = LQ + 7;
constexpr int BOYS_DENS = 20;
constexpr double BOYS_TMAX = 36.0;
constexpr int BOYS_NGRID = 36 * BOYS_DENS + 2;
__device__ double g_boys[BOYS_NGRID][BOYS_NORD];

__global__ __launch_bounds__(256) void boys_table_kernel() {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= BOYS_NGRID) return;
  double F[BOYS_NORD];
  boys_series(BOYS_NORD - 1, (double)k / BOYS_DENS, F);
  for (int n = 0; n < BOYS_NORD; ++n) g_boys[k][n] = F[n];
}

// F_n(T), n = 0..nmax (nmax <= LQ).  Below BOYS_TMAX the seven-term Taylor expansion about the nearest grid
// point (dF_n/dT = -F_{n+1}):  F_n(T) = sum_j F_{n+j}(T_k) (T_k - T)^j / j!,  |T_k - T| <= 0.025, remainder
// below 1e-15 F_n.  Above, F_0 from erf and upward recursion F_{n+1} = ((2n+1) F_n - e^-T) / (2T) (e^-T is
// then far below every (2n+1) F_n: no cancellation).
__device__ void boys_fn(int nmax, double T, double* F) {
  if (T < BOYS_TMAX) {
    const double x = T * BOYS_DENS;
    const int k = (int)(x + 0.5);
    const double d = ((double)k - x) / BOYS_DENS;
    const double* g = g_boys[k];
    for (int n = 0; n <= nmax; ++n) {
      double f = g[n + 6];
      f = g[n + 5] + d * f * (1.0 / 6.0);
      f = g[n + 4] + d * f * (1.0 / 5.0);
      f = g[n + 3] + d * f * (1.0 / 4.0);
      f = g[n + 2] + d * f * (1.0 / 3.0);
      f = g[n + 1] + d * f * (1.0 / 2.0);
      F[n] = g[n] + d * f;
    }
  } else {
    const double e = exp(-T);
    F[0] = 0.5 * sqrt(M_PI / T) * erf(sqrt(T));
    for (int n = 0; n < nmax; ++n) F[n + 1] = ((2 * n + 1) * F[n] - e) / (2.0 * T);
  }
}

// E_t^{ij} (t = 0..i+j) along one axis for exponents a, b and Q = A - B (i, j <= LF):
//   E^{00}_0 = exp(-ab/(a+b) Q^2),
//   E^{i+1,j}_t = E^{ij}_{t-1} / 2p + X_PA E^{ij}_t + (t+1) E^{ij}_{t+1},   X_PA = -b Q / p,
//   E^{i,j+1}_t = E^{ij}_{t-1} / 2p + X_PB E^{ij}_t + (t+1) E^{ij}_{t+1},   X_PB =  a Q / p.
__device__ void herm_E(int i, int j, double Q, double a, double b, double* out) {
  const double p = a + b, h = 0.5 / p, xpa = -b * Q / p, xpb = a * Q / p;
  double e[LF + 1][LF + 1][NE];
  for (int ii = 0; ii <= i; ++ii)
    for (int jj = 0; jj <= j; ++jj)
      for (int t = 0; t < NE; ++t) e[ii][jj][t] = 0.0;
  e[0][0][0] = exp(-a * b / p * Q * Q);
  for (int ii = 0; ii <= i; ++ii) {
    for (int jj = 0; jj <= j; ++jj) {
      if (ii == 0 && jj == 0) continue;
      const int pi = ii > 0 ? ii - 1 : ii, pj = ii > 0 ? jj : jj - 1;
      const double x = ii > 0 ? xpa : xpb;
      for (int t = 0; t <= ii + jj; ++t) {
        double v = x * e[pi][pj][t];
        if (t > 0) v += h * e[pi][pj][t - 1];
        if (t + 1 <= pi + pj) v += (t + 1) * e[pi][pj][t + 1];
        e[ii][jj][t] = v;
      }
    }
  }
  for (int t = 0; t <= i + j; ++t) out[t] = e[i][j][t];
}

__device__ inline int lsum(const int* l) { return l[0] + l[1] + l[2]; }

#define kNaN __longlong_as_double(0x7ff8000000000000LL)

// A table entry inside the kernels' limits (centre index below ncen, 1..APY_GTO_MAXPRIM primitives, one or
// two terms of angular momentum <= LF); entries outside them give NaN, never an out-of-bounds access.
__device__ bool gto_ok(const apy_gto& g, int64_t ncen) {
  if (g.atom < 0 || g.atom >= ncen || g.nprim < 1 || g.nprim > APY_GTO_MAXPRIM || g.nterm < 1 || g.nterm > 2)
    return false;
  for (int t = 0; t < g.nterm; ++t)
    if (g.lmn[t][0] < 0 || g.lmn[t][1] < 0 || g.lmn[t][2] < 0 || lsum(g.lmn[t]) > LF) return false;
  return true;
}

__host__ __device__ inline int apy_oei_ncomp(int which) {
  if (which <= 0 || which > 31) return 0;
  return (which & 1) + ((which >> 1) & 1) + ((which >> 2) & 1) + 3 * ((which >> 3) & 1) + 3 * ((which >> 4) & 1);
}

// Hermite Coulomb integrals R^0_tuv(alpha, PQ) for t <= Lt[0], u <= Lt[1], v <= Lt[2] (L = the sum, <= LQ;
// (Lt[0]+1)(Lt[1]+1)(Lt[2]+1) <= NRB), from F = F_n(alpha |PQ|^2), n <= L:
//   R^n_000 = (-2 alpha)^n F_n,  R^n_{t+1,u,v} = t R^{n+1}_{t-1,u,v} + PQ_x R^{n+1}_{tuv}  (and alike for u, v).
// Level n is built from level n + 1 in the two alternating buffers Rb; the result is Rb[returned index]
// at [t sy + u sz + v], sz = Lt[2]+1, sy = (Lt[1]+1) sz.
__device__ int herm_R(int L, const int* Lt, double alpha, const double* PQ, const double* F, double (*Rb)[NRB]) {
  const int sz = Lt[2] + 1, sy = (Lt[1] + 1) * sz;
  int cur = 0;
  for (int n = L; n >= 0; --n) {
    const int nxt = cur ^ 1;  // level n + 1 lives in Rb[cur]
    double* out = Rb[nxt];
    const double* prev = Rb[cur];
    const int lim = L - n;
    for (int t = 0; t <= Lt[0]; ++t)
      for (int u = 0; u <= Lt[1]; ++u)
        for (int v = 0; v <= Lt[2]; ++v) {
          if (t + u + v > lim) continue;
          double r;
          if (t > 0) {
            r = PQ[0] * prev[(t - 1) * sy + u * sz + v];
            if (t > 1) r += (t - 1) * prev[(t - 2) * sy + u * sz + v];
          } else if (u > 0) {
            r = PQ[1] * prev[u * sz - sz + v];
            if (u > 1) r += (u - 1) * prev[(u - 2) * sz + v];
          } else if (v > 0) {
            r = PQ[2] * prev[v - 1];
            if (v > 1) r += (v - 1) * prev[v - 2];
          } else {
            double s = 1.0;
            for (int k = 0; k < n; ++k) s *= -2.0 * alpha;
            r = s * F[n];
          }
          out[t * sy + u * sz + v] = r;
        }
    cur = nxt;
  }
  return cur;
}

// x = hi (hi + 1) / 2 + lo with 0 <= lo <= hi: the row-packed lower triangle.
__device__ inline void tri_split(int64_t x, int64_t& hi, int64_t& lo) {
  int64_t h = (int64_t)((sqrt(8.0 * (double)x + 1.0) - 1.0) * 0.5);
  while (h * (h + 1) / 2 > x) --h;
  while ((h + 1) * (h + 2) / 2 <= x) ++h;
  hi = h;
  lo = x - h * (h + 1) / 2;
}

// Which permutational symmetry of the real integrals (ab|cd) the launch uses: ERI_ALL when the four
// tables are one table (8 images per computed quartet: i >= j, k >= l, (ij) >= (kl)), ERI_KET when the
// ket tables are one table ((ab|cd) = (ab|dc): 2 images, k >= l), ERI_NONE otherwise.
enum EriSym { ERI_NONE = 0, ERI_KET = 1, ERI_ALL = 2 };

struct EriTab {
  const apy_gto* f[4];
  int64_t n[4];
};

// One primitive quartet of (a b | c d): terms (ta, tb, tc, td), primitives (pa, pb, pc, pd), centres ca..cd,
// qab = A - B, qcd = C - D.  The caller has checked the table entries and that the quartet's total angular
// momentum is at most LQ.
__device__ double eri_prim(const apy_gto& A, const apy_gto& B, const apy_gto& C, const apy_gto& D, int ta, int tb,
                           int tc, int td, int pa, int pb, int pc, int pd, const double* ca, const double* cb,
                           const double* cc, const double* cd, const double* qab, const double* qcd) {
  const int* la = A.lmn[ta];
  const int* lb = B.lmn[tb];
  const int* lc = C.lmn[tc];
  const int* ld = D.lmn[td];
  int L1[3], L2[3], Lt[3];
  for (int x = 0; x < 3; ++x) { L1[x] = la[x] + lb[x]; L2[x] = lc[x] + ld[x]; Lt[x] = L1[x] + L2[x]; }
  const int L = Lt[0] + Lt[1] + Lt[2];
  const int sz = Lt[2] + 1, sy = (Lt[1] + 1) * sz;  // R index (t, u, v) -> t sy + u sz + v
  const double a = A.exps[pa], b = B.exps[pb], p = a + b;
  const double c = C.exps[pc], d = D.exps[pd], q = c + d;
  double Eab[3][NE], Ecd[3][NE], PQ[3];
  for (int x = 0; x < 3; ++x) {
    herm_E(la[x], lb[x], qab[x], a, b, Eab[x]);
    herm_E(lc[x], ld[x], qcd[x], c, d, Ecd[x]);
    PQ[x] = (a * ca[x] + b * cb[x]) / p - (c * cc[x] + d * cd[x]) / q;
  }
  const double alpha = p * q / (p + q);
  double F[LQ + 1];
  boys_fn(L, alpha * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]), F);
  double Rb[2][NRB];
  const double* R = Rb[herm_R(L, Lt, alpha, PQ, F, Rb)];
  double val = 0.0;
  for (int t = 0; t <= L1[0]; ++t)
    for (int u = 0; u <= L1[1]; ++u)
      for (int v = 0; v <= L1[2]; ++v) {
        const double e1 = Eab[0][t] * Eab[1][u] * Eab[2][v];
        double s2 = 0.0;
        for (int tt = 0; tt <= L2[0]; ++tt)
          for (int uu = 0; uu <= L2[1]; ++uu)
            for (int vv = 0; vv <= L2[2]; ++vv) {
              const double e2 = Ecd[0][tt] * Ecd[1][uu] * Ecd[2][vv];
              const double sg = ((tt + uu + vv) & 1) ? -1.0 : 1.0;
              s2 += sg * e2 * R[(t + tt) * sy + (u + uu) * sz + (v + vv)];
            }
        val += e1 * s2;
      }
  const double pref0 = 2.0 * M_PI * M_PI * sqrt(M_PI);
  return A.coefs[ta][pa] * B.coefs[tb][pb] * C.coefs[tc][pc] * D.coefs[td][pd] * pref0 / (p * q * sqrt(p + q)) * val;
}

// Whether every term combination of the quartet stays within the total angular momentum LQ.
__device__ bool quartet_ok(const apy_gto& A, const apy_gto& B, const apy_gto& C, const apy_gto& D) {
  for (int ta = 0; ta < A.nterm; ++ta)
    for (int tb = 0; tb < B.nterm; ++tb)
      for (int tc = 0; tc < C.nterm; ++tc)
        for (int td = 0; td < D.nterm; ++td)
          if (lsum(A.lmn[ta]) + lsum(B.lmn[tb]) + lsum(C.lmn[tc]) + lsum(D.lmn[td]) > LQ) return false;
  return true;
}

// The elements one by one, a wavefront each (wave-uniform control flow): the lanes split the element's
// (term, primitive) quartets and a fixed-order butterfly sums them; lane 0 writes the value to every
// image of the element under the launch's symmetry.  A table entry outside the limits (angular
// momentum, primitive count, term count, atom index) gives NaN before any indexing.
__device__ __forceinline__ void eri_elements(int64_t ngeom, int64_t natom, const double* __restrict__ centers,
                                             const EriTab& T, int sym, double2* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t na = T.n[0], nb = T.n[1], nc = T.n[2], nd = T.n[3], full = na * nb * nc * nd;
  const int64_t pc = nc * (nc + 1) / 2;
  const int64_t per = sym == ERI_ALL ? pc * (pc + 1) / 2 : sym == ERI_KET ? na * nb * pc : full;
  const int64_t total = ngeom * per;
  const int64_t nwave = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t e = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6; e < total; e += nwave) {
    const int64_t g = e / per, r = e % per;
    int64_t i, j, k, l;
    if (sym == ERI_ALL) {
      int64_t bra, ket;
      tri_split(r, bra, ket);
      tri_split(bra, i, j);
      tri_split(ket, k, l);
    } else if (sym == ERI_KET) {
      tri_split(r % pc, k, l);
      j = (r / pc) % nb;
      i = r / (pc * nb);
    } else {
      l = r % nd; k = (r / nd) % nc; j = (r / (nd * nc)) % nb; i = r / (nd * nc * nb);
    }
    double2* o = out + g * full;
    // element (p, q, s, t) of the [na][nb][nc][nd] output
    auto at = [&](int64_t p, int64_t q, int64_t s2, int64_t t) { return ((p * nb + q) * nc + s2) * nd + t; };
    auto put = [&](double v) {
      const double2 w = make_double2(v, 0.0);
      o[at(i, j, k, l)] = w;
      if (sym == ERI_NONE) return;
      o[at(i, j, l, k)] = w;
      if (sym == ERI_KET) return;
      o[at(j, i, k, l)] = w;
      o[at(j, i, l, k)] = w;
      o[at(k, l, i, j)] = w;
      o[at(l, k, i, j)] = w;
      o[at(k, l, j, i)] = w;
      o[at(l, k, j, i)] = w;
    };
    const apy_gto& A = T.f[0][i];
    const apy_gto& B = T.f[1][j];
    const apy_gto& C = T.f[2][k];
    const apy_gto& D = T.f[3][l];
    if (!gto_ok(A, natom) || !gto_ok(B, natom) || !gto_ok(C, natom) || !gto_ok(D, natom) ||
        !quartet_ok(A, B, C, D)) {
      if (lane == 0) put(kNaN);
      continue;
    }
    const double* cen = centers + 3 * natom * g;
    const double* ca = cen + 3 * A.atom;
    const double* cb = cen + 3 * B.atom;
    const double* cc = cen + 3 * C.atom;
    const double* cd = cen + 3 * D.atom;
    const double qab[3] = {ca[0] - cb[0], ca[1] - cb[1], ca[2] - cb[2]};
    const double qcd[3] = {cc[0] - cd[0], cc[1] - cd[1], cc[2] - cd[2]};
    // quartet w = ((((((ta nbt + tb) nct + tc) ndt + td) npa + pa) npb + pb) npc + pc) npd + pd
    const int nt = A.nterm * B.nterm * C.nterm * D.nterm;
    const int np = A.nprim * B.nprim * C.nprim * D.nprim;
    double acc = 0.0;
    for (int w = lane; w < nt * np; w += 64) {
      int x = w;
      const int pd = x % D.nprim; x /= D.nprim;
      const int pc = x % C.nprim; x /= C.nprim;
      const int pb = x % B.nprim; x /= B.nprim;
      const int pa = x % A.nprim; x /= A.nprim;
      const int td = x % D.nterm; x /= D.nterm;
      const int tc = x % C.nterm; x /= C.nterm;
      const int tb = x % B.nterm; x /= B.nterm;
      const int ta = x;
      acc += eri_prim(A, B, C, D, ta, tb, tc, td, pa, pb, pc, pd, ca, cb, cc, cd, qab, qcd);
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) put(acc);
  }
}

__global__ __launch_bounds__(256) void eri_element_kernel(int64_t ngeom, int64_t natom,
                                                          const double* __restrict__ centers, EriTab T, int sym,
                                                          double2* __restrict__ out) {
  eri_elements(ngeom, natom, centers, T, sym, out);
}

// Functions that sit next to each other in a table on one centre with the same exponents (an sp or a d
// shell) form a group of up to EG.  A group quartet shares every primitive quartet's Boys functions and
// Hermite Coulomb integrals, which is why the work is split by group quartets and not by elements: at
// H2O2/6-31G* (34 functions, 2.1e6 primitive quartets of functions) there are 1.0e5 of groups.
//
// One workgroup computes the (up to EG^4) elements of a group quartet.  The expansion of a bra or ket
// element (ab| in Hermite Gaussians is a list of slots, one for each pair of terms and (t, u, v); primitive
// pairs are taken in batches that fit LDS; per batch
//   1. Hermite E coefficients (a thread per primitive pair, axis and bra power), G_n = pref (-2 alpha)^n F_n
//      and the powers of P - Q (a thread per primitive quartet and order),
//   2. R_tuv = sum_ijk a_ti a_uj a_vk X^(t-2i) Y^(u-2j) Z^(v-2k) G_(t+u+v-i-j-k), a_ti = t!/(i!(t-2i)!2^i)
//      (the Hermite recursion in closed form: every entry on its own, no order of evaluation between them),
//      and the slots' coefficients Lam[pair][slot] = c_a c_b E^x_t E^y_u E^z_v, signs (-1)^(t+u+v) in the ket's,
//   3. H[bra pair][ket element][tuv] += sum over the ket pairs and the element's slots of Lam R,
// and per bra batch acc[element] += sum over the bra pairs and the element's slots of Lam H.  Contracting the
// ket pairs first makes the step that touches every element run once a bra pair instead of once a primitive
// quartet.  Bound by the latency of these short phases, not by bytes or flops: the sums over slots are flat
// loops of two slots by EU primitive pairs side by side (as loops over t, u and v with the products of E in
// them, one sp quartet of three primitives took 165 us, now 50), and 168 registers and 52 KB of LDS keep three
// workgroups on a CU.  H2O2/6-31G*: 5040 us with a wave an element and every expansion redone for each
// quartet of functions, 140 us so.
constexpr int EG = 6;                 // functions of a group
constexpr int EPP = APY_GTO_MAXPRIM * APY_GTO_MAXPRIM;
constexpr int EW = 1536;              // doubles: G, powers and R of a batch
constexpr int EH = EG * EG * EG * EG; // doubles: H (a d,d pair's 35 tuv with its 36 ket elements: 1260)
constexpr int EE = 448;               // doubles: E coefficients of a batch, bra or ket (f,f: 336 a pair)
constexpr int ES = 384;               // slots by primitive pairs of a batch, bra or ket (d,d: 342 a pair; one
                                      // element: at most 108)
constexpr int ESUM = 2048;            // entries of the table of sums of two tuv (d,d against d,d: 1225)
constexpr int EU = 4;                 // primitive pairs side by side
constexpr int EACC = (EG * EG * EG * EG + 255) / 256;
constexpr int ENR = (LQ + 1) * (LQ + 2) * (LQ + 3) / 6;   // tuv with t + u + v <= LQ
constexpr int ETAB = 4096;            // group starts that LDS holds, all tables together

// index of (t, u, v) in order of t + u + v: the entries up to a total L come first
__host__ __device__ inline int tuv_index(int t, int u, int v) {
  const int r = u + v, s = t + r;
  return s * (s + 1) * (s + 2) / 6 + r * (r + 1) / 2 + v;
}
__host__ __device__ inline int tuv_count(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// w / d and w % d for 0 <= w < 2^16 and one d of a workgroup: a multiplication instead of the ~40
// instructions of an integer division (several a work item, as long as the item's own sums)
struct SmallDiv {
  unsigned inv;
  int d;
  __device__ explicit SmallDiv(int n) : inv(n > 1 ? 0xffffffffu / (unsigned)n + 1u : 0u), d(n) {}
  __device__ int div(int w) const { return d > 1 ? (int)__umulhi((unsigned)w, inv) : w; }
  __device__ int mod(int w) const { return w - div(w) * d; }
};

// an LDS value that every thread reads alike, in a scalar register
__device__ inline int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// A slot of an element: the places of E^x_t, E^y_u and E^z_v in a primitive pair's E block and the two
// functions' coefficient rows (2 member + term); ca = 255 pads an element to an even count.
struct EriSlot {
  uint16_t e[3];
  uint8_t ca, cb;
};

struct EriShared {
  double W[EW], H[EH], E[2][EE], Lam[2][ES];
  double exps[4][APY_GTO_MAXPRIM], cen[4][3], coef[4][EG][2][APY_GTO_MAXPRIM];
  double pair[2][EPP][5];             // of each primitive pair: p = a + b, 1 / p and P
  double herm[LQ + 1][LQ / 2 + 1];    // a_ti
  int16_t slot[2][EG * EG + 1];       // first slot of each element, bra and ket
  int8_t lmn[4][EG][2][3];
  uint8_t nterm[4][EG];
  uint8_t prim[2][EPP][2];            // primitives of pair b (bra) or q (ket)
  uint8_t tuv[ENR][3];
  uint8_t stuv[2][ES];                // tuv index of each slot of the slice
  uint8_t sum[ESUM];                  // tuv index of the sum of a bra and a ket (t, u, v)
  EriSlot rec[2][ES];
  int size[4], nprim[4], L[4], first[4], ngrp[4], nshort[4][2];
};

// Starts of the groups of a table into `start` (start[ngrp] = n) and over the flags of its functions (bit 0: joins
// the one before, bits 1-2: one term of L = 0 or 1) each group's class: L of such a function by itself, else ECLS;
// how many of each class into nshort.  By one wave, 64 functions at a time (by one thread 2 us at 34 functions).
constexpr int ECLS = 2;
__device__ int find_groups(int n, uint8_t* flags, uint16_t* start, int* nshort, int lane) {
  int g = 0, run = 0, ns = 0, np = 0;                  // run: where the functions that join each other began
  for (int base = 0; base < n; base += 64) {
    const int i = base + lane;
    const int f = i < n ? flags[i] : 1, next = i + 1 < n ? flags[i + 1] : 0;
    const unsigned long long cut = __ballot(i == 0 || !(f & 1)), upto = cut & ((2ull << lane) - 1ull);
    const int r = upto ? base + 63 - __clzll((long long)upto) : run;
    const bool first = i < n && (i - r) % EG == 0;
    const unsigned long long firsts = __ballot(first);
    const int cls = next & 1 ? ECLS : f & 2 ? 0 : f & 4 ? 1 : ECLS;
    if (first) {
      const int at = g + __popcll(firsts & ((1ull << lane) - 1ull));
      start[at] = (uint16_t)i;
      flags[at] = (uint8_t)cls;                        // at <= i: read by all lanes above
    }
    ns += __popcll(__ballot(first && cls == 0));
    np += __popcll(__ballot(first && cls == 1));
    g += __popcll(firsts);
    run = __shfl(r, 63, 64);
  }
  if (lane == 0) {
    start[g] = (uint16_t)n;
    nshort[0] = ns;
    nshort[1] = np;
  }
  return g;
}

// E^{ij}_t of one primitive pair and axis for this i and all j <= Lb, into out[(i (Lb+1) + j) nt + t],
// nt = La + Lb + 1, times sgn^t; the recursion of herm_E along one row, in registers.
__device__ void herm_row(int i, int La, int Lb, double Q, double a, double b, double ip, double sgn, double* out) {
  const double h = 0.5 * ip, xpa = -b * Q * ip, xpb = a * Q * ip;
  double e[NE + 1];
#pragma unroll
  for (int t = 0; t <= NE; ++t) e[t] = 0.0;
  e[0] = exp(-a * b * ip * Q * Q);
  auto raise = [&](double x) {
    double lo = 0.0;                                   // E_(t-1) of the row below
#pragma unroll
    for (int t = 0; t < NE; ++t) {
      const double c = e[t];
      e[t] = x * c + h * lo + (t + 1) * e[t + 1];
      lo = c;
    }
  };
  for (int k = 0; k < i; ++k) raise(xpa);
  const int nt = La + Lb + 1;
  double* o = out + (int64_t)i * (Lb + 1) * nt;
  for (int j = 0; j <= Lb; ++j) {
    if (j) raise(xpb);
    double s = 1.0;
#pragma unroll
    for (int t = 0; t < NE; ++t) {
      if (t < nt) o[j * nt + t] = s * e[t];
      s *= sgn;
    }
  }
}

// F_n(T) for one order (boys_fn's two ranges; erf(sqrt T) = 1 in doubles from T = 36 on).
__device__ double boys_one(int n, double T) {
  if (T < BOYS_TMAX) {
    const double x = T * BOYS_DENS;
    const int k = (int)(x + 0.5);
    const double d = ((double)k - x) / BOYS_DENS;
    const double* g = g_boys[k] + n;
    double f = g[6];
    f = g[5] + d * f * (1.0 / 6.0);
    f = g[4] + d * f * (1.0 / 5.0);
    f = g[3] + d * f * (1.0 / 4.0);
    f = g[2] + d * f * (1.0 / 3.0);
    f = g[1] + d * f * (1.0 / 2.0);
    return g[0] + d * f;
  }
  const double e = exp(-T), r = 0.5 / T;
  double F = 0.5 * sqrt(M_PI / T);
  for (int m = 0; m < n; ++m) F = ((2 * m + 1) * F - e) * r;
  return F;
}

// (ab|cd) of four functions of one term, all s but at most one p (about its own centre, axis x):
//   (ss|ss) = sum K_ab K_cd F_0,  bra p: K_ab K_cd ((P - A)_x F_0 - alpha / p (P - Q)_x F_1), ket p alike with the
// other sign of P - Q; the lanes split the primitive quartets.  A chain of 12 hydrogens in a split-valence basis
// (24 s functions, each a group by itself): 852 us as groups, 379 as elements of the general form, 235 so.
__device__ double eri_short(const apy_gto& A, const apy_gto& B, const apy_gto& C, const apy_gto& D, const double* cen,
                            int lane) {
  int pf = -1, px = 0;                                 // the p function and its axis
  double r[4][3];
  auto centre = [&](const apy_gto& f, int y) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      r[y][k] = cen[3 * f.atom + k];
      if (f.lmn[0][k]) { pf = y; px = k; }
    }
  };
  centre(A, 0);
  centre(B, 1);
  centre(C, 2);
  centre(D, 3);
  double ab = 0.0, cd = 0.0, rx[4];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    ab += (r[0][k] - r[1][k]) * (r[0][k] - r[1][k]);
    cd += (r[2][k] - r[3][k]) * (r[2][k] - r[3][k]);
  }
#pragma unroll
  for (int y = 0; y < 4; ++y) rx[y] = px == 0 ? r[y][0] : px == 1 ? r[y][1] : r[y][2];
  const double at = pf == 0 ? rx[0] : pf == 1 ? rx[1] : pf == 2 ? rx[2] : rx[3];
  const SmallDiv dD(D.nprim), dC(C.nprim), dB(B.nprim);
  const int np = A.nprim * B.nprim * C.nprim * D.nprim;
  double acc = 0.0;
  for (int w = lane; w < np; w += 64) {
    const int w1 = dD.div(w), w2 = dC.div(w1), w3 = dB.div(w2);
    const int pd = dD.mod(w), pc = dC.mod(w1), pb = dB.mod(w2), pa = w3;
    const double a = A.exps[pa], b = B.exps[pb], c = C.exps[pc], d = D.exps[pd];
    const double p = a + b, q = c + d, ip = 1.0 / p, iq = 1.0 / q, alpha = p * q / (p + q);
    double r2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double x = (a * r[0][k] + b * r[1][k]) * ip - (c * r[2][k] + d * r[3][k]) * iq;
      r2 += x * x;
    }
    const double F0 = boys_one(0, alpha * r2);
    double v = F0;
    if (pf >= 0) {
      const double P = (a * rx[0] + b * rx[1]) * ip, Q = (c * rx[2] + d * rx[3]) * iq, F1 = boys_one(1, alpha * r2);
      v = pf < 2 ? (P - at) * F0 - alpha * ip * (P - Q) * F1 : (Q - at) * F0 + alpha * iq * (P - Q) * F1;
    }
    acc += A.coefs[0][pa] * B.coefs[0][pb] * C.coefs[0][pc] * D.coefs[0][pd] *
           (2.0 * M_PI * M_PI * sqrt(M_PI) / (p * q * sqrt(p + q))) * exp(-a * b * ip * ab - c * d * iq * cd) * v;
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  return acc;
}

__global__ __launch_bounds__(256, 3) void eri_kernel(int64_t ngeom, int64_t natom, const double* __restrict__ centers,
                                                  EriTab T, int sym, double2* __restrict__ out) {
  __shared__ EriShared S;
  extern __shared__ uint16_t starts[];               // group starts, then the functions' flags, the groups' classes
  const int tid = threadIdx.x;
  const int64_t n0 = T.n[0], n1 = T.n[1], n2 = T.n[2], n3 = T.n[3], full = n0 * n1 * n2 * n3;

  // ---- once a workgroup: the tables' groups (ERI_ALL: one table, ERI_KET: the ket's twice), index tables
  const int ntab = sym == ERI_ALL ? 1 : sym == ERI_KET ? 3 : 4;
  int64_t tot = 0, off[5];
  for (int x = 0; x < 4; ++x) { off[x] = tot; if (x < ntab) tot += T.n[x] + 1; }
  uint8_t* flags = (uint8_t*)(starts + tot);
  for (int x = 0; x < ntab; ++x)
    for (int64_t i = tid; i < T.n[x]; i += 256) {
      const apy_gto& f = T.f[x][i];
      int v = 0;
      if (gto_ok(f, natom)) {
        bool same = i > 0;
        if (same) {
          const apy_gto& e = T.f[x][i - 1];
          same = gto_ok(e, natom) && e.atom == f.atom && e.nprim == f.nprim;
          for (int k = 0; same && k < f.nprim; ++k) same = e.exps[k] == f.exps[k];
        }
        const int L = lsum(f.lmn[0]);
        v = (same ? 1 : 0) | (f.nterm == 1 && L < ECLS && f.nprim <= 4 ? 2 << L : 0);
      }
      flags[off[x] + i] = (uint8_t)v;
    }
  __syncthreads();
  if (const int x = tid >> 6; x < ntab) {
    const int g = find_groups((int)T.n[x], flags + off[x], starts + off[x], S.nshort[x], tid & 63);
    if ((tid & 63) == 0) S.ngrp[x] = g;
  }
  for (int r = tid; r < ENR; r += 256) {
    int s = 0, w = 0;
    while (tuv_count(s) <= r) ++s;
    const int q = r - (s > 0 ? tuv_count(s - 1) : 0);
    while ((w + 1) * (w + 2) / 2 <= q) ++w;
    const int v = q - w * (w + 1) / 2;
    S.tuv[r][0] = (uint8_t)(s - w); S.tuv[r][1] = (uint8_t)(w - v); S.tuv[r][2] = (uint8_t)v;
  }
  if (tid <= LQ) {
    double a = 1.0;
    for (int i = 0; 2 * i <= tid; ++i) {
      S.herm[tid][i] = a;
      a *= (double)((tid - 2 * i) * (tid - 2 * i - 1)) / (2.0 * (i + 1));
    }
  }
  __syncthreads();
  // slot x's groups are those of table tx[x]
  const int tx[4] = {0, sym == ERI_ALL ? 0 : 1, sym == ERI_ALL ? 0 : 2, sym == ERI_ALL ? 0 : sym == ERI_KET ? 2 : 3};
  int64_t ng[4];
  for (int x = 0; x < 4; ++x) ng[x] = uniform(S.ngrp[tx[x]]);
  // the short form (below) where it takes most quartets: the passes over all of them that it needs beside the
  // workgroups' cost a molecule of mixed shells more than it saves there (13 geometries of H2O2/6-31G* 1.31 -> 1.36 ms)
  double all = 1.0, ss = 1.0, sp = 0.0;
  for (int x = 0; x < 4; ++x) {
    const int* c = S.nshort[tx[x]];
    all *= (double)ng[x];
    sp = sp * (double)c[0] + ss * (double)c[1];
    ss *= (double)c[0];
  }
  const bool shorts = uniform(ss + sp >= 0.5 * all);
  const int64_t pk = sym == ERI_NONE ? ng[2] * ng[3] : ng[2] * (ng[2] + 1) / 2;
  const int64_t per = sym == ERI_ALL ? pk * (pk + 1) / 2 : ng[0] * ng[1] * pk;

  // the groups of an item, and whether the short form takes it
  auto decode = [&](int64_t r0, int64_t (&G)[4]) {
    if (sym == ERI_ALL) {
      int64_t bra, ket;
      tri_split(r0, bra, ket);
      tri_split(bra, G[0], G[1]);
      tri_split(ket, G[2], G[3]);
    } else {
      if (sym == ERI_KET) {
        tri_split(r0 % pk, G[2], G[3]);
      } else {
        G[2] = (r0 % pk) / ng[3]; G[3] = r0 % ng[3];
      }
      G[1] = (r0 / pk) % ng[1];
      G[0] = r0 / (pk * ng[1]);
    }
    int c = shorts ? 0 : 2;
    for (int x = 0; shorts && x < 4; ++x) {
      const int y = flags[off[tx[x]] + G[x]];
      c += y < ECLS ? y : 2;
    }
    return c < 2;
  };
  // the value of a canonical element to every image under the launch's symmetry
  auto put = [&](int64_t g, int64_t i, int64_t j, int64_t k, int64_t l, double v) {
    const double2 y = make_double2(v, 0.0);
    double2* o = out + g * full;
    auto at = [&](int64_t p, int64_t q, int64_t s, int64_t t) { return ((p * n1 + q) * n2 + s) * n3 + t; };
    o[at(i, j, k, l)] = y;
    if (sym == ERI_NONE) return;
    o[at(i, j, l, k)] = y;
    if (sym == ERI_KET) return;
    o[at(j, i, k, l)] = y;
    o[at(j, i, l, k)] = y;
    o[at(k, l, i, j)] = y;
    o[at(l, k, i, j)] = y;
    o[at(k, l, j, i)] = y;
    o[at(l, k, j, i)] = y;
  };
  for (int64_t item = blockIdx.x; item < ngeom * per; item += gridDim.x) {
    const int64_t g = item / per, r0 = item % per;
    int64_t G[4];
    if (uniform(decode(r0, G))) continue;
    // ---- the four groups into LDS
    __syncthreads();                                  // the previous item's elements are done with LDS
    if (tid < 4) {
      const int x = tid;
      const int64_t b = starts[off[tx[x]] + G[x]], e = starts[off[tx[x]] + G[x] + 1];
      const apy_gto& f = T.f[x][b];
      const bool ok = gto_ok(f, natom);
      S.first[x] = (int)b;
      S.size[x] = (int)(e - b);
      S.nprim[x] = ok ? f.nprim : 0;
      S.L[x] = 0;
      for (int k = 0; k < 3; ++k) S.cen[x][k] = ok ? centers[3 * (natom * g + f.atom) + k] : 0.0;
    }
    __syncthreads();
    for (int w = tid; w < 4 * EG * 2 * APY_GTO_MAXPRIM; w += 256) {
      const int k = w % APY_GTO_MAXPRIM, t = (w / APY_GTO_MAXPRIM) % 2, m = (w / (2 * APY_GTO_MAXPRIM)) % EG,
                x = w / (2 * APY_GTO_MAXPRIM * EG);
      if (m >= S.size[x]) continue;
      const apy_gto& f = T.f[x][S.first[x] + m];
      S.coef[x][m][t][k] = f.coefs[t][k];
      if (m == 0 && t == 0) S.exps[x][k] = f.exps[k];
      if (k < 3) S.lmn[x][m][t][k] = (int8_t)f.lmn[t][k];
      if (k == 3 && t == 0) S.nterm[x][m] = (uint8_t)f.nterm;
      if (k == 4 && S.nprim[x] > 0 && t < f.nterm) atomicMax(&S.L[x], lsum(f.lmn[t]));
    }
    __syncthreads();
    const int La = uniform(S.L[0]), Lb = uniform(S.L[1]), Lc = uniform(S.L[2]), Ld = uniform(S.L[3]);
    const int sz1 = uniform(S.size[1]), sz3 = uniform(S.size[3]);
    const int nbc = uniform(S.size[0]) * sz1, nkc = uniform(S.size[2]) * sz3;
    const int nbp = uniform(S.nprim[0] * S.nprim[1]), nkp = uniform(S.nprim[2] * S.nprim[3]);
    const bool bad = nbp * nkp == 0;
    const int L1 = La + Lb, L2 = Lc + Ld, L = min(L1 + L2, LQ), nr = tuv_count(L), nr1 = tuv_count(min(L1, L));
    const int nr2 = tuv_count(min(L2, L));
    const int eb = 3 * (La + 1) * (Lb + 1) * (L1 + 1), ek = 3 * (Lc + 1) * (Ld + 1) * (L2 + 1);
    const int wsz = 4 * (L + 1) + nr;
    const SmallDiv dL(L + 1), dR(nr), dR1(nr1), dR2(nr2), dA(La + 1), dC(Lc + 1), d3(3), dsz1(sz1), dsz3(sz3);
    // tuv index of the sum of a bra's and a ket's; past L (read by elements past LQ only, which are NaN) 0
    auto tuv_sum = [&](int x, int y) {
      const int t = S.tuv[x][0] + S.tuv[y][0], u = S.tuv[x][1] + S.tuv[y][1], v = S.tuv[x][2] + S.tuv[y][2];
      return t + u + v <= L ? tuv_index(t, u, v) : 0;
    };
    const bool tab = nr1 * nr2 <= ESUM;
    // ---- per quartet: primitive pairs, the slots of every element, sums of tuv
    if (!bad) {
      if (tid < 128) {
        const int x = tid >> 6, b = tid & 63, n = S.nprim[2 * x + 1];
        if (b < (x ? nkp : nbp)) {
          const int pa = b / n, pb = b % n;
          const double ea = S.exps[2 * x][pa], e = S.exps[2 * x + 1][pb], p = ea + e, ip = 1.0 / p;
          S.prim[x][b][0] = (uint8_t)pa;
          S.prim[x][b][1] = (uint8_t)pb;
          S.pair[x][b][0] = p;
          S.pair[x][b][1] = ip;
          for (int k = 0; k < 3; ++k)
            S.pair[x][b][2 + k] = (ea * S.cen[2 * x][k] + e * S.cen[2 * x + 1][k]) / p;
        }
      } else {
        const int x = (tid - 128) >> 6, e = tid & 63, ne = x ? nkc : nbc;   // waves 2 (bra) and 3 (ket)
        int n = 0;
        if (e < ne) {
          const int ma = x ? dsz3.div(e) : dsz1.div(e), mb = x ? dsz3.mod(e) : dsz1.mod(e);
          for (int ta = 0; ta < S.nterm[2 * x][ma]; ++ta)
            for (int tb = 0; tb < S.nterm[2 * x + 1][mb]; ++tb) {
              int c = 1;
              for (int k = 0; k < 3; ++k) c *= S.lmn[2 * x][ma][ta][k] + S.lmn[2 * x + 1][mb][tb][k] + 1;
              n += c;
            }
          n = (n + 1) & ~1;
        }
        int sc = n;                                    // inclusive scan over the wave
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(sc, o, 64);
          if ((tid & 63) >= o) sc += y;
        }
        if (e < ne) S.slot[x][e + 1] = (int16_t)sc;
        if (e == 0) S.slot[x][0] = 0;
      }
      for (int w = tid; tab && w < nr1 * nr2; w += 256) S.sum[w] = (uint8_t)tuv_sum(dR2.div(w), dR2.mod(w));
    }
    __syncthreads();
    const int totb = bad ? 0 : uniform(S.slot[0][nbc]), totk = bad ? 0 : uniform(S.slot[1][nkc]);
    // slices of elements whose slots fit (all of them but for differentiated or f functions)
    auto slice = [&](int x, int e0, int ne, int tot, int cap) {
      if (bad) return ne - e0;
      int n = min(ne - e0, cap);
      if (tot > ES)
        while (n > 1 && uniform(S.slot[x][e0 + n] - S.slot[x][e0]) > ES) --n;
      return n;
    };
    for (int k0 = 0, nks; k0 < nkc; k0 += nks) {
      nks = slice(1, k0, nkc, totk, EH / nr1);
      for (int m0 = 0, nbs; m0 < nbc; m0 += nbs) {
      nbs = slice(0, m0, nbc, totb, EG * EG);
      const int nel = nbs * nks;
      const SmallDiv dK(nks);
      const int sk0 = bad ? 0 : uniform(S.slot[1][k0]), sb0 = bad ? 0 : uniform(S.slot[0][m0]);
      const int nsk = bad ? 1 : uniform(S.slot[1][k0 + nks]) - sk0, nsb = bad ? 1 : uniform(S.slot[0][m0 + nbs]) - sb0;
      const SmallDiv dsb(nsb), dsk(nsk);
      // the slots of the slice, a thread each
      for (int w = tid; w < nsb + nsk && !bad; w += 256) {
        const int x = w < nsb ? 0 : 1, sl = x ? w - nsb : w, g = sl + (x ? sk0 : sb0);
        int e = 0, hi = x ? nkc : nbc;                   // last element whose first slot is at most g
        while (hi - e > 1) {
          const int mid = (e + hi) >> 1;
          if (S.slot[x][mid] <= g) e = mid; else hi = mid;
        }
        const int ma = x ? dsz3.div(e) : dsz1.div(e), mb = x ? dsz3.mod(e) : dsz1.mod(e);
        int n = g - S.slot[x][e], tuv = 0;
        EriSlot r;
        r.e[0] = r.e[1] = r.e[2] = 0;
        r.ca = 255;
        r.cb = 0;
        for (int tt = 0; tt < S.nterm[2 * x][ma] * S.nterm[2 * x + 1][mb]; ++tt) {
          const int ta = tt / S.nterm[2 * x + 1][mb], tb = tt % S.nterm[2 * x + 1][mb];
          const int8_t* la = S.lmn[2 * x][ma][ta];
          const int8_t* lb = S.lmn[2 * x + 1][mb][tb];
          const int lx = la[0] + lb[0], ly = la[1] + lb[1], lz = la[2] + lb[2], c = (lx + 1) * (ly + 1) * (lz + 1);
          if (n >= 0 && n < c) {
            const int k = n % (lz + 1), j = n / (lz + 1) % (ly + 1), i = n / ((lz + 1) * (ly + 1));
            const int l2 = (x ? Ld : Lb) + 1, nt = (x ? L2 : L1) + 1, ax = (x ? ek : eb) / 3;
            r.e[0] = (uint16_t)((la[0] * l2 + lb[0]) * nt + i);
            r.e[1] = (uint16_t)(ax + (la[1] * l2 + lb[1]) * nt + j);
            r.e[2] = (uint16_t)(2 * ax + (la[2] * l2 + lb[2]) * nt + k);
            r.ca = (uint8_t)(2 * ma + ta);
            r.cb = (uint8_t)(2 * mb + tb);
            tuv = tuv_index(i, j, k);
          }
          n -= c;
        }
        S.rec[x][sl] = r;
        S.stuv[x][sl] = (uint8_t)tuv;
      }
      // batches of primitive pairs
      const int Kb = max(1, min(min(nkp, ES / nsk), min(EE / ek, EW / wsz)));
      const int Bb = max(1, min(min(nbp, ES / nsb), min(EE / eb, min(EW / (wsz * Kb), EH / (nr1 * nks)))));
      double acc[EACC];
#pragma unroll
      for (int m = 0; m < EACC; ++m) acc[m] = 0.0;
      for (int b0 = 0; b0 < nbp && !bad; b0 += Bb) {
        const int nb = min(Bb, nbp - b0);
        for (int w = tid; w < nb * nks * nr1; w += 256) S.H[w] = 0.0;
        for (int q0 = 0; q0 < nkp; q0 += Kb) {
          const int nq = min(Kb, nkp - q0), nbq = nb * nq;
          const SmallDiv dq(nq);
          // 1. E of the bra batch (once) and of the ket batch (again only if it changes), G and powers
          const bool newb = q0 == 0, newk = Kb < nkp || b0 == 0;
          // (a wave each for the bra's E and the ket's, two for G: in one wave their latencies would add up)
          const int wave = tid >> 6;
          if (wave < 2) {
            const int x = wave, l1 = x ? Lc : La, l2 = x ? Ld : Lb, p0 = x ? q0 : b0, es = x ? ek : eb;
            const int n = (x ? newk : newb) ? (x ? nq : nb) * 3 * (l1 + 1) : 0;
            for (int w = tid & 63; w < n; w += 64) {
              const int y = x ? dC.div(w) : dA.div(w), i = x ? dC.mod(w) : dA.mod(w), b = d3.div(y), ax = d3.mod(y);
              const uint8_t* pr = S.prim[x][p0 + b];
              herm_row(i, l1, l2, S.cen[2 * x][ax] - S.cen[2 * x + 1][ax], S.exps[2 * x][pr[0]],
                       S.exps[2 * x + 1][pr[1]], S.pair[x][p0 + b][1], x ? -1.0 : 1.0, S.E[x] + b * es + ax * (es / 3));
            }
          } else {
            for (int w = tid - 128; w < nbq * (L + 1); w += 128) {
              const int bq = dL.div(w), n = dL.mod(w);
              const double* B = S.pair[0][b0 + dq.div(bq)];
              const double* Q = S.pair[1][q0 + dq.mod(bq)];
              const double p = B[0], s = Q[0], alpha = p * s / (p + s);
              double* Wq = S.W + bq * wsz;
              double r2 = 0.0;
              for (int ax = 0; ax < 3; ++ax) {
                const double d = B[2 + ax] - Q[2 + ax];
                r2 += d * d;
                double pw = 1.0;
                for (int k = 0; k < n; ++k) pw *= d;
                Wq[(ax + 1) * (L + 1) + n] = pw;
              }
              double G_ = 2.0 * M_PI * M_PI * sqrt(M_PI) / (p * s * sqrt(p + s)) * boys_one(n, alpha * r2);
              for (int k = 0; k < n; ++k) G_ *= -2.0 * alpha;
              Wq[n] = G_;
            }
          }
          __syncthreads();
          // 2. R_tuv, and the slots' coefficients
          auto coulomb = [&](auto uc) {
            constexpr int U = decltype(uc)::value;
            for (int w = tid; w < nr * ((nbq + U - 1) / U); w += 256) {
              const int rr = dR.mod(w), x0 = U * dR.div(w);
              const int t = S.tuv[rr][0], u = S.tuv[rr][1], v = S.tuv[rr][2];
              const double* Wq[U];
#pragma unroll
              for (int x = 0; x < U; ++x) Wq[x] = S.W + min(x0 + x, nbq - 1) * wsz;
              double sx[U];
#pragma unroll
              for (int x = 0; x < U; ++x) sx[x] = 0.0;
              for (int i = 0; 2 * i <= t; ++i) {
                double sy[U];
#pragma unroll
                for (int x = 0; x < U; ++x) sy[x] = 0.0;
                for (int j = 0; 2 * j <= u; ++j) {
                  double sz[U];
#pragma unroll
                  for (int x = 0; x < U; ++x) sz[x] = 0.0;
                  for (int k = 0; 2 * k <= v; ++k) {
                    const double a = S.herm[v][k];
#pragma unroll
                    for (int x = 0; x < U; ++x)
                      sz[x] += a * Wq[x][3 * (L + 1) + v - 2 * k] * Wq[x][t + u + v - i - j - k];
                  }
                  const double a = S.herm[u][j];
#pragma unroll
                  for (int x = 0; x < U; ++x) sy[x] += a * Wq[x][2 * (L + 1) + u - 2 * j] * sz[x];
                }
                const double a = S.herm[t][i];
#pragma unroll
                for (int x = 0; x < U; ++x) sx[x] += a * Wq[x][L + 1 + t - 2 * i] * sy[x];
              }
#pragma unroll
              for (int x = 0; x < U; ++x)
                if (x0 + x < nbq) S.W[(x0 + x) * wsz + 4 * (L + 1) + rr] = sx[x];
            }
          };
          if (nbq == 1) coulomb(std::integral_constant<int, 1>{});
          else coulomb(std::integral_constant<int, EU>{});
          // from the first thread on that has one R less to do
          const int nlb = newb ? nb * nsb : 0, nlk = newk ? nq * nsk : 0;
          const int ncoul = nbq == 1 ? nr : nr * ((nbq + EU - 1) / EU);
          for (int w = (tid - ncoul) & 255; w < nlb + nlk; w += 256) {
            const int x = w < nlb ? 0 : 1, y = x ? w - nlb : w;
            const int q = x ? dsk.div(y) : dsb.div(y), sl = x ? dsk.mod(y) : dsb.mod(y);
            const EriSlot r = S.rec[x][sl];
            const double* E = S.E[x] + q * (x ? ek : eb);
            const uint8_t* pr = S.prim[x][(x ? q0 : b0) + q];
            double v = 0.0;
            if (r.ca != 255)
              v = (&S.coef[2 * x][0][0][0])[r.ca * APY_GTO_MAXPRIM + pr[0]] *
                  (&S.coef[2 * x + 1][0][0][0])[r.cb * APY_GTO_MAXPRIM + pr[1]] * E[r.e[0]] * E[r.e[1]] * E[r.e[2]];
            S.Lam[x][y] = v;
          }
          __syncthreads();
          // 3. the ket contraction; where the items are few, 2^sh neighbouring lanes share one
          const int items = nb * nks * nr1;
          int sh = 0;
          while (sh < 6 && (items << (sh + 1)) <= 256 && (1 << sh) < nq) ++sh;
          const int sub = tid & ((1 << sh) - 1);
          auto ket = [&](auto uc) {
            constexpr int U = decltype(uc)::value;
            for (int w = tid >> sh; w < items; w += 256 >> sh) {
              const int y = dR1.div(w), rr = dR1.mod(w), b = dK.div(y), kc = k0 + dK.mod(y);
              const int f = S.slot[1][kc] - sk0, n = S.slot[1][kc + 1] - sk0;
              const uint8_t* sm = S.sum + rr * nr2;
              const double* R = S.W + b * nq * wsz + 4 * (L + 1);
              double h = 0.0;
              for (int q = sub; q < nq; q += U << sh) {
                int lq[U], rq[U];
                double c[U];
#pragma unroll
                for (int x = 0; x < U; ++x) {
                  const int z = q + (x << sh) < nq ? q + (x << sh) : q;
                  lq[x] = z * nsk;
                  rq[x] = z * wsz;
                  c[x] = 0.0;
                }
                for (int s = f; s < n; s += 2) {
                  const int t0 = S.stuv[1][s], t1 = S.stuv[1][s + 1];
                  const int r0 = tab ? sm[t0] : tuv_sum(rr, t0), r1 = tab ? sm[t1] : tuv_sum(rr, t1);
#pragma unroll
                  for (int x = 0; x < U; ++x)
                    c[x] += S.Lam[1][lq[x] + s] * R[rq[x] + r0] + S.Lam[1][lq[x] + s + 1] * R[rq[x] + r1];
                }
#pragma unroll
                for (int x = 0; x < U; ++x)
                  if (q + (x << sh) < nq) h += c[x];
              }
              for (int o = (1 << sh) >> 1; o > 0; o >>= 1) h += __shfl_xor(h, o, 64);   // one item's lanes: all here
              if (sub == 0) S.H[w] += h;
            }
          };
          if (nq <= 1 << sh) ket(std::integral_constant<int, 1>{});
          else ket(std::integral_constant<int, EU>{});
          __syncthreads();
        }
        // the bra contraction of this batch
        auto bra = [&](auto uc) {
          constexpr int U = decltype(uc)::value;
#pragma unroll
          for (int m = 0; m < EACC; ++m) {
            const int w = tid + 256 * m;
            if (w >= nel) continue;
            const int kc = dK.mod(w), bc = m0 + dK.div(w);
            const int f = S.slot[0][bc] - sb0, n = S.slot[0][bc + 1] - sb0;
            const double* Hk = S.H + kc * nr1;
            double h = 0.0;
            for (int b = 0; b < nb; b += U) {
              int lq[U], hq[U];
              double c[U];
#pragma unroll
              for (int x = 0; x < U; ++x) {
                const int z = b + x < nb ? b + x : b;
                lq[x] = z * nsb;
                hq[x] = z * nks * nr1;
                c[x] = 0.0;
              }
              for (int s = f; s < n; s += 2) {
                // a slot past the tuv of H belongs to elements past LQ (NaN)
                const int r0 = min((int)S.stuv[0][s], nr1 - 1), r1 = min((int)S.stuv[0][s + 1], nr1 - 1);
#pragma unroll
                for (int x = 0; x < U; ++x)
                  c[x] += S.Lam[0][lq[x] + s] * Hk[hq[x] + r0] + S.Lam[0][lq[x] + s + 1] * Hk[hq[x] + r1];
              }
#pragma unroll
              for (int x = 0; x < U; ++x)
                if (b + x < nb) h += c[x];
            }
            acc[m] += h;
          }
        };
        if (nb == 1) bra(std::integral_constant<int, 1>{});
        else bra(std::integral_constant<int, EU>{});
        __syncthreads();                              // H, E and the slots of this batch are read
      }
      // ---- out
#pragma unroll
      for (int m = 0; m < EACC; ++m) {
        const int w = tid + 256 * m;
        if (w >= nel) continue;
        const int kc = k0 + dK.mod(w), bc = m0 + dK.div(w);
        const int e0 = dsz1.div(bc), e1 = dsz1.mod(bc), e2 = dsz3.div(kc), e3 = dsz3.mod(kc);
        const int64_t i = S.first[0] + e0, j = S.first[1] + e1, k = S.first[2] + e2, l = S.first[3] + e3;
        // one element an image class: an order of functions is asked for where the group quartet leaves one open
        if (sym != ERI_NONE && k < l) continue;
        if (sym == ERI_ALL && i < j) continue;
        if (sym == ERI_ALL && G[0] == G[2] && G[1] == G[3] && (i < k || (i == k && j < l))) continue;
        double v = acc[m];
        if (bad) {
          v = kNaN;
        } else {
          int Lm[4];
          const int em[4] = {e0, e1, e2, e3};
          for (int x = 0; x < 4; ++x) {
            Lm[x] = 0;
            for (int t = 0; t < S.nterm[x][em[x]]; ++t) {
              const int8_t* c = S.lmn[x][em[x]][t];
              Lm[x] = max(Lm[x], c[0] + c[1] + c[2]);
            }
          }
          if (Lm[0] + Lm[1] + Lm[2] + Lm[3] > LQ) v = kNaN;
        }
        put(g, i, j, k, l, v);
      }
      }
    }
  }
  // ---- the short form, a wave an element: one s function each, or one of them p (the derivative of an s)
  const int lane = tid & 63;
  for (int64_t item = (int64_t)blockIdx.x * 4 + (tid >> 6); shorts && item < ngeom * per;
       item += (int64_t)gridDim.x * 4) {
    const int64_t g = item / per, r0 = item % per;
    int64_t G[4];
    if (!uniform(decode(r0, G))) continue;
    int64_t f[4];
    for (int x = 0; x < 4; ++x) f[x] = starts[off[tx[x]] + G[x]];
    const double v = eri_short(T.f[0][f[0]], T.f[1][f[1]], T.f[2][f[2]], T.f[3][f[3]], centers + 3 * natom * g, lane);
    if (lane == 0) put(g, f[0], f[1], f[2], f[3], v);
  }
}

// out[m,n,l,s] = on(m) D[m,n,l,s] + on(n) D[n,m,l,s] + on(l) D[l,s,m,n] + on(s) D[s,l,m,n] with
// D = (d m/dx n | l s) and on(p) = 1 if function p sits on the displaced atom (the derivative of (mn|ls)
// when that atom moves, each function following its atom).
__global__ __launch_bounds__(256) void eri_deriv_assemble_kernel(int64_t n, const int* __restrict__ atom_of,
                                                                 int atom, const double2* __restrict__ D,
                                                                 double2* __restrict__ out) {
  const int64_t n2 = n * n, n3 = n2 * n, total = n3 * n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t s = e % n, l = (e / n) % n, q = (e / n2) % n, m = e / n3;
    double re = 0.0;
    if (atom_of[m] == atom) re += D[((m * n + q) * n + l) * n + s].x;
    if (atom_of[q] == atom) re += D[((q * n + m) * n + l) * n + s].x;
    if (atom_of[l] == atom) re += D[((l * n + s) * n + m) * n + q].x;
    if (atom_of[s] == atom) re += D[((s * n + l) * n + m) * n + q].x;
    out[e] = make_double2(re, 0.0);
  }
}


// ------------------------------------------------------------------------------ one-electron integrals
constexpr int OJ = LF + 3;  // ket powers j <= LF + 2 (the kinetic operator raises j by two)
constexpr int NOEI = 9;     // S, T, V, Dx, Dy, Dz, Lx, Ly, Lz

// 1-D overlaps S_ij = int x_A^i x_B^j exp(-a x_A^2 - b x_B^2) dx for i <= imax (<= LF), j <= jmax (< OJ),
// Obara-Saika: S_00 = sqrt(pi/p) exp(-ab/p Q^2) with Q = A - B, p = a + b, and
//   S_{i+1,j} = X_PA S_ij + (i S_{i-1,j} + j S_{i,j-1}) / 2p,   X_PA = -b Q / p,
//   S_{i,j+1} = X_PB S_ij + (i S_{i-1,j} + j S_{i,j-1}) / 2p,   X_PB =  a Q / p.
__device__ void ovl_1d(int imax, int jmax, double Q, double a, double b, double (*S)[OJ]) {
  const double p = a + b, h = 0.5 / p, xpa = -b * Q / p, xpb = a * Q / p;
  S[0][0] = sqrt(M_PI / p) * exp(-a * b / p * Q * Q);
  for (int j = 0; j < jmax; ++j) S[0][j + 1] = xpb * S[0][j] + (j > 0 ? j * h * S[0][j - 1] : 0.0);
  for (int i = 0; i < imax; ++i)
    for (int j = 0; j <= jmax; ++j) {
      double v = xpa * S[i][j];
      if (i > 0) v += i * h * S[i - 1][j];
      if (j > 0) v += j * h * S[i][j - 1];
      S[i + 1][j] = v;
    }
}

// The integrals `which` selects between bra function A at ra and ket function B at rb, accumulated into
// v[NOEI].  Per axis, from the 1-D overlaps S_ij (i = bra power, j = ket power):
//   kinetic    t = -1/2 (j(j-1) S_{i,j-2} - 2b(2j+1) S_ij + 4b^2 S_{i,j+2}),
//   moment     m = S_{i,j+1} + (B - O) S_ij             (x - O = x_B + B - O),
//   derivative d = j S_{i,j-1} - 2b S_{i,j+1}           (d/dx acting on the ket);
//   T = t_x s_y s_z + s_x t_y s_z + s_x s_y t_z,  D_x = m_x s_y s_z,  L_x = (m_y d_z - m_z d_y) s_x (cyclic).
// The nuclear attraction uses the Hermite expansion of the product:
//   V = -sum_C Z_C 2 pi / p sum_tuv E^x_t E^y_u E^z_v R_tuv(p, P - C).
// The (term, primitive) pairs w = ((ta nbt + tb) npa + pa) npb + pb from `first` in steps of `step` (the
// lanes of a wavefront split them).
__device__ void oei_pair(const apy_gto& A, const double* ra, const apy_gto& B, const double* rb, int which,
                         const double* origin, const double* nuc, const double* Z, int64_t nnuc, int first, int step,
                         double* v) {
  const double Q[3] = {ra[0] - rb[0], ra[1] - rb[1], ra[2] - rb[2]};
  const int nw = A.nterm * B.nterm * A.nprim * B.nprim;
  for (int w = first; w < nw; w += step) {
    const int pb = w % B.nprim, pa = (w / B.nprim) % A.nprim, tb = (w / (B.nprim * A.nprim)) % B.nterm,
              ta = w / (B.nprim * A.nprim * B.nterm);
    const int* la = A.lmn[ta];
    const int* lb = B.lmn[tb];
    const double a = A.exps[pa], b = B.exps[pb], p = a + b;
    const double c = A.coefs[ta][pa] * B.coefs[tb][pb];
    double S[3][LF + 1][OJ], s[3], t[3], m[3], d[3];
    for (int x = 0; x < 3; ++x) {
      const int i = la[x], j = lb[x];
      ovl_1d(i, j + 2, Q[x], a, b, S[x]);
      s[x] = S[x][i][j];
      t[x] = -0.5 * ((j > 1 ? j * (j - 1) * S[x][i][j - 2] : 0.0) - 2.0 * b * (2 * j + 1) * S[x][i][j] +
                     4.0 * b * b * S[x][i][j + 2]);
      m[x] = S[x][i][j + 1] + (rb[x] - origin[x]) * S[x][i][j];
      d[x] = (j > 0 ? j * S[x][i][j - 1] : 0.0) - 2.0 * b * S[x][i][j + 1];
    }
    if (which & APY_OEI_OVERLAP) v[0] += c * s[0] * s[1] * s[2];
    if (which & APY_OEI_KINETIC) v[1] += c * (t[0] * s[1] * s[2] + s[0] * t[1] * s[2] + s[0] * s[1] * t[2]);
    if (which & APY_OEI_DIPOLE) {
      v[3] += c * m[0] * s[1] * s[2];
      v[4] += c * s[0] * m[1] * s[2];
      v[5] += c * s[0] * s[1] * m[2];
    }
    if (which & APY_OEI_ANGMOM) {
      v[6] += c * (m[1] * d[2] - m[2] * d[1]) * s[0];
      v[7] += c * (m[2] * d[0] - m[0] * d[2]) * s[1];
      v[8] += c * (m[0] * d[1] - m[1] * d[0]) * s[2];
    }
    if (which & APY_OEI_POTENTIAL) {
      double E[3][NE], P[3];
      int Lt[3];
      for (int x = 0; x < 3; ++x) {
        herm_E(la[x], lb[x], Q[x], a, b, E[x]);
        P[x] = (a * ra[x] + b * rb[x]) / p;
        Lt[x] = la[x] + lb[x];
      }
      const int L = Lt[0] + Lt[1] + Lt[2];
      const int sz = Lt[2] + 1, sy = (Lt[1] + 1) * sz;
      double acc = 0.0;
      for (int64_t C = 0; C < nnuc; ++C) {
        const double PC[3] = {P[0] - nuc[3 * C], P[1] - nuc[3 * C + 1], P[2] - nuc[3 * C + 2]};
        double F[LQ + 1], Rb[2][NRB];
        boys_fn(L, p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), F);
        const double* R = Rb[herm_R(L, Lt, p, PC, F, Rb)];
        double sum = 0.0;
        for (int tt = 0; tt <= Lt[0]; ++tt)
          for (int u = 0; u <= Lt[1]; ++u)
            for (int vv = 0; vv <= Lt[2]; ++vv) sum += E[0][tt] * E[1][u] * E[2][vv] * R[tt * sy + u * sz + vv];
        acc -= Z[C] * sum;
      }
      v[2] += c * 2.0 * M_PI / p * acc;
    }
  }
}

// One wavefront per output element (wave-uniform control flow): the lanes split the (term, primitive)
// pairs and a fixed-order butterfly sums each component.
__global__ __launch_bounds__(256) void oei_kernel(apy_oei_args p) {
  const int lane = threadIdx.x & 63;
  const int64_t per = p.na * p.nb, total = p.nset * per;
  const int64_t nwave = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t e = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6; e < total; e += nwave) {
    const int64_t s = e / per, r = e % per, i = r / p.nb, j = r % p.nb;
    const apy_gto& A = p.fa[i];
    const apy_gto& B = p.fb[j];
    double v[NOEI];
    for (int k = 0; k < NOEI; ++k) v[k] = 0.0;
    if (gto_ok(A, p.nca) && gto_ok(B, p.ncb)) {
      oei_pair(A, p.ca + 3 * (s * p.nca + A.atom), B, p.cb + 3 * (s * p.ncb + B.atom), p.which, p.origin,
               p.nuclei ? p.nuclei + 3 * s * p.nnuc : nullptr, p.charges, p.nnuc, lane, 64, v);
#pragma unroll
      for (int k = 0; k < NOEI; ++k)
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
    } else {
      for (int k = 0; k < NOEI; ++k) v[k] = kNaN;
    }
    if (lane != 0) continue;
    // selected components in the order S, T, V, Dx, Dy, Dz, Lx, Ly, Lz
    constexpr int bit_of[NOEI] = {APY_OEI_OVERLAP, APY_OEI_KINETIC, APY_OEI_POTENTIAL, APY_OEI_DIPOLE, APY_OEI_DIPOLE,
                                  APY_OEI_DIPOLE,  APY_OEI_ANGMOM,  APY_OEI_ANGMOM,    APY_OEI_ANGMOM};
    int64_t c = 0;
    const int64_t ncomp = apy_oei_ncomp(p.which);
#pragma unroll
    for (int k = 0; k < NOEI; ++k)
      if (p.which & bit_of[k]) p.out[((s * ncomp + c++) * p.na + i) * p.nb + j] = v[k];
  }
}
// Fill g_boys on the current device before its first integral launch; the stream is synchronised once so
// that launches on other streams see the table.
int ensure_boys_table(hipStream_t st) {
  static std::mutex mu;
  static bool ready[256] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 256) return APY_E_HIP;
  std::lock_guard<std::mutex> lk(mu);
  if (ready[dev]) return APY_OK;
  boys_table_kernel<<<(BOYS_NGRID + 255) / 256, 256, 0, st>>>();
  APY_LAUNCH_CHECK();
  if (hipStreamSynchronize(st) != hipSuccess) return APY_E_HIP;
  ready[dev] = true;
  return APY_OK;
}

}  // namespace

extern "C" {

int apy_eri_gto(int64_t ngeom, int64_t natom, const double* centers, const apy_gto* fa, int64_t na,
                const apy_gto* fb, int64_t nb, const apy_gto* fc, int64_t nc, const apy_gto* fd, int64_t nd,
                void* out, void* stream) {
  if (ngeom < 1 || natom < 1 || !centers || !fa || !fb || !fc || !fd || !out || na < 1 || nb < 1 || nc < 1 ||
      nd < 1)
    return APY_E_ARG;
  // the same table in every slot: 8-fold permutational symmetry; the same ket tables: (ab|cd) = (ab|dc)
  const int sym = (fa == fb && fb == fc && fc == fd && na == nb && nb == nc && nc == nd) ? ERI_ALL
                  : (fc == fd && nc == nd)                                             ? ERI_KET
                                                                                       : ERI_NONE;
  if (na > INT32_MAX || nb > INT32_MAX || nc > INT32_MAX || nd > INT32_MAX) return APY_E_ARG;
  if (const int rc = ensure_boys_table((hipStream_t)stream); rc != APY_OK) return rc;
  const EriTab T = {{fa, fb, fc, fd}, {na, nb, nc, nd}};
  // Tables whose group starts do not fit LDS are taken element by element, and so are launches of fewer elements
  // than the waves of two a SIMD: the longest one then sets the time, and a wave has its sums sooner
  // than a workgroup its group.  us a call, elements / groups: 406 elements of H2O/STO-3G 102 / 108, their 1372
  // derivatives 178 / 186; 3081 of H2O2/STO-3G 145 / 107.
  const int64_t tot = na + 1 + (sym == ERI_ALL ? 0 : nb + nc + 2 + (sym == ERI_KET ? 0 : nd + 1));
  const double nk = (double)nc * (nc + 1) / 2;
  const double elements = (double)ngeom * (sym == ERI_ALL   ? nk * (nk + 1) / 2
                                           : sym == ERI_KET ? (double)na * nb * nk
                                                            : (double)na * nb * nc * nd);
  if (tot > ETAB || elements <= 2048.0) {
    const unsigned grid = (unsigned)std::min((elements + 3.0) / 4.0, 65536.0);
    eri_element_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(ngeom, natom, centers, T, sym, (double2*)out);
    APY_LAUNCH_CHECK();
    return APY_OK;
  }
  // a resident grid (three workgroups a CU): the groups are found once a workgroup
  const unsigned grid = (unsigned)std::min(elements, 3.0 * 256.0);
  const size_t lds = (size_t)tot * (sizeof(uint16_t) + 1);
  eri_kernel<<<grid, 256, lds, (hipStream_t)stream>>>(ngeom, natom, centers, T, sym, (double2*)out);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

int apy_eri_deriv_assemble(int64_t n, const int* atom_of, int atom, const void* D, void* out, void* stream) {
  if (n < 1 || !atom_of || !D || !out || D == out) return APY_E_ARG;
  const int64_t total = n * n * n * n;
  eri_deriv_assemble_kernel<<<apy_grid1d(total), 256, 0, (hipStream_t)stream>>>(n, atom_of, atom, (const double2*)D,
                                                                                 (double2*)out);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

int apy_oei_components(int which) { return apy_oei_ncomp(which); }

int apy_oei_gto(const apy_oei_args* a, void* stream) {
  if (!a || apy_oei_ncomp(a->which) == 0 || a->nset < 1 || !a->fa || !a->fb || a->na < 1 || a->nb < 1 || !a->ca ||
      !a->cb || a->nca < 1 || a->ncb < 1 || !a->out)
    return APY_E_ARG;
  if ((a->which & APY_OEI_POTENTIAL) && (!a->nuclei || !a->charges || a->nnuc < 1)) return APY_E_ARG;
  const int64_t total = a->nset * a->na * a->nb;
  if ((a->which & APY_OEI_POTENTIAL) != 0)
    if (const int rc = ensure_boys_table((hipStream_t)stream); rc != APY_OK) return rc;
  oei_kernel<<<apy_grid1d(64 * total), 256, 0, (hipStream_t)stream>>>(*a);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

}  // extern "C"
