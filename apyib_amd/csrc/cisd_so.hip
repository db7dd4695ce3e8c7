// Spin-orbital CISD / CID operator on MI355X.
//
// The doubles residual of ci_wfn.py:319-334 is regrouped into GEMMs on the
// FP64 matrix cores plus one fused elementwise epilogue:
//   PPL + HHL + F_oo (ci_wfn.py:326-329)  in (i<j)x(a<b) pair space:
//        R_p  = T_p . vvvv_p^T            [Po x Pv x Pv]   (t2 and <ab||cd>
//        R_p += Hoo . T_p                 [Po x Pv x Po]    antisymmetric, so
//                                                            1/2 sum_cd = sum_c<d)
//   ring (ci_wfn.py:330-333) as one product and its P(ij)P(ab) images:
//        X[(ia),(jb)] = sum_kc t2[i,k,a,c] <kb||cj>    [OV x OV x OV]
//   F_vv (ci_wfn.py:324-325):   Y[ija,b] = sum_c t2[ija,c] F_bc
//   T1 -> T2 (ci_wfn.py:320-323): U[a,b,(ij)] = sum_k t1[k,a] <kb||ij>,
//                                 Q[(ab),j,i] = sum_c <ab||cj> t1[i,c]
// and the epilogue, per packed (i<j, a<b), sums
//   <ab||ij> + R_p + P(ij)P(ab) X + P(ab) Y - P(ab) U + P(ij) Q
// then applies r = s - E t, t += r/D, writing the four antisymmetric images.
// The singles residual (ci_wfn.py:309-316) is six small GEMMs into one
// accumulator and an elementwise update.
#include "common.h"
#include "synth.h"

#include <algorithm>
#include <vector>

namespace {

__host__ __device__ inline int64_t npair(int64_t N) { return N * (N - 1) / 2; }
__host__ __device__ inline int64_t prow(int64_t p, int64_t N) { return p * (2 * N - p - 1) / 2; }

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

// ---------------------------------------------------------------- sources
struct SrcFull {
  const double2* A;
  int64_t n;
  __device__ double2 operator()(int64_t p, int64_t q, int64_t r, int64_t s) const {
    return A[((p * n + q) * n + r) * n + s];
  }
};

// <pq||rs> = <pq|rs> - <pq|sr>, <pq|rs> = (p/2 r/2 | q/2 s/2) delta(sp,sr) delta(sq,ss)
struct SrcMO {
  const double2* E;
  int64_t m;
  __device__ double2 chem(int64_t P, int64_t Q, int64_t R, int64_t S) const {
    return E[((P * m + Q) * m + R) * m + S];
  }
  __device__ double2 operator()(int64_t p, int64_t q, int64_t r, int64_t s) const {
    double2 v = make_double2(0.0, 0.0);
    if (((p ^ r) & 1) == 0 && ((q ^ s) & 1) == 0) v = chem(p >> 1, r >> 1, q >> 1, s >> 1);
    if (((p ^ s) & 1) == 0 && ((q ^ r) & 1) == 0) {
      double2 w = chem(p >> 1, s >> 1, q >> 1, r >> 1);
      v.x -= w.x;
      v.y -= w.y;
    }
    return v;
  }
};

enum Kind { K_VVVV_P = 0, K_RING, K_OOOO_P, K_OVOO_P, K_VVVO_P, K_VOVV, K_OOOV, K_VVOO_T, K_OOVV, K_COUNT };

__host__ __device__ inline int64_t kind_size(int kind, int64_t O, int64_t V) {
  const int64_t Po = npair(O), Pv = npair(V);
  switch (kind) {
    case K_VVVV_P: return Pv * Pv;
    case K_RING: return O * V * O * V;
    case K_OOOO_P: return Po * Po;
    case K_OVOO_P: return O * V * Po;
    case K_VVVO_P: return Pv * O * V;
    case K_VOVV: return V * O * Pv;
    case K_OOOV: return O * O * O * V;
    case K_VVOO_T: return O * O * V * V;
    case K_OOVV: return O * O * V * V;
  }
  return 0;
}

// Map flat index t of block `kind` to spin-orbital indices (p,q,r,s) of <pq||rs>.
__device__ inline void kind_index(int kind, int64_t t, int64_t O, int64_t V, int64_t& p, int64_t& q, int64_t& r,
                                  int64_t& s) {
  const int64_t Po = npair(O), Pv = npair(V);
  int64_t a, b, c, d, i, j, k;
  switch (kind) {
    case K_VVVV_P: {
      pdec(t / Pv, V, a, b);
      pdec(t % Pv, V, c, d);
      p = O + a; q = O + b; r = O + c; s = O + d;
      break;
    }
    case K_RING: {  // [(j,b),(k,c)] = <kb||cj>
      c = t % V; t /= V; k = t % O; t /= O; b = t % V; j = t / V;
      p = k; q = O + b; r = O + c; s = j;
      break;
    }
    case K_OOOO_P: {  // [(i<j)][(k<l)] = <kl||ij>
      int64_t l;
      pdec(t / Po, O, i, j);
      pdec(t % Po, O, k, l);
      p = k; q = l; r = i; s = j;
      break;
    }
    case K_OVOO_P: {  // [k][b][(i<j)] = <kb||ij>
      int64_t P = t % Po; t /= Po;
      b = t % V; k = t / V;
      pdec(P, O, i, j);
      p = k; q = O + b; r = i; s = j;
      break;
    }
    case K_VVVO_P: {  // [(a<b)][j][c] = <ab||cj>
      c = t % V; t /= V; j = t % O; int64_t P = t / O;
      pdec(P, V, a, b);
      p = O + a; q = O + b; r = O + c; s = j;
      break;
    }
    case K_VOVV: {  // [a][j][(c<b)] = <aj||cb>
      int64_t P = t % Pv; t /= Pv;
      j = t % O; a = t / O;
      pdec(P, V, c, b);
      p = O + a; q = j; r = O + c; s = O + b;
      break;
    }
    case K_OOOV: {  // [k][j][i][b] = <kj||ib>
      b = t % V; t /= V; i = t % O; t /= O; j = t % O; k = t / O;
      p = k; q = j; r = i; s = O + b;
      break;
    }
    case K_VVOO_T: {  // [i][j][a][b] = <ab||ij>
      b = t % V; t /= V; a = t % V; t /= V; j = t % O; i = t / O;
      p = O + a; q = O + b; r = i; s = j;
      break;
    }
    default: {  // K_OOVV [i][j][a][b] = <ij||ab>
      b = t % V; t /= V; a = t % V; t /= V; j = t % O; i = t / O;
      p = i; q = j; r = O + a; s = O + b;
      break;
    }
  }
}

// A store that leaves the caches to the integrals that are still read (past): for whole runs where the blocks of a
// call hold NT_ELEMENTS (64 MB) or more together (vvvo_p of m = 60, 158 MB, 62 -> 55 us; packed rows, which end
// inside cache lines, lose by it, 127 -> 149 us).  Fewer are still in the caches when the next kernel reads them: us
// to build the blocks and read each once, kept / past: m = 16, O = 10 178 / 247; m = 24, O = 12 144 / 166;
// m = 30, O = 20 (70 MB) 156 / 165, the build alone 62 / 57; m = 50, O = 20 (370 MB) 403 / 379, 215 / 196.
constexpr int64_t NT_ELEMENTS = 4 << 20;
__device__ inline void put_block(double2* p, double2 v, int past) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  if (past) __builtin_nontemporal_store((v2d){v.x, v.y}, (v2d*)p);
  else *p = v;
}

template <class Src>
__global__ __launch_bounds__(256) void build_block(Src src, int kind, int64_t O, int64_t V, double2* out,
                                                   int64_t total, int accumulate, double scale, int past) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    int64_t p, q, r, s;
    kind_index(kind, t, O, V, p, q, r, s);
    double2 v = src(p, q, r, s);
    if (accumulate) {
      double2 o = out[t];
      out[t] = make_double2(o.x + scale * v.x, o.y + scale * v.y);
    } else {
      put_block(out + t, v, past);
    }
  }
}

// The four large blocks of <pq||rs> from spatial MO integrals, where they are large (launch_pair_rows).  For one spatial pair (P, Q) the block's
// rows are the matrix M[x][y] = (Px|Qy) = E[P][x][Q][y] and its transpose:
//   <pq||rs> = d(p,r) d(q,s) M[R][S] - d(p,s) d(q,r) M[S][R]   (spins; capitals: p/2).
// One workgroup takes a pair (P, Q) and a 32 x 32 tile of (R, S): it reads the tile of M and the mirrored
// one along their rows into LDS and writes the rows of the up to four spin pairs along the output's
// contiguous index.  build_block read M[S][R] one element a cache line (stride m^2) and decoded four
// orbitals an element: m = 60, O = 20 (57e6 elements, 0.92 GB) 560 us in all, bound by those reads, 335 us
// so, bound by its writes.
//   KIND            p       q      columns                    output index
//   K_VVVV_P        a    <  b      r = c < s = d              [(ab)][(cd)]
//   K_VOVV          a       j      r = c < s = b              [a][j][(cb)]
//   K_VVVO_P        a    <  b      r = c, s = j               [(ab)][j][c]
//   K_RING          k       b      r = c, s = j               [(j,b)][(k,c)]
constexpr int BT = 32;   // spatial tile edge

template <int KIND>
__global__ __launch_bounds__(256) void build_pair_rows(const double2* __restrict__ E, int64_t m, int64_t O, int64_t V,
                                                       int64_t nq, int64_t nts, int past, double2* __restrict__ out) {
  constexpr bool TRI = KIND == K_VVVV_P || KIND == K_VOVV;      // columns r < s, both virtual
  constexpr bool PAIR = KIND == K_VVVV_P || KIND == K_VVVO_P;   // rows a < b
  __shared__ double2 A[BT][BT + 1], B[BT][BT + 1];              // M[R][S] and M[S][R] of the tile
  const int64_t n = O + V, v0 = O >> 1;                          // first virtual spatial orbital (O odd: shared)
  const int64_t Pv = npair(V), OV = O * V;
  int64_t w = blockIdx.x;
  int64_t tr, ts;
  if (TRI) {                                                     // tile pairs tr <= ts
    int64_t t = w % (nts * (nts + 1) / 2);
    w /= nts * (nts + 1) / 2;
    tr = 0;
    while (t >= nts - tr) { t -= nts - tr; ++tr; }
    ts = tr + t;
  } else {
    const int64_t ntv = ((n - 1) / 2 - v0) / BT + 1;
    tr = w % ntv; w /= ntv;
    ts = w % nts; w /= nts;
  }
  int64_t P, Q;
  if (PAIR) {                                                    // P <= Q of nq virtual ones
    const double b = 2.0 * (double)nq + 1.0;
    P = (int64_t)((b - sqrt(b * b - 8.0 * (double)w)) * 0.5);
    while (P > 0 && P * (2 * nq - P + 1) / 2 > w) --P;
    while ((P + 1) * (2 * nq - P) / 2 <= w) ++P;
    Q = v0 + P + w - P * (2 * nq - P + 1) / 2;
    P += v0;
  } else if (KIND == K_VOVV) {
    P = v0 + w / nq; Q = w % nq;
  } else {
    P = w / nq; Q = v0 + w % nq;
  }
  const int64_t R0 = v0 + tr * BT, S0 = (TRI ? v0 : 0) + ts * BT;
  const int64_t Rn = n / 2 + (n & 1), Sn = TRI ? Rn : (O + 1) / 2;   // ends of the spatial ranges
  const double2* M = E + (P * m * m + Q) * m;                        // M[x][y] = M[x m^2 + y]
  for (int e = threadIdx.x; e < BT * BT; e += 256) {
    const int64_t x = e / BT, y = e % BT;
    if (R0 + x < Rn && S0 + y < Sn) A[x][y] = M[(R0 + x) * m * m + S0 + y];
    if (S0 + x < Sn && R0 + y < Rn) B[x][y] = M[(S0 + x) * m * m + R0 + y];
  }
  __syncthreads();
  // the contiguous index of the output runs over the lanes: s for the packed columns, else r
  const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
  for (int pq = 0; pq < 4; ++pq) {
    const int64_t p = 2 * P + (pq >> 1), q = 2 * Q + (pq & 1);
    int64_t base;
    if (PAIR) {
      if (p < O || q < O || p >= n || q >= n || p >= q) continue;
      base = (prow(p - O, V) + q - p - 1) * (KIND == K_VVVV_P ? Pv : OV);
    } else if (KIND == K_VOVV) {
      if (p < O || p >= n || q >= O) continue;
      base = ((p - O) * O + q) * Pv;
    } else {
      if (p >= O || q < O || q >= n) continue;
      base = (q - O) * OV + p * V;
    }
    for (int k = grp; k < 2 * BT; k += 4) {
      const int x = TRI ? k : lane, y = TRI ? lane : k;              // spin offsets of r and s in the tile
      const int64_t r = 2 * R0 + x, s = 2 * S0 + y;
      if (r < O || r >= n || (TRI ? s <= r || s >= n : s >= O)) continue;
      double2 v = make_double2(0.0, 0.0);
      if (((p ^ r) & 1) == 0 && ((q ^ s) & 1) == 0) v = A[x >> 1][y >> 1];
      if (((p ^ s) & 1) == 0 && ((q ^ r) & 1) == 0) {
        const double2 u = B[y >> 1][x >> 1];
        v.x -= u.x;
        v.y -= u.y;
      }
      const int64_t o = TRI ? prow(r - O, V) + s - r - 1 : KIND == K_VVVO_P ? s * V + r - O : s * V * OV + r - O;
      if (TRI) out[base + o] = v;
      else put_block(out + base + o, v, past);
    }
  }
}

// The rows form takes a block of N elements from N >= from + 1000 per workgroup on.  Below it the fill of
// the tiles and the passes over the spin pairs (7 to 13 us whatever the size) or the padding of few occupied
// orbitals to 32 cost more than one thread an element does, us elementwise / rows:
//   vvvv_p  m = 16, O = 4  5.1 / 11.2   m = 24, O = 10   9.7 / 13.1   m = 32, O = 20  14.9 / 14.3   m = 48, O = 20  100 / 46
//   ring    m = 16, O = 4  3.7 / 6.8    m = 36, O = 20   7.7 / 9.4    m = 40, O = 20   9.4 / 9.4    m = 48, O = 20  13.5 / 10.4
//   vvvo_p  m = 16, O = 4  3.6 / 7.4    m = 48, O = 4   15.6 / 22.2   m = 32, O = 20   9.8 / 9.4    m = 48, O = 20  36.5 / 20.7
//   vovv_p  m = 16, O = 4  3.5 / 10.3   m = 36, O = 20  15.2 / 16.0   m = 40, O = 20  21.0 / 17.6   m = 48, O = 10  29.0 / 20.4
template <int KIND>
int launch_pair_rows(const double2* E, int64_t m, int64_t O, int64_t V, int past, void* out, hipStream_t st,
                     unsigned& done) {
  const int64_t N = kind_size(KIND, O, V);
  if (!out || N <= 0) return APY_OK;
  constexpr bool TRI = KIND == K_VVVV_P || KIND == K_VOVV, PAIR = KIND == K_VVVV_P || KIND == K_VVVO_P;
  constexpr int64_t from = KIND == K_VVVV_P ? 500000 : KIND == K_VVVO_P ? 330000 : KIND == K_VOVV ? 1500000 : 1200000;
  const int64_t nv = m - O / 2, no = (O + 1) / 2, ntv = (nv + BT - 1) / BT, nto = (no + BT - 1) / BT;
  const int64_t nq = PAIR ? nv : KIND == K_VOVV ? no : nv;
  const int64_t pairs = PAIR ? nv * (nv + 1) / 2 : nv * no, tiles = TRI ? ntv * (ntv + 1) / 2 : ntv * nto;
  if (pairs * tiles > 0x7fffffffLL || N < from + 1000 * pairs * tiles) return APY_OK;
  build_pair_rows<KIND><<<(unsigned)(pairs * tiles), 256, 0, st>>>(E, m, O, V, nq, TRI ? ntv : nto, past, (double2*)out);
  APY_LAUNCH_CHECK();
  done |= 1u << KIND;
  return APY_OK;
}

void* block_ptr(const apy_so_ints* I, int kind) {
  switch (kind) {
    case K_VVVV_P: return I->vvvv_p;
    case K_RING: return I->ring;
    case K_OOOO_P: return I->oooo_p;
    case K_OVOO_P: return I->ovoo_p;
    case K_VVVO_P: return I->vvvo_p;
    case K_VOVV: return I->vovv_p;
    case K_OOOV: return I->ooov;
    case K_VVOO_T: return I->vvoo_t;
    case K_OOVV: return I->oovv;
  }
  return nullptr;
}

int stored_past(const apy_so_ints* I) {
  int64_t n = 0;
  for (int kind = 0; kind < K_COUNT; ++kind)
    if (block_ptr(I, kind)) n += std::max<int64_t>(kind_size(kind, I->O, I->V), 0);
  return n >= NT_ELEMENTS;
}

template <class Src>
int build_all(const Src& src, const apy_so_ints* I, int accumulate, double scale, hipStream_t st,
              unsigned skip = 0) {
  if (!I || I->O < 0 || I->V < 0) return APY_E_ARG;
  const int past = stored_past(I);
  for (int kind = 0; kind < K_COUNT; ++kind) {
    if (skip >> kind & 1) continue;
    double2* out = (double2*)block_ptr(I, kind);
    if (!out) continue;
    int64_t total = kind_size(kind, I->O, I->V);
    if (total <= 0) continue;
    build_block<Src><<<apy_grid1d(total, 1 << 20), 256, 0, st>>>(src, kind, I->O, I->V, out, total, accumulate,
                                                                 scale, past);
    APY_LAUNCH_CHECK();
  }
  return APY_OK;
}

__global__ void so_fock_kernel(int64_t m, int64_t nb, const double2* fmo, double2* fso) {
  const int64_t n = 2 * m, total = nb * n * n;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = t / n, p = r % n, q = t % n;
    fso[t] = ((p ^ q) & 1) ? make_double2(0.0, 0.0) : fmo[((r / n) * m + (p >> 1)) * m + (q >> 1)];
  }
}

// ------------------------------------------------------------ sigma pieces
// Every sigma works from the packed doubles T_p[(i<j)][(a<b)] (the packed
// input itself, or those of a dense input); the dense images the GEMMs
// need are expanded from it with the antisymmetry signs.
//
// One launch forms all of them: the grid is cut into sections (in blocks), so that the small copies of a
// step do not follow each other at a launch's latency each (five launches of 2 to 5 us at O=10 V=4 and
// O=18 V=50 alike).  A dense input is read at its i < j, a < b elements, which are T_p.
struct PrepArgs {
  int64_t O, V;
  const double2* t2;       // dense input [i][j][a][b] (NULL: tp_in is read)
  const double2* tp_in;    // packed input
  double2* tp;             // T_p of a dense input
  double2* tr;             // T'[(i,a),(k,c)]
  double2* th;             // Th[i][j][(c<b)] (NULL: none)
  const double2* ov;       // ovoo_p (NULL: no transposes)
  double2* ovT;            // [(i<j)][k][b] = <kb||ij>
  const double2* oo;       // ooov
  double2* ooT;            // [k][i][(j,b)] = <kj||ib>
  int32_t ring, pack, half, ovb;   // ends of the sections in blocks; the rest: ooT
};

__device__ inline int64_t pidx(int64_t p, int64_t q, int64_t N) { return prow(p, N) + q - p - 1; }

constexpr int RT = 32;      // edge of a ring tile
constexpr int PREP_E = 512; // elements of a block of the other sections

__global__ __launch_bounds__(256) void prep_kernel(PrepArgs p) {
  __shared__ double2 T[RT][RT + 1];
  const int64_t O = p.O, V = p.V, Po = npair(O), Pv = npair(V), OV = O * V;
  const int blk = (int)blockIdx.x;
  if (blk < p.ring) {
    // T'[(i,a),(k,c)] = t2[i,k,a,c]: +T_p[(ik),(ac)] when i<k and a<c (or both reversed), minus when one
    // pair is reversed, zero on i == k or a == c.  One block per (i, k, 32 x 32 tile of (a, c)): the row
    // (ik) is read in two passes, the a < c half with c fastest and the a > c half with a fastest, so that
    // both read along it; the tile goes through LDS and out along c.
    const int64_t nt = (V + RT - 1) / RT;
    const int tx = threadIdx.x % RT, ty = threadIdx.x / RT;
    const int64_t tc = blk % nt, ta = (blk / nt) % nt, k = (blk / (nt * nt)) % O, i = blk / (nt * nt * O);
    const int64_t a0 = ta * RT, c0 = tc * RT, lo = i < k ? i : k, hi = i < k ? k : i;
    const double2* row = i == k ? nullptr : p.t2 ? p.t2 + (lo * O + hi) * V * V : p.tp_in + pidx(lo, hi, O) * Pv;
    auto at = [&](int64_t x, int64_t y) { return p.t2 ? x * V + y : pidx(x, y, V); };   // x < y
    const double su = i < k ? 1.0 : -1.0;     // sign of the a < c half; the a > c half has -su
#pragma unroll
    for (int r = 0; r < RT / 8; ++r) {
      const int ra = ty + 8 * r;
      // upper pass (c fastest): a < c, and every slot the lower pass does not cover (zeros)
      const int64_t a = a0 + ra, c = c0 + tx;
      if (!(row && a < V && c < V && a > c)) {
        double2 x = make_double2(0.0, 0.0);
        if (row && a < V && c < V && a < c) {
          const double2 y = row[at(a, c)];
          x = make_double2(su * y.x, su * y.y);
        }
        T[ra][tx] = x;
      }
      // lower pass (a fastest): a > c
      const int64_t al = a0 + tx, cl = c0 + ra;
      if (row && al < V && cl < V && al > cl) {
        const double2 y = row[at(cl, al)];
        T[tx][ra] = make_double2(-su * y.x, -su * y.y);
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RT / 8; ++r) {
      const int64_t a = a0 + ty + 8 * r, c = c0 + tx;
      if (a < V && c < V) p.tr[(i * V + a) * OV + k * V + c] = T[ty + 8 * r][tx];
    }
    return;
  }
  const int first = blk < p.pack ? p.ring : blk < p.half ? p.pack : blk < p.ovb ? p.half : p.ovb;
#pragma unroll
  for (int u = 0; u < PREP_E / 256; ++u) {
    const int64_t t = (int64_t)(blk - first) * PREP_E + u * 256 + threadIdx.x;
    if (blk < p.pack) {                        // T_p of a dense input
      if (t >= Po * Pv) return;
      int64_t i, j, a, b;
      pdec(t / Pv, O, i, j);
      pdec(t % Pv, V, a, b);
      p.tp[t] = p.t2[((i * O + j) * V + a) * V + b];
    } else if (blk < p.half) {                 // Th[i][j][(c<b)] = t2[i,j,c,b], zero rows for i == j
      if (t >= O * O * Pv) return;
      const int64_t P = t % Pv, j = (t / Pv) % O, i = t / (Pv * O), lo = i < j ? i : j, hi = i < j ? j : i;
      double2 v = make_double2(0.0, 0.0);
      if (i != j) {
        if (p.t2) {
          int64_t c, b;
          pdec(P, V, c, b);
          v = p.t2[((lo * O + hi) * V + c) * V + b];
        } else {
          v = p.tp_in[pidx(lo, hi, O) * Pv + P];
        }
        if (i > j) v = make_double2(-v.x, -v.y);
      }
      p.th[t] = v;
    } else if (blk < p.ovb) {                  // ovT
      if (t >= Po * OV) return;
      const int64_t b = t % V, k = (t / V) % O, P = t / OV;
      p.ovT[t] = p.ov[(k * V + b) * Po + P];
    } else {                                   // ooT
      if (t >= O * O * OV) return;
      const int64_t b = t % V, j = (t / V) % O, i = (t / OV) % O, k = t / (OV * O);
      p.ooT[t] = p.oo[((k * O + j) * O + i) * V + b];
    }
  }
}

int launch_prep(PrepArgs p, hipStream_t st) {
  const int64_t nt = (p.V + RT - 1) / RT, Po = npair(p.O), Pv = npair(p.V), OV = p.O * p.V;
  auto blocks = [](int64_t n) { return (n + PREP_E - 1) / PREP_E; };
  int64_t e = p.O * p.O * nt * nt;
  p.ring = (int32_t)e;
  e += p.t2 ? blocks(Po * Pv) : 0;
  p.pack = (int32_t)e;
  e += p.th ? blocks(p.O * p.O * Pv) : 0;
  p.half = (int32_t)e;
  e += p.ov ? blocks(Po * OV) : 0;
  p.ovb = (int32_t)e;
  e += p.ov ? blocks(p.O * p.O * OV) : 0;
  if (e > 0x7fffffffLL) return APY_E_ARG;
  prep_kernel<<<(unsigned)e, 256, 0, st>>>(p);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

__global__ __launch_bounds__(256) void ring_fock_kernel(int64_t O, int64_t V, const double2* __restrict__ F,
                                                        const double2* __restrict__ ring, double2* __restrict__ rf) {
  const int64_t n = O + V, OV = O * V, total = OV * OV;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = t / OV, col = t % OV;
    double2 v = ring[t];
    if (row / V == col / V) {
      const double2 f = F[(O + row % V) * n + O + col % V];
      v.x += 0.5 * f.x;
      v.y += 0.5 * f.y;
    }
    rf[t] = v;
  }
}

__global__ void pair_oo_kernel(const double2* __restrict__ oooo_p, const double2* __restrict__ F, int64_t n,
                               int64_t O, double2* __restrict__ hoo) {
  const int64_t Po = npair(O), total = Po * Po;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    int64_t i, j, k, l;
    pdec(t / Po, O, i, j);
    pdec(t % Po, O, k, l);
    double2 v = oooo_p ? oooo_p[t] : make_double2(0.0, 0.0);
    // -sum_m F_mj t2[i,m] - sum_m F_mi t2[m,j] expressed on t2[(k<l)]
    if (k == i) { double2 f = F[l * n + j]; v.x -= f.x; v.y -= f.y; }
    if (l == i) { double2 f = F[k * n + j]; v.x += f.x; v.y += f.y; }
    if (l == j) { double2 f = F[k * n + i]; v.x -= f.x; v.y -= f.y; }
    if (k == j) { double2 f = F[l * n + i]; v.x += f.x; v.y += f.y; }
    hoo[t] = v;
  }
}

__device__ inline void acc(double2& s, double2 v) { s.x += v.x; s.y += v.y; }
__device__ inline void dec(double2& s, double2 v) { s.x -= v.x; s.y -= v.y; }
__device__ inline double2 cm(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline void cfma(double2& s, double2 a, double2 b) {
  s.x += a.x * b.x - a.y * b.y;
  s.y += a.x * b.y + a.y * b.x;
}

// ------------------------------------------------------------ doubles epilogue
// One workgroup per (i<j) pair and pair of 32-wide virtual tiles (A <= B);
// thread (ty, tx) owns a = a0 + ty + 8q (q = 0..3), b = b0 + tx, a < b.  It sums
//   c0 <ab||ij> + R_p + X[(ia),(jb)] - X[(ja),(ib)] - X[(ib),(ja)] + X[(jb),(ia)]
//   + Q_T[j][i][(ab)] - Q_T[i][j][(ab)] - U_ab + U_ba   (U_ab = sum_k t1[k,a] <kb||ij>)
//   + the f_bj t_ia coupling (Hermitian operator only)
// -- the reference's doubles terms of ci_wfn.py:319-334 regrouped (F_vv is in X).
// The two X blocks read transposed go through LDS so every global access is a
// row segment.  Output: packed s (sigma) or, in residual mode, r = s - E t and
// t + r/D; dense outputs write the four antisymmetric images, the two
// transposed ones through LDS again.
constexpr int ET = 32;   // virtual tile edge
constexpr int EKC = 8;   // occupied chunk of the in-kernel U contraction

struct Epi2Args {
  int64_t O, V, Po, Pv, n;
  int ntile;
  const double2* drv;      // vvoo_t [i][j][a][b] = <ab||ij> (NULL: no driver term)
  const double2* Rp;       // [(ij)][(ab)]
  const double2* X;        // [(i,a)][(j,b)]
  const double2* QT;       // Q_T[j][i][(ab)] at QT + j*qj + i*Pv (NULL: no T1 -> T2 terms)
  int64_t qj;
  const double2* ovT;      // [(ij)][k][b] = <kb||ij>
  const double2* t1;       // [i][a]
  const double2* F;        // [n][n]
  int fov;
  const double* eps;
  const double2* E;
  double c0r, c0i;
  const double2* c0p;
  const double2* Tp;       // packed t2 (residual mode)
  double2* out;            // packed [(ij)][(ab)] or dense [i][j][a][b]
  double2* tn;             // residual mode: t + r/D, same layout as out
  int mode;
  int packed;
  const double2* s1;       // singles accumulator (NULL: no singles in this launch)
  double2* out1;
  double2* tn1;
  int32_t doubles;         // blocks of the doubles (0: singles only); the singles' blocks follow
};

__device__ inline void epi_dense_transposed(const Epi2Args& e, double2 (*L)[ET + 1], double2* base, int64_t i,
                                            int64_t j, int64_t a0, int64_t b0, int ty, int tx) {
  // base[i][j][b][a] = -v(a,b), base[j][i][b][a] = +v(a,b) for the tile's
  // values v(a,b) held in L[a - a0][b - b0]; rows b, lanes over a.
  const int64_t O = e.O, V = e.V;
  for (int q = 0; q < ET / 8; ++q) {
    const int lb = ty + 8 * q;
    const int64_t b = b0 + lb, a = a0 + tx;
    if (b < V && a < b) {
      const double2 v = L[tx][lb];
      base[((i * O + j) * V + b) * V + a] = make_double2(-v.x, -v.y);
      base[((j * O + i) * V + b) * V + a] = v;
    }
  }
}

__device__ __forceinline__ void epi2_doubles(const Epi2Args& e) {
  __shared__ double2 L[ET][ET + 1];
  __shared__ double2 sA[EKC][ET], sB[EKC][ET], oA[EKC][ET], oB[EKC][ET];
  const int tid = threadIdx.x, tx = tid & (ET - 1), ty = tid >> 5;
  const int64_t O = e.O, V = e.V, OV = O * V, Pv = e.Pv;
  const int ntp = e.ntile * (e.ntile + 1) / 2;
  const int64_t Pij = blockIdx.x / ntp;
  int tp = (int)(blockIdx.x % ntp), ta = 0;
  while (tp >= e.ntile - ta) { tp -= e.ntile - ta; ++ta; }
  const int tb = ta + tp;
  const int64_t a0 = (int64_t)ta * ET, b0 = (int64_t)tb * ET;
  int64_t i, j;
  pdec(Pij, O, i, j);

  // The reads of each part are issued before the first is used, outside a < b at the pair (0, 1): under
  // conditions they followed each other at a read's latency.
  constexpr int NK = ET / 8;
  const double2 c0 = e.c0p ? *e.c0p : make_double2(e.c0r, e.c0i);
  {
    // transposed X blocks: L[lb][la] = -X[(i,b),(j,a)] + X[(j,b),(i,a)]
    double2 x3[NK], x4[NK];
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      int64_t b = b0 + ty + 8 * q, a = a0 + tx;
      if (b >= V || a >= b) { a = 0; b = 1; }
      x3[q] = e.X[(i * V + b) * OV + j * V + a];
      x4[q] = e.X[(j * V + b) * OV + i * V + a];
    }
#pragma unroll
    for (int q = 0; q < NK; ++q) L[ty + 8 * q][tx] = make_double2(x4[q].x - x3[q].x, x4[q].y - x3[q].y);
  }

  double2 s[NK];
  {
    double2 dv[NK], rp[NK], x1[NK], x2[NK], q1[NK], q2[NK];
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      int64_t a = a0 + ty + 8 * q, b = b0 + tx;
      if (b >= V || a >= b) { a = 0; b = 1; }
      const int64_t Pab = pidx(a, b, V);
      if (e.drv) dv[q] = e.drv[((i * O + j) * V + a) * V + b];
      rp[q] = e.Rp[Pij * Pv + Pab];
      x1[q] = e.X[(i * V + a) * OV + j * V + b];
      x2[q] = e.X[(j * V + a) * OV + i * V + b];
      if (e.QT) {
        q1[q] = e.QT[j * e.qj + i * Pv + Pab];
        q2[q] = e.QT[i * e.qj + j * Pv + Pab];
      }
    }
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      const int64_t a = a0 + ty + 8 * q, b = b0 + tx;
      double2 v = make_double2(0.0, 0.0);
      if (b < V && a < b) {
        if (e.drv) v = cm(c0, dv[q]);
        acc(v, rp[q]);
        acc(v, x1[q]);
        dec(v, x2[q]);
        if (e.QT) {
          acc(v, q1[q]);
          dec(v, q2[q]);
        }
        if (e.fov) {
          const int64_t n = e.n;
          cfma(v, e.F[(O + b) * n + j], e.t1[i * V + a]);
          cfma(v, e.F[(O + a) * n + i], e.t1[j * V + b]);
          const double2 m1 = cm(e.F[(O + b) * n + i], e.t1[j * V + a]);
          const double2 m2 = cm(e.F[(O + a) * n + j], e.t1[i * V + b]);
          v.x -= m1.x + m2.x;
          v.y -= m1.y + m2.y;
        }
      }
      s[q] = v;
    }
  }

  // T1 -> T2 through <kb||ij>: -U_ab + U_ba, U_ab = sum_k t1[k,a] <kb||ij>
  if (e.QT) {
    double2 u[ET / 8];
    for (int q = 0; q < ET / 8; ++q) u[q] = make_double2(0.0, 0.0);
    const double2* ov = e.ovT + Pij * O * V;
    for (int64_t k0 = 0; k0 < O; k0 += EKC) {
      __syncthreads();
      {
        const int kk = ty;                     // 8 rows x 32 lanes: one element of each array per thread
        const int64_t k = k0 + kk, a = a0 + tx, b = b0 + tx;
        const bool kv = k < O;
        sA[kk][tx] = (kv && a < V) ? e.t1[k * V + a] : make_double2(0.0, 0.0);
        sB[kk][tx] = (kv && b < V) ? e.t1[k * V + b] : make_double2(0.0, 0.0);
        oA[kk][tx] = (kv && a < V) ? ov[k * V + a] : make_double2(0.0, 0.0);
        oB[kk][tx] = (kv && b < V) ? ov[k * V + b] : make_double2(0.0, 0.0);
      }
      __syncthreads();
      for (int q = 0; q < ET / 8; ++q) {
        const int la = ty + 8 * q;
        for (int kk = 0; kk < EKC; ++kk) {
          const double2 x = cm(sA[kk][la], oB[kk][tx]);   // t1[k,a] <kb||ij>
          const double2 y = cm(sB[kk][tx], oA[kk][la]);   // t1[k,b] <ka||ij>
          u[q].x += y.x - x.x;
          u[q].y += y.y - x.y;
        }
      }
    }
    for (int q = 0; q < ET / 8; ++q) acc(s[q], u[q]);
  }
  __syncthreads();                             // L complete
  for (int q = 0; q < ET / 8; ++q) acc(s[q], L[tx][ty + 8 * q]);

  double2 tnv[ET / 8];
  if (e.mode == APY_MODE_RESIDUAL) {
    const double2 E = *e.E;
    for (int q = 0; q < ET / 8; ++q) {
      const int64_t a = a0 + ty + 8 * q, b = b0 + tx;
      if (b < V && a < b) {
        const double2 tv = e.Tp[Pij * Pv + pidx(a, b, V)];
        dec(s[q], cm(E, tv));
        const double D = e.eps[i] + e.eps[j] - e.eps[O + a] - e.eps[O + b];
        tnv[q] = make_double2(tv.x + s[q].x / D, tv.y + s[q].y / D);
      } else {
        tnv[q] = make_double2(0.0, 0.0);
      }
    }
  }

  if (e.packed) {
    for (int q = 0; q < ET / 8; ++q) {
      const int64_t a = a0 + ty + 8 * q, b = b0 + tx;
      if (b < V && a < b) {
        const int64_t o = Pij * Pv + pidx(a, b, V);
        e.out[o] = s[q];
        if (e.mode == APY_MODE_RESIDUAL) e.tn[o] = tnv[q];
      }
    }
    return;
  }
  // dense: direct images [i][j][a][b] = v, [j][i][a][b] = -v
  for (int q = 0; q < ET / 8; ++q) {
    const int64_t a = a0 + ty + 8 * q, b = b0 + tx;
    if (b < V && a < b) {
      e.out[((i * O + j) * V + a) * V + b] = s[q];
      e.out[((j * O + i) * V + a) * V + b] = make_double2(-s[q].x, -s[q].y);
      if (e.mode == APY_MODE_RESIDUAL) {
        e.tn[((i * O + j) * V + a) * V + b] = tnv[q];
        e.tn[((j * O + i) * V + a) * V + b] = make_double2(-tnv[q].x, -tnv[q].y);
      }
    }
  }
  // transposed images through LDS
  __syncthreads();
  for (int q = 0; q < ET / 8; ++q) L[ty + 8 * q][tx] = s[q];
  __syncthreads();
  epi_dense_transposed(e, L, e.out, i, j, a0, b0, ty, tx);
  if (e.mode == APY_MODE_RESIDUAL) {
    __syncthreads();
    for (int q = 0; q < ET / 8; ++q) L[ty + 8 * q][tx] = tnv[q];
    __syncthreads();
    epi_dense_transposed(e, L, e.tn, i, j, a0, b0, ty, tx);
  }
}

__device__ __forceinline__ void epi_singles(const Epi2Args& e, int64_t t) {
  const int64_t O = e.O, V = e.V;
  if (t >= O * V) return;
  const double2 c0 = e.c0p ? *e.c0p : make_double2(e.c0r, e.c0i);
  const int64_t i = t / V, a = t % V;
  const double2 f = e.F[(O + a) * e.n + i];
  double2 s = e.s1[t];
  s.x += c0.x * f.x - c0.y * f.y;
  s.y += c0.x * f.y + c0.y * f.x;
  if (e.mode == APY_MODE_RESIDUAL) {
    const double2 tv = e.t1[t], E = *e.E;
    s.x -= E.x * tv.x - E.y * tv.y;
    s.y -= E.x * tv.y + E.y * tv.x;
    const double D = e.eps[i] - e.eps[O + a];
    e.tn1[t] = make_double2(tv.x + s.x / D, tv.y + s.y / D);
  }
  e.out1[t] = s;
}

__global__ __launch_bounds__(256) void epi_kernel(Epi2Args e) {
  if ((int)blockIdx.x >= e.doubles) {
    epi_singles(e, (int64_t)((int)blockIdx.x - e.doubles) * 256 + threadIdx.x);
    return;
  }
  epi2_doubles(e);
}

// Both epilogues in one launch, unless the singles are written over the t1 that the doubles still read
// (a step with t_new == t).
int launch_epi(Epi2Args e, int64_t t_len, hipStream_t st) {
  const int64_t nt = (e.V + ET - 1) / ET, nd = npair(e.O) * (nt * (nt + 1) / 2), ns = (e.O * e.V + 255) / 256;
  if (nd + ns > 0x7fffffffLL) return APY_E_ARG;
  auto hits = [&](const double2* p) { return p && p < e.t1 + t_len && e.t1 < p + t_len; };
  e.doubles = (int32_t)nd;
  const bool split = e.s1 && (hits(e.out1) || (e.mode == APY_MODE_RESIDUAL && hits(e.tn1)));
  epi_kernel<<<(unsigned)(nd + (e.s1 && !split ? ns : 0)), 256, 0, st>>>(e);
  APY_LAUNCH_CHECK();
  if (split) {
    e.doubles = 0;
    epi_kernel<<<(unsigned)ns, 256, 0, st>>>(e);
    APY_LAUNCH_CHECK();
  }
  return APY_OK;
}

// Energy partial sums: terms l < OV are t1[i,a] f[i,O+a]; the rest 1/4 t2*oovv
// (dense) or t2p*oovv over (i<j, a<b) (packed).
__global__ __launch_bounds__(256) void energy_partial(int64_t O, int64_t V, int64_t n, int singles, int packed,
                                                      const double2* __restrict__ F, const double2* __restrict__ oovv,
                                                      const double2* __restrict__ t, double2* partial) {
  const int64_t OV = O * V;
  double sr = 0.0, si = 0.0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (singles) {
    for (int64_t q = l; q < OV; q += stride) {
      const int64_t i = q / V, a = q % V;
      double2 x = t[q], f = F[i * n + O + a];
      sr += x.x * f.x - x.y * f.y;
      si += x.x * f.y + x.y * f.x;
    }
  }
  double qr = 0.0, qi = 0.0;
  if (!oovv) {
    // one-electron part only: no doubles term
  } else if (packed) {
    const int64_t Pv = npair(V), L2 = npair(O) * Pv;
    for (int64_t q = l; q < L2; q += stride) {
      int64_t i, j, a, b;
      pdec(q / Pv, O, i, j);
      pdec(q % Pv, V, a, b);
      const double2 x = t[OV + q], w = oovv[((i * O + j) * V + a) * V + b];
      qr += x.x * w.x - x.y * w.y;
      qi += x.x * w.y + x.y * w.x;
    }
  } else {
    const int64_t L2 = O * O * V * V;
    for (int64_t q = l; q < L2; q += stride) {
      double2 x = t[OV + q], w = oovv[q];
      qr += x.x * w.x - x.y * w.y;
      qi += x.x * w.y + x.y * w.x;
    }
    qr *= 0.25;
    qi *= 0.25;
  }
  sr += qr;
  si += qi;
  __shared__ double rs[256], is[256];
  rs[threadIdx.x] = sr;
  is[threadIdx.x] = si;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) { rs[threadIdx.x] += rs[threadIdx.x + w]; is[threadIdx.x] += is[threadIdx.x + w]; }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(rs[0], is[0]);
}

__global__ void finalize_sum(const double2* __restrict__ partial, int np, double2* out) {
  __shared__ double rs[256], is[256];
  double sr = 0.0, si = 0.0;
  for (int q = threadIdx.x; q < np; q += blockDim.x) { sr += partial[q].x; si += partial[q].y; }
  rs[threadIdx.x] = sr;
  is[threadIdx.x] = si;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) { rs[threadIdx.x] += rs[threadIdx.x + w]; is[threadIdx.x] += is[threadIdx.x + w]; }
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = make_double2(rs[0], is[0]);
}

constexpr int ENERGY_BLOCKS = 1024;

// Blocks of the energy's partial sums over n terms: four terms a thread, and one block (which then writes
// the energy itself) where a second launch would take longer than the terms do.
inline int energy_blocks(int64_t n) {
  if (n <= 4096) return 1;
  return (int)std::min<int64_t>(ENERGY_BLOCKS, (n + 1023) / 1024);
}

int launch_energy(int64_t O, int64_t V, int singles, int packed, const double2* F, const double2* oovv,
                  const double2* t, double2* part, double2* energy, hipStream_t st) {
  const int nb = energy_blocks(O * V + (packed ? npair(O) * npair(V) : O * O * V * V));
  energy_partial<<<nb, 256, 0, st>>>(O, V, O + V, singles, packed, F, oovv, t, nb > 1 ? part : energy);
  APY_LAUNCH_CHECK();
  if (nb > 1) {
    finalize_sum<<<1, 256, 0, st>>>(part, nb, energy);
    APY_LAUNCH_CHECK();
  }
  return APY_OK;
}

inline size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

void fill(apy_gemm_desc& d, int64_t m, int64_t n, int64_t k, int al, const void* a, int64_t lda, int bl,
          const void* b, int64_t ldb, void* c, int64_t ldc, double alr, double ber) {
  d = apy_gemm_desc{};
  d.m = m; d.n = n; d.k = k;
  d.a_layout = al; d.b_layout = bl;
  d.alpha_re = alr; d.beta_re = ber;
  d.a = a; d.lda = lda; d.b = b; d.ldb = ldb; d.c = c; d.ldc = ldc;
  d.batch = 1;
}

// Workspace of nb instances (nb = 1: one sigma step).  Regions hold
// [nb][...] per buffer; tp only for dense inputs.
struct SigmaWS {
  double2 *tp, *rp, *tr, *X, *QT, *th, *ovT, *ooT, *s1, *t1;
  void* gemm;
  size_t gemm_bytes;
  size_t total;
};

// The GEMMs of a step over nb instances (nb = 1 for apy_cisd_so_step).
//   t[k]      the instance's vector ([t1 | t2...]; only t1 is read here)
//   F[k]      its Fock matrix, hoo[k] its pair operator
//   ring_f    (nb == 1 only, optional) the ring block with F_vv folded in
// With null pointers the list is built only to size the workspace.
//   g3        the PPL and ring products in the three-product complex form
void sigma_gemms(int64_t O, int64_t V, int nb, int singles, const apy_so_ints* I, const double2* const* F,
                 const void* const* hoo, const double2* const* t, const void* ring_f, const SigmaWS& w,
                 std::vector<apy_gemm_desc>& G, int g3 = 0) {
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V, n = O + V;
  const int64_t PP = Po * Pv, R2 = OV * OV;
  G.clear();
  apy_gemm_desc d;
  auto off = [](const double2* p, int64_t o) -> const double2* { return p ? p + o : nullptr; };
  auto offw = [](double2* p, int64_t o) -> double2* { return p ? p + o : nullptr; };
  // [0] PPL over all instances: R_p = T_p . vvvv_p^T
  fill(d, nb * Po, Pv, Pv, APY_MK, w.tp, Pv, APY_NK, I ? I->vvvv_p : nullptr, Pv, w.rp, Pv, 1.0, 0.0);
  d.gauss3m = g3;
  G.push_back(d);
  // [1] ring over all instances: X = T' . ring^T (ring_f: F_vv folded in)
  fill(d, nb * OV, OV, OV, APY_MK, w.tr, OV, APY_NK, ring_f ? ring_f : (I ? I->ring : nullptr), OV, w.X, OV, 1.0, 0.0);
  d.gauss3m = g3;
  G.push_back(d);
  if (singles) {
    // Q_T[j][(k,i)][(ab)] = sum_c t1_k[i,c] <ab||cj>: batched over j, all instances' t1 stacked along M
    fill(d, nb * O, Pv, V, APY_MK, w.t1, V, APY_NK, I ? I->vvvo_p : nullptr, O * V, w.QT, Pv, 1.0, 0.0);
    d.batch = O; d.stride_a = 0; d.stride_b = V; d.stride_c = (int64_t)nb * O * Pv;
    G.push_back(d);
    // s1 += 1/2 sum_(jcb) t2 <aj||cb> = sum_j sum_(c<b) Th[(k,i)][(j,cb)] vovv_p[a][(j,cb)], all instances
    fill(d, nb * O, V, O * Pv, APY_MK, w.th, O * Pv, APY_NK, I ? I->vovv_p : nullptr, O * Pv, w.s1, V, 1.0, 0.0);
    G.push_back(d);
    // s1 += ring . t1 (all instances: M = nb)
    fill(d, nb, OV, OV, APY_MK, w.t1, OV, APY_NK, I ? I->ring : nullptr, OV, w.s1, OV, 1.0, 1.0);
    G.push_back(d);
  }
  for (int k = 0; k < nb; ++k) {
    const double2* Fk = F ? F[k] : nullptr;
    const double2* trk = off(w.tr, k * R2);
    double2* s1 = offw(w.s1, k * OV);
    // HHL + F_oo: R_p += Hoo . T_p
    fill(d, Po, Pv, Po, APY_MK, hoo ? hoo[k] : nullptr, Po, APY_KN, off(w.tp, k * PP), Pv, offw(w.rp, k * PP), Pv,
         1.0, 1.0);
    G.push_back(d);
    if (!ring_f) {
      // F_vv into X: X[(i,a,j)][b] += 1/2 sum_c T'[(i,a,j)][c] F[O+b][O+c]
      fill(d, O * V * O, V, V, APY_MK, trk, V, APY_NK, Fk ? Fk + O * n + O : nullptr, n, offw(w.X, k * R2), V, 0.5,
           1.0);
      G.push_back(d);
    }
    if (!singles) continue;
    const double2* t1 = t ? t[k] : nullptr;
    // s1 += t1 F_vv^T
    fill(d, O, V, V, APY_MK, t1, V, APY_NK, Fk ? Fk + O * n + O : nullptr, n, s1, V, 1.0, 1.0);
    G.push_back(d);
    // s1 -= F_oo^T t1
    fill(d, O, V, O, APY_KM, Fk, n, APY_KN, t1, V, s1, V, -1.0, 1.0);
    G.push_back(d);
    // s1[(ia)] += sum_j sum_b T'[(ia),(jb)] F[j][O+b]
    fill(d, OV, 1, V, APY_MK, trk, OV, APY_KN, Fk ? Fk + O : nullptr, 1, s1, 1, 1.0, 1.0);
    d.batch = O; d.stride_a = V; d.stride_b = n; d.stride_c = 0; d.reduce_batch = 1;
    G.push_back(d);
    // s1[i][a] -= 1/2 sum_k sum_(jb) <kj||ib> T'[(k,a),(j,b)]
    fill(d, O, V, OV, APY_MK, w.ooT, OV, APY_NK, trk, OV, s1, V, -0.5, 1.0);
    d.batch = O; d.stride_a = O * OV; d.stride_b = V * OV; d.stride_c = 0; d.reduce_batch = 1;
    G.push_back(d);
  }
}

// exact = 1 sizes the GEMM region for the plans that would run now instead of
// every plan the tuner may pick (the no-allocation entry point); grouped = 1: at
// least the partial sums of the products in one launch (a query's size; they are
// far below the largest single product's, and where a step's workspace does not
// hold them the products run one after another).
SigmaWS carve(int64_t O, int64_t V, int nb, int singles, int dense_in, const void* ring_f, void* base,
              int exact = 0, int grouped = 0) {
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V;
  SigmaWS w{};
  size_t off = 0;
  char* b = base ? (char*)base : (char*)256;     // a query's addresses are only compared with each other
  auto take = [&](size_t elems) -> double2* {
    double2* p = (double2*)(b + off);
    off += al256(elems * sizeof(double2));
    return p;
  };
  if (dense_in) w.tp = take((size_t)nb * Po * Pv);
  w.rp = take((size_t)nb * Po * Pv);
  w.tr = take((size_t)nb * OV * OV);
  w.X = take((size_t)nb * OV * OV);
  if (singles) {
    w.QT = take((size_t)O * nb * O * Pv);
    w.th = take((size_t)nb * O * O * Pv);
    w.ovT = take((size_t)Po * O * V);
    w.ooT = take((size_t)O * O * OV);
    w.s1 = take((size_t)nb * OV);
    w.t1 = take((size_t)nb * OV);
  }
  // GEMM split-K workspace: the largest any of the step's GEMMs asks for.
  std::vector<apy_gemm_desc> G;
  sigma_gemms(O, V, nb, singles, nullptr, nullptr, nullptr, nullptr, ring_f, w, G);
  size_t g = 0;
  for (const apy_gemm_desc& d : G) g = std::max(g, exact ? apy_zgemm_plan_ws_bytes(&d) : apy_zgemm_ws_bytes(&d));
  if (grouped) g = std::max(g, apy_zgemm_group_ws_bytes(G.data(), (int)G.size()));
  w.gemm = (void*)(b + off);
  w.gemm_bytes = g;
  off += al256(g);
  w.total = off;
  return w;
}

// Everything of a sigma over nb instances up to the epilogues: the packed
// doubles (tp: the caller's packed inputs when tp_in is given), the dense
// images, the transposed integral pieces and all GEMMs.
int sigma_body(int64_t O, int64_t V, int nb, int singles, const apy_so_ints* I, const double2* const* F,
               const void* const* hoo, const double2* const* t, int packed_in, const void* ring_f, SigmaWS& w,
               hipEvent_t ev0, hipEvent_t ev1, hipStream_t st, int g3) {
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V, PP = Po * Pv;
  if (packed_in) {
    if (nb != 1) return APY_E_ARG;
    w.tp = (double2*)(t[0] + OV);      // T_p is the packed input itself
  }
  if (singles && nb == 1) w.t1 = (double2*)t[0];   // one instance: t1 read in place
  for (int k = 0; k < nb; ++k) {
    double2* tpk = w.tp + k * PP;
    PrepArgs p{};
    p.O = O; p.V = V;
    p.t2 = packed_in ? nullptr : t[k] + OV;
    p.tp_in = tpk;
    p.tp = tpk;
    p.tr = w.tr + k * OV * OV;
    if (singles) p.th = w.th + k * O * O * Pv;
    if (singles && k == 0) {
      p.ov = (const double2*)I->ovoo_p; p.ovT = w.ovT;
      p.oo = (const double2*)I->ooov; p.ooT = w.ooT;
    }
    const int s = launch_prep(p, st);
    if (s != APY_OK) return s;
    if (singles && nb > 1)
      APY_HIP_TRY(hipMemcpyAsync(w.t1 + k * OV, t[k], OV * sizeof(double2), hipMemcpyDeviceToDevice, st));
  }
  std::vector<apy_gemm_desc> G;
  sigma_gemms(O, V, nb, singles, I, F, hoo, t, ring_f, w, G, g3);
  const int s = apy_zgemm_group(G.data(), (int)G.size(), w.gemm, w.gemm_bytes, st, ev0, ev1);
  if (s != APY_OK) return s;
  return APY_OK;
}

Epi2Args epi_args(int64_t O, int64_t V, int nb, int k, int singles, const apy_so_ints* I, const SigmaWS& w,
                  const double2* F, const double2* t, int fov) {
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V;
  Epi2Args e{};
  e.O = O; e.V = V; e.Po = Po; e.Pv = Pv; e.n = O + V;
  e.ntile = (int)((V + ET - 1) / ET);
  e.drv = (const double2*)I->vvoo_t;
  e.Rp = w.rp + k * Po * Pv;
  e.X = w.X + k * OV * OV;
  e.QT = singles ? w.QT + k * O * Pv : nullptr;
  e.qj = (int64_t)nb * O * Pv;
  e.ovT = singles ? w.ovT : nullptr;
  e.t1 = t;
  e.F = F;
  e.fov = (singles && fov) ? 1 : 0;
  e.Tp = w.tp + k * Po * Pv;
  return e;
}

}  // namespace

extern "C" {

int apy_so_ints_sizes(int64_t O, int64_t V, int64_t sizes_out[9]) {
  if (O < 0 || V < 0 || !sizes_out) return APY_E_ARG;
  for (int k = 0; k < K_COUNT; ++k) sizes_out[k] = kind_size(k, O, V);
  return APY_OK;
}

int apy_so_ints_from_full(int64_t n, const void* A, const apy_so_ints* ints, void* stream) {
  if (!A || !ints || ints->O + ints->V != n) return APY_E_ARG;
  SrcFull src{(const double2*)A, n};
  return build_all(src, ints, 0, 0.0, (hipStream_t)stream);
}

int apy_so_ints_from_mo(int64_t m, const void* eri_mo, const apy_so_ints* ints, void* stream) {
  if (!eri_mo || !ints || ints->O + ints->V != 2 * m) return APY_E_ARG;
  const double2* E = (const double2*)eri_mo;
  const int64_t O = ints->O, V = ints->V;
  hipStream_t st = (hipStream_t)stream;
  if (O < 0 || V < 0) return APY_E_ARG;
  unsigned done = 0;
  const int past = stored_past(ints);
  int s = launch_pair_rows<K_VVVV_P>(E, m, O, V, past, ints->vvvv_p, st, done);
  if (s == APY_OK) s = launch_pair_rows<K_VVVO_P>(E, m, O, V, past, ints->vvvo_p, st, done);
  if (s == APY_OK) s = launch_pair_rows<K_VOVV>(E, m, O, V, past, ints->vovv_p, st, done);
  if (s == APY_OK) s = launch_pair_rows<K_RING>(E, m, O, V, past, ints->ring, st, done);
  if (s != APY_OK) return s;
  SrcMO src{E, m};
  return build_all(src, ints, 0, 0.0, st, done);
}

int apy_synth_so_ints(uint64_t seed, uint64_t tag, double sd, int accumulate, double scale, int real_only,
                      const apy_so_ints* ints, void* stream) {
  if (!ints) return APY_E_ARG;
  SrcSynth src{seed, tag, ints->O + ints->V, sd, real_only};
  return build_all(src, ints, accumulate, scale, (hipStream_t)stream);
}

int apy_so_fock_from_mo(int64_t m, const void* f_mo, void* f_so, void* stream) {
  return apy_so_fock_from_mo_batch(m, 1, f_mo, f_so, stream);
}

int apy_so_fock_from_mo_batch(int64_t m, int64_t nb, const void* f_mo, void* f_so, void* stream) {
  if (m <= 0 || nb <= 0 || !f_mo || !f_so) return APY_E_ARG;
  so_fock_kernel<<<apy_grid1d(4 * m * m * nb), 256, 0, (hipStream_t)stream>>>(m, nb, (const double2*)f_mo,
                                                                               (double2*)f_so);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

int apy_cisd_so_pair_operator(int64_t O, int64_t V, const void* fock, const void* oooo_p, void* hoo, void* stream) {
  if (O < 0 || V < 0 || !fock || !hoo) return APY_E_ARG;
  const int64_t Po = npair(O);
  if (Po == 0) return APY_OK;
  pair_oo_kernel<<<apy_grid1d(Po * Po), 256, 0, (hipStream_t)stream>>>(
      (const double2*)oooo_p, (const double2*)fock, O + V, O, (double2*)hoo);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

int apy_cisd_so_ring_fock(int64_t O, int64_t V, const void* fock, const void* ring, void* ring_f, void* stream) {
  if (O < 1 || V < 1 || !fock || !ring || !ring_f || ring == ring_f) return APY_E_ARG;
  const int64_t OV = O * V;
  ring_fock_kernel<<<apy_grid1d(OV * OV, 1 << 20), 256, 0, (hipStream_t)stream>>>(
      O, V, (const double2*)fock, (const double2*)ring, (double2*)ring_f);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

size_t apy_cisd_so_workspace(int64_t O, int64_t V, int singles) {
  if (O < 0 || V < 0) return 0;
  // a dense input, without and with ring_f (any non-null address here): covers every call of this (O, V)
  const int sg = singles ? 1 : 0;
  return std::max(carve(O, V, 1, sg, 1, nullptr, nullptr, 0, 1).total,
                  carve(O, V, 1, sg, 1, (const void*)256, nullptr, 0, 1).total);
}

}  // extern "C"

// The step on a caller's workspace; exact = 1 sizes the GEMM region for the
// plans that run now (see carve).  Shared by the entry points below and by
// other translation units (common.h).
int apy_cisd_so_step_ws(const apy_cisd_so_args* A, void* workspace, size_t ws_bytes, void* stream, int exact) {
  if (!A || !A->ints || !A->fock || !A->eps || !A->t || !A->out || !A->hoo) return APY_E_ARG;
  if (A->out == A->t || (A->mode == APY_MODE_RESIDUAL && (!A->t_new || A->t_new == A->out))) return APY_E_ARG;
  const int64_t O = A->O, V = A->V;
  if (O < 2 || V < 2 || A->ints->O != O || A->ints->V != V) return APY_E_ARG;
  const int singles = A->singles ? 1 : 0;
  if (A->mode != APY_MODE_RESIDUAL && A->mode != APY_MODE_SIGMA) return APY_E_ARG;
  if (A->mode == APY_MODE_RESIDUAL && !A->energy) return APY_E_ARG;
  const int packed = A->packed ? 1 : 0;
  if (packed && A->mode != APY_MODE_SIGMA) return APY_E_ARG;
  const apy_so_ints* I = A->ints;
  if (!I->vvvv_p || !I->ring || !I->vvoo_t) return APY_E_ARG;
  if (singles && (!I->ovoo_p || !I->vvvo_p || !I->vovv_p || !I->ooov)) return APY_E_ARG;
  if (A->ring_f && (A->ring_f == I->ring || A->ring_f == A->out)) return APY_E_ARG;
  hipStream_t st = (hipStream_t)stream;
  SigmaWS w = carve(O, V, 1, singles, !packed, A->ring_f, workspace, exact);
  if (!workspace || ws_bytes < w.total) return APY_E_WORKSPACE;
  w.gemm_bytes = ws_bytes - (size_t)((char*)w.gemm - (char*)workspace);

  const int64_t OV = O * V;
  const double2* t = (const double2*)A->t;
  double2* tn = (double2*)A->t_new;
  double2* out = (double2*)A->out;
  const double2* F = (const double2*)A->fock;
  const double2* Fk[1] = {F};
  const void* Hk[1] = {A->hoo};
  const double2* Tk[1] = {t};
  int s = sigma_body(O, V, 1, singles, I, Fk, Hk, Tk, packed, A->ring_f, w, (hipEvent_t)A->ev_begin,
                     (hipEvent_t)A->ev_end, st, A->gauss3m ? 1 : 0);
  if (s != APY_OK) return s;

  const double c0r = A->mode == APY_MODE_RESIDUAL ? 1.0 : A->c0_re;
  const double c0i = A->mode == APY_MODE_RESIDUAL ? 0.0 : A->c0_im;
  const double2* c0p = A->mode == APY_MODE_SIGMA ? (const double2*)A->c0_dev : nullptr;
  Epi2Args e = epi_args(O, V, 1, 0, singles, I, w, F, t, A->fov_coupling);
  e.eps = A->eps;
  e.E = (const double2*)A->energy;
  e.c0r = c0r; e.c0i = c0i; e.c0p = c0p;
  e.out = out + OV;
  e.tn = tn ? tn + OV : nullptr;
  e.mode = A->mode;
  e.packed = packed;
  e.s1 = singles ? w.s1 : nullptr;
  e.out1 = out;
  e.tn1 = tn;
  return launch_epi(e, OV, st);
}

size_t apy_cisd_so_ws_exact(const apy_cisd_so_args* A) {
  if (!A || A->O < 2 || A->V < 2) return 0;
  return carve(A->O, A->V, 1, A->singles ? 1 : 0, A->packed ? 0 : 1, A->ring_f, nullptr, 1).total;
}

extern "C" {

int apy_cisd_so_step(const apy_cisd_so_args* A, void* workspace, size_t ws_bytes, void* stream) {
  return apy_cisd_so_step_ws(A, workspace, ws_bytes, stream, 0);
}

int apy_cisd_so_tune(const apy_cisd_so_args* A, void* workspace, size_t ws_bytes, int reps, void* stream) {
  if (!A || !A->ints || !A->fock || !A->t || !A->hoo) return APY_E_ARG;
  const int64_t O = A->O, V = A->V;
  if (O < 2 || V < 2 || A->ints->O != O || A->ints->V != V) return APY_E_ARG;
  const int singles = A->singles ? 1 : 0;
  const int packed = A->packed ? 1 : 0;
  SigmaWS w = carve(O, V, 1, singles, !packed, A->ring_f, workspace);
  if (!workspace || ws_bytes < w.total) return APY_E_WORKSPACE;
  if (packed) w.tp = (double2*)((const double2*)A->t + O * V);
  const double2* Fk[1] = {(const double2*)A->fock};
  const void* Hk[1] = {A->hoo};
  const double2* Tk[1] = {(const double2*)A->t};
  std::vector<apy_gemm_desc> G;
  sigma_gemms(O, V, 1, singles, A->ints, Fk, Hk, Tk, A->ring_f, w, G, A->gauss3m ? 1 : 0);
  for (const apy_gemm_desc& d : G) {
    if (!d.a || !d.b) continue;
    int s = apy_zgemm_tune_impl(&d, w.gemm, w.gemm_bytes, reps, (hipStream_t)stream, nullptr, nullptr, nullptr);
    if (s != APY_OK) return s;
  }
  return APY_OK;
}

static int energy_impl(int64_t O, int64_t V, int singles, int packed, const void* fock, const void* oovv,
                       const void* t, void* energy, void* workspace, size_t ws_bytes, void* stream) {
  if (O < 0 || V < 0 || !fock || !oovv || !t || !energy) return APY_E_ARG;
  if (!workspace || ws_bytes < ENERGY_BLOCKS * sizeof(double2)) return APY_E_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  return launch_energy(O, V, singles, packed, (const double2*)fock, (const double2*)oovv, (const double2*)t,
                       (double2*)workspace, (double2*)energy, st);
}

int apy_cisd_so_energy(int64_t O, int64_t V, int singles, const void* fock, const void* oovv, const void* t,
                       void* energy, void* workspace, size_t ws_bytes, void* stream) {
  return energy_impl(O, V, singles, 0, fock, oovv, t, energy, workspace, ws_bytes, stream);
}

int apy_cisd_so_energy_packed(int64_t O, int64_t V, int singles, const void* fock, const void* oovv,
                              const void* t, void* energy, void* workspace, size_t ws_bytes, void* stream) {
  if (O < 2 || V < 2) return APY_E_ARG;
  return energy_impl(O, V, singles, 1, fock, oovv, t, energy, workspace, ws_bytes, stream);
}

// ------------------------------------------------------------ batched sigma
// Sigma products of nb instances that share the integrals (the field-
// displaced copies of one system): the particle-particle ladder, the ring
// term, the vvvo.t1, t2.vovv and ring.t1 terms each run as ONE GEMM with the
// instances stacked along M, so the integral blocks are read once per batch;
// the Fock-dependent products and the epilogues run per instance.
size_t apy_cisd_so_sigma_batch_workspace(int64_t O, int64_t V, int nb, int singles) {
  if (O < 2 || V < 2 || nb < 1) return 0;
  return carve(O, V, nb, singles ? 1 : 0, 1, nullptr, nullptr).total;
}

int apy_cisd_so_sigma_batch(const apy_cisd_so_sigma_batch_args* A, void* workspace, size_t ws_bytes, void* stream) {
  if (!A || !A->ints || !A->fock || !A->hoo || !A->c0 || !A->t || !A->out) return APY_E_ARG;
  const int64_t O = A->O, V = A->V;
  const int nb = A->nb;
  if (O < 2 || V < 2 || nb < 1 || nb > 4096 || A->ints->O != O || A->ints->V != V) return APY_E_ARG;
  const int singles = A->singles ? 1 : 0;
  const apy_so_ints* I = A->ints;
  if (!I->vvvv_p || !I->ring || !I->vvoo_t) return APY_E_ARG;
  if (singles && (!I->ovoo_p || !I->vvvo_p || !I->vovv_p || !I->ooov)) return APY_E_ARG;
  for (int k = 0; k < nb; ++k)
    if (!A->fock[k] || !A->hoo[k] || !A->t[k] || !A->out[k] || A->out[k] == A->t[k]) return APY_E_ARG;
  SigmaWS w = carve(O, V, nb, singles, 1, nullptr, workspace);
  if (!workspace || ws_bytes < w.total) return APY_E_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const int64_t OV = O * V;
  std::vector<const double2*> F(nb), T(nb);
  std::vector<const void*> H(nb);
  for (int k = 0; k < nb; ++k) {
    F[k] = (const double2*)A->fock[k];
    H[k] = A->hoo[k];
    T[k] = (const double2*)A->t[k];
  }
  int s = sigma_body(O, V, nb, singles, I, F.data(), H.data(), T.data(), 0, nullptr, w, (hipEvent_t)A->ev_begin,
                     (hipEvent_t)A->ev_end, st, A->gauss3m ? 1 : 0);
  if (s != APY_OK) return s;
  for (int k = 0; k < nb; ++k) {
    double2* out = (double2*)A->out[k];
    Epi2Args e = epi_args(O, V, nb, k, singles, I, w, F[k], T[k], A->fov_coupling);
    e.c0r = A->c0[2 * k]; e.c0i = A->c0[2 * k + 1];
    e.out = out + OV;
    e.mode = APY_MODE_SIGMA;
    e.packed = 0;
    e.s1 = singles ? w.s1 + k * OV : nullptr;
    e.out1 = out;
    const int qs = launch_epi(e, OV, st);
    if (qs != APY_OK) return qs;
  }
  return APY_OK;
}

}  // extern "C"

// ------------------------------------------------------------ one-electron sigma
// The Fock-linear part L(F) of the Hermitian CISD sigma on a packed vector
// [c1 | c2 over (i<j, a<b) | c0]: the terms of ci_wfn.py:309-334 that carry
// F_SO (r_T1: F_vo c0, -F_oo^T c1, c1 F_vv^T, F_ov.c2; r_T2: the two F_vv and
// the two F_oo contractions) plus the Hermitian f_ov couplings (c0 row
// F_ov.c1, doubles P(ij)P(ab) f_bj c_ia).  For a one-electron perturbation
// dF of a Hamiltonian whose two-electron integrals stay fixed (the field-
// displaced copies of fin_diff.py:335-370), H(F0 + dF) = H(F0) + L(dF)
// exactly, so the sigma of every perturbed instance follows from one full
// sigma and this O^2 V^3 product.  The products are the step's own GEMMs
// (ring permutation, 1/2 T' F_vv^T into X, pair operator of F alone) and its
// epilogues with the two-electron pieces left out.
namespace {

struct FockWS {
  double2 *tr, *X, *rp, *s1, *part;
  void* gemm;
  size_t gemm_bytes;
  size_t total;
};

void fock_gemms(int64_t O, int64_t V, const double2* F, const void* hoo, const double2* t, const FockWS& w,
                std::vector<apy_gemm_desc>& G) {
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V, n = O + V;
  G.clear();
  apy_gemm_desc d;
  const double2* tp = t ? t + OV : nullptr;
  // X[(i,a,j)][b] = 1/2 sum_c T'[(i,a,j)][c] F[O+b][O+c]
  fill(d, O * V * O, V, V, APY_MK, w.tr, V, APY_NK, F ? F + O * n + O : nullptr, n, w.X, V, 0.5, 0.0);
  G.push_back(d);
  // R_p = Hoo(F) . T_p  (the F_oo terms over occupied pairs)
  fill(d, Po, Pv, Po, APY_MK, hoo, Po, APY_KN, tp, Pv, w.rp, Pv, 1.0, 0.0);
  G.push_back(d);
  // s1 = c1 F_vv^T - F_oo^T c1 + sum_jb T'[(ia),(jb)] F[j][O+b]
  fill(d, O, V, V, APY_MK, t, V, APY_NK, F ? F + O * n + O : nullptr, n, w.s1, V, 1.0, 0.0);
  G.push_back(d);
  fill(d, O, V, O, APY_KM, F, n, APY_KN, t, V, w.s1, V, -1.0, 1.0);
  G.push_back(d);
  fill(d, OV, 1, V, APY_MK, w.tr, OV, APY_KN, F ? F + O : nullptr, 1, w.s1, 1, 1.0, 1.0);
  d.batch = O; d.stride_a = V; d.stride_b = n; d.stride_c = 0; d.reduce_batch = 1;
  G.push_back(d);
}

FockWS carve_fock(int64_t O, int64_t V, void* base, int grouped = 0) {
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V;
  FockWS w{};
  size_t off = 0;
  char* b = base ? (char*)base : (char*)256;
  auto take = [&](size_t elems) -> double2* {
    double2* p = (double2*)(b + off);
    off += al256(elems * sizeof(double2));
    return p;
  };
  w.tr = take((size_t)OV * OV);
  w.X = take((size_t)OV * OV);
  w.rp = take((size_t)Po * Pv);
  w.s1 = take((size_t)OV);
  w.part = take((size_t)ENERGY_BLOCKS);
  std::vector<apy_gemm_desc> G;
  fock_gemms(O, V, nullptr, nullptr, nullptr, w, G);
  size_t g = 0;
  for (const apy_gemm_desc& d : G) g = std::max(g, apy_zgemm_ws_bytes(&d));
  if (grouped) g = std::max(g, apy_zgemm_group_ws_bytes(G.data(), (int)G.size()));
  w.gemm = (void*)(b + off);
  w.gemm_bytes = g;
  off += al256(g);
  w.total = off;
  return w;
}

}  // namespace

extern "C" {

size_t apy_cisd_so_fock_sigma_workspace(int64_t O, int64_t V) {
  if (O < 2 || V < 2) return 0;
  return carve_fock(O, V, nullptr, 1).total;
}

int apy_cisd_so_fock_sigma(const apy_cisd_so_fock_sigma_args* A, void* workspace, size_t ws_bytes, void* stream) {
  if (!A || !A->fock || !A->hoo || !A->t || !A->out) return APY_E_ARG;
  const int64_t O = A->O, V = A->V;
  const int nf = A->nf;
  if (O < 2 || V < 2 || nf < 1 || nf > 4096) return APY_E_ARG;
  for (int f = 0; f < nf; ++f)
    if (!A->fock[f] || !A->hoo[f] || !A->out[f] || A->out[f] == A->t) return APY_E_ARG;
  FockWS w = carve_fock(O, V, workspace);
  if (!workspace || ws_bytes < w.total) return APY_E_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const int64_t Po = npair(O), Pv = npair(V), OV = O * V, n = O + V, PP = Po * Pv;
  const double2* t = (const double2*)A->t;
  const double2* c0p = t + OV + PP;
  PrepArgs pa{};
  pa.O = O; pa.V = V; pa.tp_in = t + OV; pa.tr = w.tr;
  const int ps = launch_prep(pa, st);
  if (ps != APY_OK) return ps;
  std::vector<apy_gemm_desc> G;
  for (int f = 0; f < nf; ++f) {
    const double2* F = (const double2*)A->fock[f];
    double2* out = (double2*)A->out[f];
    fock_gemms(O, V, F, A->hoo[f], t, w, G);
    const int gs = apy_zgemm_group(G.data(), (int)G.size(), w.gemm,
                                   ws_bytes - (size_t)((char*)w.gemm - (char*)workspace), st);
    if (gs != APY_OK) return gs;
    Epi2Args e{};
    e.O = O; e.V = V; e.Po = Po; e.Pv = Pv; e.n = n;
    e.ntile = (int)((V + ET - 1) / ET);
    e.drv = nullptr;
    e.Rp = w.rp;
    e.X = w.X;
    e.QT = nullptr;
    e.qj = 0;
    e.ovT = nullptr;
    e.t1 = t;
    e.F = F;
    e.fov = 1;
    e.c0p = c0p;
    e.Tp = t + OV;
    e.out = out + OV;
    e.mode = APY_MODE_SIGMA;
    e.packed = 1;
    e.s1 = w.s1;
    e.out1 = out;
    const int qs = launch_epi(e, OV, st);
    if (qs != APY_OK) return qs;
    const int es = launch_energy(O, V, 1, 1, F, nullptr, t, w.part, out + OV + PP, st);
    if (es != APY_OK) return es;
  }
  return APY_OK;
}

}  // extern "C"
