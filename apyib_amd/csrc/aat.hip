// Finite-difference atomic axial tensors: determinants of displaced-orbital
// overlaps contracted with CI/MP2 amplitudes (aats.py:558-1055 spatial,
// aats.py:120-554 spin-orbital), without forming determinant tensors.
//
// For an overlap S between bra orbitals (rows) and ket orbitals (columns)
// with occupied block P = S[o,o] (no x no, d = det P), every determinant the
// reference builds by replacing up to two occupied rows (i -> a) and up to two
// occupied columns (k -> c) is d times a minor of
//     Gamma = [[ -P^-1, Y ], [ X, W ]],   X = S[v,o] P^-1,  Y = P^-1 S[o,v],
//                                         W = S[v,v] - S[v,o] P^-1 S[o,v],
// (Jacobi's complementary-minor theorem): rows = replaced columns k then the
// new rows a, columns = replaced rows i then the new columns c, sign (-1)^(r c).
// Expanding those minors turns each amplitude-determinant sum of the
// reference into contractions of the amplitudes with x = X^T, y = Y, P^-1
// and W: O(o^2 v^2 (o+v)) per overlap class instead of (ov)^4 determinants.
//
// Kernels:
//   gamma_kernel   one workgroup per overlap: Gauss-Jordan inverse of P with
//                  partial pivoting (d = product of pivots), then x, y, P^-1
//                  (active block), W into a record.
//   axpby_kernel   amplitude combinations conj?(ca A + cb B) (normalised
//                  finite differences of the displaced amplitudes).
//   contract_forms o x v contractions of the doubles with x / y.
//   hmat_g/h       H(M) = P^T M W^T for four o x v matrices.
//   sandwich       U[k,l] = W K2[k,l] W^T on the FP64 matrix cores.
//   pair_dots      the occupied transforms of U and the dots with the bra doubles.
//   scalars        one workgroup per job: the 20 scalars of APY_AAT_NTERMS.
#include "common.h"

#include <algorithm>

namespace {

constexpr int BLK = 256;

inline __host__ __device__ int64_t rnd16(int64_t n) { return (n + 15) / 16 * 16; }

struct GLayout {
  int64_t oa, nv, x, y, p, w, size;
};

inline __host__ __device__ GLayout glayout(int64_t no, int64_t nf, int64_t nv) {
  GLayout L;
  L.oa = no - nf;
  L.nv = nv;
  L.x = 16;                       // [0] = d, padded to 256 bytes
  L.y = L.x + L.oa * nv;
  L.p = L.y + L.oa * nv;
  L.w = L.p + L.oa * L.oa;
  L.size = rnd16(L.w + nv * nv);
  return L;
}

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// four FMAs (a sum of two rounded products would take six instructions)
__device__ inline void cfma(double2& acc, double2 a, double2 b) {
  acc.x = fma(-a.y, b.y, fma(a.x, b.x, acc.x));
  acc.y = fma(a.y, b.x, fma(a.x, b.y, acc.y));
}
__device__ inline double2 czero() { return make_double2(0.0, 0.0); }

// ------------------------------------------------------------------ gamma
// ws: batch x no x 2no (Gauss-Jordan [P | I]); yw: batch x no x nv (full Y).
__global__ __launch_bounds__(BLK) void gamma_kernel(int64_t n, int64_t no, int64_t nf, const double2* __restrict__ S,
                                                    int64_t stride_s, double2* __restrict__ gam, double2* ws,
                                                    double2* yw) {
  const int64_t b = blockIdx.x;
  const int64_t nv = n - no, w2 = 2 * no;
  const GLayout L = glayout(no, nf, nv);
  const double2* Sb = S + b * stride_s;
  double2* M = ws + b * no * w2;
  double2* Y = yw + b * no * nv;
  double2* R = gam + b * L.size;
  __shared__ double smax[BLK];
  __shared__ int sidx[BLK];
  __shared__ double2 fac[BLK];
  __shared__ double2 det;
  __shared__ int singular;
  for (int64_t t = threadIdx.x; t < no * w2; t += BLK) {
    const int64_t r = t / w2, c = t % w2;
    M[t] = c < no ? Sb[r * n + c] : make_double2(r == c - no ? 1.0 : 0.0, 0.0);
  }
  if (threadIdx.x == 0) {
    det = make_double2(1.0, 0.0);
    singular = 0;
  }
  __syncthreads();
  for (int64_t col = 0; col < no; ++col) {
    double best = -1.0;
    int bi = -1;
    for (int64_t r = col + threadIdx.x; r < no; r += BLK) {
      const double2 v = M[r * w2 + col];
      const double m = v.x * v.x + v.y * v.y;
      if (m > best) { best = m; bi = (int)r; }
    }
    smax[threadIdx.x] = best;
    sidx[threadIdx.x] = bi;
    __syncthreads();
    for (int s = BLK / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) {
        const double o = smax[threadIdx.x + s];
        const int oi = sidx[threadIdx.x + s];
        if (o > smax[threadIdx.x] || (o == smax[threadIdx.x] && oi >= 0 && (sidx[threadIdx.x] < 0 || oi < sidx[threadIdx.x]))) {
          smax[threadIdx.x] = o;
          sidx[threadIdx.x] = oi;
        }
      }
      __syncthreads();
    }
    const int piv = sidx[0];
    const double pm = smax[0];
    __syncthreads();
    if (!(pm > 0.0)) {                 // exactly singular occupied block: d = 0
      if (threadIdx.x == 0) singular = 1;
      __syncthreads();
      break;
    }
    if (piv != col) {
      for (int64_t c = threadIdx.x; c < w2; c += BLK) {
        const double2 t0 = M[col * w2 + c];
        M[col * w2 + c] = M[(int64_t)piv * w2 + c];
        M[(int64_t)piv * w2 + c] = t0;
      }
    }
    __syncthreads();
    const double2 p = M[col * w2 + col];
    const double inv_den = 1.0 / (p.x * p.x + p.y * p.y);
    const double2 pinv = make_double2(p.x * inv_den, -p.y * inv_den);
    __syncthreads();
    if (threadIdx.x == 0) {
      double2 d = cmul(det, p);
      if (piv != col) d = make_double2(-d.x, -d.y);
      det = d;
    }
    for (int64_t c = threadIdx.x; c < w2; c += BLK) M[col * w2 + c] = cmul(M[col * w2 + c], pinv);
    for (int64_t r = threadIdx.x; r < no; r += BLK) fac[r] = (r == col) ? czero() : M[r * w2 + col];
    __syncthreads();
    for (int64_t t = threadIdx.x; t < no * w2; t += BLK) {
      const int64_t r = t / w2, c = t % w2;
      if (r != col) M[t] = csub(M[t], cmul(fac[r], M[col * w2 + c]));
    }
    __syncthreads();
  }
  if (singular) {
    for (int64_t t = threadIdx.x; t < L.size; t += BLK) R[t] = czero();
    return;
  }
  // full Y = P^-1 S[o, v]
  for (int64_t t = threadIdx.x; t < no * nv; t += BLK) {
    const int64_t m = t / nv, c = t % nv;
    double2 acc = czero();
    for (int64_t k = 0; k < no; ++k) cfma(acc, M[m * w2 + no + k], Sb[k * n + no + c]);
    Y[t] = acc;
  }
  __syncthreads();
  if (threadIdx.x == 0) R[0] = det;
  const int64_t oa = L.oa;
  for (int64_t t = threadIdx.x; t < oa * nv; t += BLK) {
    const int64_t i = t / nv, a = t % nv;
    double2 acc = czero();                               // x[i][a] = (S[v,o] P^-1)[a][nf+i]
    for (int64_t m = 0; m < no; ++m) cfma(acc, Sb[(no + a) * n + m], M[m * w2 + no + nf + i]);
    R[L.x + t] = acc;
    R[L.y + t] = Y[(nf + i) * nv + a];
  }
  for (int64_t t = threadIdx.x; t < oa * oa; t += BLK) {
    const int64_t k = t / oa, i = t % oa;
    R[L.p + t] = M[(nf + k) * w2 + no + nf + i];
  }
  for (int64_t t = threadIdx.x; t < nv * nv; t += BLK) {
    const int64_t a = t / nv, c = t % nv;
    double2 acc = Sb[(no + a) * n + no + c];
    for (int64_t m = 0; m < no; ++m) acc = csub(acc, cmul(Sb[(no + a) * n + m], Y[m * nv + c]));
    R[L.w + t] = acc;
  }
}

// ------------------------------------------------------------------ axpby
__global__ __launch_bounds__(BLK) void axpby_kernel(const apy_aat_axpby_op* __restrict__ ops) {
  const apy_aat_axpby_op op = ops[blockIdx.y];
  const double2* A = (const double2*)op.a;
  const double2* B = (const double2*)op.b;
  double2* out = (double2*)op.out;
  for (int64_t e = blockIdx.x * (int64_t)BLK + threadIdx.x; e < op.n; e += (int64_t)gridDim.x * BLK) {
    double2 v = make_double2(op.ca * A[e].x, op.ca * A[e].y);
    if (B) { v.x += op.cb * B[e].x; v.y += op.cb * B[e].y; }
    if (op.conj) v.y = -v.y;
    out[e] = v;
  }
}

// ------------------------------------------------------------------ jobs
// Scratch of one job.  Jobs of a call share operands (the AAT elements reuse overlaps and amplitudes), so
// every intermediate is formed once, in the slot of the first job that needs it (its representative):
//   bra forms of (gamma, b2), ket forms and H matrices of (gamma, k1, k2), U of (gamma, k2), A(b2) of b2.
struct JLayout {
  int64_t ov, o2v2, small, part, per;
};
constexpr int PD_COLS = 16;       // (a,b) columns of a pair_dots block: one (e1, e2) partial each
inline __host__ __device__ JLayout jlayout(int64_t oa, int64_t nv) {
  JLayout J;
  J.ov = oa * nv;
  J.o2v2 = J.ov * J.ov;
  J.small = rnd16(16 * J.ov);     // bra forms [4], ket forms [4], G[4], H[4]
  J.part = rnd16(2 * ((nv * nv + PD_COLS - 1) / PD_COLS));   // (e1, e2) partials
  J.per = J.small + J.part + 2 * rnd16(J.o2v2);            // ... then A(b2) (U1 of the general path) and U (U2)
  return J;
}

// Representatives of a job and whether its doubles are exactly antisymmetric in both pairs (0: they are).
struct JobRep {
  int b2, k2, bra, ket;           // first job with the same b2 / k2 / (gamma, b2) / (gamma, k1, k2)
  int gen_b, gen_k;               // set on the representative by antisym_check
};

__device__ inline int64_t i4(int64_t oa, int64_t nv, int64_t i, int64_t j, int64_t a, int64_t b) {
  return ((i * oa + j) * nv + a) * nv + b;
}

// one wavefront a job, its lanes over the earlier jobs
__global__ __launch_bounds__(BLK) void job_reps(int64_t njobs, const apy_aat_job* __restrict__ jobs,
                                                JobRep* __restrict__ reps) {
  const int q = blockIdx.x * (BLK / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (q >= njobs) return;
  const apy_aat_job me = jobs[q];
  int r[4] = {q, q, q, q};
  for (int t = lane; t < q; t += 64) {
    const apy_aat_job o = jobs[t];
    const bool same[4] = {o.b2 == me.b2, o.k2 == me.k2, o.gamma == me.gamma && o.b2 == me.b2,
                          o.gamma == me.gamma && o.k2 == me.k2 && o.k1 == me.k1};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (same[k]) r[k] = min(r[k], t);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k)
    for (int off = 32; off > 0; off >>= 1) r[k] = min(r[k], __shfl_xor(r[k], off, 64));
  if (lane == 0) reps[q] = JobRep{r[0], r[1], r[2], r[3], 0, 0};
}

// Marks the doubles (z = 0: b2, 1: k2) that are not exactly antisymmetric in (i,j) and in (a,b).  The
// spin-orbital solvers' amplitudes are; the spatial ones are not.  Antisymmetric doubles need one
// contraction instead of four, half of the occupied pairs of U and no A(b2).
__global__ __launch_bounds__(BLK) void antisym_check(int64_t oa, int64_t nv, const apy_aat_job* __restrict__ jobs,
                                                     JobRep* reps) {
  const int q = blockIdx.y, ket = blockIdx.z;
  if ((ket ? reps[q].k2 : reps[q].b2) != q) return;
  const double2* T = (const double2*)(ket ? jobs[q].k2 : jobs[q].b2);
  if (!T) return;
  int* flag = ket ? &reps[q].gen_k : &reps[q].gen_b;
  for (int64_t ij = blockIdx.x; ij < oa * oa; ij += gridDim.x) {
    const int64_t i = ij / oa, j = ij % oa;
    if (i > j) continue;
    if (*(volatile int*)flag) return;
    const double2 *A = T + ij * nv * nv, *B = T + (j * oa + i) * nv * nv;
    const int n = (int)nv;
    for (int e = threadIdx.x; e < n * n; e += BLK) {
      const int a = e / n, b = e % n;
      if (a > b) continue;
      const double2 x = A[e], y = B[e], z = A[b * n + a], w = B[b * n + a];
      const bool ok = x.x == -y.x && x.y == -y.y && x.x == -z.x && x.y == -z.y && x.x == w.x && x.y == w.y;
      if (!ok) *(volatile int*)flag = 1;
    }
  }
}

// A(b2) = (T - T^ab - T^ij + T^ijab) / 4 of the doubles that are not antisymmetric themselves
__global__ __launch_bounds__(BLK) void antisymmetrize(int64_t oa, int64_t nv, const apy_aat_job* __restrict__ jobs,
                                                      const JobRep* __restrict__ reps, double2* __restrict__ wsj) {
  const int q = blockIdx.y;
  if (reps[q].b2 != q || !reps[q].gen_b || !jobs[q].b2) return;
  const JLayout J = jlayout(oa, nv);
  const double2* T = (const double2*)jobs[q].b2;
  double2* out = wsj + q * J.per + J.small + J.part;
  const int n = (int)nv;
  for (int64_t ij = blockIdx.x; ij < oa * oa; ij += gridDim.x) {
    const double2 *A = T + ij * nv * nv, *B = T + ((ij % oa) * oa + ij / oa) * nv * nv;
    double2* o = out + ij * nv * nv;
    for (int e = threadIdx.x; e < n * n; e += BLK) {
      const int at = (e % n) * n + e / n;
      const double2 v = csub(csub(A[e], A[at]), csub(B[e], B[at]));
      o[e] = make_double2(0.25 * v.x, 0.25 * v.y);
    }
  }
}

// The four contractions of a doubles tensor with an o x v vector (z = 0: b2 with x, 1: k2 with y):
//   form 0: u[p,q] = sum_rs T[p,r,q,s] v[r,s]   1: T[p,r,s,q]   2: T[r,p,q,s]   3: T[r,p,s,q]
// beta = u0, beta' = u3, beta^ = (u0 - u1 - u2 + u3)/4 of the bra; kA = u0, kB = u3, k^ = -(u0 - u1 - u2 + u3)/4
// of the ket.  Antisymmetric doubles: u1 = u2 = -u0, u3 = u0, one pass over the tensor.
// Bound by the reads of the tensors (L2 and HBM): a block takes one (form, p, 32 values of q) and reads each
// row of T along its contiguous index, forms 0 and 2 reducing along it, 1 and 3 holding it as q.  O=18 V=50,
// 324 jobs: 21.9 ms with one thread an output element and job, 0.65 ms.
__global__ __launch_bounds__(BLK) void contract_forms(int64_t oa, int64_t nv, const double2* __restrict__ gam,
                                                      int64_t rec, const apy_aat_job* __restrict__ jobs,
                                                      const JobRep* __restrict__ reps, double2* __restrict__ wsj) {
  const int q = blockIdx.y, ket = blockIdx.z;
  const JobRep rp = reps[q];
  if ((ket ? rp.ket : rp.bra) != q) return;
  const apy_aat_job jb = jobs[q];
  const double2* T = (const double2*)(ket ? jb.k2 : jb.b2);
  const bool anti = T && !(ket ? reps[rp.k2].gen_k : reps[rp.b2].gen_b);
  const int64_t nq = (nv + 31) / 32;
  int64_t r0 = blockIdx.x;
  const int64_t q0 = (r0 % nq) * 32; r0 /= nq;
  const int64_t p = r0 % oa;
  const int form = (int)(r0 / oa);
  if (anti && form) return;
  const JLayout J = jlayout(oa, nv);
  const GLayout L = glayout(oa, 0, nv);
  const double2* vec = gam + jb.gamma * rec + (ket ? L.y : L.x);
  double2* out = wsj + q * J.per + (4 * ket + form) * J.ov + p * nv;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  __shared__ double2 sh[8][33];
  if (!T) {
    if (ty == 0 && q0 + tx < nv) out[q0 + tx] = czero();
    return;
  }
  auto put = [&](int64_t qq, double2 v) {
    out[qq] = v;
    if (anti) {
      const double2 m = make_double2(-v.x, -v.y);
      out[qq + J.ov] = m;
      out[qq + 2 * J.ov] = m;
      out[qq + 3 * J.ov] = v;
    }
  };
  const int64_t vv = nv * nv, step = form < 2 ? vv : oa * vv;
  const double2* base = T + (form < 2 ? p * oa : p) * vv;   // tile r at base + r * step
  if ((form & 1) == 0) {
    double2 acc[4] = {czero(), czero(), czero(), czero()};
    for (int64_t r = 0; r < oa; ++r)
      for (int64_t s = tx; s < nv; s += 32) {
        const double2 x = vec[r * nv + s];
        const double2* t = base + r * step + s;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int64_t row = q0 + ty + 8 * m;
          if (row < nv) cfma(acc[m], t[row * nv], x);
        }
      }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      for (int off = 16; off > 0; off >>= 1) {
        acc[m].x += __shfl_xor(acc[m].x, off, 64);
        acc[m].y += __shfl_xor(acc[m].y, off, 64);
      }
      const int64_t row = q0 + ty + 8 * m;
      if (tx == 0 && row < nv) put(row, acc[m]);
    }
  } else {
    double2 acc = czero();
    const int64_t col = q0 + tx;
    if (col < nv)
      for (int64_t r = 0; r < oa; ++r) {
        const double2* t = base + r * step + col;
        for (int64_t s = ty; s < nv; s += 8) cfma(acc, t[s * nv], vec[r * nv + s]);
      }
    sh[ty][tx] = acc;
    __syncthreads();
    if (ty == 0 && col < nv) {
      for (int k = 1; k < 8; ++k) acc = cadd(acc, sh[k][tx]);
      put(col, acc);
    }
  }
}

// element e of beta^ (sign +1) or k^ (sign -1) from the forms at u
__device__ inline double2 hat(const double2* u, int64_t ov, int64_t e, double sign) {
  const double2 v = cadd(csub(csub(u[e], u[ov + e]), u[2 * ov + e]), u[3 * ov + e]);
  return make_double2(0.25 * sign * v.x, 0.25 * sign * v.y);
}

// G_w[k,b] = sum_d M_w[k,d] W[b,d]  for M = (K1, k^, kA, kB)
__global__ __launch_bounds__(BLK) void hmat_g(int64_t oa, int64_t nv, const double2* __restrict__ gam, int64_t rec,
                                              const apy_aat_job* __restrict__ jobs, const JobRep* __restrict__ reps,
                                              double2* __restrict__ wsj) {
  if (reps[blockIdx.y].ket != (int)blockIdx.y) return;
  const JLayout J = jlayout(oa, nv);
  const int64_t t = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (t >= 4 * J.ov) return;
  const apy_aat_job jb = jobs[blockIdx.y];
  const int w = (int)(t / J.ov);
  const int64_t e = t % J.ov, k = e / nv, bb = e % nv;
  const GLayout L = glayout(oa, 0, nv);
  const double2* W = gam + jb.gamma * rec + L.w;
  double2* base = wsj + blockIdx.y * J.per;
  const double2* u = base + 4 * J.ov;
  double2 acc = czero();
  if (w == 1) {
    for (int64_t d = 0; d < nv; ++d) cfma(acc, hat(u, J.ov, k * nv + d, -1.0), W[bb * nv + d]);
  } else {
    const double2* M = w == 0 ? (const double2*)jb.k1 : u + (w == 2 ? 0 : 3) * J.ov;
    if (M)
      for (int64_t d = 0; d < nv; ++d) cfma(acc, M[k * nv + d], W[bb * nv + d]);
  }
  base[(8 + w) * J.ov + e] = acc;
}

// H_w[i,b] = sum_k P[k,i] G_w[k,b]
__global__ __launch_bounds__(BLK) void hmat_h(int64_t oa, int64_t nv, const double2* __restrict__ gam, int64_t rec,
                                              const apy_aat_job* __restrict__ jobs, const JobRep* __restrict__ reps,
                                              double2* __restrict__ wsj) {
  if (reps[blockIdx.y].ket != (int)blockIdx.y) return;
  const JLayout J = jlayout(oa, nv);
  const int64_t t = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (t >= 4 * J.ov) return;
  const apy_aat_job jb = jobs[blockIdx.y];
  const int w = (int)(t / J.ov);
  const int64_t e = t % J.ov, i = e / nv, bb = e % nv;
  const GLayout L = glayout(oa, 0, nv);
  const double2* P = gam + jb.gamma * rec + L.p;
  double2* base = wsj + blockIdx.y * J.per;
  const double2* G = base + (8 + w) * J.ov;
  double2 acc = czero();
  for (int64_t k = 0; k < oa; ++k) cfma(acc, P[k * oa + i], G[k * nv + bb]);
  base[(12 + w) * J.ov + e] = acc;
}

// ------------------------------------------------------------------ e1, e2
// e2 = sum B2 T and e1 = sum A(B2) T, T = (P^T (x) P^T (x) W (x) W) K2, in two kernels.

// U[k,l] = W K2[k,l] W^T for every occupied pair on the FP64 matrix cores; when K2 is antisymmetric so is U, and
// only k < l, a < b is formed, U[k,l] holding the packed row (a < b).  A wave takes 16 columns b of one pair: K2[k,l] W^T first, its 16 x 16 result blocks staying in
// registers, where their layout (row lane/16 + 4r, column lane%16) is the B operand of step r of the second
// product, so the intermediate is never stored.  K2 is read along its rows (64 B a row and step, from L2:
// the pairs' tensors are shared by many overlaps); W comes from LDS while it fits, else from L2.
// Bound by the matrix cores; nv is padded to 16 in the rows and columns and to 4 in the sums.  O=18 V=50, 324
// jobs (225 kets): 1.8 ms, against 24 ms for two scalar quarter transforms a job.
// RB = ceil(nv / 16).
template <int RB, bool WL>
__global__ __launch_bounds__(BLK) void sandwich(int64_t oa, int64_t nv, const double2* __restrict__ gam, int64_t rec,
                                                const apy_aat_job* __restrict__ jobs, const JobRep* __restrict__ reps,
                                                double2* __restrict__ wsj) {
  extern __shared__ double2 Ws[];
  const int q = blockIdx.y;
  const JobRep rp = reps[q];
  const apy_aat_job jb = jobs[q];
  if (rp.ket != q || !jb.k2) return;
  const bool anti = !reps[rp.k2].gen_k;
  const JLayout J = jlayout(oa, nv);
  const GLayout L = glayout(oa, 0, nv);
  const double2* W = gam + jb.gamma * rec + L.w;
  const double2* K2 = (const double2*)jb.k2;
  double2* U = wsj + q * J.per + J.small + J.part + rnd16(J.o2v2);
  const int ldw = WL ? (int)nv + 1 : (int)nv;
  const double2* Wr = W;
  if (WL) {
    for (int t = threadIdx.x; t < (int)(nv * nv); t += BLK) Ws[(t / (int)nv) * ldw + t % (int)nv] = W[t];
    __syncthreads();
    Wr = Ws;
  }
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int n = (int)nv;
  const int64_t units = oa * oa * RB, vv = nv * nv;
  const int64_t nwave = (int64_t)gridDim.x * (BLK / 64);
  for (int64_t u = blockIdx.x * (int64_t)(BLK / 64) + (threadIdx.x >> 6); u < units; u += nwave) {
    const int64_t kl = u / RB;
    const int b0 = (int)(u % RB) * 16;
    if (anti && kl / oa >= kl % oa) continue;
    const double2* K = K2 + kl * vv;
    auto lda = [&](int rb, int d0) {
      const int c = rb * 16 + lr, d = d0 + lk;
      const double2 x = K[(int64_t)min(c, n - 1) * n + min(d, n - 1)];
      return (c < n && d < n) ? x : czero();
    };
    auto ldwt = [&](int row, int k) {
      const double2 x = Wr[min(row, n - 1) * ldw + min(k, n - 1)];
      return (row < n && k < n) ? x : czero();
    };
    v4d xr[RB], xi[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) { xr[r] = (v4d){0, 0, 0, 0}; xi[r] = (v4d){0, 0, 0, 0}; }
    double2 an[RB], bn;
#pragma unroll
    for (int r = 0; r < RB; ++r) an[r] = lda(r, 0);
    bn = ldwt(b0 + lr, lk);
    for (int d0 = 0; d0 < n; d0 += 4) {
      double2 av[RB];
      const double2 bv = bn;
#pragma unroll
      for (int r = 0; r < RB; ++r) av[r] = an[r];
#pragma unroll
      for (int r = 0; r < RB; ++r) an[r] = lda(r, d0 + 4);
      bn = ldwt(b0 + lr, d0 + 4 + lk);
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        xr[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[r].x, bv.x, xr[r], 0, 0, 0);
        xi[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[r].x, bv.y, xi[r], 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        xr[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(-av[r].y, bv.y, xr[r], 0, 0, 0);
        xi[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[r].y, bv.x, xi[r], 0, 0, 0);
      }
    }
    for (int a0 = 0; a0 < (anti ? min(n, b0 + 16) : n); a0 += 16) {
      v4d rr = (v4d){0, 0, 0, 0}, ri = rr, ir = rr, ii = rr;
#pragma unroll
      for (int s = 0; s < 4 * RB; ++s) {
        if (4 * s < n) {
          const double2 w = ldwt(a0 + lr, 4 * s + lk);
          rr = __builtin_amdgcn_mfma_f64_16x16x4f64(w.x, xr[s >> 2][s & 3], rr, 0, 0, 0);
          ii = __builtin_amdgcn_mfma_f64_16x16x4f64(w.y, xi[s >> 2][s & 3], ii, 0, 0, 0);
          ri = __builtin_amdgcn_mfma_f64_16x16x4f64(w.x, xi[s >> 2][s & 3], ri, 0, 0, 0);
          ir = __builtin_amdgcn_mfma_f64_16x16x4f64(w.y, xr[s >> 2][s & 3], ir, 0, 0, 0);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = a0 + lk + 4 * r, b = b0 + lr;
        const int64_t at = anti ? a * (2 * n - a - 1) / 2 + b - a - 1 : a * n + b;
        if (b < n && (anti ? a < b : a < n)) U[kl * vv + at] = make_double2(rr[r] - ii[r], ri[r] + ir[r]);
      }
    }
  }
}

// The occupied transforms of U and the dots with the bra doubles, over 16 columns (a,b) a block:
//   X[k,j] = sum_l P[l,j] U[k,l],  T[i,j] = sum_k P[k,i] X[k,j],  e2 += B2[i,j] T[i,j],  e1 += A(B2)[i,j] T[i,j]
// Antisymmetric K2: T is antisymmetric too, so only a < b and i < j are formed and e1 = e2 = 4 sum A(B2) T.
// Both products run on the FP64 matrix cores with P^T as the A operand of either, held in registers for the
// whole block; X of 16 values of j lives in LDS, T only in the accumulators.  (The same sums on the vector units
// with P from scalar loads ran at 7 TFLOP/s: too few waves beside the LDS to cover the scalar loads.)  oa is
// padded to 16 in the rows and to 4 in the sums.  One launch covers every ket; its jobs' dots are taken PD_JL at
// a time.  Blocks of 4 waves: two fit beside each other in LDS and hide each other's barriers (2.5 ms with 8
// waves a block, 1.6 ms with 4 at O=18 V=50, 324 jobs; two quarter transforms and the dots took 28 ms).
// KS = ceil(oa / 4).
constexpr int PD_NT = 256, PD_JL = 4;
template <int KS>
__global__ __launch_bounds__(PD_NT) void pair_dots(int64_t oa64, int64_t nv, const double2* __restrict__ gam,
                                                   int64_t rec, int64_t njobs, const apy_aat_job* __restrict__ jobs,
                                                   const JobRep* __restrict__ reps, double2* __restrict__ wsj) {
  extern __shared__ double2 Xs[];                      // [k][16 j][16 columns]
  __shared__ int list[PD_NT];
  __shared__ int count;
  __shared__ double2 red[2 * PD_JL][PD_NT / 64];
  const int q = blockIdx.y;
  const JobRep rp = reps[q];
  const apy_aat_job jb = jobs[q];
  if (rp.ket != q || !jb.k2) return;
  const bool anti = !reps[rp.k2].gen_k;
  const JLayout J = jlayout(oa64, nv);
  const GLayout L = glayout(oa64, 0, nv);
  const double2* P = gam + jb.gamma * rec + L.p;
  const double2* U = wsj + q * J.per + J.small + J.part + rnd16(J.o2v2);
  constexpr int NW = PD_NT / 64, RBO = (KS + 3) / 4;
  const int oa = (int)oa64, n = (int)nv;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int64_t vv = nv * nv, ncol = anti ? nv * (nv - 1) / 2 : vv, col = blockIdx.x * (int64_t)PD_COLS + lr;
  if (blockIdx.x * (int64_t)PD_COLS >= ncol) return;   // antisymmetric: fewer columns (scalars reads as many partials)
  const bool in = col < ncol;
  const int64_t uc = in ? col : 0;
  int64_t at = uc;                                     // this lane's column in a full [a][b] tile
  if (anti) {
    const double m = 2.0 * n - 1.0;
    int a = (int)((m - sqrt(m * m - 8.0 * (double)uc)) * 0.5);
    a = max(0, min(a, n - 2));
    while (a > 0 && (int64_t)a * (2 * n - a - 1) / 2 > uc) --a;
    while (a < n - 2 && (int64_t)(a + 1) * (2 * n - a - 2) / 2 <= uc) ++a;
    at = (int64_t)a * n + (uc - (int64_t)a * (2 * n - a - 1) / 2 + a + 1);
  }
  // A operand of both products: row 16 rb + lr, sum index 4 s + lk of P^T
  double2 pt[RBO][KS];
#pragma unroll
  for (int rb = 0; rb < RBO; ++rb)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int row = 16 * rb + lr, k = 4 * s + lk;
      const double2 x = P[min(k, oa - 1) * oa + min(row, oa - 1)];
      pt[rb][s] = row < oa && k < oa ? x : czero();
    }

  for (int64_t w0 = 0; w0 < njobs; w0 += PD_NT) {
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    // this ket's jobs among the next PD_NT, in order: the waves append in turn
    const int64_t cand = w0 + threadIdx.x;
    const bool mine = cand < njobs && reps[cand].ket == q && jobs[cand].b2;
    for (int w = 0; w < NW; ++w) {
      if (wave == w) {
        const unsigned long long bal = __ballot(mine);
        const int base = count;
        if (mine) list[base + __popcll(bal & ((1ull << lane) - 1ull))] = (int)cand;
        if (lane == 0) count = base + __popcll(bal);
      }
      __syncthreads();
    }
    const int nl = count;
    for (int c0 = 0; c0 < nl; c0 += PD_JL) {
      double2 e1[PD_JL], e2[PD_JL];
      const double2 *B[PD_JL], *A[PD_JL];
#pragma unroll
      for (int t = 0; t < PD_JL; ++t) {
        e1[t] = czero();
        e2[t] = czero();
        const int job = list[min(c0 + t, nl - 1)], rb = reps[job].b2;
        B[t] = (const double2*)jobs[job].b2;
        A[t] = reps[rb].gen_b ? wsj + rb * J.per + J.small + J.part : B[t];
      }
#pragma unroll
      for (int jbk = 0; jbk < RBO; ++jbk) {
        for (int k = wave; k < oa; k += NW) {
          double2 u[KS];
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const int l = min(4 * s + lk, oa - 1);
            u[s] = U[(anti && l < k ? l * oa + k : k * oa + l) * vv + uc];   // antisymmetric: k < l is stored
          }
          v4d rr = (v4d){0, 0, 0, 0}, ri = rr, ir = rr, ii = rr;
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const int l = 4 * s + lk;
            const bool zero = l >= oa || (anti && l == k), neg = anti && l < k;
            const double ux = zero ? 0.0 : neg ? -u[s].x : u[s].x, uy = zero ? 0.0 : neg ? -u[s].y : u[s].y;
            rr = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[jbk][s].x, ux, rr, 0, 0, 0);
            ii = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[jbk][s].y, uy, ii, 0, 0, 0);
            ri = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[jbk][s].x, uy, ri, 0, 0, 0);
            ir = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[jbk][s].y, ux, ir, 0, 0, 0);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r)
            Xs[(k * 16 + lk + 4 * r) * 16 + lr] = make_double2(rr[r] - ii[r], ri[r] + ir[r]);
        }
        __syncthreads();
        for (int jl = wave; jl < min(16, oa - 16 * jbk); jl += NW) {
          const int j = 16 * jbk + jl, imax = anti ? j : oa;
          double2 x[KS];
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const int k = 4 * s + lk;
            const double2 v = Xs[(min(k, oa - 1) * 16 + jl) * 16 + lr];
            x[s] = k < oa ? v : czero();
          }
#pragma unroll
          for (int ib = 0; ib < RBO; ++ib) {
            if (16 * ib >= imax) continue;
            v4d rr = (v4d){0, 0, 0, 0}, ri = rr, ir = rr, ii = rr;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                rr = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[ib][s].x, x[s].x, rr, 0, 0, 0);
              ii = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[ib][s].y, x[s].y, ii, 0, 0, 0);
              ri = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[ib][s].x, x[s].y, ri, 0, 0, 0);
              ir = __builtin_amdgcn_mfma_f64_16x16x4f64(pt[ib][s].y, x[s].x, ir, 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < PD_JL; ++t) {
              if (c0 + t >= nl) continue;
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int i = 16 * ib + lk + 4 * r;
                const bool use = in && i < imax;
                const int64_t e = (int64_t)(min(i, oa - 1) * oa + j) * vv + at;
                const double2 tv = make_double2(rr[r] - ii[r], ri[r] + ir[r]), av = A[t][e];
                if (use) cfma(e1[t], av, tv);
                if (!anti) {
                  const double2 bv = B[t][e];
                  if (use) cfma(e2[t], bv, tv);
                }
              }
            }
          }
        }
        __syncthreads();
      }
#pragma unroll
      for (int t = 0; t < PD_JL; ++t) {
        for (int off = 32; off > 0; off >>= 1) {
          e1[t].x += __shfl_xor(e1[t].x, off, 64);
          e1[t].y += __shfl_xor(e1[t].y, off, 64);
          e2[t].x += __shfl_xor(e2[t].x, off, 64);
          e2[t].y += __shfl_xor(e2[t].y, off, 64);
        }
        if (lane == 0) { red[2 * t][wave] = e1[t]; red[2 * t + 1][wave] = e2[t]; }
      }
      __syncthreads();
      if (threadIdx.x < 2 * PD_JL && c0 + (int)threadIdx.x / 2 < nl) {
        const int src = anti ? threadIdx.x & ~1 : threadIdx.x;            // antisymmetric: e2 = e1
        double2 v = red[src][0];
        for (int w = 1; w < NW; ++w) v = cadd(v, red[src][w]);
        if (anti) v = make_double2(4.0 * v.x, 4.0 * v.y);
        wsj[list[c0 + threadIdx.x / 2] * J.per + J.small + 2 * blockIdx.x + (threadIdx.x & 1)] = v;
      }
      __syncthreads();
    }
    __syncthreads();                                   // the list is read no more
  }
}

// General quarter transforms of K2 (nv or oa beyond the kernels above), stage 0..3:
//   0: U1[k,l,c,b] = sum_d K2[k,l,c,d] W[b,d]     1: U2[k,l,a,b] = sum_c W[a,c] U1[k,l,c,b]
//   2: U1[k,j,a,b] = sum_l P[l,j] U2[k,l,a,b]     3: U2[i,j,a,b] = sum_k P[k,i] U1[k,j,a,b]
__global__ __launch_bounds__(BLK) void quarter(int stage, int64_t oa, int64_t nv, const double2* __restrict__ gam,
                                               int64_t rec, const apy_aat_job* __restrict__ jobs,
                                               const JobRep* __restrict__ reps, double2* __restrict__ wsj) {
  const JLayout J = jlayout(oa, nv);
  const apy_aat_job jb = jobs[blockIdx.y];
  if (reps[blockIdx.y].ket != (int)blockIdx.y || !jb.k2) return;
  const GLayout L = glayout(oa, 0, nv);
  const double2* W = gam + jb.gamma * rec + L.w;
  const double2* P = gam + jb.gamma * rec + L.p;
  double2* U1 = wsj + blockIdx.y * J.per + J.small + J.part;
  double2* U2 = U1 + rnd16(J.o2v2);
  const double2* K2 = (const double2*)jb.k2;
  for (int64_t e = blockIdx.x * (int64_t)BLK + threadIdx.x; e < J.o2v2; e += (int64_t)gridDim.x * BLK) {
    int64_t r0 = e;
    const int64_t b = r0 % nv; r0 /= nv;
    const int64_t a = r0 % nv; r0 /= nv;
    const int64_t j = r0 % oa;
    const int64_t i = r0 / oa;
    double2 acc = czero();
    switch (stage) {
      case 0:  // (i,j,a,b) = (k,l,c,b)
        for (int64_t d = 0; d < nv; ++d) cfma(acc, K2[i4(oa, nv, i, j, a, d)], W[b * nv + d]);
        U1[e] = acc;
        break;
      case 1:  // (k,l,a,b)
        for (int64_t c = 0; c < nv; ++c) cfma(acc, W[a * nv + c], U1[i4(oa, nv, i, j, c, b)]);
        U2[e] = acc;
        break;
      case 2:  // (k,j,a,b)
        for (int64_t l = 0; l < oa; ++l) cfma(acc, P[l * oa + j], U2[i4(oa, nv, i, l, a, b)]);
        U1[e] = acc;
        break;
      default:  // (i,j,a,b)
        for (int64_t k = 0; k < oa; ++k) cfma(acc, P[k * oa + i], U1[i4(oa, nv, k, j, a, b)]);
        U2[e] = acc;
        break;
    }
  }
}

__device__ double2 block_sum(double2 v, double2* sh) {
  for (int off = 32; off > 0; off >>= 1) {
    v.x += __shfl_xor(v.x, off, 64);
    v.y += __shfl_xor(v.y, off, 64);
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double2 r = sh[0];
  for (int w = 1; w < BLK / 64; ++w) r = cadd(r, sh[w]);
  __syncthreads();
  return r;
}

// The (e1, e2) partials of the general path: one block a job and slice of T
__global__ __launch_bounds__(BLK) void general_dots(int64_t oa, int64_t nv, int64_t nslice,
                                                    const apy_aat_job* __restrict__ jobs,
                                                    const JobRep* __restrict__ reps, double2* __restrict__ wsj) {
  __shared__ double2 sh[BLK / 64];
  const JLayout J = jlayout(oa, nv);
  const int q = blockIdx.y;
  const apy_aat_job jb = jobs[q];
  if (!jb.b2 || !jb.k2) return;
  const double2* B2 = (const double2*)jb.b2;
  const double2* T = wsj + reps[q].ket * J.per + J.small + J.part + rnd16(J.o2v2);
  double2 e1 = czero(), e2 = czero();
  for (int64_t e = blockIdx.x * (int64_t)BLK + threadIdx.x; e < J.o2v2; e += nslice * BLK) {
    int64_t r0 = e;
    const int64_t b = r0 % nv; r0 /= nv;
    const int64_t a = r0 % nv; r0 /= nv;
    const int64_t j = r0 % oa;
    const int64_t i = r0 / oa;
    const double2 tv = T[e];
    double2 ta = csub(csub(tv, T[i4(oa, nv, i, j, b, a)]), csub(T[i4(oa, nv, j, i, a, b)], T[i4(oa, nv, j, i, b, a)]));
    ta = make_double2(0.25 * ta.x, 0.25 * ta.y);
    cfma(e1, B2[e], ta);
    cfma(e2, B2[e], tv);
  }
  const double2 s1 = block_sum(e1, sh), s2 = block_sum(e2, sh);
  if (threadIdx.x == 0) {
    double2* part = wsj + q * J.per + J.small + 2 * blockIdx.x;
    part[0] = s1;
    part[1] = s2;
  }
}

// One block a job: its 20 scalars from the representatives' forms and H matrices and the npart partials (for
// an antisymmetric ket of pair_dots those of its nv (nv - 1) / 2 columns, anti_cols a partial).
__global__ __launch_bounds__(BLK) void scalars(int64_t oa, int64_t nv, int64_t npart, int64_t anti_cols, const double2* __restrict__ gam,
                                               int64_t rec, const apy_aat_job* __restrict__ jobs,
                                               const JobRep* __restrict__ reps, const double2* __restrict__ wsj,
                                               double2* __restrict__ out) {
  __shared__ double2 sh[BLK / 64];
  const JLayout J = jlayout(oa, nv);
  const apy_aat_job jb = jobs[blockIdx.x];
  const JobRep rp = reps[blockIdx.x];
  const GLayout L = glayout(oa, 0, nv);
  const double2* G = gam + jb.gamma * rec;
  const double2* x = G + L.x;
  const double2* y = G + L.y;
  const double2* ub = wsj + rp.bra * J.per;
  const double2* uk = wsj + rp.ket * J.per + 4 * J.ov;
  const double2* H = wsj + rp.ket * J.per + 12 * J.ov;
  const double2* part = wsj + blockIdx.x * J.per + J.small;
  const double2* B1 = (const double2*)jb.b1;
  const double2* K1 = (const double2*)jb.k1;
  double2* o = out + blockIdx.x * (int64_t)APY_AAT_NTERMS;
  double2 r[APY_AAT_NTERMS - 1];
#pragma unroll
  for (int k = 0; k < APY_AAT_NTERMS - 1; ++k) r[k] = czero();
  for (int64_t e = threadIdx.x; e < J.ov; e += BLK) {
    const double2 xe = x[e], ye = y[e], be = ub[e], bp = ub[3 * J.ov + e], bh = hat(ub, J.ov, e, 1.0);
    const double2 h0 = H[e], h1 = H[J.ov + e], h2 = H[2 * J.ov + e], h3 = H[3 * J.ov + e];
    if (B1) {
      const double2 b1 = B1[e];
      cfma(r[0], b1, xe);         // sx
      cfma(r[6], b1, h0);         // s1
      cfma(r[9], b1, h1);         // s4
      cfma(r[10], b1, h2);        // s5
    }
    if (K1) cfma(r[1], K1[e], ye);               // sy
    cfma(r[2], be, xe);           // bxx
    cfma(r[3], bh, xe);           // axx
    cfma(r[4], uk[e], ye);        // kyyp
    cfma(r[5], hat(uk, J.ov, e, 1.0), ye);       // kyy = -sum k^ y
    cfma(r[7], be, h0);           // s2
    cfma(r[8], bh, h0);           // s3
    cfma(r[11], bh, h1);          // s6
    cfma(r[12], bh, h2);          // s7
    cfma(r[13], be, h1);          // s8
    cfma(r[14], bp, h1);          // s9
    cfma(r[15], bp, h3);          // s10
    cfma(r[16], be, h2);          // s11
  }
  if (anti_cols && !reps[rp.k2].gen_k) npart = (nv * (nv - 1) / 2 + anti_cols - 1) / anti_cols;
  if (jb.b2 && jb.k2)
    for (int64_t e = threadIdx.x; e < npart; e += BLK) {
      r[17] = cadd(r[17], part[2 * e]);
      r[18] = cadd(r[18], part[2 * e + 1]);
    }
#pragma unroll
  for (int k = 0; k < APY_AAT_NTERMS - 1; ++k) {
    const double2 v = block_sum(r[k], sh);
    if (threadIdx.x == 0) o[1 + k] = v;
  }
  if (threadIdx.x == 0) o[0] = G[0];
}

// Norm pieces of each amplitude set: |t1|^2, |t2|^2, Re sum conj(t2[ijab]) t2[ijba], as NORM_SLICES partial
// sums a set (one block each: a set of 1e6 doubles in one block took 2.3 ms) and their sum in order.
constexpr int NORM_SLICES = 64;
__global__ __launch_bounds__(BLK) void norms_partial(int64_t oa, int64_t nv, const void* const* __restrict__ t1s,
                                                     const void* const* __restrict__ t2s, double* __restrict__ part) {
  __shared__ double2 sh[BLK / 64];
  const double2* t1 = (const double2*)t1s[blockIdx.y];
  const double2* t2 = (const double2*)t2s[blockIdx.y];
  const int64_t ov = oa * nv, first = blockIdx.x * (int64_t)BLK + threadIdx.x, step = (int64_t)NORM_SLICES * BLK;
  double n1 = 0.0, n2 = 0.0, nx = 0.0;
  if (t1)
    for (int64_t e = first; e < ov; e += step) n1 += t1[e].x * t1[e].x + t1[e].y * t1[e].y;
  if (t2)
    for (int64_t ij = blockIdx.x; ij < oa * oa; ij += NORM_SLICES) {
      const double2* t = t2 + ij * nv * nv;
      const int n = (int)nv;
      for (int e = threadIdx.x; e < n * n; e += BLK) {
        const double2 u = t[e], w = t[(e % n) * n + e / n];
        n2 += u.x * u.x + u.y * u.y;
        nx += u.x * w.x + u.y * w.y;
      }
    }
  const double2 s12 = block_sum(make_double2(n1, n2), sh);
  const double2 s3 = block_sum(make_double2(nx, 0.0), sh);
  if (threadIdx.x == 0) {
    double* p = part + 3 * (blockIdx.y * (int64_t)NORM_SLICES + blockIdx.x);
    p[0] = s12.x;
    p[1] = s12.y;
    p[2] = s3.x;
  }
}

__global__ __launch_bounds__(64) void norms_sum(const double* __restrict__ part, double* __restrict__ out) {
  if (threadIdx.x >= 3) return;
  double s = 0.0;
  for (int k = 0; k < NORM_SLICES; ++k) s += part[3 * (blockIdx.x * (int64_t)NORM_SLICES + k) + threadIdx.x];
  out[3 * blockIdx.x + threadIdx.x] = s;
}

// The two tensor kernels take nv up to 160 (accumulators of the sandwich) and oa up to 36 (X of pair_dots in
// LDS: oa 4 KB <= 147 KB); other sizes run the general quarter transforms.
constexpr int64_t SANDWICH_MAXV = 160, PAIR_MAXO = 36;

template <int RB, bool WL>
int launch_sandwich(dim3 grid, int64_t oa, int64_t nv, const double2* g, int64_t rec, const apy_aat_job* dj,
                    const JobRep* reps, double2* wsj, hipStream_t st) {
  const size_t lds = WL ? (size_t)nv * (size_t)(nv + 1) * sizeof(double2) : 0;
  if (lds > 65536)
    APY_HIP_TRY(hipFuncSetAttribute((const void*)sandwich<RB, WL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  sandwich<RB, WL><<<grid, BLK, lds, st>>>(oa, nv, g, rec, dj, reps, wsj);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

template <int KS>
int launch_pair_dots(int64_t oa, int64_t nv, const double2* g, int64_t rec, int64_t njobs, const apy_aat_job* dj,
                     const JobRep* reps, double2* wsj, hipStream_t st, int64_t npart) {
  const size_t lds = (size_t)oa * 256 * sizeof(double2);
  if (lds > 65536 - 4096)
    APY_HIP_TRY(hipFuncSetAttribute((const void*)pair_dots<KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  pair_dots<KS><<<dim3((unsigned)npart, (unsigned)njobs), PD_NT, lds, st>>>(oa, nv, g, rec, njobs, dj, reps, wsj);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

inline size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

extern "C" {

int64_t apy_aat_gamma_record(int64_t no, int64_t nf, int64_t nv) {
  if (no < 1 || nf < 0 || nf >= no || nv < 1) return 0;
  return glayout(no, nf, nv).size;
}

size_t apy_aat_gamma_workspace(int64_t n, int64_t no, int64_t batch) {
  if (n <= no || no < 1 || batch < 1) return 0;
  return al256((size_t)batch * no * 2 * no * sizeof(double2)) + al256((size_t)batch * no * (n - no) * sizeof(double2));
}

int apy_aat_gamma(int64_t n, int64_t no, int64_t nf, int64_t batch, const void* s, int64_t stride_s, void* gamma,
                  void* workspace, size_t ws_bytes, void* stream) {
  if (n <= no || no < 1 || no > BLK || nf < 0 || nf >= no || batch < 1 || batch > 2147483647 || !s || !gamma ||
      stride_s < n * n)
    return APY_E_ARG;
  const size_t need = apy_aat_gamma_workspace(n, no, batch);
  if (!workspace || ws_bytes < need) return APY_E_WORKSPACE;
  double2* ws = (double2*)workspace;
  double2* yw = (double2*)((char*)workspace + al256((size_t)batch * no * 2 * no * sizeof(double2)));
  gamma_kernel<<<(unsigned)batch, BLK, 0, (hipStream_t)stream>>>(n, no, nf, (const double2*)s, stride_s,
                                                                 (double2*)gamma, ws, yw);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

size_t apy_aat_axpby_workspace(int64_t count) {
  return count < 1 ? 0 : al256((size_t)count * sizeof(apy_aat_axpby_op));
}

int apy_aat_axpby(int64_t count, const apy_aat_axpby_op* ops, void* workspace, size_t ws_bytes, void* stream) {
  if (count < 1 || count > 65535 || !ops) return APY_E_ARG;
  int64_t nmax = 0;
  for (int64_t q = 0; q < count; ++q) {
    if (ops[q].n < 0 || (ops[q].n > 0 && (!ops[q].a || !ops[q].out))) return APY_E_ARG;
    if (ops[q].n > nmax) nmax = ops[q].n;
  }
  if (nmax == 0) return APY_OK;
  if (!workspace || ws_bytes < apy_aat_axpby_workspace(count)) return APY_E_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  APY_HIP_TRY(hipMemcpyAsync(workspace, ops, count * sizeof(apy_aat_axpby_op), hipMemcpyHostToDevice, st));
  dim3 grid(apy_grid1d(nmax, 4096), (unsigned)count);
  axpby_kernel<<<grid, BLK, 0, st>>>((const apy_aat_axpby_op*)workspace);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

size_t apy_aat_terms_workspace(int64_t oa, int64_t nv, int64_t njobs) {
  if (oa < 1 || nv < 1 || njobs < 1) return 0;
  const JLayout J = jlayout(oa, nv);
  return al256((size_t)njobs * sizeof(apy_aat_job)) + al256((size_t)njobs * sizeof(JobRep)) +
         (size_t)njobs * J.per * sizeof(double2);
}

int apy_aat_terms(int64_t oa, int64_t nv, const void* gamma, int64_t rec, int64_t ngamma, int64_t njobs,
                  const apy_aat_job* jobs, void* out, void* workspace, size_t ws_bytes, void* stream) {
  if (oa < 1 || nv < 1 || njobs < 1 || njobs > 65535 || !gamma || !jobs || !out ||
      rec < glayout(oa, 0, nv).size)
    return APY_E_ARG;
  for (int64_t q = 0; q < njobs; ++q)
    if (jobs[q].gamma < 0 || jobs[q].gamma >= ngamma) return APY_E_ARG;
  const size_t need = apy_aat_terms_workspace(oa, nv, njobs);
  if (!workspace || ws_bytes < need) return APY_E_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const size_t jb = al256((size_t)njobs * sizeof(apy_aat_job)), rb = al256((size_t)njobs * sizeof(JobRep));
  apy_aat_job* dj = (apy_aat_job*)workspace;
  JobRep* reps = (JobRep*)((char*)workspace + jb);
  double2* wsj = (double2*)((char*)workspace + jb + rb);
  APY_HIP_TRY(hipMemcpyAsync(dj, jobs, njobs * sizeof(apy_aat_job), hipMemcpyHostToDevice, st));
  const JLayout J = jlayout(oa, nv);
  const double2* g = (const double2*)gamma;
  const unsigned nj = (unsigned)njobs;
  job_reps<<<(unsigned)((njobs + BLK / 64 - 1) / (BLK / 64)), BLK, 0, st>>>(njobs, dj, reps);
  APY_LAUNCH_CHECK();
  antisym_check<<<dim3((unsigned)std::min<int64_t>(oa * oa, 256), nj, 2), BLK, 0, st>>>(oa, nv, dj, reps);
  APY_LAUNCH_CHECK();
  const bool fast = nv <= SANDWICH_MAXV && oa <= PAIR_MAXO;
  if (fast) {
    antisymmetrize<<<dim3((unsigned)std::min<int64_t>(oa * oa, 256), nj), BLK, 0, st>>>(oa, nv, dj, reps, wsj);
    APY_LAUNCH_CHECK();
  }
  contract_forms<<<dim3((unsigned)(4 * oa * ((nv + 31) / 32)), nj, 2), BLK, 0, st>>>(oa, nv, g, rec, dj, reps, wsj);
  APY_LAUNCH_CHECK();
  hmat_g<<<dim3((unsigned)((4 * J.ov + BLK - 1) / BLK), nj), BLK, 0, st>>>(oa, nv, g, rec, dj, reps, wsj);
  APY_LAUNCH_CHECK();
  hmat_h<<<dim3((unsigned)((4 * J.ov + BLK - 1) / BLK), nj), BLK, 0, st>>>(oa, nv, g, rec, dj, reps, wsj);
  APY_LAUNCH_CHECK();
  int64_t npart = 0, anti_cols = 0;
  if (fast) {
    // blocks a ket: enough that W (loaded by each) is used for several pairs, few enough to balance
    const int64_t RB = (nv + 15) / 16, units = oa * oa * RB;
    const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>((units + 31) / 32, 64)), nj);
    int s = APY_OK;
    switch (RB) {
      case 1: s = launch_sandwich<1, true>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      case 2: s = launch_sandwich<2, true>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      case 3: s = launch_sandwich<3, true>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      case 4: s = launch_sandwich<4, true>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      case 5: s = launch_sandwich<5, true>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      case 6: s = launch_sandwich<6, true>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      case 7:
      case 8: s = launch_sandwich<8, false>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
      default: s = launch_sandwich<10, false>(grid, oa, nv, g, rec, dj, reps, wsj, st); break;
    }
    if (s != APY_OK) return s;
    npart = (nv * nv + PD_COLS - 1) / PD_COLS;
    anti_cols = PD_COLS;
    switch ((oa + 3) / 4) {
      case 1: s = launch_pair_dots<1>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 2: s = launch_pair_dots<2>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 3: s = launch_pair_dots<3>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 4: s = launch_pair_dots<4>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 5: s = launch_pair_dots<5>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 6: s = launch_pair_dots<6>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 7: s = launch_pair_dots<7>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      case 8: s = launch_pair_dots<8>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
      default: s = launch_pair_dots<9>(oa, nv, g, rec, njobs, dj, reps, wsj, st, npart); break;
    }
    if (s != APY_OK) return s;
  } else {
    for (int stage = 0; stage < 4; ++stage) {
      quarter<<<dim3(apy_grid1d(J.o2v2, 2048), nj), BLK, 0, st>>>(stage, oa, nv, g, rec, dj, reps, wsj);
      APY_LAUNCH_CHECK();
    }
    npart = std::min<int64_t>(64, J.part / 2);
    general_dots<<<dim3((unsigned)npart, nj), BLK, 0, st>>>(oa, nv, npart, dj, reps, wsj);
    APY_LAUNCH_CHECK();
  }
  scalars<<<nj, BLK, 0, st>>>(oa, nv, npart, anti_cols, g, rec, dj, reps, wsj, (double2*)out);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

size_t apy_aat_norms_workspace(int64_t nset) {
  return nset < 1 ? 0 : 2 * al256((size_t)nset * sizeof(void*)) + al256((size_t)nset * NORM_SLICES * 3 * sizeof(double));
}

int apy_aat_norms(int64_t oa, int64_t nv, int64_t nset, const void* const* t1, const void* const* t2, void* out,
                  void* workspace, size_t ws_bytes, void* stream) {
  if (oa < 1 || nv < 1 || nset < 1 || nset > 2147483647 || !t1 || !t2 || !out) return APY_E_ARG;
  if (!workspace || ws_bytes < apy_aat_norms_workspace(nset)) return APY_E_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const void** d1 = (const void**)workspace;
  const void** d2 = (const void**)((char*)workspace + al256((size_t)nset * sizeof(void*)));
  double* part = (double*)((char*)workspace + 2 * al256((size_t)nset * sizeof(void*)));
  APY_HIP_TRY(hipMemcpyAsync(d1, t1, nset * sizeof(void*), hipMemcpyHostToDevice, st));
  APY_HIP_TRY(hipMemcpyAsync(d2, t2, nset * sizeof(void*), hipMemcpyHostToDevice, st));
  for (int64_t s0 = 0; s0 < nset; s0 += 65535) {
    const unsigned n = (unsigned)std::min<int64_t>(65535, nset - s0);
    norms_partial<<<dim3(NORM_SLICES, n), BLK, 0, st>>>(oa, nv, d1 + s0, d2 + s0, part + s0 * NORM_SLICES * 3);
    APY_LAUNCH_CHECK();
  }
  norms_sum<<<(unsigned)nset, 64, 0, st>>>(part, (double*)out);
  APY_LAUNCH_CHECK();
  return APY_OK;
}

}  // extern "C"
