// FP64 grid stage on product grids.
//
// The grid is a product (Gauss-Hermite in z, Gauss-Laguerre in r) and every
// basis state a product of a radial and an axial function,
//   psi = f(r) c(z),   d_r psi = f1 c,   (Lambda / r) psi = f2 c,   d_z psi = f c',
//   lap psi = f4 c + f c'',
// with few different radial functions: the states of one block and spin differ
// in n_r only, and the two parities share them.  So the contractions of the
// densities and of the projection go one direction at a time:
//   Z_t[p](z)      = sum_{a in fa, b in fb} c_t1(z, a) rho(a, b) c_t2(z, b)     (k_sep_z)
//   dens_c(r, z)   = sum_t sum_p R_ct[p](r) Z_t[p](z)                           (k_sep_dens)
//   Y_t[p](z)      = sum_c sum_r R'_ct[p](r) F_c(r, z)                          (k_sep_proj)
//   h(a, b)        = 2 sum_z sum_t c_t1(z, a) Y_t[p](z) c_t2(z, b)              (k_sep_expand)
// where p runs over the pairs (fa, fb) of radial functions that occur in a
// block structure ("slots", per pair of spins) and t over the pairs of axial
// functions: (c, c), (c, c'), (c', c), (c', c') and, for the projection only,
// (c, c'') + (c'', c).  At N_sh = 16 (nxy 103 926, 40 x 40 points, 2 736 slots)
// that is 1.3e9 FLOP per frequency where the contraction over all 1 600 points
// at once takes 1.5e10; the results differ in summation order only.
//
// The tables the caller passes are not labelled with quantum numbers, so the
// factors are recovered from the tables themselves (k_sep_fit, one least-
// squares product fit per state) and the plan is used only if every table of
// every state is a product to rounding; any other basis keeps the kernels that
// contract over all points.
#pragma once

// Largest residual of a product fit, relative to the table's largest value: what a
// larger one left out would be a change of the caller's tables.  Their own rounding
// leaves up to 1.9e-15 (HO tables of 2 to 20 shells, 8 x 6 to 120 x 100 points);
// states that are no products leave 1e-3 or more.
constexpr double SEP_TOL = 1e-14;
// Radial functions this close in all four tables are one: the gauge of f4 is the
// least certain, members of one function differ by up to 9.4e-15 (64 x 64 points).
constexpr double SEP_SAME = 3e-14;
constexpr int SEP_MAX1D = 256;      // points per direction the fit's LDS holds

// ---- product fit of the tables ------------------------------------------------
struct SepFit {
  const double *tab[5];   // wf, wfdr, wfdp, wfdz, wfd2_all
  int nz, nr, dqp, nzp;
  double *fr;             // [dqp][4][nr]: f, f1, f2, f4; f of unit norm
  double *fz;             // [3][dqp][nzp]: c, c', c'', zero from nz to nzp
  double *resid;          // [dqp] largest residual of the five tables, relative to each table's largest value
};

__device__ inline double sep_max(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = red[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) s = fmax(s, red[k]);
  return s;
}

// One workgroup per state: alternating least squares from the row of the
// largest value.  c'' is the part of the Laplacian along f (its gauge against
// f4 c is that f4 is orthogonal to f), so it is the same for the states that
// share a radial function.
__global__ void __launch_bounds__(256) k_sep_fit(SepFit S) {
  __shared__ double f[SEP_MAX1D], c[SEP_MAX1D], g[SEP_MAX1D], q[SEP_MAX1D], red[4];
  __shared__ int piv;
  const int a = blockIdx.x, nz = S.nz, nr = S.nr, G = nz * nr, tid = threadIdx.x;
  const double *M = S.tab[0] + (size_t)a * G;
  double mx = 0.0;
  for (int i = tid; i < G; i += 256) mx = fmax(mx, fabs(M[i]));
  mx = sep_max(mx, red);
  if (tid == 0) piv = G;
  __syncthreads();
  for (int i = tid; i < G; i += 256)
    if (fabs(M[i]) == mx) atomicMin(&piv, i);
  __syncthreads();
  // a table with no largest value (all zero or not finite) is no product
  if (!(mx > 0.0) || !(mx < 1e300) || piv >= G) {
    if (tid == 0) S.resid[a] = 1.0;
    return;
  }
  const int rp = piv / nz;
  if (tid < nz) c[tid] = M[rp * nz + tid];
  __syncthreads();
  auto dot = [](const double *u, const double *v, int n) {
    double s = 0.0;
    for (int i = 0; i < n; ++i) s = __builtin_fma(u[i], v[i], s);
    return s;
  };
  // out(r) = sum_z T(r, z) c(z) / |c|^2 and out(z) = sum_r T(r, z) f(r) / |f|^2
  auto fit_r = [&](const double *T, double *out) {
    const double n = dot(c, c, nz);
    if (tid < nr) out[tid] = dot(T + (size_t)tid * nz, c, nz) / n;
    __syncthreads();
  };
  auto fit_z = [&](const double *T, double *out) {
    const double n = dot(f, f, nr);
    if (tid < nz) {
      double s = 0.0;
      for (int r = 0; r < nr; ++r) s = __builtin_fma(T[(size_t)r * nz + tid], f[r], s);
      out[tid] = s / n;
    }
    __syncthreads();
  };
  fit_r(M, f);
  fit_z(M, c);
  fit_r(M, f);
  // f of unit norm, its first value of at least half the largest positive
  {
    double fm = 0.0;
    for (int r = 0; r < nr; ++r) fm = fmax(fm, fabs(f[r]));
    double s = sqrt(dot(f, f, nr));
    for (int r = 0; r < nr; ++r)
      if (fabs(f[r]) >= 0.5 * fm) { if (f[r] < 0.0) s = -s; break; }
    __syncthreads();
    if (tid < nr) f[tid] /= s;
    if (tid < nz) c[tid] *= s;
    __syncthreads();
  }
  double worst = 0.0;
  // residual of table T against u(r) v(z) + u2(r) v2(z)
  auto check = [&](const double *T, const double *u, const double *v, const double *u2, const double *v2) {
    double m = 0.0, d = 0.0;
    for (int i = tid; i < G; i += 256) {
      const int r = i / nz, z = i - r * nz;
      const double t = T[i];
      double e = __builtin_fma(-u[r], v[z], t);
      if (u2) e = __builtin_fma(-u2[r], v2[z], e);
      m = fmax(m, fabs(t));
      d = (e == e) ? fmax(d, fabs(e)) : 1e300;
    }
    m = sep_max(m, red);
    d = sep_max(d, red);
    if (d > 0.0) worst = fmax(worst, m > 0.0 ? d / m : 1.0);
    __syncthreads();
  };
  auto put_r = [&](int x, const double *v) {
    if (tid < nr) S.fr[((size_t)a * 4 + x) * nr + tid] = v[tid];
  };
  auto put_z = [&](int x, const double *v) {
    if (tid < S.nzp) S.fz[((size_t)x * S.dqp + a) * S.nzp + tid] = tid < nz ? v[tid] : 0.0;
  };
  check(M, f, c, nullptr, nullptr);
  put_r(0, f);
  put_z(0, c);
  for (int x = 1; x <= 2; ++x) {
    const double *T = S.tab[x] + (size_t)a * G;
    fit_r(T, g);
    check(T, g, c, nullptr, nullptr);
    put_r(x, g);
    __syncthreads();
  }
  {
    const double *T = S.tab[3] + (size_t)a * G;
    fit_z(T, q);
    check(T, f, q, nullptr, nullptr);
    put_z(1, q);
    __syncthreads();
  }
  {
    const double *T = S.tab[4] + (size_t)a * G;
    fit_z(T, q);
    const double n = dot(c, c, nz);
    if (tid < nr) {
      double s = 0.0;
      for (int z = 0; z < nz; ++z) s = __builtin_fma(__builtin_fma(-f[tid], q[z], T[(size_t)tid * nz + z]), c[z], s);
      g[tid] = s / n;
    }
    __syncthreads();
    check(T, g, c, f, q);
    put_r(3, g);
    put_z(2, q);
  }
  if (tid == 0) S.resid[a] = worst;
}

// ---- tables of radial products -------------------------------------------------
// Rows of the density contraction per axial pair t = (c, c), (c, c'), (c', c),
// (c', c'), each a radial product; sums that only occur together are one row.
// Same spin (P of density_accumulate):
//   t0: f f | f f2 + f2 f | f1 f1 + f2 f2 | f f1 - f1 f     t1: f f | f1 f | f2 f
//   t2: f f | f f1 | f f2                                   t3: f f
// opposite spins (Q), e = +1 for (up, down), -1 for (down, up):
//   t0: f f | f2 f + f f2 | e (f f2 - f2 f) + f f1 + f1 f | f1 f1 + e (f1 f2 - f2 f1) / 2 |
//       e f2 f2 + (f2 f1 - f1 f2) / 2 | f f1 - f1 f
//   t1: f f | (f1 - e f2) f     t2: f f | f (f1 + e f2)     t3: f f
// pairing: t0: f f.
// Each t's rows are padded to whole 16-row tiles.
constexpr int SEP_NT = 4;
__host__ __device__ constexpr int sep_rows(int kind, bool same, int t) {
  return kind ? (t == 0 ? 1 : 0) : (same ? (t == 0 ? 4 : (t == 3 ? 1 : 3)) : (t == 0 ? 6 : (t == 3 ? 1 : 2)));
}
__host__ __device__ inline int sep_row0(int kind, bool same, int t, int nr) {
  int o = 0;
  for (int k = 0; k < t; ++k) o += (sep_rows(kind, same, k) * nr + 15) / 16 * 16;
  return o;
}

// Terms of the projection per axial pair (t4 is (c, c'') + (c'', c)): field
// (z, z') and radial product.  The fields' own symmetries (k_fields) merge
//   F04 = F40:  f f4 + f4 f (t0) and f f (t4);
//   same spin:  F22 = F11: f1 f1 + f2 f2, F21 = F12: f1 f2 + f2 f1;
//   opposite:   F21 = -F12: f1 f2 - f2 f1 (F22 on its own).
constexpr int SEP_PT = 5;
__host__ __device__ constexpr int sep_terms(int kind, bool same, int t) {
  return kind ? (t == 0 ? 1 : 0) : (t == 0 ? (same ? 8 : 9) : (t <= 2 ? 3 : 1));
}
__host__ __device__ inline int sep_k0(int kind, bool same, int t, int nr4) {
  int o = 0;
  for (int k = 0; k < t; ++k) o += sep_terms(kind, same, k) * nr4;
  return o;
}
// field component (index of the 104) of term c of axial pair t
inline int sep_field(int kind, int t, int c, int sa, int sb) {
  if (kind) return 100 + (sb == 0 ? (sa == 0 ? 0 : 1) : (sa == 0 ? 2 : 3));
  int z, zp;
  if (t == 0) {   // 00, 01, 10, 02, 20, 11, 12, 04, 22
    z = (c == 2 || c == 5 || c == 6) ? 1 : (c == 4 || c == 8 ? 2 : 0);
    zp = (c == 1 || c == 5) ? 1 : (c == 3 || c == 6 || c == 8 ? 2 : (c == 7 ? 4 : 0));
  } else if (t == 1) {
    z = c; zp = 3;
  } else if (t == 2) {
    z = 3; zp = c;
  } else if (t == 3) {
    z = zp = 3;
  } else {
    z = 0; zp = 4;
  }
  return mf_index(z, zp, sa, sb);
}

struct SepTab {           // one (block structure, pair of spins): the slots' radial products
  const int2 *key;        // [n] radial functions of the rows and the columns
  int n, kind, sa, sb;
  double *rd;             // density [pad4(n)][rows], null: not needed
  double *rp;             // projection [k][pad16(n)], null: not needed
};

__global__ void k_sep_rtab(SepTab T, const double *__restrict__ ftab, int nr, int ncls) {
  const bool same = T.sa == T.sb;
  const double e = T.sb == 1 ? 1.0 : -1.0;
  auto F = [&](int cls, int x, int r) { return ftab[((size_t)x * ncls + cls) * nr + r]; };
  if (T.rd) {
    const int L = sep_row0(T.kind, same, SEP_NT, nr), np = (T.n + 3) & ~3;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < (long)L * np; i += (long)gridDim.x * blockDim.x) {
      const int p = (int)(i / L), row = (int)(i - (long)p * L);
      int t = 0, r0 = 0;
      for (int k = 1; k < SEP_NT; ++k) {
        const int q = sep_row0(T.kind, same, k, nr);
        if (sep_rows(T.kind, same, k) > 0 && row >= q) { t = k; r0 = q; }
      }
      const int c = (row - r0) / nr, r = (row - r0) - c * nr;
      double v = 0.0;
      if (p < T.n && c < sep_rows(T.kind, same, t)) {
        const int2 k = T.key[p];
        const double a0 = F(k.x, 0, r), a1 = F(k.x, 1, r), a2 = F(k.x, 2, r);
        const double b0 = F(k.y, 0, r), b1 = F(k.y, 1, r), b2 = F(k.y, 2, r);
        if (c == 0) v = a0 * b0;
        else if (t == 0 && same) v = c == 1 ? a0 * b2 + a2 * b0 : (c == 2 ? a1 * b1 + a2 * b2 : a0 * b1 - a1 * b0);
        else if (t == 0) {
          const double x = a1 * b2 - a2 * b1;
          v = c == 1 ? a2 * b0 + a0 * b2
                     : (c == 2 ? e * (a0 * b2 - a2 * b0) + (a0 * b1 + a1 * b0)
                               : (c == 3 ? a1 * b1 + 0.5 * e * x : (c == 4 ? e * (a2 * b2) - 0.5 * x : a0 * b1 - a1 * b0)));
        } else if (same) v = t == 1 ? (c == 1 ? a1 : a2) * b0 : a0 * (c == 1 ? b1 : b2);
        else v = t == 1 ? (a1 - e * a2) * b0 : a0 * (b1 + e * b2);
      }
      T.rd[i] = v;
    }
  }
  if (T.rp) {
    const int nr4 = (nr + 3) & ~3, np = (T.n + 15) & ~15, nk = sep_k0(T.kind, same, SEP_PT, nr4);
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < (long)nk * np; i += (long)gridDim.x * blockDim.x) {
      const int k = (int)(i / np), p = (int)(i - (long)k * np);
      int t = 0, k0 = 0;
      for (int u = 1; u < SEP_PT; ++u) {
        const int q = sep_k0(T.kind, same, u, nr4);
        if (sep_terms(T.kind, same, u) > 0 && k >= q) { t = u; k0 = q; }
      }
      const int c = (k - k0) / nr4, r = (k - k0) - c * nr4;
      double v = 0.0;
      if (p < T.n && r < nr) {
        const int2 s = T.key[p];
        const double a0 = F(s.x, 0, r), a1 = F(s.x, 1, r), a2 = F(s.x, 2, r), a4 = F(s.x, 3, r);
        const double b0 = F(s.y, 0, r), b1 = F(s.y, 1, r), b2 = F(s.y, 2, r), b4 = F(s.y, 3, r);
        if (t == 0)
          switch (c) {
            case 0: v = a0 * b0; break;
            case 1: v = a0 * b1; break;
            case 2: v = a1 * b0; break;
            case 3: v = a0 * b2; break;
            case 4: v = a2 * b0; break;
            case 5: v = same ? a1 * b1 + a2 * b2 : a1 * b1; break;
            case 6: v = same ? a1 * b2 + a2 * b1 : a1 * b2 - a2 * b1; break;
            case 7: v = a0 * b4 + a4 * b0; break;
            default: v = a2 * b2; break;
          }
        else if (t == 1) v = (c == 0 ? a0 : (c == 1 ? a1 : a2)) * b0;
        else if (t == 2) v = a0 * (c == 0 ? b0 : (c == 1 ? b1 : b2));
        else v = a0 * b0;
      }
      T.rp[i] = v;
    }
  }
}

// ---- densities: axial contraction ----------------------------------------------
// A slot's matrix elements: offset in the structure's storage, row and column state.
struct SepSlot { int first, count, mat, zoff; };   // elements; offset of its Z rows (densities) or Y rows (projection)
// The slots of one structure, pair of spins and radial function of the columns
// form a bundle: they read (write) rows of the same matrix columns.
struct SepArgs {
  int nz, nr, dqp, nzp;       // nzp: nz padded to 8, the stride of the axial tables and of Y
  long nxy;
  const double *fz;           // [3][dqp][nzp]
  const double *tab;          // tables of radial products
  const double *rsp;          // [w][8][nxy]
  int slot_of[4];             // rsp slots (pairs) of rho0, kap0, rho1, kap1
  double *zy;                 // per active point: Z, later Y
  long zstride, ystride;
  double *acc;                // [split][active][rows][2 nz] partial densities
  long astride;               // doubles per active point
  double *dens, *flds, *hsp;
  const double *wdcori;
  const int *act;
  int na, skip;
};

// Z_t(z) = sum over the slot's elements of rho(a, b) c_t1(z, a) c_t2(z, b): a
// product of [8 frequencies x (re, im)] x elements by elements x [z], four
// elements per v_mfma_f64_16x16x4 step, the four axial products formed in
// registers from the states' axial functions (four loads and four multiplies
// for the four products' matrix instructions of a 16-point tile).  One wave
// per slot, 8 frequencies and ZT tiles of 16 axial points; few frequencies
// leave rows of the matrix instructions empty, which costs less than the
// scalar loads of a vector kernel did (one lane per axial point, rho through
// scalar loads: 2.3 ms for 48 points of N_sh = 16, 75 us for one).
// The prefetched loads are unconditional (clamped to the list) so that they stay
// in flight across the products: a load under a branch is waited for at its end.
template <int ZT, bool MEAN>
__device__ inline void sep_z_slot(const SepArgs &A, const SepSlot S, const int4 *__restrict__ elems) {
  constexpr int NX = MEAN ? 4 : 1;
  const int lane = threadIdx.x & 63, mi = lane & 15, mk = lane >> 4;
  const int y = min((int)blockIdx.y * 8 + (mi >> 1), A.na - 1);
  const double *__restrict__ rho = A.rsp + ((size_t)A.act[y] * 8 + 2 * A.slot_of[S.mat] + (mi & 1)) * A.nxy;
  const size_t xs = (size_t)A.dqp * A.nzp;
  // rows this lane stores (row 4 v + mk of the product)
  bool st[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int yo = blockIdx.y * 8 + 2 * v + (mk >> 1);
    st[v] = yo < A.na && A.act[min(yo, A.na - 1)] != A.skip;
  }
  int z[ZT];
#pragma unroll
  for (int t = 0; t < ZT; ++t) z[t] = min((int)(blockIdx.z * ZT + t) * 16 + mi, A.nzp - 1);
  v4d C[ZT][NX];
#pragma unroll
  for (int t = 0; t < ZT; ++t)
#pragma unroll
    for (int k = 0; k < NX; ++k) C[t][k] = v4d{0, 0, 0, 0};
  const int4 *__restrict__ el = elems + S.first;
  auto load = [&](int4 r, double (&c)[ZT][4]) {
    const double *fa = A.fz + (size_t)r.y * A.nzp, *fb = A.fz + (size_t)r.z * A.nzp;
#pragma unroll
    for (int t = 0; t < ZT; ++t) {
      c[t][0] = fa[z[t]];
      c[t][2] = fb[z[t]];
      if (MEAN) {
        c[t][1] = fa[xs + z[t]];
        c[t][3] = fb[xs + z[t]];
      }
    }
  };
  const int n = S.count;
  int4 rn = el[min(mk, n - 1)];
  double vn = rho[rn.x], cn[ZT][4];
  load(rn, cn);
  rn = el[min(4 + mk, n - 1)];
  for (int s = 0; s < n; s += 4) {
    const double v = s + mk < n ? vn : 0.0;
    double X[ZT][NX];
#pragma unroll
    for (int t = 0; t < ZT; ++t) {
      X[t][0] = cn[t][0] * cn[t][2];
      if (MEAN) {
        X[t][NX / 2 - 1] = cn[t][0] * cn[t][3];
        X[t][NX / 2] = cn[t][1] * cn[t][2];
        X[t][NX - 1] = cn[t][1] * cn[t][3];
      }
    }
    vn = rho[rn.x];
    load(rn, cn);
    rn = el[min(s + 8 + mk, n - 1)];
    loads_first();
#pragma unroll
    for (int k = 0; k < NX; ++k)
#pragma unroll
      for (int t = 0; t < ZT; ++t) C[t][k] = mfma64(v, X[t][k], C[t][k]);
  }
  double *out = A.zy + (size_t)(blockIdx.y * 8 + (mk >> 1)) * A.zstride + S.zoff + (size_t)(mk & 1) * A.nz;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    if (st[v])
#pragma unroll
      for (int t = 0; t < ZT; ++t) {
        const int zt = (blockIdx.z * ZT + t) * 16 + mi;
        if (zt < A.nz)
#pragma unroll
          for (int k = 0; k < NX; ++k) out[(size_t)(2 * k) * A.nz + zt] = C[t][k][v];
      }
    out += 2 * A.zstride;
  }
}

// Four slots of a bundle per workgroup, one per wave; the host deals the bundles
// to the XCDs (workgroup x runs on XCD x % 8), so that a bundle's lines are
// fetched into one L2.
template <int ZT>
__global__ void __launch_bounds__(256) k_sep_z(SepArgs A, const SepSlot *__restrict__ slots,
                                               const int4 *__restrict__ elems) {
  const SepSlot S = slots[__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)))];
  if (S.count == 0) return;
  if ((S.mat & 1) == 0) sep_z_slot<ZT, true>(A, S, elems);
  else sep_z_slot<ZT, false>(A, S, elems);
}

// The same for more than 8 points: the NW waves of a workgroup take the same slot for
// 8 frequencies each, the axial products of 8 elements formed once for all of them
// and kept in LDS in the layout of the operand, the loads of the next 8 in flight
// during the products of these.  In k_sep_z every wave loads the functions for
// itself, and the L1 serves those at its limit: N_sh = 16, 128 points 1.75 ms,
// here 1.31 ms (0.34 ms at the peak matrix rate, and 1.9 GB of Z to write).
template <int ZT, int NW, bool MEAN>
__device__ inline void sep_z_wide(const SepArgs &A, const SepSlot S, const int4 *__restrict__ elems,
                                  double (*__restrict__ buf)[2 * 4 * ZT * 64]) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int NX = MEAN ? 4 : 1, NP = (ZT + NW - 1) / NW;   // products' element and pair of z per thread
  const int tid = threadIdx.x, lane = tid & 63, mi = lane & 15, mk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), y0 = ((int)blockIdx.y * NW + wv) * 8;
  const bool on = y0 < A.na;               // waves past the last point wait with the others
  const double *__restrict__ rho =
      A.rsp + ((size_t)A.act[min(y0 + (mi >> 1), A.na - 1)] * 8 + 2 * A.slot_of[S.mat] + (mi & 1)) * A.nxy;
  const size_t xs = (size_t)A.dqp * A.nzp;
  const int4 *__restrict__ el = elems + S.first;
  const int n = S.count;
  // this thread's products: element pe[i] of the chunk, axial points zp[i] and + 1
  int pe[NP], zp[NP], at[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int q = min(tid + 64 * NW * i, 64 * ZT - 1), z = 2 * (q % (8 * ZT));
    pe[i] = q / (8 * ZT);
    zp[i] = min((int)blockIdx.z * ZT * 16 + z, A.nzp - 2);
    at[i] = ((pe[i] >> 2) * NX * ZT + (z >> 4)) * 64 + (pe[i] & 3) * 16 + (z & 15);
  }
  v4d C[ZT][NX];
#pragma unroll
  for (int t = 0; t < ZT; ++t)
#pragma unroll
    for (int k = 0; k < NX; ++k) C[t][k] = v4d{0, 0, 0, 0};
  v2d f[NP][4];
  int4 rx[NP];
  int rr[2];
  double vn[2];
  auto next = [&](int e0) {                // list entries of a chunk
#pragma unroll
    for (int i = 0; i < NP; ++i) rx[i] = el[min(e0 + pe[i], n - 1)];
#pragma unroll
    for (int s = 0; s < 2; ++s) rr[s] = el[min(e0 + 4 * s + mk, n - 1)].x;
  };
  auto load = [&] {                        // its functions and matrix elements
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const double *fa = A.fz + (size_t)rx[i].y * A.nzp + zp[i], *fb = A.fz + (size_t)rx[i].z * A.nzp + zp[i];
      f[i][0] = *(const v2d *)fa;
      f[i][2] = *(const v2d *)fb;
      if (MEAN) {
        f[i][1] = *(const v2d *)(fa + xs);
        f[i][3] = *(const v2d *)(fb + xs);
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) vn[s] = rho[rr[s]];
  };
  auto form = [&](double *d) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      v2d *p = (v2d *)(d + at[i]);
      p[0] = f[i][0] * f[i][2];
      if (MEAN) {
        p[1 * ZT * 32] = f[i][0] * f[i][3];
        p[2 * ZT * 32] = f[i][1] * f[i][2];
        p[3 * ZT * 32] = f[i][1] * f[i][3];
      }
    }
  };
  next(0);
  load();
  next(8);
  form(buf[0]);
  __syncthreads();
  int cur = 0;
  for (int e0 = 0; e0 < n; e0 += 8) {
    double v[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) v[s] = e0 + 4 * s + mk < n ? vn[s] : 0.0;
    load();
    next(e0 + 16);
    loads_first();
    const double *d = buf[cur] + lane;
    if (on)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (s == 0 || e0 + 4 < n)
#pragma unroll
          for (int k = 0; k < NX; ++k)
#pragma unroll
            for (int t = 0; t < ZT; ++t) C[t][k] = mfma64(v[s], d[((s * NX + k) * ZT + t) * 64], C[t][k]);
    cur ^= 1;
    if (e0 + 8 < n) form(buf[cur]);
    __syncthreads();
  }
  if (!on) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int yo = y0 + 2 * v + (mk >> 1);           // row 4 v + mk of the product
    if (yo < A.na && A.act[yo] != A.skip) {
      double *out = A.zy + (size_t)yo * A.zstride + S.zoff + (size_t)(mk & 1) * A.nz;
#pragma unroll
      for (int t = 0; t < ZT; ++t) {
        const int zt = (blockIdx.z * ZT + t) * 16 + mi;
        if (zt < A.nz)
#pragma unroll
          for (int k = 0; k < NX; ++k) out[(size_t)(2 * k) * A.nz + zt] = C[t][k][v];
      }
    }
  }
}

// One slot per workgroup, in the order of k_sep_z's workgroups of four.
template <int ZT, int NW>
__global__ void __launch_bounds__(64 * NW, ZT > 2 ? 3 : 4) k_sep_z_wide(SepArgs A, const SepSlot *__restrict__ slots,
                                                                        const int4 *__restrict__ elems) {
  __shared__ __attribute__((aligned(16))) double buf[2][2 * 4 * ZT * 64];
  const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
  const SepSlot S = slots[((i >> 2) * 8 + x) * 4 + (i & 3)];
  if (S.count == 0) return;
  if ((S.mat & 1) == 0) sep_z_wide<ZT, NW, true>(A, S, elems, buf);
  else sep_z_wide<ZT, NW, false>(A, S, elems, buf);
}

// ---- densities: radial contraction ----------------------------------------------
struct SepDJob {            // 16-row tiles of one axial pair of one (structure, spins)
  int64_t rd;               // offset of the class's table
  int n, ld;                // slots; rows per slot
  int row, nrt;             // first table row, tiles (1..4; 0: an empty job)
  int zoff, zld;            // Z of the class's first slot at this axial pair; stride between slots
  int arow, pad;            // output row of the first tile
};

// The jobs of the two radial contractions: workgroup b runs on XCD b % 8 and takes
// that XCD's jobs (list entries [x len, (x + 1) len), len = njob / 8), `run` jobs
// at a time for every point: the tables of a run stay in the XCD's L2 while the
// points pass by, and its jobs, which read the same operands of a point, run side
// by side.
__device__ inline int sep_job(int njob, int run, int na, int &y) {
  const int x = blockIdx.x & 7, i = blockIdx.x >> 3, g = i / (run * na), r = i - g * run * na;
  y = r / run;
  return x * (njob >> 3) + g * run + r % run;
}

// One job with RT row tiles.  No branch in the loop (a job's tile count is a
// template argument, the load after the last step repeats it), so that the loads
// of a step stay in flight across the products of the one before.
template <int CT, int RT>
__device__ inline void sep_dens_job(const SepArgs &A, const SepDJob &J, int y, int ncg, int nsplit) {
  const int lane = threadIdx.x, mi = lane & 15, mk = lane >> 4;
  const int cg = blockIdx.y % ncg, spl = blockIdx.y / ncg;
  const int W = 2 * A.nz;
  const int nst = (J.n + 3) >> 2;
  const int s0 = (int)((long)spl * nst / nsplit), s1 = (int)((long)(spl + 1) * nst / nsplit);
  v4d C[RT][CT];
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int c = 0; c < CT; ++c) C[q][c] = v4d{0, 0, 0, 0};
  if (s0 < s1) {
    const double *__restrict__ R = A.tab + J.rd + J.row + mi;
    const double *__restrict__ Z = A.zy + (size_t)y * A.zstride + J.zoff;
    int col[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) col[c] = min((cg * CT + c) * 16 + mi, W - 1);
    double an[RT], bn[CT];
    auto load = [&](int s) {
      const int p = 4 * s + mk;                    // table rows are zero past the last slot
      const double *r = R + (size_t)p * J.ld, *z = Z + (size_t)min(p, J.n - 1) * J.zld;
#pragma unroll
      for (int q = 0; q < RT; ++q) an[q] = r[16 * q];
#pragma unroll
      for (int c = 0; c < CT; ++c) bn[c] = z[col[c]];
    };
    load(s0);
    for (int s = s0; s < s1; ++s) {
      double a[RT], b[CT];
#pragma unroll
      for (int q = 0; q < RT; ++q) a[q] = an[q];
#pragma unroll
      for (int c = 0; c < CT; ++c) b[c] = bn[c];
      load(min(s + 1, s1 - 1));
      loads_first();
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int c = 0; c < CT; ++c) C[q][c] = mfma64(a[q], b[c], C[q][c]);
    }
  }
  double *out = A.acc + ((size_t)spl * A.na + y) * A.astride + (size_t)J.arow * W;
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int k = (cg * CT + c) * 16 + mi;
      if (k < W)
#pragma unroll
        for (int v = 0; v < 4; ++v) out[(size_t)(16 * q + 4 * v + mk) * W + k] = C[q][c][v];
    }
}

// acc(row, (ri, z)) = sum_p R[p][row] Z_t[p][(ri, z)] on v_mfma_f64_16x16x4:
// up to 4 row tiles by CT column tiles per wave, four slots per step, the
// operands of the next step in flight during the products of this one.  One
// wave's 20 products of a step (1 280 cycles at 40 points) hide its 9 operand
// loads; an XCD reads its own part of the tables only.  With few points the slots
// are split (blockIdx.y), the parts added in order by k_sep_sum.
template <int CT>
__global__ void __launch_bounds__(64, 2) k_sep_dens(SepArgs A, const SepDJob *__restrict__ jobs, int njob, int ncg,
                                                    int nsplit) {
  int y;
  const SepDJob J = jobs[sep_job(njob, njob >> 3, A.na, y)];
  if (A.act[y] == A.skip) return;
  switch (J.nrt) {
    case 1: sep_dens_job<CT, 1>(A, J, y, ncg, nsplit); break;
    case 2: sep_dens_job<CT, 2>(A, J, y, ncg, nsplit); break;
    case 3: sep_dens_job<CT, 3>(A, J, y, ncg, nsplit); break;
    case 4: sep_dens_job<CT, 4>(A, J, y, ncg, nsplit); break;
    default: break;
  }
}

// acc of split 0 += those of the other splits, in order
__global__ void k_sep_sum(double *__restrict__ acc, int nsplit, long n) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    double v = acc[e];
    for (int s = 1; s < nsplit; ++s) v += acc[(size_t)s * n + e];
    acc[e] = v;
  }
}

struct SepAcc {     // first output row of each (structure, spins) class, -1: the class has no slots
  int row[16];
};

// The 28 densities of a grid point from the class sums (the combinations of
// density_accumulate), weights stripped; those with same-spin sums and the others
// on threads of their own, so that a thread's loads fit its registers and are in
// flight together (one point: 14 -> 8 us).
__global__ void __launch_bounds__(64, 2) k_sep_combine(SepArgs A, SepAcc B) {
  const int G = A.nz * A.nr, g = blockIdx.x * blockDim.x + threadIdx.x;
  const int w = A.act[blockIdx.y];
  if (g >= G || w == A.skip) return;
  const int sec = blockIdx.z & 1, nr = A.nr, nz = A.nz, r = g / nz, z = g - r * nz, W = 2 * nz;
  const double *acc = A.acc + (size_t)blockIdx.y * A.astride + z;
  auto get = [&](int cls, int kind, bool same, int t, int c) {
    // a class without slots reads row 0 and drops it: no branch, so that the loads
    // of all densities are in flight together
    const int b = B.row[cls];
    const double *p = acc + (size_t)(b < 0 ? 0 : b + sep_row0(kind, same, t, nr) + c * nr + r) * W;
    const double re = p[0], im = p[nz];
    return b < 0 ? cplx{0.0, 0.0} : cplx{re, im};
  };
  const double wc = A.wdcori[g];
  double *out = A.dens + (((size_t)w * 2 + sec) * 2 * NDENS) * G + g;
  cplx val[NDENS];         // stored at the end: a store would hold back the loads after it
  auto put = [&](int d, cplx v) { val[d] = v; };
  auto store = [&](int d) { out[(size_t)(2 * d) * G] = val[d].r * wc; out[(size_t)(2 * d + 1) * G] = val[d].i * wc; };
  auto store_all = [&](auto... d) { (store(d), ...); };
  const int m = 8 * sec;   // classes: rho uu ud du dd, then kappa
  auto P = [&](int t, int c, double s) {   // up-up + s down-down
    return get(m, 0, true, t, c) + s * get(m + 3, 0, true, t, c);
  };
  auto Q = [&](int t, int c, double s) {   // (up, down) + s (down, up)
    return get(m + 1, 0, false, t, c) + s * get(m + 2, 0, false, t, c);
  };
  if (blockIdx.z < 2) {
    put(D_RHO, P(0, 0, 1.0));
    put(D_SZ, P(0, 0, -1.0));
    put(D_JP, 0.5 * P(0, 1, 1.0));
    put(D_TJPZ, 0.5 * P(0, 1, -1.0));
    const cplx p33 = P(3, 0, 1.0), m33 = P(3, 0, -1.0);
    put(D_TAU, P(0, 2, 1.0) + p33);
    put(D_TZ, P(0, 2, -1.0) + m33);
    put(D_JR, 0.5 * mul_i(P(0, 3, 1.0)));
    put(D_TJRZ, 0.5 * mul_i(P(0, 3, -1.0)));
    put(D_JZ, 0.5 * mul_i(P(1, 0, 1.0) - P(2, 0, 1.0)));
    const cplx m03 = P(1, 0, -1.0), m30 = P(2, 0, -1.0);
    put(D_TJZZ, 0.5 * mul_i(m03 - m30));
    put(D_GS, m03 + m30 + Q(0, 2, 1.0));
    put(D_FR, 0.5 * (P(1, 1, -1.0) + P(2, 1, -1.0)) + Q(0, 3, 1.0));
    put(D_FP, mul_i(0.5 * (P(1, 2, -1.0) - P(2, 2, -1.0)) + Q(0, 4, 1.0)));
    put(D_FZ, m33 + 0.5 * (Q(1, 1, 1.0) + Q(2, 1, 1.0)));
    store_all(D_RHO, D_SZ, D_JP, D_TJPZ, D_TAU, D_TZ, D_JR, D_TJRZ, D_JZ, D_TJZZ, D_GS, D_FR, D_FP, D_FZ);
  } else {
    put(D_SR, Q(0, 0, 1.0));
    put(D_SP, mul_i(Q(0, 0, -1.0)));
    put(D_TJPR, 0.5 * Q(0, 1, 1.0));
    put(D_TJPP, 0.5 * mul_i(Q(0, 1, -1.0)));
    // f1 f1 + f2 f2 = (F_r row) + e (F_phi row)
    put(D_TR, Q(0, 3, 1.0) + Q(0, 4, -1.0) + Q(3, 0, 1.0));
    put(D_TP, mul_i(Q(0, 3, -1.0) + Q(0, 4, 1.0) + Q(3, 0, -1.0)));
    put(D_TJRR, 0.5 * mul_i(Q(0, 5, 1.0)));
    put(D_TJRP, -0.5 * Q(0, 5, -1.0));
    put(D_TJZR, 0.5 * mul_i(Q(1, 0, 1.0) - Q(2, 0, 1.0)));
    put(D_TJZP, -0.5 * (Q(1, 0, -1.0) - Q(2, 0, -1.0)));
    const cplx kuu = get(m + 4, 1, true, 0, 0), kud = get(m + 5, 1, false, 0, 0), kdu = get(m + 6, 1, false, 0, 0),
               kdd = get(m + 7, 1, true, 0, 0);
    put(D_RB, 2.0 * (kud - kdu));
    put(D_SBZ, 2.0 * (kud + kdu));
    put(D_SBR, 2.0 * (kdd - kuu));
    put(D_SBP, -2.0 * mul_i(kuu + kdd));
    store_all(D_SR, D_SP, D_TJPR, D_TJPP, D_TR, D_TP, D_TJRR, D_TJRP, D_TJZR, D_TJZP, D_RB, D_SBZ, D_SBR, D_SBP);
  }
}

// ---- projection: radial contraction ----------------------------------------------
constexpr int SEP_PRUN = 4;   // jobs of a run (k_sep_proj)
struct SepPJob {
  int64_t rp;               // offset of the class's table at this axial pair: [k][ld]
  uint64_t fields;          // the terms' field components, seven bits each
  int ld, n, s0, nst;       // slots padded to 16, slots, first slot, slot tiles (1..4; 0: an empty job)
  int nc, sec;              // terms, sector
  int yoff, yld;            // Y of the class's first slot at this axial pair; stride between slots
};
static_assert(9 * 7 <= 64 && NFLD <= 128, "a job's nine field components fit 64 bits");

// One job with RT slot tiles (the loop as in sep_dens_job); the loads of U steps
// are in flight during the products of the U before.
template <int CT, int RT, int U>
__device__ inline void sep_proj_job(const SepArgs &A, const SepPJob &J, int w, int y) {
  const int lane = threadIdx.x, mi = lane & 15, mk = lane >> 4;
  const int nz = A.nz, nr = A.nr, W = 2 * A.nzp, nr4 = (nr + 3) & ~3;
  const long G = (long)nz * nr;
  v4d C[RT][CT];
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int c = 0; c < CT; ++c) C[q][c] = v4d{0, 0, 0, 0};
  const __amdgpu_buffer_rsrc_t F = rsrc64(A.flds + (((size_t)w * 2 + J.sec) * 2 * NFLD) * G, (int)(2 * NFLD * G));
  // columns past the last axial point repeat it: finite, and multiplied by the
  // axial tables' zeros later
  int col[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int k = min(((int)blockIdx.y * CT + c) * 16 + mi, W - 1);
    col[c] = k < A.nzp ? min(k, nz - 1) : (int)G + min(k - A.nzp, nz - 1);
  }
  // step k: points r0 .. r0 + 3 of a term (table rows are zero past the last
  // point, whose fields the lanes past it repeat)
  const int rl = mk * nz, rt = (min(nr4 - 4 + mk, nr - 1) - (nr4 - 4)) * nz;
  const int nk = J.nc * (nr4 >> 2);
  uint64_t fields = J.fields;
  const int step = 4 * J.ld, G2 = 2 * (int)G;
  const __amdgpu_buffer_rsrc_t R = rsrc64(A.tab + J.rp + J.s0, nk * step - J.s0);
  const int ra = mk * J.ld + mi;
  int r0 = 0, fo = (int)(fields & 127) * G2, p = 0;   // point, offsets in the fields and the table
  double an[U][RT], bn[U][CT];
  int kl = 0;               // the step the next load takes; after the last one the last again
  auto load = [&] {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = r0 + 4 < nr4 ? rl : rt;
#pragma unroll
      for (int k = 0; k < CT; ++k) bn[u][k] = load64(F, col[k] + q, fo);
#pragma unroll
      for (int k = 0; k < RT; ++k) an[u][k] = load64(R, ra + 16 * k, p);
      const bool more = ++kl < nk, next = r0 + 4 == nr4;
      fields = more && next ? fields >> 7 : fields;
      fo = !more ? fo : (next ? (int)(fields & 127) * G2 : fo + 4 * nz);
      r0 = !more ? r0 : (next ? 0 : r0 + 4);
      p += more ? step : 0;
    }
  };
  load();
  for (int k = 0; k < nk; k += U) {
    double a[U][RT], b[U][CT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int q = 0; q < RT; ++q) a[u][q] = an[u][q];
#pragma unroll
      for (int i = 0; i < CT; ++i) b[u][i] = bn[u][i];
    }
    load();
    loads_first();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u > 0 && k + u >= nk) break;
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int i = 0; i < CT; ++i) C[q][i] = mfma64(a[u][q], b[u][i], C[q][i]);
    }
  }
  double *out = A.zy + (size_t)y * A.ystride + J.yoff;
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k = ((int)blockIdx.y * CT + i) * 16 + mi, s = J.s0 + 16 * q + 4 * v + mk;
        if (k < W && s < J.n) out[(size_t)s * J.yld + k] = C[q][i][v];
      }
}

// Y[p][(ri, z)] = sum_{c, r} R'_c[r][p] F_c(r, z) on v_mfma_f64_16x16x4: up to RT
// tiles of 16 slots by CT tiles of 16 (ri, z) per wave, four radial points per
// step.  The fields are read where k_fields put them.  With many points (RT = 4)
// the products of two steps hide the loads of the next two (N_sh = 16, 128 points
// 2.01 ms, 2.09 with one; 1.10 at the peak matrix rate).  With few, a wave's
// chain of steps (some 90) is what takes the time: one slot tile per wave, four
// steps ahead, and where that leaves the device unfilled one column tile, eight
// ahead (one point, N_sh = 8: 46 -> 21 us; N_sh = 16: 50 -> 39 us).
template <int CT, int RT>
__global__ void __launch_bounds__(64, RT > 1 ? 2 : 3) k_sep_proj(SepArgs A, const SepPJob *__restrict__ jobs, int njob) {
  int y;
  const SepPJob J = jobs[sep_job(njob, SEP_PRUN, A.na, y)];
  const int w = A.act[y];
  if (w == A.skip) return;
  if (RT == 1) {
    if (J.nst) sep_proj_job<CT, 1, CT == 1 ? 8 : 4>(A, J, w, y);
    return;
  }
  switch (J.nst) {
    case 1: sep_proj_job<CT, 1, 2>(A, J, w, y); break;
    case 2: sep_proj_job<CT, 2, 2>(A, J, w, y); break;
    case 3: sep_proj_job<CT, 3, 2>(A, J, w, y); break;
    case 4: sep_proj_job<CT, 4, 2>(A, J, w, y); break;
    default: break;
  }
}

// ---- projection: axial expansion ----------------------------------------------------
// h(a, b) = 2 sum_t sum_z Y_t[p](z) c_t1(z, a) c_t2(z, b) over the slot's elements:
// the transpose of k_sep_z's product, [8 frequencies x (re, im)] x [(t, z)] by
// [(t, z)] x elements, 16 elements per tile, up to SEP_EN tiles at a time.  A
// lane holds two neighbouring axial points (16-byte loads, two matrix steps).
// Up to 8 points: one wave per slot, the five axial products of an element and z
// formed in registers.
constexpr int SEP_EN = 2;
template <bool MEAN>
__device__ inline void sep_expand_slot(const SepArgs &A, const SepSlot S, const int4 *__restrict__ elems) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int NT = MEAN ? 5 : 1, NX = MEAN ? 3 : 1;
  const int lane = threadIdx.x & 63, mi = lane & 15, mk = lane >> 4;
  const int nzp = A.nzp;
  // a row of a point past the last repeats it: finite, not stored
  const double *__restrict__ Y =
      A.zy + (size_t)min(mi >> 1, A.na - 1) * A.ystride + S.zoff + (size_t)(mi & 1) * nzp + 2 * mk;
  double *out[4];          // where this lane stores (row 4 v + mk of the product), null: nowhere
  const int out_slot = S.mat == 0 ? 0 : (S.mat == 1 ? 1 : (S.mat == 2 ? 3 : 2));
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int yo = 2 * v + (mk >> 1), w = A.act[min(yo, A.na - 1)];
    out[v] = yo < A.na && w != A.skip ? A.hsp + ((size_t)w * 8 + 2 * out_slot + (mk & 1)) * A.nxy : nullptr;
  }
  const double *__restrict__ fz = A.fz + 2 * mk;
  const size_t xs = (size_t)A.dqp * nzp;
  const int4 *__restrict__ el = elems + S.first;
  for (int e0 = 0; e0 < S.count; e0 += 16 * SEP_EN) {
    const double *fa[SEP_EN], *fb[SEP_EN];
    int off[SEP_EN];
#pragma unroll
    for (int k = 0; k < SEP_EN; ++k) {
      const int4 r = el[min(e0 + 16 * k + mi, S.count - 1)];
      off[k] = r.x; fa[k] = fz + (size_t)r.y * nzp; fb[k] = fz + (size_t)r.z * nzp;
    }
    const bool two = SEP_EN > 1 && e0 + 16 < S.count;     // the second tile has elements
    v4d C[SEP_EN];
#pragma unroll
    for (int k = 0; k < SEP_EN; ++k) C[k] = v4d{0, 0, 0, 0};
    v2d yn[NT], an[SEP_EN][NX], bn[SEP_EN][NX];
    auto load = [&](int zb) {
#pragma unroll
      for (int t = 0; t < NT; ++t) yn[t] = *(const v2d *)(Y + (size_t)(2 * t) * nzp + zb);
#pragma unroll
      for (int k = 0; k < SEP_EN; ++k)
#pragma unroll
        for (int x = 0; x < NX; ++x) {
          an[k][x] = *(const v2d *)(fa[k] + x * xs + zb);
          bn[k][x] = *(const v2d *)(fb[k] + x * xs + zb);
        }
    };
    load(0);
    for (int zb = 0; zb < nzp; zb += 8) {
      v2d yv[NT], X[SEP_EN][NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) yv[t] = yn[t];
#pragma unroll
      for (int k = 0; k < SEP_EN; ++k)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          X[k][0][u] = an[k][0][u] * bn[k][0][u];
          if constexpr (MEAN) {
            X[k][1][u] = an[k][0][u] * bn[k][1][u];
            X[k][2][u] = an[k][1][u] * bn[k][0][u];
            X[k][3][u] = an[k][1][u] * bn[k][1][u];
            X[k][4][u] = __builtin_fma(an[k][0][u], bn[k][2][u], an[k][2][u] * bn[k][0][u]);
          }
        }
      load(min(zb + 8, nzp - 8));
      loads_first();
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t) C[0] = mfma64(yv[t][u], X[0][t][u], C[0]);
      if (two)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int t = 0; t < NT; ++t) C[SEP_EN - 1] = mfma64(yv[t][u], X[SEP_EN - 1][t][u], C[SEP_EN - 1]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (out[v])
#pragma unroll
        for (int k = 0; k < SEP_EN; ++k)
          if (e0 + 16 * k + mi < S.count) out[v][off[k]] = 2.0 * C[k][v];
  }
}

__global__ void __launch_bounds__(256) k_sep_expand(SepArgs A, const SepSlot *__restrict__ slots,
                                                    const int4 *__restrict__ elems) {
  const SepSlot S = slots[__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)))];
  if (S.count == 0) return;
  if ((S.mat & 1) == 0) sep_expand_slot<true>(A, S, elems);
  else sep_expand_slot<false>(A, S, elems);
}

// The same for more than 8 points: the NW waves of a workgroup take the same slot for
// 8 frequencies each, the axial products of up to SEP_EW element tiles and 8 axial
// points formed once for all of them and kept in LDS in the layout of the
// operand, the next chunk's loads in flight during the products of this one.
// With a wave per slot for 16 frequencies, the products in registers, one wave
// filled a SIMD's registers and the functions' loads were repeated for every 16
// points: N_sh = 16, 128 points 2.25 ms, here 1.71 ms (0.40 ms at the peak matrix
// rate; 4.6 GB read and 2.3 written, 2.7 times what h holds: a slot's elements
// lie in lines it shares with other slots).
constexpr int SEP_EW = 4;
template <int NW, bool MEAN>
__device__ inline void sep_expand_wide(const SepArgs &A, const SepSlot S, const int4 *__restrict__ elems,
                                       double (*__restrict__ buf)[5 * 2 * SEP_EW * 64]) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int NT = MEAN ? 5 : 1, NX = MEAN ? 3 : 1, NP = SEP_EW / NW;   // element and pair of z per thread
  const int lane = threadIdx.x & 63, mi = lane & 15, mk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), y0 = ((int)blockIdx.y * NW + wv) * 8;
  const bool on = y0 < A.na;               // waves past the last point wait with the others
  const int nzp = A.nzp;
  // a row of a point past the last repeats it: finite, not stored
  const double *__restrict__ Y =
      A.zy + (size_t)min(y0 + (mi >> 1), A.na - 1) * A.ystride + S.zoff + (size_t)(mi & 1) * nzp + 2 * mk;
  const int out_slot = S.mat == 0 ? 0 : (S.mat == 1 ? 1 : (S.mat == 2 ? 3 : 2));
  const size_t xs = (size_t)A.dqp * nzp;
  const int4 *__restrict__ el = elems + S.first;
  const int q = threadIdx.x & 3;
  for (int e0 = 0; e0 < S.count; e0 += 16 * SEP_EW) {
    const int nk = min(SEP_EW, (S.count - e0 + 15) >> 4);
    int fa[NP], fb[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int4 r = el[min(e0 + ((int)threadIdx.x >> 2) + 16 * NW * i, S.count - 1)];
      fa[i] = r.y * nzp + 2 * q; fb[i] = r.z * nzp + 2 * q;
    }
    v4d C[SEP_EW];
#pragma unroll
    for (int k = 0; k < SEP_EW; ++k) C[k] = v4d{0, 0, 0, 0};
    v2d yn[NT], an[NP][NX], bn[NP][NX];
    auto load = [&](int zb) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int x = 0; x < NX; ++x) {
          an[i][x] = *(const v2d *)(A.fz + x * xs + zb + fa[i]);
          bn[i][x] = *(const v2d *)(A.fz + x * xs + zb + fb[i]);
        }
#pragma unroll
      for (int t = 0; t < NT; ++t) yn[t] = *(const v2d *)(Y + (size_t)(2 * t) * nzp + zb);
    };
    // value (t, u = z % 2, tile k, mk = z / 2, mi) at ((t 2 + u) SEP_EW + k) 64 + lane
    auto form = [&](double *d) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int e = ((int)threadIdx.x >> 2) + 16 * NW * i;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          double *p = d + (u * SEP_EW + (e >> 4)) * 64 + q * 16 + (e & 15);
          p[0] = an[i][0][u] * bn[i][0][u];
          if constexpr (MEAN) {
            p[1 * 2 * SEP_EW * 64] = an[i][0][u] * bn[i][1][u];
            p[2 * 2 * SEP_EW * 64] = an[i][1][u] * bn[i][0][u];
            p[3 * 2 * SEP_EW * 64] = an[i][1][u] * bn[i][1][u];
            p[4 * 2 * SEP_EW * 64] = __builtin_fma(an[i][0][u], bn[i][2][u], an[i][2][u] * bn[i][0][u]);
          }
        }
      }
    };
    load(0);
    form(buf[0]);
    __syncthreads();
    int cur = 0;
    for (int zb = 0; zb < nzp; zb += 8) {
      v2d yv[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) yv[t] = yn[t];
      load(min(zb + 8, nzp - 8));
      loads_first();
      const double *d = buf[cur] + lane;
      if (on)
#pragma unroll
        for (int k = 0; k < SEP_EW; ++k)
          if (k < nk)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int t = 0; t < NT; ++t) C[k] = mfma64(yv[t][u], d[((t * 2 + u) * SEP_EW + k) * 64], C[k]);
      cur ^= 1;
      if (zb + 8 < nzp) form(buf[cur]);
      __syncthreads();
    }
    if (on) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int yo = y0 + 2 * v + (mk >> 1), w = A.act[min(yo, A.na - 1)];
        if (yo < A.na && w != A.skip) {
          double *out = A.hsp + ((size_t)w * 8 + 2 * out_slot + (mk & 1)) * A.nxy;
#pragma unroll
          for (int k = 0; k < SEP_EW; ++k)
            if (e0 + 16 * k + mi < S.count) out[el[e0 + 16 * k + mi].x] = 2.0 * C[k][v];
        }
      }
    }
  }
}

// One slot per workgroup, in the order of k_sep_expand's workgroups of four.
template <int NW>
__global__ void __launch_bounds__(64 * NW, NW == 4 ? 3 : 2) k_sep_expand_wide(SepArgs A, const SepSlot *__restrict__ slots,
                                                             const int4 *__restrict__ elems) {
  __shared__ double buf[2][5 * 2 * SEP_EW * 64];
  const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
  const SepSlot S = slots[((i >> 2) * 8 + x) * 4 + (i & 3)];
  if (S.count == 0) return;
  if ((S.mat & 1) == 0) sep_expand_wide<NW, true>(A, S, elems, buf);
  else sep_expand_wide<NW, false>(A, S, elems, buf);
}
