// pnFAM iteration engine for MI355X (gfx950): kernels + C ABI (include/pnfam_gpu.h).
//
// Per-frequency state lives in HBM as frequency-major arrays:
//   vin/vout [w][4][nxy]  mixed / new amplitudes  (ReX, ReY, ImX, ImY) -- the
//                         Broyden vector layout of pnfam_broyden.f90:50-53
//   rsp      [w][8][nxy]  drho_sp quadrants re/im (m11, m12, m21, m22)
//   hsp      [w][8][nxy]  dH_sp quadrants re/im
//   hqp      [w][4][nxy]  dH_qp (H20 re, H02 re, H20 im, H02 im)
//   dens     [w][2][56][nghl]   local densities of the two sectors
//   flds     [w][2][208][nghl]  mean fields mf(z,z',sa,sb) and pairing fields
// Converged frequencies leave the active list and are skipped by every launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <map>
#include <chrono>
#include <cstdlib>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <numeric>
#include <set>
#include <string>
#include <vector>

#include <rocblas/rocblas.h>

#include "../../include/pnfam_gpu.h"
#include "plan.hpp"

using namespace pnfam;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                                          \
  do {                                                                                         \
    hipError_t e_ = (expr);                                                                    \
    if (e_ != hipSuccess)                                                                      \
      return fail(PNFAM_GPU_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));       \
  } while (0)

constexpr int NDENS = 28;          // complex local densities per sector
constexpr int NFLD = 104;          // complex fields per sector: 100 mf(z,z',sa,sb) + 4 pairing
constexpr double PI = 3.14159265358979323846;

// density indices (order of the density_set, pnfam_type_densityset.f90:14-33)
enum { D_RHO, D_TAU, D_TJRR, D_TJPR, D_TJZR, D_TJRP, D_TJPP, D_TJZP, D_TJRZ, D_TJPZ, D_TJZZ,
       D_SR, D_SP, D_SZ, D_TR, D_TP, D_TZ, D_JR, D_JP, D_JZ, D_FR, D_FP, D_FZ, D_GS,
       D_RB, D_SBR, D_SBP, D_SBZ };

__host__ __device__ constexpr int mf_index(int z, int zp, int sa, int sb) {  // sa/sb: 0 up, 1 down
  return ((z * 5 + zp) * 2 + sa) * 2 + sb;
}

typedef double v4d __attribute__((ext_vector_type(4)));

// v_mfma_f64_16x16x4: lane i + 16k supplies A[i][k] and B[k][i]; the result
// D[i][j] is held by lane j + 16 (i % 4) in register i / 4.
__device__ inline v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

struct DevPtr {
  void *p = nullptr;
  size_t bytes = 0;
  ~DevPtr() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr; bytes = 0;
  }
  int alloc(size_t n) {
    if (p && bytes >= n) return 0;
    release();
    if (n == 0) n = 8;
    if (hipMalloc(&p, n) != hipSuccess) {
      (void)hipGetLastError();   // reported here, not by the next check of a launch as well
      p = nullptr;
      return fail(PNFAM_GPU_ENOMEM, "hipMalloc of " + std::to_string(n) + " bytes failed");
    }
    bytes = n;
    return 0;
  }
  template <class T> T *as() const { return static_cast<T *>(p); }
};

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

__global__ void k_fill(double *__restrict__ p, size_t n, double v) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

// zero slots [s0, s0+ns) of every active frequency's [w][nslot][nxy] array
__global__ void k_zero_slots(double *__restrict__ base, const int *__restrict__ act, int nslot, int s0, int ns,
                             long nxy, int skip) {
  int w = act[blockIdx.y];
  if (w == skip) return;
  double *p = base + ((size_t)w * nslot + s0) * nxy;
  size_t n = (size_t)ns * nxy;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0.0;
}

// Block triple products out[i,j] = sum_terms s op(A) op(B_w) op(C); one workgroup per
// (output block, frequency).  T = s op(A) op(B) is staged in LDS.
__global__ void __launch_bounds__(256) k_triprod(const Group *__restrict__ groups, const Term *__restrict__ terms,
                                                 const double *__restrict__ m0, const double *__restrict__ m1,
                                                 const double *__restrict__ m2, const double *__restrict__ m3,
                                                 const double *__restrict__ bbase, long bstride, int bslots,
                                                 double *__restrict__ obase, long ostride, int oslots,
                                                 const int *__restrict__ act, long nxy) {
  extern __shared__ double lds[];
  const Group g = groups[blockIdx.x];
  const int w = act ? act[blockIdx.y] : (int)blockIdx.y;
  const double *B = bbase + (size_t)w * bstride;
  double *O = obase + (size_t)w * ostride + (size_t)g.out_slot * nxy + g.out_off;
  const double *mats[4] = {m0, m1, m2, m3};
  const int n = g.nrow * g.ncol;
  for (int t = 0; t < g.count; ++t) {
    const Term tm = terms[g.first + t];
    const double *A = (tm.a_id == 0 ? m0 : tm.a_id == 1 ? m1 : tm.a_id == 2 ? m2 : m3) + tm.a_off;
    const double *Bb = B + (size_t)tm.b_slot * nxy + tm.b_off;
    const double *C = (tm.c_id == 0 ? m0 : tm.c_id == 1 ? m1 : tm.c_id == 2 ? m2 : m3) + tm.c_off;
    const int nda = tm.nda, ndc = tm.ndc;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
      const int i = e % nda, j = e / nda;
      double acc = 0.0;
      for (int k = 0; k < nda; ++k) {
        const double a = tm.ta ? A[k + i * nda] : A[i + k * nda];
        const double b = tm.tb ? Bb[j + k * tm.ldb] : Bb[k + j * tm.ldb];
        acc += a * b;
      }
      lds[e] = tm.s * acc;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
      const int i = e % nda, j = e / nda;
      double acc = 0.0;
      for (int l = 0; l < ndc; ++l) {
        const double c = tm.tc ? C[j + l * ndc] : C[l + j * ndc];
        acc += lds[i + l * nda] * c;
      }
      O[e] = (t == 0) ? acc : O[e] + acc;
    }
    __syncthreads();
  }
}

// Keeps the loads of the next step above the products of the current one: nothing
// in the program orders the two, and the compiler otherwise sinks each load to
// its use in the next trip of the loop, where its latency is not hidden.
__device__ inline void loads_first() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Buffer of n doubles at a uniform p: loads with one address register (offsets of
// the lanes; soff: a uniform offset on top), zero past the end.
__device__ inline __amdgpu_buffer_rsrc_t rsrc64(const double *p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, 8 * n, 0x00020000);
}
__device__ inline double load64(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, 8 * off, 8 * soff, 0));
}

constexpr int TP_MAXCT = 8;    // column tiles of 16 per strip (block sizes up to 128)
constexpr int TP_MERGE_N = 8;  // at most this many points: one launch over all tile classes (bf16 triple products, projection)
constexpr int TP_SPLIT_N = 4;  // at most this many points: FP64 triple products in one launch, a strip's columns on four waves

// Resident matrices of the FP64 triple products: every block zero-padded to a
// pitch P of 32 k, as stored (cm) and transposed (rm), so that op(A) is read with
// its rows and op(C) with its columns along the lanes, aligned and unmasked.
struct Tp64 {
  const double *cm, *rm;
  long mstride;          // doubles per matrix
};

__global__ void k_tp_pack(const double *__restrict__ m, const int4 *__restrict__ blocks, double *__restrict__ cm,
                          double *__restrict__ rm) {
  const int4 b = blocks[blockIdx.y];    // FP64 offset, padded offset, d, P
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < b.w * b.w; e += gridDim.x * blockDim.x) {
    const int i = e % b.w, j = e / b.w;
    const bool in = i < b.z && j < b.z;
    cm[b.y + e] = in ? m[b.x + i + (size_t)j * b.z] : 0.0;
    rm[b.y + e] = in ? m[b.x + j + (size_t)i * b.z] : 0.0;
  }
}

// Block triple products on the matrix cores: the strips (16 rows) of an output
// block on the waves of a workgroup, per group and frequency.
//
// A strip's first product is formed transposed, T^T(j, i) = sum_k op(B)(k, j)
// op(A)(i, k): register v of tile c then holds T(i, 16 c + 4 v + lane / 16) for
// i = lane % 16, which is the A operand of the second product's step
// l = 16 c + 4 v, so T needs neither LDS nor a barrier.
// op(B) and op(C), which all strips read, go through LDS in chunks of 16 rows,
// the next chunk's loads in flight during the products of this one.  Read
// straight into the operand layout, a matrix whose rows are contiguous gives
// every lane a cache line of its own; the L1 then serves one lane a cycle, and
// that, not the matrix rate, bound the kernel (counters: 0.6 to 0.7 L1 accesses
// per cycle and CU, 25 to 28 per load, matrix cores busy 29 to 37 % of the time;
// now 0.4 to 0.5, 20 to 26 and 63 to 71 %).
// op(A), with its rows along the lanes, is read from the packed copies.  Buffer
// loads keep an address in one register, which lets three waves of up to 96
// columns (four of up to 64) share a SIMD.
// N_sh = 16, both term sets of a stage at 128 points: 1.55 ms (0.87 ms at the
// peak matrix rate), 2.4 ms with the operands read straight from memory and the
// term sets in launches of their own.
// NCT: 16-column tiles of the launch's groups; NW: waves.
template <int NCT, int NW>
__global__ void __launch_bounds__(64 * NW, NCT <= 4 ? 4 : (NCT <= 6 || (NCT == 7 && NW == 4) ? 3 : 2))
    k_triprod_mfma(const Group *__restrict__ groups, const Term *__restrict__ terms, Tp64 M,
                   const double *__restrict__ bbase, long bstride, double *__restrict__ obase, long ostride,
                   const int *__restrict__ act, long nxy, int skip) {
  constexpr int PJ = 16 * NCT + 1;   // chunk row pitch: odd, so that neither a column written nor four rows read collide much
  __shared__ double buf[2][16 * PJ];
  const Group g = groups[blockIdx.x];
  const int w = act ? act[blockIdx.y] : (int)blockIdx.y;
  if (w == skip) return;
  const int tid = threadIdx.x, lane = tid & 63, mi = lane & 15, mk = lane >> 4;
  constexpr int nth = 64 * NW;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = 16 * ((int)blockIdx.z * NW + wv);
  const bool on = i0 < g.nrow;               // waves past the block load and wait with the others
  const double *B = bbase + (size_t)w * bstride;
  // A chunk is 16 rows by 16 NCT columns, in runs of 16 values: thread group u0
  // (16 threads) takes the runs u0 + 4 NW i.  All addresses are one register plus
  // what is uniform or a constant.
  constexpr int NG = 4 * NW, NL = 16 * NCT / NG;
  const int l16 = tid & 15, u0 = tid >> 4;
  v4d acc[NCT];
#pragma unroll
  for (int c = 0; c < NCT; ++c) acc[c] = v4d{0, 0, 0, 0};
  for (int t = 0; t < g.count; ++t) {
    const Term tm = terms[g.first + t];
    const int nda = tm.nda, ndc = tm.ndc, Pa = (nda + 31) & ~31, Pc = (ndc + 31) & ~31;
    const __amdgpu_buffer_rsrc_t Ap =
        rsrc64((tm.ta ? M.rm : M.cm) + tm.a_id * M.mstride + tm.pad0 + (on ? i0 : 0), Pa * Pa - (on ? i0 : 0));
    const __amdgpu_buffer_rsrc_t Cp = rsrc64((tm.tc ? M.cm : M.rm) + tm.c_id * M.mstride + tm.pad1, Pc * Pc);
    // Rows and columns of op(B) past the block: zeros past its end (the buffer's
    // bound), else other values of the same block; the padding of A and C takes
    // both out.
    const __amdgpu_buffer_rsrc_t Bb = rsrc64(B + (size_t)tm.b_slot * nxy + tm.b_off, nda * ndc);
    // stored with its columns contiguous (tb): run u is row u % 16, columns 16 (u / 16)
    // to + 15; else column u, 16 rows
    const int ldb = tm.ldb, bk = tm.tb ? ldb : 1, bc = tm.tb ? 16 : 16 * ldb;
    const int bd = tm.tb ? u0 * PJ + l16 : l16 * PJ + u0, br = tm.tb ? PJ : 1;
    double st[NL];
    auto bload = [&](int k0) {
#pragma unroll
      for (int i = 0; i < NL; ++i)
        st[i] = load64(Bb, u0 * ldb + l16 + k0 * bk + NG * i % 16 * ldb + NG * i / 16 * bc, 0);
    };
    auto bstore = [&](double *d) {
#pragma unroll
      for (int i = 0; i < NL; ++i) d[bd + NG * i % 16 * br + NG * i / 16 * 16] = st[i];
    };
    auto cload = [&](int l0) {
#pragma unroll
      for (int i = 0; i < NL; ++i) st[i] = load64(Cp, u0 * Pc + l16, (l0 + NG * i % 16) * Pc + NG * i / 16 * 16);
    };
    auto cstore = [&](double *d) {
#pragma unroll
      for (int i = 0; i < NL; ++i) d[u0 * PJ + l16 + NG * i % 16 * PJ + NG * i / 16 * 16] = st[i];
    };
    v4d T[NCT];
#pragma unroll
    for (int c = 0; c < NCT; ++c) T[c] = v4d{0, 0, 0, 0};
    double an[4];
    auto aload = [&](int k0) {
#pragma unroll
      for (int s = 0; s < 4; ++s) an[s] = load64(Ap, mk * Pa + mi, (k0 + 4 * s) * Pa);
    };
    bload(0);
    aload(0);
    __syncthreads();                         // the previous term's last chunk has been read
    bstore(buf[0]);
    __syncthreads();
    int cur = 0, k0 = 0;
    for (; k0 + 16 < nda; k0 += 16) {
      double a[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) a[s] = an[s];
      bload(k0 + 16);
      aload(k0 + 16);
      loads_first();
      const double *d = buf[cur];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int c = 0; c < NCT; ++c) T[c] = mfma64(d[(4 * s + mk) * PJ + 16 * c + mi], a[s], T[c]);
        if (NCT > 3) __builtin_amdgcn_sched_barrier(0);
      }
      cur ^= 1;
      bstore(buf[cur]);
      __syncthreads();
    }
    cload(0);
    loads_first();
    {
      const double *d = buf[cur];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s > 0 && k0 + 4 * s >= nda) break;
#pragma unroll
        for (int c = 0; c < NCT; ++c) T[c] = mfma64(d[(4 * s + mk) * PJ + 16 * c + mi], an[s], T[c]);
        if (NCT > 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    cur ^= 1;
    cstore(buf[cur]);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      if (c + 1 < NCT) cload(16 * (c + 1));
      loads_first();
      const double *d = buf[cur];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (c == NCT - 1 && v > 0 && 16 * c + 4 * v >= ndc) break;   // only the last tile may end early
        const double a = tm.s * T[c][v];
#pragma unroll
        for (int q = 0; q < NCT; ++q)
          acc[q] = mfma64(a, d[(4 * v + mk) * PJ + 16 * q + mi], acc[q]);
        if (NCT > 3) __builtin_amdgcn_sched_barrier(0);
      }
      cur ^= 1;
      if (c + 1 < NCT) {
        cstore(buf[cur]);
        __syncthreads();
      }
    }
  }
  if (!on) return;
  double *O = obase + (size_t)w * ostride + (size_t)g.out_slot * nxy + g.out_off;
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int j = c * 16 + mi;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = i0 + 4 * v + mk;
      if (i < g.nrow && j < g.ncol) O[i + (size_t)j * g.nrow] = acc[c][v];
    }
  }
}

// The same for the fewest points: one strip per workgroup, its column tiles dealt
// to four waves (tile c to wave c % 4), of T for up to two terms, then of the
// output, so that the chains run side by side and every sum keeps its order (and
// its bits).  A wave turns its tiles of op(B) over in an LDS patch of its own;
// T passes between the waves in the layout in which they read it.
// N_sh = 16, one point: 50 us a stage, 141 us with the terms one after another
// on one wave and re and im in launches of their own.
template <int NCT>
__global__ void __launch_bounds__(256, 3) k_triprod_split(const Group *__restrict__ groups,
                                                          const Term *__restrict__ terms, Tp64 M,
                                                          const double *__restrict__ bbase, long bstride,
                                                          double *__restrict__ obase, long ostride,
                                                          const int *__restrict__ act, long nxy, int skip) {
  constexpr int NT = (NCT + 3) / 4, TS = 2;      // tiles per wave; terms per pass
  __shared__ double tl[TS * 4 * NT * 256];
  __shared__ double patch[4 * NT * 16 * 17];
  const Group g = groups[blockIdx.x];
  const int w = act ? act[blockIdx.y] : (int)blockIdx.y;
  const int lane = threadIdx.x & 63, mi = lane & 15, mk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int i0 = 16 * (int)blockIdx.z;
  if (w == skip || i0 >= g.nrow) return;          // uniform per workgroup
  const double *B = bbase + (size_t)w * bstride;
  double *d = patch + wave * NT * 16 * 17;
  v4d acc[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) acc[u] = v4d{0, 0, 0, 0};
  for (int t0 = 0; t0 < g.count; t0 += TS) {
    const int nt = min(TS, g.count - t0);
    const Term *tp = terms + g.first + t0;
    // loads of the next 16 k, across the ends of the terms
    Term tm = tp[0];
    __amdgpu_buffer_rsrc_t Ap, Bb, Cp;
    double an[4], bn[NT][4], cn[4][NT];
    auto open_ab = [&](int t) {
      tm = tp[t];
      const int Pa = (tm.nda + 31) & ~31;
      Ap = rsrc64((tm.ta ? M.rm : M.cm) + tm.a_id * M.mstride + tm.pad0 + i0, Pa * Pa - i0);
      // past the block: zeros or other values of it, as in k_triprod_mfma
      Bb = rsrc64(B + (size_t)tm.b_slot * nxy + tm.b_off, tm.nda * tm.ndc);
    };
    auto load_ab = [&](int k0) {
      const int Pa = (tm.nda + 31) & ~31, bk = tm.tb ? tm.ldb : 1, bj = tm.tb ? 1 : tm.ldb;
#pragma unroll
      for (int s = 0; s < 4; ++s) an[s] = load64(Ap, mk * Pa + mi, (k0 + 4 * s) * Pa);
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          bn[u][s] = load64(Bb, mk * tm.ldb + mi + 4 * s * tm.ldb + k0 * bk + 16 * (wave + 4 * u) * bj, 0);
    };
    auto open_c = [&](int t) {
      tm = tp[t];
      const int Pc = (tm.ndc + 31) & ~31;
      // columns past the block's padding read the next row: of output tiles that are not stored
      Cp = rsrc64((tm.tc ? M.cm : M.rm) + tm.c_id * M.mstride + tm.pad1, Pc * Pc);
    };
    auto load_c = [&](int l0) {
      const int Pc = (tm.ndc + 31) & ~31;
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int u = 0; u < NT; ++u) cn[v][u] = load64(Cp, mk * Pc + mi, (l0 + 4 * v) * Pc + 16 * (wave + 4 * u));
    };
    open_ab(0);
    load_ab(0);
    for (int t = 0; t < nt; ++t) {
      const int nda = tm.nda, dw = tm.tb ? mk * 17 + mi : mi * 17 + mk, ds = tm.tb ? 4 * 17 : 4;
      const double sc = tm.s;
      v4d T[NT];
#pragma unroll
      for (int u = 0; u < NT; ++u) T[u] = v4d{0, 0, 0, 0};
      for (int k0 = 0; k0 < nda; k0 += 16) {
        double a[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) a[s] = an[s];
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int s = 0; s < 4; ++s) d[u * 16 * 17 + dw + s * ds] = bn[u][s];
        int kn = k0 + 16;
        if (kn >= nda) {
          kn = 0;
          open_ab(min(t + 1, nt - 1));
        }
        load_ab(kn);
        loads_first();                            // also: the patch is written before other lanes' values are read
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (s > 0 && k0 + 4 * s >= nda) break;
#pragma unroll
          for (int u = 0; u < NT; ++u) T[u] = mfma64(d[(u * 16 + 4 * s + mk) * 17 + mi], a[s], T[u]);
        }
        loads_first();                            // read before it is written again
      }
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) tl[((t * 4 * NT + wave + 4 * u) * 4 + v) * 64 + lane] = sc * T[u][v];
    }
    open_c(0);
    load_c(0);
    loads_first();
    __syncthreads();
    for (int t = 0; t < nt; ++t) {
      const int ndc = tm.ndc;
      const double *T = tl + t * 4 * NT * 256 + lane;
      for (int l0 = 0; l0 < ndc; l0 += 16) {
        double cv[4][NT];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int u = 0; u < NT; ++u) cv[v][u] = cn[v][u];
        int ln = l0 + 16;
        if (ln >= ndc) {
          ln = 0;
          open_c(min(t + 1, nt - 1));
        }
        load_c(ln);
        loads_first();
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (v > 0 && l0 + 4 * v >= ndc) break;
          const double a = T[(l0 / 4 + v) * 64];
#pragma unroll
          for (int u = 0; u < NT; ++u) acc[u] = mfma64(a, cv[v][u], acc[u]);
        }
      }
    }
    __syncthreads();                              // T has been read
  }
  double *O = obase + (size_t)w * ostride + (size_t)g.out_slot * nxy + g.out_off;
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int j = 16 * (wave + 4 * u) + mi;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = i0 + 4 * v + mk;
      if (i < g.nrow && j < g.ncol) O[i + (size_t)j * g.nrow] = acc[u][v];
    }
  }
}

struct PairList {       // block pairs (row block, col block, element offset) of a block map
  const int4 *p;
  int n;
};

struct DensArgs {
  const double *wf, *wfdr, *wfdp, *wfdz, *wdcori;
  const int *isstart, *db, *nsu, *ns;
  const double *rsp;   // [w][8][nxy]
  long nxy;
  int nghl;
  PairList rho[2], kap[2];   // per sector
  int rho_slot[2], kap_slot[2];
  double *dens;        // [w][2][56][nghl]
  double *part;        // k_density_mfma split over block pairs: [split][active index][2][56][nghl]; null: dens
  const int *act;
  int skip = -1;       // an active-list entry whose workgroups return at once (graph replay's spare slot)
};

// Local densities (pnfam_hamiltonian_blas.f90:124-711): per grid point r and
// column b, T_x^s(r,b) = sum_{a in block, spin s} psi_x(r,a) rho(a,b) followed by
// the products with psi_y(r,b).  One lane per grid point; a workgroup loops over
// all block pairs, so every density is a deterministic per-thread sum.
__global__ void __launch_bounds__(64) k_density(DensArgs A) {
  const int r = blockIdx.x * 64 + threadIdx.x;
  const int w = A.act[blockIdx.y];
  if (w == A.skip) return;
  const int sec = blockIdx.z;
  const int G = A.nghl;
  const bool live = r < G;
  const int rr = live ? r : 0;
  double acc[2 * NDENS];
#pragma unroll
  for (int d = 0; d < 2 * NDENS; ++d) acc[d] = 0.0;
  const double *rho_re = A.rsp + ((size_t)w * 8 + 2 * A.rho_slot[sec]) * A.nxy;
  const double *rho_im = rho_re + A.nxy;
  const double *tab[4] = {A.wf, A.wfdr, A.wfdp, A.wfdz};
#define ACC(d, ri) acc[2 * (d) + (ri)]
  const PairList pl = A.rho[sec];
  for (int p = 0; p < pl.n; ++p) {
    const int4 pr = pl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy], nsu = A.nsu[ix];
    for (int bl = 0; bl < dy; ++bl) {
      const int b = ib0 + bl;
      double Tr[4][2], Ti[4][2];  // [x][spin of a: 0 up, 1 down]
#pragma unroll
      for (int x = 0; x < 4; ++x) { Tr[x][0] = Tr[x][1] = Ti[x][0] = Ti[x][1] = 0.0; }
      const double *cr = rho_re + off + (size_t)bl * dx;
      const double *ci = rho_im + off + (size_t)bl * dx;
      for (int al = 0; al < dx; ++al) {
        const int sp = al < nsu ? 0 : 1;
        const double vr = cr[al], vi = ci[al];
        const size_t o = (size_t)(ia + al) * G + rr;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const double psi = tab[x][o];
          Tr[x][sp] += psi * vr;
          Ti[x][sp] += psi * vi;
        }
      }
      const int s = A.ns[b];
      const int sd = s > 0 ? 0 : 1, so = 1 - sd;
      const size_t ob = (size_t)b * G + rr;
      const double y[4] = {A.wf[ob], A.wfdr[ob], A.wfdp[ob], A.wfdz[ob]};
      // P[x][y] = T_x(spin of b) psi_y(b); Q[x][y] = T_x(opposite spin) psi_y(b)
      double Pr[4][4], Pi[4][4], Qr[4][4], Qi[4][4];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int yy = 0; yy < 4; ++yy) {
          Pr[x][yy] = Tr[x][sd] * y[yy]; Pi[x][yy] = Ti[x][sd] * y[yy];
          Qr[x][yy] = Tr[x][so] * y[yy]; Qi[x][yy] = Ti[x][so] * y[yy];
        }
      double ar, ai;
      ACC(D_RHO, 0) += Pr[0][0]; ACC(D_RHO, 1) += Pi[0][0];
      ACC(D_SZ, 0) += s * Pr[0][0]; ACC(D_SZ, 1) += s * Pi[0][0];
      ar = 0.5 * (Pr[0][2] + Pr[2][0]); ai = 0.5 * (Pi[0][2] + Pi[2][0]);
      ACC(D_JP, 0) += ar; ACC(D_JP, 1) += ai;
      ACC(D_TJPZ, 0) += s * ar; ACC(D_TJPZ, 1) += s * ai;
      ar = Pr[1][1] + Pr[2][2] + Pr[3][3]; ai = Pi[1][1] + Pi[2][2] + Pi[3][3];
      ACC(D_TAU, 0) += ar; ACC(D_TAU, 1) += ai;
      ACC(D_TZ, 0) += s * ar; ACC(D_TZ, 1) += s * ai;
      ar = 0.5 * (Pr[0][1] - Pr[1][0]); ai = 0.5 * (Pi[0][1] - Pi[1][0]);   // j_r = i*aux
      ACC(D_JR, 0) -= ai; ACC(D_JR, 1) += ar;
      ACC(D_TJRZ, 0) -= s * ai; ACC(D_TJRZ, 1) += s * ar;
      ar = 0.5 * (Pr[0][3] - Pr[3][0]); ai = 0.5 * (Pi[0][3] - Pi[3][0]);
      ACC(D_JZ, 0) -= ai; ACC(D_JZ, 1) += ar;
      ACC(D_TJZZ, 0) -= s * ai; ACC(D_TJZZ, 1) += s * ar;
      ACC(D_GS, 0) += s * (Pr[0][3] + Pr[3][0]); ACC(D_GS, 1) += s * (Pi[0][3] + Pi[3][0]);
      ACC(D_FR, 0) += 0.5 * s * (Pr[1][3] + Pr[3][1]); ACC(D_FR, 1) += 0.5 * s * (Pi[1][3] + Pi[3][1]);
      ar = Pr[2][3] - Pr[3][2]; ai = Pi[2][3] - Pi[3][2];
      ACC(D_FP, 0) -= 0.5 * s * ai; ACC(D_FP, 1) += 0.5 * s * ar;
      ACC(D_FZ, 0) += s * Pr[3][3]; ACC(D_FZ, 1) += s * Pi[3][3];
      // spin-flip part; e = -s: +1 for (a up, b down), -1 for (a down, b up)
      const double e = -(double)s;
      ACC(D_SR, 0) += Qr[0][0]; ACC(D_SR, 1) += Qi[0][0];
      ACC(D_SP, 0) -= e * Qi[0][0]; ACC(D_SP, 1) += e * Qr[0][0];
      const double t2r = 0.5 * (Qr[2][0] + Qr[0][2]), t2i = 0.5 * (Qi[2][0] + Qi[0][2]);
      ACC(D_TJPR, 0) += t2r; ACC(D_TJPR, 1) += t2i;
      ACC(D_TJPP, 0) -= e * t2i; ACC(D_TJPP, 1) += e * t2r;
      ACC(D_GS, 0) += e * (Qr[0][2] - Qr[2][0]) + (Qr[0][1] + Qr[1][0]);
      ACC(D_GS, 1) += e * (Qi[0][2] - Qi[2][0]) + (Qi[0][1] + Qi[1][0]);
      const double tkr = Qr[1][1] + Qr[2][2] + Qr[3][3], tki = Qi[1][1] + Qi[2][2] + Qi[3][3];
      ACC(D_TR, 0) += tkr; ACC(D_TR, 1) += tki;
      ACC(D_TP, 0) -= e * tki; ACC(D_TP, 1) += e * tkr;
      const double jrr = 0.5 * (Qr[0][1] - Qr[1][0]), jri = 0.5 * (Qi[0][1] - Qi[1][0]);
      ACC(D_TJRR, 0) -= jri; ACC(D_TJRR, 1) += jrr;
      ACC(D_TJRP, 0) -= e * jrr; ACC(D_TJRP, 1) -= e * jri;
      const double jzr = 0.5 * (Qr[0][3] - Qr[3][0]), jzi = 0.5 * (Qi[0][3] - Qi[3][0]);
      ACC(D_TJZR, 0) -= jzi; ACC(D_TJZR, 1) += jzr;
      ACC(D_TJZP, 0) -= e * jzr; ACC(D_TJZP, 1) -= e * jzi;
      ar = Qr[1][1] + e * 0.5 * (Qr[1][2] - Qr[2][1]);
      ai = Qi[1][1] + e * 0.5 * (Qi[1][2] - Qi[2][1]);
      ACC(D_FR, 0) += ar; ACC(D_FR, 1) += ai;
      ar = e * Qr[2][2] + 0.5 * (Qr[2][1] - Qr[1][2]);
      ai = e * Qi[2][2] + 0.5 * (Qi[2][1] - Qi[1][2]);
      ACC(D_FP, 0) -= ai; ACC(D_FP, 1) += ar;
      ar = Qr[3][1] + Qr[1][3] + e * (Qr[3][2] - Qr[2][3]);
      ai = Qi[3][1] + Qi[1][3] + e * (Qi[3][2] - Qi[2][3]);
      ACC(D_FZ, 0) += 0.5 * ar; ACC(D_FZ, 1) += 0.5 * ai;
    }
  }
  // pairing densities from kappa (pnfam_hamiltonian_blas.f90:596-675)
  const double *kap_re = A.rsp + ((size_t)w * 8 + 2 * A.kap_slot[sec]) * A.nxy;
  const double *kap_im = kap_re + A.nxy;
  const PairList kl = A.kap[sec];
  for (int p = 0; p < kl.n; ++p) {
    const int4 pr = kl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy], nsu = A.nsu[ix];
    for (int bl = 0; bl < dy; ++bl) {
      const int b = ib0 + bl;
      double Tr[2] = {0.0, 0.0}, Ti[2] = {0.0, 0.0};
      const double *cr = kap_re + off + (size_t)bl * dx;
      const double *ci = kap_im + off + (size_t)bl * dx;
      for (int al = 0; al < dx; ++al) {
        const int sp = al < nsu ? 0 : 1;
        const double psi = A.wf[(size_t)(ia + al) * G + rr];
        Tr[sp] += psi * cr[al];
        Ti[sp] += psi * ci[al];
      }
      const int s = A.ns[b];
      const int sd = s > 0 ? 0 : 1, so = 1 - sd;
      const double wb = A.wf[(size_t)b * G + rr];
      double pr_ = 2.0 * Tr[so] * wb, pi_ = 2.0 * Ti[so] * wb;
      ACC(D_RB, 0) -= s * pr_; ACC(D_RB, 1) -= s * pi_;
      ACC(D_SBZ, 0) += pr_; ACC(D_SBZ, 1) += pi_;
      pr_ = 2.0 * Tr[sd] * wb; pi_ = 2.0 * Ti[sd] * wb;
      ACC(D_SBR, 0) += s < 0 ? pr_ : -pr_; ACC(D_SBR, 1) += s < 0 ? pi_ : -pi_;
      ACC(D_SBP, 0) += pi_; ACC(D_SBP, 1) -= pr_;
    }
  }
#undef ACC
  if (!live) return;
  const double wc = A.wdcori[r];
  double *out = A.dens + (((size_t)w * 2 + sec) * 2 * NDENS) * G + r;
#pragma unroll
  for (int d = 0; d < 2 * NDENS; ++d) out[(size_t)d * G] = acc[d] * wc;
}


// Accumulates the local-density contributions of one column b at one grid
// point from T_x^s (x = psi, d_r psi, d_phi psi, d_z psi; s = spin of a) and
// psi_y(b) (pnfam_hamiltonian_blas.f90:255-581).
// P[x][y] = sum over a of the spin of b, Q[x][y] = sum over a of the other
// spin, of psi_x(a) rho(a, b) psi_y(b), for columns b of spin s (+1/-1).
template <class R, class A>
__device__ inline void density_accumulate(A *acc, const R (&Pr)[4][4], const R (&Pi)[4][4],
                                          const R (&Qr)[4][4], const R (&Qi)[4][4], int s) {
#define ACC(d, ri) acc[2 * (d) + (ri)]
  const A half = A(0.5);
  A ar, ai;
  ACC(D_RHO, 0) += Pr[0][0]; ACC(D_RHO, 1) += Pi[0][0];
  ACC(D_SZ, 0) += s * Pr[0][0]; ACC(D_SZ, 1) += s * Pi[0][0];
  ar = half * (Pr[0][2] + Pr[2][0]); ai = half * (Pi[0][2] + Pi[2][0]);
  ACC(D_JP, 0) += ar; ACC(D_JP, 1) += ai;
  ACC(D_TJPZ, 0) += s * ar; ACC(D_TJPZ, 1) += s * ai;
  ar = Pr[1][1] + Pr[2][2] + Pr[3][3]; ai = Pi[1][1] + Pi[2][2] + Pi[3][3];
  ACC(D_TAU, 0) += ar; ACC(D_TAU, 1) += ai;
  ACC(D_TZ, 0) += s * ar; ACC(D_TZ, 1) += s * ai;
  ar = half * (Pr[0][1] - Pr[1][0]); ai = half * (Pi[0][1] - Pi[1][0]);
  ACC(D_JR, 0) -= ai; ACC(D_JR, 1) += ar;
  ACC(D_TJRZ, 0) -= s * ai; ACC(D_TJRZ, 1) += s * ar;
  ar = half * (Pr[0][3] - Pr[3][0]); ai = half * (Pi[0][3] - Pi[3][0]);
  ACC(D_JZ, 0) -= ai; ACC(D_JZ, 1) += ar;
  ACC(D_TJZZ, 0) -= s * ai; ACC(D_TJZZ, 1) += s * ar;
  ACC(D_GS, 0) += s * (Pr[0][3] + Pr[3][0]); ACC(D_GS, 1) += s * (Pi[0][3] + Pi[3][0]);
  ACC(D_FR, 0) += half * s * (Pr[1][3] + Pr[3][1]); ACC(D_FR, 1) += half * s * (Pi[1][3] + Pi[3][1]);
  ar = Pr[2][3] - Pr[3][2]; ai = Pi[2][3] - Pi[3][2];
  ACC(D_FP, 0) -= half * s * ai; ACC(D_FP, 1) += half * s * ar;
  ACC(D_FZ, 0) += s * Pr[3][3]; ACC(D_FZ, 1) += s * Pi[3][3];
  const A e = A(-s);
  ACC(D_SR, 0) += Qr[0][0]; ACC(D_SR, 1) += Qi[0][0];
  ACC(D_SP, 0) -= e * Qi[0][0]; ACC(D_SP, 1) += e * Qr[0][0];
  const A t2r = half * (Qr[2][0] + Qr[0][2]), t2i = half * (Qi[2][0] + Qi[0][2]);
  ACC(D_TJPR, 0) += t2r; ACC(D_TJPR, 1) += t2i;
  ACC(D_TJPP, 0) -= e * t2i; ACC(D_TJPP, 1) += e * t2r;
  ACC(D_GS, 0) += e * (Qr[0][2] - Qr[2][0]) + (Qr[0][1] + Qr[1][0]);
  ACC(D_GS, 1) += e * (Qi[0][2] - Qi[2][0]) + (Qi[0][1] + Qi[1][0]);
  const A tkr = Qr[1][1] + Qr[2][2] + Qr[3][3], tki = Qi[1][1] + Qi[2][2] + Qi[3][3];
  ACC(D_TR, 0) += tkr; ACC(D_TR, 1) += tki;
  ACC(D_TP, 0) -= e * tki; ACC(D_TP, 1) += e * tkr;
  const A jrr = half * (Qr[0][1] - Qr[1][0]), jri = half * (Qi[0][1] - Qi[1][0]);
  ACC(D_TJRR, 0) -= jri; ACC(D_TJRR, 1) += jrr;
  ACC(D_TJRP, 0) -= e * jrr; ACC(D_TJRP, 1) -= e * jri;
  const A jzr = half * (Qr[0][3] - Qr[3][0]), jzi = half * (Qi[0][3] - Qi[3][0]);
  ACC(D_TJZR, 0) -= jzi; ACC(D_TJZR, 1) += jzr;
  ACC(D_TJZP, 0) -= e * jzr; ACC(D_TJZP, 1) -= e * jzi;
  ar = Qr[1][1] + e * half * (Qr[1][2] - Qr[2][1]);
  ai = Qi[1][1] + e * half * (Qi[1][2] - Qi[2][1]);
  ACC(D_FR, 0) += ar; ACC(D_FR, 1) += ai;
  ar = e * Qr[2][2] + half * (Qr[2][1] - Qr[1][2]);
  ai = e * Qi[2][2] + half * (Qi[2][1] - Qi[1][2]);
  ACC(D_FP, 0) -= ai; ACC(D_FP, 1) += ar;
  ar = Qr[3][1] + Qr[1][3] + e * (Qr[3][2] - Qr[2][3]);
  ai = Qi[3][1] + Qi[1][3] + e * (Qi[3][2] - Qi[2][3]);
  ACC(D_FZ, 0) += half * ar; ACC(D_FZ, 1) += half * ai;
#undef ACC
}

__device__ inline void density_column(double *acc, const double (&Tr)[4][2], const double (&Ti)[4][2],
                                      const double (&y)[4], int s) {
  const int sd = s > 0 ? 0 : 1, so = 1 - sd;
  double Pr[4][4], Pi[4][4], Qr[4][4], Qi[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int yy = 0; yy < 4; ++yy) {
      Pr[x][yy] = Tr[x][sd] * y[yy]; Pi[x][yy] = Ti[x][sd] * y[yy];
      Qr[x][yy] = Tr[x][so] * y[yy]; Qi[x][yy] = Ti[x][so] * y[yy];
    }
  density_accumulate(acc, Pr, Pi, Qr, Qi, s);
}

// Local densities with FP64 MFMA (v_mfma_f64_16x16x4).  One wave per
// (16 grid points, frequency, sector), looping over all block pairs.  With few
// frequencies the third grid dimension also splits the pair lists
// (blockIdx.z = sector + 2 split): split z takes pairs [z n / Z, (z + 1) n / Z)
// of each list and writes its partial densities to A.part, which k_dens_sum
// adds split by split.  With one split the kernel is the unsplit one.
// T_x^s(r, b) = sum_a psi_x(r,a) rho(a,b) runs on the matrix cores (rows r,
// k = a in steps of 4, 16 columns b per tile, re and im tiles), per-spin ranges
// of a accumulated separately; the tile goes through LDS to a lane-per-(r, 4 b)
// layout for the density products, whose sums over b stay in registers.
__global__ void __launch_bounds__(64) k_density_mfma(DensArgs A) {
  __shared__ double sT[16][16][17];     // [(x, s, ri)][r][b]
  const int lane = threadIdx.x;
  const int r0 = blockIdx.x * 16;
  const int w = A.act[blockIdx.y];
  if (w == A.skip) return;
  const int sec = blockIdx.z & 1;
  const int spl = blockIdx.z >> 1, nspl = gridDim.z >> 1;
  const int G = A.nghl;
  const int mi = lane & 15, mk = lane >> 4;     // MFMA operand lane coordinates
  const int er = lane & 15, eg = lane >> 4;     // epilogue: row er, columns eg + 4q
  const int rA = r0 + mi;
  const bool rA_ok = rA < G;
  const int rE = r0 + er;
  const bool rE_ok = rE < G;
  const int rEc = rE_ok ? rE : 0;
  double acc[2 * NDENS];
#pragma unroll
  for (int d = 0; d < 2 * NDENS; ++d) acc[d] = 0.0;
  const double *rho_re = A.rsp + ((size_t)w * 8 + 2 * A.rho_slot[sec]) * A.nxy;
  const double *rho_im = rho_re + A.nxy;
  const double *tab[4] = {A.wf, A.wfdr, A.wfdp, A.wfdz};
  const PairList pl = A.rho[sec];
  const int p0 = (int)((long)spl * pl.n / nspl), p1 = (int)((long)(spl + 1) * pl.n / nspl);
  for (int p = p0; p < p1; ++p) {
    const int4 pr = pl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy], nsu = A.nsu[ix];
    for (int b0 = 0; b0 < dy; b0 += 16) {
      v4d C[4][2][2];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) { C[x][s2][0] = v4d{0, 0, 0, 0}; C[x][s2][1] = v4d{0, 0, 0, 0}; }
      const int bj = b0 + mi;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int lo = s2 ? nsu : 0, hi = s2 ? dx : nsu;
        // operands of the k step at a (zero outside the block and the grid)
        auto load = [&](int a, double (&av)[4], double &br, double &bi) {
          const int ak = a + mk;
          const bool ok = ak < hi;
          const size_t oa = (size_t)(ia + (ok ? ak : lo)) * G + (rA_ok ? rA : 0);
#pragma unroll
          for (int x = 0; x < 4; ++x) av[x] = (ok && rA_ok) ? tab[x][oa] : 0.0;
          const bool bok = ok && bj < dy;
          const size_t ob = off + (size_t)(bok ? bj : 0) * dx + (ok ? ak : 0);
          br = bok ? rho_re[ob] : 0.0;
          bi = bok ? rho_im[ob] : 0.0;
        };
        // the loads of step a + 4 are issued before the products of step a
        double avn[4], brn, bin;
        load(lo, avn, brn, bin);
        for (int a = lo; a < hi; a += 4) {
          double av[4];
#pragma unroll
          for (int x = 0; x < 4; ++x) av[x] = avn[x];
          const double br = brn, bi = bin;
          if (a + 4 < hi) load(a + 4, avn, brn, bin);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            C[x][s2][0] = mfma64(av[x], br, C[x][s2][0]);
            C[x][s2][1] = mfma64(av[x], bi, C[x][s2][1]);
          }
        }
      }
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
          for (int ri = 0; ri < 2; ++ri)
#pragma unroll
            for (int v = 0; v < 4; ++v) sT[(x * 2 + s2) * 2 + ri][4 * v + mk][mi] = C[x][s2][ri][v];
      __syncthreads();
      for (int q = 0; q < 4; ++q) {
        const int bl = eg + 4 * q;
        if (b0 + bl >= dy) break;
        const int b = ib0 + b0 + bl;
        double Tr[4][2], Ti[4][2];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            Tr[x][s2] = sT[(x * 2 + s2) * 2 + 0][er][bl];
            Ti[x][s2] = sT[(x * 2 + s2) * 2 + 1][er][bl];
          }
        const size_t oy = (size_t)b * G + rEc;
        const double y[4] = {A.wf[oy], A.wfdr[oy], A.wfdp[oy], A.wfdz[oy]};
        density_column(acc, Tr, Ti, y, A.ns[b]);
      }
      __syncthreads();
    }
  }
  // pairing densities from kappa: x = 0 only
  const double *kap_re = A.rsp + ((size_t)w * 8 + 2 * A.kap_slot[sec]) * A.nxy;
  const double *kap_im = kap_re + A.nxy;
  const PairList kl = A.kap[sec];
  const int q0 = (int)((long)spl * kl.n / nspl), q1 = (int)((long)(spl + 1) * kl.n / nspl);
  for (int p = q0; p < q1; ++p) {
    const int4 pr = kl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy], nsu = A.nsu[ix];
    for (int b0 = 0; b0 < dy; b0 += 16) {
      v4d C[2][2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) { C[s2][0] = v4d{0, 0, 0, 0}; C[s2][1] = v4d{0, 0, 0, 0}; }
      const int bj = b0 + mi;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int lo = s2 ? nsu : 0, hi = s2 ? dx : nsu;
        auto load = [&](int a, double &av, double &br, double &bi) {
          const int ak = a + mk;
          const bool ok = ak < hi;
          av = (ok && rA_ok) ? A.wf[(size_t)(ia + ak) * G + rA] : 0.0;
          const bool bok = ok && bj < dy;
          const size_t ob = off + (size_t)(bok ? bj : 0) * dx + (ok ? ak : 0);
          br = bok ? kap_re[ob] : 0.0;
          bi = bok ? kap_im[ob] : 0.0;
        };
        double avn, brn, bin;
        load(lo, avn, brn, bin);
        for (int a = lo; a < hi; a += 4) {
          const double av = avn, br = brn, bi = bin;
          if (a + 4 < hi) load(a + 4, avn, brn, bin);
          C[s2][0] = mfma64(av, br, C[s2][0]);
          C[s2][1] = mfma64(av, bi, C[s2][1]);
        }
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int ri = 0; ri < 2; ++ri)
#pragma unroll
          for (int v = 0; v < 4; ++v) sT[s2 * 2 + ri][4 * v + mk][mi] = C[s2][ri][v];
      __syncthreads();
      for (int q = 0; q < 4; ++q) {
        const int bl = eg + 4 * q;
        if (b0 + bl >= dy) break;
        const int b = ib0 + b0 + bl;
        const int s = A.ns[b];
        const int sd = s > 0 ? 0 : 1, so = 1 - sd;
        const double wb = A.wf[(size_t)b * G + rEc];
        double pr_ = 2.0 * sT[so * 2 + 0][er][bl] * wb, pi_ = 2.0 * sT[so * 2 + 1][er][bl] * wb;
        acc[2 * D_RB] -= s * pr_; acc[2 * D_RB + 1] -= s * pi_;
        acc[2 * D_SBZ] += pr_; acc[2 * D_SBZ + 1] += pi_;
        pr_ = 2.0 * sT[sd * 2 + 0][er][bl] * wb; pi_ = 2.0 * sT[sd * 2 + 1][er][bl] * wb;
        acc[2 * D_SBR] += s < 0 ? pr_ : -pr_; acc[2 * D_SBR + 1] += s < 0 ? pi_ : -pi_;
        acc[2 * D_SBP] += pi_; acc[2 * D_SBP + 1] -= pr_;
      }
      __syncthreads();
    }
  }
  // sum the four column subgroups (lanes er, er+16, er+32, er+48)
  const double wc = rE_ok ? A.wdcori[rE] : 0.0;
  double *out = (A.part ? A.part + (((size_t)spl * gridDim.y + blockIdx.y) * 2 + sec) * 2 * NDENS * G
                        : A.dens + (((size_t)w * 2 + sec) * 2 * NDENS) * G) + rEc;
#pragma unroll
  for (int d = 0; d < 2 * NDENS; ++d) {
    double v = acc[d];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (eg == 0 && rE_ok) out[(size_t)d * G] = v * wc;
  }
}

// Local densities with FP64 MFMA, two waves per (16 grid points, frequency,
// sector, split).  For each block pair and 16-column tile the waves share the
// products T_x^s(r, b) = sum_a psi_x(r,a) rho(a,b): wave 0 computes x = 0, 1
// and wave 1 x = 2, 3 into LDS (the pairing products: wave 0 the spin-up rows
// of a, wave 1 the spin-down rows).  The epilogue is split by spin relation:
// wave 0 accumulates the same-spin terms (P) of the densities and the pairing
// densities built from them (s-breve_r, s-breve_phi), wave 1 the opposite-spin
// terms (Q) and the pairing densities rho-breve and s-breve_z; the four
// densities with both (gs and the three F) are summed through LDS at the end.
// Each wave holds 16 complex accumulators instead of 28, so two waves fit
// where one did; the terms are those of density_accumulate.
constexpr int DPQ_NACC = 16;
__device__ constexpr int kDensP[DPQ_NACC] = {D_RHO, D_SZ, D_JP, D_TJPZ, D_TAU, D_TZ, D_JR, D_TJRZ,
                                             D_JZ, D_TJZZ, D_GS, D_FR, D_FP, D_FZ, D_SBR, D_SBP};
__device__ constexpr int kDensQ[DPQ_NACC] = {D_SR, D_SP, D_TJPR, D_TJPP, D_GS, D_TR, D_TP, D_TJRR,
                                             D_TJRP, D_TJZR, D_TJZP, D_FR, D_FP, D_FZ, D_RB, D_SBZ};

// same-spin (P) terms of density_accumulate; acc in kDensP order
// (the products T_x y_y are formed where they are used, so only T and y stay live)
__device__ inline void density_acc_p(double *acc, const double (&tr)[4], const double (&ti)[4], const double (&y)[4],
                                     int s) {
#define Pr(x, yy) (tr[x] * y[yy])
#define Pi(x, yy) (ti[x] * y[yy])
#define AP(k, ri) acc[2 * (k) + (ri)]
  const double half = 0.5;
  double ar, ai;
  AP(0, 0) += Pr(0, 0); AP(0, 1) += Pi(0, 0);                       // rho
  AP(1, 0) += s * Pr(0, 0); AP(1, 1) += s * Pi(0, 0);               // s_z
  ar = half * (Pr(0, 2) + Pr(2, 0)); ai = half * (Pi(0, 2) + Pi(2, 0));
  AP(2, 0) += ar; AP(2, 1) += ai;                                   // j_phi
  AP(3, 0) += s * ar; AP(3, 1) += s * ai;                           // J_phi z
  ar = Pr(1, 1) + Pr(2, 2) + Pr(3, 3); ai = Pi(1, 1) + Pi(2, 2) + Pi(3, 3);
  AP(4, 0) += ar; AP(4, 1) += ai;                                   // tau
  AP(5, 0) += s * ar; AP(5, 1) += s * ai;                           // T_z
  ar = half * (Pr(0, 1) - Pr(1, 0)); ai = half * (Pi(0, 1) - Pi(1, 0));
  AP(6, 0) -= ai; AP(6, 1) += ar;                                   // j_r
  AP(7, 0) -= s * ai; AP(7, 1) += s * ar;                           // J_rz
  ar = half * (Pr(0, 3) - Pr(3, 0)); ai = half * (Pi(0, 3) - Pi(3, 0));
  AP(8, 0) -= ai; AP(8, 1) += ar;                                   // j_z
  AP(9, 0) -= s * ai; AP(9, 1) += s * ar;                           // J_zz
  AP(10, 0) += s * (Pr(0, 3) + Pr(3, 0)); AP(10, 1) += s * (Pi(0, 3) + Pi(3, 0));                 // gs
  AP(11, 0) += half * s * (Pr(1, 3) + Pr(3, 1)); AP(11, 1) += half * s * (Pi(1, 3) + Pi(3, 1));   // F_r
  ar = Pr(2, 3) - Pr(3, 2); ai = Pi(2, 3) - Pi(3, 2);
  AP(12, 0) -= half * s * ai; AP(12, 1) += half * s * ar;          // F_phi
  AP(13, 0) += s * Pr(3, 3); AP(13, 1) += s * Pi(3, 3);             // F_z
#undef AP
#undef Pr
#undef Pi
}

// opposite-spin (Q) terms of density_accumulate; acc in kDensQ order
__device__ inline void density_acc_q(double *acc, const double (&tr)[4], const double (&ti)[4], const double (&y)[4],
                                     int s) {
#define Qr(x, yy) (tr[x] * y[yy])
#define Qi(x, yy) (ti[x] * y[yy])
#define AQ(k, ri) acc[2 * (k) + (ri)]
  const double half = 0.5;
  const double e = -s;
  double ar, ai;
  AQ(0, 0) += Qr(0, 0); AQ(0, 1) += Qi(0, 0);                       // s_r
  AQ(1, 0) -= e * Qi(0, 0); AQ(1, 1) += e * Qr(0, 0);               // s_phi
  const double t2r = half * (Qr(2, 0) + Qr(0, 2)), t2i = half * (Qi(2, 0) + Qi(0, 2));
  AQ(2, 0) += t2r; AQ(2, 1) += t2i;                                 // J_phi r
  AQ(3, 0) -= e * t2i; AQ(3, 1) += e * t2r;                         // J_phi phi
  AQ(4, 0) += e * (Qr(0, 2) - Qr(2, 0)) + (Qr(0, 1) + Qr(1, 0));   // gs
  AQ(4, 1) += e * (Qi(0, 2) - Qi(2, 0)) + (Qi(0, 1) + Qi(1, 0));
  const double tkr = Qr(1, 1) + Qr(2, 2) + Qr(3, 3), tki = Qi(1, 1) + Qi(2, 2) + Qi(3, 3);
  AQ(5, 0) += tkr; AQ(5, 1) += tki;                                 // T_r
  AQ(6, 0) -= e * tki; AQ(6, 1) += e * tkr;                         // T_phi
  const double jrr = half * (Qr(0, 1) - Qr(1, 0)), jri = half * (Qi(0, 1) - Qi(1, 0));
  AQ(7, 0) -= jri; AQ(7, 1) += jrr;                                 // J_rr
  AQ(8, 0) -= e * jrr; AQ(8, 1) -= e * jri;                         // J_r phi
  const double jzr = half * (Qr(0, 3) - Qr(3, 0)), jzi = half * (Qi(0, 3) - Qi(3, 0));
  AQ(9, 0) -= jzi; AQ(9, 1) += jzr;                                 // J_zr
  AQ(10, 0) -= e * jzr; AQ(10, 1) -= e * jzi;                       // J_z phi
  ar = Qr(1, 1) + e * half * (Qr(1, 2) - Qr(2, 1));
  ai = Qi(1, 1) + e * half * (Qi(1, 2) - Qi(2, 1));
  AQ(11, 0) += ar; AQ(11, 1) += ai;                                 // F_r
  ar = e * Qr(2, 2) + half * (Qr(2, 1) - Qr(1, 2));
  ai = e * Qi(2, 2) + half * (Qi(2, 1) - Qi(1, 2));
  AQ(12, 0) -= ai; AQ(12, 1) += ar;                                 // F_phi
  ar = Qr(3, 1) + Qr(1, 3) + e * (Qr(3, 2) - Qr(2, 3));
  ai = Qi(3, 1) + Qi(1, 3) + e * (Qi(3, 2) - Qi(2, 3));
  AQ(13, 0) += half * ar; AQ(13, 1) += half * ai;                   // F_z
#undef AQ
#undef Qr
#undef Qi
}

__global__ void __launch_bounds__(128) k_density_pq(DensArgs A) {
  __shared__ double sT[16][16][17];     // [(x, s, ri)][r][b]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r0 = blockIdx.x * 16;
  const int w = A.act[blockIdx.y];
  if (w == A.skip) return;
  const int sec = blockIdx.z & 1;
  const int spl = blockIdx.z >> 1, nspl = gridDim.z >> 1;
  const int G = A.nghl;
  const int mi = lane & 15, mk = lane >> 4;     // MFMA operand lane coordinates
  const int er = lane & 15, eg = lane >> 4;     // epilogue: row er, columns eg + 4q
  const int rA = r0 + mi;
  const bool rA_ok = rA < G;
  const int rE = r0 + er;
  const bool rE_ok = rE < G;
  const int rEc = rE_ok ? rE : 0;
  double acc[2 * DPQ_NACC];
#pragma unroll
  for (int d = 0; d < 2 * DPQ_NACC; ++d) acc[d] = 0.0;
  const double *rho_re = A.rsp + ((size_t)w * 8 + 2 * A.rho_slot[sec]) * A.nxy;
  const double *rho_im = rho_re + A.nxy;
  const double *tab[4] = {A.wf, A.wfdr, A.wfdp, A.wfdz};
  const double *tw0 = tab[2 * wave], *tw1 = tab[2 * wave + 1];   // this wave's two tables
  const PairList pl = A.rho[sec];
  const int p0 = (int)((long)spl * pl.n / nspl), p1 = (int)((long)(spl + 1) * pl.n / nspl);
  for (int p = p0; p < p1; ++p) {
    const int4 pr = pl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy], nsu = A.nsu[ix];
    for (int b0 = 0; b0 < dy; b0 += 16) {
      v4d C[2][2][2];
#pragma unroll
      for (int xl = 0; xl < 2; ++xl)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) { C[xl][s2][0] = v4d{0, 0, 0, 0}; C[xl][s2][1] = v4d{0, 0, 0, 0}; }
      const int bj = b0 + mi;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int lo = s2 ? nsu : 0, hi = s2 ? dx : nsu;
        auto load = [&](int a, double (&av)[2], double &br, double &bi) {
          const int ak = a + mk;
          const bool ok = ak < hi;
          const size_t oa = (size_t)(ia + (ok ? ak : lo)) * G + (rA_ok ? rA : 0);
          av[0] = (ok && rA_ok) ? tw0[oa] : 0.0;
          av[1] = (ok && rA_ok) ? tw1[oa] : 0.0;
          const bool bok = ok && bj < dy;
          const size_t ob = off + (size_t)(bok ? bj : 0) * dx + (ok ? ak : 0);
          br = bok ? rho_re[ob] : 0.0;
          bi = bok ? rho_im[ob] : 0.0;
        };
        double avn[2], brn, bin;
        load(lo, avn, brn, bin);
        for (int a = lo; a < hi; a += 4) {
          const double av0 = avn[0], av1 = avn[1], br = brn, bi = bin;
          if (a + 4 < hi) load(a + 4, avn, brn, bin);
          C[0][s2][0] = mfma64(av0, br, C[0][s2][0]);
          C[0][s2][1] = mfma64(av0, bi, C[0][s2][1]);
          C[1][s2][0] = mfma64(av1, br, C[1][s2][0]);
          C[1][s2][1] = mfma64(av1, bi, C[1][s2][1]);
        }
      }
#pragma unroll
      for (int xl = 0; xl < 2; ++xl)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
          for (int ri = 0; ri < 2; ++ri)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              sT[((2 * wave + xl) * 2 + s2) * 2 + ri][4 * v + mk][mi] = C[xl][s2][ri][v];
      __syncthreads();
      for (int q = 0; q < 4; ++q) {
        const int bl = eg + 4 * q;
        if (b0 + bl >= dy) break;
        const int b = ib0 + b0 + bl;
        const int s = A.ns[b];
        const int sd = s > 0 ? 0 : 1;
        const int sx = wave == 0 ? sd : 1 - sd;   // the spin of a this wave contracts
        const size_t oy = (size_t)b * G + rEc;
        const double y[4] = {A.wf[oy], A.wfdr[oy], A.wfdp[oy], A.wfdz[oy]};
        double tr[4], ti[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          tr[x] = sT[(x * 2 + sx) * 2 + 0][er][bl];
          ti[x] = sT[(x * 2 + sx) * 2 + 1][er][bl];
        }
        if (wave == 0) density_acc_p(acc, tr, ti, y, s);
        else density_acc_q(acc, tr, ti, y, s);
      }
      __syncthreads();
    }
  }
  // pairing densities from kappa: x = 0; wave 0 the spin-up rows of a, wave 1 the spin-down rows
  const double *kap_re = A.rsp + ((size_t)w * 8 + 2 * A.kap_slot[sec]) * A.nxy;
  const double *kap_im = kap_re + A.nxy;
  const PairList kl = A.kap[sec];
  const int q0 = (int)((long)spl * kl.n / nspl), q1 = (int)((long)(spl + 1) * kl.n / nspl);
  for (int p = q0; p < q1; ++p) {
    const int4 pr = kl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy], nsu = A.nsu[ix];
    for (int b0 = 0; b0 < dy; b0 += 16) {
      v4d C0 = v4d{0, 0, 0, 0}, C1 = v4d{0, 0, 0, 0};
      const int bj = b0 + mi;
      const int s2 = wave;
      const int lo = s2 ? nsu : 0, hi = s2 ? dx : nsu;
      auto load = [&](int a, double &av, double &br, double &bi) {
        const int ak = a + mk;
        const bool ok = ak < hi;
        av = (ok && rA_ok) ? A.wf[(size_t)(ia + ak) * G + rA] : 0.0;
        const bool bok = ok && bj < dy;
        const size_t ob = off + (size_t)(bok ? bj : 0) * dx + (ok ? ak : 0);
        br = bok ? kap_re[ob] : 0.0;
        bi = bok ? kap_im[ob] : 0.0;
      };
      double avn, brn, bin;
      load(lo, avn, brn, bin);
      for (int a = lo; a < hi; a += 4) {
        const double av = avn, br = brn, bi = bin;
        if (a + 4 < hi) load(a + 4, avn, brn, bin);
        C0 = mfma64(av, br, C0);
        C1 = mfma64(av, bi, C1);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        sT[s2 * 2 + 0][4 * v + mk][mi] = C0[v];
        sT[s2 * 2 + 1][4 * v + mk][mi] = C1[v];
      }
      __syncthreads();
      for (int q = 0; q < 4; ++q) {
        const int bl = eg + 4 * q;
        if (b0 + bl >= dy) break;
        const int b = ib0 + b0 + bl;
        const int s = A.ns[b];
        const int sd = s > 0 ? 0 : 1, so = 1 - sd;
        const double wb = A.wf[(size_t)b * G + rEc];
        if (wave == 1) {   // rho-breve, s-breve_z (opposite spin)
          const double pr_ = 2.0 * sT[so * 2 + 0][er][bl] * wb, pi_ = 2.0 * sT[so * 2 + 1][er][bl] * wb;
          acc[2 * 14] -= s * pr_; acc[2 * 14 + 1] -= s * pi_;
          acc[2 * 15] += pr_; acc[2 * 15 + 1] += pi_;
        } else {           // s-breve_r, s-breve_phi (same spin)
          const double pr_ = 2.0 * sT[sd * 2 + 0][er][bl] * wb, pi_ = 2.0 * sT[sd * 2 + 1][er][bl] * wb;
          acc[2 * 14] += s < 0 ? pr_ : -pr_; acc[2 * 14 + 1] += s < 0 ? pi_ : -pi_;
          acc[2 * 15] += pi_; acc[2 * 15 + 1] -= pr_;
        }
      }
      __syncthreads();
    }
  }
  // sum the four column subgroups (lanes er, er+16, er+32, er+48)
#pragma unroll
  for (int d = 0; d < 2 * DPQ_NACC; ++d) {
    double v = acc[d];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    acc[d] = v;
  }
  // gs, F_r, F_phi, F_z: wave 1's part through LDS to wave 0
  double *xch = &sT[0][0][0];
  if (wave == 1 && eg == 0)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int lq = k == 0 ? 4 : 10 + k;   // kDensQ slots of gs, F_r, F_phi, F_z
      xch[(2 * k) * 16 + er] = acc[2 * lq];
      xch[(2 * k + 1) * 16 + er] = acc[2 * lq + 1];
    }
  __syncthreads();
  if (wave == 0 && eg == 0)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int lp = 10 + k;                // kDensP slots of gs, F_r, F_phi, F_z
      acc[2 * lp] += xch[(2 * k) * 16 + er];
      acc[2 * lp + 1] += xch[(2 * k + 1) * 16 + er];
    }
  const double wc = rE_ok ? A.wdcori[rE] : 0.0;
  double *out = (A.part ? A.part + (((size_t)spl * gridDim.y + blockIdx.y) * 2 + sec) * 2 * NDENS * G
                        : A.dens + (((size_t)w * 2 + sec) * 2 * NDENS) * G) + rEc;
  if (eg == 0 && rE_ok)
#pragma unroll
    for (int k = 0; k < DPQ_NACC; ++k) {
      const int d = wave == 0 ? kDensP[k] : kDensQ[k];
      const bool shared = wave == 1 && (k == 4 || (k >= 11 && k <= 13));   // written by wave 0
      if (!shared) {
        out[(size_t)(2 * d) * G] = acc[2 * k] * wc;
        out[(size_t)(2 * d + 1) * G] = acc[2 * k + 1] * wc;
      }
    }
}

// Local densities with FP64 MFMA, two waves and no exchange (fp64_density 2).
// The columns b of block iy go in 16-column tiles within each spin range
// (block states are spin-sorted: [0, nsu) up, [nsu, d) down), so a tile's
// columns share one spin; wave 0 contracts the rows a of that spin (the
// same-spin, P densities), wave 1 the rows of the other spin (Q), each for all
// four psi_x.  The products are the transpose of k_density_pq's,
// T_x^T(b, r) = sum_a rho(a, b) psi_x(r, a): lane i + 16 k supplies
// rho(a + k, b0 + i) and psi_x(r0 + i, a + k), and lane r + 16 g receives the
// columns b0 + 4 v + g of grid point r0 + r -- the layout of the density
// products, so the tile needs neither an LDS pass nor a barrier, and the two
// waves run through their pairs independently.  The pairing densities
// (kappa, x = 0) go the same way.  Splits (few frequencies), outputs and the
// four densities both waves contribute to are as in k_density_pq.
__global__ void __launch_bounds__(128, 2) k_density_pq2(DensArgs A) {
  __shared__ double xch[8 * 16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r0 = blockIdx.x * 16;
  const int w = A.act[blockIdx.y];
  if (w == A.skip) return;
  const int sec = blockIdx.z & 1;
  const int spl = blockIdx.z >> 1, nspl = gridDim.z >> 1;
  const int G = A.nghl;
  const int li = lane & 15, lk = lane >> 4;     // MFMA operand lane coordinates
  const int er = lane & 15, eg = lane >> 4;     // products: grid point er, columns 4 v + eg
  const int rB = r0 + li;
  const bool rB_ok = rB < G;
  const int rBc = rB_ok ? rB : 0;
  const int rE = r0 + er;
  const bool rE_ok = rE < G;
  const int rEc = rE_ok ? rE : 0;
  double acc[2 * DPQ_NACC];
#pragma unroll
  for (int d = 0; d < 2 * DPQ_NACC; ++d) acc[d] = 0.0;
  const double *rho_re = A.rsp + ((size_t)w * 8 + 2 * A.rho_slot[sec]) * A.nxy;
  const double *rho_im = rho_re + A.nxy;
  const double *tab[4] = {A.wf, A.wfdr, A.wfdp, A.wfdz};
  const PairList pl = A.rho[sec];
  const int p0 = (int)((long)spl * pl.n / nspl), p1 = (int)((long)(spl + 1) * pl.n / nspl);
  for (int p = p0; p < p1; ++p) {
    const int4 pr = pl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy];
    const int nsu = A.nsu[ix], nsuy = A.nsu[iy];
    for (int h = 0; h < 2; ++h) {                   // spin range of the columns
      const int c0 = h ? nsuy : 0, c1 = h ? dy : nsuy;
      const int sx = wave == 0 ? h : 1 - h;          // the spin range of a this wave contracts
      const int lo = sx ? nsu : 0, hi = sx ? dx : nsu;
      for (int b0 = c0; b0 < c1; b0 += 16) {
        v4d C[4][2];
#pragma unroll
        for (int x = 0; x < 4; ++x) { C[x][0] = v4d{0, 0, 0, 0}; C[x][1] = v4d{0, 0, 0, 0}; }
        const int bj = b0 + li;
        const bool bcol = bj < c1;
        auto load = [&](int a, double (&pv)[4], double &br, double &bi) {
          const int ak = a + lk;
          const bool ok = ak < hi;
          const size_t oa = (size_t)(ia + (ok ? ak : lo)) * G + rBc;
#pragma unroll
          for (int x = 0; x < 4; ++x) pv[x] = (ok && rB_ok) ? tab[x][oa] : 0.0;
          const bool bok = ok && bcol;
          const size_t ob = off + (size_t)(bok ? bj : 0) * dx + (ok ? ak : 0);
          br = bok ? rho_re[ob] : 0.0;
          bi = bok ? rho_im[ob] : 0.0;
        };
        if (lo < hi) {
          double pvn[4], brn, bin;
          load(lo, pvn, brn, bin);
          for (int a = lo; a < hi; a += 4) {
            double pv[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) pv[x] = pvn[x];
            const double br = brn, bi = bin;
            if (a + 4 < hi) load(a + 4, pvn, brn, bin);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              C[x][0] = mfma64(br, pv[x], C[x][0]);
              C[x][1] = mfma64(bi, pv[x], C[x][1]);
            }
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int bl = 4 * v + eg;
          if (b0 + bl < c1) {
            const int b = ib0 + b0 + bl;
            const int s = A.ns[b];
            const size_t oy = (size_t)b * G + rEc;
            const double y[4] = {A.wf[oy], A.wfdr[oy], A.wfdp[oy], A.wfdz[oy]};
            double tr[4], ti[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) { tr[x] = C[x][0][v]; ti[x] = C[x][1][v]; }
            if (wave == 0) density_acc_p(acc, tr, ti, y, s);
            else density_acc_q(acc, tr, ti, y, s);
          }
          // one column at a time: the loads of the next column's psi_y wait here
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  // pairing densities from kappa (x = 0): wave 0 the rows of the columns' spin,
  // wave 1 the others
  const double *kap_re = A.rsp + ((size_t)w * 8 + 2 * A.kap_slot[sec]) * A.nxy;
  const double *kap_im = kap_re + A.nxy;
  const PairList kl = A.kap[sec];
  const int q0 = (int)((long)spl * kl.n / nspl), q1 = (int)((long)(spl + 1) * kl.n / nspl);
  for (int p = q0; p < q1; ++p) {
    const int4 pr = kl.p[p];
    const int ix = pr.x, iy = pr.y, off = pr.z;
    const int ia = A.isstart[ix], ib0 = A.isstart[iy], dx = A.db[ix], dy = A.db[iy];
    const int nsu = A.nsu[ix], nsuy = A.nsu[iy];
    for (int h = 0; h < 2; ++h) {
      const int c0 = h ? nsuy : 0, c1 = h ? dy : nsuy;
      const int sx = wave == 0 ? h : 1 - h;
      const int lo = sx ? nsu : 0, hi = sx ? dx : nsu;
      for (int b0 = c0; b0 < c1; b0 += 16) {
        v4d C0 = v4d{0, 0, 0, 0}, C1 = v4d{0, 0, 0, 0};
        const int bj = b0 + li;
        const bool bcol = bj < c1;
        auto load = [&](int a, double &pv, double &br, double &bi) {
          const int ak = a + lk;
          const bool ok = ak < hi;
          pv = (ok && rB_ok) ? A.wf[(size_t)(ia + ak) * G + rB] : 0.0;
          const bool bok = ok && bcol;
          const size_t ob = off + (size_t)(bok ? bj : 0) * dx + (ok ? ak : 0);
          br = bok ? kap_re[ob] : 0.0;
          bi = bok ? kap_im[ob] : 0.0;
        };
        if (lo < hi) {
          double pvn, brn, bin;
          load(lo, pvn, brn, bin);
          for (int a = lo; a < hi; a += 4) {
            const double pv = pvn, br = brn, bi = bin;
            if (a + 4 < hi) load(a + 4, pvn, brn, bin);
            C0 = mfma64(br, pv, C0);
            C1 = mfma64(bi, pv, C1);
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int bl = 4 * v + eg;
          if (b0 + bl < c1) {
            const int b = ib0 + b0 + bl;
            const int s = A.ns[b];
            const double wb = A.wf[(size_t)b * G + rEc];
            const double pr_ = 2.0 * C0[v] * wb, pi_ = 2.0 * C1[v] * wb;
            if (wave == 1) {   // rho-breve, s-breve_z (opposite spin)
              acc[2 * 14] -= s * pr_; acc[2 * 14 + 1] -= s * pi_;
              acc[2 * 15] += pr_; acc[2 * 15 + 1] += pi_;
            } else {           // s-breve_r, s-breve_phi (same spin)
              acc[2 * 14] += s < 0 ? pr_ : -pr_; acc[2 * 14 + 1] += s < 0 ? pi_ : -pi_;
              acc[2 * 15] += pi_; acc[2 * 15 + 1] -= pr_;
            }
          }
        }
      }
    }
  }
  // sum the four column subgroups (lanes er, er+16, er+32, er+48)
#pragma unroll
  for (int d = 0; d < 2 * DPQ_NACC; ++d) {
    double v = acc[d];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    acc[d] = v;
  }
  // gs, F_r, F_phi, F_z: wave 1's part through LDS to wave 0
  if (wave == 1 && eg == 0)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int lq = k == 0 ? 4 : 10 + k;   // kDensQ slots of gs, F_r, F_phi, F_z
      xch[(2 * k) * 16 + er] = acc[2 * lq];
      xch[(2 * k + 1) * 16 + er] = acc[2 * lq + 1];
    }
  __syncthreads();
  if (wave == 0 && eg == 0)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int lp = 10 + k;                // kDensP slots of gs, F_r, F_phi, F_z
      acc[2 * lp] += xch[(2 * k) * 16 + er];
      acc[2 * lp + 1] += xch[(2 * k + 1) * 16 + er];
    }
  const double wc = rE_ok ? A.wdcori[rE] : 0.0;
  double *out = (A.part ? A.part + (((size_t)spl * gridDim.y + blockIdx.y) * 2 + sec) * 2 * NDENS * G
                        : A.dens + (((size_t)w * 2 + sec) * 2 * NDENS) * G) + rEc;
  if (eg == 0 && rE_ok)
#pragma unroll
    for (int k = 0; k < DPQ_NACC; ++k) {
      const int d = wave == 0 ? kDensP[k] : kDensQ[k];
      const bool shared = wave == 1 && (k == 4 || (k >= 11 && k <= 13));   // written by wave 0
      if (!shared) {
        out[(size_t)(2 * d) * G] = acc[2 * k] * wc;
        out[(size_t)(2 * d + 1) * G] = acc[2 * k + 1] * wc;
      }
    }
}

// densities of the active frequency y = the sum of its nsplit partial
// densities, split by split (k_density_mfma with split pair lists)
__global__ void k_dens_sum(const double *__restrict__ part, int nsplit, int na, long nd, const int *__restrict__ act,
                           double *__restrict__ dens) {
  const int y = blockIdx.y;
  double *out = dens + (size_t)act[y] * nd;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < nd; e += (long)gridDim.x * blockDim.x) {
    double v = 0.0;
    for (int s = 0; s < nsplit; ++s) v += part[((size_t)s * na + y) * nd + e];
    out[e] = v;
  }
}

struct FieldArgs {
  const double *dens;     // [w][2][56][nghl]
  double *flds;           // [w][2][208][nghl]
  const double *crho, *cs, *cpair, *cspair;
  double cdrho, ctau, ctj0, ctj1, ctj2, crdj, cds, ct, cj, cgs, cf, csdj;
  int nghl;
  const int *act;
  int skip = -1;          // as DensArgs::skip
};

struct cplx { double r, i; };
__device__ inline cplx operator+(cplx a, cplx b) { return {a.r + b.r, a.i + b.i}; }
__device__ inline cplx operator-(cplx a, cplx b) { return {a.r - b.r, a.i - b.i}; }
__device__ inline cplx operator*(double s, cplx a) { return {s * a.r, s * a.i}; }
__device__ inline cplx mul_i(cplx a) { return {-a.i, a.r}; }   // i*a

// Mean and pairing fields in closed form.  The sequence of assignments of
// pnfam_hamiltonian_blas.f90:774-1093 (and 1200-1208 for pairing) resolved per
// field mf(z, z', s_a, s_b) with s = +1/-1 (index 0/1 here).
// GRID1D: for the contraction one grid direction at a time, which reads neither the
// components that are always zero nor (4, 0) and (2, 1), its (0, 4) and +-(1, 2);
// nor the same-spin (2, 2), its (1, 1), which is stored with the rest.
// Stores bound the kernel: 68 for it, 180 without (N_sh = 16, 128 points 195 -> 110 us).
template <bool GRID1D>
__global__ void __launch_bounds__(128) k_fields(FieldArgs F) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= F.nghl) return;
  const int w = F.act[blockIdx.y];
  if (w == F.skip) return;
  const int sec = blockIdx.z;
  const int G = F.nghl;
  const double *dn = F.dens + (((size_t)w * 2 + sec) * 2 * NDENS) * G + r;
  auto D = [&](int d) { return cplx{dn[(size_t)(2 * d) * G], dn[(size_t)(2 * d + 1) * G]}; };
  const cplx rho = D(D_RHO), tau = D(D_TAU), sr = D(D_SR), sp = D(D_SP), sz = D(D_SZ), tr = D(D_TR), tp = D(D_TP),
             tz = D(D_TZ), jr = D(D_JR), jp = D(D_JP), jz = D(D_JZ), fr = D(D_FR), fp = D(D_FP), fz = D(D_FZ),
             gs = D(D_GS), tjrr = D(D_TJRR), tjpr = D(D_TJPR), tjzr = D(D_TJZR), tjrp = D(D_TJRP),
             tjpp = D(D_TJPP), tjzp = D(D_TJZP), tjrz = D(D_TJRZ), tjpz = D(D_TJPZ), tjzz = D(D_TJZZ),
             rb = D(D_RB), sbr = D(D_SBR), sbp = D(D_SBP), sbz = D(D_SBZ);
  const double crho = F.crho[r], cs = F.cs[r], cpair = F.cpair[r], cspair = F.cspair[r];
  const double cdrho = F.cdrho, ctau = F.ctau, ctj0 = F.ctj0, ctj1 = F.ctj1, ctj2 = F.ctj2, crdj = F.crdj,
               cds = F.cds, ct = F.ct, cj = F.cj, cgs = F.cgs, cf = F.cf, csdj = F.csdj;
  const cplx c0 = ctj0 * (tjrr + tjpp + tjzz), c1a = ctj1 * (tjzr - tjrz), c1b = ctj1 * (tjpz - tjzp),
             c2a = ctj2 * (tjrz + tjzr), c2b = ctj2 * (tjpz + tjzp);
  double *out = F.flds + (((size_t)w * 2 + sec) * 2 * NFLD) * G + r;
  auto put = [&](int idx, cplx v) { out[(size_t)(2 * idx) * G] = v.r; out[(size_t)(2 * idx + 1) * G] = v.i; };
  if (!GRID1D)
    for (int k = 0; k < NFLD; ++k) put(k, cplx{0.0, 0.0});
  // spin-diagonal fields, sigma = +1 (index 0) and -1 (index 1)
  for (int si = 0; si < 2; ++si) {
    const double sg = si == 0 ? 1.0 : -1.0;
    put(mf_index(0, 0, si, si), 2.0 * crho * rho + ctau * tau + sg * (2.0 * cs * sz + ct * tz + cf * fz));
    const cplx b01 = -crdj * (tjpz - tjzp) - sg * csdj * jp;
    const cplx x01 = sg * mul_i(c1a - 0.5 * c2a) - mul_i(cj * jr);
    put(mf_index(0, 1, si, si), b01 + x01);
    put(mf_index(1, 0, si, si), b01 - x01);
    const cplx b02 = cj * jp + sg * (c1b + 0.5 * c2b);
    const cplx x02 = sg * mul_i(csdj * jr) - mul_i(crdj * (tjzr - tjrz));
    put(mf_index(0, 2, si, si), b02 + x02);
    put(mf_index(2, 0, si, si), b02 - x02);
    const cplx b03 = -crdj * (tjrp - tjpr) + 2.0 * sg * cgs * gs;
    const cplx x03 = -sg * mul_i(c0 - (ctj2 / 3.0) * (tjrr + tjpp - 2.0 * tjzz)) - mul_i(cj * jz);
    put(mf_index(0, 3, si, si), b03 + x03);
    put(mf_index(3, 0, si, si), b03 - x03);
    const cplx f04 = 2.0 * cdrho * rho + 2.0 * sg * cds * sz;
    put(mf_index(0, 4, si, si), f04);
    if (!GRID1D) put(mf_index(4, 0, si, si), f04);
    const cplx f12 = csdj * sz + sg * crdj * rho;
    put(mf_index(1, 2, si, si), f12);
    if (!GRID1D) put(mf_index(2, 1, si, si), f12);
    put(mf_index(1, 3, si, si), sg * 0.5 * cf * sr + mul_i(csdj * sp));
    put(mf_index(3, 1, si, si), sg * 0.5 * cf * sr - mul_i(csdj * sp));
    put(mf_index(2, 3, si, si), -csdj * sr - sg * mul_i(0.5 * cf * sp));
    put(mf_index(3, 2, si, si), -csdj * sr + sg * mul_i(0.5 * cf * sp));
    const cplx f11 = (4.0 * cdrho + ctau) * rho + sg * (4.0 * cds + ct) * sz;
    put(mf_index(1, 1, si, si), f11);
    put(mf_index(2, 2, si, si), f11);
    put(mf_index(3, 3, si, si), f11 + sg * cf * sz);
  }
  // spin-flip fields: (sa, sb) = (up, down) eps = +1, (down, up) eps = -1
  const cplx a2 = -ctj1 * (tjrp - tjpr);
  const cplx a3 = -1.0 * mul_i(c0);
  const cplx a4 = -0.5 * ctj2 * (tjrp + tjpr);
  const cplx a5 = mul_i((ctj2 / 3.0) * (-2.0 * tjrr + tjpp + tjzz));
  const cplx a6 = mul_i((ctj2 / 3.0) * (tjrr - 2.0 * tjpp + tjzz));
  for (int k = 0; k < 2; ++k) {
    const int sa = k, sb = 1 - k;
    const double e = k == 0 ? 1.0 : -1.0;
    put(mf_index(0, 0, sa, sb), (2.0 * cs * sr + ct * tr + cf * fr) - e * mul_i(2.0 * cs * sp + ct * tp + cf * fp));
    const cplx g = 2.0 * cgs * gs;
    const cplx iz = mul_i(csdj * jz);
    put(mf_index(0, 1, sa, sb), g - e * iz + e * a2 + a3 + e * a4 + a5);
    put(mf_index(1, 0, sa, sb), g - e * iz - e * a2 - a3 - e * a4 - a5);
    put(mf_index(0, 2, sa, sb), e * g - iz + a2 + e * a3 - a4 + e * a6);
    put(mf_index(2, 0, sa, sb), -e * g + iz + a2 + e * a3 - a4 + e * a6);
    const cplx b3 = csdj * jp + e * mul_i(csdj * jr);
    put(mf_index(0, 3, sa, sb), b3 - mul_i(c1a + 0.5 * c2a) + e * (c1b - 0.5 * c2b));
    put(mf_index(3, 0, sa, sb), b3 + mul_i(c1a + 0.5 * c2a) - e * (c1b - 0.5 * c2b));
    const cplx f04 = 2.0 * cds * (sr - e * mul_i(sp));
    put(mf_index(0, 4, sa, sb), f04);
    if (!GRID1D) put(mf_index(4, 0, sa, sb), f04);
    const cplx f12 = mul_i(0.5 * cf * sp) + e * 0.5 * cf * sr;
    put(mf_index(1, 2, sa, sb), f12);
    if (!GRID1D) put(mf_index(2, 1, sa, sb), -1.0 * f12);
    put(mf_index(1, 3, sa, sb), 0.5 * cf * sz + e * crdj * rho);
    put(mf_index(3, 1, sa, sb), 0.5 * cf * sz - e * crdj * rho);
    put(mf_index(2, 3, sa, sb), -e * 0.5 * cf * sz - crdj * rho);
    put(mf_index(3, 2, sa, sb), e * 0.5 * cf * sz - crdj * rho);
    const cplx f33 = (ct + 4.0 * cds) * (sr - e * mul_i(sp));
    put(mf_index(3, 3, sa, sb), f33);
    put(mf_index(1, 1, sa, sb), f33 + cf * sr);
    put(mf_index(2, 2, sa, sb), f33 - e * mul_i(cf * sp));
  }
  // pairing fields P(sa, sb) (pnfam_hamiltonian_blas.f90:1200-1208)
  put(100 + 0, cspair * (sbr - mul_i(sbp)));             // (up, up)
  put(100 + 1, -cpair * rb - cspair * sbz);              // (down, up)
  put(100 + 2, cpair * rb - cspair * sbz);               // (up, down)
  put(100 + 3, cspair * (-1.0 * sbr - mul_i(sbp)));      // (down, down)
}

#include "mixed.hpp"

struct Tile {        // output tile of one block of a projected matrix
  int32_t ix, iy, off, sec;   // row block, col block, element offset, sector
  int32_t a0, b0, na, nb_;    // tile origin / size inside the block
  int32_t out_slot, kind, pad0, pad1;   // kind 0: mean field (5 psi), 1: pairing (psi only)
};
static_assert(sizeof(Tile) == 48, "Tile layout");

struct ProjArgs {
  const double *psi[5];   // wf, wfdr, wfdp, wfdz, wfd2_all
  const int *isstart, *db, *nsu, *ns;
  const double *flds;     // [w][2][208][nghl]
  double *hsp;            // [w][8][nxy]
  double *part;           // k_project_mfma split over grid points: [split][active index][8][nxy]; null: hsp
  long nxy;
  int nghl;
  const Tile *tiles;
  const int *act;
  int na;                 // active frequencies (k_project_mfma: the last group may be partial)
  int skip = -1;          // as DensArgs::skip (a group of frequencies returns when its first is it)
};

constexpr int PT = 32;   // tile edge
constexpr int PR = 8;    // grid points per LDS chunk

// h_ab = 2 sum_r sum_z psi_z(r,a) hpsi_z^{s_a}(r,b),
// hpsi_z^{s_a}(r,b) = sum_z' mf(z,z',s_a,s_b)(r) psi_z'(r,b)      (:1105-1167)
// Delta_ab = 2 sum_r psi_0(r,a) P_{s_a s_b}(r) psi_0(r,b)        (:1210-1260)
__global__ void __launch_bounds__(256) k_project(ProjArgs P) {
  __shared__ double sA[5][PR][PT];
  __shared__ double sH[5][2][2][PR][PT];  // [z][s_a][re/im][r][b]
  const Tile t = P.tiles[blockIdx.x];
  const int w = P.act[blockIdx.y];
  if (w == P.skip) return;
  const int G = P.nghl;
  const int ia = P.isstart[t.ix] + t.a0, ib = P.isstart[t.iy] + t.b0;
  const int nsu = P.nsu[t.ix];
  const int nz = t.kind == 0 ? 5 : 1;
  const double *fl = P.flds + (((size_t)w * 2 + t.sec) * 2 * NFLD) * G;
  // each thread owns 4 output elements: (a = tid%32, b = tid/32 + 8k)
  const int ta = threadIdx.x % PT, tb0 = threadIdx.x / PT;
  double accr[4] = {0, 0, 0, 0}, acci[4] = {0, 0, 0, 0};
  const int sa_own = (t.a0 + ta) < nsu ? 0 : 1;
  for (int r0 = 0; r0 < G; r0 += PR) {
    // stage psi_z(r, a)
    for (int e = threadIdx.x; e < nz * PR * PT; e += 256) {
      const int a = e % PT, rr = (e / PT) % PR, z = e / (PT * PR);
      const int r = r0 + rr;
      sA[z][rr][a] = (a < t.na && r < G) ? P.psi[z][(size_t)(ia + a) * G + r] : 0.0;
    }
    // hpsi for (rr, b): one pair per thread
    {
      const int b = threadIdx.x % PT, rr = threadIdx.x / PT;
      const int r = r0 + rr;
      if (b < t.nb_ && r < G) {
        const size_t ob = (size_t)(ib + b) * G + r;
        const int sb = P.ns[ib + b] > 0 ? 0 : 1;
        if (t.kind == 0) {
          double pv[5];
#pragma unroll
          for (int z = 0; z < 5; ++z) pv[z] = P.psi[z][ob];
#pragma unroll
          for (int sa = 0; sa < 2; ++sa)
#pragma unroll
            for (int z = 0; z < 5; ++z) {
              double hr = 0.0, hi = 0.0;
#pragma unroll
              for (int zp = 0; zp < 5; ++zp) {
                const int idx = mf_index(z, zp, sa, sb);
                hr += fl[(size_t)(2 * idx) * G + r] * pv[zp];
                hi += fl[(size_t)(2 * idx + 1) * G + r] * pv[zp];
              }
              sH[z][sa][0][rr][b] = hr;
              sH[z][sa][1][rr][b] = hi;
            }
        } else {
          const double p0 = P.psi[0][ob];
#pragma unroll
          for (int sa = 0; sa < 2; ++sa) {
            const int idx = 100 + (sb == 0 ? (sa == 0 ? 0 : 1) : (sa == 0 ? 2 : 3));
            sH[0][sa][0][rr][b] = fl[(size_t)(2 * idx) * G + r] * p0;
            sH[0][sa][1][rr][b] = fl[(size_t)(2 * idx + 1) * G + r] * p0;
          }
        }
      } else {
        for (int z = 0; z < nz; ++z)
          for (int sa = 0; sa < 2; ++sa) { sH[z][sa][0][rr][b] = 0.0; sH[z][sa][1][rr][b] = 0.0; }
      }
    }
    __syncthreads();
    for (int k = 0; k < 4; ++k) {
      const int b = tb0 + 8 * k;
      double hr = 0.0, hi = 0.0;
      for (int z = 0; z < nz; ++z)
#pragma unroll
        for (int rr = 0; rr < PR; ++rr) {
          const double a = sA[z][rr][ta];
          hr += a * sH[z][sa_own][0][rr][b];
          hi += a * sH[z][sa_own][1][rr][b];
        }
      accr[k] += hr;
      acci[k] += hi;
    }
    __syncthreads();
  }
  const int dx = P.db[t.ix];
  double *ore = P.hsp + ((size_t)w * 8 + 2 * t.out_slot) * P.nxy + t.off;
  double *oim = ore + P.nxy;
  for (int k = 0; k < 4; ++k) {
    const int b = tb0 + 8 * k;
    if (ta < t.na && b < t.nb_) {
      const size_t o = (size_t)(t.a0 + ta) + (size_t)(t.b0 + b) * dx;
      ore[o] = 2.0 * accr[k];
      oim[o] = 2.0 * acci[k];
    }
  }
}

struct Tile2 {        // one wave's output of a projected matrix: rows of one spin, 16 columns
  int32_t ix, iy, off, sec;
  int32_t a_lo, a_hi, sa, b0;     // row range inside block ix (single spin sa), column tile origin
  int32_t out_slot, kind, pad0, pad1;
};
static_assert(sizeof(Tile2) == 48, "Tile2 layout");

constexpr int P2_MAXRT = 4;   // row tiles of 16 per wave
// FP64 density and projection with few frequencies: splits of the serial loop
// (pairs, grid points) per frequency, and the most (split, frequency) partial
// outputs they write
constexpr int FEW_SPLIT_SLABS = 32;
inline int few_split(int na) { return na <= 4 ? 8 : (na <= 8 ? 4 : 1); }

// h_ab / Delta_ab with FP64 MFMA: D[a][b] = sum_{z,r} psi_z(r,a) B_z(r,b), with
// B_z(r,b) = sum_z' mf(z,z',s_a,s_b)(r) psi_z'(r,b) built in registers from
// fields staged in LDS per 16 grid points (KIND 1: B = P_{s_a s_b}(r) psi_0(r,b)).
// Rows: NRT x 16 states of spin s_a of block ix; columns: 16 states of block iy.
// Instantiated per (NRT, KIND) with tiles sorted accordingly on the host, so the
// row-tile and table loops carry no branches.  The fields are staged with the
// grid point fastest across lanes (128-byte reads) and no integer division.
// Grid (tile, frequency), tiles fastest.  Ordering frequencies fastest within
// an XCD (so a tile's psi rows are fetched once per L2) cut the HBM fetch 4x
// but ran 1.4x slower: the kernel is not bound by HBM traffic.
// With few frequencies a third grid dimension splits the grid points: split z
// takes the 16-point chunks [z n / Z, (z + 1) n / Z) and writes its partial
// tile to P.part, and k_proj_sum adds the splits in order.  With one split the
// loop and the output are those of the unsplit kernel.
// (z, z') pairs of the mean field that are not identically zero
// (pnfam_hamiltonian_blas.f90:774-1093): z = 0 couples to z' = 0..4, z = 1..3 to
// z' = 0..3, z = 4 to z' = 0; numbered in (z, z') order
__host__ __device__ constexpr int mf_zp_count(int z) { return z == 0 ? 5 : (z == 4 ? 1 : 4); }
__host__ __device__ constexpr int mf_zp_first(int z) { return z == 0 ? 0 : (z == 4 ? 17 : 5 + 4 * (z - 1)); }
constexpr int MF_NZP = 18;

// h_ab / Delta_ab with FP64 MFMA: D[a][b] = sum_{z,r} psi_z(r,a) B_z(r,b), with
// B_z(r,b) = sum_z' mf(z,z',s_a,s_b)(r) psi_z'(r,b) built in registers from
// fields staged in LDS per 16 grid points (KIND 1: B = P_{s_a s_b}(r) psi_0(r,b)).
// Rows: NRT x 16 states of spin s_a of block ix; columns: 16 states of block iy.
// One wave computes the tile for NF frequencies (active indices NF y .. NF y +
// NF - 1): the psi operands, which do not depend on the frequency, are loaded
// once per k step for all of them, and each frequency builds its own B from
// its staged fields.  Instantiated per (NRT, KIND, NF) with tiles sorted on the
// host, so the row-tile and table loops carry no branches.  The operands of the
// next k step are loaded before the products of the current one.
// Grid (tile, frequency group, split), tiles fastest.  With few frequencies the
// third grid dimension splits the grid points: split z takes the 16-point
// chunks [z n / Z, (z + 1) n / Z) and writes its partial tile to P.part, which
// k_proj_sum adds in order.  With one split the output is the unsplit kernel's,
// and every output element is summed in the same order whatever NRT and NF.
// NS: depth of the operand pipeline (the loads of NS k steps ahead are in
// flight while the products of one run); the sums keep their order.
template <int NRT, int KIND, int NF, int NS>
__global__ void __launch_bounds__(64) k_project_mfma(ProjArgs P, const Tile2 *__restrict__ tiles) {
  static_assert(4 % NS == 0, "a 16-point chunk holds 4 k steps");
  constexpr int NZ = KIND == 0 ? 5 : 1;
  constexpr int NC = KIND == 0 ? MF_NZP : 1;
  __shared__ double sMF[NF][16][2][NC][2];     // [frequency][r][s_b][(z, z') pair][ri]
  const Tile2 t = tiles[blockIdx.x];
  if (P.act[blockIdx.y * NF] == P.skip) return;   // the group's slots are all the spare one
  const int G = P.nghl;
  const int lane = threadIdx.x;
  const int mi = lane & 15, mk = lane >> 4;
  const int ia = P.isstart[t.ix], ib0 = P.isstart[t.iy];
  const int dx = P.db[t.ix], dy = P.db[t.iy];
  const int nrows = t.a_hi - t.a_lo;
  int wf[NF];
  bool fon[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int y = blockIdx.y * NF + f;
    fon[f] = y < P.na;
    wf[f] = P.act[fon[f] ? y : blockIdx.y * NF];
  }
  const int bj = t.b0 + mi;             // this lane's B column
  const bool bcol = bj < dy;
  const int sb = bcol ? (P.ns[ib0 + bj] > 0 ? 0 : 1) : 0;
  v4d C[NF][NRT][2];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int q = 0; q < NRT; ++q) { C[f][q][0] = v4d{0, 0, 0, 0}; C[f][q][1] = v4d{0, 0, 0, 0}; }
  const int nch = (G + 15) / 16;
  const int c0 = (int)((long)blockIdx.z * nch / gridDim.z), c1 = (int)((long)(blockIdx.z + 1) * nch / gridDim.z);
  const int rend = 16 * c1;
  // operands of the k step at grid point r (this lane's k index): psi_z'(r, b)
  // of its column and psi_z(r, a) of its rows, zero outside the blocks and the grid
  auto load = [&](int r, double (&pz)[NZ], double (&av)[NRT][NZ]) {
    const bool rok = r < G;
    const size_t ob = (size_t)(ib0 + (bcol ? bj : 0)) * G + (rok ? r : 0);
#pragma unroll
    for (int z = 0; z < NZ; ++z) pz[z] = (bcol && rok) ? P.psi[z][ob] : 0.0;
#pragma unroll
    for (int q = 0; q < NRT; ++q) {
      const int arow = q * 16 + mi;
      const bool aok = arow < nrows && rok;
      const size_t oa = (size_t)(ia + t.a_lo + (aok ? arow : 0)) * G + (rok ? r : 0);
#pragma unroll
      for (int z = 0; z < NZ; ++z) av[q][z] = aok ? P.psi[z][oa] : 0.0;
    }
  };
  double pzs[NS][NZ], avs[NS][NRT][NZ];
#pragma unroll
  for (int s = 0; s < NS; ++s) load(16 * c0 + 4 * s + mk, pzs[s], avs[s]);
  for (int rc = 16 * c0; rc < rend; rc += 16) {
    // stage each frequency's fields of 16 grid points for this spin of a;
    // lanes run along r
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const double *fl = P.flds + (((size_t)wf[f] * 2 + t.sec) * 2 * NFLD) * G;
      if (KIND == 0) {
        for (int e = lane; e < 16 * 2 * NC * 2; e += 64) {
          const int rr = e & 15, q = e >> 4, ri = q & 1, jz = q >> 1;   // jz = s_b * NC + pair
          const int sbb = jz >= NC ? 1 : 0, cc = jz - NC * sbb;
          const int z = cc >= 17 ? 4 : (cc >= 5 ? 1 + (cc - 5) / 4 : 0);
          const int zp = cc >= 17 ? 0 : (cc >= 5 ? (cc - 5) % 4 : cc);
          const int r = rc + rr;
          const int idx = mf_index(z, zp, t.sa, sbb);
          sMF[f][rr][sbb][cc][ri] = r < G ? fl[(size_t)(2 * idx + ri) * G + r] : 0.0;
        }
      } else {
        for (int e = lane; e < 16 * 2 * 2; e += 64) {
          const int rr = e & 15, ri = (e >> 4) & 1, sbb = e >> 5;
          const int r = rc + rr;
          const int idx = 100 + (sbb == 0 ? (t.sa == 0 ? 0 : 1) : (t.sa == 0 ? 2 : 3));
          sMF[f][rr][sbb][0][ri] = r < G ? fl[(size_t)(2 * idx + ri) * G + r] : 0.0;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int kc = 0; kc < 16; kc += 4) {
      const int st = (kc / 4) % NS;   // static after unrolling
      double pz[NZ], av[NRT][NZ];
#pragma unroll
      for (int z = 0; z < NZ; ++z) pz[z] = pzs[st][z];
#pragma unroll
      for (int q = 0; q < NRT; ++q)
#pragma unroll
        for (int z = 0; z < NZ; ++z) av[q][z] = avs[st][q][z];
      if (rc + kc + 4 * NS < rend) load(rc + kc + 4 * NS + mk, pzs[st], avs[st]);
      const int rr = kc + mk;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        // B operand (k = r, column bj): B_z = sum_z' mf * psi_z'(r, b)
        double Bre[NZ], Bim[NZ];
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
          double br = 0.0, bi = 0.0;
#pragma unroll
          for (int k = 0; k < (KIND == 0 ? mf_zp_count(z) : 1); ++k) {
            const int cc = KIND == 0 ? mf_zp_first(z) + k : 0;
            const int zp = KIND == 0 ? (z == 4 ? 0 : k) : 0;
            br += sMF[f][rr][sb][cc][0] * pz[zp];
            bi += sMF[f][rr][sb][cc][1] * pz[zp];
          }
          Bre[z] = br;
          Bim[z] = bi;
        }
        // z outer: consecutive products go to 2 NRT different accumulators, so a
        // product does not wait for the one before it (each accumulator still
        // adds z = 0..NZ-1 in order)
#pragma unroll
        for (int z = 0; z < NZ; ++z)
#pragma unroll
          for (int q = 0; q < NRT; ++q) {
            C[f][q][0] = mfma64(av[q][z], Bre[z], C[f][q][0]);
            C[f][q][1] = mfma64(av[q][z], Bim[z], C[f][q][1]);
          }
      }
    }
    __syncthreads();
  }
  const int bcolo = t.b0 + (lane & 15);
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    if (!fon[f]) continue;
    const int y = blockIdx.y * NF + f;
    double *obase = P.part ? P.part + ((size_t)blockIdx.z * P.na + y) * 8 * P.nxy : P.hsp + (size_t)wf[f] * 8 * P.nxy;
    double *ore = obase + (size_t)(2 * t.out_slot) * P.nxy + t.off;
    double *oim = ore + P.nxy;
#pragma unroll
    for (int q = 0; q < NRT; ++q) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int arow = q * 16 + 4 * v + (lane >> 4);
        if (arow < nrows && bcolo < dy) {
          const size_t o = (size_t)(t.a_lo + arow) + (size_t)bcolo * dx;
          ore[o] = 2.0 * C[f][q][0][v];
          oim[o] = 2.0 * C[f][q][1][v];
        }
      }
    }
  }
}

// h_ab / Delta_ab for four frequencies per workgroup, the psi operands shared
// through LDS: wave v computes the tile of active frequency 4 y + v, as
// k_project_mfma<NRT, KIND, 1, .> does, but the rows psi_z(r, a) of the tile and
// the columns psi_z'(r, b), which do not depend on the frequency, are loaded
// once per 16-point chunk by all 256 threads (coalesced along r) into LDS, and
// the loads of the next chunk are in flight in registers while the products of
// the current one run.  Every output element is summed in the order of
// k_project_mfma (chunks, k steps of 4 points, z), so the results are bitwise
// the same.  Used with four or more active frequencies and no grid split.
template <int NRT, int KIND>
__global__ void __launch_bounds__(256) k_project_lds(ProjArgs P, const Tile2 *__restrict__ tiles) {
  constexpr int NZ = KIND == 0 ? 5 : 1;
  constexpr int NC = KIND == 0 ? MF_NZP : 1;
  constexpr int NR = 16 * NRT;              // tile rows
  constexpr int NS = NR + 16;               // staged states: rows, then the 16 columns
  constexpr int NSTG = NZ * NS * 16;        // staged values per chunk
  constexpr int PER = (NSTG + 255) / 256;   // per thread
  // [z][state slot][chunk point rr ^ (slot & 15)]: the XOR swizzle spreads the
  // 16 rows a wave reads at one rr over distinct LDS banks
  __shared__ double sPsi[NZ][NS][16];
  __shared__ double sMF[4][16][2][NC][2];   // [wave][r][s_b][(z, z') pair][ri]
  const Tile2 t = tiles[blockIdx.x];
  if (P.act[blockIdx.y * 4] == P.skip) return;    // the group's slots are all the spare one
  const int G = P.nghl;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int mi = lane & 15, mk = lane >> 4;
  const int ia = P.isstart[t.ix], ib0 = P.isstart[t.iy];
  const int dx = P.db[t.ix], dy = P.db[t.iy];
  const int nrows = t.a_hi - t.a_lo;
  const int y = blockIdx.y * 4 + wave;
  const bool fon = y < P.na;
  const int w = P.act[fon ? y : blockIdx.y * 4];
  const int bj = t.b0 + mi;
  const bool bcol = bj < dy;
  const int sb = bcol ? (P.ns[ib0 + bj] > 0 ? 0 : 1) : 0;
  const double *fl = P.flds + (((size_t)w * 2 + t.sec) * 2 * NFLD) * G;
  v4d C[NRT][2];
#pragma unroll
  for (int q = 0; q < NRT; ++q) { C[q][0] = v4d{0, 0, 0, 0}; C[q][1] = v4d{0, 0, 0, 0}; }
  // staged value i of this thread: chunk point rr = tid & 15, state slot
  // s = ((tid >> 4) + 16 i) % NS, table z = ((tid >> 4) + 16 i) / NS; the
  // clamped addresses stay inside the tables and the selects zero what lies
  // outside the tile or the grid
  const int rr_own = tid & 15;
  double stg[PER];
  auto gload = [&](int rc) {
    const int r = rc + rr_own;
    const bool rok = r < G;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int q = (tid >> 4) + 16 * i;
      const int z = q / NS, s = q - z * NS;
      bool ok = rok && z < NZ;
      int st;
      if (s < NR) { ok = ok && s < nrows; st = ia + t.a_lo + (ok ? s : 0); }
      else { ok = ok && t.b0 + (s - NR) < dy; st = ib0 + t.b0 + (ok ? s - NR : 0); }
      const double v = P.psi[z < NZ ? z : 0][(size_t)st * G + (rok ? r : 0)];
      stg[i] = ok ? v : 0.0;
    }
  };
  auto sstore = [&]() {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int q = (tid >> 4) + 16 * i;
      const int z = q / NS, s = q - z * NS;
      if (z < NZ) sPsi[z][s][rr_own ^ (s & 15)] = stg[i];
    }
  };
  const int rend = G;
  gload(0);
  for (int rc = 0; rc < rend; rc += 16) {
    sstore();
    // this wave's fields of the chunk (as k_project_mfma stages them)
    if (KIND == 0) {
      for (int e = lane; e < 16 * 2 * NC * 2; e += 64) {
        const int rr = e & 15, q = e >> 4, ri = q & 1, jz = q >> 1;
        const int sbb = jz >= NC ? 1 : 0, cc = jz - NC * sbb;
        const int z = cc >= 17 ? 4 : (cc >= 5 ? 1 + (cc - 5) / 4 : 0);
        const int zp = cc >= 17 ? 0 : (cc >= 5 ? (cc - 5) % 4 : cc);
        const int r = rc + rr;
        const int idx = mf_index(z, zp, t.sa, sbb);
        sMF[wave][rr][sbb][cc][ri] = r < G ? fl[(size_t)(2 * idx + ri) * G + r] : 0.0;
      }
    } else {
      for (int e = lane; e < 16 * 2 * 2; e += 64) {
        const int rr = e & 15, ri = (e >> 4) & 1, sbb = e >> 5;
        const int r = rc + rr;
        const int idx = 100 + (sbb == 0 ? (t.sa == 0 ? 0 : 1) : (t.sa == 0 ? 2 : 3));
        sMF[wave][rr][sbb][0][ri] = r < G ? fl[(size_t)(2 * idx + ri) * G + r] : 0.0;
      }
    }
    __syncthreads();
    if (rc + 16 < rend) gload(rc + 16);   // in flight during the products below
#pragma unroll
    for (int kc = 0; kc < 16; kc += 4) {
      const int rr = kc + mk;
      double pz[NZ];
#pragma unroll
      for (int z = 0; z < NZ; ++z) pz[z] = sPsi[z][NR + mi][rr ^ mi];
      double Bre[NZ], Bim[NZ];
#pragma unroll
      for (int z = 0; z < NZ; ++z) {
        double br = 0.0, bi = 0.0;
#pragma unroll
        for (int k = 0; k < (KIND == 0 ? mf_zp_count(z) : 1); ++k) {
          const int cc = KIND == 0 ? mf_zp_first(z) + k : 0;
          const int zp = KIND == 0 ? (z == 4 ? 0 : k) : 0;
          br += sMF[wave][rr][sb][cc][0] * pz[zp];
          bi += sMF[wave][rr][sb][cc][1] * pz[zp];
        }
        Bre[z] = br;
        Bim[z] = bi;
      }
#pragma unroll
      for (int z = 0; z < NZ; ++z)
#pragma unroll
        for (int q = 0; q < NRT; ++q) {
          const double av = sPsi[z][q * 16 + mi][rr ^ mi];
          C[q][0] = mfma64(av, Bre[z], C[q][0]);
          C[q][1] = mfma64(av, Bim[z], C[q][1]);
        }
    }
    __syncthreads();
  }
  if (!fon) return;
  double *obase = P.hsp + (size_t)w * 8 * P.nxy;
  double *ore = obase + (size_t)(2 * t.out_slot) * P.nxy + t.off;
  double *oim = ore + P.nxy;
#pragma unroll
  for (int q = 0; q < NRT; ++q) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int arow = q * 16 + 4 * v + (lane >> 4);
      if (arow < nrows && bj < dy) {
        const size_t o = (size_t)(t.a_lo + arow) + (size_t)bj * dx;
        ore[o] = 2.0 * C[q][0][v];
        oim[o] = 2.0 * C[q][1][v];
      }
    }
  }
}

// hsp of the active frequency y = the sum of its nsplit partial projections,
// split by split (k_project_mfma with a split grid)
__global__ void k_proj_sum(const double *__restrict__ part, int nsplit, int na, long n8, const int *__restrict__ act,
                           double *__restrict__ hsp) {
  const int y = blockIdx.y;
  double *out = hsp + (size_t)act[y] * n8;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n8; e += (long)gridDim.x * blockDim.x) {
    double v = 0.0;
    for (int s = 0; s < nsplit; ++s) v += part[((size_t)s * na + y) * n8 + e];
    out[e] = v;
  }
}

#include "factored.hpp"
#include "separable.hpp"

struct GreenArgs {
  const double *hqp;     // [w][4][nxy]
  const double *f20, *f02;
  const double *e1, *e2; // row / column qp energies (Ep,En for beta-)
  const int *xrow, *xcol, *yrow, *ycol;
  const double *wre, *wim;   // per frequency
  double *vout;          // [w][4][nxy]
  long nxy;
  double quench;
  int use_h;
  const int *act;
  int skip = -1;         // as DensArgs::skip
};

// X = g_X (F20 + q H20), Y = g_Y (F02 + q H02), g = -1/(E1_i + E2_j -+ w)
// (pnfam_solver.f90:169-179, matrix_2qp :510-544)
__global__ void k_green(GreenArgs A) {
  const int w = A.act[blockIdx.y];
  if (w == A.skip) return;
  const long n = A.nxy;
  const double wr = A.wre[w], wi = A.wim[w];
  const double *h = A.hqp + (size_t)w * 4 * n;
  double *v = A.vout + (size_t)w * 4 * n;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < 2 * n; e += (long)gridDim.x * blockDim.x) {
    const bool isx = e < n;
    const long k = isx ? e : e - n;
    // quench the induced field, then add the (real) external field (:169-175)
    const double f = isx ? A.f20[k] : A.f02[k];
    const double hr = A.use_h ? A.quench * h[(isx ? 0 : n) + k] + f : f;
    const double hi = A.use_h ? A.quench * h[(isx ? 2 * n : 3 * n) + k] : 0.0;
    const double E = isx ? A.e1[A.xrow[k]] + A.e2[A.xcol[k]] : A.e1[A.yrow[k]] + A.e2[A.ycol[k]];
    // x = E -+ w ; g = -1/x
    const double xr = isx ? E - wr : E + wr;
    const double xi = isx ? -wi : wi;
    const double den = xr * xr + xi * xi;
    const double gr = -xr / den, gi = xi / den;
    v[(isx ? 0 : n) + k] = gr * hr - gi * hi;
    v[(isx ? 2 * n : 3 * n) + k] = gi * hr + hi * gr;
  }
}

// ---- mixed path: the hamiltonian is linear in vin, so H(vin_k) is carried as
// an FP64 sum of H applied to the increments vin_k - vin_{k-1}; the increment
// is the step the Broyden update adds (k_bro_update writes it) --------------
// hacc = hqp (set != 0, a full evaluation) or hacc += hqp (an increment)
__global__ void k_hacc(double *__restrict__ hacc, const double *__restrict__ hqp, long n, int set,
                       const int *__restrict__ act) {
  const size_t w = act[blockIdx.y];
  double *a = hacc + w * n;
  const double *b = hqp + w * n;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    a[e] = set ? b[e] : a[e] + b[e];
}

// ---- Broyden (pnfam_broyden.f90:117-216), per frequency, FP64 ---------------
constexpr int BRO_WG = 256;
constexpr int BRO_NWG_FEW = 1024;   // workgroups per point of the FP32-history kernels with few points
constexpr int BRO_FEW = 8;          // "few": at most this many active points
constexpr int BRO_MAXM = 64;

struct BroArgs {
  double *vin, *vout;     // [w][N]
  void *df, *dv;          // history [w][M][N]: double, or float on the mixed path
  double *pdf;            // float history: the pending raw vout [w][N] (FP64)
  double *part;           // [w][nwg][2*M+2]
  double *gram;           // [w][M][M]
  double *coef;           // [w][M] gamma
  double *si;             // [w]
  double *vmax;           // [w] max |vin|
  double *scal;           // [w][4]: normi, ...
  double *dvin;           // mixed path: [w][N] the step added to vin (the next increment); null for FP64
  const int *drop;        // [w] 1: this iteration's history pair is zeroed (mixed refinement); null: none
  long N;
  int M, nwg, iter, ipos, inext, iter_used;
  double alpha;
  const int *act;
  const int *iterp;       // graph replay: the iteration is iterp[0] in device memory; null: iter above
  const int *lag;         // [w] iterations point w has waited for its refinement group: its own
                          // iteration is the batch's less lag[w]; null: none waited
  int skip = -1;          // as DensArgs::skip
};

// The iteration-dependent fields of point w (Broyden steps with a history:
// M > 0, iteration >= 1), with the host's formulas, when they are not the ones
// the host set: the iteration read from device memory (graph replay), less the
// iterations the point waited for its refinement group.
__device__ inline void bro_iter(BroArgs &B, int w) {
  if (!B.iterp && !B.lag) return;
  const int it = (B.iterp ? B.iterp[0] : B.iter) - (B.lag ? B.lag[w] : 0), M = B.M;
  B.iter = it;
  B.iter_used = min(it - 1, M);
  B.ipos = it < 2 ? 0 : (it - 1 - ((it - 2) / M) * M) - 1;
  B.inext = (it - ((it - 1) / M) * M) - 1;
}

// Partial sums of the Broyden reductions, value-major so that the readers'
// lanes load consecutive workgroups: part[(w * (2 BRO_MAXM + 2) + i) * nwg + q]
// for workgroup q; i = 0 max|vout|, 1 |df|^2, 2 max|vin| (resid, norm), then
// 2 + 2 j, 3 + 2 j the dots of history entry j (dots, solve; slot 2 is reused).
__device__ inline double *bro_part(const BroArgs &B, int w, int i, int q) {
  return B.part + ((size_t)w * (2 * BRO_MAXM + 2) + i) * B.nwg + q;
}

__device__ inline double wg_sum(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64;
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int k = 0; k < (int)(blockDim.x / 64); ++k) s += red[k];
  return s;  // valid on thread 0
}
__device__ inline double wg_max(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64;
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int k = 0; k < (int)(blockDim.x / 64); ++k) s = fmax(s, red[k]);
  return s;
}

// ifam's exit tests on the device, for the graph replay of the FP64 iteration
// (pnfam_solver.f90:93-221): a point not yet done stops as converged (si below
// the tolerance; its iteration count is the iteration index) or interrupted
// (at max_iter; -1), or stays active.  The active points go to act in ascending
// order, the remaining of the nslots entries to the spare slot `dummy`, whose
// results nothing reads.  ctl[2] is the iteration to run: ctl[0] = active
// count, ctl[1] = this iteration (read by the Broyden kernels), ctl[2] += 1;
// ctl[3] = 1 flags more active points than slots.
__global__ void __launch_bounds__(1024) k_select(const double *__restrict__ si, int *__restrict__ done,
                                                int *__restrict__ iters, int *__restrict__ act, int *ctl, int npts,
                                                int nslots, double eps, int max_iter, int dummy) {
  __shared__ int wsum[16];
  __shared__ int base;
  const int it = ctl[2];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (threadIdx.x == 0) base = 0;
  __syncthreads();
  for (int w0 = 0; w0 < npts; w0 += 1024) {
    const int w = w0 + threadIdx.x;
    int a = 0;
    if (w < npts && !done[w]) {
      if (si[w] < eps) { done[w] = 1; iters[w] = it; }
      else if (it >= max_iter) { done[w] = 1; iters[w] = -1; }
      else a = 1;
    }
    const unsigned long long m = __ballot(a);
    const int pre = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wsum[wv] = __popcll(m);
    __syncthreads();
    int off = 0, tot = 0;
    for (int k = 0; k < 16; ++k) {
      off += k < wv ? wsum[k] : 0;
      tot += wsum[k];
    }
    const int pos = base + off + pre;
    if (a && pos < nslots) act[pos] = w;
    __syncthreads();
    if (threadIdx.x == 0) base += tot;
    __syncthreads();
  }
  const int n = base;
  for (int i = n + threadIdx.x; i < nslots; i += blockDim.x) act[i] = dummy;
  if (threadIdx.x == 0) {
    ctl[0] = n < nslots ? n : nslots;
    ctl[1] = it;
    ctl[2] = n > 0 ? it + 1 : it;   // with none active it stays the iteration that found them done
    if (n > nslots) ctl[3] = 1;
  }
}

// vout <- vout - vin; partial max|vout|; for iter >= 2 also the partial squared
// norm of the history difference at slot ipos, which an FP64 history forms again
// in k_bro_dots (from values that kernel reads anyway), so that nothing but vout
// is written here.
// H: element type of the history (double; float on the mixed path, whose
// pending raw vout stays FP64 in pdf, so the residual difference is formed
// exactly, and whose dv is the step the last update wrote to dvin).
// The Broyden kernels of an FP64 history run at the memory's rate (4.8 to 5.2 TB/s
// at 128 points, a large copy 4.9): up to 8 pairs k, 4 + (k + 6) + (k + 5) vectors
// of 4 nxy pass per iteration in resid, dots and update (7 + (k + 8) + (k + 5) with
// the difference written here; N_sh = 16, 128 points, this kernel 617 -> 337 us).
template <class H>
__global__ void __launch_bounds__(BRO_WG) k_bro_resid(BroArgs B) {
  constexpr bool f64 = sizeof(H) == 8;
  __shared__ double red[BRO_WG / 64];
  const int w = B.act[blockIdx.y];
  if (w == B.skip) return;
  bro_iter(B, w);
  const long N = B.N;
  double *vo = B.vout + (size_t)w * N;
  const double *vi = B.vin + (size_t)w * N;
  const bool hist = B.iter >= 2 && B.M > 0;
  H *dfp = (H *)B.df + ((size_t)w * B.M + (hist ? B.ipos : 0)) * N;
  H *dvp = (H *)B.dv + ((size_t)w * B.M + (hist ? B.ipos : 0)) * N;
  const double *qf = f64 ? nullptr : B.pdf + (size_t)w * N;
  // float history (mixed path): the new dv is the step the last update added,
  // which that update left in dvin
  const double *qv = f64 ? nullptr : B.dvin + (size_t)w * N;
  double mx = 0.0, nr = 0.0, vm = 0.0;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
    const double d = vo[e] - vi[e];
    vo[e] = d;
    mx = fmax(mx, fabs(d));
    vm = fmax(vm, fabs(vi[e]));
    if (hist) {
      const double f = d - (f64 ? (double)dfp[e] : qf[e]);
      if constexpr (!f64) {
        dfp[e] = (H)f;
        dvp[e] = (H)qv[e];
      }
      nr += f * f;
    }
  }
  const double m = wg_max(mx, red);
  const double s = wg_sum(nr, red);
  const double v = wg_max(vm, red);
  if (threadIdx.x == 0) {
    *bro_part(B, w, 0, blockIdx.x) = m;
    *bro_part(B, w, 1, blockIdx.x) = s;
    *bro_part(B, w, 2, blockIdx.x) = v;   // read by k_bro_norm before k_bro_dots reuses the slot
  }
}

// One wave per frequency: lane l folds the partials l, l + 64, ... in order,
// then the lanes are combined by a fixed butterfly.
__global__ void __launch_bounds__(64) k_bro_norm(BroArgs B) {
  const int w = B.act[blockIdx.x];
  if (w == B.skip) return;
  bro_iter(B, w);
  double m = 0.0, s = 0.0, v = 0.0;
  for (int k = threadIdx.x; k < B.nwg; k += 64) {
    m = fmax(m, *bro_part(B, w, 0, k));
    s += *bro_part(B, w, 1, k);
    v = fmax(v, *bro_part(B, w, 2, k));
  }
  for (int o = 32; o > 0; o >>= 1) {
    m = fmax(m, __shfl_xor(m, o, 64));
    s += __shfl_xor(s, o, 64);
    v = fmax(v, __shfl_xor(v, o, 64));
  }
  if (threadIdx.x != 0) return;
  B.si[w] = m;
  B.vmax[w] = v;
  // a dropped pair is scaled to zero: its Gram row is then w0^2 + 1 on the
  // diagonal only and its coefficient zero, so it adds nothing to the step
  const bool drop = B.drop != nullptr && B.drop[w] != 0;
  B.scal[(size_t)w * 4 + 0] = (B.iter >= 2 && B.M > 0) ? (drop ? 0.0 : 1.0 / sqrt(s)) : 1.0;
}

// scale the history slot, then partial dots df_j . df_ipos and df_j . vout, up to
// BRO_JB history vectors per pass over the new difference and vout.  An FP64
// history's slot holds the last vout and vin until here: its difference is formed,
// scaled and stored in the first pass, u_j = dv_j + alpha df_j in the dv slot, the
// only form the update reads (one vector per history entry instead of two)
constexpr int BRO_JB = 8;
template <class H, int NJ, bool FIRST>
__device__ inline void bro_dots_pass(const BroArgs &B, int w, int j0, double normi, double *red) {
  constexpr bool f64 = sizeof(H) == 8;
  const long N = B.N;
  H *dfp = (H *)B.df + ((size_t)w * B.M + B.ipos) * N;
  H *dvp = (H *)B.dv + ((size_t)w * B.M + B.ipos) * N;
  const double *vo = B.vout + (size_t)w * N, *vi = B.vin + (size_t)w * N;
  double g[NJ], v[NJ];
  const H *hj[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    g[j] = 0.0; v[j] = 0.0;
    hj[j] = (const H *)B.df + ((size_t)w * B.M + j0 + j) * N;
  }
  const int own = B.ipos - j0;              // the new difference itself (what memory held before it does not count)
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
    const double o = vo[e];
    double a[NJ], p;
#pragma unroll
    for (int j = 0; j < NJ; ++j) a[j] = hj[j][e];
    if constexpr (f64 && FIRST) {
      const double f = o - dfp[e], q = vi[e] - dvp[e];
      p = f * normi;
      dfp[e] = p;
      dvp[e] = __builtin_fma(B.alpha, p, q * normi);
    } else if constexpr (FIRST) {
      const H f = (H)(dfp[e] * normi);
      dfp[e] = f;
      dvp[e] = (H)(dvp[e] * normi);
      p = f;
    } else {
      p = dfp[e];
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const double x = j == own ? p : a[j];
      g[j] += x * p;
      v[j] += x * o;
    }
  }
  // the 2 NJ sums of the pass together: per value the shuffle tree and wave order
  // of wg_sum, one LDS exchange for all of them
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    for (int o = 32; o > 0; o >>= 1) {
      g[j] += __shfl_down(g[j], o, 64);
      v[j] += __shfl_down(v[j], o, 64);
    }
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64;
  __syncthreads();
  if (lane == 0)
#pragma unroll
    for (int j = 0; j < NJ; ++j) { red[(2 * j) * (BRO_WG / 64) + wid] = g[j]; red[(2 * j + 1) * (BRO_WG / 64) + wid] = v[j]; }
  __syncthreads();
  if (threadIdx.x < 2 * NJ) {
    double t = 0.0;
    for (int q = 0; q < BRO_WG / 64; ++q) t += red[threadIdx.x * (BRO_WG / 64) + q];
    *bro_part(B, w, 2 + 2 * j0 + threadIdx.x, blockIdx.x) = t;
  }
}

template <class H, bool FIRST>
__device__ inline void bro_dots_step(const BroArgs &B, int w, int j0, double normi, double *red) {
  switch (min(BRO_JB, B.iter_used - j0)) {
    case 1: bro_dots_pass<H, 1, FIRST>(B, w, j0, normi, red); break;
    case 2: bro_dots_pass<H, 2, FIRST>(B, w, j0, normi, red); break;
    case 3: bro_dots_pass<H, 3, FIRST>(B, w, j0, normi, red); break;
    case 4: bro_dots_pass<H, 4, FIRST>(B, w, j0, normi, red); break;
    case 5: bro_dots_pass<H, 5, FIRST>(B, w, j0, normi, red); break;
    case 6: bro_dots_pass<H, 6, FIRST>(B, w, j0, normi, red); break;
    case 7: bro_dots_pass<H, 7, FIRST>(B, w, j0, normi, red); break;
    default: bro_dots_pass<H, 8, FIRST>(B, w, j0, normi, red); break;
  }
}

template <class H>
__global__ void __launch_bounds__(BRO_WG) k_bro_dots(BroArgs B) {
  __shared__ double red[2 * BRO_JB * (BRO_WG / 64)];
  const int w = B.act[blockIdx.y];
  if (w == B.skip) return;
  bro_iter(B, w);
  if (B.iter_used < 1) return;
  const double normi = B.scal[(size_t)w * 4 + 0];
  bro_dots_step<H, true>(B, w, 0, normi, red);
  for (int j0 = BRO_JB; j0 < B.iter_used; j0 += BRO_JB) bro_dots_step<H, false>(B, w, j0, normi, red);
}

// Lane l's value, l uniform.
__device__ inline double wave_read(double v, int l) {
  const long b = __builtin_bit_cast(long, v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, l), hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __builtin_bit_cast(double, (long)(((unsigned long)hi << 32) | lo));
}

// Largest value of the wave (every lane must hold a number).
__device__ inline double wave_max(double v) {
  auto step = [&](auto f) {
    const long b = __builtin_bit_cast(long, v);
    const unsigned lo = f((int)(unsigned)b), hi = f((int)(unsigned)(b >> 32));
    v = fmax(v, __builtin_bit_cast(double, (long)(((unsigned long)hi << 32) | lo)));
  };
  // lanes without a partner keep their own value; lane 63 ends with the whole wave's
  step([](int x) { return __builtin_amdgcn_update_dpp(x, x, 0x111, 0xf, 0xf, false); });   // row_shr:1
  step([](int x) { return __builtin_amdgcn_update_dpp(x, x, 0x112, 0xf, 0xf, false); });
  step([](int x) { return __builtin_amdgcn_update_dpp(x, x, 0x114, 0xf, 0xf, false); });
  step([](int x) { return __builtin_amdgcn_update_dpp(x, x, 0x118, 0xf, 0xf, false); });
  step([](int x) { return __builtin_amdgcn_update_dpp(x, x, 0x142, 0xa, 0xf, false); });   // row_bcast:15
  step([](int x) { return __builtin_amdgcn_update_dpp(x, x, 0x143, 0xc, 0xf, false); });   // row_bcast:31
  return wave_read(v, 63);
}

// Gram row update, beta = (w0^2+1) I + offdiag(Gram), gamma = beta^-1 work
// (Gauss-Jordan on one workgroup per frequency)
__global__ void __launch_bounds__(512) k_bro_solve(BroArgs B) {
  __shared__ double a[BRO_MAXM][2 * BRO_MAXM + 1];
  __shared__ double work[BRO_MAXM];
  const int w = B.act[blockIdx.x];
  if (w == B.skip) return;
  bro_iter(B, w);
  const int M = B.M, k = B.iter_used;
  double *gram = B.gram + (size_t)w * M * M;
  // reduce the partial dots: one wave per history entry j, lane l folds the
  // partials l, l + 64, ... in order, then a fixed butterfly over the lanes
  {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    for (int j = wv; j < k; j += nwv) {
      double sg = 0.0, sv = 0.0;
      for (int q = lane; q < B.nwg; q += 64) {
        sg += *bro_part(B, w, 2 + 2 * j, q);
        sv += *bro_part(B, w, 3 + 2 * j, q);
      }
      for (int o = 32; o > 0; o >>= 1) {
        sg += __shfl_xor(sg, o, 64);
        sv += __shfl_xor(sv, o, 64);
      }
      if (lane == 0) {
        if (B.iter >= 2) { gram[(size_t)B.ipos * M + j] = sg; gram[(size_t)j * M + B.ipos] = sg; }
        work[j] = sv;
      }
    }
  }
  __syncthreads();
  const double w0 = 0.010;
  // rows over the waves, columns over the lanes (no integer division per element)
  const int gl = threadIdx.x & 63, gw = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), gnw = blockDim.x >> 6;
  for (int i = gw; i < k; i += gnw)
    for (int j = gl; j < 2 * k; j += 64) {
      double v;
      if (j < k) v = (i == j) ? w0 * w0 + 1.0 : gram[(size_t)i * M + j];
      else v = (j - k == i) ? 1.0 : 0.0;
      a[i][j] = v;
    }
  __syncthreads();
  // Gauss-Jordan with partial pivoting (the first largest |a[i][c]|).  What a
  // column takes is latency, so it has one barrier (three, and the shuffles of the
  // search through LDS: 65 us for 50 pairs, now 40): rows stay where they are
  // (lane l of every wave holds the row at position l and swaps it there), every
  // wave finds the pivot by itself, column c and the pivot row are only read in
  // step c (columns up to c are not needed any more), and the pivot row is scaled
  // when the next step reads it.
  int row = gl;
  double dl = 1.0;                          // scale of the last pivot row (position c - 1)
  for (int c = 0; c < k; ++c) {
    const bool cand = gl >= c && gl < k;
    const double av = cand ? a[row][c] : 0.0;
    const double x = cand && fabs(av) > -1.0 ? fabs(av) : -1.0;
    const double big = wave_max(x);
    const int pos = __builtin_ctzll(__ballot(cand && x == big));
    const double d = 1.0 / wave_read(av, pos);
    const int rp = __builtin_amdgcn_readlane(row, pos), rc = __builtin_amdgcn_readlane(row, c);
    row = gl == c ? rp : (gl == pos ? rc : row);
    for (int i = gw; i < k; i += gnw) {
      if (i == c) continue;
      const int r = __builtin_amdgcn_readlane(row, i);
      const double sc = i == c - 1 ? dl : 1.0, f = a[r][c] * sc;
      for (int j = gl; j < 2 * k; j += 64)
        if (j > c) a[r][j] = __builtin_fma(-f, a[rp][j] * d, a[r][j] * sc);
    }
    dl = d;
    __syncthreads();
  }
  // position k - 1 still waits for its scale
  for (int i0 = 0; i0 < k; i0 += blockDim.x) {
    const int i = i0 + (int)threadIdx.x;
    double g = 0.0;
    for (int j = 0; j < k; ++j) {           // beta(j,i)
      const double b = a[__builtin_amdgcn_readlane(row, j)][k + min(i, k - 1)];
      g = __builtin_fma(j == k - 1 ? b * dl : b, work[j], g);
    }
    if (i < k)
      B.coef[(size_t)w * M + i] = g;
  }
}

// curv = alpha vout - sum_i gamma_i (dv_i + alpha df_i); df[inext] = vout;
// dv[inext] = vin; vin += curv.  With iter_used = 0 this is also the first
// Broyden step; mode 1/2 give linear mixing / no mixing.  An FP64 history
// holds dv_i + alpha df_i already (k_bro_dots forms it).
template <class H>
__global__ void __launch_bounds__(BRO_WG) k_bro_update(BroArgs B, int mode) {
  constexpr bool f64 = sizeof(H) == 8;
  const H *hdf = (const H *)B.df, *hdv = (const H *)B.dv;
  const int w = B.act[blockIdx.y];
  if (w == B.skip) return;
  bro_iter(B, w);
  const long N = B.N;
  double *vi = B.vin + (size_t)w * N;
  const double *vo = B.vout + (size_t)w * N;
  const double *gm = B.coef + (size_t)w * (B.M > 0 ? B.M : 1);
  double *dv_out = B.dvin ? B.dvin + (size_t)w * N : nullptr;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
    const double r = vo[e];
    double c;
    if (mode == 2) {
      c = r;
    } else if (mode == 1) {
      c = B.alpha * r;
    } else {
      c = B.alpha * r;
#pragma unroll 8
      for (int i = 0; i < B.iter_used; ++i) {
        const size_t o = ((size_t)w * B.M + i) * N + e;
        if (f64) c -= gm[i] * (double)hdv[o];
        else c -= gm[i] * __builtin_fma(B.alpha, (double)hdf[o], (double)hdv[o]);
      }
      if (f64) {
        const size_t on = ((size_t)w * B.M + B.inext) * N + e;
        ((double *)B.df)[on] = r;
        ((double *)B.dv)[on] = vi[e];
      } else {
        B.pdf[(size_t)w * N + e] = r;
      }
    }
    vi[e] += c;
    if (dv_out) dv_out[e] = c;
  }
}

// S = -(1/pi) (F20.X + F02.Y) for re and im (contract_bbm, pnfam_type_bbm.f90:393-421),
// for nop operators stored fstride apart (blockIdx.z; the strength itself and the
// cross-term operators, pnfam_solver.f90:190-203)
__global__ void __launch_bounds__(256) k_contract(const double *__restrict__ vin, const double *__restrict__ f20,
                                                  const double *__restrict__ f02, long nxy, double *__restrict__ part,
                                                  int nwg, const int *__restrict__ act, long fstride, int nop,
                                                  int skip) {
  __shared__ double red[4];
  const int w = act[blockIdx.y];
  if (w == skip) return;
  const double *v = vin + (size_t)w * 4 * nxy;
  const double *g20 = f20 + (size_t)blockIdx.z * fstride, *g02 = f02 + (size_t)blockIdx.z * fstride;
  double sr = 0.0, si = 0.0;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < nxy; e += (long)gridDim.x * blockDim.x) {
    sr += g20[e] * v[e] + g02[e] * v[nxy + e];
    si += g20[e] * v[2 * nxy + e] + g02[e] * v[3 * nxy + e];
  }
  const double a = wg_sum(sr, red);
  const double b = wg_sum(si, red);
  const size_t o = (((size_t)w * nop + blockIdx.z) * nwg + blockIdx.x) * 2;
  if (threadIdx.x == 0) { part[o] = a; part[o + 1] = b; }
}

// res: where the host reads the iteration's results (mapped memory: si, max|vin| and
// S of every point), null: nowhere.
struct HostRes {
  double *res;
  const double *si, *vmax;
  int npts;
};
__global__ void k_contract_fin(const double *__restrict__ part, int nwg, double *__restrict__ S,
                               const int *__restrict__ act, int nop, int skip, HostRes R) {
  const int w = act[blockIdx.x];
  if (w == skip) return;
  // one operator z per workgroup (one wave); the partials come in together and are
  // added in order
  __shared__ double p[128];
  const int z = blockIdx.y;
  const double *q = part + ((size_t)w * nop + z) * nwg * 2;
  double a = 0.0, b = 0.0;
  for (int k0 = 0; k0 < nwg; k0 += 64) {
    const int n = min(64, nwg - k0);
    __syncthreads();
    for (int e = threadIdx.x; e < 2 * n; e += 64) p[e] = q[2 * k0 + e];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int k = 0; k < n; ++k) { a += p[2 * k]; b += p[2 * k + 1]; }
  }
  if (threadIdx.x > 0) return;
  S[((size_t)w * nop + z) * 2] = -a / PI;
  S[((size_t)w * nop + z) * 2 + 1] = -b / PI;
  if (R.res && z == 0) {
    R.res[w] = R.si[w];
    R.res[R.npts + w] = R.vmax[w];
    R.res[2 * R.npts + 2 * w] = -a / PI;
    R.res[2 * R.npts + 2 * w + 1] = -b / PI;
  }
}

// dst = src for every active point's [w][n] slot
__global__ void k_copy_slots(double *__restrict__ dst, const double *__restrict__ src, long n,
                             const int *__restrict__ act) {
  const size_t w = act[blockIdx.y];
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    dst[w * n + e] = src[w * n + e];
}

}  // namespace

// ---------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------
struct pnfam_gpu_ctx {
  int device = 0;   // the device current at pnfam_gpu_create
  int nb = 0, dqp = 0, nghl = 0;
  std::vector<int> db, isstart, nsu, ns;
  std::vector<double> cscal;
  hipStream_t stream = nullptr;
  // resident
  DevPtr d_wf, d_wfdr, d_wfdz, d_wfdp, d_wfd2, d_wdcori, d_Ep, d_En;
  DevPtr d_U[4];
  DevPtr d_crho, d_cs, d_cpair, d_cspair;
  DevPtr d_isstart, d_db, d_nsu, d_ns;
  // operator
  bool have_op = false;
  bool bminus = true;
  long nxy = 0;
  BlockMap fmap, xmap, ymap, rspmap[4], hspmap[4];
  DevPtr d_f20, d_f02, d_xrow, d_xcol, d_yrow, d_ycol;
  DevPtr d_terms_q2s[2], d_groups_q2s[2], d_terms_s2q[2], d_groups_s2q[2];
  int ngroups_q2s[2] = {0, 0}, ngroups_s2q[2] = {0, 0};
  size_t lds_q2s = 0, lds_s2q = 0;
  int strips = 1;   // 16-row strips of the largest output block
  DevPtr d_pairs;   // rho0, kap0, rho1, kap1 pair lists
  int pair_off[4] = {0, 0, 0, 0}, pair_n[4] = {0, 0, 0, 0};
  DevPtr d_tiles, d_tiles2;
  int ntiles = 0, ntiles2 = 0;
  int pj_first[16] = {}, pj_count[16] = {};   // projection tiles per kind * 8 + row tiles
  bool basic_kernels = false;   // PNFAM_GPU_BASIC=1: the plain FP64 kernels (cross-check path)
  int proj_nf1 = 0;             // proj_freqs of the one-row-tile mean-field tiles, 0: proj_nf (option proj_freqs_rt1)
  int fac_nf = 0;               // factored BF16 projection: frequencies per wave, 0 auto (option fac_freqs)
  bool sorted_spins = false;    // every block's states spin-sorted (k_density_pq2 needs it)
  int dens_pq = 2;              // FP64 densities: 2 two waves by row spin, transposed products, no
                                // exchange; 1 two waves by table with an LDS exchange; 0 one wave
  int proj_ns = 2;              // k_project_mfma operand pipeline depth, 1 or 2 (option proj_stages)
  int graph_mode = 0;           // FP64 batches: iterations as graph replays (option graph)
  int few_split_on = 1;         // few-point splits of the FP64 grid loops (option few_split)
  bool q2s_cover = false, s2q_cover = false;   // the transforms' groups write every output element
  bool proj_cover = false;      // the projection tiles write every dH_sp element
  int zero_skip = 1;            // 1: no zeroing of fully covered transform outputs (option zero_skip)
  bool graph_capturing = false; // a graph is being captured: no allocations
  long graph_launches = 0;      // graph replays of the last batch (option graph_launches)
  int skip_slot = -1;           // while a replay is captured: the spare slot, whose workgroups return at once
  long graph_captures = 0;      // graphs captured for it (option graph_captures)
  double graph_capture_ms = 0;  // host time spent capturing and instantiating them (option graph_capture_ms)
  DevPtr d_gdone, d_giters, d_gctl;
  int proj_maxrt = P2_MAXRT;    // projection: 16-row tiles per wave (option proj_rows)
  int proj_nf = 1;              // projection: frequencies per wave, 1 or 2, or 4 per workgroup with the
                                // psi operands shared through LDS (option proj_freqs)
  // per-frequency workspace
  int cap = 0;
  int hist_cap = -1;
  DevPtr d_vin, d_vout, d_rsp, d_hsp, d_hqp, d_dens, d_flds, d_part, d_cpart, d_S, d_si, d_vmax, d_scal;
  DevPtr d_df, d_dv, d_pdf, d_gram, d_coef, d_wre, d_wim, d_act;
  // mixed path: the next increment of vin, accumulated FP64 H20/H02
  DevPtr d_act64, d_actlo, d_dvin, d_hacc, d_drop, d_lag;
  DevPtr d_ppart;   // partial projections of a grid-point split (few frequencies)
  DevPtr d_dpart;   // partial densities of a pair split (few frequencies)
  // split-BF16 grid stage: one element layout per block structure (the mean-field
  // set in map f, one pairing set per sector), pair tables and operands
  struct MixSet {
    int Kp = 0;
    int kbeg[5] = {0, 0, 0, 0, 0};
    int ntp = 0, ntd = 0;
    DevPtr d_elem, d_sa, d_sb, TPh, TPl, TDh, TDl, d_jobs_dens, d_jobs_proj;
    DevPtr Bh, Bl, O, Fh, Fl;   // per-batch operands
    int maxcount = 0;            // largest class
  };
  MixSet mix[3];                 // 0: mean field (f); 1: kappa+/Delta+ (sector 0); 2: kappa-/Delta- (sector 1)
  bool mix_ready = false;
  int RP = 0, mix_cap = 0;
  // contractions: rocBLAS bf16 GEMMs (default) or the hand-written k_mix_gemm
  // (PNFAM_GPU_MIX_GEMM=own)
  rocblas_handle blas = nullptr;
  bool own_gemm = false;
  DevPtr d_Oproj;   // projection results [Kp][ncol] of the largest set (FP32)
  DevPtr d_Psplit;  // split-K partial planes (FP32)
  // factored split-BF16 grid stage: psi tables, chunk maps, pair lists, operand segments
  int mix_grid = 0;             // 0 auto, 1 pair tables, 2 factored (PNFAM_GPU_MIX_GRID)
  int mix_auto_n = 6;           // auto: factored at or below this many active points
  double mix_table_frac = 0.5;  // auto: pair tables only within this fraction of free device memory
  double mix_table_bytes = 0;   // their size, as estimated by the last auto choice
  bool fac_ready = false;
  DevPtr PAh, PAl, PS32, DBh, DBl, d_fac_blk, d_fac_pairs, d_fac_segs, FRh, FRl, d_fac_dpart, FFm, FFp;
  long fac_L = 0, fac_pz = 0, fac_dbx = 0;
  int fac_nseg = 0, fac_cap = 0;
  int fac_first[4] = {0, 0, 0, 0}, fac_n[4] = {0, 0, 0, 0};   // rho0, kap0, rho1, kap1 pair ranges
  // split-BF16 block triple products (mixed path): padded hi/lo copies of U/V
  bool tp_bf16 = true;          // PNFAM_GPU_MIX_TRIPROD = bf16 | fp64
  bool tp_ready = false;
  bool tp64_ok = true;          // the terms' A and C are whole blocks (FP64 matrix-core products)
  DevPtr tp_cm64, tp_rm64;      // padded FP64 copies of U/V for them
  std::vector<int4> tp_blocks;  // (fp64 offset, padded offset, d, P) per block
  long tp_mstride = 0;
  DevPtr tp_rmh, tp_rml, tp_cmh, tp_cml, d_tp_blocks;
  // per stage, the re and im term sets together (one launch per tile class
  // covers both): terms, groups sorted by tile count, B operand offsets and
  // conversion jobs
  std::vector<Term> tpa_terms_h[2];
  std::vector<Group> tpa_groups_h[2];
  std::vector<int> tpa_toff_h[2];
  std::vector<int2> tpa_jobs_h[2];
  DevPtr d_tpa_terms[2], d_tpa_groups[2], d_tpa_toff[2], d_tpa_jobs[2], tp_Bh, tp_Bl;
  int tpa_njobs[2] = {0, 0};
  int tpa_first[2][TP_MAXCT + 1] = {}, tpa_count[2][TP_MAXCT + 1] = {}, tpa_strips[2][TP_MAXCT + 1] = {};
  long tp_L[2] = {0, 0}, tp_Lcap = 0;                        // per active point, per stage
  int unit_precision = PNFAM_GPU_FP64;   // grid stage of the per-unit entry points
  // pinned host staging of the per-iteration transfers: active lists [3][cap]
  // (all, FP64, low precision) and results [4][cap] (si, vmax, re S, im S)
  int *pin_act = nullptr;
  double *pin_res = nullptr;
  int pin_cap = 0;
  int bro_nwg = 0;
  int bro_nwg_few = 0;          // FP32-history Broyden with few active points: more workgroups per point
  double flops_q2s = 0, flops_s2q = 0;
  // per-kernel event timing (pnfam_gpu_profile)
  bool prof = false;
  struct KStat { double ms = 0; int64_t launches = 0; double units = 0; };
  KStat kstat[32];
  struct Pending { int kid; hipEvent_t a, b; int units; };
  std::vector<Pending> pending;
  std::vector<hipEvent_t> event_pool;
  double flops_unit[32] = {0};   // algorithmic FLOP per frequency, per kernel id
  // kernel classes (name and template arguments) launched while profiling is on
  std::set<std::string> classes;
  // per-unit entry points: batch slots their one frequency runs in (option
  // unit_replicas), so that they take the batched launch paths
  int unit_reps = 1;
  bool unit_general = false;   // the grid stage of the FP64 unit calls runs the general kernels (set with unit_replicas)
  std::vector<int> unit_act;
  // mixed-path options (environment defaults, pnfam_gpu_set_option)
  double mix_tau = 3e-3;        // one-product threshold (PNFAM_GPU_MIX_TAU)
  int mix_hist64 = 0;           // Broyden history in FP64 (PNFAM_GPU_MIX_HIST=fp64)
  int mix_drop = 1;             // zero the Broyden pair across a refinement (PNFAM_GPU_MIX_DROP)
  double mix_refine_at = 1.0;   // MIXED refines when si < mix_refine_at * tolerance
  int mix_refine_every = 8;     // MIXED refinements run on batch iterations that are multiples of this
  bool mix_grid_set = false, mix_auto_set = false;   // set by pnfam_gpu_set_option (over the environment)
  // per-unit Broyden hook (pnfam_gpu_broyden_step): history size and mixing in use
  int hook_M = -2;
  double hook_alpha = 0.0;
  // FP64 grid stage on product grids (separable.hpp): the basis part, found when
  // the context is created, and the plan of the operator's block structures
  struct SepGroup { int cls, first, count; };   // radial function, members of the state list
  bool sep_basis = false, sep_plan = false;
  bool sep_nomem = false;      // the workspace could not be had: the rest of this call takes the general kernels
  size_t sep_limit = 0;        // option fp64_grid_bytes
  double sep_resid = 1.0;      // largest residual of the tables' product fit
  int sep_nz = 0, sep_nr = 0, sep_ncls = 0;
  std::vector<SepGroup> sep_groups;              // per (block, spin), in order of sep_gfirst
  std::vector<int> sep_gfirst;                   // [2 nb + 1]
  std::vector<int> sep_members;                  // local state indices
  DevPtr d_sep_f, d_sep_fz;
  DevPtr d_sep_keys, d_sep_tabs, d_sep_djobs, d_sep_pjobs;
  DevPtr d_sep_slots[2], d_sep_elems[2];         // density, projection
  int sep_nslot[2] = {0, 0}, sep_ndjob = 0, sep_nwork = 0, sep_npjob[2] = {0, 0}, sep_pjob0[2] = {0, 0};
  int sep_ct[2] = {1, 1}, sep_ncg[2] = {1, 1};   // density, projection: column tiles per wave, column groups
  int sep_nct1 = 1;                              // column tiles of the projection
  SepAcc sep_acc{};
  long sep_zstride = 0, sep_ystride = 0, sep_arows = 0;
  double sep_flops_d = 0, sep_flops_p = 0;       // FLOP per point of the two halves; gen_: of the general kernels
  double gen_flops_d = 0, gen_flops_p = 0;
  DevPtr d_sep_zy, d_sep_part;                   // Z / Y and partial densities of a chunk of points
  int fp64_grid = 0;                             // 0: the separable stage where there is a plan, 1: never
  // cross-term operators in the qp basis, g20 / g02 [nx][nxy], and their
  // contractions with every point's amplitudes [w][nx][2]
  int nx = 0;
  DevPtr d_g20, d_g02, d_xpart, d_xs;
  // plan of the qp transform W^T g W of a single-particle operator with f's structure
  std::vector<Term> fq_terms;
  std::vector<Group> fq_groups;
  size_t fq_lds = 8;
  // host state of the last batch: what a checkpoint holds besides the device
  // arrays (the next iteration to run and per point the residual, largest
  // amplitude, strength, status and refinement flag)
  struct Batch {
    bool valid = false;
    int npts = 0, iter = 0, M = 0, precision = 0, hist32 = 0, nx = 0;
    double eps = 0, quench = 0, alpha = 0;
    std::vector<double> wre, wim, si, vmax, S;
    std::vector<int> done, refined, iters;
    std::vector<int> lag;   // iterations each point waited for its refinement group
  } bs;
  ~pnfam_gpu_ctx() {
    if (blas) (void)rocblas_destroy_handle(blas);
    if (pin_act) (void)hipHostFree(pin_act);
    if (pin_res) (void)hipHostFree(pin_res);
    for (auto &p : pending) { (void)hipEventDestroy(p.a); (void)hipEventDestroy(p.b); }
    for (auto e : event_pool) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

enum KernelId { K_TRIPROD_Q2S, K_DENSITY, K_FIELDS, K_PROJECT, K_TRIPROD_S2Q, K_GREEN, K_BRO_RESID, K_BRO_NORM,
                K_BRO_DOTS, K_BRO_SOLVE, K_BRO_UPDATE, K_CONTRACT, K_CONTRACT_FIN, K_ZERO, K_MIXACC,
                K_MIX_CVT, K_MIX_GEMM_D, K_MIX_DENS, K_MIX_GEMM_P, K_FAC_CVT, K_FAC_DENS, K_FAC_PROJ, K_NKERNEL };
const char *kKernelNames[K_NKERNEL] = {"triprod_qp2sp", "density", "fields", "project", "triprod_sp2qp", "green",
                                       "bro_resid", "bro_norm", "bro_dots", "bro_solve", "bro_update", "contract",
                                       "contract_fin", "zero_slots", "mix_accumulate", "mix_convert",
                                       "mix_gemm_density", "mix_densities", "mix_gemm_project", "fac_convert",
                                       "fac_density", "fac_project"};

hipEvent_t pool_event(pnfam_gpu_ctx *h) {
  if (!h->event_pool.empty()) { hipEvent_t e = h->event_pool.back(); h->event_pool.pop_back(); return e; }
  hipEvent_t e = nullptr;
  (void)hipEventCreate(&e);
  return e;
}

// Brackets one launch with events on the engine stream when profiling is on.
struct Prof {
  pnfam_gpu_ctx *h; int kid; int units; hipEvent_t a = nullptr;
  Prof(pnfam_gpu_ctx *h_, int kid_, int units_) : h(h_), kid(kid_), units(units_) {
    if (h->prof) { a = pool_event(h); (void)hipEventRecord(a, h->stream); }
  }
  ~Prof() {
    if (!h->prof) return;
    hipEvent_t b = pool_event(h);
    (void)hipEventRecord(b, h->stream);
    h->pending.push_back({kid, a, b, units});
  }
};

// Records one launched kernel class while profiling is on.
// Every block's states spin-sorted: [0, nsu) up, [nsu, d) down (the HFB
// preparation sorts them; k_density_pq2 relies on it, so a context whose basis
// is not sorted runs k_density_pq instead).
bool spin_sorted(const pnfam_gpu_ctx *h) {
  for (size_t i = 0; i < h->db.size(); ++i)
    for (int j = 0; j < h->db[i]; ++j)
      if ((h->ns[h->isstart[i] + j] > 0) != (j < h->nsu[i])) return false;
  return true;
}

void note(pnfam_gpu_ctx *h, const char *name, int a = -1, int b = -1) {
  if (!h->prof) return;
  char buf[64];
  if (a < 0) std::snprintf(buf, sizeof buf, "%s", name);
  else if (b < 0) std::snprintf(buf, sizeof buf, "%s<%d>", name, a);
  else std::snprintf(buf, sizeof buf, "%s<%d,%d>", name, a, b);
  h->classes.insert(buf);
}

// Call after a stream synchronisation: folds finished launches into the totals.
void prof_collect(pnfam_gpu_ctx *h) {
  for (auto &p : h->pending) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
      h->kstat[p.kid].ms += ms;
      h->kstat[p.kid].launches += 1;
      h->kstat[p.kid].units += p.units;
    }
    h->event_pool.push_back(p.a);
    h->event_pool.push_back(p.b);
  }
  h->pending.clear();
}

int upload(DevPtr &d, const void *h, size_t bytes, hipStream_t s) {
  if (int e = d.alloc(bytes)) return e;
  HIP_TRY(hipMemcpyAsync(d.p, h, bytes, hipMemcpyHostToDevice, s));
  return 0;
}

std::vector<int4> pair_list(const BlockMap &m) {
  std::vector<int4> v;
  for (size_t i = 0; i < m.ir2c.size(); ++i)
    if (m.ir2c[i] >= 0) v.push_back(make_int4((int)i, m.ir2c[i], m.ir2m[i], 0));
  return v;
}

// Padded layout of the resident block-diagonal matrices for the matrix-core
// triple products (BF16 and FP64): block i (dimension d, FP64 offset sum d_j^2) at the padded offset
// sum P_j^2, P = d rounded up to 32.
void tp_layout(pnfam_gpu_ctx *h) {
  h->tp_blocks.clear();
  long off = 0, poff = 0;
  for (size_t i = 0; i < h->db.size(); ++i) {
    const int d = h->db[i], P = (d + 31) & ~31;
    h->tp_blocks.push_back(make_int4((int)off, (int)poff, d, P));
    off += (long)d * d;
    poff += (long)P * P;
  }
  h->tp_mstride = std::max<long>(poff, 8);
}

// Term fields pad0 / pad1: padded offsets of the A and C blocks (-1 if the FP64
// offset is not a block start).
void tp_patch_terms(const pnfam_gpu_ctx *h, std::vector<Term> &terms) {
  auto pad = [&](int off) {
    for (const auto &b : h->tp_blocks)
      if (b.x == off) return b.y;
    return -1;
  };
  for (auto &t : terms) { t.pad0 = pad(t.a_off); t.pad1 = pad(t.c_off); }
}

// B operand layout of one (stage, ri) term set, appended to the stage's
// combined lists: term offsets (after base) and conversion jobs; returns the
// end offset.
long tp_b_layout(pnfam_gpu_ctx *h, int stage, const std::vector<Term> &terms, const std::vector<Group> &groups,
                 long base) {
  const int t0 = (int)h->tpa_terms_h[stage].size();
  long off = base;
  // terms that read the same block of B the same way share one converted copy
  std::map<std::array<int, 5>, int> seen;
  for (size_t i = 0; i < terms.size(); ++i) {
    const Term &t = terms[i];
    const std::array<int, 5> key{t.b_slot, t.b_off, t.tb, t.nda, t.ndc};
    const auto it = seen.find(key);
    if (it != seen.end()) { h->tpa_toff_h[stage].push_back(it->second); continue; }
    const int nj = (t.ndc + 15) / 16, nk = ((t.nda + 31) & ~31) / TP_TK;
    h->tpa_toff_h[stage].push_back((int)off);
    seen[key] = (int)off;
    for (int q = 0; q < nj * nk; ++q) h->tpa_jobs_h[stage].push_back(make_int2(t0 + (int)i, q));
    off += (long)nj * TP_TJ * nk * TP_TK;
  }
  h->tpa_terms_h[stage].insert(h->tpa_terms_h[stage].end(), terms.begin(), terms.end());
  for (Group g : groups) {
    g.first += t0;
    h->tpa_groups_h[stage].push_back(g);
  }
  return off;
}

// Sorts a stage's combined groups by tile count and uploads the combined lists.
int tp_finish_stage(pnfam_gpu_ctx *h, int stage) {
  auto &groups = h->tpa_groups_h[stage];
  auto nct = [](const Group &g) { return (g.ncol + 15) / 16; };
  std::stable_sort(groups.begin(), groups.end(), [&](const Group &a, const Group &b) { return nct(a) < nct(b); });
  for (int c = 0; c <= TP_MAXCT; ++c) { h->tpa_first[stage][c] = 0; h->tpa_count[stage][c] = 0; h->tpa_strips[stage][c] = 0; }
  for (size_t i = 0; i < groups.size(); ++i) {
    const int c = nct(groups[i]);
    if (h->tpa_count[stage][c] == 0) h->tpa_first[stage][c] = (int)i;
    h->tpa_count[stage][c]++;
    h->tpa_strips[stage][c] = std::max(h->tpa_strips[stage][c], (groups[i].nrow + 15) / 16);
  }
  auto &terms = h->tpa_terms_h[stage];
  auto &toff = h->tpa_toff_h[stage];
  auto &jobs = h->tpa_jobs_h[stage];
  h->tpa_njobs[stage] = (int)jobs.size();
  if (terms.empty()) terms.push_back(Term{});
  if (toff.empty()) toff.push_back(0);
  if (jobs.empty()) jobs.push_back(make_int2(0, 0));
  if (groups.empty()) groups.push_back(Group{});
  int e;
  if ((e = upload(h->d_tpa_terms[stage], terms.data(), terms.size() * sizeof(Term), h->stream)) ||
      (e = upload(h->d_tpa_groups[stage], groups.data(), groups.size() * sizeof(Group), h->stream)) ||
      (e = upload(h->d_tpa_toff[stage], toff.data(), toff.size() * 4, h->stream)) ||
      (e = upload(h->d_tpa_jobs[stage], jobs.data(), jobs.size() * sizeof(int2), h->stream)))
    return e;
  HIP_TRY(hipStreamSynchronize(h->stream));   // the host lists are released below
  terms.clear(); toff.clear(); jobs.clear(); groups.clear();
  return 0;
}

bool tp_terms_ok(const std::vector<Term> &terms) {
  for (const auto &t : terms)
    if (t.pad0 < 0 || t.pad1 < 0) return false;
  return true;
}

int tp_prepare(pnfam_gpu_ctx *h) {
  if (h->tp_ready) return 0;
  const size_t n = 4 * (size_t)h->tp_mstride * 2;
  int e;
  if ((e = h->tp_rmh.alloc(n)) || (e = h->tp_rml.alloc(n)) || (e = h->tp_cmh.alloc(n)) || (e = h->tp_cml.alloc(n)))
    return e;
  for (int m = 0; m < 4; ++m) {
    const size_t o = (size_t)m * h->tp_mstride;
    hipLaunchKernelGGL(k_tp_copy, dim3(16, (unsigned)h->tp_blocks.size()), dim3(256), 0, h->stream,
                       h->d_U[m].as<double>(), h->d_tp_blocks.as<int4>(), (int)h->tp_blocks.size(),
                       h->tp_rmh.as<__bf16>() + o, h->tp_rml.as<__bf16>() + o, h->tp_cmh.as<__bf16>() + o,
                       h->tp_cml.as<__bf16>() + o);
  }
  HIP_TRY(hipGetLastError());
  h->tp_ready = true;
  return 0;
}

// FP64 triple products of a stage, both term sets (re and im): one launch per
// tile count present, or up to TP_SPLIT_N points one launch of k_triprod_split for
// all of them (beyond that the groups alone fill the device: N_sh = 16, 129 us at
// 4 points, as much as the launches per count; 42 to 56 us at one).
int launch_triprod(pnfam_gpu_ctx *h, int stage, const double *bbase, long bstride, double *obase, long ostride, int na,
                   const int *act) {
  const Tp64 M{h->tp_cm64.as<double>(), h->tp_rm64.as<double>(), h->tp_mstride};
  const Term *terms = h->d_tpa_terms[stage].as<Term>();
  const Group *groups = h->d_tpa_groups[stage].as<Group>();
  const bool split = na <= TP_SPLIT_N;
  int cmax = 0, smax = 0, ntot = 0;
  for (int c = 1; c <= TP_MAXCT; ++c)
    if (h->tpa_count[stage][c]) { cmax = c; smax = std::max(smax, h->tpa_strips[stage][c]); ntot += h->tpa_count[stage][c]; }
  for (int c = split ? cmax : 1; c <= TP_MAXCT && c >= 1; ++c) {
    const int n = split ? ntot : h->tpa_count[stage][c];
    if (!n) continue;
    const int ns = split ? smax : h->tpa_strips[stage][c];
    // four strips of a group to a workgroup, or two where that leaves fewer waves idle
    const int nw = split || (ns + 1) % 4 < 2 ? 4 : 2, nz = split ? ns : (ns + nw - 1) / nw;
    const dim3 grid(n, na, nz), block(64 * nw);
    const Group *g = groups + (split ? 0 : h->tpa_first[stage][c]);
    // the column class, whichever kernel takes it, and the kernel
    note(h, "k_triprod_mfma", std::min(c, TP_MAXCT));
    if (split) note(h, "k_triprod_split", std::min(c, TP_MAXCT));
    else note(h, "k_triprod_mfma", std::min(c, TP_MAXCT), nw);
#define TP_GO(K) \
  hipLaunchKernelGGL(K, grid, block, 0, h->stream, g, terms, M, bbase, bstride, obase, ostride, act, h->nxy, h->skip_slot)
#define TP_LAUNCH(NC)                                      \
  do {                                                     \
    if (split) TP_GO(k_triprod_split<NC>);                 \
    else if (nw == 4) TP_GO((k_triprod_mfma<NC, 4>));      \
    else TP_GO((k_triprod_mfma<NC, 2>));                   \
  } while (0)
    switch (c) {
      case 1: TP_LAUNCH(1); break;
      case 2: TP_LAUNCH(2); break;
      case 3: TP_LAUNCH(3); break;
      case 4: TP_LAUNCH(4); break;
      case 5: TP_LAUNCH(5); break;
      case 6: TP_LAUNCH(6); break;
      case 7: TP_LAUNCH(7); break;
      default: TP_LAUNCH(8); break;
    }
#undef TP_LAUNCH
#undef TP_GO
    if (split) break;
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Both term sets (re and im) of a stage: one conversion launch and one launch
// per tile class (one launch in all for few points).
int launch_triprod_bf16(pnfam_gpu_ctx *h, int stage, const double *bbase, long bstride, double *obase, long ostride,
                        int na, const int *act, int n3) {
  if (int e = tp_prepare(h)) return e;
  const long L = std::max(h->tp_L[0], h->tp_L[1]);
  if (h->tp_Lcap < L * h->cap) {
    h->tp_Lcap = 0;
    if (int e = h->tp_Bh.alloc((size_t)L * h->cap * 2)) return e;
    if (int e = h->tp_Bl.alloc((size_t)L * h->cap * 2)) return e;
    h->tp_Lcap = L * h->cap;
  }
  if (na > h->cap) return fail(PNFAM_GPU_EINVAL, "more active points than the batch capacity");
  const Term *terms = h->d_tpa_terms[stage].as<Term>();
  const Group *groups = h->d_tpa_groups[stage].as<Group>();
  if (const int nj = h->tpa_njobs[stage]) {
    // four waves per workgroup; with many points each wave takes four jobs
    const int per = na >= 16 ? 16 : 4;
    hipLaunchKernelGGL(k_tp_bconv, dim3((nj + per - 1) / per, na), dim3(256), 0, h->stream, terms,
                       h->d_tpa_toff[stage].as<int>(), h->d_tpa_jobs[stage].as<int2>(), nj, bbase, bstride, h->nxy,
                       act, L, h->tp_Bh.as<__bf16>(), h->tp_Bl.as<__bf16>());
  }
  TpMats M{h->tp_rmh.as<__bf16>(), h->tp_rml.as<__bf16>(), h->tp_cmh.as<__bf16>(), h->tp_cml.as<__bf16>(),
           h->tp_mstride};
  TpB BB{h->tp_Bh.as<__bf16>(), h->tp_Bl.as<__bf16>(), L, h->d_tpa_toff[stage].as<int>()};
  // few points: one launch over all tile classes (the widest template), so the
  // classes' dependency chains overlap instead of running one after another
  const bool merge = na <= TP_MERGE_N;
  int cmax = 0, smax = 0, ntot = 0;
  for (int c = 1; c <= TP_MAXCT; ++c)
    if (h->tpa_count[stage][c]) { cmax = c; smax = std::max(smax, h->tpa_strips[stage][c]); ntot += h->tpa_count[stage][c]; }
  for (int c = merge ? cmax : 1; c <= TP_MAXCT && c >= 1; ++c) {
    const int n = merge ? ntot : h->tpa_count[stage][c];
    if (!n) continue;
    const int ns = merge ? smax : h->tpa_strips[stage][c];
    // strips per workgroup (one launch per tile class with many points): qp -> sp
    // classes of four or more strips take one strip per wave (shared B and C
    // loads; 17 % faster for that stage).  The sp -> qp groups hold more terms:
    // two and four strips per workgroup measured 5 % and 10 % slower there, and
    // merged few-point launches want the parallelism of the term split.
    const int spw = (!merge && stage == 0 && ns >= 4) ? 4 : 1;
    const long units8 = ((long)n * na + 7) / 8;
    const dim3 grid((unsigned)(units8 * ((ns + spw - 1) / spw) * 8));
    const Group *g = groups + (merge ? 0 : h->tpa_first[stage][c]);
    note(h, "k_triprod_bf16", std::min(c, TP_MAXCT), spw);
#define TB_LAUNCH(NC)                                                                                          \
  do {                                                                                                         \
    if (spw == 4)                                                                                              \
      hipLaunchKernelGGL((k_triprod_bf16<NC, 4>), grid, dim3(64 * TP_NW), 0, h->stream, g, n, ns, terms, M, BB, \
                         obase, ostride, act, na, h->nxy, n3);                                                 \
    else                                                                                                       \
      hipLaunchKernelGGL((k_triprod_bf16<NC, 1>), grid, dim3(64 * TP_NW), 0, h->stream, g, n, ns, terms, M, BB, \
                         obase, ostride, act, na, h->nxy, n3);                                                 \
  } while (0)
    switch (c) {
      case 1: TB_LAUNCH(1); break;
      case 2: TB_LAUNCH(2); break;
      case 3: TB_LAUNCH(3); break;
      case 4: TB_LAUNCH(4); break;
      case 5: TB_LAUNCH(5); break;
      case 6: TB_LAUNCH(6); break;
      case 7: TB_LAUNCH(7); break;
      default: TB_LAUNCH(8); break;
    }
#undef TB_LAUNCH
    if (merge) break;
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

int grow_workspace(pnfam_gpu_ctx *h, int npts, int M) {
  // an allocation that fails below leaves its buffer freed: the recorded
  // capacity is cleared first and set only once every buffer is in place
  h->cap = 0;
  h->hist_cap = -1;
  const size_t n = (size_t)std::max(npts, 1);
  const size_t nxy = (size_t)h->nxy;
  const int Mh = std::max(M, 1);
  int e;
  if ((e = h->d_vin.alloc(n * 4 * nxy * 8))) return e;
  if ((e = h->d_vout.alloc(n * 4 * nxy * 8))) return e;
  if ((e = h->d_rsp.alloc(n * 8 * nxy * 8))) return e;
  if ((e = h->d_hsp.alloc(n * 8 * nxy * 8))) return e;
  if ((e = h->d_hqp.alloc(n * 4 * nxy * 8))) return e;
  if ((e = h->d_dens.alloc(n * 2 * 2 * NDENS * (size_t)h->nghl * 8))) return e;
  if ((e = h->d_flds.alloc(n * 2 * 2 * NFLD * (size_t)h->nghl * 8))) return e;
  h->bro_nwg = (int)std::min<long>(256, std::max<long>(1, (long)(4 * nxy + BRO_WG - 1) / BRO_WG));
  h->bro_nwg_few = (int)std::min<long>(BRO_NWG_FEW, std::max<long>(1, (long)(4 * nxy + BRO_WG - 1) / BRO_WG));
  if ((e = h->d_part.alloc(n * std::max(h->bro_nwg, h->bro_nwg_few) * (2 * BRO_MAXM + 2) * 8))) return e;
  if ((e = h->d_cpart.alloc(n * 64 * 2 * 8))) return e;
  if ((e = h->d_S.alloc(n * 2 * 8))) return e;
  if ((e = h->d_si.alloc(n * 8))) return e;
  if ((e = h->d_vmax.alloc(n * 8))) return e;
  if ((e = h->d_scal.alloc(n * 4 * 8))) return e;
  if ((e = h->d_df.alloc(n * Mh * 4 * nxy * 8))) return e;
  if ((e = h->d_dv.alloc(n * Mh * 4 * nxy * 8))) return e;
  if ((e = h->d_pdf.alloc(n * 4 * nxy * 8))) return e;
  if ((e = h->d_gram.alloc(n * Mh * Mh * 8))) return e;
  if ((e = h->d_coef.alloc(n * Mh * 8))) return e;
  if ((e = h->d_wre.alloc(n * 8))) return e;
  if ((e = h->d_wim.alloc(n * 8))) return e;
  if ((int)n > h->pin_cap) {
    if (h->pin_act) { (void)hipHostFree(h->pin_act); h->pin_act = nullptr; }
    if (h->pin_res) { (void)hipHostFree(h->pin_res); h->pin_res = nullptr; }
    h->pin_cap = 0;
    if (hipHostMalloc((void **)&h->pin_act, 6 * n * 4) != hipSuccess ||
        hipHostMalloc((void **)&h->pin_res, 4 * n * 8) != hipSuccess) {
      (void)hipGetLastError();
      return fail(PNFAM_GPU_ENOMEM, "hipHostMalloc of the pinned staging buffers failed");
    }
    h->pin_cap = (int)n;
  }
  if ((e = h->d_act.alloc(n * 4))) return e;
  if ((e = h->d_act64.alloc(n * 4))) return e;
  if ((e = h->d_drop.alloc(n * 4))) return e;
  if ((e = h->d_lag.alloc(n * 4))) return e;
  if ((e = h->d_actlo.alloc(n * 4))) return e;
  if ((e = h->d_dvin.alloc(n * 4 * nxy * 8))) return e;
  if ((e = h->d_hacc.alloc(n * 4 * nxy * 8))) return e;
  h->cap = (int)n;
  h->hist_cap = M;
  return 0;
}

void sep_release(pnfam_gpu_ctx *h) {
  h->d_sep_zy.release();
  h->d_sep_part.release();
}

int ensure_workspace(pnfam_gpu_ctx *h, int npts, int M) {
  if (npts <= h->cap && M == h->hist_cap) return 0;
  int e = grow_workspace(h, npts, M);
  // the factored grid stage can do without its workspace, a batch cannot
  if (e == PNFAM_GPU_ENOMEM && h->d_sep_zy.p) {
    sep_release(h);
    e = grow_workspace(h, npts, M);
  }
  return e;
}

dim3 grid1(size_t n, int bs, int maxb = 2048) {
  size_t b = (n + bs - 1) / bs;
  return dim3((unsigned)std::max<size_t>(1, std::min<size_t>(b, maxb)));
}

// ---- pipeline stages over the active list (device pointer act, count na) --
// lowp: split-BF16 triple products (the mixed path's increments), the first
// n3 active points with three products.
int stage_qp2sp(pnfam_gpu_ctx *h, const double *vin, int na, const int *act, bool lowp = false, int n3 = 0) {
  const long nxy = h->nxy;
  if (!(h->zero_skip && h->q2s_cover && !h->basic_kernels)) {
    Prof pr(h, K_ZERO, na);
    hipLaunchKernelGGL(k_zero_slots, dim3(64, na), dim3(256), 0, h->stream, h->d_rsp.as<double>(), act, 8, 0, 8, nxy,
                       h->skip_slot); }
  Prof pr(h, K_TRIPROD_Q2S, na);
  if (lowp) return launch_triprod_bf16(h, 0, vin, 4 * nxy, h->d_rsp.as<double>(), 8 * nxy, na, act, n3);
  if (!h->basic_kernels && h->tp64_ok)
    return launch_triprod(h, 0, vin, 4 * nxy, h->d_rsp.as<double>(), 8 * nxy, na, act);
  for (int ri = 0; ri < 2; ++ri) {
    if (!h->ngroups_q2s[ri]) continue;
    hipLaunchKernelGGL(k_triprod, dim3(h->ngroups_q2s[ri], na), dim3(256), h->lds_q2s, h->stream,
                       h->d_groups_q2s[ri].as<Group>(), h->d_terms_q2s[ri].as<Term>(), h->d_U[0].as<double>(),
                       h->d_U[1].as<double>(), h->d_U[2].as<double>(), h->d_U[3].as<double>(), vin, 4 * nxy, 4,
                       h->d_rsp.as<double>(), 8 * nxy, 8, act, nxy);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

int stage_fields(pnfam_gpu_ctx *h, int na, const int *act, const double *dens = nullptr, double *flds = nullptr,
                 bool grid1d = false) {
  FieldArgs F{};
  F.dens = dens ? dens : h->d_dens.as<double>(); F.flds = flds ? flds : h->d_flds.as<double>();
  F.crho = h->d_crho.as<double>(); F.cs = h->d_cs.as<double>(); F.cpair = h->d_cpair.as<double>();
  F.cspair = h->d_cspair.as<double>();
  const double *c = h->cscal.data();
  F.cdrho = c[0]; F.ctau = c[1]; F.ctj0 = c[2]; F.ctj1 = c[3]; F.ctj2 = c[4]; F.crdj = c[5];
  F.cds = c[6]; F.ct = c[7]; F.cj = c[8]; F.cgs = c[9]; F.cf = c[10]; F.csdj = c[11];
  F.nghl = h->nghl; F.act = act; F.skip = h->skip_slot;
  { Prof pr(h, K_FIELDS, na);
    if (grid1d) hipLaunchKernelGGL(k_fields<true>, dim3((h->nghl + 127) / 128, na, 2), dim3(128), 0, h->stream, F);
    else hipLaunchKernelGGL(k_fields<false>, dim3((h->nghl + 127) / 128, na, 2), dim3(128), 0, h->stream, F); }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Buffers of the FP64 grid stage: the context's batch workspace by default.
// rsp in the slot layout [w][8][nxy] with the sector-1 rho / kappa pairs at
// rho1 / kap1 (3 and 2 there; 2 and 3 in calc_dHsp_interface's argument
// order); split: few-point splits of the grid loops allowed (they need the
// partial buffers the context allocates).
struct GridBufs {
  const double *rsp;
  int rho1, kap1;
  double *dens, *flds, *hsp;
  bool split;
};

int stage_hamiltonian_on(pnfam_gpu_ctx *h, int na, const int *act, const GridBufs &gb) {
  DensArgs A{};
  A.wf = h->d_wf.as<double>(); A.wfdr = h->d_wfdr.as<double>(); A.wfdp = h->d_wfdp.as<double>();
  A.wfdz = h->d_wfdz.as<double>(); A.wdcori = h->d_wdcori.as<double>();
  A.isstart = h->d_isstart.as<int>(); A.db = h->d_db.as<int>(); A.nsu = h->d_nsu.as<int>(); A.ns = h->d_ns.as<int>();
  A.rsp = gb.rsp; A.nxy = h->nxy; A.nghl = h->nghl;
  const int4 *pl = h->d_pairs.as<int4>();
  A.rho[0] = PairList{pl + h->pair_off[0], h->pair_n[0]};
  A.kap[0] = PairList{pl + h->pair_off[1], h->pair_n[1]};
  A.rho[1] = PairList{pl + h->pair_off[2], h->pair_n[2]};
  A.kap[1] = PairList{pl + h->pair_off[3], h->pair_n[3]};
  // sector 0: rho_pn = m11 (slot 0), kappa+ = m12 (slot 1); sector 1: rho_np = m22 (3), kappa- = m21 (2)
  A.rho_slot[0] = 0; A.kap_slot[0] = 1; A.rho_slot[1] = gb.rho1; A.kap_slot[1] = gb.kap1;
  A.dens = gb.dens; A.act = act; A.skip = h->skip_slot;
  h->flops_unit[K_DENSITY] = h->gen_flops_d;
  h->flops_unit[K_PROJECT] = h->gen_flops_p;
  { Prof pr(h, K_DENSITY, na);
    if (h->basic_kernels) {
      note(h, "k_density");
      hipLaunchKernelGGL(k_density, dim3((h->nghl + 63) / 64, na, 2), dim3(64), 0, h->stream, A);
    } else {
      // few frequencies: split the pair lists so that the waves fill the device
      const int nsplit = gb.split ? few_split(na) : 1;
      note(h, (h->dens_pq == 2 && h->sorted_spins) ? "k_density_pq2" : (h->dens_pq ? "k_density_pq" : "k_density_mfma"),
           nsplit);
      const long nd = 2L * 2 * NDENS * h->nghl;
      if (nsplit > 1) {
        if (int e = h->d_dpart.alloc((size_t)FEW_SPLIT_SLABS * nd * 8)) return e;
        A.part = h->d_dpart.as<double>();
      }
      if (h->dens_pq == 2 && h->sorted_spins)
        hipLaunchKernelGGL(k_density_pq2, dim3((h->nghl + 15) / 16, na, 2 * nsplit), dim3(128), 0, h->stream, A);
      else if (h->dens_pq)
        hipLaunchKernelGGL(k_density_pq, dim3((h->nghl + 15) / 16, na, 2 * nsplit), dim3(128), 0, h->stream, A);
      else
        hipLaunchKernelGGL(k_density_mfma, dim3((h->nghl + 15) / 16, na, 2 * nsplit), dim3(64), 0, h->stream, A);
      if (nsplit > 1)
        hipLaunchKernelGGL(k_dens_sum, dim3((unsigned)std::min<long>(1024, (nd + 255) / 256), na), dim3(256), 0,
                           h->stream, A.part, nsplit, na, nd, act, gb.dens);
    } }
  if (int e = stage_fields(h, na, act, gb.dens, gb.flds)) return e;
  if (!(h->zero_skip && h->proj_cover && !h->basic_kernels)) {
    Prof pr(h, K_ZERO, na);
    hipLaunchKernelGGL(k_zero_slots, dim3(64, na), dim3(256), 0, h->stream, gb.hsp, act, 8, 0, 8, h->nxy,
                       h->skip_slot); }
  ProjArgs P{};
  P.psi[0] = h->d_wf.as<double>(); P.psi[1] = h->d_wfdr.as<double>(); P.psi[2] = h->d_wfdp.as<double>();
  P.psi[3] = h->d_wfdz.as<double>(); P.psi[4] = h->d_wfd2.as<double>();
  P.isstart = h->d_isstart.as<int>(); P.db = h->d_db.as<int>(); P.nsu = h->d_nsu.as<int>(); P.ns = h->d_ns.as<int>();
  P.flds = gb.flds; P.hsp = gb.hsp; P.nxy = h->nxy; P.nghl = h->nghl;
  P.tiles = h->d_tiles.as<Tile>(); P.act = act; P.skip = h->skip_slot;
  if (h->basic_kernels && h->ntiles) {
    Prof pr(h, K_PROJECT, na);
    note(h, "k_project");
    hipLaunchKernelGGL(k_project, dim3(h->ntiles, na), dim3(256), 0, h->stream, P);
  } else if (h->ntiles2) {
    Prof pr(h, K_PROJECT, na);
    const Tile2 *tl = h->d_tiles2.as<Tile2>();
    // few frequencies: split the grid points so that the waves fill the device
    // (one frequency leaves about one wave per SIMD with a serial loop over all
    // grid points)
    const int nsplit = gb.split ? few_split(na) : 1;
    const long n8 = 8 * h->nxy;
    if (nsplit > 1) {
      if (int e = h->d_ppart.alloc((size_t)FEW_SPLIT_SLABS * n8 * 8)) return e;
      P.part = h->d_ppart.as<double>();
      hipLaunchKernelGGL(k_fill, grid1((size_t)nsplit * na * n8, 256), dim3(256), 0, h->stream, P.part,
                         (size_t)nsplit * na * n8, 0.0);
    }
    const int ns = h->proj_ns;
    P.na = na;
    for (int k = 0; k < 16; ++k) {
      const int n = h->pj_count[k];
      if (!n) continue;
      // frequencies per wave: proj_freqs, or proj_freqs_rt1 for the mean-field
      // tiles of one row tile, whose few products per staged chunk make the
      // shared-operand workgroups slower than one frequency per wave (measured
      // at 128 points: 9.4 against 14.5 ms); with few points one (the split
      // keeps the device busy); the four-frequency workgroups below 16 points
      // leave too many waves idle (measured at 9 points: 1.4x slower)
      const int nfk = (k == 1 && h->proj_nf1) ? h->proj_nf1 : h->proj_nf;
      const int nf = (nsplit > 1 || na < 2 || (nfk == 4 && na < 16)) ? 1 : nfk;
      const dim3 grid(n, (na + nf - 1) / nf, nsplit);
      const Tile2 *tk = tl + h->pj_first[k];
      note(h, nf == 1 ? "k_project_mfma" : (nf == 2 ? "k_project_mfma_f2" : "k_project_lds"), k & 7, k >> 3);
      if (nsplit > 1) note(h, "k_proj_sum", nsplit);
#define PJ_LAUNCH(NRT, KIND)                                                                                  \
  do {                                                                                                        \
    if (nf == 4) hipLaunchKernelGGL((k_project_lds<NRT, KIND>), grid, dim3(256), 0, h->stream, P, tk);               \
    else if (nf == 2 && ns == 2) hipLaunchKernelGGL((k_project_mfma<NRT, KIND, 2, 2>), grid, dim3(64), 0, h->stream, P, tk); \
    else if (nf == 2) hipLaunchKernelGGL((k_project_mfma<NRT, KIND, 2, 1>), grid, dim3(64), 0, h->stream, P, tk);  \
    else if (ns == 2) hipLaunchKernelGGL((k_project_mfma<NRT, KIND, 1, 2>), grid, dim3(64), 0, h->stream, P, tk);  \
    else hipLaunchKernelGGL((k_project_mfma<NRT, KIND, 1, 1>), grid, dim3(64), 0, h->stream, P, tk);          \
  } while (0)
      switch (k) {
        case 1: PJ_LAUNCH(1, 0); break;
        case 2: PJ_LAUNCH(2, 0); break;
        case 3: PJ_LAUNCH(3, 0); break;
        case 4: PJ_LAUNCH(4, 0); break;
        case 9: PJ_LAUNCH(1, 1); break;
        case 10: PJ_LAUNCH(2, 1); break;
        case 11: PJ_LAUNCH(3, 1); break;
        case 12: PJ_LAUNCH(4, 1); break;
        default: return fail(PNFAM_GPU_EINVAL, "projection tile class out of range");
      }
#undef PJ_LAUNCH
    }
    if (nsplit > 1)
      hipLaunchKernelGGL(k_proj_sum, dim3((unsigned)std::min<long>(1024, (n8 + 255) / 256), na), dim3(256), 0,
                         h->stream, P.part, nsplit, na, n8, act, gb.hsp);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

// ---- FP64 grid stage on product grids (separable.hpp) ------------------------
constexpr int sep_pad8(int n) { return (n + 7) & ~7; }

// Points along z of the product grid: the first divisor of nghl, from nz on, for
// which the values of a few states are rank-one matrices; 0 if there is none.  The
// few can be rank one for a wrong one too: where they vanish on the outer half of
// the axis, so they are with half its points.
int sep_axial_points(const pnfam_gpu_basis *b, int nz) {
  const int G = b->nghl;
  for (; nz <= G / 2; ++nz) {
    if (G % nz || nz > SEP_MAX1D || G / nz > SEP_MAX1D) continue;
    bool ok = true;
    for (int k = 0; k < 3 && ok; ++k) {
      const double *M = b->wf + (size_t)((long)k * (b->dqp - 1) / 2) * G;
      int p = 0;
      for (int i = 1; i < G; ++i)
        if (std::fabs(M[i]) > std::fabs(M[p])) p = i;
      const int rp = p / nz, zp = p % nz;
      const double m = M[p], tol = 1e-12 * m * m;
      ok = m != 0.0;
      for (int i = 0; i < G && ok; ++i)
        ok = std::fabs(M[i] * m - M[rp * nz + i % nz] * M[(i / nz) * nz + zp]) <= tol;
    }
    if (ok) return nz;
  }
  return 0;
}

// Factors of the wavefunction tables, nz axial points; *ok: they are products.
int sep_fit(pnfam_gpu_ctx *h, int nz, std::vector<double> &fr, bool *ok) {
  const int nr = h->nghl / nz, D = h->dqp;
  DevPtr dfr, dres;
  int e;
  if ((e = dfr.alloc((size_t)D * 4 * nr * 8)) || (e = dres.alloc((size_t)D * 8)) ||
      (e = h->d_sep_fz.alloc((size_t)3 * D * sep_pad8(nz) * 8)))
    return e;
  SepFit S{};
  S.tab[0] = h->d_wf.as<double>(); S.tab[1] = h->d_wfdr.as<double>(); S.tab[2] = h->d_wfdp.as<double>();
  S.tab[3] = h->d_wfdz.as<double>(); S.tab[4] = h->d_wfd2.as<double>();
  S.nz = nz; S.nr = nr; S.dqp = D; S.nzp = sep_pad8(nz); S.fr = dfr.as<double>(); S.fz = h->d_sep_fz.as<double>();
  S.resid = dres.as<double>();
  hipLaunchKernelGGL(k_sep_fit, dim3(D), dim3(256), 0, h->stream, S);
  HIP_TRY(hipGetLastError());
  fr.resize((size_t)D * 4 * nr);
  std::vector<double> res(D);
  HIP_TRY(hipMemcpyAsync(fr.data(), dfr.p, fr.size() * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipMemcpyAsync(res.data(), dres.p, res.size() * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->sep_resid = 0.0;
  for (double r : res) h->sep_resid = r <= 1.0 ? std::max(h->sep_resid, r) : 1.0;
  *ok = h->sep_resid <= SEP_TOL;
  return 0;
}

// Factors of the wavefunction tables and the radial functions they share.
// Leaves sep_basis false where the tables are no products.
int sep_prepare(pnfam_gpu_ctx *h, const pnfam_gpu_basis *b) {
  std::vector<double> fr;
  bool ok = false;
  int nz = 1, e;
  while (!ok) {
    if (!(nz = sep_axial_points(b, nz + 1))) return 0;
    if ((e = sep_fit(h, nz, fr, &ok))) return e;
  }
  const int nr = b->nghl / nz, D = b->dqp;
  // radial functions equal to rounding (all four tables) form one class,
  // represented by the mean of its members
  std::vector<int> cls(D), first;
  std::vector<int> cnt;
  auto same = [&](int a, int c) {
    for (int x = 0; x < 4; ++x) {
      const double *u = &fr[((size_t)a * 4 + x) * nr], *v = &fr[((size_t)c * 4 + x) * nr];
      double m = 0.0;
      for (int r = 0; r < nr; ++r) m = std::max(m, std::fabs(v[r]));
      for (int r = 0; r < nr; ++r)
        if (!(std::fabs(u[r] - v[r]) <= SEP_SAME * m)) return false;
    }
    return true;
  };
  for (int a = 0; a < D; ++a) {
    int c = -1;
    for (size_t k = 0; k < first.size() && c < 0; ++k)
      if (same(a, first[k])) c = (int)k;
    if (c < 0) { c = (int)first.size(); first.push_back(a); cnt.push_back(0); }
    cls[a] = c;
    ++cnt[c];
  }
  const int nc = (int)first.size();
  std::vector<double> f((size_t)4 * nc * nr, 0.0);
  for (int a = 0; a < D; ++a)
    for (int x = 0; x < 4; ++x)
      for (int r = 0; r < nr; ++r) f[((size_t)x * nc + cls[a]) * nr + r] += fr[((size_t)a * 4 + x) * nr + r];
  for (int x = 0; x < 4; ++x)
    for (int c = 0; c < nc; ++c)
      for (int r = 0; r < nr; ++r) f[((size_t)x * nc + c) * nr + r] /= cnt[c];
  h->sep_groups.clear(); h->sep_members.clear();
  h->sep_gfirst.assign(2 * h->nb + 1, 0);
  for (int i = 0; i < h->nb; ++i)
    for (int s = 0; s < 2; ++s) {
      const int lo = s ? h->nsu[i] : 0, hi = s ? h->db[i] : h->nsu[i];
      std::vector<int> order;
      for (int k = lo; k < hi; ++k) order.push_back(k);
      std::stable_sort(order.begin(), order.end(),
                       [&](int a, int c) { return cls[h->isstart[i] + a] < cls[h->isstart[i] + c]; });
      h->sep_gfirst[2 * i + s] = (int)h->sep_groups.size();
      for (int k : order) {
        const int c = cls[h->isstart[i] + k];
        if ((int)h->sep_groups.size() == h->sep_gfirst[2 * i + s] || h->sep_groups.back().cls != c)
          h->sep_groups.push_back({c, (int)h->sep_members.size(), 0});
        h->sep_members.push_back(k);
        ++h->sep_groups.back().count;
      }
    }
  h->sep_gfirst[2 * h->nb] = (int)h->sep_groups.size();
  if ((e = upload(h->d_sep_f, f.data(), f.size() * 8, h->stream))) return e;
  HIP_TRY(hipStreamSynchronize(h->stream));   // pageable sources
  h->sep_nz = nz; h->sep_nr = nr; h->sep_ncls = nc;
  h->sep_basis = true;
  return 0;
}

// Plan for the block structures of the operator: slots, tables of radial
// products and the jobs of the four kernels.
int sep_build(pnfam_gpu_ctx *h) {
  h->sep_plan = false;
  if (!h->sep_basis) return 0;
  const int nz = h->sep_nz, nr = h->sep_nr, W = 2 * nz, W8 = 2 * sep_pad8(nz), nr4 = (nr + 3) & ~3;
  const BlockMap *dm[4] = {&h->rspmap[0], &h->rspmap[1], &h->rspmap[3], &h->rspmap[2]};   // rho0, kap0, rho1, kap1
  const BlockMap *pm[4] = {&h->hspmap[0], &h->hspmap[1], &h->hspmap[3], &h->hspmap[2]};   // h0, D0, h1, D1
  const int out_slot[4] = {0, 1, 3, 2};
  typedef std::vector<std::pair<int, int>> Keys;
  struct Tab { int kind, sa, sb; Keys keys; bool d = false, p = false; size_t key0 = 0, rd = 0, rp = 0; };
  std::vector<Tab> tabs;
  auto groups = [&](int blk, int s) {
    return std::make_pair(h->sep_gfirst[2 * blk + s], h->sep_gfirst[2 * blk + s + 1]);
  };
  // slots of one structure and pair of spins, in the order of (row, column) function
  auto keys_of = [&](const BlockMap &m, int sa, int sb) {
    Keys k;
    for (auto &p : pair_list(m)) {
      const auto ga = groups(p.x, sa), gb = groups(p.y, sb);
      for (int i = ga.first; i < ga.second; ++i)
        for (int j = gb.first; j < gb.second; ++j) k.push_back({h->sep_groups[i].cls, h->sep_groups[j].cls});
    }
    std::sort(k.begin(), k.end());
    k.erase(std::unique(k.begin(), k.end()), k.end());
    return k;
  };
  int dtab[16], ptab[16];
  for (int q = 0; q < 16; ++q) {
    const int mat = q >> 2, sa = (q >> 1) & 1, sb = q & 1, kind = mat & 1;
    for (int side = 0; side < 2; ++side) {
      Keys k = keys_of(side ? *pm[mat] : *dm[mat], sa, sb);
      int t = -1;
      for (size_t i = 0; i < tabs.size() && t < 0; ++i)
        if (tabs[i].kind == kind && tabs[i].sa == sa && tabs[i].sb == sb && tabs[i].keys == k) t = (int)i;
      if (t < 0) {
        t = (int)tabs.size();
        tabs.push_back({kind, sa, sb, std::move(k)});
      }
      (side ? tabs[t].p : tabs[t].d) = true;
      (side ? ptab : dtab)[q] = t;
    }
  }
  auto slot_id = [&](const Tab &t, int ca, int cb) {
    return (int)(std::lower_bound(t.keys.begin(), t.keys.end(), std::make_pair(ca, cb)) - t.keys.begin());
  };
  // a point's Z and Y; their offsets are 32-bit: a larger basis keeps the other kernels
  // (decided before the first copy, whose sources end with this function)
  long zall = 0, yall = 0;
  for (int q = 0; q < 16; ++q) {
    const bool pair = (q >> 2) & 1;
    zall += (long)tabs[dtab[q]].keys.size() * (pair ? 1 : SEP_NT) * W;
    yall += (long)tabs[ptab[q]].keys.size() * (pair ? 1 : SEP_PT) * W8;
  }
  if (zall > (1L << 30) || yall > (1L << 30)) return 0;
  std::vector<int2> keys;
  size_t doubles = 0;
  for (auto &t : tabs) {
    const size_t n = t.keys.size();
    const bool same = t.sa == t.sb;
    t.key0 = keys.size();
    for (auto &k : t.keys) keys.push_back(make_int2(k.first, k.second));
    if (t.d) { t.rd = doubles; doubles += ((n + 3) & ~size_t(3)) * sep_row0(t.kind, same, SEP_NT, nr); }
    if (t.p) { t.rp = doubles; doubles += ((n + 15) & ~size_t(15)) * sep_k0(t.kind, same, SEP_PT, nr4); }
  }
  int e;
  if ((e = upload(h->d_sep_keys, keys.data(), std::max<size_t>(1, keys.size()) * sizeof(int2), h->stream)) ||
      (e = h->d_sep_tabs.alloc(std::max<size_t>(1, doubles) * 8)))
    return e;
  double *tb = h->d_sep_tabs.as<double>();
  for (auto &t : tabs) {
    if (t.keys.empty()) continue;
    const SepTab T{h->d_sep_keys.as<int2>() + t.key0, (int)t.keys.size(), t.kind, t.sa, t.sb, t.d ? tb + t.rd : nullptr,
                   t.p ? tb + t.rp : nullptr};
    hipLaunchKernelGGL(k_sep_rtab, dim3(512), dim3(256), 0, h->stream, T, h->d_sep_f.as<double>(), nr, h->sep_ncls);
  }
  HIP_TRY(hipGetLastError());
  // column tiles per wave: at most five (20 accumulator tiles)
  for (int k = 0; k < 2; ++k) {
    const int nct = ((k ? W8 : W) + 15) / 16;
    h->sep_ncg[k] = (nct + 4) / 5;
    h->sep_ct[k] = (nct + h->sep_ncg[k] - 1) / h->sep_ncg[k];
    if (k) h->sep_nct1 = nct;
  }
  std::vector<SepSlot> slots[2];
  std::vector<int4> elems[2];
  struct Bundle { int first, count; };   // slots with the same columns
  std::vector<Bundle> bundles[2];
  std::vector<std::vector<SepDJob>> dgroups;
  std::vector<std::vector<SepPJob>> pgroups[2];
  long zoff = 0, yoff = 0, arow = 0;
  h->sep_flops_d = h->sep_flops_p = 0;
  // the slots of one class with their elements; each slot takes `ld` doubles from `at` on
  auto put_slots = [&](int side, int q, const Tab &T, const BlockMap &m, long at, long ld) {
    const int mat = q >> 2, sa = (q >> 1) & 1, sb = q & 1;
    std::vector<std::vector<int4>> el(T.keys.size());
    for (auto &p : pair_list(m)) {
      const auto ga = groups(p.x, sa), gb = groups(p.y, sb);
      for (int i = ga.first; i < ga.second; ++i)
        for (int j = gb.first; j < gb.second; ++j) {
          const auto &A = h->sep_groups[i], &B = h->sep_groups[j];
          auto &v = el[slot_id(T, A.cls, B.cls)];
          for (int b = 0; b < B.count; ++b)
            for (int a = 0; a < A.count; ++a) {
              const int al = h->sep_members[A.first + a], bl = h->sep_members[B.first + b];
              v.push_back(make_int4(p.z + al + bl * h->db[p.x], h->isstart[p.x] + al, h->isstart[p.y] + bl, 0));
            }
        }
    }
    // in the order of the columns' function, one bundle for each
    std::vector<int> order(el.size());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int c) { return T.keys[a].second < T.keys[c].second; });
    for (size_t k = 0; k < order.size(); ++k) {
      const int s = order[k];
      if (k == 0 || T.keys[s].second != T.keys[order[k - 1]].second) bundles[side].push_back({(int)slots[side].size(), 0});
      ++bundles[side].back().count;
      slots[side].push_back({(int)elems[side].size(), (int)el[s].size(), mat, (int)(at + (long)s * ld)});
      elems[side].insert(elems[side].end(), el[s].begin(), el[s].end());
    }
  };
  for (int q = 0; q < 16; ++q) {
    const int mat = q >> 2, sa = (q >> 1) & 1, sb = q & 1, kind = mat & 1;
    const bool same = sa == sb;
    {   // densities
      const Tab &T = tabs[dtab[q]];
      const int n = (int)T.keys.size(), nt = kind ? 1 : SEP_NT, ld = sep_row0(kind, same, SEP_NT, nr);
      put_slots(0, q, T, *dm[mat], zoff, (long)nt * W);
      h->sep_acc.row[q] = n ? (int)arow : -1;
      for (int t = 0; t < nt && n; ++t) {
        const int r0 = sep_row0(kind, same, t, nr), r1 = sep_row0(kind, same, t + 1, nr), tiles = (r1 - r0) / 16;
        const int nw = (tiles + 3) / 4;             // waves: at most four row tiles each, evenly
        std::vector<SepDJob> g;                     // one group: they read the same Z rows
        for (int k = 0, r = r0; k < nw; ++k) {
          const int q = tiles / nw + (k < tiles % nw ? 1 : 0);
          g.push_back({(int64_t)T.rd, n, ld, r, q, (int)(zoff + (long)t * W), nt * W, (int)arow + r, 0});
          r += 16 * q;
        }
        dgroups.push_back(g);
        h->sep_flops_d += 2.0 * n * sep_rows(kind, same, t) * nr * W;
      }
      zoff += (long)n * nt * W;
      arow += n ? ld : 0;
    }
    {   // projection
      const Tab &T = tabs[ptab[q]];
      const int n = (int)T.keys.size(), nt = kind ? 1 : SEP_PT, ld = (n + 15) & ~15;
      put_slots(1, q, T, *pm[mat], yoff, (long)nt * W8);
      for (int t = 0; t < nt && n; ++t) {
        h->sep_flops_p += 2.0 * n * sep_terms(kind, same, t) * nr * W;
        uint64_t fields = 0;
        for (int c = sep_terms(kind, same, t) - 1; c >= 0; --c) fields = fields << 7 | (uint64_t)sep_field(kind, t, c, sa, sb);
        for (int v = 0; v < 2; ++v) {
          const int rt = v ? 4 : 1;
          std::vector<SepPJob> g;                   // one group: they read the same fields
          for (int s = 0; s < ld; s += 16 * rt) {
            if ((int)g.size() == SEP_PRUN) { pgroups[v].push_back(g); g.clear(); }
            g.push_back({(int64_t)(T.rp + (size_t)sep_k0(kind, same, t, nr4) * ld), fields, ld, n, s,
                         std::min(rt, (ld - s) / 16), sep_terms(kind, same, t), mat >> 1, (int)(yoff + (long)t * W8),
                         nt * W8});
          }
          g.resize(SEP_PRUN, SepPJob{});
          pgroups[v].push_back(g);
        }
      }
      yoff += (long)n * nt * W8;
    }
    // per element: the axial products of the densities and of the expansion
    h->sep_flops_d += (kind ? 4.0 : 16.0) * nz * (double)dm[mat]->nelem(h->db) / 4;
    h->sep_flops_p += (kind ? 4.0 : 20.0) * nz * (double)pm[mat]->nelem(h->db) / 4;
  }
  // the job groups go to the XCD with the least work so far, the costliest group
  // first; lists of unequal length end in empty jobs
  auto deal = [](auto &groups, auto cost, auto &all) {
    auto sum = [&](const auto &g) {
      long c = 0;
      for (auto &j : g) c += cost(j);
      return c;
    };
    std::stable_sort(groups.begin(), groups.end(), [&](const auto &a, const auto &b) { return sum(a) > sum(b); });
    typename std::remove_reference<decltype(groups[0])>::type list[8];
    long load[8] = {};
    for (auto &g : groups) {
      const int x = (int)(std::min_element(load, load + 8) - load);
      load[x] += sum(g);
      list[x].insert(list[x].end(), g.begin(), g.end());
    }
    size_t len = 0;
    for (auto &l : list) len = std::max(len, l.size());
    all.assign(8 * len, typename std::remove_reference<decltype(all[0])>::type{});
    for (int x = 0; x < 8; ++x) std::copy(list[x].begin(), list[x].end(), all.begin() + x * len);
  };
  std::vector<SepDJob> djobs;
  std::vector<SepPJob> pjobs[2];
  deal(dgroups, [](const SepDJob &j) { return (long)j.n * j.nrt; }, djobs);
  for (int v = 0; v < 2; ++v) deal(pgroups[v], [](const SepPJob &j) { return (long)j.nc * j.nst; }, pjobs[v]);
  // the bundles dealt to the eight XCDs in turn, the costliest first; workgroup x
  // (four slots) runs on XCD x % 8, lists of unequal length end in empty slots
  for (int k = 0; k < 2; ++k) {
    auto cost = [&](const Bundle &b) {
      long c = 0;
      for (int i = 0; i < b.count; ++i) {
        const SepSlot &s = slots[k][b.first + i];
        c += (long)(s.count + 16) * ((s.mat & 1) ? 1 : 4);
      }
      return c;
    };
    std::stable_sort(bundles[k].begin(), bundles[k].end(), [&](const Bundle &a, const Bundle &b) { return cost(a) > cost(b); });
    std::vector<SepSlot> xcd[8];
    for (size_t i = 0; i < bundles[k].size(); ++i) {
      auto &x = xcd[i % 8];
      const auto first = slots[k].begin() + bundles[k][i].first;
      x.insert(x.end(), first, first + bundles[k][i].count);
    }
    size_t len = 0;
    for (auto &x : xcd) len = std::max(len, (x.size() + 3) / 4 * 4);
    std::vector<SepSlot> all(8 * len, SepSlot{0, 0, 0, 0});
    for (int x = 0; x < 8; ++x)
      for (size_t i = 0; i < xcd[x].size(); ++i) all[((i / 4) * 8 + x) * 4 + i % 4] = xcd[x][i];
    slots[k].swap(all);
  }
  std::vector<SepPJob> pj(pjobs[0]);
  pj.insert(pj.end(), pjobs[1].begin(), pjobs[1].end());
  for (int k = 0; k < 2; ++k) {
    h->sep_nslot[k] = (int)slots[k].size();
    if ((e = upload(h->d_sep_slots[k], slots[k].data(), std::max<size_t>(1, slots[k].size()) * sizeof(SepSlot), h->stream)) ||
        (e = upload(h->d_sep_elems[k], elems[k].data(), std::max<size_t>(1, elems[k].size()) * sizeof(int4), h->stream)))
      return e;
  }
  if ((e = upload(h->d_sep_djobs, djobs.data(), std::max<size_t>(1, djobs.size()) * sizeof(SepDJob), h->stream)) ||
      (e = upload(h->d_sep_pjobs, pj.data(), std::max<size_t>(1, pj.size()) * sizeof(SepPJob), h->stream)))
    return e;
  HIP_TRY(hipStreamSynchronize(h->stream));   // pageable sources
  h->sep_ndjob = (int)djobs.size();
  h->sep_nwork = (int)std::count_if(djobs.begin(), djobs.end(), [](const SepDJob &j) { return j.n > 0; });
  for (int v = 0; v < 2; ++v) {
    h->sep_pjob0[v] = v ? (int)pjobs[0].size() : 0;
    h->sep_npjob[v] = (int)pjobs[v].size();
  }
  h->sep_zstride = zoff; h->sep_ystride = yoff; h->sep_arows = arow;
  h->sep_plan = !djobs.empty() && !pj.empty();
  return 0;
}

bool sep_active(const pnfam_gpu_ctx *h) {
  return h->sep_plan && h->fp64_grid == 0 && !h->basic_kernels && !h->sep_nomem;
}

// Projection below eight points: one column tile per wave while that gives at most
// this many waves (16 per CU; beyond, the operands read once per column tile cost
// more than the shorter chains save: one point 21 us against 29 at N_sh = 8,
// 18 against 25 at N_sh = 10).
constexpr long SEP_PFEW = 4096;

// Points a pass of the separable stage takes at once, and the splits of its
// density contraction: with few points the slots are split so that about 2 048
// waves run.  The limit only bounds the memory (N_sh = 16: 20 MB per point; 128
// points in passes of 32 take 4 % longer than in one, 64 1 %); a pass of one point
// may exceed it, unless the caller has set the limit (option fp64_grid_bytes): then
// 0 points a pass, where not even one fits.
constexpr size_t SEP_CHUNK_BYTES = size_t(4) << 30;
size_t sep_point_bytes(const pnfam_gpu_ctx *h) {
  return (size_t)std::max<long>(1, std::max(h->sep_zstride, h->sep_ystride)) * 8;
}
int sep_chunk(const pnfam_gpu_ctx *h, int na) {
  const size_t n = (h->sep_limit ? h->sep_limit : SEP_CHUNK_BYTES) / sep_point_bytes(h);
  return (int)std::min<size_t>((size_t)na, h->sep_limit ? n : std::max<size_t>(1, n));
}
int sep_split(const pnfam_gpu_ctx *h, int nc, bool split) {
  if (!split) return 1;
  const long waves = (long)h->sep_nwork * h->sep_ncg[0] * nc;
  return (int)std::max<long>(1, std::min<long>(16, 2048 / std::max<long>(1, waves)));
}

// Device memory of a pass over na points, before any launch (a captured pass
// cannot allocate); without it nothing is held.
int sep_workspace(pnfam_gpu_ctx *h, int na) {
  const int nc = sep_chunk(h, na);
  // split counts fall as the points rise: the most partial sums any count up to nc needs
  long parts = 0;
  for (int n = 1; n <= nc; ++n) parts = std::max(parts, (long)n * sep_split(h, n, true));
  int e = nc ? h->d_sep_zy.alloc((size_t)nc * sep_point_bytes(h))
             : fail(PNFAM_GPU_ENOMEM, "fp64_grid_bytes is below the need of one point");
  if (!e) e = h->d_sep_part.alloc((size_t)parts * h->sep_arows * 2 * h->sep_nz * 8);
  if (e) sep_release(h);
  return e;
}

// Densities, fields and projection through the separable kernels.
int stage_hamiltonian_sep(pnfam_gpu_ctx *h, int na, const int *act, const GridBufs &gb) {
  SepArgs A{};
  A.nz = h->sep_nz; A.nr = h->sep_nr; A.dqp = h->dqp; A.nxy = h->nxy;
  A.nzp = sep_pad8(A.nz); A.fz = h->d_sep_fz.as<double>(); A.tab = h->d_sep_tabs.as<double>();
  A.rsp = gb.rsp; A.dens = gb.dens; A.flds = gb.flds; A.hsp = gb.hsp; A.wdcori = h->d_wdcori.as<double>();
  A.slot_of[0] = 0; A.slot_of[1] = 1; A.slot_of[2] = gb.rho1; A.slot_of[3] = gb.kap1;
  A.zy = h->d_sep_zy.as<double>(); A.zstride = h->sep_zstride; A.ystride = h->sep_ystride;
  A.acc = h->d_sep_part.as<double>(); A.astride = h->sep_arows * 2 * h->sep_nz; A.skip = h->skip_slot;
  h->flops_unit[K_DENSITY] = h->sep_flops_d;
  h->flops_unit[K_PROJECT] = h->sep_flops_p;
  const int C = sep_chunk(h, na), G = h->nghl;
  for (int c0 = 0; c0 < na; c0 += C) {
    const int nc = std::min(C, na - c0);
    A.act = act + c0;
    A.na = nc;
    { Prof pr(h, K_DENSITY, nc);
      const int ns = sep_split(h, nc, gb.split);
      note(h, "k_sep_dens", h->sep_ct[0], ns);
      const int zt = (h->sep_nz + 15) / 16, zg = (zt + 2) / 3;
      if (nc > 8) note(h, "k_sep_z_wide", nc > 16 ? 4 : 2);
      else note(h, "k_sep_z");
      const SepSlot *sl = h->d_sep_slots[0].as<SepSlot>();
      const int4 *el = h->d_sep_elems[0].as<int4>();
#define SEP_Z(ZT)                                                                                                      \
  do {                                                                                                                 \
    if (nc > 16)                                                                                                       \
      hipLaunchKernelGGL((k_sep_z_wide<ZT, 4>), dim3(h->sep_nslot[0], (nc + 31) / 32, zg), dim3(256), 0, h->stream, A, \
                         sl, el);                                                                                      \
    else if (nc > 8)                                                                                                   \
      hipLaunchKernelGGL((k_sep_z_wide<ZT, 2>), dim3(h->sep_nslot[0], 1, zg), dim3(128), 0, h->stream, A, sl, el);     \
    else                                                                                                               \
      hipLaunchKernelGGL(k_sep_z<ZT>, dim3(h->sep_nslot[0] / 4, 1, zg), dim3(256), 0, h->stream, A, sl, el);           \
  } while (0)
      switch ((zt + zg - 1) / zg) {
        case 1: SEP_Z(1); break;
        case 2: SEP_Z(2); break;
        default: SEP_Z(3); break;
      }
#undef SEP_Z
      const dim3 grid(h->sep_ndjob * nc, h->sep_ncg[0] * ns);
#define SEP_D(CT) hipLaunchKernelGGL(k_sep_dens<CT>, grid, dim3(64), 0, h->stream, A, h->d_sep_djobs.as<SepDJob>(), h->sep_ndjob, h->sep_ncg[0], ns)
      switch (h->sep_ct[0]) {
        case 1: SEP_D(1); break;
        case 2: SEP_D(2); break;
        case 3: SEP_D(3); break;
        case 4: SEP_D(4); break;
        default: SEP_D(5); break;
      }
#undef SEP_D
      if (ns > 1)
        hipLaunchKernelGGL(k_sep_sum, grid1((size_t)nc * A.astride, 256), dim3(256), 0, h->stream, A.acc, ns,
                           (long)nc * A.astride);
      hipLaunchKernelGGL(k_sep_combine, dim3((G + 63) / 64, nc, 4), dim3(64), 0, h->stream, A, h->sep_acc);
    }
    if (int e = stage_fields(h, nc, A.act, gb.dens, gb.flds, true)) return e;
    if (!(h->zero_skip && h->proj_cover)) {
      Prof pr(h, K_ZERO, nc);
      hipLaunchKernelGGL(k_zero_slots, dim3(64, nc), dim3(256), 0, h->stream, gb.hsp, A.act, 8, 0, 8, h->nxy,
                         h->skip_slot);
    }
    { Prof pr(h, K_PROJECT, nc);
      const int v = nc >= 8 ? 1 : 0;   // four slot tiles per wave from eight points, one below
      const int np = h->sep_npjob[v], ct = !v && (long)np * nc * h->sep_nct1 <= SEP_PFEW ? 1 : h->sep_ct[1];
      note(h, "k_sep_proj", ct, v ? 4 : 1);
      const dim3 grid(np * nc, (h->sep_nct1 + ct - 1) / ct);
      const SepPJob *pj = h->d_sep_pjobs.as<SepPJob>() + h->sep_pjob0[v];
#define SEP_P(CT)                                                                                    \
  do {                                                                                               \
    if (v) hipLaunchKernelGGL((k_sep_proj<CT, 4>), grid, dim3(64), 0, h->stream, A, pj, np);         \
    else hipLaunchKernelGGL((k_sep_proj<CT, 1>), grid, dim3(64), 0, h->stream, A, pj, np);           \
  } while (0)
      switch (ct) {
        case 1: SEP_P(1); break;
        case 2: SEP_P(2); break;
        case 3: SEP_P(3); break;
        case 4: SEP_P(4); break;
        default: SEP_P(5); break;
      }
#undef SEP_P
      if (nc > 8) note(h, "k_sep_expand_wide", nc > 16 ? 4 : 2);
      else note(h, "k_sep_expand");
      const SepSlot *sl = h->d_sep_slots[1].as<SepSlot>();
      const int4 *el = h->d_sep_elems[1].as<int4>();
      if (nc > 16)
        hipLaunchKernelGGL(k_sep_expand_wide<4>, dim3(h->sep_nslot[1], (nc + 31) / 32), dim3(256), 0, h->stream, A, sl, el);
      else if (nc > 8)
        hipLaunchKernelGGL(k_sep_expand_wide<2>, dim3(h->sep_nslot[1], 1), dim3(128), 0, h->stream, A, sl, el);
      else
        hipLaunchKernelGGL(k_sep_expand, dim3(h->sep_nslot[1] / 4), dim3(256), 0, h->stream, A, sl, el);
    }
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

int stage_hamiltonian(pnfam_gpu_ctx *h, int na, const int *act) {
  const GridBufs gb{h->d_rsp.as<double>(), 3, 2, h->d_dens.as<double>(), h->d_flds.as<double>(), h->d_hsp.as<double>(),
                    h->few_split_on != 0};
  // without memory for the separable stage's intermediates the general kernels run,
  // to the end of the call: an allocation that failed is not tried every iteration
  if (sep_active(h)) {
    if (sep_workspace(h, na) == 0) return stage_hamiltonian_sep(h, na, act, gb);
    h->sep_nomem = true;
  }
  return stage_hamiltonian_on(h, na, act, gb);
}

// ---- split-BF16 grid stage (mixed path) ------------------------------------
bool same_pairs(const BlockMap &a, const BlockMap &b) {
  const auto pa = pair_list(a), pb = pair_list(b);
  if (pa.size() != pb.size()) return false;
  for (size_t i = 0; i < pa.size(); ++i)
    if (pa[i].x != pb[i].x || pa[i].y != pb[i].y || pa[i].z != pb[i].z) return false;
  return true;
}

// Element order, pair tables and GEMM jobs of one block structure.
int mix_build_set(pnfam_gpu_ctx *h, pnfam_gpu_ctx::MixSet &S, const BlockMap &m, int ntp, int ntd) {
  std::vector<int> elem, sa, sb;
  const auto pl = pair_list(m);
  for (int cls = 0; cls < 4; ++cls) {
    S.kbeg[cls] = (int)elem.size();
    const int ca = cls >> 1, cb = cls & 1;
    for (const auto &p : pl) {
      const int dx = h->db[p.x], dy = h->db[p.y], nx = h->nsu[p.x], ny = h->nsu[p.y];
      const int a0 = ca ? nx : 0, a1 = ca ? dx : nx, b0 = cb ? ny : 0, b1 = cb ? dy : ny;
      for (int b = b0; b < b1; ++b)
        for (int a = a0; a < a1; ++a) {
          elem.push_back(p.z + a + b * dx);
          sa.push_back(h->isstart[p.x] + a);
          sb.push_back(h->isstart[p.y] + b);
        }
    }
    while (elem.size() % MIX_KALIGN) { elem.push_back(-1); sa.push_back(-1); sb.push_back(-1); }
  }
  S.kbeg[4] = (int)elem.size();
  S.Kp = S.kbeg[4];
  S.ntp = ntp; S.ntd = ntd;
  S.maxcount = 0;
  for (int c = 0; c < 4; ++c) S.maxcount = std::max(S.maxcount, S.kbeg[c + 1] - S.kbeg[c]);
  int e;
  if ((e = upload(S.d_elem, elem.data(), elem.size() * 4, h->stream)) ||
      (e = upload(S.d_sa, sa.data(), sa.size() * 4, h->stream)) ||
      (e = upload(S.d_sb, sb.data(), sb.size() * 4, h->stream)))
    return e;
  const size_t ntab = (size_t)S.Kp * h->RP;
  if ((e = S.TPh.alloc(ntp * ntab * 2)) || (e = S.TPl.alloc(ntp * ntab * 2)) || (e = S.TDh.alloc(ntd * ntab * 2)) ||
      (e = S.TDl.alloc(ntd * ntab * 2)))
    return e;
  TabArgs T{};
  T.psi[0] = h->d_wf.as<double>(); T.psi[1] = h->d_wfdr.as<double>(); T.psi[2] = h->d_wfdp.as<double>();
  T.psi[3] = h->d_wfdz.as<double>(); T.psi[4] = h->d_wfd2.as<double>();
  T.sa = S.d_sa.as<int>(); T.sb = S.d_sb.as<int>();
  for (int c = 0; c < 5; ++c) T.kbeg[c] = S.kbeg[c];
  T.Kp = S.Kp; T.nghl = h->nghl; T.RP = h->RP; T.single = ntp == 1;
  T.nc = ntp; T.dens = 0; T.hi = S.TPh.as<__bf16>(); T.lo = S.TPl.as<__bf16>();
  hipLaunchKernelGGL(k_mix_tables, dim3(2048, ntp), dim3(256), 0, h->stream, T);
  T.nc = ntd; T.dens = 1; T.hi = S.TDh.as<__bf16>(); T.lo = S.TDl.as<__bf16>();
  hipLaunchKernelGGL(k_mix_tables, dim3(2048, ntd), dim3(256), 0, h->stream, T);
  HIP_TRY(hipGetLastError());
  // density jobs: table rows (c, r), K = the class range; projection jobs: table
  // rows = the class range, K = (c, r)
  GemmJob jd[4], jp[4];
  for (int c = 0; c < 4; ++c) {
    jd[c] = GemmJob{0, ntd * h->RP, S.kbeg[c], S.kbeg[c + 1] - S.kbeg[c], c, 0};
    jp[c] = GemmJob{S.kbeg[c], S.kbeg[c + 1] - S.kbeg[c], 0, h->RP, c, 0};
  }
  if ((e = upload(S.d_jobs_dens, jd, sizeof(jd), h->stream)) || (e = upload(S.d_jobs_proj, jp, sizeof(jp), h->stream)))
    return e;
  return 0;
}

int fac_prepare(pnfam_gpu_ctx *h);

int mix_prepare(pnfam_gpu_ctx *h) {
  if (h->mix_ready) return 0;
  if (!same_pairs(h->rspmap[0], h->fmap) || !same_pairs(h->rspmap[3], h->fmap))
    return fail(PNFAM_GPU_EINVAL, "mixed path: rho_pn / rho_np structure differs from f");
  if (!same_pairs(h->rspmap[1], h->hspmap[1]) || !same_pairs(h->rspmap[2], h->hspmap[2]))
    return fail(PNFAM_GPU_EINVAL, "mixed path: kappa structure differs from Delta");
  h->RP = (h->nghl + MIX_RALIGN - 1) / MIX_RALIGN * MIX_RALIGN;
  if (const char *ev = std::getenv("PNFAM_GPU_MIX_GEMM")) h->own_gemm = std::strcmp(ev, "own") == 0;
  if (!h->mix_grid_set) {
    h->mix_grid = 0;
    if (const char *ev = std::getenv("PNFAM_GPU_MIX_GRID")) {
      if (std::strcmp(ev, "tables") == 0) h->mix_grid = 1;
      else if (std::strcmp(ev, "factored") == 0) h->mix_grid = 2;
      else if (std::strcmp(ev, "auto") != 0) return fail(PNFAM_GPU_EINVAL, "PNFAM_GPU_MIX_GRID must be tables, factored or auto");
    }
  }
  if (!h->mix_auto_set)
    if (const char *ev = std::getenv("PNFAM_GPU_MIX_AUTO_N")) h->mix_auto_n = std::atoi(ev);
  if (h->mix_grid == 0) {
    // auto: the pair tables only where they take at most mix_table_frac of the
    // free device memory (BF16 hi and lo, NPROJ_C + NDENS_C combinations of the
    // mean-field structure, one of each pairing structure); otherwise the
    // factored kernels take every pass
    auto elems = [&](const BlockMap &m) {
      double n = 0;
      for (const auto &p : pair_list(m)) n += (double)h->db[p.x] * h->db[p.y];
      return n;
    };
    const double bytes = ((NPROJ_C + NDENS_C) * elems(h->fmap) + 2.0 * (elems(h->hspmap[1]) + elems(h->hspmap[2]))) *
                         (double)h->RP * 4.0;
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) return fail(PNFAM_GPU_EDEVICE, "hipMemGetInfo failed");
    h->mix_table_bytes = bytes;
    if (bytes > h->mix_table_frac * (double)fr) h->mix_grid = 2;
  }
  if (h->mix_grid != 1)
    if (int e = fac_prepare(h)) return e;
  if (h->mix_grid == 2) {   // factored only: no pair tables
    h->mix_ready = true;
    return 0;
  }
  if (!h->own_gemm && !h->blas) {
    if (rocblas_create_handle(&h->blas) != rocblas_status_success)
      return fail(PNFAM_GPU_EDEVICE, "rocblas_create_handle failed");
    if (rocblas_set_stream(h->blas, h->stream) != rocblas_status_success)
      return fail(PNFAM_GPU_EDEVICE, "rocblas_set_stream failed");
  }
  int e;
  if ((e = mix_build_set(h, h->mix[0], h->fmap, NPROJ_C, NDENS_C))) return e;
  if ((e = mix_build_set(h, h->mix[1], h->hspmap[1], 1, 1))) return e;
  if ((e = mix_build_set(h, h->mix[2], h->hspmap[2], 1, 1))) return e;
  h->mix_ready = true;
  h->mix_cap = 0;
  // MFMA-issued FLOP per frequency and BF16 product (a pass issues one or
  // three products; padded element and grid ranges included)
  double fd = 0, fp = 0;
  for (int si = 0; si < 3; ++si) {
    const double cols = si == 0 ? 4.0 : 2.0;
    fd += 2.0 * h->mix[si].ntd * (double)h->RP * h->mix[si].Kp * cols;
    fp += 2.0 * h->mix[si].ntp * (double)h->RP * h->mix[si].Kp * cols;
  }
  h->flops_unit[K_MIX_GEMM_D] = fd;
  h->flops_unit[K_MIX_GEMM_P] = fp;
  return 0;
}

constexpr int64_t MIX_KCHUNK = 2048;   // K chunk of the split-K contractions

int mix_workspace(pnfam_gpu_ctx *h, int cap) {
  if (cap <= h->mix_cap) return 0;
  h->mix_cap = 0;   // set again only once every buffer below is in place
  const size_t RP = h->RP;
  for (int si = 0; si < 3; ++si) {
    auto &S = h->mix[si];
    const size_t ncol = (si == 0 ? 4 : 2) * (size_t)cap;
    const size_t nF = (si == 0 ? 4 * (size_t)NPROJ_C : 4) * ncol * RP;
    int e;
    if ((e = S.Bh.alloc(ncol * S.Kp * 2)) || (e = S.Bl.alloc(ncol * S.Kp * 2)) ||
        (e = S.O.alloc(4 * (size_t)S.ntd * RP * ncol * 4)) || (e = S.Fh.alloc(nF * 2)) || (e = S.Fl.alloc(nF * 2)))
      return e;
  }
  size_t kmax = 0;
  for (int si = 0; si < 3; ++si) kmax = std::max(kmax, (size_t)h->mix[si].Kp);
  if (int e = h->d_Oproj.alloc(kmax * 4 * (size_t)cap * 4)) return e;
  // split-K planes of the pairing-set density contractions and of the
  // mean-field ones (at most four planes: dens_kchunk splits in three)
  size_t psz = 4 * (size_t)h->mix[0].ntd * RP * 4 * (size_t)cap;
  for (int si = 1; si < 3; ++si) {
    const auto &S = h->mix[si];
    for (int c = 0; c < 4; ++c) {
      const size_t kl = (size_t)(S.kbeg[c + 1] - S.kbeg[c]);
      const size_t np = kl / MIX_KCHUNK + 1;
      psz = std::max(psz, np * (size_t)S.ntd * RP * 2 * (size_t)cap);
    }
  }
  if (int e = h->d_Psplit.alloc(std::max<size_t>(psz, 1) * 4)) return e;
  h->mix_cap = cap;
  return 0;
}

// C[s][t] (t-major, ld = ldc) (+)= sum_k S[s][k] T[t][k]: column-major
// C(s, t) = S^T(s, k) T(k, t) with both operands K-contiguous.
int blas_nt(pnfam_gpu_ctx *h, int64_t ns, int64_t nt, int64_t k, const __bf16 *S, int64_t lds, const __bf16 *T,
            int64_t ldt, float *C, int64_t ldc, bool accumulate) {
  const float alpha = 1.0f, beta = accumulate ? 1.0f : 0.0f;
  const rocblas_status st = rocblas_gemm_ex_64(h->blas, rocblas_operation_transpose, rocblas_operation_none, ns, nt, k,
                                               &alpha, S, rocblas_datatype_bf16_r, lds, T, rocblas_datatype_bf16_r, ldt,
                                               &beta, C, rocblas_datatype_f32_r, ldc, C, rocblas_datatype_f32_r, ldc,
                                               rocblas_datatype_f32_r, rocblas_gemm_algo_standard, 0, 0);
  if (st != rocblas_status_success) return fail(PNFAM_GPU_EDEVICE, "rocblas_gemm_ex failed: " + std::to_string(st));
  return 0;
}

// As blas_nt for `batch` consecutive K chunks of length k: chunk j reads
// S + j k, T + j k and writes its own output plane C + j cstride.
int blas_nt_chunks(pnfam_gpu_ctx *h, int64_t ns, int64_t nt, int64_t k, int64_t batch, const __bf16 *S, int64_t lds,
                   const __bf16 *T, int64_t ldt, float *C, int64_t ldc, int64_t cstride, bool accumulate) {
  const float alpha = 1.0f, beta = accumulate ? 1.0f : 0.0f;
  const rocblas_status st = rocblas_gemm_strided_batched_ex_64(
      h->blas, rocblas_operation_transpose, rocblas_operation_none, ns, nt, k, &alpha, S, rocblas_datatype_bf16_r, lds,
      k, T, rocblas_datatype_bf16_r, ldt, k, &beta, C, rocblas_datatype_f32_r, ldc, cstride, C, rocblas_datatype_f32_r,
      ldc, cstride, batch, rocblas_datatype_f32_r, rocblas_gemm_algo_standard, 0, 0);
  if (st != rocblas_status_success)
    return fail(PNFAM_GPU_EDEVICE, "rocblas_gemm_strided_batched_ex failed: " + std::to_string(st));
  return 0;
}

// The split products of one contraction: hi*hi over all ns columns of the
// small operand, hi*lo + lo*hi over its first ns3 columns (the points that
// take three products come first in the active list).
int blas_split(pnfam_gpu_ctx *h, int64_t ns, int64_t nt, int64_t k, const __bf16 *Sh, const __bf16 *Sl, int64_t lds,
               const __bf16 *Th, const __bf16 *Tl, int64_t ldt, float *C, int64_t ldc, int64_t ns3) {
  if (int e = blas_nt(h, ns, nt, k, Sh, lds, Th, ldt, C, ldc, false)) return e;
  if (ns3 == 0) return 0;
  if (int e = blas_nt(h, ns3, nt, k, Sh, lds, Tl, ldt, C, ldc, true)) return e;
  return blas_nt(h, ns3, nt, k, Sl, lds, Th, ldt, C, ldc, true);
}

// Split-K form of blas_split for contractions with few output tiles: K chunks
// of kchunk go to separate FP32 planes of P in one batched call each, the
// remainder to the next plane, and k_sum_planes adds the first ns rows of every
// plane column into C.  Used for the pairing densities (one grid-point row per
// table row) and, with two or three chunks, for the mean-field densities when
// the column count leaves rocBLAS too few output tiles for the device.

__global__ void k_sum_planes(const float *__restrict__ P, int nplanes, int64_t ns, int64_t nt, int64_t ldc,
                             float *__restrict__ C) {
  const size_t plane = (size_t)nt * ldc, n = (size_t)nt * ns;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const size_t i = (e / ns) * ldc + e % ns;
    float v = 0.0f;
    for (int j = 0; j < nplanes; ++j) v += P[(size_t)j * plane + i];
    C[i] = v;
  }
}

int blas_split_k(pnfam_gpu_ctx *h, int64_t ns, int64_t nt, int64_t k, const __bf16 *Sh, const __bf16 *Sl, int64_t lds,
                 const __bf16 *Th, const __bf16 *Tl, int64_t ldt, float *C, int64_t ldc, int64_t ns3, float *P,
                 size_t pcap, int64_t kchunk) {
  note(h, "rocblas_split_k");
  const int64_t nfull = k / kchunk, rem = k - nfull * kchunk;
  const int64_t plane = nt * ldc;
  if ((size_t)(nfull + 1) * (size_t)plane > pcap) return fail(PNFAM_GPU_EINVAL, "split-K planes exceed their buffer");
  const __bf16 *Ss[3] = {Sh, Sh, Sl}, *Ts[3] = {Th, Tl, Th};
  for (int p = 0; p < 3; ++p) {
    const int64_t nsp = p == 0 ? ns : ns3;
    if (nsp == 0) break;
    if (nfull > 0)
      if (int e = blas_nt_chunks(h, nsp, nt, kchunk, nfull, Ss[p], lds, Ts[p], ldt, P, ldc, plane, p > 0)) return e;
    if (rem > 0)
      if (int e = blas_nt(h, nsp, nt, rem, Ss[p] + nfull * kchunk, lds, Ts[p] + nfull * kchunk, ldt,
                          P + nfull * plane, ldc, p > 0))
        return e;
  }
  const int np = (int)(nfull + (rem > 0 ? 1 : 0));
  const size_t n = (size_t)nt * ns;
  hipLaunchKernelGGL(k_sum_planes, dim3((unsigned)std::min<size_t>(2048, (n + 255) / 256)), dim3(256), 0, h->stream, P,
                     np, ns, nt, ldc, C);
  HIP_TRY(hipGetLastError());
  return 0;
}

// K chunk for a mean-field density contraction of ns columns: rocBLAS tiles
// these shapes 256 columns wide, so below about 384 columns its grid leaves most
// of the device idle; two or three K chunks in one batched call fill it (split
// count measured on MI355X for 14400 table rows and K = 26112: 512 columns
// 0.55 -> 0.37 ms with two, 256 columns 0.49 -> 0.21 ms with three).  The chunk
// is rounded down to 64 so that the split count of chunks runs in one batched
// call; the remainder (under 64 per chunk) takes one more small call.  0: no split.
int64_t dens_kchunk(int64_t ns, int64_t k) {
  const int nsplit = ns >= 384 ? 2 : (ns >= 96 ? 3 : 1);
  if (nsplit == 1 || k < 4096) return 0;
  return k / nsplit / 64 * 64;
}

void mix_gemm(pnfam_gpu_ctx *h, GemmArgs G, const pnfam_gpu_ctx::MixSet &S, int tmax) {
  const int ntt = (tmax + GT_ROWS - 1) / GT_ROWS;
  const int ntt8 = (ntt + 7) / 8 * 8;
  G.nst = (G.nS + GS_ROWS - 1) / GS_ROWS;
  hipLaunchKernelGGL(k_mix_gemm, dim3((unsigned)(ntt8 * G.nst), 4), dim3(512), 0, h->stream, G);
  (void)S;
}

// calc_hamiltonian for the active columns on split-BF16 MFMA: rsp -> hsp.
// n3: the first n3 active points take three BF16 products, the rest one.
int stage_hamiltonian_mixed(pnfam_gpu_ctx *h, int na, const int *act, int n3) {
  if (int e = mix_workspace(h, h->cap)) return e;
  note(h, h->own_gemm ? "k_mix_gemm" : "rocblas_pair_tables");
  const size_t RP = h->RP;
  const int cap = h->mix_cap;
  // 1. rho and kappa -> BF16 hi/lo columns
  { Prof pr(h, K_MIX_CVT, na);
    for (int si = 0; si < 3; ++si) {
      auto &S = h->mix[si];
      CvtRhoArgs C{};
      C.rsp = h->d_rsp.as<double>(); C.elem = S.d_elem.as<int>(); C.act = act; C.nxy = h->nxy; C.Kp = S.Kp;
      C.nsec = si == 0 ? 2 : 1;
      C.q0 = si == 0 ? 0 : (si == 1 ? 1 : 2);   // quadrants: rho_pn, kappa+, kappa-, rho_np
      C.q1 = 3;
      C.hi = S.Bh.as<__bf16>(); C.lo = S.Bl.as<__bf16>();
      hipLaunchKernelGGL(k_mix_rho, dim3((unsigned)std::min(1024, (S.Kp + 255) / 256), na), dim3(256), 0, h->stream, C);
    } }
  // 2. density contractions
  if (!h->own_gemm) {
    Prof pr(h, K_MIX_GEMM_D, na + 2 * n3);
    for (int si = 0; si < 3; ++si) {
      auto &S = h->mix[si];
      const long ncol = (si == 0 ? 4 : 2) * (long)cap;
      const int64_t nS = (si == 0 ? 4 : 2) * (int64_t)na, nT = (int64_t)S.ntd * RP;
      for (int c = 0; c < 4; ++c) {
        const int64_t k0 = S.kbeg[c], kl = S.kbeg[c + 1] - S.kbeg[c];
        float *O = S.O.as<float>() + (size_t)c * nT * ncol;
        if (kl == 0) {
          hipLaunchKernelGGL(k_fill_f32, dim3(1024), dim3(256), 0, h->stream, O, (size_t)nT * ncol);
          continue;
        }
        const int64_t nS3 = (si == 0 ? 4 : 2) * (int64_t)n3;
        if (si != 0) {   // pairing sets: one table row per grid point, too few output tiles
          if (int e = blas_split_k(h, nS, nT, kl, S.Bh.as<__bf16>() + k0, S.Bl.as<__bf16>() + k0, S.Kp,
                                   S.TDh.as<__bf16>() + k0, S.TDl.as<__bf16>() + k0, S.Kp, O, ncol, nS3,
                                   h->d_Psplit.as<float>(), h->d_Psplit.bytes / 4, MIX_KCHUNK))
            return e;
        } else if (const int64_t kc = dens_kchunk(nS, kl)) {
          if (int e = blas_split_k(h, nS, nT, kl, S.Bh.as<__bf16>() + k0, S.Bl.as<__bf16>() + k0, S.Kp,
                                   S.TDh.as<__bf16>() + k0, S.TDl.as<__bf16>() + k0, S.Kp, O, ncol, nS3,
                                   h->d_Psplit.as<float>(), h->d_Psplit.bytes / 4, kc))
            return e;
        } else if (int e = blas_split(h, nS, nT, kl, S.Bh.as<__bf16>() + k0, S.Bl.as<__bf16>() + k0, S.Kp,
                                      S.TDh.as<__bf16>() + k0, S.TDl.as<__bf16>() + k0, S.Kp, O, ncol, nS3))
          return e;
      }
    }
  } else {
    Prof pr(h, K_MIX_GEMM_D, na + 2 * n3);
    for (int si = 0; si < 3; ++si) {
      auto &S = h->mix[si];
      const long ncol = (si == 0 ? 4 : 2) * (long)cap;
      GemmArgs G{};
      G.Th = S.TDh.as<__bf16>(); G.Tl = S.TDl.as<__bf16>(); G.ldT = S.Kp; G.segT = 0;
      G.Sh = S.Bh.as<__bf16>(); G.Sl = S.Bl.as<__bf16>(); G.ldS = S.Kp; G.segS = 0;
      G.nseg = 1; G.nS = (si == 0 ? 4 : 2) * na; G.s_cls = 0;
      G.o_cls = (long)S.ntd * RP * ncol; G.jobs = S.d_jobs_dens.as<GemmJob>();
      G.mode = 0; G.O = S.O.as<float>(); G.ldO = ncol;
      mix_gemm(h, G, S, S.ntd * (int)RP);
    } }
  // 3. densities
  { Prof pr(h, K_MIX_DENS, na);
    CombArgs A{};
    A.Of = h->mix[0].O.as<float>(); A.Ok0 = h->mix[1].O.as<float>(); A.Ok1 = h->mix[2].O.as<float>();
    A.ldf = 4L * cap; A.ldk = 2L * cap; A.RP = (int)RP; A.nghl = h->nghl; A.na = na;
    A.wdcori = h->d_wdcori.as<double>(); A.dens = h->d_dens.as<double>(); A.act = act;
    hipLaunchKernelGGL(k_mix_dens, dim3((h->nghl + 15) / 16, (2 * na + 15) / 16), dim3(256), 0, h->stream, A); }
  // 4. fields (FP64, closed forms)
  if (int e = stage_fields(h, na, act)) return e;
  // 5. fields -> BF16 hi/lo
  { Prof pr(h, K_MIX_CVT, na);
    for (int si = 0; si < 3; ++si) {
      auto &S = h->mix[si];
      CvtFldArgs C{};
      C.flds = h->d_flds.as<double>(); C.act = act; C.nghl = h->nghl; C.RP = (int)RP;
      C.ncap = (si == 0 ? 4 : 2) * cap; C.pair = si != 0; C.sec = si == 2 ? 1 : 0;
      C.hi = S.Fh.as<__bf16>(); C.lo = S.Fl.as<__bf16>();
      hipLaunchKernelGGL(k_mix_fields, dim3((unsigned)((RP + 127) / 128), na), dim3(128), 0, h->stream, C);
    } }
  // 6. projections: rocBLAS into O[k][n] and a scatter into the FP64 block
  // matrices, or the hand-written kernel writing them directly
  if (!h->own_gemm) {
    Prof pr(h, K_MIX_GEMM_P, na + 2 * n3);
    for (int si = 0; si < 3; ++si) {
      auto &S = h->mix[si];
      const long ncol = (si == 0 ? 4 : 2) * (long)cap;
      const int64_t nS = (si == 0 ? 4 : 2) * (int64_t)na, KK = (int64_t)S.ntp * RP;
      float *O = h->d_Oproj.as<float>();
      for (int c = 0; c < 4; ++c) {
        const int64_t k0 = S.kbeg[c], kl = S.kbeg[c + 1] - S.kbeg[c];
        if (kl == 0) continue;
        const size_t fo = (size_t)c * ncol * KK;
        // the mean-field set uses proj_ncomb(c) of the NPROJ_C table combinations
        const int64_t Kc = si == 0 ? (int64_t)proj_ncomb(c) * RP : KK;
        if (int e = blas_split(h, nS, kl, Kc, S.Fh.as<__bf16>() + fo, S.Fl.as<__bf16>() + fo, KK,
                               S.TPh.as<__bf16>() + (size_t)k0 * KK, S.TPl.as<__bf16>() + (size_t)k0 * KK, KK,
                               O + (size_t)k0 * ncol, ncol, (si == 0 ? 4 : 2) * (int64_t)n3))
          return e;
      }
      hipLaunchKernelGGL(k_mix_scatter, dim3((unsigned)((S.Kp + 63) / 64), (unsigned)((nS + 63) / 64)),
                         dim3(256), 0, h->stream, O, ncol, S.d_elem.as<int>(), S.Kp, (int)nS, si == 0 ? 2 : 1,
                         si == 0 ? 0 : (si == 1 ? 1 : 2), 3, act, h->d_hsp.as<double>(), h->nxy);
    }
  } else {
    Prof pr(h, K_MIX_GEMM_P, na + 2 * n3);
    for (int si = 0; si < 3; ++si) {
      auto &S = h->mix[si];
      const long ncol = (si == 0 ? 4 : 2) * (long)cap;
      GemmArgs G{};
      G.Th = S.TPh.as<__bf16>(); G.Tl = S.TPl.as<__bf16>(); G.ldT = (long)S.ntp * RP; G.segT = RP;
      G.Sh = S.Fh.as<__bf16>(); G.Sl = S.Fl.as<__bf16>(); G.ldS = (long)S.ntp * RP; G.segS = RP;
      G.nseg = S.ntp; G.nS = (si == 0 ? 4 : 2) * na; G.s_cls = ncol * (long)S.ntp * RP; G.o_cls = 0;
      G.jobs = S.d_jobs_proj.as<GemmJob>();
      G.mode = 1; G.hsp = h->d_hsp.as<double>(); G.elem = S.d_elem.as<int>(); G.act = act; G.nxy = h->nxy;
      G.nsec = si == 0 ? 2 : 1; G.q0 = si == 0 ? 0 : (si == 1 ? 1 : 2); G.q1 = 3;
      mix_gemm(h, G, S, S.maxcount);
    } }
  HIP_TRY(hipGetLastError());
  return 0;
}

// ---- factored split-BF16 grid stage (mixed path) -----------------------------
// psi tables, chunk map of every (block, spin), the density pair lists with
// their operand offsets and the conversion segments of the four density
// structures (rho_pn, kappa+, rho_np, kappa- as the FP64 density kernel reads them).
int fac_prepare(pnfam_gpu_ctx *h) {
  if (h->fac_ready) return 0;
  const int nb = (int)h->db.size();
  const int RP = h->RP;
  // spin order inside every block: states [0, nsu) up, [nsu, d) down
  for (int i = 0; i < nb; ++i)
    for (int j = 0; j < h->db[i]; ++j)
      if ((h->ns[h->isstart[i] + j] > 0) != (j < h->nsu[i]))
        return fail(PNFAM_GPU_EINVAL, "factored grid stage: block states are not ordered spin up, spin down");
  std::vector<FacBlock> blk(nb);
  std::vector<int2> chunks;
  for (int i = 0; i < nb; ++i) {
    const int n0 = h->nsu[i], n1 = h->db[i] - h->nsu[i];
    blk[i].nc0 = (n0 + FAC_CH - 1) / FAC_CH;
    blk[i].nc1 = (n1 + FAC_CH - 1) / FAC_CH;
    blk[i].cb0 = (int)chunks.size();
    for (int c = 0; c < blk[i].nc0; ++c) chunks.push_back(make_int2(h->isstart[i] + c * FAC_CH, std::min(FAC_CH, n0 - c * FAC_CH)));
    blk[i].cb1 = (int)chunks.size();
    for (int c = 0; c < blk[i].nc1; ++c)
      chunks.push_back(make_int2(h->isstart[i] + n0 + c * FAC_CH, std::min(FAC_CH, n1 - c * FAC_CH)));
  }
  const int nchunk = std::max<int>(1, (int)chunks.size());
  if (chunks.empty()) chunks.push_back(make_int2(0, 0));
  // pairs and segments: structure order rho0 (m11), kap0 (m12), rho1 (m22), kap1 (m21)
  const int quad[4] = {0, 1, 3, 2};
  std::vector<int4> pairs;
  std::vector<FacSeg> segs;
  long L = 0;
  for (int st = 0; st < 4; ++st) {
    h->fac_first[st] = (int)pairs.size();
    for (const auto &pq : pair_list(h->rspmap[quad[st]])) {
      const int ix = pq.x, iy = pq.y, dx = h->db[ix], dy = h->db[iy];
      const int nchT = blk[ix].nc0 + blk[ix].nc1;
      pairs.push_back(make_int4(ix, iy, (int)L, 0));
      for (int b = 0; b < dy; ++b)
        for (int sa = 0; sa < 2; ++sa) {
          const int n = sa ? dx - h->nsu[ix] : h->nsu[ix];
          if (n == 0) continue;
          FacSeg g;
          g.src = pq.z + b * dx + (sa ? h->nsu[ix] : 0);
          g.n = n;
          g.dst = (int)(L + ((long)b * nchT + (sa ? blk[ix].nc0 : 0)) * FAC_CH);
          g.q = quad[st];
          segs.push_back(g);
        }
      L += (long)dy * nchT * FAC_CH;
    }
    h->fac_n[st] = (int)pairs.size() - h->fac_first[st];
  }
  if (L >= (1L << 31)) return fail(PNFAM_GPU_EINVAL, "factored grid stage: operand too large");
  h->fac_L = std::max<long>(L, FAC_CH);
  h->fac_nseg = (int)segs.size();
  int e;
  if ((e = upload(h->d_fac_blk, blk.data(), std::max<size_t>(1, blk.size()) * sizeof(FacBlock), h->stream)) ||
      (e = upload(h->d_fac_pairs, pairs.data(), std::max<size_t>(1, pairs.size()) * sizeof(int4), h->stream)) ||
      (e = upload(h->d_fac_segs, segs.data(), std::max<size_t>(1, segs.size()) * sizeof(FacSeg), h->stream)))
    return e;
  DevPtr d_chunks;
  if ((e = upload(d_chunks, chunks.data(), chunks.size() * sizeof(int2), h->stream))) return e;
  const int nst = (int)std::accumulate(h->db.begin(), h->db.end(), 0);
  h->fac_pz = (long)nst * RP;
  h->fac_dbx = (long)nchunk * RP * FAC_CH;
  if ((e = h->PAh.alloc(5 * h->fac_pz * 2)) || (e = h->PAl.alloc(5 * h->fac_pz * 2)) ||
      (e = h->PS32.alloc(5 * h->fac_pz * 4)) || (e = h->DBh.alloc(4 * h->fac_dbx * 2)) ||
      (e = h->DBl.alloc(4 * h->fac_dbx * 2)))
    return e;
  hipLaunchKernelGGL(k_fac_ptab, dim3(2048, 5), dim3(256), 0, h->stream, h->d_wf.as<double>(), h->d_wfdr.as<double>(),
                     h->d_wfdp.as<double>(), h->d_wfdz.as<double>(), h->d_wfd2.as<double>(), nst, h->nghl, RP,
                     h->PAh.as<__bf16>(), h->PAl.as<__bf16>(), h->PS32.as<float>());
  hipLaunchKernelGGL(k_fac_dtab, dim3(2048, 4), dim3(256), 0, h->stream, h->d_wf.as<double>(), h->d_wfdr.as<double>(),
                     h->d_wfdp.as<double>(), h->d_wfdz.as<double>(), d_chunks.as<int2>(), nchunk, h->nghl, RP,
                     h->DBh.as<__bf16>(), h->DBl.as<__bf16>());
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(h->stream));   // d_chunks is freed on return
  // MFMA-issued FLOP per frequency and BF16 product: density tiles of 16 grid
  // points x 16 columns per chunk (4 tables mean field, 1 pairing, re + im);
  // projection tiles of NRT x 16 rows x 16 columns per 32 grid points
  double fd = 0;
  for (int st = 0; st < 4; ++st) {
    const int nx = (st == 0 || st == 2) ? 4 : 1;
    for (int p = h->fac_first[st]; p < h->fac_first[st] + h->fac_n[st]; ++p) {
      const int ix = pairs[p].x, iy = pairs[p].y;
      const int ny = h->nsu[iy], dy = h->db[iy];
      const int bt = (ny + 15) / 16 + (dy - ny + 15) / 16;
      fd += (double)bt * (blk[ix].nc0 + blk[ix].nc1) * nx * 2 * (2.0 * 16 * 16 * FAC_CH);
    }
  }
  h->flops_unit[K_FAC_DENS] = fd * (RP / 16);
  double fpj = 0;
  for (int k = 0; k < 16; ++k) {
    const int nrt = k & 7, kind = k >> 3;
    fpj += (double)h->pj_count[k] * nrt * (kind ? 1 : 5) * 2 * (2.0 * 16 * 16 * FAC_RT);
  }
  h->flops_unit[K_FAC_PROJ] = fpj * (RP / FAC_RT);
  h->fac_cap = 0;
  h->fac_ready = true;
  return 0;
}

constexpr int FAC_DPART = 32;   // partial density planes (parts x slots) of the split density launch

int fac_workspace(pnfam_gpu_ctx *h, int cap) {
  if (cap <= h->fac_cap) return 0;
  h->fac_cap = 0;   // set again only once every buffer below is in place
  const size_t n = (size_t)cap * 2 * h->fac_L * 2;
  if (int e = h->FRh.alloc(n)) return e;
  if (int e = h->FRl.alloc(n)) return e;
  if (int e = h->FFm.alloc((size_t)cap * 4 * h->RP * FAC_FM * 4)) return e;
  if (int e = h->FFp.alloc((size_t)cap * 4 * h->RP * FAC_FP * 4)) return e;
  h->fac_cap = cap;
  return 0;
}

// calc_hamiltonian for the active columns with the factored split-BF16 kernels.
int stage_hamiltonian_fac(pnfam_gpu_ctx *h, int na, const int *act, int n3) {
  if (int e = fac_workspace(h, h->cap)) return e;
  { Prof pr(h, K_FAC_CVT, na);
    if (h->fac_nseg)
      hipLaunchKernelGGL(k_fac_rho, dim3((h->fac_nseg + 3) / 4, na), dim3(256), 0, h->stream, h->d_rsp.as<double>(),
                         h->d_fac_segs.as<FacSeg>(), h->fac_nseg, h->nxy, h->fac_L, act, h->FRh.as<__bf16>(),
                         h->FRl.as<__bf16>()); }
  FacDensArgs D{};
  D.FRh = h->FRh.as<__bf16>(); D.FRl = h->FRl.as<__bf16>(); D.L = h->fac_L;
  D.DBh = h->DBh.as<__bf16>(); D.DBl = h->DBl.as<__bf16>(); D.dbx = h->fac_dbx;
  D.blk = h->d_fac_blk.as<FacBlock>(); D.pairs = h->d_fac_pairs.as<int4>();
  D.rho_first[0] = h->fac_first[0]; D.rho_n[0] = h->fac_n[0]; D.kap_first[0] = h->fac_first[1]; D.kap_n[0] = h->fac_n[1];
  D.rho_first[1] = h->fac_first[2]; D.rho_n[1] = h->fac_n[2]; D.kap_first[1] = h->fac_first[3]; D.kap_n[1] = h->fac_n[3];
  D.PS = h->PS32.as<float>(); D.pz = h->fac_pz; D.wdcori = h->d_wdcori.as<double>();
  D.isstart = h->d_isstart.as<int>(); D.db = h->d_db.as<int>(); D.nsu = h->d_nsu.as<int>();
  D.nghl = h->nghl; D.RP = h->RP; D.dens = h->d_dens.as<double>(); D.act = act; D.n3 = n3;
  // few points: the pairs of a grid tile spread over psplit workgroups (psplit * na <= FAC_DPART)
  // (at most four parts: 2, 4, 8 and 16 measured 280, 254, 264 and 264 us for one point)
  D.psplit = std::max(1, std::min(4, FAC_DPART / na));
  if (D.psplit > 1) {
    if (int e = h->d_fac_dpart.alloc((size_t)FAC_DPART * 2 * 2 * NDENS * h->nghl * 4)) return e;
    D.part = h->d_fac_dpart.as<float>();
  }
  { Prof pr(h, K_FAC_DENS, na + 2 * n3);
    note(h, "k_fac_density", D.psplit);
    hipLaunchKernelGGL(k_fac_density, dim3(h->RP / 16, na, 2 * D.psplit), dim3(64 * FAC_NW), 0, h->stream, D);
    if (D.psplit > 1)
      hipLaunchKernelGGL(k_fac_dsum, dim3((2 * NDENS * h->nghl + 255) / 256, na, 2), dim3(256), 0, h->stream, D.part,
                         D.psplit, na, h->nghl, h->d_wdcori.as<double>(), act, h->d_dens.as<double>()); }
  if (int e = stage_fields(h, na, act)) return e;
  if (!(h->zero_skip && h->proj_cover)) {
    Prof pr(h, K_ZERO, na);
    hipLaunchKernelGGL(k_zero_slots, dim3(64, na), dim3(256), 0, h->stream, h->d_hsp.as<double>(), act, 8, 0, 8,
                       h->nxy, h->skip_slot); }
  FacProjArgs P{};
  P.PAh = h->PAh.as<__bf16>(); P.PAl = h->PAl.as<__bf16>(); P.PS = h->PS32.as<float>(); P.pz = h->fac_pz;
  P.isstart = h->d_isstart.as<int>(); P.db = h->d_db.as<int>(); P.nsu = h->d_nsu.as<int>();
  P.FFm = h->FFm.as<float>(); P.FFp = h->FFp.as<float>();
  P.hsp = h->d_hsp.as<double>(); P.nxy = h->nxy; P.nghl = h->nghl; P.RP = h->RP;
  P.act = act; P.n3 = n3;
  { Prof pr(h, K_FAC_CVT, 0);   // its units (points) are counted once per pass, with k_fac_rho
    const int nconv = h->RP * (FAC_FM + FAC_FP);
    hipLaunchKernelGGL(k_fac_fconv, dim3((nconv + 255) / 256, na, 4), dim3(256), 0, h->stream, h->d_flds.as<double>(),
                       h->nghl, h->RP, act, h->FFm.as<float>(), h->FFp.as<float>()); }
  { Prof pr(h, K_FAC_PROJ, na + 2 * n3);
    const Tile2 *tl = h->d_tiles2.as<Tile2>();
    // few points: one launch per kind over all row-tile classes (widest template)
    const bool merge = na <= TP_MERGE_N;
    int mk[2] = {0, 0}, mfirst[2] = {-1, -1}, mcount[2] = {0, 0};
    for (int k = 0; k < 16; ++k) {
      if (!h->pj_count[k]) continue;
      const int kind = k >> 3;
      mk[kind] = k;
      if (mfirst[kind] < 0) mfirst[kind] = h->pj_first[k];
      mcount[kind] += h->pj_count[k];
    }
    for (int k = 0; k < 16; ++k) {
      const int kind = k >> 3;
      if (merge && k != mk[kind]) continue;
      const int n = merge ? mcount[kind] : h->pj_count[k];
      if (!n) continue;
      // frequencies per wave (option fac_freqs; 0: two from 16 points, below
      // which the halved grid costs more than the shared loads save; one for
      // four row tiles, whose accumulators leave no registers for a second)
      const int want = h->fac_nf ? h->fac_nf : (na >= 16 ? 2 : 1);
      const int nf = (want == 2 && (k & 7) <= 3 && na > 1) ? 2 : 1;
      const int ngrp = (na + nf - 1) / nf;
      // XCD chunks of eight consecutive tiles for every slot group
      P.na = na; P.ntiles = n; P.chunk = std::min(1024, 8 * ngrp);
      const long units = (long)n * ngrp, per = 8L * P.chunk;
      const dim3 grid((unsigned)((units + per - 1) / per * per));
      const Tile2 *tk = tl + (merge ? mfirst[kind] : h->pj_first[k]);
      note(h, nf == 2 ? "k_fac_project_f2" : "k_fac_project", k & 7, k >> 3);
#define FP_LAUNCH(NRT, KIND)                                                                                        \
  do {                                                                                                            \
    if (nf == 2) hipLaunchKernelGGL((k_fac_project<NRT, KIND, (NRT <= 3 ? 2 : 1)>), grid, dim3(64 * FAC_NW), 0,   \
                                    h->stream, P, tk);                                                            \
    else hipLaunchKernelGGL((k_fac_project<NRT, KIND, 1>), grid, dim3(64 * FAC_NW), 0, h->stream, P, tk);         \
  } while (0)
      switch (k) {
        case 1: FP_LAUNCH(1, 0); break;
        case 2: FP_LAUNCH(2, 0); break;
        case 3: FP_LAUNCH(3, 0); break;
        case 4: FP_LAUNCH(4, 0); break;
        case 9: FP_LAUNCH(1, 1); break;
        case 10: FP_LAUNCH(2, 1); break;
        case 11: FP_LAUNCH(3, 1); break;
        case 12: FP_LAUNCH(4, 1); break;
        default: return fail(PNFAM_GPU_EINVAL, "projection tile class out of range");
      }
#undef FP_LAUNCH
    } }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Grid stage of the mixed path for na active points, the first n3 of which
// take three BF16 products: the pair-table GEMMs or the factored kernels
// (PNFAM_GPU_MIX_GRID = tables | factored | auto).  A pass over the tables
// costs at least one stream of them whatever the column count, the factored
// kernels cost per point; auto gives the factored kernels any group of at most
// PNFAM_GPU_MIX_AUTO_N points: the whole pass, or the few three-product points
// while the one-product majority streams the tables once.
int stage_hamiltonian_lowp(pnfam_gpu_ctx *h, int na, const int *act, int n3) {
  if (h->mix_grid == 2) return stage_hamiltonian_fac(h, na, act, n3);
  if (h->mix_grid == 1) return stage_hamiltonian_mixed(h, na, act, n3);
  if (na <= h->mix_auto_n) return stage_hamiltonian_fac(h, na, act, n3);
  if (n3 > 0 && n3 <= h->mix_auto_n) {
    if (int e = stage_hamiltonian_fac(h, n3, act, n3)) return e;
    return stage_hamiltonian_mixed(h, na - n3, act + n3, 0);
  }
  return stage_hamiltonian_mixed(h, na, act, n3);
}

int stage_sp2qp(pnfam_gpu_ctx *h, int na, const int *act, bool lowp = false, int n3 = 0) {
  const long nxy = h->nxy;
  if (!(h->zero_skip && h->s2q_cover && !h->basic_kernels)) {
    Prof pr(h, K_ZERO, na);
    hipLaunchKernelGGL(k_zero_slots, dim3(64, na), dim3(256), 0, h->stream, h->d_hqp.as<double>(), act, 4, 0, 4, nxy,
                       h->skip_slot); }
  Prof pr(h, K_TRIPROD_S2Q, na);
  if (lowp) return launch_triprod_bf16(h, 1, h->d_hsp.as<double>(), 8 * nxy, h->d_hqp.as<double>(), 4 * nxy, na, act, n3);
  if (!h->basic_kernels && h->tp64_ok)
    return launch_triprod(h, 1, h->d_hsp.as<double>(), 8 * nxy, h->d_hqp.as<double>(), 4 * nxy, na, act);
  for (int ri = 0; ri < 2; ++ri) {
    if (!h->ngroups_s2q[ri]) continue;
    hipLaunchKernelGGL(k_triprod, dim3(h->ngroups_s2q[ri], na), dim3(256), h->lds_s2q, h->stream,
                       h->d_groups_s2q[ri].as<Group>(), h->d_terms_s2q[ri].as<Term>(), h->d_U[0].as<double>(),
                       h->d_U[1].as<double>(), h->d_U[2].as<double>(), h->d_U[3].as<double>(), h->d_hsp.as<double>(),
                       8 * nxy, 8, h->d_hqp.as<double>(), 4 * nxy, 4, act, nxy);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Projection tiles of the MFMA projection kernels (FP64 and factored BF16):
// per output block and spin of its rows, row ranges of at most proj_maxrt
// 16-row tiles by 16 columns, ordered by (kind, row tiles) for the templated
// kernels.  The row tiles per wave change the work per wave, not any output
// element's sum.
int build_tiles2(pnfam_gpu_ctx *h) {
  const std::vector<int> &db = h->db;
  const int slot_sec[4] = {0, 0, 1, 1};
  const int maxrt = h->proj_maxrt;
  std::vector<Tile2> tiles2;
  for (int q = 0; q < 4; ++q) {
    for (auto &p : pair_list(h->hspmap[q])) {
      const int dx = db[p.x], dy = db[p.y], nsu = h->nsu[p.x];
      for (int sa = 0; sa < 2; ++sa) {
        const int lo = sa ? nsu : 0, hi = sa ? dx : nsu;
        for (int a0 = lo; a0 < hi; a0 += 16 * maxrt)
          for (int b0 = 0; b0 < dy; b0 += 16) {
            Tile2 t{};
            t.ix = p.x; t.iy = p.y; t.off = p.z; t.sec = slot_sec[q];
            t.a_lo = a0; t.a_hi = std::min(hi, a0 + 16 * maxrt); t.sa = sa; t.b0 = b0;
            t.out_slot = q; t.kind = (q == 1 || q == 2) ? 1 : 0;
            tiles2.push_back(t);
          }
      }
    }
  }
  // the tiles' kernels store every element of a tile: complete coverage of the
  // eight dH_sp slots lets the projection skip zeroing them first
  {
    const size_t nxy = (size_t)h->fmap.nelem(db);   // h->nxy is set after the first call
    std::vector<char> cov(8 * nxy, 0);
    bool ok = true;
    for (const auto &t : tiles2) {
      const int dx = db[t.ix], dy = db[t.iy];
      for (int s = 0; s < 2; ++s)
        for (int b = t.b0; b < std::min(dy, t.b0 + 16); ++b) {
          const size_t o = (size_t)(2 * t.out_slot + s) * nxy + t.off + (size_t)b * dx;
          if (o + t.a_hi > cov.size()) { ok = false; continue; }
          std::fill(cov.begin() + o + t.a_lo, cov.begin() + o + t.a_hi, 1);
        }
    }
    h->proj_cover = ok && std::find(cov.begin(), cov.end(), 0) == cov.end();
  }
  auto tkey = [](const Tile2 &t) { return t.kind * 8 + (t.a_hi - t.a_lo + 15) / 16; };
  std::stable_sort(tiles2.begin(), tiles2.end(), [&](const Tile2 &a, const Tile2 &b) { return tkey(a) < tkey(b); });
  for (int k = 0; k < 16; ++k) { h->pj_first[k] = 0; h->pj_count[k] = 0; }
  for (size_t i = 0; i < tiles2.size(); ++i) {
    const int k = tkey(tiles2[i]);
    if (h->pj_count[k] == 0) h->pj_first[k] = (int)i;
    h->pj_count[k]++;
  }
  h->ntiles2 = (int)tiles2.size();
  if (int e = upload(h->d_tiles2, tiles2.data(), std::max<size_t>(1, tiles2.size()) * sizeof(Tile2), h->stream))
    return e;
  HIP_TRY(hipStreamSynchronize(h->stream));   // the host list is released on return
  return 0;
}

// W^T g W for n single-particle operators with f's block structure (host
// g_elem [n][nxy]): the quadrants 20 and 02 go to out20 / out02 [n][nxy]
// (device).  The same plan as Fqp (pnfam_solver.f90:364-372).
int to_qp(pnfam_gpu_ctx *h, const double *g_elem, int n, double *out20, double *out02) {
  const long nxy = h->nxy;
  DevPtr dt, dg, df, dout, dact;
  std::vector<int> act(n);
  std::iota(act.begin(), act.end(), 0);
  const auto &terms = h->fq_terms;
  const auto &groups = h->fq_groups;
  int e;
  if ((e = upload(dt, terms.data(), std::max<size_t>(1, terms.size()) * sizeof(Term), h->stream)) ||
      (e = upload(dg, groups.data(), std::max<size_t>(1, groups.size()) * sizeof(Group), h->stream)) ||
      (e = upload(df, g_elem, (size_t)n * nxy * 8, h->stream)) || (e = dout.alloc((size_t)n * 2 * nxy * 8)) ||
      (e = upload(dact, act.data(), (size_t)n * 4, h->stream)))
    return e;
  hipLaunchKernelGGL(k_fill, grid1((size_t)n * 2 * nxy, 256), dim3(256), 0, h->stream, dout.as<double>(),
                     (size_t)n * 2 * nxy, 0.0);
  if (!groups.empty())
    hipLaunchKernelGGL(k_triprod, dim3((unsigned)groups.size(), n), dim3(256), h->fq_lds, h->stream, dg.as<Group>(),
                       dt.as<Term>(), h->d_U[0].as<double>(), h->d_U[1].as<double>(), h->d_U[2].as<double>(),
                       h->d_U[3].as<double>(), df.as<double>(), nxy, 1, dout.as<double>(), 2 * nxy, 2, dact.as<int>(),
                       nxy);
  HIP_TRY(hipGetLastError());
  for (int k = 0; k < n; ++k) {
    HIP_TRY(hipMemcpyAsync(out20 + (size_t)k * nxy, dout.as<double>() + (size_t)k * 2 * nxy, nxy * 8,
                           hipMemcpyDeviceToDevice, h->stream));
    HIP_TRY(hipMemcpyAsync(out02 + (size_t)k * nxy, dout.as<double>() + (size_t)k * 2 * nxy + nxy, nxy * 8,
                           hipMemcpyDeviceToDevice, h->stream));
  }
  HIP_TRY(hipStreamSynchronize(h->stream));   // the temporaries are released on return
  return 0;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

const char *pnfam_gpu_last_error(void) { return g_err.c_str(); }

const char *pnfam_gpu_version(void) { return "pnfam_gpu 0.1 gfx950 fp64"; }

int pnfam_gpu_create(const pnfam_gpu_basis *b, pnfam_gpu_ctx **out) {
  if (!b || !out) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (b->nb <= 0 || b->nb % 2 || b->dqp <= 0 || b->nghl <= 0)
    return fail(PNFAM_GPU_EINVAL, "nb must be positive and even, dqp and nghl positive");
  std::unique_ptr<pnfam_gpu_ctx> h(new pnfam_gpu_ctx);
  h->nb = b->nb; h->dqp = b->dqp; h->nghl = b->nghl;
  h->db.assign(b->db, b->db + b->nb);
  h->nsu.assign(b->num_spin_up, b->num_spin_up + b->nb);
  h->ns.assign(b->ns, b->ns + b->dqp);
  h->isstart.resize(b->nb);
  int s = 0;
  for (int i = 0; i < b->nb; ++i) {
    if (h->db[i] <= 0 || h->nsu[i] < 0 || h->nsu[i] > h->db[i]) return fail(PNFAM_GPU_EINVAL, "bad block size");
    h->isstart[i] = s;
    s += h->db[i];
  }
  if (s != b->dqp) return fail(PNFAM_GPU_EINVAL, "sum(db) != dqp");
  h->sorted_spins = spin_sorted(h.get());
  for (int i = 0; i < b->nb / 2; ++i)
    if (h->db[i] != h->db[i + b->nb / 2]) return fail(PNFAM_GPU_EINVAL, "time-reversed blocks must match");
  for (int i = 0; i < b->dqp; ++i)
    if (h->ns[i] != 1 && h->ns[i] != -1) return fail(PNFAM_GPU_EINVAL, "ns must be +1 or -1");
  for (int i = 0; i < b->nb; ++i)   // spin-up states first in each block
    for (int k = 0; k < h->db[i]; ++k)
      if ((k < h->nsu[i]) != (h->ns[h->isstart[i] + k] > 0))
        return fail(PNFAM_GPU_EINVAL, "states must be spin-sorted within blocks");
  h->cscal.assign(b->cscal, b->cscal + 12);
  if (const char *ev = std::getenv("PNFAM_GPU_BASIC")) h->basic_kernels = ev[0] == '1';
  if (const char *ev = std::getenv("PNFAM_GPU_MIX_TAU")) h->mix_tau = std::atof(ev);
  if (const char *ev = std::getenv("PNFAM_GPU_MIX_HIST")) h->mix_hist64 = std::strcmp(ev, "fp64") == 0;
  if (const char *ev = std::getenv("PNFAM_GPU_MIX_DROP")) h->mix_drop = ev[0] != '0';
  if (const char *ev = std::getenv("PNFAM_GPU_MIX_TRIPROD")) {
    if (std::strcmp(ev, "fp64") == 0) h->tp_bf16 = false;
    else if (std::strcmp(ev, "bf16") != 0) return fail(PNFAM_GPU_EINVAL, "PNFAM_GPU_MIX_TRIPROD must be bf16 or fp64");
  }
  tp_layout(h.get());
  HIP_TRY(hipGetDevice(&h->device));
  HIP_TRY(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  const size_t tab = (size_t)b->nghl * b->dqp * 8;
  size_t dmat = 0;
  for (int i = 0; i < b->nb; ++i) dmat += (size_t)h->db[i] * h->db[i];
  int e;
  if ((e = upload(h->d_wf, b->wf, tab, h->stream)) || (e = upload(h->d_wfdr, b->wfdr, tab, h->stream)) ||
      (e = upload(h->d_wfdz, b->wfdz, tab, h->stream)) || (e = upload(h->d_wfdp, b->wfdp, tab, h->stream)) ||
      (e = upload(h->d_wfd2, b->wfd2_all, tab, h->stream)) ||
      (e = upload(h->d_wdcori, b->wdcori, (size_t)b->nghl * 8, h->stream)) ||
      (e = upload(h->d_Ep, b->Ep, (size_t)b->dqp * 8, h->stream)) ||
      (e = upload(h->d_En, b->En, (size_t)b->dqp * 8, h->stream)) ||
      (e = upload(h->d_U[MAT_UP], b->Up, dmat * 8, h->stream)) ||
      (e = upload(h->d_U[MAT_VP], b->Vp, dmat * 8, h->stream)) ||
      (e = upload(h->d_U[MAT_UN], b->Un, dmat * 8, h->stream)) ||
      (e = upload(h->d_U[MAT_VN], b->Vn, dmat * 8, h->stream)) ||
      (e = upload(h->d_crho, b->crho, (size_t)b->nghl * 8, h->stream)) ||
      (e = upload(h->d_cs, b->cs, (size_t)b->nghl * 8, h->stream)) ||
      (e = upload(h->d_cpair, b->cpair, (size_t)b->nghl * 8, h->stream)) ||
      (e = upload(h->d_cspair, b->cspair, (size_t)b->nghl * 8, h->stream)) ||
      (e = upload(h->d_isstart, h->isstart.data(), (size_t)b->nb * 4, h->stream)) ||
      (e = upload(h->d_db, h->db.data(), (size_t)b->nb * 4, h->stream)) ||
      (e = upload(h->d_nsu, h->nsu.data(), (size_t)b->nb * 4, h->stream)) ||
      (e = upload(h->d_ns, h->ns.data(), (size_t)b->dqp * 4, h->stream)))
    return e;
  HIP_TRY(hipStreamSynchronize(h->stream));
  // padded copies of U and V for the FP64 triple products
  if ((e = h->tp_cm64.alloc(4 * (size_t)h->tp_mstride * 8)) || (e = h->tp_rm64.alloc(4 * (size_t)h->tp_mstride * 8)) ||
      (e = upload(h->d_tp_blocks, h->tp_blocks.data(), h->tp_blocks.size() * sizeof(int4), h->stream)))
    return e;
  for (int m = 0; m < 4; ++m)
    hipLaunchKernelGGL(k_tp_pack, dim3(16, (unsigned)h->tp_blocks.size()), dim3(256), 0, h->stream,
                       h->d_U[m].as<double>(), h->d_tp_blocks.as<int4>(),
                       h->tp_cm64.as<double>() + (size_t)m * h->tp_mstride,
                       h->tp_rm64.as<double>() + (size_t)m * h->tp_mstride);
  HIP_TRY(hipGetLastError());
  if ((e = sep_prepare(h.get(), b))) return e;
  *out = h.release();
  return 0;
}

void pnfam_gpu_destroy(pnfam_gpu_ctx *h) { delete h; }

int pnfam_gpu_set_operator(pnfam_gpu_ctx *h, int32_t beta_minus, const int32_t *f_ir2c, const double *f_elem,
                           int64_t *nxy_out) {
  if (!h || !f_ir2c || !f_elem) return fail(PNFAM_GPU_EINVAL, "null argument");
  const int nb = h->nb;
  std::vector<int> rows(f_ir2c, f_ir2c + nb);
  std::vector<int> seen(nb, 0);
  for (int i = 0; i < nb; ++i) {
    if (rows[i] < -1 || rows[i] >= nb) return fail(PNFAM_GPU_EINVAL, "f_ir2c out of range");
    if (rows[i] >= 0 && seen[rows[i]]++) return fail(PNFAM_GPU_EINVAL, "f has two blocks in one block column");
  }
  h->have_op = false;
  h->mix_ready = false;
  h->tp64_ok = true;
  h->bminus = beta_minus != 0;
  const std::vector<int> &db = h->db;
  std::vector<int> diag(nb), tr(nb);
  for (int i = 0; i < nb; ++i) { diag[i] = i; tr[i] = i < nb / 2 ? i + nb / 2 : i - nb / 2; }
  BlockMap U = BlockMap::from_rows(db, diag), V = BlockMap::from_rows(db, tr);
  // V storage follows U's offsets (pnfam_setup.f90:314-320)
  for (int i = 0; i < nb; ++i) V.ir2m[i] = U.ir2m[i];
  for (int i = 0; i < nb; ++i) V.ic2m[V.ir2c[i]] = V.ir2m[i];
  h->fmap = BlockMap::from_rows(db, rows);
  const long nxy = h->fmap.nelem(db);
  if (nxy <= 0) return fail(PNFAM_GPU_EINVAL, "operator has no blocks");
  const int L_U = h->bminus ? MAT_UP : MAT_UN, L_V = h->bminus ? MAT_VP : MAT_VN;
  const int R_U = h->bminus ? MAT_UN : MAT_UP, R_V = h->bminus ? MAT_VN : MAT_VP;
  SymBBM WL, WR;
  WL.m[0] = &U; WL.m[1] = &V; WL.m[2] = &V; WL.m[3] = &U;
  WL.id[0] = L_U; WL.id[1] = L_V; WL.id[2] = L_V; WL.id[3] = L_U;
  WR = WL;
  WR.id[0] = R_U; WR.id[1] = R_V; WR.id[2] = R_V; WR.id[3] = R_U;
  // Fqp = WL^T Fsp WR : quadrants 12 (s=+1) and 21 (s=-1)
  SymBBM Fsp;
  Fsp.m[0] = &h->fmap; Fsp.id[0] = 0;
  BlockMap fq[4] = {BlockMap(nb), BlockMap(nb), BlockMap(nb), BlockMap(nb)};
  SymBBM Fqp;
  Fqp.m[1] = &fq[1]; Fqp.m[2] = &fq[2]; Fqp.id[1] = 0; Fqp.id[2] = 1;
  Fqp.s[2] = -1; Fqp.s[3] = -1;
  Planner pf; pf.db = db;
  BlockMap *fout[4] = {&fq[0], &fq[1], &fq[2], &fq[3]};
  if (!pf.product('t', WL, 'n', Fsp, 'n', WR, Fqp, fout)) return fail(PNFAM_GPU_EINVAL, pf.err);
  h->xmap = fq[1];
  h->ymap = fq[2];
  if (h->xmap.nelem(db) != nxy || h->ymap.nelem(db) != nxy)
    return fail(PNFAM_GPU_EINVAL, "operator block structure not supported (X/Y sizes differ from f)");
  // which elements of the transforms' outputs the groups write (both kernels
  // store every element of a group's block): complete coverage lets the stages
  // skip zeroing the outputs first
  auto cover = [&](std::vector<char> &cov, const std::vector<Group> &groups) {
    for (const auto &g : groups) {
      const int nct = (g.ncol + 15) / 16;
      if (g.nrow <= 0 || nct < 1 || nct > TP_MAXCT) continue;
      const size_t o = (size_t)g.out_slot * nxy + g.out_off, n = (size_t)g.nrow * g.ncol;
      if (o + n > cov.size()) continue;
      std::fill(cov.begin() + o, cov.begin() + o + n, 1);
    }
  };
  auto full = [](const std::vector<char> &cov) { return std::find(cov.begin(), cov.end(), 0) == cov.end(); };
  std::vector<char> cov_q2s((size_t)8 * nxy, 0), cov_s2q((size_t)4 * nxy, 0);
  // dR_sp = WL dR_qp WR^T, per re/im: quadrant signs/transposes of pnfam_solver.f90:354-363
  for (int ri = 0; ri < 2; ++ri) {
    SymBBM dR;
    dR.m[1] = &h->xmap; dR.m[2] = &h->ymap;
    dR.id[1] = 2 * ri; dR.id[2] = 2 * ri + 1;   // vin slots: ReX ReY ImX ImY
    dR.s[2] = -1; dR.s[3] = -1;
    dR.imag = ri == 1;
    SymBBM out;
    BlockMap om[4] = {BlockMap(nb), BlockMap(nb), BlockMap(nb), BlockMap(nb)};
    for (int q = 0; q < 4; ++q) { out.m[q] = &om[q]; out.id[q] = 2 * q + ri; }
    if (ri == 0) { out.s[1] = -1; out.s[3] = -1; } else { out.s[1] = -1; out.s[2] = -1; out.s[3] = -1; }
    out.t[1] = out.t[2] = out.t[3] = 't';
    out.imag = ri == 1;
    Planner p; p.db = db;
    BlockMap *omp[4] = {&om[0], &om[1], &om[2], &om[3]};
    if (!p.product('n', WL, 'n', dR, 't', WR, out, omp)) return fail(PNFAM_GPU_EINVAL, p.err);
    if (ri == 0) for (int q = 0; q < 4; ++q) h->rspmap[q] = om[q];
    for (int q = 0; q < 4; ++q)
      if (om[q].nelem(db) > nxy) return fail(PNFAM_GPU_EINVAL, "density quadrant larger than nxy");
    std::vector<Term> terms; std::vector<Group> groups;
    p.finish(terms, groups);
    cover(cov_q2s, groups);
    size_t lds = 0;
    for (auto &g : groups) lds = std::max(lds, (size_t)g.nrow * g.ncol * 8);
    h->lds_q2s = std::max(h->lds_q2s, lds);
    if (ri == 0) h->flops_q2s = 0;
    for (auto &t : terms) h->flops_q2s += 2.0 * t.nda * t.nda * t.ndc + 2.0 * t.nda * t.ndc * t.ndc;
    tp_patch_terms(h, terms);
    if (!tp_terms_ok(terms)) h->tp_bf16 = h->tp64_ok = false;   // A or C not whole blocks: the plain FP64 products only
    int e;
    if (ri == 0) { h->tpa_terms_h[0].clear(); h->tpa_groups_h[0].clear(); h->tpa_toff_h[0].clear(); h->tpa_jobs_h[0].clear(); }
    h->tp_L[0] = tp_b_layout(h, 0, terms, groups, ri == 0 ? 0 : h->tp_L[0]);
    if (ri == 1 && (e = tp_finish_stage(h, 0))) return e;
    if ((e = upload(h->d_terms_q2s[ri], terms.data(), std::max<size_t>(1, terms.size()) * sizeof(Term), h->stream)) ||
        (e = upload(h->d_groups_q2s[ri], groups.data(), std::max<size_t>(1, groups.size()) * sizeof(Group), h->stream)))
      return e;
    h->ngroups_q2s[ri] = (int)groups.size();
  }
  // dH_sp structures preset as the reference (pnfam_solver.f90:402-413):
  // h_pn, h_np like f; Delta+ like X; Delta- like Y
  h->hspmap[0] = h->fmap; h->hspmap[1] = h->xmap; h->hspmap[2] = h->ymap; h->hspmap[3] = h->fmap;
  for (int ri = 0; ri < 2; ++ri) {
    SymBBM dH;
    for (int q = 0; q < 4; ++q) { dH.m[q] = &h->hspmap[q]; dH.id[q] = 2 * q + ri; }
    if (ri == 0) { dH.s[2] = -1; dH.s[3] = -1; } else { dH.s[3] = -1; }
    dH.t[3] = 't';
    dH.imag = ri == 1;
    SymBBM out;
    BlockMap om[4] = {BlockMap(nb), BlockMap(nb), BlockMap(nb), BlockMap(nb)};
    out.m[1] = &om[1]; out.m[2] = &om[2];
    out.id[1] = ri == 0 ? 0 : 2; out.id[2] = ri == 0 ? 1 : 3;   // hqp slots
    out.s[2] = -1; out.s[3] = -1;
    out.imag = ri == 1;
    Planner p; p.db = db;
    BlockMap *omp[4] = {&om[0], &om[1], &om[2], &om[3]};
    if (!p.product('t', WL, 'n', dH, 'n', WR, out, omp)) return fail(PNFAM_GPU_EINVAL, p.err);
    for (int i = 0; i < nb; ++i)
      if (om[1].ir2c[i] != h->xmap.ir2c[i] || om[2].ir2c[i] != h->ymap.ir2c[i])
        return fail(PNFAM_GPU_EINVAL, "dH_qp structure differs from dR_qp");
    std::vector<Term> terms; std::vector<Group> groups;
    p.finish(terms, groups);
    cover(cov_s2q, groups);
    size_t lds = 0;
    for (auto &g : groups) lds = std::max(lds, (size_t)g.nrow * g.ncol * 8);
    h->lds_s2q = std::max(h->lds_s2q, lds);
    if (ri == 0) h->flops_s2q = 0;
    for (auto &t : terms) h->flops_s2q += 2.0 * t.nda * t.nda * t.ndc + 2.0 * t.nda * t.ndc * t.ndc;
    tp_patch_terms(h, terms);
    if (!tp_terms_ok(terms)) h->tp_bf16 = h->tp64_ok = false;   // A or C not whole blocks: the plain FP64 products only
    int e;
    if (ri == 0) { h->tpa_terms_h[1].clear(); h->tpa_groups_h[1].clear(); h->tpa_toff_h[1].clear(); h->tpa_jobs_h[1].clear(); }
    h->tp_L[1] = tp_b_layout(h, 1, terms, groups, ri == 0 ? 0 : h->tp_L[1]);
    if (ri == 1 && (e = tp_finish_stage(h, 1))) return e;
    if ((e = upload(h->d_terms_s2q[ri], terms.data(), std::max<size_t>(1, terms.size()) * sizeof(Term), h->stream)) ||
        (e = upload(h->d_groups_s2q[ri], groups.data(), std::max<size_t>(1, groups.size()) * sizeof(Group), h->stream)))
      return e;
    h->ngroups_s2q[ri] = (int)groups.size();
  }
  h->q2s_cover = full(cov_q2s);
  h->s2q_cover = full(cov_s2q);
  // density pair lists: sector 0 (rho_pn = m11, kappa+ = m12), sector 1 (rho_np = m22, kappa- = m21)
  std::vector<int4> pl;
  const BlockMap *pm[4] = {&h->rspmap[0], &h->rspmap[1], &h->rspmap[3], &h->rspmap[2]};
  for (int k = 0; k < 4; ++k) {
    auto v = pair_list(*pm[k]);
    h->pair_off[k] = (int)pl.size();
    h->pair_n[k] = (int)v.size();
    pl.insert(pl.end(), v.begin(), v.end());
  }
  int e;
  if ((e = upload(h->d_pairs, pl.data(), std::max<size_t>(1, pl.size()) * sizeof(int4), h->stream))) return e;
  // projection tiles: h_pn (slot 0, sector 0), Delta+ (slot 1, sector 0), Delta- (slot 2, sector 1), h_np (slot 3, sector 1)
  std::vector<Tile> tiles;
  const int slot_sec[4] = {0, 0, 1, 1};
  for (int q = 0; q < 4; ++q) {
    for (auto &p : pair_list(h->hspmap[q])) {
      const int dx = db[p.x], dy = db[p.y];
      for (int a0 = 0; a0 < dx; a0 += PT)
        for (int b0 = 0; b0 < dy; b0 += PT) {
          Tile t{};
          t.ix = p.x; t.iy = p.y; t.off = p.z; t.sec = slot_sec[q];
          t.a0 = a0; t.b0 = b0; t.na = std::min(PT, dx - a0); t.nb_ = std::min(PT, dy - b0);
          t.out_slot = q; t.kind = (q == 1 || q == 2) ? 1 : 0;
          tiles.push_back(t);
        }
    }
  }
  h->ntiles = (int)tiles.size();
  if ((e = upload(h->d_tiles, tiles.data(), std::max<size_t>(1, tiles.size()) * sizeof(Tile), h->stream))) return e;
  if ((e = build_tiles2(h))) return e;
  // element -> (row state, column state) for the Green's function
  auto rc = [&](const BlockMap &m, std::vector<int> &row, std::vector<int> &col) {
    row.assign(nxy, 0); col.assign(nxy, 0);
    for (int i = 0; i < nb; ++i) {
      int j = m.ir2c[i];
      if (j < 0) continue;
      for (int c = 0; c < db[j]; ++c)
        for (int r = 0; r < db[i]; ++r) {
          long e2 = m.ir2m[i] + r + (long)c * db[i];
          row[e2] = h->isstart[i] + r;
          col[e2] = h->isstart[j] + c;
        }
    }
  };
  std::vector<int> xr, xc, yr, yc;
  rc(h->xmap, xr, xc);
  rc(h->ymap, yr, yc);
  if ((e = upload(h->d_xrow, xr.data(), nxy * 4, h->stream)) || (e = upload(h->d_xcol, xc.data(), nxy * 4, h->stream)) ||
      (e = upload(h->d_yrow, yr.data(), nxy * 4, h->stream)) || (e = upload(h->d_ycol, yc.data(), nxy * 4, h->stream)))
    return e;
  // Fqp on the device with the same product machinery (one "frequency": B = f)
  h->nxy = nxy;
  {
    int dmax = 0;
    for (int i = 0; i < nb; ++i) dmax = std::max(dmax, db[i]);
    if (dmax > 16 * TP_MAXCT) return fail(PNFAM_GPU_EINVAL, "block size above 128 is not supported");
    h->strips = (dmax + 15) / 16;
  }
  {
    Planner p; p.db = db;
    SymBBM F1 = Fsp;
    BlockMap om[4] = {BlockMap(nb), BlockMap(nb), BlockMap(nb), BlockMap(nb)};
    SymBBM out = Fqp;
    out.m[1] = &om[1]; out.m[2] = &om[2];
    BlockMap *omp[4] = {&om[0], &om[1], &om[2], &om[3]};
    if (!p.product('t', WL, 'n', F1, 'n', WR, out, omp)) return fail(PNFAM_GPU_EINVAL, p.err);
    p.finish(h->fq_terms, h->fq_groups);
    h->fq_lds = 8;
    for (auto &g : h->fq_groups) h->fq_lds = std::max(h->fq_lds, (size_t)g.nrow * g.ncol * 8);
    if ((e = h->d_f20.alloc(nxy * 8)) || (e = h->d_f02.alloc(nxy * 8))) return e;
    if ((e = to_qp(h, f_elem, 1, h->d_f20.as<double>(), h->d_f02.as<double>()))) return e;
  }
  h->nx = 0;
  // algorithmic FLOP per frequency and iteration for the kernels that carry the arithmetic
  for (double &f : h->flops_unit) f = 0.0;
  {
    const double G = h->nghl;
    double q2s = 0, s2q = 0;
    // recompute from the term tables kept on the host side of the planner
    q2s = h->flops_q2s; s2q = h->flops_s2q;
    const double nr0 = (double)h->rspmap[0].nelem(db), nk0 = (double)h->rspmap[1].nelem(db);
    const double nr1 = (double)h->rspmap[3].nelem(db), nk1 = (double)h->rspmap[2].nelem(db);
    h->flops_unit[K_TRIPROD_Q2S] = q2s;
    h->flops_unit[K_TRIPROD_S2Q] = s2q;
    h->gen_flops_d = G * (16.0 * (nr0 + nr1) + 4.0 * (nk0 + nk1));
    h->gen_flops_p = G * (20.0 * (double)(h->hspmap[0].nelem(db) + h->hspmap[3].nelem(db)) +
                          4.0 * (double)(h->hspmap[1].nelem(db) + h->hspmap[2].nelem(db)));
    h->flops_unit[K_DENSITY] = h->gen_flops_d;
    h->flops_unit[K_PROJECT] = h->gen_flops_p;
  }
  if ((e = sep_build(h))) return e;
  h->have_op = true;
  h->cap = 0;
  h->hist_cap = -1;
  if (nxy_out) *nxy_out = nxy;
  return 0;
}

int pnfam_gpu_profile(pnfam_gpu_ctx *h, int32_t enable) {
  if (!h) return fail(PNFAM_GPU_EINVAL, "null context");
  HIP_TRY(hipStreamSynchronize(h->stream));
  prof_collect(h);
  for (auto &k : h->kstat) k = pnfam_gpu_ctx::KStat();
  h->classes.clear();
  h->prof = enable != 0;
  return 0;
}

int pnfam_gpu_profile_read(pnfam_gpu_ctx *h, int32_t max_kernels, char *names, double *ms, int64_t *launches,
                           double *units, double *flops_per_unit, int32_t *n_out) {
  if (!h || !n_out) return fail(PNFAM_GPU_EINVAL, "null argument");
  HIP_TRY(hipStreamSynchronize(h->stream));
  prof_collect(h);
  const int n = std::min<int>(max_kernels, K_NKERNEL);
  for (int k = 0; k < n; ++k) {
    if (names) { std::memset(names + 32 * k, 0, 32); std::strncpy(names + 32 * k, kKernelNames[k], 31); }
    if (ms) ms[k] = h->kstat[k].ms;
    if (launches) launches[k] = h->kstat[k].launches;
    if (units) units[k] = h->kstat[k].units;
    if (flops_per_unit) flops_per_unit[k] = h->flops_unit[k];
  }
  *n_out = n;
  return 0;
}

int pnfam_gpu_structures(pnfam_gpu_ctx *h, int32_t *maps, int32_t *xy_maps) {
  if (!h || !h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  for (int q = 0; q < 4; ++q)
    if (maps) std::copy(h->rspmap[q].ir2c.begin(), h->rspmap[q].ir2c.end(), maps + q * h->nb);
  if (xy_maps) {
    std::copy(h->xmap.ir2c.begin(), h->xmap.ir2c.end(), xy_maps);
    std::copy(h->ymap.ir2c.begin(), h->ymap.ir2c.end(), xy_maps + h->nb);
  }
  return 0;
}

int pnfam_gpu_get_fqp(pnfam_gpu_ctx *h, double *f20, double *f02) {
  if (!h || !h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  HIP_TRY(hipMemcpy(f20, h->d_f20.p, h->nxy * 8, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(f02, h->d_f02.p, h->nxy * 8, hipMemcpyDeviceToHost));
  return 0;
}

// The per-unit entry points run their one frequency in unit_reps batch slots
// with identical inputs (slot 0 copied to the others) and return the last slot.
static int one_point(pnfam_gpu_ctx *h) {
  if (!h || !h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  const int R = h->unit_reps;
  h->bs.valid = false;
  h->sep_nomem = false;
  h->hook_M = -2;
  if (int e = ensure_workspace(h, R, h->hist_cap < 0 ? 1 : h->hist_cap)) return e;
  h->unit_act.resize(R);
  std::iota(h->unit_act.begin(), h->unit_act.end(), 0);
  HIP_TRY(hipMemcpy(h->d_act.p, h->unit_act.data(), (size_t)R * 4, hipMemcpyHostToDevice));
  return 0;
}

static int replicate(pnfam_gpu_ctx *h, double *base, size_t stride) {
  for (int r = 1; r < h->unit_reps; ++r)
    HIP_TRY(hipMemcpyAsync(base + r * stride, base, stride * 8, hipMemcpyDeviceToDevice, h->stream));
  return 0;
}

int pnfam_gpu_qp2sp(pnfam_gpu_ctx *h, const double *x_re, const double *x_im, const double *y_re, const double *y_im,
                    double *rsp) {
  if (int e = one_point(h)) return e;
  const long n = h->nxy;
  const int R = h->unit_reps;
  double *v = h->d_vin.as<double>();
  HIP_TRY(hipMemcpyAsync(v, x_re, n * 8, hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(v + n, y_re, n * 8, hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(v + 2 * n, x_im, n * 8, hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(v + 3 * n, y_im, n * 8, hipMemcpyHostToDevice, h->stream));
  if (int e = replicate(h, v, 4 * n)) return e;
  if (int e = stage_qp2sp(h, v, R, h->d_act.as<int>(), h->unit_precision != PNFAM_GPU_FP64 && h->tp_bf16, R)) return e;
  HIP_TRY(hipMemcpyAsync(rsp, h->d_rsp.as<double>() + (size_t)(R - 1) * 8 * n, 8 * n * 8, hipMemcpyDeviceToHost,
                         h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return 0;
}

// The 16-array argument order of calc_dHsp_interface (rho_pn, kappa+, rho_np,
// kappa-; h_pn, Delta+, h_np, Delta-) maps to quadrant slots m11, m12, m22, m21.
static const int kArgSlot[8] = {0, 1, 2, 3, 6, 7, 4, 5};

static int upload_args(pnfam_gpu_ctx *h, DevPtr &dst, const double *in) {
  const long n = h->nxy;
  for (int k = 0; k < 8; ++k)
    HIP_TRY(hipMemcpyAsync(dst.as<double>() + (size_t)kArgSlot[k] * n, in + (size_t)k * n, n * 8,
                           hipMemcpyHostToDevice, h->stream));
  return replicate(h, dst.as<double>(), 8 * (size_t)n);
}

static int unit_hamiltonian(pnfam_gpu_ctx *h) {
  const int R = h->unit_reps;
  if (h->unit_precision == PNFAM_GPU_FP64) {
    const GridBufs gb{h->d_rsp.as<double>(), 3, 2, h->d_dens.as<double>(), h->d_flds.as<double>(),
                      h->d_hsp.as<double>(), h->few_split_on != 0};
    return h->unit_general ? stage_hamiltonian_on(h, R, h->d_act.as<int>(), gb) : stage_hamiltonian(h, R, h->d_act.as<int>());
  }
  if (int e = mix_prepare(h)) return e;
  return stage_hamiltonian_lowp(h, R, h->d_act.as<int>(), R);
}

int pnfam_gpu_set_unit_precision(pnfam_gpu_ctx *h, int32_t precision) {
  if (!h) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (precision != PNFAM_GPU_FP64 && precision != PNFAM_GPU_MIXED)
    return fail(PNFAM_GPU_EINVAL, "unit precision must be FP64 or MIXED");
  h->unit_precision = precision;
  return 0;
}

int pnfam_gpu_calc_hamiltonian(pnfam_gpu_ctx *h, const double *in, double *out) {
  if (int e = one_point(h)) return e;
  const long n = h->nxy;
  if (int e = upload_args(h, h->d_rsp, in)) return e;
  if (int e = unit_hamiltonian(h)) return e;
  const double *last = h->d_hsp.as<double>() + (size_t)(h->unit_reps - 1) * 8 * n;
  for (int k = 0; k < 8; ++k)
    HIP_TRY(hipMemcpyAsync(out + (size_t)k * n, last + (size_t)kArgSlot[k] * n, n * 8, hipMemcpyDeviceToHost,
                           h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return 0;
}

int pnfam_gpu_densities(pnfam_gpu_ctx *h, const double *in, int32_t sector, double *dens) {
  if (sector != 0 && sector != 1) return fail(PNFAM_GPU_EINVAL, "sector must be 0 or 1");
  if (int e = one_point(h)) return e;
  if (int e = upload_args(h, h->d_rsp, in)) return e;
  if (int e = unit_hamiltonian(h)) return e;
  HIP_TRY(hipMemcpyAsync(dens, h->d_dens.as<double>() + ((size_t)(h->unit_reps - 1) * 2 + sector) * 2 * NDENS * h->nghl,
                         (size_t)2 * NDENS * h->nghl * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return 0;
}

int pnfam_gpu_sp2qp(pnfam_gpu_ctx *h, const double *hsp, double *h20_re, double *h20_im, double *h02_re,
                    double *h02_im) {
  if (int e = one_point(h)) return e;
  const long n = h->nxy;
  if (int e = upload_args(h, h->d_hsp, hsp)) return e;
  const int R = h->unit_reps;
  if (int e = stage_sp2qp(h, R, h->d_act.as<int>(), h->unit_precision != PNFAM_GPU_FP64 && h->tp_bf16, R)) return e;
  const double *q = h->d_hqp.as<double>() + (size_t)(R - 1) * 4 * n;
  HIP_TRY(hipMemcpyAsync(h20_re, q, n * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipMemcpyAsync(h02_re, q + n, n * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipMemcpyAsync(h20_im, q + 2 * n, n * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipMemcpyAsync(h02_im, q + 3 * n, n * 8, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return 0;
}

// ---- batched ifam --------------------------------------------------------

// One modified-Broyden step (pnfam_broyden.f90:117-216) for the na points of
// act: vout <- vout - vin, si = max|vout|, vin <- mixed update.  M < 0: no mixing;
// M = 0 or iter = 0: linear mixing; else the incremental-Gram Broyden update.
static int bro_run(pnfam_gpu_ctx *h, int M, int iter, double alpha, int na, const int *dact, bool hist32,
                   const int *drop, bool mixed, const int *iterp = nullptr, const int *lag = nullptr) {
  hipStream_t st = h->stream;
  const long N = 4 * h->nxy;
  BroArgs B{};
  B.vin = h->d_vin.as<double>(); B.vout = h->d_vout.as<double>(); B.df = h->d_df.p; B.dv = h->d_dv.p;
  B.pdf = h->d_pdf.as<double>();
  B.part = h->d_part.as<double>(); B.gram = h->d_gram.as<double>();
  B.coef = h->d_coef.as<double>(); B.si = h->d_si.as<double>(); B.scal = h->d_scal.as<double>();
  B.vmax = h->d_vmax.as<double>();
  B.dvin = mixed ? h->d_dvin.as<double>() : nullptr;
  B.drop = drop;
  // with the FP32 history (its reductions need not match the FP64 path's order)
  // and few points, more workgroups per point keep more loads in flight
  const int nwg_it = (hist32 && na <= BRO_FEW) ? h->bro_nwg_few : h->bro_nwg;
  B.N = N; B.M = std::max(M, 0); B.nwg = nwg_it; B.iter = iter; B.alpha = alpha; B.act = dact; B.skip = h->skip_slot;
  int mode = 0;
  if (M < 0) mode = 2;
  else if (M == 0 || iter == 0) mode = 1;
  if (mode == 0) {
    B.iter_used = std::min(iter - 1, M);
    B.ipos = (iter - 1 - ((iter - 2) / M) * M) - 1;   // 0-based slots
    B.inext = (iter - ((iter - 1) / M) * M) - 1;
    if (iter < 2) B.ipos = 0;
  }
  B.iter = mode == 0 ? iter : 0;
  B.iterp = mode == 0 ? iterp : nullptr;
  B.lag = mode == 0 ? lag : nullptr;
  { Prof pr(h, K_BRO_RESID, na);
    if (hist32) hipLaunchKernelGGL(k_bro_resid<float>, dim3(nwg_it, na), dim3(BRO_WG), 0, st, B);
    else hipLaunchKernelGGL(k_bro_resid<double>, dim3(nwg_it, na), dim3(BRO_WG), 0, st, B); }
  { Prof pr(h, K_BRO_NORM, na); hipLaunchKernelGGL(k_bro_norm, dim3(na), dim3(64), 0, st, B); }
  if (mode == 0) {
    { Prof pr(h, K_BRO_DOTS, na);
      if (hist32) hipLaunchKernelGGL(k_bro_dots<float>, dim3(nwg_it, na), dim3(BRO_WG), 0, st, B);
      else hipLaunchKernelGGL(k_bro_dots<double>, dim3(nwg_it, na), dim3(BRO_WG), 0, st, B); }
    { Prof pr(h, K_BRO_SOLVE, na); hipLaunchKernelGGL(k_bro_solve, dim3(na), dim3(512), 0, st, B); }
  }
  { Prof pr(h, K_BRO_UPDATE, na);
    if (hist32) hipLaunchKernelGGL(k_bro_update<float>, dim3(nwg_it, na), dim3(BRO_WG), 0, st, B, mode);
    else hipLaunchKernelGGL(k_bro_update<double>, dim3(nwg_it, na), dim3(BRO_WG), 0, st, B, mode); }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Strength (and cross-terms) of the active points from their current amplitudes.
static int contract_active(pnfam_gpu_ctx *h, int na, const int *dact, HostRes R = {}) {
  hipStream_t st = h->stream;
  const int cnwg = 64;
  { Prof pr(h, K_CONTRACT, na);
    hipLaunchKernelGGL(k_contract, dim3(cnwg, na, 1), dim3(256), 0, st, h->d_vin.as<double>(), h->d_f20.as<double>(),
                       h->d_f02.as<double>(), h->nxy, h->d_cpart.as<double>(), cnwg, dact, 0L, 1, h->skip_slot);
    if (h->nx > 0)
      hipLaunchKernelGGL(k_contract, dim3(cnwg, na, h->nx), dim3(256), 0, st, h->d_vin.as<double>(),
                         h->d_g20.as<double>(), h->d_g02.as<double>(), h->nxy, h->d_xpart.as<double>(), cnwg, dact,
                         h->nxy, h->nx, h->skip_slot); }
  { Prof pr(h, K_CONTRACT_FIN, na);
    hipLaunchKernelGGL(k_contract_fin, dim3(na), dim3(64), 0, st, h->d_cpart.as<double>(), cnwg, h->d_S.as<double>(),
                       dact, 1, h->skip_slot, R);
    if (h->nx > 0)
      hipLaunchKernelGGL(k_contract_fin, dim3(na, h->nx), dim3(64), 0, st, h->d_xpart.as<double>(), cnwg,
                         h->d_xs.as<double>(), dact, h->nx, h->skip_slot, HostRes{}); }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Initial state of a batch: nothing (all amplitudes zero, ifam's fresh start),
// stored amplitudes (the reference's restart), or a full checkpoint (resume).
struct Start {
  const double *x_in = nullptr, *si_in = nullptr, *s_in_re = nullptr, *s_in_im = nullptr;
  const unsigned char *ckpt = nullptr;
  int64_t ckpt_bytes = 0;
};

constexpr uint64_t CKPT_MAGIC = 0x31544b4d41464e50ull;   // "PNFAMKT1"
struct CkptHead {
  uint64_t magic;
  int32_t npts, iter, M, precision, hist32, nx;
  int64_t nxy, bytes;
  double eps, quench, alpha;
};

// Device arrays of a checkpoint: pointer and bytes of each, in file order.
static std::vector<std::pair<void *, size_t>> ckpt_arrays(pnfam_gpu_ctx *h, int npts, int M, bool hist32, bool mixed) {
  const size_t N = 4 * (size_t)h->nxy, n = (size_t)npts, Mh = (size_t)std::max(M, 1);
  const size_t hb = hist32 ? 4 : 8;
  std::vector<std::pair<void *, size_t>> v;
  v.push_back({h->d_vin.p, n * N * 8});
  if (M > 0) {
    v.push_back({h->d_df.p, n * Mh * N * hb});
    v.push_back({h->d_dv.p, n * Mh * N * hb});
    v.push_back({h->d_gram.p, n * Mh * Mh * 8});
    if (hist32) v.push_back({h->d_pdf.p, n * N * 8});
  }
  if (mixed) {
    v.push_back({h->d_dvin.p, n * N * 8});
    v.push_back({h->d_hacc.p, n * N * 8});
  }
  if (h->nx > 0) v.push_back({h->d_xs.p, n * (size_t)h->nx * 2 * 8});
  return v;
}

static int64_t ckpt_size(pnfam_gpu_ctx *h, const pnfam_gpu_ctx::Batch &b) {
  int64_t sz = sizeof(CkptHead) + (int64_t)b.npts * (5 * 8 + 4 * 4 + 2 * 8);
  for (auto &a : ckpt_arrays(h, b.npts, b.M, b.hist32 != 0, b.precision != PNFAM_GPU_FP64)) sz += (int64_t)a.second;
  return sz;
}

static int solve_core(pnfam_gpu_ctx *h, int32_t npts, const double *re_w, const double *im_w, const pnfam_gpu_opts *o,
                      const Start &start, double *re_s, double *im_s, int32_t *iters, double *si_final,
                      double *x_out) {
  if (!h || !o || !re_s || !im_s || !iters) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  if (npts <= 0) return fail(PNFAM_GPU_EINVAL, "npts must be positive");
  if (o->max_iter < 0) return fail(PNFAM_GPU_EINVAL, "max_iter must be >= 0");
  if (o->precision != PNFAM_GPU_FP64 && o->precision != PNFAM_GPU_MIXED && o->precision != PNFAM_GPU_MIXED_NOREFINE)
    return fail(PNFAM_GPU_EINVAL, "unknown precision");
  const bool mixed = o->precision != PNFAM_GPU_FP64;
  const bool refine = o->precision == PNFAM_GPU_MIXED;
  int M = o->broyden_history;
  const bool skip_res = std::fabs(o->quench) < 1e-10;
  if (skip_res) M = -1;   // no residual interaction: no mixing (pnfam_solver.f90:261-264)
  if (M > BRO_MAXM) return fail(PNFAM_GPU_EINVAL, "broyden_history above " + std::to_string(BRO_MAXM));
  // the mixed path keeps the Broyden history in FP32 unless mix_hist64 is set
  const bool hist32 = mixed && !h->mix_hist64 && M > 0;
  const CkptHead *ck = nullptr;
  if (start.ckpt) {
    if (start.ckpt_bytes < (int64_t)sizeof(CkptHead)) return fail(PNFAM_GPU_EINVAL, "checkpoint too short");
    ck = reinterpret_cast<const CkptHead *>(start.ckpt);
    if (ck->magic != CKPT_MAGIC) return fail(PNFAM_GPU_EINVAL, "not a pnfam_gpu checkpoint");
    if (ck->npts != npts || ck->nxy != h->nxy || ck->M != std::max(M, 0) || ck->precision != o->precision ||
        ck->hist32 != (int)hist32 || ck->nx != h->nx || ck->eps != o->convergence_epsilon ||
        ck->quench != o->quench || ck->alpha != o->alpha_mix || ck->bytes != start.ckpt_bytes)
      return fail(PNFAM_GPU_EINVAL, "checkpoint does not match this context, batch or options (only max_iter may change)");
    if (ck->iter > o->max_iter) return fail(PNFAM_GPU_EINVAL, "checkpoint is past max_iter");
  } else if (!re_w || !im_w) {
    return fail(PNFAM_GPU_EINVAL, "null frequencies");
  }
  if (mixed)
    if (int e = mix_prepare(h)) return e;
  const long nxy = h->nxy, N = 4 * nxy;
  h->bs.valid = false;
  h->sep_nomem = false;
  h->hook_M = -2;   // the Broyden hook's history shares this workspace
  // graph replay of the FP64 iteration (option graph): one more slot, the
  // spare one the replays give the entries of retired points
  const bool graph_ok = h->graph_mode && !mixed && !h->prof && M > 0 && !h->basic_kernels;
  const int nslot_alloc = npts + (graph_ok ? 1 : 0);
  h->graph_launches = 0;
  h->graph_captures = 0;
  h->graph_capture_ms = 0;
  if (int e = ensure_workspace(h, nslot_alloc, std::max(M, 0))) return e;
  if (h->nx > 0) {
    if (int e = h->d_xpart.alloc((size_t)nslot_alloc * h->nx * 64 * 2 * 8)) return e;
    if (int e = h->d_xs.alloc((size_t)nslot_alloc * h->nx * 2 * 8)) return e;
  }
  hipStream_t st = h->stream;
  auto &b = h->bs;
  b.npts = npts; b.M = std::max(M, 0); b.precision = o->precision; b.hist32 = hist32; b.nx = h->nx;
  b.eps = o->convergence_epsilon; b.quench = o->quench; b.alpha = o->alpha_mix;
  int iter0 = 0;
  bool warm = false;
  if (ck) {
    const unsigned char *q = start.ckpt + sizeof(CkptHead);
    auto take = [&](void *dst, size_t n) { std::memcpy(dst, q, n); q += n; };
    b.wre.resize(npts); b.wim.resize(npts); b.si.resize(npts); b.vmax.resize(npts); b.S.resize(2 * npts);
    b.done.resize(npts); b.refined.resize(npts); b.iters.resize(npts); b.lag.resize(npts);
    take(b.wre.data(), npts * 8); take(b.wim.data(), npts * 8); take(b.si.data(), npts * 8);
    take(b.vmax.data(), npts * 8); take(b.S.data(), 2 * npts * 8);
    take(b.done.data(), npts * 4); take(b.refined.data(), npts * 4); take(b.iters.data(), npts * 4);
    take(b.lag.data(), npts * 4);
    for (auto &a : ckpt_arrays(h, npts, M, hist32, mixed)) {
      HIP_TRY(hipMemcpyAsync(a.first, q, a.second, hipMemcpyHostToDevice, st));
      q += a.second;
    }
    // interrupted points run on; converged ones keep their result
    for (int w = 0; w < npts; ++w)
      if (b.done[w] && b.iters[w] < 0) b.done[w] = 0;
    iter0 = ck->iter;
    HIP_TRY(hipMemcpyAsync(h->d_wre.p, b.wre.data(), npts * 8, hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(h->d_wim.p, b.wim.data(), npts * 8, hipMemcpyHostToDevice, st));
    HIP_TRY(hipStreamSynchronize(st));   // pageable sources
  } else {
    b.wre.assign(re_w, re_w + npts); b.wim.assign(im_w, im_w + npts);
    b.si.assign(npts, 1.0); b.vmax.assign(npts, 1.0); b.S.assign(2 * npts, 0.0);
    b.done.assign(npts, 0); b.refined.assign(npts, 0); b.iters.assign(npts, -1); b.lag.assign(npts, 0);
    HIP_TRY(hipMemcpyAsync(h->d_wre.p, re_w, npts * 8, hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(h->d_wim.p, im_w, npts * 8, hipMemcpyHostToDevice, st));
    if (start.x_in) {
      // restart (pnfam_solver.f90:63-71): the stored amplitudes, residual and
      // strength; the Broyden history starts empty
      warm = true;
      HIP_TRY(hipMemcpyAsync(h->d_vin.p, start.x_in, (size_t)npts * N * 8, hipMemcpyHostToDevice, st));
      for (int w = 0; w < npts; ++w) {
        if (start.si_in) b.si[w] = start.si_in[w];
        if (start.s_in_re) b.S[2 * w] = start.s_in_re[w];
        if (start.s_in_im) b.S[2 * w + 1] = start.s_in_im[w];
      }
    } else {
      hipLaunchKernelGGL(k_fill, grid1((size_t)npts * N, 256), dim3(256), 0, st, h->d_vin.as<double>(),
                         (size_t)npts * N, 0.0);
    }
    if (M > 0)
      hipLaunchKernelGGL(k_fill, grid1((size_t)npts * M * M, 256), dim3(256), 0, st, h->d_gram.as<double>(),
                         (size_t)npts * M * M, 0.0);
    if (h->nx > 0)
      hipLaunchKernelGGL(k_fill, grid1((size_t)npts * h->nx * 2, 256), dim3(256), 0, st, h->d_xs.as<double>(),
                         (size_t)npts * h->nx * 2, 0.0);
    HIP_TRY(hipStreamSynchronize(st));   // pageable sources
  }
  const double *e1 = h->bminus ? h->d_Ep.as<double>() : h->d_En.as<double>();
  const double *e2 = h->bminus ? h->d_En.as<double>() : h->d_Ep.as<double>();
  std::vector<int> act, act64, actlo, sent;   // sent: the list d_act holds
  const double tau = h->mix_tau;
  const long nq = 4 * nxy;   // doubles of H20/H02 (re, im) per frequency
  // PNFAM_GPU_TRACE=1: one line per iteration on stderr (active points, BF16
  // products of the grid stage, wall time of the iteration)
  const bool trace = std::getenv("PNFAM_GPU_TRACE") != nullptr;
  // The refinement's FP64 evaluation moves the residual by the error the
  // accumulated field carried.  That jump is not a secant of the fixed-point map,
  // so the Broyden pair formed across it is zeroed (option mix_drop = 0 keeps it).
  const bool drop_pairs = mixed && refine && !skip_res && M > 0 && h->mix_drop;
  const bool needs_refine = mixed && refine && !skip_res;
  // the refinement runs when a point's residual first drops below refine_at
  // (option mix_refine_at, a multiple of the tolerance, at least 1)
  const double refine_at = h->mix_refine_at * o->convergence_epsilon;
  int *pin_drop = h->pin_act + 3 * npts;
  // Refinements in groups (option mix_refine_every = q > 1): a point that meets
  // refine_at on a batch iteration that is not a multiple of q waits, without
  // iterating, for the next one, so that its FP64 evaluation runs with those of
  // the other points that got there meanwhile.  Its own iteration (the batch's
  // less lag[w]) drives its Broyden history, its three-product test and the
  // count it reports, so its arithmetic is that of an unwaiting point; only the
  // composition of the launches it joins changes.  max_iter stays a limit on
  // the batch's iterations: every point still running stops on the same one,
  // so a resumed batch continues exactly (a point that waited may so stop with
  // up to q - 1 fewer iterations of its own).
  const int group = needs_refine ? h->mix_refine_every : 1;
  int *pin_lag = h->pin_act + 5 * npts;
  bool lag_used = false;
  for (int w = 0; w < npts; ++w) lag_used = lag_used || b.lag[w] != 0;
  auto t_last = std::chrono::steady_clock::now();
  int n3_last = 0;
  // the iteration whose hamiltonian is the first one evaluated: 1 from zero
  // amplitudes (H(0) = 0 at iteration 0), 0 from stored ones
  const int first_h = warm ? 0 : 1;
  int iter = iter0;
  // Graph replay (FP64, option graph): from the third iteration of the call on,
  // each iteration is one hipGraph launch -- k_select runs ifam's exit tests on
  // the device and writes the active list, then the transforms, grid stage,
  // G(w), Broyden (its iteration read from device memory) and strength over a
  // fixed number of slots, retired points' slots going to the spare slot npts,
  // whose workgroups return at once (skip_slot).
  // The host only launches and keeps at most three launches in flight: it waits
  // for the launch two back and reads its active count; when an eighth of the
  // slots has retired it waits for the stream and captures a graph with fewer
  // slots, and when the count is zero the batch is done (the launches after it
  // find nothing active).  The arithmetic of every point is that of the eager
  // loop, except that the few-point splits of the grid loops follow the number
  // of captured slots rather than of active points (option few_split 0 turns
  // them off in both).
  auto graph_phase = [&](int it0) -> int {
    const long n4 = (long)4 * nxy;
    HIP_TRY(hipMemcpyAsync(h->d_gdone.p, b.done.data(), npts * 4, hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(h->d_giters.p, b.iters.data(), npts * 4, hipMemcpyHostToDevice, st));
    const int ctl0[4] = {0, it0, it0, 0};
    HIP_TRY(hipMemcpyAsync(h->d_gctl.p, ctl0, sizeof ctl0, hipMemcpyHostToDevice, st));
    // the spare slot starts from zeros (its results are never read)
    hipLaunchKernelGGL(k_fill, grid1(n4, 256), dim3(256), 0, st, h->d_vin.as<double>() + npts * n4, (size_t)n4, 0.0);
    hipLaunchKernelGGL(k_fill, grid1(n4, 256), dim3(256), 0, st, h->d_vout.as<double>() + npts * n4, (size_t)n4, 0.0);
    hipLaunchKernelGGL(k_fill, grid1((size_t)M * n4, 256), dim3(256), 0, st,
                       h->d_df.as<double>() + (size_t)npts * M * n4, (size_t)M * n4, 0.0);
    hipLaunchKernelGGL(k_fill, grid1((size_t)M * n4, 256), dim3(256), 0, st,
                       h->d_dv.as<double>() + (size_t)npts * M * n4, (size_t)M * n4, 0.0);
    hipLaunchKernelGGL(k_fill, grid1((size_t)M * M, 256), dim3(256), 0, st,
                       h->d_gram.as<double>() + (size_t)npts * M * M, (size_t)M * M, 0.0);
    // the partial buffers of the few-point splits, which a capture cannot allocate
    if (h->few_split_on) {
      if (int e = h->d_dpart.alloc((size_t)FEW_SPLIT_SLABS * 2 * 2 * NDENS * h->nghl * 8)) return e;
      if (int e = h->d_ppart.alloc((size_t)FEW_SPLIT_SLABS * 8 * nxy * 8)) return e;
    }
    HIP_TRY(hipStreamSynchronize(st));   // pageable sources
    int nslots = 0;
    for (int w = 0; w < npts; ++w) nslots += b.done[w] ? 0 : 1;
    if (nslots == 0) { iter = it0; return 0; }
    // (without memory for the separable stage every capture takes the general kernels)
    if (sep_active(h) && sep_workspace(h, nslots) != 0) h->sep_nomem = true;
    int *dact = h->d_act.as<int>();
    int *ctl = h->d_gctl.as<int>();
    auto body = [&](int ns) -> int {
      hipLaunchKernelGGL(k_select, dim3(1), dim3(1024), 0, st, h->d_si.as<double>(), h->d_gdone.as<int>(),
                         h->d_giters.as<int>(), dact, ctl, npts, ns, o->convergence_epsilon, o->max_iter, npts);
      if (int e = stage_qp2sp(h, h->d_vin.as<double>(), ns, dact)) return e;
      if (int e = stage_hamiltonian(h, ns, dact)) return e;
      if (int e = stage_sp2qp(h, ns, dact)) return e;
      GreenArgs G{};
      G.hqp = h->d_hqp.as<double>(); G.f20 = h->d_f20.as<double>(); G.f02 = h->d_f02.as<double>();
      G.e1 = e1; G.e2 = e2;
      G.xrow = h->d_xrow.as<int>(); G.xcol = h->d_xcol.as<int>(); G.yrow = h->d_yrow.as<int>(); G.ycol = h->d_ycol.as<int>();
      G.wre = h->d_wre.as<double>(); G.wim = h->d_wim.as<double>(); G.vout = h->d_vout.as<double>();
      G.nxy = nxy; G.quench = o->quench; G.use_h = true; G.act = dact; G.skip = h->skip_slot;
      hipLaunchKernelGGL(k_green, dim3((unsigned)std::min<long>(1024, (2 * nxy + 255) / 256), ns), dim3(256), 0, st, G);
      // iteration 2 here only selects the Broyden step with a history; the
      // kernels read the iteration from ctl[1]
      if (int e = bro_run(h, M, 2, o->alpha_mix, ns, dact, false, nullptr, false, ctl + 1)) return e;
      return contract_active(h, ns, dact);
    };
    hipGraphExec_t ge = nullptr;
    auto capture = [&](int ns) -> int {
      const auto tc = std::chrono::steady_clock::now();
      ++h->graph_captures;
      if (hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed) != hipSuccess)
        return fail(PNFAM_GPU_EDEVICE, "hipStreamBeginCapture failed");
      h->graph_capturing = true;
      h->skip_slot = npts;   // the spare slot's workgroups return at once
      const int e = body(ns);
      h->skip_slot = -1;
      hipGraph_t g = nullptr;
      const hipError_t ce = hipStreamEndCapture(st, &g);
      h->graph_capturing = false;
      if (e) { if (g) (void)hipGraphDestroy(g); return e; }
      if (ce != hipSuccess || !g) return fail(PNFAM_GPU_EDEVICE, "hipStreamEndCapture failed");
      const hipError_t ie = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      if (ie != hipSuccess) { ge = nullptr; return fail(PNFAM_GPU_EDEVICE, "hipGraphInstantiate failed"); }
      h->graph_capture_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tc).count();
      return 0;
    };
    hipEvent_t ev[4] = {};
    int err = 0;
    for (int k = 0; k < 4 && !err; ++k)
      if (hipEventCreateWithFlags(&ev[k], hipEventDisableTiming) != hipSuccess) err = fail(PNFAM_GPU_EDEVICE, "hipEventCreate failed");
    int *ring = h->pin_act + 4 * npts;   // four ints past the staging lists (capacity npts + 1)
    int cur = nslots, launched = 0;
    if (!err) err = capture(cur);
    while (!err) {
      if (hipGraphLaunch(ge, st) != hipSuccess) { err = fail(PNFAM_GPU_EDEVICE, "hipGraphLaunch failed"); break; }
      ++launched;
      ++h->graph_launches;
      const int r = launched & 3;
      if (hipMemcpyAsync(ring + r, ctl, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
          hipEventRecord(ev[r], st) != hipSuccess) { err = fail(PNFAM_GPU_EDEVICE, "active-count copy failed"); break; }
      if (it0 + launched - 1 >= o->max_iter) break;   // that launch ends every point
      if (launched <= 2) continue;
      // at most three launches in flight: wait for the one two back (the GPU
      // keeps the two newer ones), whose active count then tells what to do
      const int rl = (launched - 2) & 3;
      if (hipEventSynchronize(ev[rl]) != hipSuccess) { err = fail(PNFAM_GPU_EDEVICE, "hipEventSynchronize failed"); break; }
      const int nl = ring[rl];
      if (nl == 0) break;
      const int retired = cur - nl;
      if (retired < 1 || 8 * retired < cur) continue;
      // an eighth of the slots (at least one) has retired: wait, and replay with
      // fewer slots (the spare-slot work is the price of not re-capturing)
      int now = 0;
      if (hipStreamSynchronize(st) != hipSuccess || hipMemcpy(&now, ctl, 4, hipMemcpyDeviceToHost) != hipSuccess) {
        err = fail(PNFAM_GPU_EDEVICE, "active-count read failed");
        break;
      }
      if (now == 0) break;
      (void)hipGraphExecDestroy(ge);
      ge = nullptr;
      cur = now;
      err = capture(cur);
    }
    const hipError_t se = hipStreamSynchronize(st);
    if (ge) (void)hipGraphExecDestroy(ge);
    for (auto e : ev) if (e) (void)hipEventDestroy(e);
    if (err) return err;
    if (se != hipSuccess) return fail(PNFAM_GPU_EDEVICE, "graph replay failed");
    int c[4];
    HIP_TRY(hipMemcpy(c, ctl, sizeof c, hipMemcpyDeviceToHost));
    if (c[3]) return fail(PNFAM_GPU_EDEVICE, "graph replay: more active points than slots");
    HIP_TRY(hipMemcpy(b.done.data(), h->d_gdone.p, npts * 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(b.iters.data(), h->d_giters.p, npts * 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(b.si.data(), h->d_si.p, npts * 8, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(b.S.data(), h->d_S.p, 2 * npts * 8, hipMemcpyDeviceToHost));
    iter = c[2];
    return 0;
  };
  if (graph_ok) {
    if (int e = h->d_gdone.alloc((size_t)npts * 4)) return e;
    if (int e = h->d_giters.alloc((size_t)npts * 4)) return e;
    if (int e = h->d_gctl.alloc(16)) return e;
  }
  for (; iter <= o->max_iter; ++iter) {
    if (graph_ok && iter >= iter0 + 2) {
      if (int e = graph_phase(iter)) return e;
      break;
    }
    act.clear(); act64.clear(); actlo.clear();
    bool any_drop = false;
    int nwait = 0;
    if (drop_pairs) std::fill(pin_drop, pin_drop + npts, 0);
    for (int w = 0; w < npts; ++w) {
      if (b.done[w]) continue;
      const int pit = iter - b.lag[w];   // the point's own iteration
      if (needs_refine && !b.refined[w] && b.si[w] < refine_at) {
        if (iter < o->max_iter) {
          if (group > 1 && pit >= 3 && iter % group != 0) {
            ++b.lag[w]; ++nwait; lag_used = true;
            continue;
          }
          // (nearly) converged on the accumulated field: one full FP64
          // evaluation replaces it, and the point iterates on until it meets
          // the tolerance
          b.refined[w] = 1;
          act.push_back(w); act64.push_back(w);
          if (drop_pairs) { pin_drop[w] = 1; any_drop = true; }
          continue;
        }
        // no iteration left for the refinement: interrupted
        b.done[w] = 1; b.iters[w] = -1; continue;
      }
      if (b.si[w] < o->convergence_epsilon) { b.done[w] = 1; b.iters[w] = pit; continue; }
      if (iter == o->max_iter) { b.done[w] = 1; b.iters[w] = -1; continue; }
      act.push_back(w);
      (mixed ? actlo : act64).push_back(w);
    }
    if (act.empty()) {
      if (nwait > 0) continue;   // only waiting points: on to their group's iteration
      break;
    }
    const int na = (int)act.size();
    int *dact = h->d_act.as<int>();
    // the device keeps the list until points retire; the results come back through
    // mapped memory (k_contract_fin): a copy is some 10 us of an iteration of 130 to
    // 180 (one point, N_sh = 8)
    if (act != sent) {
      std::memcpy(h->pin_act, act.data(), na * 4);
      HIP_TRY(hipMemcpyAsync(dact, h->pin_act, na * 4, hipMemcpyHostToDevice, st));
      sent = act;
    }
    // vin = 0 at iteration 0 of a fresh start, so H(vin) = 0 exactly there and
    // the chain is not run
    const bool use_h = !skip_res && iter >= first_h;
    if (use_h && !act64.empty()) {
      const int n64 = (int)act64.size();
      int *d64 = n64 == na ? dact : h->d_act64.as<int>();   // all active points: the same list
      if (n64 < na) {
        std::memcpy(h->pin_act + npts, act64.data(), n64 * 4);
        HIP_TRY(hipMemcpyAsync(d64, h->pin_act + npts, n64 * 4, hipMemcpyHostToDevice, st));
      }
      if (int e = stage_qp2sp(h, h->d_vin.as<double>(), n64, d64)) return e;
      if (int e = stage_hamiltonian(h, n64, d64)) return e;
      if (int e = stage_sp2qp(h, n64, d64)) return e;
      if (mixed) {
        Prof pr(h, K_MIXACC, n64);
        hipLaunchKernelGGL(k_hacc, dim3(256, n64), dim3(256), 0, st, h->d_hacc.as<double>(), h->d_hqp.as<double>(),
                           nq, 1, d64);
      }
    }
    if (use_h && !actlo.empty()) {
      // increments below tau of the amplitudes (judged by the last residual)
      // take one BF16 product: their rounding error is scaled by the increment.
      // After its FP64 refinement a point takes three products again: the
      // increments that follow carry the last digits the refinement restored.
      // Points that need three go first; n3 counts them.
      auto three = [&](int w) {
        return iter - b.lag[w] < 3 || b.refined[w] || b.si[w] >= tau * std::max(b.vmax[w], 1e-300);
      };
      std::stable_partition(actlo.begin(), actlo.end(), three);
      int n3 = 0;
      for (int w : actlo) n3 += three(w) ? 1 : 0;
      n3_last = n3;
      const int nlo = (int)actlo.size();
      int *dlo = h->d_actlo.as<int>();
      std::memcpy(h->pin_act + 2 * npts, actlo.data(), nlo * 4);
      HIP_TRY(hipMemcpyAsync(dlo, h->pin_act + 2 * npts, nlo * 4, hipMemcpyHostToDevice, st));
      // from stored amplitudes the first increment is the amplitudes themselves
      if (iter == first_h && warm)
        hipLaunchKernelGGL(k_copy_slots, dim3(256, nlo), dim3(256), 0, st, h->d_dvin.as<double>(),
                           h->d_vin.as<double>(), N, dlo);
      const bool tpl = h->tp_bf16 && !h->basic_kernels;
      if (int e = stage_qp2sp(h, h->d_dvin.as<double>(), nlo, dlo, tpl, n3)) return e;
      if (int e = (h->basic_kernels ? stage_hamiltonian(h, nlo, dlo) : stage_hamiltonian_lowp(h, nlo, dlo, n3)))
        return e;
      if (int e = stage_sp2qp(h, nlo, dlo, tpl, n3)) return e;
      { Prof pr(h, K_MIXACC, nlo);
        hipLaunchKernelGGL(k_hacc, dim3(256, nlo), dim3(256), 0, st, h->d_hacc.as<double>(), h->d_hqp.as<double>(),
                           nq, iter == first_h ? 1 : 0, dlo); }
    }
    GreenArgs G{};
    G.hqp = mixed ? h->d_hacc.as<double>() : h->d_hqp.as<double>();
    G.f20 = h->d_f20.as<double>(); G.f02 = h->d_f02.as<double>();
    G.e1 = e1; G.e2 = e2;
    G.xrow = h->d_xrow.as<int>(); G.xcol = h->d_xcol.as<int>(); G.yrow = h->d_yrow.as<int>(); G.ycol = h->d_ycol.as<int>();
    G.wre = h->d_wre.as<double>(); G.wim = h->d_wim.as<double>(); G.vout = h->d_vout.as<double>();
    G.nxy = nxy; G.quench = o->quench; G.use_h = use_h; G.act = dact;
    { Prof pr(h, K_GREEN, na);
      hipLaunchKernelGGL(k_green, dim3((unsigned)std::min<long>(1024, (2 * nxy + 255) / 256), na), dim3(256), 0, st, G); }
    const int *ddrop = nullptr;
    if (any_drop) {
      HIP_TRY(hipMemcpyAsync(h->d_drop.p, pin_drop, npts * 4, hipMemcpyHostToDevice, st));
      ddrop = h->d_drop.as<int>();
    }
    const int *dlag = nullptr;
    if (lag_used) {
      std::memcpy(pin_lag, b.lag.data(), npts * 4);
      HIP_TRY(hipMemcpyAsync(h->d_lag.p, pin_lag, npts * 4, hipMemcpyHostToDevice, st));
      dlag = h->d_lag.as<int>();
    }
    if (int e = bro_run(h, M, iter, o->alpha_mix, na, dact, hist32, ddrop, mixed, nullptr, dlag)) return e;
    const double *pr = h->pin_res;
    if (int e = contract_active(h, na, dact, HostRes{h->pin_res, h->d_si.as<double>(), h->d_vmax.as<double>(), npts}))
      return e;
    HIP_TRY(hipStreamSynchronize(st));
    for (int w : act) {
      b.si[w] = pr[w];
      if (mixed) b.vmax[w] = pr[npts + w];
      b.S[2 * w] = pr[2 * npts + 2 * w];
      b.S[2 * w + 1] = pr[2 * npts + 2 * w + 1];
    }
    if (h->prof) prof_collect(h);
    if (trace) {
      const auto t = std::chrono::steady_clock::now();
      std::fprintf(stderr, "pnfam_gpu iter %4d active %4d fp64 %4d three-product %4d ms %.3f\n", iter, na,
                   (int)act64.size(), actlo.empty() ? 0 : n3_last,
                   std::chrono::duration<double, std::milli>(t - t_last).count());
      t_last = t;
    }
  }
  b.iter = std::min(iter, o->max_iter);
  b.valid = true;
  for (int w = 0; w < npts; ++w) {
    iters[w] = b.iters[w];
    re_s[w] = b.S[2 * w];
    im_s[w] = b.S[2 * w + 1];
    if (si_final) si_final[w] = b.si[w];
  }
  if (x_out) HIP_TRY(hipMemcpy(x_out, h->d_vin.p, (size_t)npts * N * 8, hipMemcpyDeviceToHost));
  return 0;
}

int pnfam_gpu_solve_batch(pnfam_gpu_ctx *h, int32_t npts, const double *re_w, const double *im_w,
                          const pnfam_gpu_opts *o, double *re_s, double *im_s, int32_t *iters, double *si_final,
                          double *x_out) {
  return solve_core(h, npts, re_w, im_w, o, Start{}, re_s, im_s, iters, si_final, x_out);
}

int pnfam_gpu_solve_batch_restart(pnfam_gpu_ctx *h, int32_t npts, const double *re_w, const double *im_w,
                                  const pnfam_gpu_opts *o, const double *x_in, const double *si_in,
                                  const double *re_s_in, const double *im_s_in, double *re_s, double *im_s,
                                  int32_t *iters, double *si_final, double *x_out) {
  if (!x_in) return fail(PNFAM_GPU_EINVAL, "null stored amplitudes");
  Start s;
  s.x_in = x_in; s.si_in = si_in; s.s_in_re = re_s_in; s.s_in_im = im_s_in;
  return solve_core(h, npts, re_w, im_w, o, s, re_s, im_s, iters, si_final, x_out);
}

int pnfam_gpu_checkpoint_size(pnfam_gpu_ctx *h, int64_t *bytes) {
  if (!h || !bytes) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->bs.valid) return fail(PNFAM_GPU_ESTATE, "no batch state to checkpoint");
  *bytes = ckpt_size(h, h->bs);
  return 0;
}

int pnfam_gpu_checkpoint_save(pnfam_gpu_ctx *h, void *buf, int64_t bytes) {
  if (!h || !buf) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->bs.valid) return fail(PNFAM_GPU_ESTATE, "no batch state to checkpoint");
  const auto &b = h->bs;
  const int64_t need = ckpt_size(h, b);
  if (bytes < need) return fail(PNFAM_GPU_EINVAL, "checkpoint buffer too small: " + std::to_string(need) + " bytes");
  CkptHead hd{};
  hd.magic = CKPT_MAGIC; hd.npts = b.npts; hd.iter = b.iter; hd.M = b.M; hd.precision = b.precision;
  hd.hist32 = b.hist32; hd.nx = b.nx; hd.nxy = h->nxy; hd.bytes = need; hd.eps = b.eps; hd.quench = b.quench;
  hd.alpha = b.alpha;
  unsigned char *q = static_cast<unsigned char *>(buf);
  auto put = [&](const void *src, size_t n) { std::memcpy(q, src, n); q += n; };
  const int n = b.npts;
  put(&hd, sizeof hd);
  put(b.wre.data(), n * 8); put(b.wim.data(), n * 8); put(b.si.data(), n * 8); put(b.vmax.data(), n * 8);
  put(b.S.data(), 2 * n * 8); put(b.done.data(), n * 4); put(b.refined.data(), n * 4); put(b.iters.data(), n * 4);
  put(b.lag.data(), n * 4);
  for (auto &a : ckpt_arrays(h, n, b.M, b.hist32 != 0, b.precision != PNFAM_GPU_FP64)) {
    HIP_TRY(hipMemcpy(q, a.first, a.second, hipMemcpyDeviceToHost));
    q += a.second;
  }
  return 0;
}

int pnfam_gpu_solve_resume(pnfam_gpu_ctx *h, const void *buf, int64_t bytes, const pnfam_gpu_opts *o, double *re_s,
                           double *im_s, int32_t *iters, double *si_final, double *x_out) {
  if (!buf) return fail(PNFAM_GPU_EINVAL, "null checkpoint");
  Start s;
  s.ckpt = static_cast<const unsigned char *>(buf);
  s.ckpt_bytes = bytes;
  if (bytes < (int64_t)sizeof(CkptHead)) return fail(PNFAM_GPU_EINVAL, "checkpoint too short");
  const CkptHead *hd = reinterpret_cast<const CkptHead *>(buf);
  if (hd->magic != CKPT_MAGIC) return fail(PNFAM_GPU_EINVAL, "not a pnfam_gpu checkpoint");
  const int npts = hd->npts;
  return solve_core(h, npts, nullptr, nullptr, o, s, re_s, im_s, iters, si_final, x_out);
}

int pnfam_gpu_set_crossterms(pnfam_gpu_ctx *h, int32_t n, const double *g_elem) {
  if (!h || (n > 0 && !g_elem)) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  if (n < 0 || n > 64) return fail(PNFAM_GPU_EINVAL, "between 0 and 64 cross-term operators");
  h->nx = 0;
  h->bs.valid = false;
  if (n == 0) return 0;
  const size_t sz = (size_t)n * h->nxy * 8;
  if (int e = h->d_g20.alloc(sz)) return e;
  if (int e = h->d_g02.alloc(sz)) return e;
  if (int e = to_qp(h, g_elem, n, h->d_g20.as<double>(), h->d_g02.as<double>())) return e;
  h->nx = n;
  return 0;
}

int pnfam_gpu_get_crossterms(pnfam_gpu_ctx *h, int32_t npts, double *re_x, double *im_x) {
  if (!h || !re_x || !im_x) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->bs.valid || h->bs.nx != h->nx || h->nx == 0) return fail(PNFAM_GPU_ESTATE, "no cross-terms of a batch");
  if (npts != h->bs.npts) return fail(PNFAM_GPU_EINVAL, "npts differs from the last batch");
  std::vector<double> v((size_t)npts * h->nx * 2);
  HIP_TRY(hipMemcpy(v.data(), h->d_xs.p, v.size() * 8, hipMemcpyDeviceToHost));
  for (size_t k = 0; k < (size_t)npts * h->nx; ++k) { re_x[k] = v[2 * k]; im_x[k] = v[2 * k + 1]; }
  return 0;
}

int pnfam_gpu_broyden_step(pnfam_gpu_ctx *h, const pnfam_gpu_opts *o, int32_t iter, double *vout, double *vin,
                           double *si, char *flag) {
  if (!h || !o || !vout || !vin) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  if (iter < 0) return fail(PNFAM_GPU_EINVAL, "iter must be >= 0");
  const int M = o->broyden_history;
  if (M > BRO_MAXM) return fail(PNFAM_GPU_EINVAL, "broyden_history above " + std::to_string(BRO_MAXM));
  if (iter > 0 && M != h->hook_M) return fail(PNFAM_GPU_ESTATE, "history size changed without iter = 0");
  // the FP64 history stores dv + alpha df: alpha is fixed for a history
  if (iter > 0 && o->alpha_mix != h->hook_alpha)
    return fail(PNFAM_GPU_ESTATE, "alpha_mix changed without iter = 0");
  h->bs.valid = false;
  if (int e = ensure_workspace(h, 1, std::max(M, 0))) return e;
  const long N = 4 * h->nxy;
  hipStream_t st = h->stream;
  if (iter == 0) {
    h->hook_M = M;
    h->hook_alpha = o->alpha_mix;
    if (M > 0)
      hipLaunchKernelGGL(k_fill, grid1((size_t)M * M, 256), dim3(256), 0, st, h->d_gram.as<double>(), (size_t)M * M, 0.0);
  }
  int zero = 0;
  HIP_TRY(hipMemcpy(h->d_act.p, &zero, 4, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpyAsync(h->d_vin.p, vin, N * 8, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(h->d_vout.p, vout, N * 8, hipMemcpyHostToDevice, st));
  if (int e = bro_run(h, M, iter, o->alpha_mix, 1, h->d_act.as<int>(), false, nullptr, false)) return e;
  HIP_TRY(hipMemcpyAsync(vin, h->d_vin.p, N * 8, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipMemcpyAsync(vout, h->d_vout.p, N * 8, hipMemcpyDeviceToHost, st));
  double s = 0.0;
  HIP_TRY(hipMemcpyAsync(&s, h->d_si.p, 8, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (si) *si = s;
  if (flag) *flag = M < 0 ? 'N' : ((M == 0 || iter == 0) ? 'L' : 'B');
  return 0;
}

int pnfam_gpu_set_option(pnfam_gpu_ctx *h, const char *name, double value) {
  if (!h || !name) return fail(PNFAM_GPU_EINVAL, "null argument");
  const std::string n(name);
  if (n == "unit_replicas") {
    if (value < 1 || value > 256 || value != std::floor(value)) return fail(PNFAM_GPU_EINVAL, "unit_replicas in 1..256");
    h->unit_reps = (int)value;
    h->unit_general = true;
  } else if (n == "unit_general") {
    if (value != 0 && value != 1) return fail(PNFAM_GPU_EINVAL, "unit_general: 0 or 1");
    h->unit_general = value != 0;
  } else if (n == "mix_tau") {
    if (!(value >= 0)) return fail(PNFAM_GPU_EINVAL, "mix_tau must be >= 0");
    h->mix_tau = value;
  } else if (n == "mix_hist64") {
    h->mix_hist64 = value != 0;
  } else if (n == "mix_drop") {
    h->mix_drop = value != 0;
  } else if (n == "mix_refine_at") {
    if (!(value >= 1.0 && value <= 1e6)) return fail(PNFAM_GPU_EINVAL, "mix_refine_at in 1..1e6");
    h->mix_refine_at = value;
  } else if (n == "mix_refine_every") {
    if (!(value >= 1 && value <= 64) || value != std::floor(value)) return fail(PNFAM_GPU_EINVAL, "mix_refine_every in 1..64");
    h->mix_refine_every = (int)value;
  } else if (n == "mix_auto_n") {
    if (value < 0 || value > 4096) return fail(PNFAM_GPU_EINVAL, "mix_auto_n in 0..4096");
    h->mix_auto_n = (int)value;
    h->mix_auto_set = true;
  } else if (n == "proj_rows") {
    if (value < 1 || value > P2_MAXRT || value != std::floor(value))
      return fail(PNFAM_GPU_EINVAL, "proj_rows in 1.." + std::to_string(P2_MAXRT));
    h->proj_maxrt = (int)value;
    if (h->have_op)
      if (int e = build_tiles2(h)) return e;
  } else if (n == "proj_freqs") {
    if (value != 1 && value != 2 && value != 4) return fail(PNFAM_GPU_EINVAL, "proj_freqs: 1, 2 or 4");
    h->proj_nf = (int)value;
  } else if (n == "fp64_density") {
    if (value != 0 && value != 1 && value != 2)
      return fail(PNFAM_GPU_EINVAL, "fp64_density: 0 one wave, 1 two waves, 2 two waves without exchange");
    h->dens_pq = (int)value;
  } else if (n == "proj_freqs_rt1") {
    if (value != 0 && value != 1 && value != 2 && value != 4)
      return fail(PNFAM_GPU_EINVAL, "proj_freqs_rt1: 0 (as proj_freqs), 1, 2 or 4");
    h->proj_nf1 = (int)value;
  } else if (n == "fac_freqs") {
    if (value != 0 && value != 1 && value != 2) return fail(PNFAM_GPU_EINVAL, "fac_freqs: 0 (auto), 1 or 2");
    h->fac_nf = (int)value;
  } else if (n == "graph") {
    if (value != 0 && value != 1) return fail(PNFAM_GPU_EINVAL, "graph: 0 or 1");
    h->graph_mode = (int)value;
  } else if (n == "few_split") {
    if (value != 0 && value != 1) return fail(PNFAM_GPU_EINVAL, "few_split: 0 or 1");
    h->few_split_on = (int)value;
  } else if (n == "fp64_grid") {
    if (value != 0 && value != 1) return fail(PNFAM_GPU_EINVAL, "fp64_grid: 0 (separable where the basis allows) or 1 (general)");
    h->fp64_grid = (int)value;
  } else if (n == "fp64_grid_bytes") {
    if (!(value >= 0) || value > 1e15 || value != std::floor(value))
      return fail(PNFAM_GPU_EINVAL, "fp64_grid_bytes: 0 (default) or bytes");
    h->sep_limit = (size_t)value;
    h->sep_nomem = false;
    sep_release(h);
  } else if (n == "proj_stages") {
    if (value != 1 && value != 2) return fail(PNFAM_GPU_EINVAL, "proj_stages: 1 or 2");
    h->proj_ns = (int)value;
  } else if (n == "zero_skip") {
    if (value != 0 && value != 1) return fail(PNFAM_GPU_EINVAL, "zero_skip: 0 or 1");
    h->zero_skip = (int)value;
  } else if (n == "mix_table_frac") {
    if (!(value >= 0.0 && value <= 1.0)) return fail(PNFAM_GPU_EINVAL, "mix_table_frac in 0..1");
    h->mix_table_frac = value;
  } else if (n == "mix_grid") {
    if (value != 0 && value != 1 && value != 2) return fail(PNFAM_GPU_EINVAL, "mix_grid: 0 auto, 1 tables, 2 factored");
    if (h->mix_ready && (int)value != h->mix_grid) return fail(PNFAM_GPU_ESTATE, "mix_grid is fixed once the mixed path is prepared");
    h->mix_grid = (int)value;
    h->mix_grid_set = true;
  } else {
    return fail(PNFAM_GPU_EINVAL, "unknown option " + n);
  }
  return 0;
}

int pnfam_gpu_get_option(pnfam_gpu_ctx *h, const char *name, double *value) {
  if (!h || !name || !value) return fail(PNFAM_GPU_EINVAL, "null argument");
  const std::string n(name);
  if (n == "unit_replicas") *value = h->unit_reps;
  else if (n == "unit_general") *value = h->unit_general ? 1 : 0;
  else if (n == "mix_tau") *value = h->mix_tau;
  else if (n == "mix_hist64") *value = h->mix_hist64;
  else if (n == "mix_drop") *value = h->mix_drop;
  else if (n == "mix_refine_at") *value = h->mix_refine_at;
  else if (n == "mix_refine_every") *value = h->mix_refine_every;
  else if (n == "refine_waits") {   // iterations the points of the last batch waited for their refinement groups
    long t = 0;
    for (int x : h->bs.lag) t += x;
    *value = (double)t;
  }
  else if (n == "mix_auto_n") *value = h->mix_auto_n;
  else if (n == "mix_grid") *value = h->mix_grid;
  else if (n == "mix_table_frac") *value = h->mix_table_frac;
  else if (n == "zero_skip") *value = h->zero_skip;
  else if (n == "zero_skips") *value = (h->q2s_cover ? 1 : 0) + (h->s2q_cover ? 2 : 0) + (h->proj_cover ? 4 : 0);
  else if (n == "mix_table_bytes") *value = h->mix_table_bytes;
  else if (n == "fp64_density") *value = h->dens_pq;
  else if (n == "fac_freqs") *value = h->fac_nf;
  else if (n == "proj_freqs_rt1") *value = h->proj_nf1;
  else if (n == "proj_rows") *value = h->proj_maxrt;
  else if (n == "proj_freqs") *value = h->proj_nf;
  else if (n == "proj_stages") *value = h->proj_ns;
  else if (n == "graph") *value = h->graph_mode;
  else if (n == "few_split") *value = h->few_split_on;
  else if (n == "fp64_grid") *value = h->fp64_grid;
  else if (n == "fp64_separable") *value = sep_active(h) ? 1 : 0;
  else if (n == "fp64_residual") *value = h->sep_resid;
  else if (n == "fp64_grid_bytes") *value = (double)h->sep_limit;
  else if (n == "fp64_point_bytes") *value = h->sep_plan ? (double)sep_point_bytes(h) : 0;
  else if (n == "fp64_held_bytes") *value = (double)(h->d_sep_zy.bytes + h->d_sep_part.bytes);
  else if (n == "graph_launches") *value = (double)h->graph_launches;
  else if (n == "graph_captures") *value = (double)h->graph_captures;
  else if (n == "graph_capture_ms") *value = h->graph_capture_ms;
  else return fail(PNFAM_GPU_EINVAL, "unknown option " + n);
  return 0;
}

// ---- calc_hamiltonian without allocation ------------------------------------
// For callers that cannot allocate device memory (code under HIP graph capture,
// tight serving loops, harnesses that forbid hipMalloc): the grid stage's
// intermediates (local densities, fields, the dH_sp quadrants in slot order)
// live in this file-scope array, one copy per device, whose address is looked
// up once per device.  Every call on a device shares that device's copy: calls
// that overlap on one device race.
constexpr size_t NOALLOC_SCRATCH = size_t(32) << 20;   // bytes per device
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH];

constexpr int NOALLOC_MAXDEV = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[NOALLOC_MAXDEV] = {};

// Device address of this device's scratch (looked up on the first call).
static int scratch_address(int dev, void **out) {
  if (dev < 0 || dev >= NOALLOC_MAXDEV) return fail(PNFAM_GPU_EDEVICE, "device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(PNFAM_GPU_EDEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

__global__ void k_first_slot(int *act) {
  if (threadIdx.x == 0) act[0] = 0;
}

// out (calc_dHsp_interface argument order h_pn, Delta+, h_np, Delta-, re and im)
// from the dH_sp quadrants in slot order (m11, m12, m21, m22)
__global__ void k_unit_out(const double *__restrict__ hsp, double *__restrict__ out, long nxy) {
  const int k = blockIdx.y;
  const int slot = k < 4 ? k : (k < 6 ? k + 2 : k - 2);
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < nxy; e += (long)gridDim.x * blockDim.x)
    out[(size_t)k * nxy + e] = hsp[(size_t)slot * nxy + e];
}

int pnfam_gpu_calc_hamiltonian_noalloc(pnfam_gpu_ctx *h, const double *d_in, double *d_out) {
  if (!h || !d_in || !d_out) return fail(PNFAM_GPU_EINVAL, "null argument");
  if (!h->have_op) return fail(PNFAM_GPU_ESTATE, "no operator set");
  if (h->unit_precision != PNFAM_GPU_FP64) return fail(PNFAM_GPU_EINVAL, "the allocation-free call is FP64 only");
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev != h->device) return fail(PNFAM_GPU_EINVAL, "call on the device the context was created on");
  auto up = [](size_t n) { return (n + 255) & ~size_t(255); };
  const size_t b_act = 256, b_dens = up((size_t)2 * 2 * NDENS * h->nghl * 8),
               b_flds = up((size_t)2 * 2 * NFLD * h->nghl * 8), b_hsp = up((size_t)8 * h->nxy * 8);
  const size_t need = b_act + b_dens + b_flds + b_hsp;
  if (need > NOALLOC_SCRATCH)
    return fail(PNFAM_GPU_EINVAL, "problem needs " + std::to_string(need) + " bytes of scratch, above the " +
                                      std::to_string(NOALLOC_SCRATCH) + " of the allocation-free call");
  void *base = nullptr;
  if (int e = scratch_address(dev, &base)) return e;
  unsigned char *q = static_cast<unsigned char *>(base);
  int *act = reinterpret_cast<int *>(q);
  double *dens = reinterpret_cast<double *>(q + b_act);
  double *flds = reinterpret_cast<double *>(q + b_act + b_dens);
  double *hsp = reinterpret_cast<double *>(q + b_act + b_dens + b_flds);
  h->bs.valid = false;
  const bool prof = h->prof;   // event timing draws events from a pool: off for this call
  h->prof = false;
  hipLaunchKernelGGL(k_first_slot, dim3(1), dim3(64), 0, h->stream, act);
  // the input is read in the argument order: sector 1 rho_np / kappa- are pairs 2 / 3
  const GridBufs gb{d_in, 2, 3, dens, flds, hsp, false};
  int e = stage_hamiltonian_on(h, 1, act, gb);
  if (!e) {
    hipLaunchKernelGGL(k_unit_out, dim3((unsigned)std::min<long>(1024, (h->nxy + 255) / 256), 8), dim3(256), 0,
                       h->stream, hsp, d_out, h->nxy);
    const hipError_t le = hipGetLastError();
    const hipError_t se = hipStreamSynchronize(h->stream);
    if (le != hipSuccess || se != hipSuccess)
      e = fail(PNFAM_GPU_EDEVICE, std::string("calc_hamiltonian_noalloc: ") +
                                      hipGetErrorString(le != hipSuccess ? le : se));
  }
  h->prof = prof;
  return e;
}

int pnfam_gpu_kernel_classes(pnfam_gpu_ctx *h, char *buf, int32_t len, int32_t *len_out) {
  if (!h) return fail(PNFAM_GPU_EINVAL, "null context");
  std::string all;
  for (const auto &c : h->classes) { if (!all.empty()) all += ';'; all += c; }
  if (len_out) *len_out = (int32_t)all.size() + 1;
  if (buf && len > 0) {
    const size_t n = std::min<size_t>(all.size(), (size_t)len - 1);
    std::memcpy(buf, all.data(), n);
    buf[n] = 0;
  }
  return 0;
}

}  // extern "C"
