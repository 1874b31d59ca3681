// Mesh handle, sparsity pattern and the global x tier.
//
// Assembly is atomic-free and sort-free at run time. Set-up (host, once per
// mesh) builds the sorted vertex-pair block pattern, the element -> block map
// and, per block on or above the diagonal, the list of its contributions in
// ascending element order. Each Hessian evaluation is then two launches:
//   1. element pass: one lane per tet computes F, the 9x9 Hessian, its
//      vol-weighted PSD projection and the upper triangle of
//      K_e = B_e^T H+ B_e, staged per element (kKst values);
//   2. block gather: sums each block's contributions in a fixed order and
//      writes the 3 row segments of the block and of its transpose. No two
//      lanes write the same value, so values are bit-reproducible.
#include "sk_elem.h"
#include "sk_internal.h"
#include "sk_materials.h"
#include "sk_resident.h"

#include <algorithm>
#include <exception>
#include <numeric>
#include <thread>

namespace sk {

// ---------------------------------------------------------------------------
// Element passes
// ---------------------------------------------------------------------------
struct EnergyArgs {
  ElemView m;
  int64_t nv;
  const double* x;
  const double* F0;  // optional per-element offset added to F (u tier: F = J u + J x_bar)
  const double* dx;  // non-null: evaluate E(x + t dx) - E(x)
  double t;
  const double* mu;
  const double* lam;
  const double* vol;
  double* elem_energy;
  const double* mass;  // per DOF; non-null adds the kinetic and load difference
  const double* xt;
  const double* fext;
  const uint8_t* fixed;
  double inv_h2;
  double* partials;
};

template <class M>
__global__ __launch_bounds__(kBlock) void elem_energy_kernel(EnergyArgs a) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0.0;
  if (e < a.m.nt) {
    int32_t v[4];
    double D[12], xe[12], F[9];
    load_elem(a.m, e, v, D);
    gather_x(a.x, v, xe);
    make_F(xe, D, F);
    add_F0(a.F0, e, F);
    const double mu = a.mu[e], lam = a.lam ? a.lam[e] : 0.0, vol = a.vol[e];
    double val = vol * M::energy(F, mu, lam);
    if (a.dx) {
      double de[12], F1[9];
      gather_x(a.dx, v, de);
#pragma unroll
      for (int k = 0; k < 12; ++k) de[k] = xe[k] + a.t * de[k];
      make_F(de, D, F1);
      add_F0(a.F0, e, F1);
      val = vol * M::energy(F1, mu, lam) - val;
    }
    if (a.elem_energy) a.elem_energy[e] = val;
    acc = val;
  }
  if (a.mass && e < a.nv) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int64_t k = 3 * e + c;
      if (a.fixed && a.fixed[k]) continue;
      const double x0 = a.x[k];
      const double x1 = x0 + a.t * a.dx[k];
      const double d0 = x0 - a.xt[k], d1 = x1 - a.xt[k];
      acc += 0.5 * a.inv_h2 * a.mass[k] * (d1 - d0) * (d1 + d0);
      if (a.fext) acc -= a.fext[k] * (x1 - x0);
    }
  }
  double v1[1] = {acc};
  store_block_partials<1>(v1, a.partials);
}

struct ElemArgs {
  ElemView m;
  const double* x;
  const double* F0;
  const double* mu;
  const double* lam;
  const double* vol;
  double* fst;
  double* Kst;
  int psd;
  const int* active;    // optional (batched problems): skip elements whose problem is inactive
  const int32_t* pid;   // problem of each vertex, with `active`
  unsigned long long* fp64_count;  // optional: += elements whose FP32 Hessian took the FP64 polar branch
  uint8_t* flags;       // closed-form eigensystem passes: 1 where the element falls back to the Jacobi pass
};

template <class M>
__global__ __launch_bounds__(kBlock) void elem_grad_kernel(ElemArgs a) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.m.nt) return;
  int32_t v[4];
  double D[12], xe[12], F[9], P[9];
  load_elem(a.m, e, v, D);
  gather_x(a.x, v, xe);
  make_F(xe, D, F);
  add_F0(a.F0, e, F);
  M::gradient(F, a.mu[e], a.lam ? a.lam[e] : 0.0, P);
  const double vol = a.vol[e];
  double* out = a.fst + kFst * e;
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int i = 0; i < 3; ++i)
      out[3 * k + i] = vol * (P[3 * i] * D[k] + P[3 * i + 1] * D[4 + k] + P[3 * i + 2] * D[8 + k]);
}

// Element Hessian in precision R (double, or float for the mixed-precision
// path). F is formed in FP64 from the FP64 positions and rounded to R; in FP32
// the densities that use the polar decomposition (ARAP, FCR) still evaluate
// elements with det F < 1e-3 in FP64, where the FP32 SVD of a near-singular F
// loses the rotation. Returns whether that FP64 branch was taken.
template <template <typename> class M, typename R>
__device__ __forceinline__ bool elem_hessian_eval(const double (&F)[9], double mu, double lam, R (&H)[45]) {
  if (sizeof(R) == 4 && M<R>::kPolar) {
    if (det3(F) < 1e-3) {
      double Hd[45];
      M<double>::hessian(F, mu, lam, Hd);
#pragma unroll
      for (int k = 0; k < 45; ++k) H[k] = (R)Hd[k];
      return true;
    }
  }
  R Fr[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) Fr[k] = (R)F[k];
  M<R>::hessian(Fr, (R)mu, (R)lam, H);
  return false;
}

// Adds the number of lanes of the wave with `flag` set to *count: one atomic
// per wave, by the lowest flagged lane (integer sums do not depend on order).
__device__ __forceinline__ void wave_count(bool flag, unsigned long long* count) {
  const unsigned long long m = __ballot(flag);
  if (flag && (int)__lane_id() == __ffsll((long long)m) - 1) atomicAdd(count, (unsigned long long)__popcll(m));
}

// kMode 0: Hessian, vol weight and 9x9 Jacobi PSD projection for every
// element. kMode 1 (densities with a closed-form eigensystem, PSD on): the
// eigenvalue modification from that eigensystem; elements it declines are
// flagged and left to kMode 2, which runs the kMode 0 path on flagged
// elements only. Splitting the two paths over two kernels keeps the
// closed-form kernel's registers (and occupancy) free of the 9x9 Jacobi's.
template <template <typename> class M, int PSD, typename R, int kMode = 0>
__global__ __launch_bounds__(kBlock) void elem_hess_kernel(ElemArgs a) {
  __shared__ __align__(16) R stage[kBlock / kWave][kWave * 18];
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool live = e < a.m.nt && !(a.active && !a.active[a.pid[a.m.T[e]]]) && !(kMode == 2 && !a.flags[e]);
  R H[45], D[12];
  if (live) {
    int32_t v[4];
    double Dd[12], xe[12], F[9];
    load_elem(a.m, e, v, Dd);
    gather_x(a.x, v, xe);
    make_F(xe, Dd, F);
    add_F0(a.F0, e, F);
    if constexpr (kMode == 1) {
      R Fr[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) Fr[k] = (R)F[k];
      live = M<R>::hessian_psd_analytic(Fr, (R)a.mu[e], a.lam ? (R)a.lam[e] : R(0), (R)a.vol[e], PSD, R(1e-6), H);
      a.flags[e] = live ? 0 : 1;
    } else {
      const bool fp64_polar = elem_hessian_eval<M, R>(F, a.mu[e], a.lam ? a.lam[e] : 0.0, H);
      if (sizeof(R) == 4 && M<R>::kPolar && a.fp64_count) wave_count(fp64_polar, a.fp64_count);
      const R vol = (R)a.vol[e];
#pragma unroll
      for (int k = 0; k < 45; ++k) H[k] *= vol;
      if (PSD != SK_PSD_NONE) psd_project_sym<9, R>(H, PSD, R(1e-6));
    }
#pragma unroll
    for (int k = 0; k < 12; ++k) D[k] = (R)Dd[k];
    // the corners in ascending vertex order
    int32_t key[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) key[k] = 4 * v[k] + k;
    auto order = [&](int i, int j) {
      const bool swap = key[i] > key[j];
      const int32_t ki = key[i];
      key[i] = swap ? key[j] : ki;
      key[j] = swap ? ki : key[j];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const R di = D[4 * c + i], dj = D[4 * c + j];
        D[4 * c + i] = swap ? dj : di;
        D[4 * c + j] = swap ? di : dj;
      }
    };
    order(0, 1);
    order(2, 3);
    order(0, 2);
    order(1, 3);
    order(1, 2);
  }
  // K_e[3i+p][3j+q] = sum_{c,c'} D[c][i] H[3p+c][3q+c'] D[c'][j], a few values of the wave's elements at a
  // time through LDS, so that neighbouring lanes store neighbouring words: a record written by its own lane
  // reached L2 as 8- and 16-byte pieces, whose number and not their bytes took the time (48^3 with PSD, FP64
  // 254 -> 136 us, FP32 95 -> 88 us).
  const uint64_t lives = __ballot(live);
  if (!lives) return;
  const int lane = threadIdx.x % kWave;
  R* mine = stage[threadIdx.x / kWave];
  R* out = reinterpret_cast<R*>(a.Kst) + (int64_t)kKst * (e - lane);
  using W = std::conditional_t<sizeof(R) == 8, double2, float3>;  // what a lane stores at once
  constexpr int kW = sizeof(W) / sizeof(R);
  // the NV values of every lane at mine[NV lane] to its record's offset `at`
  auto flush = [&](auto nv, int at) {
    constexpr int NV = decltype(nv)::value, kPer = NV / kW;
    wave_lds_fence();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int n = k * kWave + lane, el = n / kPer;
      if (lives >> el & 1)
        *reinterpret_cast<W*>(out + (int64_t)kKst * el + at + n % kPer * kW) = reinterpret_cast<const W*>(mine)[n];
    }
    wave_lds_fence();
  };
  using Pair = std::integral_constant<int, 18>;
  using Diag = std::integral_constant<int, 6>;
  R w[3][9];  // w[p][3q+c'] = sum_c D[c][i] H[3p+c][3q+c']
  auto left = [&](int i) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int m = 0; m < 9; ++m)
        w[p][m] = D[i] * H[Sym<9>::idx(3 * p, m)] + D[4 + i] * H[Sym<9>::idx(3 * p + 1, m)] +
                  D[8 + i] * H[Sym<9>::idx(3 * p + 2, m)];
  };
  auto entry = [&](int j, int p, int q) { return w[p][3 * q] * D[j] + w[p][3 * q + 1] * D[4 + j] + w[p][3 * q + 2] * D[8 + j]; };
  auto block = [&](int j, R* o) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = 0; q < 3; ++q) o[3 * p + q] = entry(j, p, q);
  };
  auto diagonal = [&](int i) {
    if (live) {
#pragma unroll
      for (int u = 0; u < 6; ++u) mine[6 * lane + u] = entry(i, kBinvPQ[u][0], kBinvPQ[u][1]);
    }
    flush(Diag{}, kKstDiag + 6 * i);
  };
  R b03[9];
  if (live) {
    left(0);
    block(1, mine + 18 * lane);
    block(2, mine + 18 * lane + 9);
    block(3, b03);
  }
  flush(Pair{}, 0);
  diagonal(0);
  if (live) {
    left(2);
#pragma unroll
    for (int m = 0; m < 9; ++m) mine[18 * lane + m] = b03[m];
    block(3, mine + 18 * lane + 9);
  }
  flush(Pair{}, 18);
  diagonal(2);
  if (live) {
    left(1);
    block(2, mine + 18 * lane);
    block(3, mine + 18 * lane + 9);
  }
  flush(Pair{}, 36);
  diagonal(1);
  if (live) left(3);
  diagonal(3);
}

// ---------------------------------------------------------------------------
// Gathers
// ---------------------------------------------------------------------------
// Sum over the four lanes of a quad, in each of them: (x0 + x1) + (x2 + x3).
template <int kPerm>
__device__ __forceinline__ float quad_perm(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kPerm, 0xf, 0xf, true));
}
template <int kPerm>
__device__ __forceinline__ double quad_perm(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kPerm, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), kPerm, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <typename R>
__device__ __forceinline__ R quad_sum(R x) {
  x += quad_perm<0xB1>(x);         // [1, 0, 3, 2]
  return x + quad_perm<0x4E>(x);   // [2, 3, 0, 1]
}
constexpr int kQuad = 4;

struct GatherGArgs {
  int64_t nv;
  const int32_t* vptr;
  const int32_t* vlist;
  const double* fst;
  double* g;
  const double* mass;
  const double* x;
  const double* xt;
  const double* fext;
  const uint8_t* fixed;
  double inv_h2;
  double* partials;
};

// Four lanes per vertex: lane s sums the incidences s, s + 4, ... of the list,
// then lane c writes DOF c. A lane per vertex was a chain of up to 32 dependent
// loads on few waves: 10^3 22.5 -> 5.7 us, a 29 x 13 x 21 box 20 -> 11.5; at 48^3
// the reads themselves bound it (42 -> 41 us).
__global__ __launch_bounds__(kBlock) void gather_grad_kernel(GatherGArgs a) {
  const int s = threadIdx.x % kQuad;
  double nrm = 0.0;
  for (int64_t v = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kQuad; v < a.nv;
       v += (int64_t)gridDim.x * (kBlock / kQuad)) {
    double acc[3] = {0.0, 0.0, 0.0};
    const int32_t k1 = a.vptr[v + 1];
#pragma unroll 2
    for (int32_t k = a.vptr[v] + s; k < k1; k += kQuad) {
      const int32_t pk = a.vlist[k];
      const double* f = a.fst + (int64_t)kFst * (pk >> 2) + 3 * (pk & 3);
      acc[0] += f[0];
      acc[1] += f[1];
      acc[2] += f[2];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[c] = quad_sum(acc[c]);
    if (s < 3) {
      const int64_t k = 3 * v + s;
      double gk = s == 0 ? acc[0] : s == 1 ? acc[1] : acc[2];
      if (a.mass) {
        gk += a.mass[k] * (a.x[k] - a.xt[k]) * a.inv_h2;
        if (a.fext) gk -= a.fext[k];
        if (a.fixed && a.fixed[k]) gk = 0.0;
        nrm += gk * gk;
      }
      a.g[k] = gk;
    }
  }
  if (a.mass) {
    double v1[1] = {nrm};
    store_block_partials<1>(v1, a.partials);
  }
}

struct GatherHArgs {
  int64_t nv;
  int64_t noff;             // off-diagonal blocks above the diagonal
  int64_t dgrid;            // workgroups of the diagonal blocks
  const int4* gmeta;        // [nv + noff]
  const uint32_t* glist;
  const int32_t* bptr;
  const int32_t* brow;
  const void* Kst;
  void* values;
  const double* mass;
  double inv_h2;
  const uint8_t* fixed;
  void* binv;
  const int32_t* sell_pos;  // non-null: sliced layout (slot_index; slot of each block): the
  int quad;                 //   SELL <kSellC, 1>, or with quad = 1 <kQuadC, kQuadVW> (FP32)
  const int32_t* binv_pos;  // non-null: the diagonal inverses in the quad layout (slot of each vertex)
  int bsr;                  // 1: BSR layout (block b at values[9 b + 3 p + q])
  const int* active;        // optional (batched problems): skip blocks whose problem is inactive
  const int32_t* pid;
};

// A staged block above the diagonal (9 values) or on it (its upper triangle, 6).
typedef double sk_d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef float sk_f4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void load_staged(const double* __restrict__ s, double (&B)[9]) {
  const sk_d2u* v = reinterpret_cast<const sk_d2u*>(s);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const sk_d2u d = v[t];
    B[2 * t] = d.x;
    B[2 * t + 1] = d.y;
  }
  B[8] = s[8];
}
__device__ __forceinline__ void load_staged(const float* __restrict__ s, float (&B)[9]) {
  const sk_f4u a = *reinterpret_cast<const sk_f4u*>(s), b = *reinterpret_cast<const sk_f4u*>(s + 4);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    B[t] = a[t];
    B[4 + t] = b[t];
  }
  B[8] = s[8];
}
template <typename R>
__device__ __forceinline__ void load_staged_diag(const R* __restrict__ s, R (&B)[6]) {
  using R2 = std::conditional_t<sizeof(R) == 8, double2, float2>;
  const R2* v = reinterpret_cast<const R2*>(s);
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const R2 d = v[t];
    B[2 * t] = d.x;
    B[2 * t + 1] = d.y;
  }
}

// Sums the staged contributions of a block (precision R), adds the lumped mass
// / h^2 on diagonal blocks, writes the block in CSR, BSR or a sliced order and,
// for diagonal blocks, the inverse of the fixed-DOF-masked block (inverse of
// diag(f) A diag(f) + diag(1 - f), masked to the free DOFs).
//
// The matrix is symmetric: only blocks on and above the diagonal are summed,
// an off-diagonal one by one lane that also writes its transpose. Diagonal
// blocks have several times the contributions of the others (on a grid of five
// tets per cell 32 or 8 against 4 to 6), so four lanes share one, lane s taking
// contributions s, s + 4, ..., and workgroups hold either diagonal or
// off-diagonal blocks. Workgroups of one XCD take consecutive rows, the diagonal
// ones among the others, for the records they share. Bound by the scattered
// reads of the records (80 to 216 bytes at a time) and writes of the blocks. One
// lane per block in row order, every off-diagonal block read twice, took 314 us
// at 48^3 (FP64, CSR order), this 241 us; 10^3 19.9 -> 9.4 us, FP32 at 48^3 193 -> 160 us.
// Two contributions at a time: one or four took 70 and 15 us more.
template <typename R>
__global__ __launch_bounds__(kBlock) void gather_hess_kernel(GatherHArgs a) {
  // workgroup `wg` in matrix order: an eighth of the list per XCD, the diagonal workgroups spread evenly
  const int64_t eighth = gridDim.x / 8, wg = blockIdx.x < 8 * eighth ? blockIdx.x % 8 * eighth + blockIdx.x / 8 : blockIdx.x;
  const int64_t d0 = wg * a.dgrid / gridDim.x, d1 = (wg + 1) * a.dgrid / gridDim.x;  // diagonal ones before it, and with it
  const bool diag = d1 > d0;
  const int64_t at = (diag ? d0 : wg - d0) * kBlock + threadIdx.x;
  const int64_t n = diag ? at / kQuad : at;
  if (n >= (diag ? a.nv : a.noff)) return;
  const int4 gm = a.gmeta[diag ? n : a.nv + n];  // block, its transpose, contributions [z, w)
  const int32_t v = a.brow[gm.x], w = a.brow[gm.y];
  if (a.active && !a.active[a.pid[v]]) return;
  const R* __restrict__ Kst = reinterpret_cast<const R*>(a.Kst);
  auto record = [&](uint32_t c) { return Kst + kKst * (int64_t)(c >> 5); };
  R acc[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) acc[k] = R(0);
  if (diag) {
    const int s = threadIdx.x % kQuad;
#pragma unroll 2
    for (int32_t k = gm.z + s; k < gm.w; k += kQuad) {
      const uint32_t c = a.glist[k], u = c >> 1 & 15;
      if (u >= 6) {
        R B[6];
        load_staged_diag(record(c) + kKstDiag + 6 * (u - 6), B);
#pragma unroll
        for (int m = 0; m < 6; ++m) acc[3 * kBinvPQ[m][0] + kBinvPQ[m][1]] += B[m];
      } else {  // a tet that has the vertex twice: K_ij + K_ji, half of the sum for each of the two entries
        R B[9];
        load_staged(record(c) + 9 * u, B);
#pragma unroll
        for (int m = 0; m < 6; ++m) {
          const int p = kBinvPQ[m][0], q = kBinvPQ[m][1];
          acc[3 * p + q] += R(0.5) * (B[3 * p + q] + B[3 * q + p]);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      const int p = kBinvPQ[m][0], q = kBinvPQ[m][1];
      acc[3 * q + p] = acc[3 * p + q] = quad_sum(acc[3 * p + q]);
    }
    if (s != 0) return;
  } else {
#pragma unroll 2
    for (int32_t k = gm.z; k < gm.w; ++k) {
      const uint32_t c = a.glist[k];
      R B[9];
      load_staged(record(c) + 9 * (c >> 1 & 15), B);
#pragma unroll
      for (int m = 0; m < 9; ++m) acc[m] += B[m];
    }
  }
  if (diag && a.mass) {
#pragma unroll
    for (int p = 0; p < 3; ++p) acc[4 * p] += (R)(a.mass[3 * (int64_t)v + p] * a.inv_h2);
  }
  R* values = reinterpret_cast<R*>(a.values);
  auto write = [&](int64_t b, int32_t row, const R (&B)[9]) {
    if (a.sell_pos) {
      const int64_t q = a.sell_pos[b];
#pragma unroll
      for (int m = 0; m < 9; ++m)
        values[a.quad ? slot_index<kQuadC, kQuadVW>(q, m) : slot_index<kSellC, 1>(q, m)] = B[m];
    } else if (a.bsr) {
      R* out = values + 9 * b;
#pragma unroll
      for (int m = 0; m < 9; ++m) out[m] = B[m];
    } else {
      const int32_t b0 = a.bptr[row], deg = a.bptr[row + 1] - b0;
      R* out = values + 9 * (int64_t)b0 + 3 * (b - b0);
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) out[3 * p * deg + q] = B[3 * p + q];
    }
  };
  write(gm.x, v, acc);
  if (!diag) {
    const R t[9] = {acc[0], acc[3], acc[6], acc[1], acc[4], acc[7], acc[2], acc[5], acc[8]};
    write(gm.y, w, t);
  }
  if (diag && a.binv) {
    R f[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) f[p] = (a.fixed && a.fixed[3 * (int64_t)v + p]) ? R(0) : R(1);
    R A[9];
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = 0; q < 3; ++q) A[3 * p + q] = f[p] * f[q] * acc[3 * p + q] + (p == q ? R(1) - f[p] : R(0));
    R c[9];
    cofactor3(A, c);
    const R det = A[0] * c[0] + A[1] * c[1] + A[2] * c[2];
    const R inv = R(1) / det;
    R* binv = reinterpret_cast<R*>(a.binv);
    if (a.binv_pos) {  // quad layout: all 9 values
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q)
          binv[slot_index<kQuadC, kQuadVW>(a.binv_pos[v], 3 * p + q)] = f[p] * f[q] * c[3 * q + p] * inv;
    } else {  // the upper triangle (the inverse of a symmetric block)
#pragma unroll
      for (int u = 0; u < kBinv; ++u) {
        const int p = kBinvPQ[u][0], q = kBinvPQ[u][1];
        binv[kBinv * (int64_t)v + u] = f[p] * f[q] * c[3 * q + p] * inv;
      }
    }
  }
}

// Per-block partial counts of elements with det F(x) <= 0 (inverted or
// collapsed), summed by a finalize launch.
__global__ __launch_bounds__(kBlock) void count_inverted_kernel(ElemView m, const double* __restrict__ x,
                                                                double* partials) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double c[1] = {0.0};
  if (e < m.nt) {
    int32_t v[4];
    double D[12], xe[12], F[9];
    load_elem(m, e, v, D);
    gather_x(x, v, xe);
    make_F(xe, D, F);
    c[0] = det3(F) <= 0.0 ? 1.0 : 0.0;
  }
  store_block_partials<1>(c, partials);
}

__global__ void csr_pattern_kernel(int64_t nv, int64_t nblk, const int32_t* bptr, const int32_t* bcol,
                                   const int32_t* brow, int32_t* indptr, int32_t* indices) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (indptr && b <= nv) {
    if (b == nv) {
      indptr[3 * nv] = (int32_t)(9 * nblk);
    } else {
      const int32_t b0 = bptr[b], deg = bptr[b + 1] - b0;
#pragma unroll
      for (int p = 0; p < 3; ++p) indptr[3 * b + p] = 9 * b0 + 3 * p * deg;
    }
  }
  if (indices && b < nblk) {
    const int32_t v = brow[b], w = bcol[b];
    const int32_t b0 = bptr[v], deg = bptr[v + 1] - b0, r = (int32_t)(b - b0);
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = 0; q < 3; ++q) indices[9 * (int64_t)b0 + 3 * p * deg + 3 * r + q] = 3 * w + q;
  }
}

__global__ void element_nnz_kernel(int64_t nt, const int32_t* T, const int32_t* bptr, const int32_t* emap,
                                   int32_t* out) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int32_t v = T[i * nt + e];
    const int32_t b0 = bptr[v], deg = bptr[v + 1] - b0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int32_t r = emap[(4 * i + j) * nt + e] - b0;
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) out[144 * e + 12 * (3 * i + p) + 3 * j + q] = 9 * b0 + 3 * p * deg + 3 * r + q;
    }
  }
}

__global__ void aos_to_soa_kernel(const double* __restrict__ D, int64_t nt, double* __restrict__ Ds) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
#pragma unroll
  for (int k = 0; k < 12; ++k) Ds[k * nt + e] = D[12 * e + k];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

int launch_elem_energy(sk_mesh* m, int material, const double* x, const double* F0, const double* dx, double t,
                       const double* mu,
                       const double* lam, const double* vol, double* elem_energy, const double* mass,
                       const double* xt, const double* fext, const uint8_t* fixed, double inv_h2,
                       hipStream_t st, double* result) {
  EnergyArgs a{view(m), m->nv, x, F0, dx, t, mu, lam, vol, elem_energy, mass, xt, fext, fixed, inv_h2,
               m->red.partials.p};
  const int64_t n = std::max<int64_t>(m->nt, mass ? m->nv : 0);
  const int g = grid_for(n);
  SK_REQUIRE(g <= Reducer::kMaxBlocks, "mesh too large for the energy reduction");
  SK_REQUIRE(dispatch_material(material, [&](auto tag) {
               elem_energy_kernel<typename decltype(tag)::template type<double>><<<g, kBlock, 0, st>>>(a);
             }),
             "unknown material");
  finalize_sum_kernel<1><<<1, kBlock, 0, st>>>(m->red.partials.p, g, result ? result : m->red.result.p);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

int launch_elem_grad(sk_mesh* m, int material, const double* x, const double* F0, const double* mu,
                     const double* lam, const double* vol, hipStream_t st) {
  ElemArgs a{view(m), x, F0, mu, lam, vol, m->fst.p, m->Kst.p, 0, nullptr, nullptr, nullptr};
  const int g = grid_for(m->nt);
  SK_REQUIRE(dispatch_material(material, [&](auto tag) {
               elem_grad_kernel<typename decltype(tag)::template type<double>><<<g, kBlock, 0, st>>>(a);
             }),
             "unknown material");
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

template <template <typename> class M, typename R>
static void hess_dispatch(int psd, int g, hipStream_t st, const ElemArgs& a) {
  if constexpr (M<R>::kAnalyticEig) {
    if (a.flags && psd != SK_PSD_NONE) {
      if (psd == SK_PSD_PROJ) {
        elem_hess_kernel<M, SK_PSD_PROJ, R, 1><<<g, kBlock, 0, st>>>(a);
        elem_hess_kernel<M, SK_PSD_PROJ, R, 2><<<g, kBlock, 0, st>>>(a);
      } else {
        elem_hess_kernel<M, SK_PSD_ABS, R, 1><<<g, kBlock, 0, st>>>(a);
        elem_hess_kernel<M, SK_PSD_ABS, R, 2><<<g, kBlock, 0, st>>>(a);
      }
      return;
    }
  }
  if (psd == SK_PSD_PROJ) elem_hess_kernel<M, SK_PSD_PROJ, R><<<g, kBlock, 0, st>>>(a);
  else if (psd == SK_PSD_ABS) elem_hess_kernel<M, SK_PSD_ABS, R><<<g, kBlock, 0, st>>>(a);
  else elem_hess_kernel<M, SK_PSD_NONE, R><<<g, kBlock, 0, st>>>(a);
}

template <template <typename> class M>
static void hess_dispatch_prec(bool fp32, int psd, int g, hipStream_t st, const ElemArgs& a) {
  if (fp32) hess_dispatch<M, float>(psd, g, st, a);
  else hess_dispatch<M, double>(psd, g, st, a);
}

int launch_elem_hess(sk_mesh* m, int material, const double* x, const double* F0, const double* mu,
                     const double* lam, const double* vol, int psd, bool fp32, hipStream_t st, const int* active,
                     const int32_t* pid, unsigned long long* fp64_count, bool closed_form) {
  SK_REQUIRE(psd == SK_PSD_NONE || psd == SK_PSD_PROJ || psd == SK_PSD_ABS, "invalid psd method");
  SK_REQUIRE(!active == !pid, "launch_elem_hess: active and pid go together");
  ElemArgs a{view(m), x, F0, mu, lam, vol, m->fst.p, m->Kst.p, psd, active, pid, fp64_count,
             closed_form ? m->eflag.p : nullptr};
  const int g = grid_for(m->nt);
  bool known = true;
  switch (material) {
    case SK_SNH: hess_dispatch_prec<SNH>(fp32, psd, g, st, a); break;
    case SK_ARAP: hess_dispatch_prec<ARAP>(fp32, psd, g, st, a); break;
    case SK_LINEAR: hess_dispatch_prec<Linear>(fp32, psd, g, st, a); break;
    case SK_MMNH: hess_dispatch_prec<MMNH>(fp32, psd, g, st, a); break;
    case SK_FCR: hess_dispatch_prec<FCR>(fp32, psd, g, st, a); break;
    default: known = false;
  }
  SK_REQUIRE(known, "unknown material");
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

int launch_count_inverted(sk_mesh* m, const double* x, double* result, hipStream_t st) {
  const int g = grid_for(m->nt);
  SK_REQUIRE(g <= Reducer::kMaxBlocks, "mesh too large for the inverted-element count");
  count_inverted_kernel<<<g, kBlock, 0, st>>>(view(m), x, m->red.partials.p);
  finalize_sum_kernel<1><<<1, kBlock, 0, st>>>(m->red.partials.p, g, result);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

int launch_gather_grad(sk_mesh* m, double* g, const double* mass, const double* x, const double* xt,
                       const double* fext, const uint8_t* fixed, double inv_h2, hipStream_t st) {
  GatherGArgs a{m->nv, m->vptr.p, m->vlist.p, m->fst.p, g, mass, x, xt, fext, fixed, inv_h2, m->red.partials.p};
  SK_REQUIRE(grid_for(m->nv) <= Reducer::kMaxBlocks, "mesh too large for the gradient reduction");
  const int gr = std::min(grid_for(kQuad * m->nv), 2048);  // eight workgroups per CU, then several vertices a quad
  gather_grad_kernel<<<gr, kBlock, 0, st>>>(a);
  if (mass) finalize_sum_kernel<1><<<1, kBlock, 0, st>>>(m->red.partials.p, gr, m->red.result.p);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

static GatherHArgs gather_args(const sk_mesh* m, void* values, const double* mass, double inv_h2, const uint8_t* fixed,
                               void* binv, const int* active, const int32_t* pid) {
  GatherHArgs a{};
  a.nv = m->nv;
  a.noff = (m->nblk - m->nv) / 2;
  a.dgrid = grid_for(kQuad * m->nv);
  a.gmeta = m->gmeta.p;
  a.glist = m->glist.p;
  a.bptr = m->bptr.p;
  a.brow = m->brow.p;
  a.Kst = m->Kst.p;
  a.values = values;
  a.mass = mass;
  a.inv_h2 = inv_h2;
  a.fixed = fixed;
  a.binv = binv;
  a.active = active;
  a.pid = pid;
  return a;
}

static int run_gather_hess(const GatherHArgs& a, bool fp32, hipStream_t st) {
  const unsigned g = (unsigned)(a.dgrid + (a.noff ? grid_for(a.noff) : 0));
  if (fp32) gather_hess_kernel<float><<<g, kBlock, 0, st>>>(a);
  else gather_hess_kernel<double><<<g, kBlock, 0, st>>>(a);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

int launch_gather_hess(sk_mesh* m, void* values, const double* mass, double inv_h2, const uint8_t* fixed,
                       void* binv, int layout, bool fp32, hipStream_t st, const int* active, const int32_t* pid) {
  SK_REQUIRE(layout == kLayoutCSR || layout == kLayoutSELL || layout == kLayoutBSR, "invalid value layout");
  SK_REQUIRE(!active == !pid, "launch_gather_hess: active and pid go together");
  GatherHArgs a = gather_args(m, values, mass, inv_h2, fixed, binv, active, pid);
  a.sell_pos = layout == kLayoutSELL ? m->sell_pos.p : nullptr;
  a.bsr = layout == kLayoutBSR ? 1 : 0;
  return run_gather_hess(a, fp32, st);
}

int launch_gather_hess_quad(sk_mesh* m, void* values, const double* mass, double inv_h2, const uint8_t* fixed,
                            void* binv, const int32_t* pos, const int32_t* row_pos, bool fp32, hipStream_t st,
                            const int* active, const int32_t* pid) {
  SK_REQUIRE(pos && (!binv || row_pos), "launch_gather_hess_quad: missing slot map");
  SK_REQUIRE(fp32, "launch_gather_hess_quad: the quad layout holds FP32 values");
  SK_REQUIRE(!active == !pid, "launch_gather_hess_quad: active and pid go together");
  GatherHArgs a = gather_args(m, values, mass, inv_h2, fixed, binv, active, pid);
  a.sell_pos = pos;
  a.quad = 1;
  a.binv_pos = row_pos;
  return run_gather_hess(a, fp32, st);
}

int read_scalars(sk_mesh* m, const double* dev, int n, hipStream_t st) {
  SK_HIP_CHECK(hipMemcpyAsync(m->pinned, dev, n * sizeof(double), hipMemcpyDeviceToHost, st));
  SK_HIP_CHECK(hipStreamSynchronize(st));
  return SK_OK;
}

// ---------------------------------------------------------------------------
// Host pattern build (once per mesh)
// ---------------------------------------------------------------------------
// Host threads for a mesh of nt tets: one per 20,000, at most 8.
static int host_threads(int64_t nt) {
  const int64_t hw = std::max(1u, std::thread::hardware_concurrency());
  return (int)std::min<int64_t>({8, hw, nt / 20000 + 1});
}

static int build_mesh(const int32_t* T, int64_t nv, int64_t nt, sk_mesh* m) {
  SK_REQUIRE(nt < (int64_t(1) << 27), "sk_mesh_create: at most 2^27 tets");
  SK_REQUIRE(nv < (int64_t(1) << 29), "sk_mesh_create: too many vertices");
  for (int64_t k = 0; k < 4 * nt; ++k)
    SK_REQUIRE(T[k] >= 0 && T[k] < nv, "sk_mesh_create: tet index out of range");

  // vertex -> (element, local corner), ascending element order
  std::vector<int32_t> vptr(nv + 1, 0), vlist(4 * nt);
  for (int64_t k = 0; k < 4 * nt; ++k) vptr[T[k] + 1]++;
  std::partial_sum(vptr.begin(), vptr.end(), vptr.begin());
  {
    std::vector<int32_t> fill(vptr.begin(), vptr.end() - 1);
    for (int64_t e = 0; e < nt; ++e)
      for (int i = 0; i < 4; ++i) vlist[fill[T[4 * e + i]]++] = (int32_t)((e << 2) | i);
  }
  // Row by row, ranges of rows on several threads: each row's sorted neighbour
  // blocks (itself included), then the element -> block map and the blocks'
  // contribution lists, from the row's incidences and a table of its blocks.
  std::vector<int32_t> bptr(nv + 1, 0);
  const int nth = host_threads(nt);
  std::vector<std::vector<int32_t>> cols(nth);
  auto ranges = [&](auto&& fn) {
    std::vector<std::exception_ptr> failed(nth);  // a thread must not end by an exception
    auto run = [&](int k) {
      try {
        fn(k, nv * k / nth, nv * (k + 1) / nth);
      } catch (...) {
        failed[k] = std::current_exception();
      }
    };
    std::vector<std::thread> pool;
    pool.reserve(nth);
    for (int k = 1; k < nth; ++k) {
      try {
        pool.emplace_back(run, k);
      } catch (...) {  // no thread to be had: here, then
        run(k);
      }
    }
    run(0);
    for (auto& t : pool) t.join();
    for (auto& e : failed)
      if (e) std::rethrow_exception(e);
  };
  ranges([&](int k, int64_t v0, int64_t v1) {
    std::vector<int32_t> seen(nv, -1), nb;
    std::vector<int32_t>& out = cols[k];
    out.reserve(16 * (v1 - v0));
    for (int64_t v = v0; v < v1; ++v) {
      nb.assign(1, (int32_t)v);
      seen[v] = (int32_t)v;
      for (int32_t q = vptr[v]; q < vptr[v + 1]; ++q) {
        const int32_t* c = T + 4 * (int64_t)(vlist[q] >> 2);
        for (int j = 0; j < 4; ++j)
          if (seen[c[j]] != v) {
            seen[c[j]] = (int32_t)v;
            nb.push_back(c[j]);
          }
      }
      std::sort(nb.begin(), nb.end());
      out.insert(out.end(), nb.begin(), nb.end());
      bptr[v + 1] = (int32_t)nb.size();
    }
  });
  int64_t nblk = 0;
  for (auto& c : cols) nblk += (int64_t)c.size();
  SK_REQUIRE(9 * nblk < (int64_t(1) << 31), "sk_mesh_create: nnz exceeds int32 indexing");
  std::partial_sum(bptr.begin(), bptr.end(), bptr.begin());
  std::vector<int32_t> bcol(nblk), brow(nblk), emap(16 * nt), cnt(nblk, 0);
  ranges([&](int k, int64_t v0, int64_t v1) {
    std::copy(cols[k].begin(), cols[k].end(), bcol.begin() + bptr[v0]);
    std::vector<int32_t> at(nv);  // block of the current row at each of its columns
    for (int64_t v = v0; v < v1; ++v) {
      for (int32_t b = bptr[v]; b < bptr[v + 1]; ++b) {
        brow[b] = (int32_t)v;
        at[bcol[b]] = b;
      }
      for (int32_t q = vptr[v]; q < vptr[v + 1]; ++q) {
        const int64_t e = vlist[q] >> 2;
        const int i = vlist[q] & 3;
        for (int j = 0; j < 4; ++j) {
          const int32_t b = at[T[4 * e + j]];
          emap[(4 * i + j) * nt + e] = b;
          cnt[b]++;
        }
      }
    }
  });
  // The blocks that the gather sums, diagonal ones first, then those above the diagonal row by row, and their
  // contribution lists in that order.
  const int64_t noff = (nblk - nv) / 2;
  std::vector<int4> gmeta(nv + noff);
  std::vector<int32_t> goff(nv + 1, 0);  // off-diagonal blocks of the rows before
  for (int64_t v = 0; v < nv; ++v)
    goff[v + 1] = goff[v] + (int32_t)(bcol.begin() + bptr[v + 1] -
                                      std::upper_bound(bcol.begin() + bptr[v], bcol.begin() + bptr[v + 1], (int32_t)v));
  ranges([&](int, int64_t v0, int64_t v1) {
    for (int64_t v = v0; v < v1; ++v) {
      int32_t o = goff[v];
      for (int32_t b = bptr[v]; b < bptr[v + 1]; ++b) {
        const int32_t w = bcol[b];
        if (w == v) gmeta[v] = make_int4(b, b, 0, cnt[b]);
        if (w <= v) continue;
        const auto r = bcol.begin() + bptr[w];
        const int32_t t = (int32_t)(std::lower_bound(r, bcol.begin() + bptr[w + 1], (int32_t)v) - bcol.begin());
        gmeta[nv + o++] = make_int4(b, t, 0, cnt[b]);
      }
    }
  });
  int32_t nlist = 0;
  for (int4& g : gmeta) {
    g.z = nlist;
    nlist += g.w;
    g.w = nlist;
  }
  std::vector<uint32_t> glist(nlist);
  ranges([&](int, int64_t v0, int64_t v1) {
    std::vector<int32_t> fill(nv);  // next entry of the current row's block at each of its columns w >= v
    for (int64_t v = v0; v < v1; ++v) {
      fill[v] = gmeta[v].z;
      for (int32_t o = goff[v]; o < goff[v + 1]; ++o) fill[bcol[gmeta[nv + o].x]] = gmeta[nv + o].z;
      for (int32_t q = vptr[v]; q < vptr[v + 1]; ++q) {
        const int64_t e = vlist[q] >> 2;
        const int i = vlist[q] & 3;
        const int32_t* c = T + 4 * e;
        auto place = [&](int j) {  // of corner j in ascending vertex order
          int r = 0;
          for (int k = 0; k < 4; ++k) r += c[k] < c[j] || (c[k] == c[j] && k < j);
          return r;
        };
        for (int j = 0; j < 4; ++j) {
          if (c[j] < v) continue;
          const int pi = place(i), pj = place(j);
          glist[fill[c[j]]++] = (uint32_t)e << 5 | (uint32_t)kst_block(std::min(pi, pj), std::max(pi, pj)) << 1;
        }
      }
    }
  });
  // SELL-C-sigma layout: rows sorted by block count (descending, stable, so
  // rows of equal degree keep their spatial order), chunks of kSellC rows.
  std::vector<int32_t> order(nv);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    return bptr[a + 1] - bptr[a] > bptr[b + 1] - bptr[b];
  });
  const int64_t nchunk = (nv + kSellC - 1) / kSellC;
  std::vector<int32_t> sell_row(nchunk * kSellC, -1), chunk_deg(nchunk), chunk_off(nchunk + 1, 0);
  for (int64_t i = 0; i < nv; ++i) sell_row[i] = order[i];
  for (int64_t c = 0; c < nchunk; ++c) {
    int32_t d = 0;
    for (int i = 0; i < kSellC; ++i) {
      const int32_t r = sell_row[c * kSellC + i];
      if (r >= 0) d = std::max(d, bptr[r + 1] - bptr[r]);
    }
    chunk_deg[c] = d;
    SK_REQUIRE((int64_t)chunk_off[c] + (int64_t)kSellC * d < (int64_t(1) << 31) / 9, "sk_mesh_create: SELL too large");
    chunk_off[c + 1] = chunk_off[c] + kSellC * d;
  }
  const int64_t nslot = chunk_off[nchunk];
  // XCD-balanced chunk order (see sk_mesh::corder). Within an XCD's list the
  // runs are merged by relative position (the k-th of n chunks of a run's
  // share sorts at k / n): on a spatially ordered mesh, chunks of different
  // degree from the same region share columns, and now run at about the same
  // time on the same XCD, whose L2 then serves their common vector entries.
  std::vector<std::vector<int32_t>> xl(8);
  std::vector<std::vector<std::pair<double, int32_t>>> xk(8);
  for (int64_t c0 = 0; c0 < nchunk;) {
    int64_t c1 = c0;
    while (c1 < nchunk && chunk_deg[c1] == chunk_deg[c0]) ++c1;
    for (int j = 0; j < 8; ++j) {
      const int64_t a0 = c0 + (c1 - c0) * j / 8, a1 = c0 + (c1 - c0) * (j + 1) / 8;
      for (int64_t c = a0; c < a1; ++c) xk[j].emplace_back((double)(c - a0) / (double)(a1 - a0), (int32_t)c);
    }
    c0 = c1;
  }
  for (int j = 0; j < 8; ++j) {
    std::stable_sort(xk[j].begin(), xk[j].end(),
                     [](const std::pair<double, int32_t>& a, const std::pair<double, int32_t>& b) {
                       return a.first < b.first;
                     });
    for (const auto& e : xk[j]) xl[j].push_back(e.second);
  }
  size_t lmax = 1;
  for (auto& l : xl) lmax = std::max(lmax, l.size());
  const int64_t lpad = (int64_t)((lmax + 3) / 4 * 4);
  std::vector<int32_t> corder(8 * lpad, -1);
  for (int j = 0; j < 8; ++j) std::copy(xl[j].begin(), xl[j].end(), corder.begin() + j * lpad);
  std::vector<int4> cmeta(8 * lpad);
  for (size_t e = 0; e < cmeta.size(); ++e) {
    const int32_t c = corder[e];
    cmeta[e] = make_int4(c, chunk_deg[c >= 0 ? c : 0], chunk_off[c >= 0 ? c : 0], 0);
  }
  std::vector<int32_t> scol(nslot, 0), sell_pos(nblk);
  for (int64_t c = 0; c < nchunk; ++c)
    for (int i = 0; i < kSellC; ++i) {
      const int32_t r = sell_row[c * kSellC + i];
      for (int32_t s = 0; s < chunk_deg[c]; ++s) {
        const int32_t q = chunk_off[c] + s * kSellC + i;
        if (r >= 0 && s < bptr[r + 1] - bptr[r]) {
          scol[q] = bcol[bptr[r] + s];
          sell_pos[bptr[r] + s] = q;
        } else {
          scol[q] = r >= 0 ? r : 0;  // padding slot: value 0, any valid column
        }
      }
    }
  std::vector<int32_t> Tsoa(4 * nt);
  for (int64_t e = 0; e < nt; ++e)
    for (int k = 0; k < 4; ++k) Tsoa[k * nt + e] = T[4 * e + k];

  m->nv = nv;
  m->nt = nt;
  m->nblk = nblk;
  SK_TRY(m->T.upload(Tsoa));
  SK_TRY(m->bptr.upload(bptr));
  SK_TRY(m->bcol.upload(bcol));
  SK_TRY(m->brow.upload(brow));
  SK_TRY(m->emap.upload(emap));
  SK_TRY(m->gmeta.upload(gmeta));
  SK_TRY(m->glist.upload(glist));
  SK_TRY(m->vptr.upload(vptr));
  SK_TRY(m->vlist.upload(vlist));
  SK_TRY(m->sell_row.upload(sell_row));
  SK_TRY(m->chunk_deg.upload(chunk_deg));
  SK_TRY(m->chunk_off.upload(chunk_off));
  SK_TRY(m->scol.upload(scol));
  SK_TRY(m->sell_pos.upload(sell_pos));
  SK_TRY(m->corder.upload(corder));
  SK_TRY(m->cmeta.upload(cmeta));
  m->lpad = lpad;
  m->nchunk = nchunk;
  m->nslot = nslot;
  SK_TRY(m->D.alloc(12 * (size_t)nt));
  SK_TRY(m->Kst.alloc((size_t)kKst * nt));
  SK_TRY(m->fst.alloc((size_t)kFst * nt));
  SK_TRY(m->eflag.alloc((size_t)nt));
  SK_TRY(m->red.init());
  SK_HIP_CHECK(hipHostMalloc((void**)&m->pinned, 16 * sizeof(double), hipHostMallocDefault));
  m->h_bptr = std::move(bptr);
  m->h_bcol = std::move(bcol);
  return SK_OK;
}

void degree_order(const std::vector<int32_t>& deg, int32_t* order) {
  std::iota(order, order + deg.size(), 0);
  std::stable_sort(order, order + deg.size(), [&](int32_t a, int32_t b) { return deg[a] > deg[b]; });
}

void vertex_degrees(const int32_t* T, int64_t nv, int64_t nt, std::vector<int32_t>& deg) {
  std::vector<int32_t> vptr(nv + 1, 0), vlist(4 * nt);
  for (int64_t k = 0; k < 4 * nt; ++k) vptr[T[k] + 1]++;
  std::partial_sum(vptr.begin(), vptr.end(), vptr.begin());
  {
    std::vector<int32_t> fill(vptr.begin(), vptr.end() - 1);
    for (int64_t e = 0; e < nt; ++e)
      for (int i = 0; i < 4; ++i) vlist[fill[T[4 * e + i]]++] = (int32_t)e;
  }
  // each vertex's neighbours once: seen[w] is the last vertex that counted w
  std::vector<int32_t> seen(nv, -1);
  deg.resize(nv);
  for (int64_t v = 0; v < nv; ++v) {
    int32_t d = 1;
    seen[v] = (int32_t)v;
    for (int32_t k = vptr[v]; k < vptr[v + 1]; ++k) {
      const int32_t* c = T + 4 * (int64_t)vlist[k];
      for (int j = 0; j < 4; ++j)
        if (seen[c[j]] != v) {
          seen[c[j]] = (int32_t)v;
          ++d;
        }
    }
    deg[v] = d;
  }
}

}  // namespace sk

using namespace sk;

static hipStream_t as_stream(sk_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

extern "C" {

int sk_mesh_create(const int32_t* T_host, const double* D, int64_t nv, int64_t nt, sk_mesh** out) {
  SK_REQUIRE(out, "sk_mesh_create: null out");
  *out = nullptr;
  SK_REQUIRE(nv > 0 && nt > 0, "sk_mesh_create: empty mesh");
  SK_REQUIRE(T_host && D, "sk_mesh_create: null T or D");
  sk_mesh* m = nullptr;
  int s = no_throw([&] {
    m = new sk_mesh();
    return build_mesh(T_host, nv, nt, m);
  });
  if (s == SK_OK) {
    aos_to_soa_kernel<<<grid_for(nt), kBlock>>>(D, nt, m->D.p);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
      set_error(std::string("sk_mesh_create: ") + hipGetErrorString(e));
      s = SK_ERR_HIP;
    }
  }
  if (s != SK_OK) {
    sk_mesh_destroy(m);
    return s;
  }
  *out = m;
  return SK_OK;
}

int sk_sell_order(const int32_t* T, int64_t nv, int64_t nt, int32_t* order) {
  SK_REQUIRE(T && order, "sk_sell_order: null argument");
  SK_REQUIRE(nv > 0 && nt > 0, "sk_sell_order: empty mesh");
  for (int64_t k = 0; k < 4 * nt; ++k) SK_REQUIRE(T[k] >= 0 && T[k] < nv, "sk_sell_order: tet index out of range");
  return no_throw([&] {
    std::vector<int32_t> deg;
    vertex_degrees(T, nv, nt, deg);
    degree_order(deg, order);
    return (int)SK_OK;
  });
}

int sk_mesh_destroy(sk_mesh* m) {
  if (!m) return SK_OK;
  if (m->pinned) (void)hipHostFree(m->pinned);
  delete m;
  return SK_OK;
}

int sk_mesh_info(const sk_mesh* m, int64_t* nv, int64_t* nt, int64_t* nnz, int64_t* nblocks) {
  SK_REQUIRE(m, "sk_mesh_info: null mesh");
  if (nv) *nv = m->nv;
  if (nt) *nt = m->nt;
  if (nnz) *nnz = 9 * m->nblk;
  if (nblocks) *nblocks = m->nblk;
  return SK_OK;
}

int sk_mesh_csr_pattern(const sk_mesh* m, int32_t* indptr, int32_t* indices, sk_stream_t s) {
  SK_REQUIRE(m, "sk_mesh_csr_pattern: null mesh");
  const int64_t n = std::max<int64_t>(m->nv + 1, m->nblk);
  csr_pattern_kernel<<<grid_for(n), kBlock, 0, as_stream(s)>>>(m->nv, m->nblk, m->bptr.p, m->bcol.p, m->brow.p,
                                                                indptr, indices);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

int sk_mesh_element_nnz(const sk_mesh* m, int32_t* elem_nnz, sk_stream_t s) {
  SK_REQUIRE(m && elem_nnz, "sk_mesh_element_nnz: null argument");
  element_nnz_kernel<<<grid_for(m->nt), kBlock, 0, as_stream(s)>>>(m->nt, m->T.p, m->bptr.p, m->emap.p, elem_nnz);
  SK_HIP_CHECK(hipGetLastError());
  return SK_OK;
}

int sk_mesh_energy(sk_mesh* m, int material, const double* x, const double* F0, const double* mu,
                   const double* lam, const double* vol, double* energy_host, double* elem_energy, sk_stream_t s) {
  SK_REQUIRE(m && x && mu && vol, "sk_mesh_energy: null argument");
  SK_REQUIRE(!material_needs_lam(material) || lam, "sk_mesh_energy: this material needs lam");
  hipStream_t st = as_stream(s);
  SK_TRY(launch_elem_energy(m, material, x, F0, nullptr, 0.0, mu, lam, vol, elem_energy, nullptr, nullptr, nullptr,
                            nullptr, 0.0, st));
  if (energy_host) {
    SK_TRY(read_scalars(m, m->red.result.p, 1, st));
    *energy_host = m->pinned[0];
  }
  return SK_OK;
}

int sk_mesh_gradient(sk_mesh* m, int material, const double* x, const double* F0, const double* mu,
                     const double* lam, const double* vol, double* g, sk_stream_t s) {
  SK_REQUIRE(m && x && mu && vol && g, "sk_mesh_gradient: null argument");
  SK_REQUIRE(!material_needs_lam(material) || lam, "sk_mesh_gradient: this material needs lam");
  hipStream_t st = as_stream(s);
  SK_TRY(launch_elem_grad(m, material, x, F0, mu, lam, vol, st));
  SK_TRY(launch_gather_grad(m, g, nullptr, nullptr, nullptr, nullptr, nullptr, 0.0, st));
  return SK_OK;
}

int sk_mesh_hessian(sk_mesh* m, int material, const double* x, const double* F0, const double* mu,
                    const double* lam, const double* vol, int psd, double* values, sk_stream_t s) {
  SK_REQUIRE(m && x && mu && vol && values, "sk_mesh_hessian: null argument");
  SK_REQUIRE(!material_needs_lam(material) || lam, "sk_mesh_hessian: this material needs lam");
  hipStream_t st = as_stream(s);
  SK_TRY(launch_elem_hess(m, material, x, F0, mu, lam, vol, psd, false, st, nullptr, nullptr, nullptr, true));
  SK_TRY(launch_gather_hess(m, values, nullptr, 0.0, nullptr, nullptr, kLayoutCSR, false, st));
  return SK_OK;
}

}  // extern "C"
