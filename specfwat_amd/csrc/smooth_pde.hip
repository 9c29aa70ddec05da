// PDE (explicit diffusion) kernel smoothing on the device.
//
// Drop-in for smooth_pde_cuda_ (src/postproc/smooth_sem_pde.cu:298-479,
// called from smooth_sem_pde, src/postproc/smooth.f90:392-402) with the same
// 42 by-reference arguments.  One diffusion step is
//   ddat = - sum_e  W (hprimewgll^T) [ J c(grad dat) ]      (element pass, scatter-add)
//   dat += rvol * ddat ;  ddat = 0                          (one streaming pass)
//   dat(PML points) = dat_bak                               (only when PML elements exist)
// for ntstep steps.  Geometry per element follows the reference: irregular
// elements read their nine inverse-Jacobian terms, regular elements use
// xix_regular; faithful mode (the default, as the reference's CUDA and CPU
// paths) puts xix_regular in all nine slots, the alternative uses the
// diagonal map of an axis-aligned cube.
//
// Differences in mechanism (not in result): the reference scatters with
// atomics into ddat, launches 4-5 kernels per diffusion step (memset, two
// phase launches, apply_mass, keep_pml) and exchanges halos over MPI; here
// the element pass finishes the points that belong to one element only and
// writes element-local terms of the others, one gather launch per step sums
// those per point in element order (the reference CPU loop's order, no
// atomics, run-to-run reproducible) fused with dat += rvol * ddat, the
// element phases are merged (single GPU), and up to 24 fields share one
// geometry read with the fields innermost in HBM ([nglob][fields]).
#include "sem_device.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

namespace {

constexpr int SM_TPB = 256;
constexpr int SM_NFMAX = 24;  // fields per device run (a larger batch runs in chunks)

inline unsigned sm_blocks(size_t n) { return (unsigned)((n + SM_TPB - 1) / SM_TPB); }

struct SmoothArgs {
  const int* ibool;       // 0-based [nspec][125]
  const int* irregular;   // [nspec]
  const realw* jinv9;     // [9][nirr][125], as the caller's nine arrays
  size_t jstride;         // nirr * 125
  const realw* jac;       // [nspec][125]  (jacobian_all)
  const realw* rot;       // [nspec][3][125] when spherical
  const realw* tables;    // hprimeT[25] hprimewgll[25] wgllwgll_yz[25] _xz[25] _xy[25]
  const realw* rvol;      // [nglob]
  realw* dat;             // [nglob][NFP]
  realw* dloc;            // [nspec][125][NFP] element-local -(weak-form stiffness term), rows by sem_floc_slot
  int nspec, nfield;
  int n_shared;           // points from here on belong to one element
  int nblocks_padded;
  realw cv, ch, xix_regular;
  realw cxh, cxv;         // ch and cv times xix_regular^2
  int is_sph;
  int faithful;
};

// Rows of NFP values per point in pieces of 16 bytes when NFP is a multiple of 4, else of 4 bytes.
template <int W>
struct SmoothPiece {
  using T = realw;
  __device__ static __forceinline__ T zero() { return 0.0f; }
  __device__ static __forceinline__ T fma_s(T x, realw h, T y) { return fmaf(x, h, y); }
  __device__ static __forceinline__ T mul_s(T x, realw h) { return x * h; }
};
template <>
struct SmoothPiece<4> {
  using T = float4;
  __device__ static __forceinline__ T zero() { return make_float4(0.0f, 0.0f, 0.0f, 0.0f); }
  __device__ static __forceinline__ T fma_s(T x, realw h, T y) {
    return make_float4(fmaf(x.x, h, y.x), fmaf(x.y, h, y.y), fmaf(x.z, h, y.z), fmaf(x.w, h, y.w));
  }
  __device__ static __forceinline__ T mul_s(T x, realw h) { return make_float4(x.x * h, x.y * h, x.z * h, x.w * h); }
};
template <int NFP>
struct SmoothRow {
  static constexpr int W = NFP % 4 == 0 ? 4 : 1, C = NFP / W;  // values per piece, pieces per row
};

// Element pass: one element per 128-lane workgroup.  The rows of the element's points go to LDS
// by consecutive lanes taking consecutive pieces of a row (a wave's access then covers eleven
// 96-byte rows whole at 24 fields; a lane per row touches 64 rows in 16-byte pieces), the fields
// are then processed a piece (four fields) at a time between two barriers, geometry read once for
// all, and the element-local terms leave LDS the same way, into rows in the order of sem_floc_slot.
//   * Points of one element only (numbered last, [n_shared, nglob)) have no other term: their
//     diffusion step dat += rvol * term is taken here and nothing of them is stored (27 of an
//     element's 125 rows), in place, since no other element reads them.
//   * REG: axis-aligned cubes with the diagonal map, whose fluxes are one factor per direction.
// LDS holds the pieces as they are: gfx950 reads 16 bytes a lane at twice the rate of 4
// (5.7e7 LDS cycles a launch with one value per lane and read, 4.4e7 with pieces).  Rows of 1 to 3 values
// are moved by the lane of their point, which needs no second trip through LDS.
// 32x32x16 cubes, 21 fields: 119 us a step with a lane per row, one field between two barriers and
// every row stored, 118 us with a third of the gather's work done here (the gather 94 -> 46 us);
// of the cycles of busy compute units LDS works in 71 %, a fifth of them conflicts, VALU in 62 %.
template <int NFP, bool REG>
__global__ __launch_bounds__(128) void k_smooth_elem(SmoothArgs A) {
  constexpr int W = SmoothRow<NFP>::W, C = SmoothRow<NFP>::C;
  using P = SmoothPiece<W>;
  using T = typename P::T;
  constexpr int SU = 131;  // pieces c and c + 1 of a point 12 banks apart, where rows go in and out
  __shared__ realw s_tab[128];
  __shared__ int s_g[125];
  __shared__ uint8_t s_row[125];  // local point of each row
  __shared__ T s_u[C * SU];       // piece c of local point p at c * SU + p
  constexpr int NB = C <= 2 ? 2 : 1;  // two halves of the fluxes in turn save a barrier a piece; with
                                      // more pieces their LDS costs waves (six: 120 -> 135 us)
  __shared__ T s_t[NB][3][128];
  const int t = threadIdx.x;
  const int e = xcd_remap(blockIdx.x, A.nblocks_padded);
  if (e >= A.nspec) return;  // block-uniform
  const int tt = min(t, 124);
  const int I = tt % 5, J = (tt / 5) % 5, K = tt / 25;
  const size_t L0 = (size_t)e * 125, Lg = L0 + tt;
  if (t < 125) {
    s_tab[t] = A.tables[t];
    if constexpr (W == 4) {
      s_g[t] = A.ibool[Lg];
      s_row[sem_floc_slot(t)] = (uint8_t)t;
    }
  }
  // geometry, requested with the points
  const realw jl = A.jac[Lg];
  realw g[REG ? 1 : 3][3], r[3] = {0.0f, 0.0f, 1.0f};
  if constexpr (!REG) {
    const int ir = A.irregular[e];
    if (ir) {
      const realw* Gm = A.jinv9 + (size_t)(ir - 1) * 125 + tt;
#pragma unroll
      for (int q = 0; q < 9; ++q) g[q / 3][q % 3] = Gm[q * A.jstride];
    } else {
#pragma unroll
      for (int q = 0; q < 9; ++q) g[q / 3][q % 3] = A.faithful || q % 4 == 0 ? A.xix_regular : 0.0f;
    }
    if (A.is_sph)
#pragma unroll
      for (int c = 0; c < 3; ++c) r[c] = A.rot[(size_t)e * 375 + 125 * c + tt];
  }
  T* dat = reinterpret_cast<T*>(A.dat);
  const int own = A.ibool[Lg];
  if constexpr (W == 1) {
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (t < 125) s_u[c * SU + t] = dat[(size_t)own * C + c];
  }
  __syncthreads();
  if constexpr (W == 4)
    for (int q = t; q < 125 * C; q += 128) {
      const int p = q / C, c = q - p * C;
      s_u[c * SU + p] = dat[(size_t)s_g[p] * C + c];
    }
  // mxm_opt{x,y,z} of the reference: u(l,J,K) * hprimeT[I*5+l], etc.; the quadrature factor and
  // the sign are folded into the second tables
  realw hpI[5], hpJ[5], hpK[5], hwI[5], hwJ[5], hwK[5];
  {
    const realw fac1 = -s_tab[50 + K * 5 + J], fac2 = -s_tab[75 + K * 5 + I], fac3 = -s_tab[100 + J * 5 + I];
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      hpI[l] = s_tab[I * 5 + l];
      hpJ[l] = s_tab[J * 5 + l];
      hpK[l] = s_tab[K * 5 + l];
      hwI[l] = s_tab[25 + I * 5 + l] * fac1;
      hwJ[l] = s_tab[25 + J * 5 + l] * fac2;
      hwK[l] = s_tab[25 + K * 5 + l] * fac3;
    }
  }
  // The fluxes are f_a = sum_b M[a][b] t_b with M = J (ch g_a . g_b + (cv - ch) (g_a . r)(g_b . r)),
  // g_a the gradient of reference coordinate a and r the vertical (z, or rot when spherical)
  realw M[3][3] = {};
  if constexpr (REG) {
    M[0][0] = M[1][1] = A.cxh * jl;
    M[2][2] = A.cxv * jl;
  } else {
    const realw cv = A.cv, ch = A.ch;
    realw v[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) v[a] = r[0] * g[a][0] + r[1] * g[a][1] + r[2] * g[a][2];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b)
        M[a][b] = jl * (ch * (g[a][0] * g[b][0] + g[a][1] * g[b][1] + g[a][2] * g[b][2]) + (cv - ch) * v[a] * v[b]);
  }
  const int La0 = 5 * J + 25 * K, Lb0 = I + 25 * K, Lc0 = I + 5 * J;
  if constexpr (W == 4) __syncthreads();
  T* dloc = reinterpret_cast<T*>(A.dloc);
#pragma unroll 1
  for (int c = 0; c < C; ++c) {
    T* U = s_u + c * SU;
    T t1 = P::zero(), t2 = P::zero(), t3 = P::zero();
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      t1 = P::fma_s(U[La0 + l], hpI[l], t1);
      t2 = P::fma_s(U[Lb0 + 5 * l], hpJ[l], t2);
      t3 = P::fma_s(U[Lc0 + 25 * l], hpK[l], t3);
    }
    auto& S = s_t[NB == 2 ? c & 1 : 0];
    if constexpr (REG) {
      S[0][t] = P::mul_s(t1, M[0][0]);
      S[1][t] = P::mul_s(t2, M[1][1]);
      S[2][t] = P::mul_s(t3, M[2][2]);
    } else {
#pragma unroll
      for (int a = 0; a < 3; ++a)
        S[a][t] = P::fma_s(t3, M[a][2], P::fma_s(t2, M[a][1], P::mul_s(t1, M[a][0])));
    }
    __syncthreads();  // fluxes complete; every lane is done reading this piece of s_u
    T d = P::zero();
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      d = P::fma_s(S[0][La0 + l], hwI[l], d);
      d = P::fma_s(S[1][Lb0 + 5 * l], hwJ[l], d);
      d = P::fma_s(S[2][Lc0 + 25 * l], hwK[l], d);
    }
    if constexpr (W == 1) {
      if (t < 125) {
        if (own >= A.n_shared) dat[(size_t)own * C + c] = P::fma_s(d, A.rvol[own], U[t]);
        else dloc[(L0 + sem_floc_slot(t)) * C + c] = d;
      }
    } else if (t < 125) {
      U[t] = d;  // own slot only
    }
    if (NB == 1 && c + 1 < C) __syncthreads();  // the fluxes are read
  }
  if constexpr (W == 1) return;
  __syncthreads();  // the terms are in s_u
  for (int q = t; q < 125 * C; q += 128) {
    const int row = q / C, c = q - row * C;
    const int p = s_row[row], ig = s_g[p];
    const T v = s_u[c * SU + p];
    if (ig >= A.n_shared) {
      T* D = dat + (size_t)ig * C + c;
      *D = P::fma_s(v, A.rvol[ig], *D);
    } else {
      dloc[(L0 + row) * C + c] = v;
    }
  }
}

// ddat(g) = sum of the element-local terms of g in element order (the reference CPU loop's
// accumulation order); dat += rvol * ddat, for the points of more than one element.  One lane per
// piece of a point's row, so consecutive lanes read and write whole rows (32x32x16 cubes, 21
// fields: 94 us a step with a lane per row over all points, 45 now; one field 11 us with a row at
// a time, 8 in groups; bound by the rows' traffic, and for few fields by the chain offset, index, row).
template <int NFP>
__global__ void k_smooth_gather(int npts, const int* __restrict__ off, const int* __restrict__ idx,
                                const realw* __restrict__ dloc, const realw* __restrict__ rvol,
                                realw* __restrict__ dat) {
  constexpr int W = SmoothRow<NFP>::W, C = SmoothRow<NFP>::C;
  const size_t h = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= (size_t)npts * C) return;
  const int g = (int)(h / C), c = (int)(h - (size_t)g * C);
  const int k1 = off[g + 1];
  int k = off[g];
  const realw r = rvol[g];
  using P = SmoothPiece<W>;
  using T = typename P::T;
  const T* rows = reinterpret_cast<const T*>(dloc) + c;
  T* D = reinterpret_cast<T*>(dat) + h;
  const T v = *D;
  T d = P::zero();
  // four, two and one rows at a time, all of a group requested before the first is added
  auto add = [&](auto n) {
    constexpr int M = decltype(n)::value;
    T a[M];
#pragma unroll
    for (int m = 0; m < M; ++m) a[m] = rows[(size_t)idx[k + m] * C];
#pragma unroll
    for (int m = 0; m < M; ++m) d = P::fma_s(a[m], 1.0f, d);
    k += M;
  };
  while (k + 3 < k1) add(std::integral_constant<int, 4>());
  if (k + 1 < k1) add(std::integral_constant<int, 2>());
  if (k < k1) add(std::integral_constant<int, 1>());
  *D = P::fma_s(d, r, v);
}

// pin PML points: dat(iglob) = dat_bak(local), in element/point order
__global__ void k_keep_pml(int npml, int nfield, int nfp, const int* __restrict__ pml_iglob,
                           const realw* __restrict__ pml_val, realw* __restrict__ dat) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npml) return;
  for (int f = 0; f < nfield; ++f) dat[(size_t)pml_iglob[q] * nfp + f] = pml_val[(size_t)f * npml + q];
}

// [nfield][nglob] <-> [nglob][nfp], the rows in library numbering; a lane per point, so that the
// caller's side is contiguous over the lanes
__global__ void k_to_point_major(int nglob, int nfield, int nfp, const int* __restrict__ perm,
                                 const realw* __restrict__ a, realw* __restrict__ b) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nglob) return;
  realw* B = b + (size_t)perm[g] * nfp;
  for (int f = 0; f < nfp; ++f) B[f] = f < nfield ? a[(size_t)f * nglob + g] : 0.0f;
}

__global__ void k_to_field_major(int nglob, int nfield, int nfp, const int* __restrict__ perm,
                                 const realw* __restrict__ b, realw* __restrict__ a) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nglob) return;
  const realw* B = b + (size_t)perm[g] * nfp;
  for (int f = 0; f < nfield; ++f) a[(size_t)f * nglob + g] = B[f];
}

int g_smooth_faithful = 1;

// fields per point row in HBM: 1-3 as they are (rows of 4, 8 or 12 bytes),
// more padded to a multiple of 4 for 16-byte vector access
int padded_fields(int nf) { return nf <= 3 ? nf : ((nf + 3) / 4) * 4; }

struct SmoothPlan {
  int nspec = 0, nglob = 0, nirr = 0, npml = 0, nfield = 0, nfp = 1;
  int n_shared = 0;         // points of more than one element come first, in the caller's order
  int* d_perm = nullptr;    // caller's point -> library point
  int* d_ibool = nullptr;
  int* d_irr = nullptr;
  realw* d_jinv9 = nullptr;
  realw* d_jac = nullptr;
  realw* d_rot = nullptr;
  realw* d_tables = nullptr;
  realw* d_rvol = nullptr;
  int* d_off = nullptr;     // CSR point -> local points, element order
  int* d_idx = nullptr;
  realw* d_dat = nullptr;   // [nglob][nfp]
  realw* d_dloc = nullptr;  // [nloc][nfp]
  realw* d_io = nullptr;    // [nfield][nglob] staging of the caller's layout
  int* d_pml_iglob = nullptr;
  realw* d_pml_val = nullptr;
  hipStream_t stream = nullptr;
  double elem_ms = 0, update_ms = 0;
};

void plan_free(SmoothPlan& p) {
  dev_free(p.d_ibool); dev_free(p.d_irr); dev_free(p.d_jinv9); dev_free(p.d_jac); dev_free(p.d_rot);
  dev_free(p.d_tables); dev_free(p.d_rvol); dev_free(p.d_off); dev_free(p.d_idx); dev_free(p.d_dat);
  dev_free(p.d_dloc); dev_free(p.d_io); dev_free(p.d_pml_iglob); dev_free(p.d_pml_val); dev_free(p.d_perm);
  if (p.stream) HIP_CHECK(hipStreamDestroy(p.stream));
  p = SmoothPlan();
}

// elem_ms / update_ms of a timed run: the element and gather launches of every
// stride-th step (at most about 256 steps) timed by their dispatch timestamps,
// scaled to all nstep steps
template <int NFP, bool REG>
void launch_steps(SmoothPlan& p, const SmoothArgs& a, int nstep, bool timed) {
  const int stride = std::max(1, nstep / 256), nsamp = (nstep + stride - 1) / stride;
  std::vector<hipEvent_t> ev;
  if (timed) {
    ev.resize(4 * (size_t)nsamp);
    for (auto& x : ev) HIP_CHECK(hipEventCreate(&x));
  }
  for (int it = 0; it < nstep; ++it) {
    const bool tm = timed && it % stride == 0;
    const size_t q = 4 * (size_t)(it / stride);
    if (tm) sem_arm_launch_events(ev[q], ev[q + 1]);
    SEM_LAUNCH((k_smooth_elem<NFP, REG>), dim3(a.nblocks_padded), dim3(128), 0, p.stream, a);
    if (tm) sem_arm_launch_events(ev[q + 2], ev[q + 3]);
    SEM_LAUNCH(k_smooth_gather<NFP>, dim3(std::max(1u, sm_blocks((size_t)p.n_shared * SmoothRow<NFP>::C))), dim3(SM_TPB),
               0, p.stream, p.n_shared, p.d_off, p.d_idx, p.d_dloc, p.d_rvol, p.d_dat);
    if (p.npml > 0)
      hipLaunchKernelGGL(k_keep_pml, dim3((p.npml + SM_TPB - 1) / SM_TPB), dim3(SM_TPB), 0, p.stream, p.npml,
                         p.nfield, p.nfp, p.d_pml_iglob, p.d_pml_val, p.d_dat);
  }
  HIP_CHECK(hipGetLastError());
  if (timed) {
    HIP_CHECK(hipStreamSynchronize(p.stream));
    double e = 0.0, u = 0.0;
    for (int k = 0; k < nsamp; ++k) {
      float a1 = 0, a2 = 0;
      HIP_CHECK(hipEventElapsedTime(&a1, ev[4 * (size_t)k], ev[4 * (size_t)k + 1]));
      HIP_CHECK(hipEventElapsedTime(&a2, ev[4 * (size_t)k + 2], ev[4 * (size_t)k + 3]));
      e += a1;
      u += a2;
    }
    p.elem_ms += e * nstep / nsamp;
    p.update_ms += u * nstep / nsamp;
    for (auto x : ev) HIP_CHECK(hipEventDestroy(x));
  }
}

template <bool REG>
void launch_fields(SmoothPlan& p, const SmoothArgs& a, int nstep, bool timed) {
  switch (p.nfp) {
    case 1: launch_steps<1, REG>(p, a, nstep, timed); break;
    case 2: launch_steps<2, REG>(p, a, nstep, timed); break;
    case 3: launch_steps<3, REG>(p, a, nstep, timed); break;
    case 4: launch_steps<4, REG>(p, a, nstep, timed); break;
    case 8: launch_steps<8, REG>(p, a, nstep, timed); break;
    case 12: launch_steps<12, REG>(p, a, nstep, timed); break;
    case 16: launch_steps<16, REG>(p, a, nstep, timed); break;
    case 20: launch_steps<20, REG>(p, a, nstep, timed); break;
    case 24: launch_steps<24, REG>(p, a, nstep, timed); break;
    default: SEM_FAIL("smooth: %d padded fields not supported", p.nfp);
  }
}

void run_steps(SmoothPlan& p, int nstep, realw cv, realw ch, realw xix_regular, int is_sph, bool timed) {
  SmoothArgs a{};
  a.ibool = p.d_ibool; a.irregular = p.d_irr; a.jinv9 = p.d_jinv9; a.jstride = (size_t)p.nirr * 125; a.jac = p.d_jac; a.rot = p.d_rot;
  a.tables = p.d_tables; a.rvol = p.d_rvol; a.dat = p.d_dat; a.dloc = p.d_dloc;
  a.n_shared = p.n_shared;
  a.cxh = (realw)((double)ch * xix_regular * xix_regular);
  a.cxv = (realw)((double)cv * xix_regular * xix_regular);
  a.nspec = p.nspec; a.nfield = p.nfield;
  a.nblocks_padded = xcd_pad(p.nspec);
  a.cv = cv; a.ch = ch; a.xix_regular = xix_regular; a.is_sph = is_sph; a.faithful = g_smooth_faithful;
  p.elem_ms = p.update_ms = 0;
  // cubes with the diagonal map everywhere: one flux factor per direction (faithful mode and
  // irregular or spherical meshes need the whole map)
  if (p.nirr == 0 && !g_smooth_faithful && !is_sph) launch_fields<true>(p, a, nstep, timed);
  else launch_fields<false>(p, a, nstep, timed);
}

// Build the device plan from the reference's host arrays.
void plan_build(SmoothPlan& p, int nspec, int nglob, int nirr, int is_sph, const realw* const* jin,
                const realw* jaco, const realw* rotate0, const realw* wxy, const realw* wxz,
                const realw* wyz, const realw* hprimeT, const realw* hprime_wgll, const int* ibool,
                const int* is_CPML, const int* irregular, const realw* rvol, int nfield) {
  if (nfield < 1 || nfield > SM_NFMAX) SEM_FAIL("smooth: %d fields per run (1..%d)", nfield, SM_NFMAX);
  HIP_CHECK(hipStreamCreateWithFlags(&p.stream, hipStreamNonBlocking));
  hipStream_t s = p.stream;
  p.nspec = nspec; p.nglob = nglob; p.nirr = nirr; p.nfield = nfield; p.nfp = padded_fields(nfield);
  const size_t nloc = (size_t)nspec * 125;
  if (nloc >= (size_t)INT32_MAX) SEM_FAIL("smooth: too many local points for 32-bit CSR indices");
  std::vector<int> ib(nloc), touch(nglob, 0);
  for (size_t L = 0; L < nloc; ++L) {
    int g = ibool[L] - 1;
    if (g < 0 || g >= nglob) SEM_FAIL("smooth_pde: ibool(%zu)=%d outside 1..%d", L, g + 1, nglob);
    ib[L] = g;
    ++touch[g];
  }
  // library numbering: points of more than one element first, in the caller's order, then the
  // others element by element; CSR shared point -> element rows in element order, by their place
  // in the rows, in the same pass over the elements
  std::vector<int> perm(nglob, -1);
  {
    std::vector<int> off(1, 0);
    off.reserve(nglob + 1);
    for (int g = 0; g < nglob; ++g)
      if (touch[g] != 1) {
        perm[g] = (int)off.size() - 1;
        off.push_back(off.back() + touch[g]);
      }
    p.n_shared = (int)off.size() - 1;
    int slot[125], n = p.n_shared;
    for (int L = 0; L < 125; ++L) slot[L] = sem_floc_slot(L);
    std::vector<int> fill(off.begin(), off.end() - 1), idx((size_t)off[p.n_shared]);
    for (int e = 0; e < nspec; ++e)
      for (int L = 0; L < 125; ++L) {
        int& g = ib[(size_t)e * 125 + L];
        if (touch[g] == 1) perm[g] = n++;
        else idx[fill[perm[g]]++] = e * 125 + slot[L];
        g = perm[g];
      }
    p.d_perm = dev_upload(perm.data(), perm.size(), s);
    p.d_ibool = dev_upload(ib.data(), nloc, s);
    p.d_off = dev_upload(off.data(), off.size(), s);
    p.d_idx = dev_upload(idx.data(), idx.size(), s);
    HIP_CHECK(hipStreamSynchronize(s));
  }
  std::vector<int> irr(irregular, irregular + nspec);
  for (int e = 0; e < nspec; ++e)
    if (irr[e] < 0 || irr[e] > nirr) SEM_FAIL("smooth_pde: irregular_element_number(%d)=%d outside 0..%d", e + 1, irr[e], nirr);
  p.d_irr = dev_upload(irr.data(), (size_t)nspec, s);
  if (nirr > 0) {
    const size_t nj = (size_t)nirr * 125;
    p.d_jinv9 = dev_alloc<realw>(9 * nj);
    for (int c = 0; c < 9; ++c)
      HIP_CHECK(hipMemcpyAsync(p.d_jinv9 + c * nj, jin[c], nj * sizeof(realw), hipMemcpyHostToDevice, s));
  }
  p.d_jac = dev_upload(jaco, nloc, s);
  if (is_sph) {
    // rotate_r(NDIM,NGLLX,NGLLY,NGLLZ,NSPEC) -> [nspec][3][125]
    std::vector<realw> r(nloc * 3);
    for (size_t e = 0; e < (size_t)nspec; ++e)
      for (int c = 0; c < 3; ++c)
        for (int L = 0; L < 125; ++L) r[(e * 3 + c) * 125 + L] = rotate0[((e * 125) + L) * 3 + c];
    p.d_rot = dev_upload(r.data(), r.size(), s);
  }
  realw tab[125];
  for (int q = 0; q < 25; ++q) {
    tab[q] = hprimeT[q];
    tab[25 + q] = hprime_wgll[q];
    tab[50 + q] = wyz[q];
    tab[75 + q] = wxz[q];
    tab[100 + q] = wxy[q];
  }
  p.d_tables = dev_upload(tab, 125, s);
  std::vector<realw> rv(nglob);
  for (int g = 0; g < nglob; ++g) rv[perm[g]] = rvol[g];
  p.d_rvol = dev_upload(rv.data(), (size_t)nglob, s);
  p.d_dat = dev_alloc<realw>((size_t)nglob * p.nfp);
  p.d_dloc = dev_alloc<realw>(nloc * p.nfp);
  p.d_io = dev_alloc<realw>((size_t)nglob * nfield);
  // PML points in element order (last writer of a shared point wins, as the
  // reference's sequential CPU loop)
  std::vector<int> piglob;  // in the caller's point order, as smooth_pde_cuda_ lists the values
  if (is_CPML) {
    std::vector<int> last(nglob, -1);
    for (int e = 0; e < nspec; ++e)
      if (is_CPML[e])
        for (int L = 0; L < 125; ++L) last[ib[(size_t)e * 125 + L]] = e * 125 + L;
    for (int g = 0; g < nglob; ++g)
      if (last[perm[g]] >= 0) piglob.push_back(perm[g]);
  }
  p.npml = (int)piglob.size();
  if (p.npml) {
    p.d_pml_iglob = dev_upload(piglob.data(), piglob.size(), s);
    std::vector<realw> zero((size_t)nfield * p.npml, 0.0f);
    p.d_pml_val = dev_upload(zero.data(), zero.size(), s);
  }
  HIP_CHECK(hipStreamSynchronize(s));
}

// caller layout (NGLOB_AB, nfield) <-> device layout [nglob][nfp]
void upload_fields(SmoothPlan& p, const realw* dat_glob) {
  const size_t n = (size_t)p.nglob * p.nfield;
  HIP_CHECK(hipMemcpyAsync(p.d_io, dat_glob, n * sizeof(realw), hipMemcpyHostToDevice, p.stream));
  hipLaunchKernelGGL(k_to_point_major, dim3(sm_blocks((size_t)p.nglob)), dim3(SM_TPB), 0, p.stream, p.nglob, p.nfield,
                     p.nfp, p.d_perm, p.d_io, p.d_dat);
  HIP_CHECK(hipGetLastError());
}

void download_fields(SmoothPlan& p, realw* dat_glob) {
  const size_t n = (size_t)p.nglob * p.nfield;
  hipLaunchKernelGGL(k_to_field_major, dim3(sm_blocks((size_t)p.nglob)), dim3(SM_TPB), 0, p.stream, p.nglob, p.nfield,
                     p.nfp, p.d_perm, p.d_dat, p.d_io);
  HIP_CHECK(hipGetLastError());
  sem_to_host(dat_glob, p.d_io, n * sizeof(realw), p.stream);
}

double g_last_elem_ms = 0.0, g_last_update_ms = 0.0;

}  // namespace

extern "C" {

// smooth_sem_pde.cu:298-316 signature.  dat_bak is the ZERO_PML pinned value
// (all zero in the reference, smooth.f90:21,184-188).
void smooth_pde_cuda_(int* h_is_sph, int* h_nspec, int* h_nglob, int* nprocs, int* h_nstep,
                      int* nspec_max, int* phase_ispec_inner_elastic, int* h_nspec_outer,
                      int* h_nspec_inner, const realw* xix, const realw* xiy, const realw* xiz,
                      const realw* etax, const realw* etay, const realw* etaz, const realw* gamx,
                      const realw* gamy, const realw* gamz, const realw* jaco, const realw* rotate0,
                      const realw* wgllwgll_xy, const realw* wgllwgll_xz, const realw* wgllwgll_yz,
                      const realw* hprimeT, const realw* hprime_wgll, const int* ibool,
                      const int* is_CPML, const realw* h_cv, const realw* h_ch, int* h_num_intfs,
                      int* h_max_nibool, const int* my_neighbors, const int* nibool_intf,
                      const int* ibool_intf, const realw* dat_bak, realw* dat, const realw* rvol,
                      realw* dat_glob, realw* ddat_glob, const int* irregular_element_number,
                      const realw* h_xix_regular, const int* h_nspec_irregular) {
  (void)nspec_max; (void)phase_ispec_inner_elastic; (void)h_num_intfs; (void)h_max_nibool;
  (void)my_neighbors; (void)nibool_intf; (void)ibool_intf; (void)ddat_glob;
  if (*nprocs != 1)
    SEM_FAIL("smooth_pde_cuda_: multi-rank halo assembly is not part of this single-GPU build (nprocs=%d)", *nprocs);
  if (*h_nspec_outer + *h_nspec_inner != *h_nspec)
    SEM_FAIL("smooth_pde_cuda_: phases do not cover all elements");
  const int nspec = *h_nspec, nglob = *h_nglob;
  const realw* jin[9] = {xix, xiy, xiz, etax, etay, etaz, gamx, gamy, gamz};
  SmoothPlan p;
  plan_build(p, nspec, nglob, *h_nspec_irregular, *h_is_sph, jin, jaco, rotate0, wgllwgll_xy,
             wgllwgll_xz, wgllwgll_yz, hprimeT, hprime_wgll, ibool, is_CPML,
             irregular_element_number, rvol, 1);
  if (p.npml) {
    // pinned values from dat_bak at the last-writer local point
    std::vector<int> last(nglob, -1);
    for (int e = 0; e < nspec; ++e)
      if (is_CPML[e])
        for (int L = 0; L < 125; ++L) last[ibool[(size_t)e * 125 + L] - 1] = e * 125 + L;
    std::vector<realw> v;
    for (int g = 0; g < nglob; ++g)
      if (last[g] >= 0) v.push_back(dat_bak[last[g]]);
    HIP_CHECK(hipMemcpyAsync(p.d_pml_val, v.data(), v.size() * sizeof(realw), hipMemcpyHostToDevice, p.stream));
  }
  upload_fields(p, dat_glob);
  run_steps(p, *h_nstep, *h_cv, *h_ch, *h_xix_regular, *h_is_sph, false);
  download_fields(p, dat_glob);
  for (size_t L = 0; L < (size_t)nspec * 125; ++L) dat[L] = dat_glob[ibool[L] - 1];
  plan_free(p);
}

// 1 = reference arithmetic on regular elements (xix_regular in all nine
// inverse-Jacobian slots, smooth_sem_pde.cu:161-171), 0 = diagonal map.
void fwat_smooth_set_faithful_(int* faithful) { g_smooth_faithful = *faithful != 0; }

// Several fields smoothed together, sharing one geometry read per element:
// dat_glob (NGLOB_AB, nfield) in/out, already projected and rvol-scaled as
// smooth_sem_pde does before calling smooth_pde_cuda_.  No PML, Cartesian or
// spherical.  timed = 1 records the element-pass time (fwat_smooth_last_time_).
void fwat_smooth_pde_batch_(int* h_is_sph, int* h_nspec, int* h_nglob, int* h_nstep, int* h_nfield,
                            const realw* xix, const realw* xiy, const realw* xiz, const realw* etax,
                            const realw* etay, const realw* etaz, const realw* gamx, const realw* gamy,
                            const realw* gamz, const realw* jaco, const realw* rotate0,
                            const realw* wgllwgll_xy, const realw* wgllwgll_xz, const realw* wgllwgll_yz,
                            const realw* hprimeT, const realw* hprime_wgll, const int* ibool,
                            const realw* h_cv, const realw* h_ch, const realw* rvol, realw* dat_glob,
                            const int* irregular_element_number, const realw* h_xix_regular,
                            const int* h_nspec_irregular, int* timed) {
  const int nspec = *h_nspec, nglob = *h_nglob, nf = *h_nfield;
  if (nf <= 0) SEM_FAIL("fwat_smooth_pde_batch_: nfield must be positive");
  const realw* jin[9] = {xix, xiy, xiz, etax, etay, etaz, gamx, gamy, gamz};
  g_last_elem_ms = g_last_update_ms = 0;
  for (int f0 = 0; f0 < nf; f0 += SM_NFMAX) {  // chunks of at most SM_NFMAX fields
    const int nc = std::min(SM_NFMAX, nf - f0);
    SmoothPlan p;
    plan_build(p, nspec, nglob, *h_nspec_irregular, *h_is_sph, jin, jaco, rotate0, wgllwgll_xy,
               wgllwgll_xz, wgllwgll_yz, hprimeT, hprime_wgll, ibool, nullptr,
               irregular_element_number, rvol, nc);
    realw* chunk = dat_glob + (size_t)f0 * nglob;
    upload_fields(p, chunk);
    HIP_CHECK(hipStreamSynchronize(p.stream));
    run_steps(p, *h_nstep, *h_cv, *h_ch, *h_xix_regular, *h_is_sph, *timed != 0);
    download_fields(p, chunk);
    g_last_elem_ms += p.elem_ms;
    g_last_update_ms += p.update_ms;
    plan_free(p);
  }
}

void fwat_smooth_last_time_(double* elem_ms, double* update_ms) {
  *elem_ms = g_last_elem_ms;
  *update_ms = g_last_update_ms;
}

}  // extern "C"
