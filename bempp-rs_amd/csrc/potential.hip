// potential.hip -- potential (off-surface) operators on triangle grids:
// P[j][i] = sum over cells and rule points q of K(x_j, y_q) psi_i(y_q) w_q J, K = G (single
// layer) or grad_y G . n_y (double layer).
//
// A workgroup takes 64 evaluation points (lane = point); its wavefronts walk cells with wave-uniform
// scalar loads. Where cells share DOFs it also owns kPotentialDofs consecutive DOFs, whose entries it
// alone writes: P1 entries are summed in LDS at [DOF][point] (lane = point, so the LDS adds of a
// wavefront never collide) and each is written once, 64 consecutive points a column. A cell at the
// border of two DOF blocks is evaluated for both (1.6 times where the cell order has locality, 2.5 in
// random order): cheaper than adding every cell's three entries to the output with global FP64 atomics, which
// ran at ~83 G/s and bounded the kernel, except for many evaluations or few workgroups. Without shared
// DOFs the entries are stored where they are computed, 64 consecutive points a column.
//
// The phase is taken relative to kR, R the distance of the point from the cell's centroid:
// |k (r - R)| <= |k| |y - c| for every point y of the cell wherever the evaluation point is, so the
// small-argument tiers hold by the cells' size alone and e^{ikR} is applied once per (point, cell).
//
// Bound by FP64 VALU issue (92 % busy). Helmholtz single layer, P1, 10007 points, 5120 cells, 6-point rule,
// complex128: 3.83 ms with the atomics and a full phase reduction per point pair, 0.69 ms so.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "core.hpp"
#include "kernels.hpp"

namespace bempp_amd {

#define HIP_CHECK_P(expr)                                                                         \
  do {                                                                                            \
    hipError_t _e = (expr);                                                                       \
    if (_e != hipSuccess) throw Error(std::string(#expr) + " failed: " + hipGetErrorString(_e)); \
  } while (0)

namespace dev {

struct PotentialArgs {
  const double* x;         // [np][3] evaluation points
  long long np;
  long long npblocks;      // blocks of 64 evaluation points
  const double* pts;       // [cells][Q][4]
  const double* geo;       // [cells][kGeoStride]
  const double* rule_tab;  // [nq][4] weight x basis values and weight of each rule point
  const double* vtx;       // the cells' vertex offsets and the rule in groups (PotentialInputs)
  const double* gq;
  const double* groups;
  int n21, ngroups;
  double wc, wc_trial;
  const int* off;          // DOF blocks (PotentialInputs); without blocks null
  const int* cells;
  const int* ldof;         // without blocks: the cells' DOFs
  int ncells;
  long long ndofs;
  int nq;
  double k;
  double wphi[kMaxQ][3];   // rule weight x basis value (a P0 space: {w, 0, 0})
  void* out;               // [np x ndofs] column-major
  int out_type;
  int mode;                // kStore or kAccumulate (one writer per entry), or kAtomic (cells once)
  int parts;               // workgroups the cells are split over (1 with blocks)
  long long first;         // first group (of a DOF block and a block of points) of the launch
};

// TIER (Helmholtz): 0 full argument reduction per point pair; 1, 2, 3: |k| t rad <= 0.5 / 0.25 /
// 1.5 for every cell, t the rule's largest point radius in a cell of radius 1. NB: DOFs per cell
// (1 or 3). BLOCKS: sums in LDS by DOF blocks; else a workgroup takes every cell in turn and adds or
// stores its entries. Q = 0: a rule of any point count (A.nq).
template <int Q, int OP, bool HELM, int TIER, int NB, bool BLOCKS>
__global__ void __launch_bounds__(1024) potential_kernel(const PotentialArgs A) {
  constexpr int NC = HELM ? 2 : 1;
  __shared__ double acc[BLOCKS ? NC : 1][BLOCKS ? kPotentialDofs : 1][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = blockIdx.x % A.parts;
  const long long group = A.first + blockIdx.x / A.parts;
  const long long block = group / A.npblocks;
  const long long t = (group - block * A.npblocks) * 64 + lane;
  const bool ok = t < A.np;
  const long long tl = ok ? t : A.np - 1;  // clamped: loads stay in bounds
  const double x[3] = {A.x[3 * tl], A.x[3 * tl + 1], A.x[3 * tl + 2]};
  if constexpr (BLOCKS) {
    for (int e = threadIdx.x; e < NC * kPotentialDofs * 64; e += blockDim.x) (&acc[0][0][0])[e] = 0.0;
    __syncthreads();
  }
  const auto pts = constant_view(A.pts);
  const auto geo = constant_view(A.geo);
  const auto tab = constant_view(A.rule_tab);
  const auto cells = constant_view(A.cells);
  const auto ldof = constant_view(A.ldof);
  const int e0 = BLOCKS ? constant_view(A.off)[block] : 0, e1 = BLOCKS ? constant_view(A.off)[block + 1] : A.ncells;
  const int nwaves = blockDim.x >> 6;
  const int nq = Q > 0 ? Q : A.nq;
  constexpr int kUnroll = Q > 0 ? Q : 4;
  for (int e = e0 + part * nwaves + wave; e < e1; e += nwaves * A.parts) {
    const int j = BLOCKS ? cells[e] : e;
    const auto sp = pts + (size_t)j * nq * 4;
    const auto sg = geo + (size_t)j * kGeoStride;
    const double ny[3] = {sg[9], sg[10], sg[11]};
    const double X[3] = {x[0] - sg[kGeoCentroid], x[1] - sg[kGeoCentroid + 1], x[2] - sg[kGeoCentroid + 2]};
    const double R2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
    const double kappa = HELM ? fabs(A.k) : 0.0;
    double kR = 0.0;
    cplx er = {sg[12], 0.0};  // the Jacobian, times e^{i kappa R} when centred
    if constexpr (TIER > 0) {
      // an evaluation point at the centroid is allowed (R = 0); below 1e-100 R is taken as 0
      kR = R2 > 1e-200 ? kappa * (R2 * rsqrt_nr(R2)) : 0.0;
      double s, c;
      sincos_cw(kR, &s, &c);
      er = {sg[12] * c, sg[12] * s};
    }
    cplx T[NB];
    // three radii away for the whole wavefront: r^2 from cell-relative terms (group_sum.hpp), which
    // lose at most a few bits there; nearer points take the difference of the coordinates
    if (__all(R2 >= 9.0 * sg[kGeoRadius] * sg[kGeoRadius])) {
      const auto sv = constant_view(A.vtx) + (size_t)j * 12;
      const double d[2][3] = {{sv[0], sv[1], sv[2]}, {sv[4], sv[5], sv[6]}}, g[3] = {sv[3], sv[7], sv[11]};
      const double none[3] = {0.0, 0.0, 0.0}, khalf = 0.5 * kappa;
      group_trial_sum<Q, OP, HELM, TIER, NB == 3>(A, X, 0.0, none, d, g, constant_view(A.gq) + (size_t)j * 3 * A.ngroups,
                                                  TIER > 0 ? khalf * khalf : 1.0, kR, khalf, T);
      double f = group_factor<OP, HELM, TIER>(kappa);
      if constexpr (OP == 1) f *= X[0] * ny[0] + X[1] * ny[1] + X[2] * ny[2];
      er = {er.re * f, er.im * f};
    } else {
#pragma unroll
      for (int b = 0; b < NB; ++b) T[b] = {0.0, 0.0};
#pragma unroll kUnroll
      for (int q = 0; q < nq; ++q) {
        const double d[3] = {x[0] - sp[4 * q], x[1] - sp[4 * q + 1], x[2] - sp[4 * q + 2]};
        const cplx kv = kernel_scalar<OP, HELM, TIER>(d[0], d[1], d[2], kappa, ny, ny, kR);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const double f = Q > 0 ? A.wphi[q < kMaxQ ? q : 0][b] : tab[4 * q + (NB == 1 ? 3 : b)];
          T[b].re = fma(kv.re, f, T[b].re);
          if constexpr (HELM) T[b].im = fma(kv.im, f, T[b].im);
        }
      }
    }
    er = {er.re * kInv4Pi, er.im * kInv4Pi};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int l = ldof[(size_t)e * NB + b];  // without blocks: the DOF itself
      if (BLOCKS && l < 0) continue;           // wave-uniform: a DOF of another block
      cplx v = {T[b].re * er.re, T[b].im * er.re};
      if constexpr (TIER > 0) v = cmul(T[b], er);
      if (HELM && A.k < 0.0) v.im = -v.im;  // e^{-i kappa r} is the conjugate
      if constexpr (BLOCKS) {
        atomicAdd(&acc[0][l][lane], v.re);
        if constexpr (HELM) atomicAdd(&acc[NC - 1][l][lane], v.im);
      } else if (ok) {
        store_value(A.out, t + A.np * l, v, A.out_type, A.mode);
      }
    }
  }
  if constexpr (BLOCKS) {
    __syncthreads();
    if (!ok) return;
    for (int l = wave; l < kPotentialDofs; l += nwaves) {
      const long long col = block * kPotentialDofs + l;
      if (col >= A.ndofs) break;
      store_value(A.out, t + A.np * col, {acc[0][l][lane], HELM ? acc[NC - 1][l][lane] : 0.0}, A.out_type, A.mode);
    }
  }
}

}  // namespace dev

namespace {

template <int Q, int OP, bool HELM, int TIER>
void launch_nb(int nb, dim3 grid, hipStream_t s, const dev::PotentialArgs& P) {
  if (!P.off) {
    if (nb == 1) dev::potential_kernel<Q, OP, HELM, TIER, 1, false><<<grid, 256, 0, s>>>(P);
    else dev::potential_kernel<Q, OP, HELM, TIER, 3, false><<<grid, 256, 0, s>>>(P);
    return;
  }
  // wavefronts a workgroup splits its cells over: 4 once that fills the card eight waves a SIMD
  // deep (8192 in all), up to 16 for fewer workgroups, which would otherwise leave it idle
  const unsigned threads = grid.x >= 2048 ? 256 : grid.x >= 1024 ? 512 : 1024;
  dev::potential_kernel<Q, OP, HELM, TIER, 3, true><<<grid, threads, 0, s>>>(P);
}

template <int Q, int OP>
void launch_tier(bool helm, int tier, int nb, dim3 grid, hipStream_t s, const dev::PotentialArgs& P) {
  if (!helm) launch_nb<Q, OP, false, 0>(nb, grid, s, P);
  else if (tier == 2) launch_nb<Q, OP, true, 2>(nb, grid, s, P);
  else if (tier == 1) launch_nb<Q, OP, true, 1>(nb, grid, s, P);
  else if (tier == 3) launch_nb<Q, OP, true, 3>(nb, grid, s, P);
  else launch_nb<Q, OP, true, 0>(nb, grid, s, P);
}

template <int OP>
void launch_potential(int Q, bool helm, int tier, int nb, dim3 grid, hipStream_t s, const dev::PotentialArgs& P) {
  switch (Q) {
    case 1: launch_tier<1, OP>(helm, tier, nb, grid, s, P); break;
    case 3: launch_tier<3, OP>(helm, tier, nb, grid, s, P); break;
    case 6: launch_tier<6, OP>(helm, tier, nb, grid, s, P); break;
    case 7: launch_tier<7, OP>(helm, tier, nb, grid, s, P); break;
    default: launch_tier<0, OP>(helm, tier, nb, grid, s, P); break;  // point count at run time
  }
}

}  // namespace

void assemble_potential_device(const Assembler& a, const FunctionSpace& space, const double* dev_points,
                               int64_t npoints, void* dev_out, bool accumulate, void* stream) {
  require_triangles(space, "potential assembly");
  if (a.op != kSL && a.op != kDL) throw Error("potential operators exist for the single and double layer only");
  if ((a.kind == kLaplace) == is_complex(a.dtype)) throw Error("dtype does not match the kernel");
  if (npoints < 0) throw Error("negative point count");
  if (npoints == 0) return;
  if (!dev_points || !dev_out) throw Error("points or output pointer is null");
  const PotentialInputs in = potential_inputs(a, space, npoints, stream);
  const bool shared_dofs = space.size < (int64_t)space.nb * space.grid->nc();
  if (in.ndofs == 0) return;
  std::vector<double> xi, w;
  triangle_rule(in.Q, xi, w);
  dev::PotentialArgs P{};
  P.x = dev_points;
  P.np = npoints;
  P.npblocks = (npoints + 63) / 64;
  P.pts = in.pts;
  P.geo = in.geo;
  P.rule_tab = in.rule_tab;
  P.vtx = in.vtx;
  P.gq = in.gq;
  P.groups = in.groups;
  P.n21 = in.n21;
  P.ngroups = in.ngroups;
  P.wc = in.wc;
  P.wc_trial = in.wc_trial;
  P.off = in.off;
  P.cells = in.cells;
  P.ldof = in.ldof;
  P.ndofs = in.ndofs;
  P.nq = in.Q;
  P.k = a.k;
  for (int p = 0; p < std::min(in.Q, dev::kMaxQ); ++p) {
    const double phi[3] = {1.0 - xi[2 * p] - xi[2 * p + 1], xi[2 * p], xi[2 * p + 1]};
    for (int b = 0; b < 3; ++b) P.wphi[p][b] = in.nb == 3 ? w[p] * phi[b] : (b == 0 ? w[p] : 0.0);
  }
  P.out = dev_out;
  P.out_type = in.out_type;
  P.mode = accumulate ? dev::kAccumulate : dev::kStore;
  hipStream_t s = (hipStream_t)stream;
  P.ncells = in.ncells;
  long long groups = P.npblocks;
  if (in.off) {
    groups *= in.nblocks;
    P.parts = 1;
  } else {
    // the cells split over as many workgroups as give 8192 in all, at least a cell a wavefront; P0
    // Helmholtz single layer, 5000 points, 20480 cells, 2048 / 4096 / 8192 / 16384: 1010 / 877 / 844 / 843 us,
    // Laplace, 3000 points, 5120 cells: 58.7 / 58.3 / 51.4 / 55.4
    P.parts = (int)std::clamp<long long>(8192 / groups, 1, (in.ncells + 3) / 4);
    if (shared_dofs) {
      P.mode = dev::kAtomic;
      if (!accumulate) {
        // a fill kernel, not a memset node: the caller may capture this stream in a graph
        const long long n = (long long)npoints * in.ndofs * (is_complex(a.dtype) ? 2 : 1);
        if (a.dtype == kF32 || a.dtype == kC32) dev::fill_zero_kernel<<<256, 256, 0, s>>>((float*)dev_out, n);
        else dev::fill_zero_kernel<<<256, 256, 0, s>>>((double*)dev_out, n);
        HIP_CHECK_P(hipGetLastError());
      }
    }
  }
  const bool helm = a.kind == kHelmholtz;
  // |k (r - R)| <= |k| t rad (with a margin for the rounding of r and R)
  const double bound = std::fabs(a.k) * in.rule_radius * in.max_radius * (1.0 + 1e-12);
  const int tier = !helm || !dev::scalable(a.k, in.max_radius) ? 0 : bound <= 0.25 ? 2 : bound <= 0.5 ? 1 : bound <= 1.5 ? 3 : 0;
  in_launches(groups, [&](long long first, unsigned n) {
    P.first = first;
    const dim3 g(n * P.parts);  // (parts > 1 only where that gives at most 8192)
    if (a.op == kSL) launch_potential<0>(in.Q, helm, tier, in.nb, g, s, P);
    else launch_potential<1>(in.Q, helm, tier, in.nb, g, s, P);
  });
  HIP_CHECK_P(hipGetLastError());
}

}  // namespace bempp_amd
