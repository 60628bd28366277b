// HIP kernels of libgdx for gfx950 (MI355X).
//
// The numeric assembly of a Lagrangian Q_K Poisson operator on a Cartesian
// mesh is done "owner computes rows": every workgroup owns a tile of owned
// rows (free dofs) of one part and computes their complete rows -- including
// the contributions of cells that belong to neighbouring parts -- with the
// tensor-product structure of the mesh, the basis and the Gauss rule:
//
//   A_ij = sum_q kappa(x_q) * [ G1 M2 M3 + M1 G2 M3 + M1 M2 G3 ](q; i,j)
//   G_d(q; i_d,j_d) = w_q dphi_a(q) dphi_b(q) / h_d
//   M_d(q; i_d,j_d) = w_q h_d  phi_a(q)  phi_b(q)
//
// which is exactly sum over cells c containing i and j of the cell matrix
// entry int_c kappa grad(phi_i).grad(phi_j) for the affine Cartesian map
// (J = diag(h), detJ = h1 h2 h3, J^{-T} grad = grad_ref / h).  The three
// contractions over x-, y- and z-quadrature points are done one dimension at
// a time (sum factorisation), so each stored value costs O(1) FMAs.  Every row is
// written once, contiguously, through a position pattern (stencil slot <-> offset
// within the CSR row): no float atomics, bit-for-bit repeatable.  The
// SubAssembledRows owner/ghost exchange is folded in: owned rows receive the
// neighbouring parts' contributions at the source, ghost rows stay zero.
// The matrix kernels are in gdx_lattice.hip (the default), gdx_march3d.hip and
// gdx_tile3d.hip; this file has the coefficients at the quadrature points and the
// numeric phase's launchers.
#include <hip/hip_runtime.h>

#include <new>
#include <vector>

#include "gdx_device.h"

namespace gdx {

// ---------------------------------------------------------------------------
// Coefficient and source at every quadrature point of the global lattice.
// a_m exp(i theta_m) = [a_m exp(i phi_m) exp(2 pi i k_m1 x)] exp(2 pi i k_m2 y) exp(2 pi i k_m3 z)
// with the three 1D factors tabulated once per launch.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void fourier_table(const double *__restrict__ modes, const KParams &kp, int qnmax,
                                              double *__restrict__ E, int m, int d, int first, int step) {
  const double *M = modes + 5 * m;
  for (int q = first; q < qnmax; q += step) {
    double x = 0.0;
    if (d < kp.dim && q < kp.qn[d]) {
      const int c = q / kp.NQ, t = q % kp.NQ;
      x = kp.x0[d] + kp.h[d] * ((double)c + kp.qx[t]);
    }
    double s, co;
    sincos(2.0 * M_PI * M[d] * x, &s, &co);
    if (d == 0) {  // fold the amplitude and phase into the x factor
      double ps, pc;
      sincos(M[4], &ps, &pc);
      const double cr = M[3] * pc, ci = M[3] * ps;
      const double r = cr * co - ci * s, i = cr * s + ci * co;
      co = r;
      s = i;
    }
    double *e = E + 2 * (((size_t)d * kp.nmodes + m) * qnmax + q);
    e[0] = co;
    e[1] = s;
  }
}

__global__ void k_fourier_tables(const double *__restrict__ modes, KParams kp, int qnmax, double *__restrict__ E) {
  fourier_table(modes, kp, qnmax, E, blockIdx.y, blockIdx.z, threadIdx.x + blockIdx.x * blockDim.x,
                blockDim.x * gridDim.x);
}

// One block = LINES consecutive x-lines (q2 .. q2+LINES-1 at fixed q3) of the
// quadrature lattice; thread <-> q1.  The x factors of a chunk of modes stay
// in registers across the lines; the per-line (y,z) products b = e2 e3 and
// (k.c) b are tabulated in LDS, so each (point, mode) costs four FMAs:
//   g += Re(e1 b),  s += Im(e1 (k.c) b).
//
// A wave reads two (four) of the tabulated doubles from LDS for every two (four)
// FMAs, and four SIMDs share that LDS port: the reads bound it (7.1 M points, 16
// modes, both sums: 48 us, at 128 B per clock and CU the reads alone 46).  So a
// problem whose source is constant makes the first sum only and stores no f
// where no kernel reads one (SOURCE = false), and up to 8 modes go in a chunk of
// 8: 32 Q1 cubes of 16..48 cells with 8 modes 97 -> 43 us.
constexpr int kCoefLines = 8;

template <bool SOURCE, int MODES>
__device__ __forceinline__ void coefficient_lines(const double *__restrict__ modes, const double *__restrict__ E,
                                                  const KParams &kp, int qnmax, double *__restrict__ W,
                                                  double *__restrict__ F, int bx, int by, int q3) {
  __shared__ double tb[kCoefLines][MODES][SOURCE ? 4 : 2];  // br, bi, (k.c) br, (k.c) bi
  const int q1 = bx * blockDim.x + threadIdx.x;
  const int q2b = by * kCoefLines;
  const bool active = q1 < kp.qn[0];
  const int nm = kp.nmodes;
  double g[kCoefLines], s[kCoefLines];
#pragma unroll
  for (int l = 0; l < kCoefLines; ++l) g[l] = s[l] = 0.0;
  for (int m0 = 0; m0 < nm; m0 += MODES) {
    __syncthreads();
    for (int i = threadIdx.x; i < kCoefLines * MODES; i += blockDim.x) {
      const int l = i / MODES, j = i % MODES, m = m0 + j;
      const int q2 = q2b + l < kp.qn[1] ? q2b + l : kp.qn[1] - 1;
      double br = 0.0, bi = 0.0, kc = 0.0;
      if (m < nm) {
        const double *M = modes + 5 * m;
        const double *e2 = E + 2 * ((size_t)(1 * nm + m) * qnmax + q2);
        const double *e3 = E + 2 * ((size_t)(2 * nm + m) * qnmax + q3);
        br = e2[0] * e3[0] - e2[1] * e3[1];
        bi = e2[0] * e3[1] + e2[1] * e3[0];
        kc = M[0] * kp.dir_coef[1] + M[1] * kp.dir_coef[2] + M[2] * kp.dir_coef[3];
      }
      tb[l][j][0] = br;
      tb[l][j][1] = bi;
      if constexpr (SOURCE) {
        tb[l][j][2] = kc * br;
        tb[l][j][3] = kc * bi;
      }
    }
    __syncthreads();
    double e1r[MODES], e1i[MODES];
#pragma unroll
    for (int j = 0; j < MODES; ++j) {
      const bool ok = active && m0 + j < nm;
      const double *e1 = E + 2 * ((size_t)(ok ? m0 + j : 0) * qnmax + (active ? q1 : 0));
      e1r[j] = ok ? e1[0] : 0.0;
      e1i[j] = ok ? e1[1] : 0.0;
    }
#pragma unroll
    for (int l = 0; l < kCoefLines; ++l) {
#pragma unroll
      for (int j = 0; j < MODES; ++j) {
        g[l] = fma(e1r[j], tb[l][j][0], fma(-e1i[j], tb[l][j][1], g[l]));
        if constexpr (SOURCE) s[l] = fma(e1r[j], tb[l][j][3], fma(e1i[j], tb[l][j][2], s[l]));
      }
    }
  }
  if (!active) return;
#pragma unroll
  for (int l = 0; l < kCoefLines; ++l) {
    const int q2 = q2b + l;
    if (q2 >= kp.qn[1]) break;
    const double kap = kp.coef_const * exp(g[l]);
    const size_t idx = q1 + (size_t)kp.qn[0] * (q2 + (size_t)kp.qn[1] * q3);
    W[idx] = kap;
    // f = -div(kappa grad uD) = -kappa grad(g).c = kappa 2 pi sum_m (k_m.c) a_m sin(theta_m)
    if (F) F[idx] = SOURCE && kp.rhs_kind == GDX_RHS_MANUFACTURED ? kap * 2.0 * M_PI * s[l] : kp.rhs_const;
  }
}

template <bool SOURCE, int MODES>
__global__ __launch_bounds__(256) void k_coefficients(const double *__restrict__ modes,
                                                      const double *__restrict__ E, KParams kp, int qnmax,
                                                      double *__restrict__ W, double *__restrict__ F) {
  coefficient_lines<SOURCE, MODES>(modes, E, kp, qnmax, W, F, blockIdx.x, blockIdx.y, blockIdx.z);
}

// The same for many problems at once: a block finds its problem and its place
// in that problem's grid in a table.
struct CoefProblem {
  KParams kp;
  const double *modes;
  double *E, *W, *F;
  int qnmax;
};
// one wave per block: small problems' lines are 32..96 points, a larger block
// would leave most of its lanes idle
struct CoefBlock {
  int prob, x, y, z;
};

__global__ __launch_bounds__(256) void k_fourier_tables_batch(const CoefProblem *__restrict__ probs,
                                                              const CoefBlock *__restrict__ blocks) {
  const CoefBlock b = blocks[blockIdx.x];
  const CoefProblem &p = probs[b.prob];
  fourier_table(p.modes, p.kp, p.qnmax, p.E, b.y, b.z, threadIdx.x, blockDim.x);
}

template <bool SOURCE, int MODES>  // what the problem that needs most needs
__global__ __launch_bounds__(64) void k_coefficients_batch(const CoefProblem *__restrict__ probs,
                                                           const CoefBlock *__restrict__ blocks) {
  const CoefBlock b = blocks[blockIdx.x];
  const CoefProblem &p = probs[b.prob];
  coefficient_lines<SOURCE, MODES>(p.modes, p.E, p.kp, p.qnmax, p.W, p.F, b.x, b.y, b.z);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int longest_line(const KParams &kp) {
  int qnmax = kp.qn[0];
  for (int d = 1; d < 3; ++d) qnmax = qnmax > kp.qn[d] ? qnmax : kp.qn[d];
  return qnmax;
}

bool points_used(const gdx_problem *p) { return !lattice_used(p) || (!p->coef_cell && p->kp.nmodes > 0); }

// f at the quadrature points, where a kernel reads it: the pair-lattice kernel
// takes a constant f in closed form
static double *source_array(const gdx_problem *p) {
  return lattice_used(p) && p->kp.rhs_kind != GDX_RHS_MANUFACTURED ? nullptr : p->dev.F;
}

int launch_coefficients(gdx_problem *p, hipStream_t st) {
  // the pair-lattice kernel takes a coefficient that is constant on every cell as it is
  if (!points_used(p)) return GDX_OK;
  if (p->coef_cell) return launch_cell_coefficients(p, st);
  const KParams &kp = p->kp;
  const int qnmax = longest_line(kp);
  if (kp.nmodes > 0) {
    dim3 g1((qnmax + 255) / 256, kp.nmodes, 3);
    hipLaunchKernelGGL(k_fourier_tables, g1, dim3(256), 0, st, p->dev.modes, kp, qnmax, p->dev.E);
  }
  const int bx = kp.qn[0] < 256 ? 64 * ((kp.qn[0] + 63) / 64) : 256;
  dim3 g2((kp.qn[0] + bx - 1) / bx, (kp.qn[1] + kCoefLines - 1) / kCoefLines, kp.qn[2]);
  const bool source = kp.rhs_kind == GDX_RHS_MANUFACTURED, few = kp.nmodes <= 8;
  const auto kernel = source ? (few ? k_coefficients<true, 8> : k_coefficients<true, 16>)
                             : (few ? k_coefficients<false, 8> : k_coefficients<false, 16>);
  hipLaunchKernelGGL(kernel, g2, dim3(bx), 0, st, p->dev.modes, p->dev.E, kp, qnmax, p->dev.W, source_array(p));
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

// Coefficients of many problems in two launches.  Alone each problem's pair of
// launches fills a few CUs and ends in a gap: 32 Q1 cubes of 16..48 cells took
// 32 x (4 + 10) us of kernels.
struct CoefBatch {
  CoefProblem *probs = nullptr;
  CoefBlock *tables = nullptr, *lines = nullptr;
  unsigned ntables = 0, nlines = 0;
  bool source = false, few = true;
};

void coef_batch_free(CoefBatch *b) {
  if (!b) return;
  void *ptrs[] = {b->probs, b->tables, b->lines};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  delete b;
}

int coef_batch_build(const std::vector<gdx_problem *> &ps, CoefBatch **out) {
  *out = nullptr;
  std::vector<CoefProblem> probs;
  std::vector<CoefBlock> tables, lines;
  for (gdx_problem *p : ps) {
    const KParams &kp = p->kp;
    const int i = (int)probs.size();
    probs.push_back({kp, p->dev.modes, p->dev.E, p->dev.W, source_array(p), longest_line(kp)});
    for (int d = 0; d < 3; ++d)
      for (int m = 0; m < kp.nmodes; ++m) tables.push_back({i, 0, m, d});
    for (int z = 0; z < kp.qn[2]; ++z)
      for (int y = 0; y < (kp.qn[1] + kCoefLines - 1) / kCoefLines; ++y)
        for (int x = 0; x < (kp.qn[0] + 63) / 64; ++x) lines.push_back({i, x, y, z});
  }
  CoefBatch *b = new (std::nothrow) CoefBatch;
  if (!b) return GDX_ERR_ALLOC;
  auto put = [](auto **dst, const auto &src) {
    const size_t n = src.size() * sizeof(src[0]);
    return hipMalloc(reinterpret_cast<void **>(dst), n ? n : 1) == hipSuccess &&
           (!n || hipMemcpy(*dst, src.data(), n, hipMemcpyHostToDevice) == hipSuccess);
  };
  if (!put(&b->probs, probs) || !put(&b->tables, tables) || !put(&b->lines, lines)) {
    coef_batch_free(b);
    return GDX_ERR_ALLOC;
  }
  b->ntables = (unsigned)tables.size();
  b->nlines = (unsigned)lines.size();
  for (gdx_problem *p : ps) {
    b->source |= p->kp.rhs_kind == GDX_RHS_MANUFACTURED;
    b->few &= p->kp.nmodes <= 8;
  }
  *out = b;
  return GDX_OK;
}

int coef_batch_launch(const CoefBatch *b, hipStream_t st) {
  if (b->ntables) hipLaunchKernelGGL(k_fourier_tables_batch, dim3(b->ntables), dim3(256), 0, st, b->probs, b->tables);
  const auto lines = b->source ? (b->few ? k_coefficients_batch<true, 8> : k_coefficients_batch<true, 16>)
                               : (b->few ? k_coefficients_batch<false, 8> : k_coefficients_batch<false, 16>);
  if (b->nlines) hipLaunchKernelGGL(lines, dim3(b->nlines), dim3(64), 0, st, b->probs, b->lines);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

int launch_matrix3d(gdx_problem *p, hipStream_t st, int precision);

bool matrix_kernel_supported(int dim, int K, int NQ) {
  if (dim == 3) return (K == 2 && (NQ == 2 || NQ == 3)) || (K == 1 && NQ == 2);
  return dim == 2 && (K == 1 || K == 2) && (NQ == 2 || NQ == 3);
}

int launch_source(gdx_problem *p, hipStream_t st);

// the pair-lattice kernel takes a constant f in closed form, and the other
// kernels but the per-tile one write b themselves
bool source_used(const gdx_problem *p) {
  const bool varies = p->ngdofs > 0 && p->kp.rhs_kind == GDX_RHS_MANUFACTURED && p->kp.nmodes > 0 && !p->coef_cell;
  return lattice_used(p) ? varies : p->kvariant3d == 1;
}

int launch_rhs(gdx_problem *p, hipStream_t st) { return source_used(p) ? launch_source(p, st) : GDX_OK; }

int launch_matrix(gdx_problem *p, hipStream_t st) {
  if (lattice_used(p)) return launch_lattice(p, st);  // either precision: its contractions are FP64
  if (p->tiles.empty()) return GDX_OK;
  if (p->kvariant3d == 0) return launch_matrix3d(p, st, p->precision);
  if (p->kvariant3d == 3) return launch_matrix_tile3d_wslab(p, st);
  return launch_matrix_tile3d(p, st);
}

}  // namespace gdx
