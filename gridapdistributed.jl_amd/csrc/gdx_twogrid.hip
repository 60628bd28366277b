// Learned two-grid preconditioner of libgdx for 3D Q1 problems on a cube of
// 2n x 2n x 2n cells with Dirichlet data on the whole boundary:
//
//   z  = w D^-1 r                          damped Jacobi pre-smoothing
//   rc = R (r - A z)                       full weighting (R = P^T, trilinear P)
//   ec = s N( D^-1 rc / s, log-diagonal )  network coarse solve, s = rms(D^-1 rc)
//   ec += w Dc^-1 (rc - Ac ec), k times     damped-Jacobi sweeps on the Galerkin
//                                          coarse operator Ac = P^T A P (27-point
//                                          stencil computed from the fine matrix)
//   z += a P ec, a = (P ec).s / (P ec).A(P ec) with s = r - A z: the
//                                          energy-optimal step along the correction
//   z += w D^-1 (r - A z)                  damped Jacobi post-smoothing (A z from
//                                          the two products above: no third SpMV)
//
// The coarse unknowns are the fine nodes with even indices; the (n-1)^3
// interior ones sit on the network's n^3 grid (the last plane is zero
// padding).  The network is trained on device from the problem's own matrix:
// a smooth random coarse error ec (white noise smoothed by repeated 3x3x3
// means), r = A P ec, target ec for the input built from r exactly as above
// (loss 1 - cos^2(N, ec): the preconditioner rescales the network's output to
// the coarse energy optimum, so only its direction matters).  Every reduction
// has a fixed order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "gdx_nn.h"

// Staging of r and z for gdx_nn_apply_noalloc: one file-scope array per GPU
// (each device that loads the library holds its own copy until the process
// ends).  Host code never passes the array's name to a kernel or a copy: it
// uses the per-device address that noalloc_setup obtains.
static constexpr size_t kNoAllocDoubles = (size_t)4 << 20;  // 32 MiB: r and z of up to 2,097,152 dofs
static __device__ __align__(256) double scratch[kNoAllocDoubles];

namespace gdx {

namespace {

constexpr int kB = 256;
constexpr int kRed = 256;  // partial sums per reduction
constexpr int kS = 3 * kRed;  // scalar slots of 'red' after three partial-sum areas
constexpr double kOmega = 2.0 / 3.0;
constexpr double kOmegaC = 2.0 / 3.0;  // coarse sweeps

// A structured coarse level: m cells per direction, unknowns at the interior
// nodes 1..m-1 stored at [0, m-1) of an m^3 array (the last plane is padding).
struct Level {
  int m = 0;
  double *cst = nullptr;  // Galerkin operator as a 27-point stencil [27][m^3]
  bool own_cst = true;    // false for the network grid (its stencil is TwoGrid::cst)
  double *rhs = nullptr, *e = nullptr, *e2 = nullptr;  // [m^3]
};

struct TwoGrid {
  gdx_problem *prob = nullptr;
  int n = 0;       // network grid = coarse cells per direction
  int nf = 0;      // fine lattice extent per direction (2n + 1)
  int ng = 0;      // free dofs
  long long *gid_node = nullptr;
  double *flat = nullptr, *dlat = nullptr;   // fine lattice vectors
  double *t1 = nullptr, *t2 = nullptr, *t3 = nullptr;  // global-id temporaries
  double *rho = nullptr;                     // coarse scaled residual [n^3]
  double *red = nullptr;                     // reduction partials + scalars
  double *ec = nullptr, *ec2 = nullptr;      // training: coarse error [n^3]
  float *tgt = nullptr;
  const double *dinv = nullptr;
  int *asym = nullptr;     // 1: fst is not symmetric to the bit
  double *lat = nullptr;   // lattice vectors of the flexible CG: x r z p q t1 t2 t3 dinv, nf^3 each
  double *fst = nullptr;   // fine matrix as a 27-point stencil on the lattice [27][nf^3]
  double *cst = nullptr;   // Galerkin coarse operator P^T A P as a stencil [27][n^3]
  double *rc = nullptr;    // coarse residual R s [n^3]
  double *ca = nullptr, *cb = nullptr;  // coarse correction (ping-pong) [n^3]
  int sweeps = 8;          // coarse damped-Jacobi sweeps after the network (two-grid form)
  bool use_net = true;     // false: the coarse correction starts from zero
  // multigrid form: a V-cycle from the network grid down to a grid of <= 8^3
  // cells replaces the coarse sweeps; lv[0] is the network grid
  bool mg = true;
  int nu = 1;              // damped-Jacobi sweeps before and after each coarse-grid correction
  int coarsest_sweeps = 24;
  std::vector<Level> lv;
};

TwoGrid *tg_of(gdx_nn *nn) { return reinterpret_cast<TwoGrid *>(nn->tg); }
inline unsigned nb(int64_t n) { return (unsigned)((n + kB - 1) / kB); }

__global__ void k_scatter(int ng, const long long *__restrict__ gn, const double *__restrict__ x, double *__restrict__ lat) {
  const int g = blockIdx.x * kB + threadIdx.x;
  if (g < ng) lat[gn[g]] = x[g];
}
__global__ void k_gather(int ng, const long long *__restrict__ gn, const double *__restrict__ lat, double *__restrict__ x) {
  const int g = blockIdx.x * kB + threadIdx.x;
  if (g < ng) x[g] = lat[gn[g]];
}

// rho[j] = dlat(2I) * sum_{|o|<=1} w(o) r(2I + o), I = j + 1, for interior coarse nodes; 0 on the padding plane
__global__ void k_restrict(int n, int nf, const double *__restrict__ flat, const double *__restrict__ dlat,
                           double *__restrict__ rho, double *__restrict__ rcoarse, double w,
                           const double *__restrict__ cst, double *__restrict__ e) {
  const unsigned tot = (unsigned)n * n * n, j = blockIdx.x * kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % n), jy = (int)(j / n % n), jz = (int)(j / ((unsigned)n * n));
  if (jx == n - 1 || jy == n - 1 || jz == n - 1) {
    rho[j] = 0.0;
    rcoarse[j] = 0.0;
    if (e) e[j] = 0.0;
    return;
  }
  const int fx = 2 * (jx + 1), fy = 2 * (jy + 1), fz = 2 * (jz + 1);
  double acc = 0.0;
  for (int oz = -1; oz <= 1; ++oz)
    for (int oy = -1; oy <= 1; ++oy)
      for (int ox = -1; ox <= 1; ++ox) {
        const double w = (ox ? 0.5 : 1.0) * (oy ? 0.5 : 1.0) * (oz ? 0.5 : 1.0);
        acc = fma(w, flat[(fx + ox) + (int64_t)nf * ((fy + oy) + (int64_t)nf * (fz + oz))], acc);
      }
  rcoarse[j] = acc;
  if (e) e[j] = w * acc / cst[(size_t)13 * tot + j];  // the V-cycle's first damped-Jacobi sweep from zero
  rho[j] = acc * dlat[fx + (int64_t)nf * (fy + (int64_t)nf * fz)];
}

// fine matrix rows -> 27-point stencil on the lattice: fst[slot][node], slot of
// the column's offset (dx+1) + 3(dy+1) + 9(dz+1); Dirichlet columns are absent
// from the free x free matrix and stay zero (fst is cleared before).
//
// kFsRows consecutive rows per block.  When their entries are stored back to
// back, the block reads them coalesced (one entry per thread, its row found by
// bisection over the block's row starts), places each value in an LDS tile
// [slot][row] and then writes the tile plane by plane, so consecutive lanes
// store consecutive lattice nodes.  Other blocks walk their rows one thread
// each.  The slot comes from the node difference: b - a + (1 + nf + nf^2) has
// base-nf digits (dx+1, dy+1, dz+1) in 0..2, found by comparisons.
constexpr int kFsRows = 64;
__device__ __forceinline__ int stencil_slot(long long d, int nf) {
  const long long nf2 = (long long)nf * nf;
  long long t = d + 1 + nf + nf2;
  if (t < 0 || t >= 3 * nf2) return -1;
  const int dz1 = t >= 2 * nf2 ? 2 : (t >= nf2 ? 1 : 0);
  t -= dz1 * nf2;
  const int dy1 = t >= 2 * (long long)nf ? 2 : (t >= nf ? 1 : 0);
  t -= (long long)dy1 * nf;
  return t > 2 ? -1 : (int)t + 3 * dy1 + 9 * dz1;
}
__global__ __launch_bounds__(kB) void k_fine_stencil(int ng, int nf, const long long *__restrict__ rstart,
                                                     const int *__restrict__ rlen, const int *__restrict__ cgid,
                                                     const double *__restrict__ val,
                                                     const long long *__restrict__ gn, double *__restrict__ fst) {
  constexpr int CAP = 27 * kFsRows;
  __shared__ double tile[27][kFsRows];
  __shared__ long long rs[kFsRows], an[kFsRows];
  __shared__ int rl[kFsRows];
  __shared__ unsigned int present[kFsRows];
  const int t = threadIdx.x, g0 = blockIdx.x * kFsRows;
  const int nr = min(kFsRows, ng - g0);
  if (nr <= 0) return;  // uniform over the block
  const int64_t nfl = (int64_t)nf * nf * nf;
  if (t < nr) {
    rs[t] = rstart[g0 + t];
    rl[t] = rlen[g0 + t];
    an[t] = gn[g0 + t];
    present[t] = 0u;
  }
  __syncthreads();
  int ok = 1;
  if (t < nr - 1) ok = rs[t] + rl[t] == rstart[g0 + t + 1];
  const long long A = rs[0], B = rs[nr - 1] + rl[nr - 1];
  ok = __syncthreads_and(ok && (B - A) <= CAP);
  if (!ok) {
    if (t < nr) {
      const long long a = an[t], s0 = rs[t];
      for (int k = 0; k < rl[t]; ++k) {
        const int sl = stencil_slot(gn[cgid[s0 + k]] - a, nf);
        if (sl >= 0) fst[(int64_t)sl * nfl + a] = val[s0 + k];
      }
    }
    return;
  }
  const int m = (int)(B - A);
  // the thread's entries k = t + kB i: column ids and values, then their
  // lattice nodes, each group of loads issued together
  constexpr int IT = (CAP + kB - 1) / kB;
  int cg[IT];
  double vv[IT];
  long long gg[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int k = t + kB * i;
    cg[i] = k < m ? cgid[A + k] : 0;
    vv[i] = k < m ? val[A + k] : 0.0;
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) gg[i] = t + kB * i < m ? gn[cg[i]] : 0;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int k = t + kB * i;
    if (k >= m) break;
    int lo = 0, hi = nr - 1;  // the row holding entry k: the last r with rs[r] - A <= k
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (rs[mid] - A <= k) lo = mid;
      else hi = mid - 1;
    }
    const int sl = stencil_slot(gg[i] - an[lo], nf);
    if (sl >= 0) {
      tile[sl][lo] = vv[i];
      atomicOr(&present[lo], 1u << sl);
    }
  }
  __syncthreads();
  for (int i = t; i < 27 * nr; i += kB) {
    const int sl = i / nr, r = i - sl * nr;
    if (present[r] >> sl & 1u) fst[(int64_t)sl * nfl + an[r]] = tile[sl][r];
  }
}

// Galerkin product, one thread per output entry (coarse node J, offset d):
//   Ac(J, J+d) = sum_{a = 2J+oa, b = 2(J+d)+ob} w(oa) A(a, b) w(ob)
// Per direction only the (oa, ob) with |2d + ob - oa| <= 1 meet the 27-point
// stencil of A: 7 pairs for d = 0, 3 for d = +-1, summed in a fixed order.
// The fine operator is a stencil [27][.] on a grid of stride S whose node I
// sits at index I - off (off = 0: the fine lattice, 1: a padded coarse level).
__constant__ signed char kGalPairs[3][7][2] = {
    {{-1, 0}, {-1, 1}, {0, 1}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},                  // d = -1
    {{-1, -1}, {-1, 0}, {0, -1}, {0, 0}, {0, 1}, {1, 0}, {1, 1}},                // d = 0
    {{0, -1}, {1, -1}, {1, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}}};                 // d = +1
// L lanes per output entry (a power of two <= 64, so a group sits in one wave)
// split its (oa, ob) pairs, flattened z-major, and sum them with a fixed
// shuffle tree; with L = 1 the order is the nested loops' order.  Small levels
// use many lanes: one lane's chain of up to 7^3 dependent loads would bound them.
template <int L>
__global__ __launch_bounds__(kB) void k_galerkin_e(int mc, int S, int off, int64_t fine_tot,
                                                   const double *__restrict__ af, double *__restrict__ cst) {
  const int64_t tot = (int64_t)mc * mc * mc;
  const int64_t tq = blockIdx.x * (int64_t)kB + threadIdx.x;
  const int64_t t = tq / L;
  const int sub = (int)(tq % L);
  if (t >= 27 * tot) return;  // whole lane groups: kB is a multiple of L
  const int k = (int)(t / tot);  // output slot: consecutive outputs share it (coalesced stores)
  const int64_t j = t - k * tot;
  const int jx = (int)(j % mc), jy = (int)((j / mc) % mc), jz = (int)(j / ((int64_t)mc * mc));
  const int dx = k % 3 - 1, dy = (k / 3) % 3 - 1, dz = k / 9 - 1;
  const int Jx = jx + 1, Jy = jy + 1, Jz = jz + 1;
  double acc = 0.0;
  const bool live = jx < mc - 1 && jy < mc - 1 && jz < mc - 1 && Jx + dx >= 1 && Jy + dy >= 1 && Jz + dz >= 1 &&
                    Jx + dx <= mc - 1 && Jy + dy <= mc - 1 && Jz + dz <= mc - 1;
  if (live && L == 1) {
    const int nx = dx ? 3 : 7, ny = dy ? 3 : 7, nz = dz ? 3 : 7;
    // y and x unrolled to their largest count (7) with the counts as
    // predicates, so that a z plane's loads are issued together; the sums
    // keep the nested loops' order
    for (int pz = 0; pz < nz; ++pz) {
      const int oaz = kGalPairs[dz + 1][pz][0], obz = kGalPairs[dz + 1][pz][1];
      const double wz = (oaz ? 0.5 : 1.0) * (obz ? 0.5 : 1.0);
      const int ez = 2 * dz + obz - oaz + 1;
      const int64_t az = 2 * Jz + oaz - off;
#pragma unroll
      for (int py = 0; py < 7; ++py) {
        if (py >= ny) break;
        const int oay = kGalPairs[dy + 1][py][0], oby = kGalPairs[dy + 1][py][1];
        const double wyz = wz * (oay ? 0.5 : 1.0) * (oby ? 0.5 : 1.0);
        const int ey = 2 * dy + oby - oay + 1;
        const int64_t ayz = (2 * Jy + oay - off) + (int64_t)S * az;
#pragma unroll
        for (int px = 0; px < 7; ++px) {
          if (px >= nx) break;
          const int oax = kGalPairs[dx + 1][px][0], obx = kGalPairs[dx + 1][px][1];
          const double w = wyz * (oax ? 0.5 : 1.0) * (obx ? 0.5 : 1.0);
          const int ex = 2 * dx + obx - oax + 1;
          const int64_t a = (2 * Jx + oax - off) + (int64_t)S * ayz;
          acc = fma(w, af[(int64_t)(ex + 3 * ey + 9 * ez) * fine_tot + a], acc);
        }
      }
    }
  } else if (live) {
    const int nx = dx ? 3 : 7, ny = dy ? 3 : 7, nz = dz ? 3 : 7;
    const int n = nx * ny * nz;
    for (int q = sub; q < n; q += L) {
      const int px = q % nx, py = (q / nx) % ny, pz = q / (nx * ny);
      const int oaz = kGalPairs[dz + 1][pz][0], obz = kGalPairs[dz + 1][pz][1];
      const int oay = kGalPairs[dy + 1][py][0], oby = kGalPairs[dy + 1][py][1];
      const int oax = kGalPairs[dx + 1][px][0], obx = kGalPairs[dx + 1][px][1];
      const double wz = (oaz ? 0.5 : 1.0) * (obz ? 0.5 : 1.0);
      const double wyz = wz * (oay ? 0.5 : 1.0) * (oby ? 0.5 : 1.0);
      const double w = wyz * (oax ? 0.5 : 1.0) * (obx ? 0.5 : 1.0);
      const int ex = 2 * dx + obx - oax + 1, ey = 2 * dy + oby - oay + 1, ez = 2 * dz + obz - oaz + 1;
      const int64_t az = 2 * Jz + oaz - off;
      const int64_t ayz = (2 * Jy + oay - off) + (int64_t)S * az;
      const int64_t a = (2 * Jx + oax - off) + (int64_t)S * ayz;
      acc = fma(w, af[(int64_t)(ex + 3 * ey + 9 * ez) * fine_tot + a], acc);
    }
  }
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, L);
  if (sub == 0) cst[k * tot + j] = acc;
}

// Galerkin product launch: lanes per output so that a level has about 2^20 threads
void galerkin(int mc, int S, int off, int64_t fine_tot, const double *af, double *cst, hipStream_t st) {
  const int64_t outs = 27 * (int64_t)mc * mc * mc;
  int L = 1;
  while (L < 64 && outs * L < (1 << 20)) L *= 2;
  const dim3 g((unsigned)((outs * L + kB - 1) / kB)), b(kB);
  switch (L) {
    case 1: hipLaunchKernelGGL(k_galerkin_e<1>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
    case 2: hipLaunchKernelGGL(k_galerkin_e<2>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
    case 4: hipLaunchKernelGGL(k_galerkin_e<4>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
    case 8: hipLaunchKernelGGL(k_galerkin_e<8>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
    case 16: hipLaunchKernelGGL(k_galerkin_e<16>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
    case 32: hipLaunchKernelGGL(k_galerkin_e<32>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
    default: hipLaunchKernelGGL(k_galerkin_e<64>, g, b, 0, st, mc, S, off, fine_tot, af, cst); break;
  }
}

// ec = s * out (network units -> coarse error), 0 on the padding plane; or 0 everywhere
__global__ void k_out_to_coarse(int n, const float *__restrict__ out, const double *__restrict__ s, int use,
                                double *__restrict__ ec) {
  const int64_t tot = (int64_t)n * n * n;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % n), jy = (int)((j / n) % n), jz = (int)(j / ((int64_t)n * n));
  ec[j] = (use && jx < n - 1 && jy < n - 1 && jz < n - 1) ? (double)out[j] * *s : 0.0;
}

// b = Ac a on the network grid (padding plane 0)
__global__ void k_coarse_apply(int n, const double *__restrict__ cst, const double *__restrict__ a,
                               double *__restrict__ b) {
  const int64_t tot = (int64_t)n * n * n;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % n), jy = (int)((j / n) % n), jz = (int)(j / ((int64_t)n * n));
  double r = 0.0;
  if (jx < n - 1 && jy < n - 1 && jz < n - 1)
    for (int k = 0; k < 27; ++k) {
      const int x = jx + k % 3 - 1, y = jy + (k / 3) % 3 - 1, z = jz + k / 9 - 1;
      if (x < 0 || y < 0 || z < 0 || x > n - 2 || y > n - 2 || z > n - 2) continue;
      r = fma(cst[k * tot + j], a[x + (int64_t)n * (y + (int64_t)n * z)], r);
    }
  b[j] = r;
}

__global__ void k_scale_by(int64_t tot, const double *__restrict__ alpha, double *__restrict__ a) {
  const int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (i < tot) a[i] *= *alpha;
}

// partial sums of out.tgt, out.out, tgt.tgt (three areas of kRed)
__global__ __launch_bounds__(kB) void k_dot3f(int64_t tot, const float *__restrict__ a, const float *__restrict__ b,
                                             double *__restrict__ part) {
  __shared__ double s1[kB], s2[kB], s3[kB];
  double p1 = 0.0, p2 = 0.0, p3 = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x; i < tot; i += (int64_t)gridDim.x * kB) {
    const double x = a[i], y = b[i];
    p1 = fma(x, y, p1);
    p2 = fma(x, x, p2);
    p3 = fma(y, y, p3);
  }
  s1[threadIdx.x] = p1;
  s2[threadIdx.x] = p2;
  s3[threadIdx.x] = p3;
  __syncthreads();
  for (int o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
      s3[threadIdx.x] += s3[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s1[0];
    part[kRed + blockIdx.x] = s2[0];
    part[2 * kRed + blockIdx.x] = s3[0];
  }
}

// sums of the three partial areas into out[0..3), and the loss
// 1 - (N.t)^2 / (|N|^2 |t|^2) into out[3]
__global__ __launch_bounds__(kB) void k_finish3(const double *__restrict__ part, double *__restrict__ out) {
  __shared__ double s1[kB], s2[kB], s3[kB];
  double p1 = 0.0, p2 = 0.0, p3 = 0.0;
  for (int i = threadIdx.x; i < kRed; i += kB) {
    p1 += part[i];
    p2 += part[kRed + i];
    p3 += part[2 * kRed + i];
  }
  s1[threadIdx.x] = p1;
  s2[threadIdx.x] = p2;
  s3[threadIdx.x] = p3;
  __syncthreads();
  for (int o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
      s3[threadIdx.x] += s3[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = s1[0];
    out[1] = s2[0] > 0.0 ? s2[0] : 1e-300;
    out[2] = s3[0] > 0.0 ? s3[0] : 1e-300;
    out[3] = 1.0 - s1[0] * s1[0] / (out[1] * out[2]);
  }
}

// gradient of 1 - (N.t)^2 / (|N|^2 |t|^2) with respect to N:
// -2 (N.t) / (|N|^2 |t|^2) (t - (N.t) / |N|^2 N)
__global__ void k_cos_grad(int64_t tot, const float *__restrict__ out, const float *__restrict__ tgt,
                           const double *__restrict__ sums, float *__restrict__ dout) {
  const int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (i >= tot) return;
  const double nt = sums[0], nn = sums[1], tt = sums[2];
  dout[i] = (float)(-2.0 * nt / (nn * tt) * ((double)tgt[i] - nt / nn * (double)out[i]));
}

// one damped-Jacobi sweep on the coarse system: b = a + w Dc^-1 (rc - Ac a)
// r0 - sum over the interior neighbours of cst[k][j] x[neighbour k], in stencil
// order.  The 54 loads are predicated (zero outside the interior) and issued
// before the subtractions, so a small grid is not one chain of dependent
// loads; a skipped term subtracts 0 * 0, which leaves r unchanged exactly.
__device__ __forceinline__ double stencil_residual(double r0, int n, int64_t tot, int64_t j, int jx, int jy, int jz,
                                                   const double *__restrict__ cst,
                                                   const double *__restrict__ x) {
  double cv[27], xv[27];
#pragma unroll
  for (int k = 0; k < 27; ++k) {
    const int ox = k % 3 - 1, oy = (k / 3) % 3 - 1, oz = k / 9 - 1;
    const int X = jx + ox, Y = jy + oy, Z = jz + oz;
    const bool in = X >= 0 && Y >= 0 && Z >= 0 && X <= n - 2 && Y <= n - 2 && Z <= n - 2;
    cv[k] = in ? cst[k * tot + j] : 0.0;
    xv[k] = in ? x[j + ox + (int64_t)n * (oy + (int64_t)n * oz)] : 0.0;
  }
  double r = r0;
#pragma unroll
  for (int k = 0; k < 27; ++k) r -= cv[k] * xv[k];
  return r;
}

__global__ void k_coarse_sweep(int n, double w, const double *__restrict__ cst, const double *__restrict__ rc,
                               const double *__restrict__ a, double *__restrict__ b) {
  const int64_t tot = (int64_t)n * n * n;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % n), jy = (int)((j / n) % n), jz = (int)(j / ((int64_t)n * n));
  if (jx == n - 1 || jy == n - 1 || jz == n - 1) {
    b[j] = 0.0;
    return;
  }
  const double r = stencil_residual(rc[j], n, tot, j, jx, jy, jz, cst, a);
  b[j] = a[j] + w * r / cst[13 * tot + j];
}

// fine lattice value of P ec (double coarse field on the network grid)
// trilinear value at node (x, y, z) of a level of 2 mc cells from the interior
// nodes of its coarse level: the 8 loads are predicated and issued together
__device__ __forceinline__ double prolonged(int mc, int x, int y, int z, const double *__restrict__ ec) {
  double v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int kx = k & 1, ky = k >> 1 & 1, kz = k >> 2;
    const int Jx = (x >> 1) + kx, Jy = (y >> 1) + ky, Jz = (z >> 1) + kz;
    const bool in = kx <= (x & 1) && ky <= (y & 1) && kz <= (z & 1) && Jx >= 1 && Jy >= 1 && Jz >= 1 &&
                    Jx <= mc - 1 && Jy <= mc - 1 && Jz <= mc - 1;
    v[k] = in ? ec[(Jx - 1) + (int64_t)mc * ((Jy - 1) + (int64_t)mc * (Jz - 1))] : 0.0;
  }
  const double w = ((x & 1) ? 0.5 : 1.0) * ((y & 1) ? 0.5 : 1.0) * ((z & 1) ? 0.5 : 1.0);
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < 8; ++k) acc = fma(w, v[k], acc);
  return acc;
}

// (32-bit node numbers: a lattice of 2^31 nodes would need a 464 GB stencil)
__global__ void k_prolong_d(int n, int nf, const double *__restrict__ ec, double *__restrict__ flat) {
  const unsigned tot = (unsigned)nf * nf * nf, i = blockIdx.x * kB + threadIdx.x;
  if (i >= tot) return;
  const int x = (int)(i % nf), y = (int)(i / nf % nf), z = (int)(i / ((unsigned)nf * nf));
  if (x == 0 || y == 0 || z == 0 || x == nf - 1 || y == nf - 1 || z == nf - 1) {
    flat[i] = 0.0;
    return;
  }
  flat[i] = prolonged(n, x, y, z, ec);
}

// ---------------------------------------------------------------------------
// multigrid on the structured coarse levels (padded interior storage)
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool padding(int64_t j, int m, int &x, int &y, int &z) {
  x = (int)(j % m);
  y = (int)((j / m) % m);
  z = (int)(j / ((int64_t)m * m));
  return x == m - 1 || y == m - 1 || z == m - 1;
}

// res = rhs - A e
__global__ void k_resid(int m, const double *__restrict__ cst, const double *__restrict__ rhs,
                        const double *__restrict__ e, double *__restrict__ res) {
  const int64_t tot = (int64_t)m * m * m;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  int jx, jy, jz;
  if (padding(j, m, jx, jy, jz)) {
    res[j] = 0.0;
    return;
  }
  res[j] = stencil_residual(rhs[j], m, tot, j, jx, jy, jz, cst, e);
}

// first damped-Jacobi sweep from zero: e = w Dc^-1 rhs
__global__ void k_sweep0(int m, double w, const double *__restrict__ cst, const double *__restrict__ rhs,
                         double *__restrict__ e) {
  const int64_t tot = (int64_t)m * m * m;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  int jx, jy, jz;
  e[j] = padding(j, m, jx, jy, jz) ? 0.0 : w * rhs[j] / cst[13 * tot + j];
}

// full weighting from level mf to mf/2: rc[J] = sum_o w(o) r[2J + o], and that
// level's first damped-Jacobi sweep from zero, ec = w Dc^-1 rc (ec null: the
// coarsest level, which starts its own)
__global__ void k_restrict_c(int mf, double w, const double *__restrict__ rf, const double *__restrict__ ccst,
                             double *__restrict__ rc, double *__restrict__ ec) {
  const int mc = mf / 2;
  const unsigned tot = (unsigned)mc * mc * mc, j = blockIdx.x * kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % mc), jy = (int)(j / mc % mc), jz = (int)(j / ((unsigned)mc * mc));
  double acc = 0.0, e0 = 0.0;
  if (jx < mc - 1 && jy < mc - 1 && jz < mc - 1) {
    for (int oz = 0; oz < 3; ++oz)  // storage of the fine nodes 2J + o: 2j .. 2j + 2
      for (int oy = 0; oy < 3; ++oy)
        for (int ox = 0; ox < 3; ++ox) {
          const double wt = (ox != 1 ? 0.5 : 1.0) * (oy != 1 ? 0.5 : 1.0) * (oz != 1 ? 0.5 : 1.0);
          acc = fma(wt, rf[(2 * jx + ox) + (size_t)mf * ((2 * jy + oy) + (size_t)mf * (2 * jz + oz))], acc);
        }
    if (ec) e0 = w * acc / ccst[(size_t)13 * tot + j];
  }
  rc[j] = acc;
  if (ec) ec[j] = e0;
}

// The residual rhs - A e and k_restrict_c's work in one launch, for levels up to
// kDownMax.  A workgroup owns 16 x 2 x 2 coarse nodes and keeps the residual at
// the 33 x 5 x 5 fine nodes below them in LDS, 1.6 of them per own node.  Small
// levels are bound by the launch and one round of loads: 7.5 us against 14 for
// residual, weighting and sweep apart at 8^3 to 32^3.  Where the planes' bytes
// bound the residual the extra nodes cost more than the launches: at 64^3 29 us
// against 15 for k_resid and k_restrict_c.
constexpr int kDownMax = 32;
constexpr int kDnX = 16, kDnY = 2, kDnZ = 2, kDnThreads = 832;
__global__ __launch_bounds__(kDnThreads) void k_down(int m, double w, const double *__restrict__ cst,
                                                     const double *__restrict__ rhs, const double *__restrict__ e,
                                                     const double *__restrict__ ccst, double *__restrict__ rc,
                                                     double *__restrict__ ec) {
  constexpr int FX = 2 * kDnX + 1, FY = 2 * kDnY + 1, FZ = 2 * kDnZ + 1;
  __shared__ double res[FX * FY * FZ];
  const int mc = m / 2, t = threadIdx.x;
  const int X0 = kDnX * blockIdx.x, Y0 = kDnY * blockIdx.y, Z0 = kDnZ * blockIdx.z;
  const int64_t tot = (int64_t)m * m * m, totc = (int64_t)mc * mc * mc;
  // coarse storage index J has fine storage nodes 2J .. 2J + 2
  for (int q = t; q < FX * FY * FZ; q += kDnThreads) {
    const int x = 2 * X0 + q % FX, y = 2 * Y0 + (q / FX) % FY, z = 2 * Z0 + q / (FX * FY);
    double r = 0.0;
    if (x <= m - 2 && y <= m - 2 && z <= m - 2) {
      const int64_t j = x + (int64_t)m * (y + (int64_t)m * z);
      r = stencil_residual(rhs[j], m, tot, j, x, y, z, cst, e);
    }
    res[q] = r;
  }
  __syncthreads();
  if (t >= kDnX * kDnY * kDnZ) return;
  const int lx = t % kDnX, ly = (t / kDnX) % kDnY, lz = t / (kDnX * kDnY);
  const int X = X0 + lx, Y = Y0 + ly, Z = Z0 + lz;
  if (X >= mc || Y >= mc || Z >= mc) return;
  const int64_t j = X + (int64_t)mc * (Y + (int64_t)mc * Z);
  double acc = 0.0, e0 = 0.0;
  if (X < mc - 1 && Y < mc - 1 && Z < mc - 1) {
    for (int oz = 0; oz < 3; ++oz)
      for (int oy = 0; oy < 3; ++oy)
        for (int ox = 0; ox < 3; ++ox) {
          const double wt = (ox != 1 ? 0.5 : 1.0) * (oy != 1 ? 0.5 : 1.0) * (oz != 1 ? 0.5 : 1.0);
          acc = fma(wt, res[2 * lx + ox + FX * (2 * ly + oy + FY * (2 * lz + oz))], acc);
        }
    if (ec) e0 = w * acc / ccst[13 * totc + j];
  }
  rc[j] = acc;
  if (ec) ec[j] = e0;
}

// One launch up a level: a' = a + P ec (trilinear, from level m/2) and one
// damped-Jacobi sweep, b = a' + w D^-1 (rhs - A a').  A workgroup owns 16 x 4 x 4
// nodes and keeps a' there and on the layer around them in LDS.
constexpr int kUpX = 16, kUpY = 4, kUpZ = 4, kUpThreads = kUpX * kUpY * kUpZ;
__global__ __launch_bounds__(kUpThreads) void k_up(int m, double w, const double *__restrict__ cst,
                                                   const double *__restrict__ rhs, const double *__restrict__ a,
                                                   const double *__restrict__ ec, double *__restrict__ b) {
  constexpr int HX = kUpX + 2, HY = kUpY + 2, HZ = kUpZ + 2;
  __shared__ double ap[HX * HY * HZ];
  const int mc = m / 2, t = threadIdx.x;
  const int64_t tot = (int64_t)m * m * m;
  const int X0 = kUpX * blockIdx.x, Y0 = kUpY * blockIdx.y, Z0 = kUpZ * blockIdx.z;
  const int lx = t % kUpX, ly = (t / kUpX) % kUpY, lz = t / (kUpX * kUpY);
  const int X = X0 + lx, Y = Y0 + ly, Z = Z0 + lz;
  const bool live = X <= m - 2 && Y <= m - 2 && Z <= m - 2;
  const int64_t j = live ? X + (int64_t)m * (Y + (int64_t)m * Z) : 0;
  // the node's coefficients (zero towards the boundary) load while a' is formed
  double cv[27];
#pragma unroll
  for (int k = 0; k < 27; ++k) cv[k] = live ? cst[k * tot + j] : 0.0;
  const double r0 = live ? rhs[j] : 0.0;
  for (int q = t; q < HX * HY * HZ; q += kUpThreads) {
    const int ix = X0 + q % HX - 1, iy = Y0 + (q / HX) % HY - 1, iz = Z0 + q / (HX * HY) - 1;
    double v = 0.0;
    if (ix >= 0 && iy >= 0 && iz >= 0 && ix <= m - 2 && iy <= m - 2 && iz <= m - 2) {
      v = a[ix + (int64_t)m * (iy + (int64_t)m * iz)] + prolonged(mc, ix + 1, iy + 1, iz + 1, ec);
    }
    ap[q] = v;
  }
  __syncthreads();
  if (X >= m || Y >= m || Z >= m) return;
  const int64_t js = X + (int64_t)m * (Y + (int64_t)m * Z);
  if (!live) {
    b[js] = 0.0;
    return;
  }
  const int c = (lx + 1) + HX * ((ly + 1) + HY * (lz + 1));
  double r = r0;
#pragma unroll
  for (int k = 0; k < 27; ++k) r -= cv[k] * ap[c + (k % 3 - 1) + HX * (((k / 3) % 3 - 1) + HY * (k / 9 - 1))];
  b[js] = ap[c] + w * r / cv[13];
}

// coarsest level (m <= 8): damped-Jacobi sweeps from zero in one workgroup;
// the stencil is staged in LDS when it fits (m <= 6).  L lanes per grid point
// (the largest power of two with L * m^3 <= 1024) split the point's 27
// stencil terms and sum them with a fixed shuffle tree, so a sweep is not one
// lane's chain of 27 dependent LDS reads.
constexpr int kCoarsestMax = 8;
constexpr int kCoarsestLds = 6 * 6 * 6;
constexpr int kCoarsestThreads = 1024;
__host__ __device__ constexpr int coarsest_lanes(int tot) {
  int L = 32;
  while (L > 1 && L * tot > kCoarsestThreads) L >>= 1;
  return L;
}

template <int L>
__global__ __launch_bounds__(kCoarsestThreads) void k_coarsest(int m, double w, int sweeps,
                                                               const double *__restrict__ cstg,
                                                               const double *__restrict__ rhs,
                                                               double *__restrict__ e) {
  __shared__ double ea[512], eb[512], cl[27 * kCoarsestLds];
  const int tot = m * m * m;
  const int t = threadIdx.x, j = t / L, sub = t % L;  // the L lanes of a point share one wave
  int jx = 0, jy = 0, jz = 0;
  const bool live = j < tot && !padding(j, m, jx, jy, jz);
  const bool staged = tot <= kCoarsestLds;
  if (staged)
    for (int i = t; i < 27 * tot; i += blockDim.x) cl[i] = cstg[i];
  const double *cst = staged ? cl : cstg;
  if (sub == 0 && j < tot) ea[j] = 0.0;
  // the right-hand side and the diagonal are read once, not per sweep
  const double rj = live ? rhs[j] : 0.0;
  __syncthreads();
  const double dj = live ? cst[13 * tot + j] : 1.0;
  // this lane's stencil slots inside the interior, as a bit mask
  uint32_t nbr = 0;
  for (int k = sub; k < 27; k += L) {
    const int x = jx + k % 3 - 1, y = jy + (k / 3) % 3 - 1, z = jz + k / 9 - 1;
    if (live && x >= 0 && y >= 0 && z >= 0 && x <= m - 2 && y <= m - 2 && z <= m - 2) nbr |= 1u << k;
  }
  // this lane's stencil coefficients and neighbour offsets (slots k = sub + L i),
  // the same every sweep: read once into registers
  constexpr int KL = (27 + L - 1) / L;
  double cf[KL];
  int of[KL];
#pragma unroll
  for (int i = 0; i < KL; ++i) {
    const int k = sub + L * i;
    const bool use = k < 27 && (nbr >> k & 1u);
    cf[i] = use ? cst[k * tot + j] : 0.0;
    of[i] = use ? (k % 3 - 1) + m * ((k / 3) % 3 - 1) + m * m * (k / 9 - 1) : 0;
  }
  double *a = ea, *b = eb;
  for (int s = 0; s < sweeps; ++s) {
    double part = 0.0;
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int k = sub + L * i;
      if (k >= 27 || !(nbr >> k & 1u)) continue;
      part = fma(cf[i], a[j + of[i]], part);
    }
    for (int o = L / 2; o > 0; o >>= 1) part += __shfl_xor(part, o, L);
    if (sub == 0 && j < tot) b[j] = live ? a[j] + w * (rj - part) / dj : 0.0;
    __syncthreads();
    double *tmp = a;
    a = b;
    b = tmp;
  }
  if (sub == 0 && j < tot) e[j] = a[j];
}

// the same sweeps where one wave holds the level (m <= 5: at most 64 interior
// points, where halving stops for 2^k and 3 2^k): L lanes per point, the grid in
// LDS with a zero layer around it, the point's lanes summed by lane moves.  A
// sweep is one chain of LDS reads, multiply-adds and a write, without a barrier
// between waves.
constexpr int kWaveLevel = 5;
template <int CTRL>
__device__ __forceinline__ double lane_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

template <int L>
__global__ __launch_bounds__(64) void k_coarsest_wave(int m, double w, int sweeps, const double *__restrict__ cst,
                                                      const double *__restrict__ rhs, double *__restrict__ e) {
  constexpr int KL = (27 + L - 1) / L, M = kWaveLevel + 1;
  __shared__ double g[2][M * M * M];
  const int t = threadIdx.x, p = t / L, sub = t % L, mi = m - 1, tot = m * m * m;
  const bool live = p < mi * mi * mi;
  const int jx = live ? p % mi : 0, jy = live ? (p / mi) % mi : 0, jz = live ? p / (mi * mi) : 0;
  const int j = jx + m * (jy + m * jz), c = (jx + 1) + M * ((jy + 1) + M * (jz + 1));
  for (int i = t; i < 2 * M * M * M; i += 64) (&g[0][0])[i] = 0.0;
  for (int i = t; i < tot; i += 64) e[i] = 0.0;  // the padding; the points follow at the end
  double cf[KL];
  int of[KL];
#pragma unroll
  for (int i = 0; i < KL; ++i) {
    const int k = sub + L * i;
    cf[i] = live && k < 27 ? cst[k * tot + j] : 0.0;  // zero towards the boundary
    of[i] = k < 27 ? c + (k % 3 - 1) + M * ((k / 3) % 3 - 1) + M * M * (k / 9 - 1) : c;
  }
  const double rj = live ? rhs[j] : 0.0, wd = live ? w / cst[13 * tot + j] : 0.0;
  double a = 0.0;
  __syncthreads();
  for (int s = 0; s < sweeps; ++s) {
    double v[KL], p0 = 0.0, p1 = 0.0;
#pragma unroll
    for (int i = 0; i < KL; ++i) v[i] = g[s & 1][of[i]];
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      if (i & 1) p1 = fma(cf[i], v[i], p1);
      else p0 = fma(cf[i], v[i], p0);
    }
    double part = p0 + p1;
    if (L >= 2) part += lane_move<0xB1>(part);   // lane ^ 1
    if (L >= 4) part += lane_move<0x4E>(part);   // lane ^ 2
    if (L >= 8) part += lane_move<0x141>(part);  // the other four of eight
    a = fma(wd, rj - part, a);
    if (sub == 0 && live) g[(s & 1) ^ 1][c] = a;
    __syncthreads();
  }
  if (sub == 0 && live) e[j] = a;
}

// partial sums of squares (and of a*b) over a grid-stride slice
__global__ __launch_bounds__(kB) void k_sumsq(int64_t n, const double *__restrict__ a, const float *__restrict__ fa,
                                             double *__restrict__ part) {
  __shared__ double sh[kB];
  double s = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x; i < n; i += (int64_t)gridDim.x * kB) {
    const double v = a ? a[i] : (double)fa[i];
    s = fma(v, v, s);
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// out = sum of the partials (one block, fixed order); mode 0: out = rms over
// 'count' values, mode 1: out = plain sum
__global__ __launch_bounds__(kB) void k_finish(const double *__restrict__ part, int nparts, double count, int mode,
                                              double *__restrict__ out) {
  __shared__ double sh[kB];
  double s = 0.0;
  for (int i = threadIdx.x; i < nparts; i += kB) s += part[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double v = mode == 0 ? sqrt(sh[0] / count) : sh[0];
    if (mode == 0 && !(v > 0.0)) v = 1.0;  // zero residual: any scale
    *out = v;
  }
}

// network input channel 0 = rho / s
__global__ void k_input0(int64_t tot, const double *__restrict__ rho, const double *__restrict__ s, float *__restrict__ inp) {
  const int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (i < tot) inp[i] = (float)(rho[i] / *s);
}

// channel 1 = log of the fine diagonal at the coarse node (scaled by h), centred
__global__ void k_input1(int n, int nf, double h, const double *__restrict__ dlat, float *__restrict__ inp1) {
  const int64_t tot = (int64_t)n * n * n;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % n), jy = (int)((j / n) % n), jz = (int)(j / ((int64_t)n * n));
  float v = 0.0f;
  if (jx < n - 1 && jy < n - 1 && jz < n - 1) {
    const double d = dlat[2 * (jx + 1) + (int64_t)nf * (2 * (jy + 1) + (int64_t)nf * 2 * (jz + 1))];
    v = (float)(0.5 * (-log(d * h) - log(8.0 / 3.0)));
  }
  inp1[j] = v;
}

// fine lattice value of P ec at interior fine nodes: trilinear from the coarse
// nodes (ec = s * out on interior coarse nodes, 0 on the boundary)
__global__ void k_prolong(int n, int nf, const float *__restrict__ out, const double *__restrict__ s,
                          double *__restrict__ flat) {
  const int64_t tot = (int64_t)nf * nf * nf;
  const int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (i >= tot) return;
  const int x = (int)(i % nf), y = (int)((i / nf) % nf), z = (int)(i / ((int64_t)nf * nf));
  if (x == 0 || y == 0 || z == 0 || x == nf - 1 || y == nf - 1 || z == nf - 1) {
    flat[i] = 0.0;
    return;
  }
  const int nc = n;  // coarse cells: coarse nodes 0..nc, interior 1..nc-1
  double acc = 0.0;
  for (int kz = 0; kz < 2; ++kz) {
    const int Iz = (z >> 1) + kz * (z & 1);
    if (kz && !(z & 1)) break;
    for (int ky = 0; ky < 2; ++ky) {
      const int Iy = (y >> 1) + ky * (y & 1);
      if (ky && !(y & 1)) break;
      for (int kx = 0; kx < 2; ++kx) {
        const int Ix = (x >> 1) + kx * (x & 1);
        if (kx && !(x & 1)) break;
        if (Ix < 1 || Iy < 1 || Iz < 1 || Ix > nc - 1 || Iy > nc - 1 || Iz > nc - 1) continue;
        const double w = ((x & 1) ? 0.5 : 1.0) * ((y & 1) ? 0.5 : 1.0) * ((z & 1) ? 0.5 : 1.0);
        acc = fma(w, (double)out[(Ix - 1) + (int64_t)n * ((Iy - 1) + (int64_t)n * (Iz - 1))], acc);
      }
    }
  }
  flat[i] = acc * *s;
}

__global__ void k_jacobi0(int n, double w, const double *__restrict__ dinv, const double *__restrict__ r,
                          double *__restrict__ z) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i < n) z[i] = w * dinv[i] * r[i];
}
// t = r - t (t held A z)
__global__ void k_rminus(int n, const double *__restrict__ r, double *__restrict__ t) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i < n) t[i] = r[i] - t[i];
}
// z += c
__global__ void k_add(int n, double *__restrict__ z, const double *__restrict__ c) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i < n) z[i] += c[i];
}
__host__ __device__ inline uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// white noise on the interior coarse nodes of the network grid (0 on the padding)
__global__ void k_coarse_noise(int n, uint64_t seed, double *__restrict__ e) {
  const int64_t tot = (int64_t)n * n * n;
  const int64_t j = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (j >= tot) return;
  const int jx = (int)(j % n), jy = (int)((j / n) % n), jz = (int)(j / ((int64_t)n * n));
  const uint64_t z = mix64(seed * 0x9E3779B97F4A7C15ull + (uint64_t)(j + 1) * 0xD1B54A32D192ED03ull);
  const double u = ((double)(z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  e[j] = (jx < n - 1 && jy < n - 1 && jz < n - 1) ? 2.0 * u - 1.0 : 0.0;
}

// P 3x3x3 means, one after another, over the interior coarse nodes (zero
// Dirichlet outside).  A workgroup owns 16 x 8 x 8 nodes and keeps what they
// depend on in LDS, shrinking by a layer a pass.  One pass a launch is bound by
// the launch and its chain of predicated loads (64^3: 7.7 us); P passes read and
// write memory once, for (5704 / 3072 at P = 3) more means.  Each mean adds its
// 27 terms in the same order at any P.  64^3: 13.6 us at P = 3
// (23 for three launches).
constexpr int kBoxX = 16, kBoxY = 8, kBoxZ = 8, kBoxThreads = 512, kBoxPasses = 3;

template <int LEFT>  // from a, which reaches LEFT layers beyond the tile, the pass's means into b, LEFT - 1
__device__ __forceinline__ void box_pass(int n, int X0, int Y0, int Z0, const double *a, double *b) {
  constexpr int AX = kBoxX + 2 * LEFT, AY = kBoxY + 2 * LEFT;
  constexpr int H = LEFT - 1, BX = kBoxX + 2 * H, BY = kBoxY + 2 * H, BZ = kBoxZ + 2 * H;
  for (int q = threadIdx.x; q < BX * BY * BZ; q += kBoxThreads) {
    const int lx = q % BX, ly = (q / BX) % BY, lz = q / (BX * BY);
    const int x = X0 + lx - H, y = Y0 + ly - H, z = Z0 + lz - H;
    double s = 0.0;
    if (x >= 0 && y >= 0 && z >= 0 && x <= n - 2 && y <= n - 2 && z <= n - 2) {
#pragma unroll
      for (int o = 0; o < 27; ++o) s += a[lx + o % 3 + AX * (ly + (o / 3) % 3 + AY * (lz + o / 9))];
      s *= 1.0 / 27.0;
    }
    b[q] = s;
  }
  __syncthreads();
}

template <int P>
__global__ __launch_bounds__(kBoxThreads) void k_box(int n, const double *__restrict__ a, double *__restrict__ b) {
  constexpr int AX = kBoxX + 2 * P, AY = kBoxY + 2 * P, AZ = kBoxZ + 2 * P;
  __shared__ double sa[AX * AY * AZ], sb[(AX - 2) * (AY - 2) * (AZ - 2)];
  const int X0 = kBoxX * blockIdx.x, Y0 = kBoxY * blockIdx.y, Z0 = kBoxZ * blockIdx.z;
  for (int q = threadIdx.x; q < AX * AY * AZ; q += kBoxThreads) {
    const int x = X0 + q % AX - P, y = Y0 + (q / AX) % AY - P, z = Z0 + q / (AX * AY) - P;
    const bool in = x >= 0 && y >= 0 && z >= 0 && x <= n - 2 && y <= n - 2 && z <= n - 2;
    sa[q] = in ? a[x + (int64_t)n * (y + (int64_t)n * z)] : 0.0;
  }
  __syncthreads();
  box_pass<P>(n, X0, Y0, Z0, sa, sb);
  if constexpr (P > 1) box_pass<P - 1>(n, X0, Y0, Z0, sb, sa);
  if constexpr (P > 2) box_pass<P - 2>(n, X0, Y0, Z0, sa, sb);
  static_assert(P <= 3);
  const double *r = P == 2 ? sa : sb;
  for (int q = threadIdx.x; q < kBoxX * kBoxY * kBoxZ; q += kBoxThreads) {
    const int x = X0 + q % kBoxX, y = Y0 + (q / kBoxX) % kBoxY, z = Z0 + q / (kBoxX * kBoxY);
    if (x < n && y < n && z < n) b[x + (int64_t)n * (y + (int64_t)n * z)] = r[q];  // the padding plane's means are 0
  }
}

__global__ void k_set(double *__restrict__ p, double v) { *p = v; }

// partial sums of a.b and c.d (grid-stride slices), part[0..kRed) and part[kRed..2kRed)
__global__ __launch_bounds__(kB) void k_dot2p(int n, const double *__restrict__ a, const double *__restrict__ b,
                                             const double *__restrict__ c, const double *__restrict__ d,
                                             double *__restrict__ part) {
  __shared__ double s1[kB], s2[kB];
  double p1 = 0.0, p2 = 0.0;
  for (int i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) {
    p1 = fma(a[i], b[i], p1);
    p2 = fma(c[i], d[i], p2);
  }
  s1[threadIdx.x] = p1;
  s2[threadIdx.x] = p2;
  __syncthreads();
  for (int o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s1[0];
    part[kRed + blockIdx.x] = s2[0];
  }
}

// alpha = (c.s) / (c.Ac): the energy-optimal step along the coarse correction
// (0 when the correction vanishes or is not finite)
__global__ __launch_bounds__(kB) void k_alpha(const double *__restrict__ part, double *__restrict__ alpha) {
  __shared__ double s1[kB], s2[kB];
  double p1 = 0.0, p2 = 0.0;
  for (int i = threadIdx.x; i < kRed; i += kB) {
    p1 += part[i];
    p2 += part[kRed + i];
  }
  s1[threadIdx.x] = p1;
  s2[threadIdx.x] = p2;
  __syncthreads();
  for (int o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double a = s1[0] / s2[0];
    *alpha = (s2[0] > 0.0 && isfinite(a)) ? a : 0.0;
  }
}

// z += alpha c ; z += w D^-1 (s - alpha Ac)   (r - A z = s - alpha Ac after the coarse step)
__global__ void k_coarse_post(int n, double w, const double *__restrict__ alpha, const double *__restrict__ dinv,
                              const double *__restrict__ s, const double *__restrict__ c,
                              const double *__restrict__ ac, double *__restrict__ z) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i < n) {
    const double a = *alpha;
    z[i] = fma(a, c[i], z[i]) + w * dinv[i] * fma(-a, ac[i], s[i]);
  }
}

// ec (double) -> network-output units for the prolongation (float) and the target ec / s
__global__ void k_ec_to_float(int64_t tot, const double *__restrict__ ec, float *__restrict__ outf) {
  const int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (i < tot) outf[i] = (float)ec[i];
}
__global__ void k_target(int64_t tot, const double *__restrict__ ec, const double *__restrict__ s, float *__restrict__ tgt) {
  const int64_t i = blockIdx.x * (int64_t)kB + threadIdx.x;
  if (i < tot) tgt[i] = (float)(ec[i] / *s);
}
// sum of squares / rms into a scalar slot of red
void rms(TwoGrid *T, const double *a, const float *fa, int64_t count, double *dst, int mode, hipStream_t st) {
  hipLaunchKernelGGL(k_sumsq, dim3(kRed), dim3(kB), 0, st, count, a, fa, T->red);
  hipLaunchKernelGGL(k_finish, dim3(1), dim3(kB), 0, st, T->red, kRed, (double)count, mode, dst);
}

// offset of the stencil's slot s on the lattice
__device__ __forceinline__ int slot_offset(int s, int nf) {
  return (s % 3 - 1) + nf * ((s / 3) % 3 - 1) + nf * nf * (s / 9 - 1);
}

// *asym = 1 if the stencil is not symmetric to the bit
__global__ __launch_bounds__(kB) void k_asymmetric(int nf, const double *__restrict__ fst, int *__restrict__ asym) {
  const int tot = nf * nf * nf, i = blockIdx.x * kB + threadIdx.x;
  int bad = 0;
  if (i < tot) {
#pragma unroll
    for (int s = 14; s < 27; ++s) {
      const int j = i + slot_offset(s, nf);
      const double u = fst[(size_t)s * tot + i], l = j < tot ? fst[(size_t)(26 - s) * tot + j] : 0.0;
      bad |= __double_as_longlong(u) != __double_as_longlong(l);
    }
  }
  if (__syncthreads_or(bad) && threadIdx.x == 0) *asym = 1;
}

// the workgroup's sums of a and b into part[blk] and part[nblk + blk]
__device__ __forceinline__ void block_dots(double a, double b, int blk, int nblk, double *__restrict__ part) {
  __shared__ double sh[2][kB / 64];
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o);
    b += __shfl_xor(b, o);
  }
  if (threadIdx.x % 64 == 0) {
    sh[0][threadIdx.x / 64] = a;
    sh[1][threadIdx.x / 64] = b;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  a = sh[0][0];
  b = sh[1][0];
  for (int k = 1; k < kB / 64; ++k) {
    a += sh[0][k];
    b += sh[1][k];
  }
  part[blk] = a;
  part[nblk + blk] = b;
}

// y = A x on the fine lattice (boundary nodes 0), or y = r - A x.  A is the
// 27-plane stencil fst; where it is symmetric only its upper 14 planes are
// read, the lower offsets' coefficients being the upper ones of the neighbour,
// which the same XCD has read shortly before (each takes a contiguous run of
// nodes).  The bound is the planes' bytes: 14 x 8 per node against 10 x 27 + 28
// for the CSR product with 16-bit column codes, and no gather through ids.
// 128^3 cells: 80 us (the CSR product 144); 96^3: 25 us, its planes staying in the
// last-level cache (62).  back walks the nodes from their end: after a product in
// the other direction the planes read last are still in that cache (70 us).
// The other form also leaves the workgroup's part of x.y and x.r in part: a dot
// of two vectors that pass by here anyway, at no pass of its own.
template <bool RESID>
__global__ __launch_bounds__(kB, 5) void k_lattice_product(int nf, int back, const double *__restrict__ fst,
                                                        const int *__restrict__ asym, const double *__restrict__ x,
                                                        const double *__restrict__ r, double *__restrict__ y,
                                                        double *__restrict__ part) {
  const int tot = nf * nf * nf, nblk = (tot + kB - 1) / kB, per = (nblk + 7) / 8;
  const int at = (int)(blockIdx.x / 8), blk = (int)(blockIdx.x % 8) * per + (back ? per - 1 - at : at);
  const int i = blk * kB + threadIdx.x;
  if (blk >= nblk) return;
  const int a = i % nf, b = (i / nf) % nf, c = i / (nf * nf);
  const bool in = i < tot && a > 0 && b > 0 && c > 0 && a < nf - 1 && b < nf - 1 && c < nf - 1;
  double acc = 0.0, xi = 0.0, ri = 0.0;
  if (in) {
    const bool sym = __builtin_amdgcn_readfirstlane(*asym) == 0;
    double up[13], lo[13], xu[13], xl[13];
#pragma unroll
    for (int k = 0; k < 13; ++k) {
      const int s = 14 + k, o = slot_offset(s, nf);
      up[k] = fst[(size_t)s * tot + i];
      lo[k] = (fst + (sym ? (int64_t)s * tot - o : (int64_t)(26 - s) * tot))[i];
      xu[k] = x[i + o];
      xl[k] = x[i - o];
    }
    xi = x[i];
    ri = r[i];
    acc = fst[(size_t)13 * tot + i] * xi;
#pragma unroll
    for (int k = 0; k < 13; ++k) acc = fma(up[k], xu[k], fma(lo[k], xl[k], acc));
  }
  if (i < tot) y[i] = RESID ? ri - acc : acc;
  if (!RESID) block_dots(xi * acc, xi * ri, blk, nblk, part);
}

// sums of both halves of the partials, in a fixed order: into out[0..2), or for
// alpha their ratio out[0] = second / first (0 when the first vanishes or the
// ratio is not finite)
template <bool ALPHA>
__global__ __launch_bounds__(1024) void k_sum2(const double *__restrict__ part, int nblk, double *__restrict__ out) {
  __shared__ double s1[1024], s2[1024];
  const int t = threadIdx.x;
  double p1 = 0.0, p2 = 0.0;
  for (int i = t; i < nblk; i += 1024) {
    p1 += part[i];
    p2 += part[nblk + i];
  }
  s1[t] = p1;
  s2[t] = p2;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (t < o) {
      s1[t] += s1[t + o];
      s2[t] += s2[t + o];
    }
    __syncthreads();
  }
  if (t != 0) return;
  if (ALPHA) {
    const double al = s2[0] / s1[0];
    out[0] = s1[0] > 0.0 && isfinite(al) ? al : 0.0;
  } else {
    out[0] = s1[0];
    out[1] = s2[0];
  }
}

// x += alpha p, r -= alpha q, alpha = p.r / p.q, and z = w D^-1 r, the first sweep
__global__ __launch_bounds__(kB) void k_lattice_update(int n, double w, const double *__restrict__ sc,
                                                       const double *__restrict__ dinv, const double *__restrict__ p,
                                                       const double *__restrict__ q, double *__restrict__ x,
                                                       double *__restrict__ r, double *__restrict__ z) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i >= n) return;
  const double alpha = sc[1] / sc[0], ri = fma(-alpha, q[i], r[i]);
  x[i] = fma(alpha, p[i], x[i]);
  r[i] = ri;
  z[i] = w * dinv[i] * ri;
}

// k_coarse_post, with the workgroup's part of z.q and r.r
__global__ __launch_bounds__(kB) void k_lattice_post(int n, double w, const double *__restrict__ alpha,
                                                     const double *__restrict__ dinv, const double *__restrict__ s,
                                                     const double *__restrict__ c, const double *__restrict__ ac,
                                                     const double *__restrict__ q, const double *__restrict__ r,
                                                     double *__restrict__ z, double *__restrict__ part) {
  const int i = blockIdx.x * kB + threadIdx.x;
  double zi = 0.0, qi = 0.0, ri = 0.0;
  if (i < n) {
    const double a = *alpha;
    zi = fma(a, c[i], z[i]) + w * dinv[i] * fma(-a, ac[i], s[i]);
    qi = q[i];
    ri = r[i];
    z[i] = zi;
  }
  block_dots(zi * qi, ri * ri, blockIdx.x, gridDim.x, part);
}

__global__ void k_lattice_dir(int n, const double *__restrict__ sc, const double *__restrict__ z,
                              double *__restrict__ p) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i < n) p[i] = fma(-sc[2] / sc[0], p[i], z[i]);
}

// network input from a fine residual in global-id order, or on the lattice (s
// into red[kS]); with the network off only the coarse residual rc is formed, and
// with e0 the V-cycle's first sweep for it
void make_input(gdx_nn *nn, TwoGrid *T, const double *r, hipStream_t st, bool for_net = true, bool lattice = false,
                double *e0 = nullptr) {
  nn::Net &N = nn->net;
  const int64_t v = (int64_t)T->n * T->n * T->n;
  // restriction reads only interior lattice nodes, all of which the scatter
  // writes: no clearing (and no memset, so this can be captured in a graph)
  if (!lattice) hipLaunchKernelGGL(k_scatter, dim3(nb(T->ng)), dim3(kB), 0, st, T->ng, T->gid_node, r, T->flat);
  hipLaunchKernelGGL(k_restrict, dim3(nb(v)), dim3(kB), 0, st, T->n, T->nf, lattice ? r : T->flat, T->dlat, T->rho,
                     T->rc, kOmegaC, T->cst, e0);
  if (!for_net) return;
  rms(T, T->rho, nullptr, v, T->red + kS, 0, st);
  hipLaunchKernelGGL(k_input0, dim3(nb(v)), dim3(kB), 0, st, v, T->rho, T->red + kS, N.inp_f);
  N.input_from_f32(N.inp_f);
}

void mg_free(TwoGrid *T) {
  for (Level &L : T->lv) {
    void *ptrs[] = {L.own_cst ? L.cst : nullptr, L.rhs, L.e, L.e2};
    for (void *q : ptrs)
      if (q) (void)hipFree(q);
  }
  T->lv.clear();
}

// levels below the network grid: halve while the cell count is even and > 4
// (the coarsest grid has at most 8 cells per direction); buffers are kept
// across attachments to the same problem, the operators are recomputed
int mg_setup(TwoGrid *T, hipStream_t st) {
  if (T->lv.empty()) {
    std::vector<int> ms{T->n};
    while (ms.back() % 2 == 0 && ms.back() > 4) ms.push_back(ms.back() / 2);
    if (ms.back() > kCoarsestMax) ms.clear();  // no coarsest grid small enough: two-grid form only
    for (size_t l = 0; l < ms.size(); ++l) {
      Level L;
      L.m = ms[l];
      const size_t v = (size_t)L.m * L.m * L.m;
      T->lv.push_back(L);
      Level &M = T->lv.back();
      bool ok = dev_malloc(reinterpret_cast<void **>(&M.rhs), v * sizeof(double)) == hipSuccess &&
                dev_malloc(reinterpret_cast<void **>(&M.e), v * sizeof(double)) == hipSuccess &&
                dev_malloc(reinterpret_cast<void **>(&M.e2), v * sizeof(double)) == hipSuccess;
      if (l == 0) {
        M.cst = T->cst;
        M.own_cst = false;
      } else {
        ok = ok && dev_malloc(reinterpret_cast<void **>(&M.cst), 27 * v * sizeof(double)) == hipSuccess;
      }
      if (!ok) {
        mg_free(T);
        return GDX_ERR_ALLOC;
      }
    }
  }
  for (size_t l = 1; l < T->lv.size(); ++l) {
    const Level &F = T->lv[l - 1];
    galerkin(T->lv[l].m, F.m, 1, (int64_t)F.m * F.m * F.m, F.cst, T->lv[l].cst, st);
  }
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

// V-cycle on level l for the right-hand side rhs, from a zero guess whose first
// sweep is already in lv[l].e (not on the coarsest level):
// nu damped-Jacobi sweeps, coarse-grid correction, nu sweeps (the coarsest
// level: sweeps in one workgroup).  Returns the buffer holding the correction.
double *vcycle(TwoGrid *T, size_t l, const double *rhs, hipStream_t st) {
  Level &L = T->lv[l];
  const int64_t v = (int64_t)L.m * L.m * L.m;
  if (l + 1 == T->lv.size()) {
    const int np = (L.m - 1) * (L.m - 1) * (L.m - 1);
    if (L.m <= kWaveLevel) {
      hipLaunchKernelGGL(np <= 8 ? k_coarsest_wave<8> : np <= 32 ? k_coarsest_wave<2> : k_coarsest_wave<1>, dim3(1),
                         dim3(64), 0, st, L.m, kOmegaC, T->coarsest_sweeps, L.cst, rhs, L.e);
      return L.e;
    }
    switch (coarsest_lanes(L.m * L.m * L.m)) {  // 6 <= m <= 8: 2 or 4 lanes per point
#define GDX_COARSEST(NL)                                                                                           \
  case NL:                                                                                                         \
    hipLaunchKernelGGL(k_coarsest<NL>, dim3(1), dim3(kCoarsestThreads), 0, st, L.m, kOmegaC, T->coarsest_sweeps, \
                       L.cst, rhs, L.e);                                                                           \
    break;
      GDX_COARSEST(2) GDX_COARSEST(4)
#undef GDX_COARSEST
      default: break;
    }
    return L.e;
  }
  double *a = L.e, *b = L.e2;
  for (int k = 1; k < T->nu; ++k) {
    hipLaunchKernelGGL(k_coarse_sweep, dim3(nb(v)), dim3(kB), 0, st, L.m, kOmegaC, L.cst, rhs, a, b);
    std::swap(a, b);
  }
  Level &C = T->lv[l + 1];
  const bool last = l + 2 == T->lv.size();
  const auto per = [](int n, int w) { return (unsigned)((n + w - 1) / w); };
  double *e0 = last ? nullptr : C.e;
  if (L.m > kDownMax) {
    hipLaunchKernelGGL(k_resid, dim3(nb(v)), dim3(kB), 0, st, L.m, L.cst, rhs, a, b);
    hipLaunchKernelGGL(k_restrict_c, dim3(nb((int64_t)C.m * C.m * C.m)), dim3(kB), 0, st, L.m, kOmegaC, b, C.cst,
                       C.rhs, e0);
  } else {
    hipLaunchKernelGGL(k_down, dim3(per(C.m, kDnX), per(C.m, kDnY), per(C.m, kDnZ)), dim3(kDnThreads), 0, st, L.m,
                       kOmegaC, L.cst, rhs, a, C.cst, C.rhs, e0);
  }
  const double *c = vcycle(T, l + 1, C.rhs, st);
  hipLaunchKernelGGL(k_up, dim3(per(L.m, kUpX), per(L.m, kUpY), per(L.m, kUpZ)), dim3(kUpThreads), 0, st, L.m,
                     kOmegaC, L.cst, rhs, a, c, b);
  std::swap(a, b);
  for (int k = 1; k < T->nu; ++k) {
    hipLaunchKernelGGL(k_coarse_sweep, dim3(nb(v)), dim3(kB), 0, st, L.m, kOmegaC, L.cst, rhs, a, b);
    std::swap(a, b);
  }
  return a;
}

}  // namespace

gdx_problem *twogrid_problem(gdx_nn *nn) { return tg_of(nn) ? tg_of(nn)->prob : nullptr; }

int twogrid_export_coarse(gdx_nn *nn, double *h) {
  TwoGrid *T = tg_of(nn);
  const int64_t v = (int64_t)T->n * T->n * T->n;
  hipStream_t st = T->prob->ctx->stream;
  if (hipMemcpyAsync(h, T->cst, 27 * v * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return GDX_ERR_HIP;
  return GDX_OK;
}

// level l of the V-cycle: its cell count m, and (h != NULL) its stencil [27][m^3]
int twogrid_export_level(gdx_nn *nn, int l, int *m, double *h) {
  TwoGrid *T = tg_of(nn);
  if (l < 0 || l >= (int)T->lv.size()) return GDX_ERR_ARG;
  const Level &L = T->lv[l];
  *m = L.m;
  if (!h) return GDX_OK;
  const int64_t v = (int64_t)L.m * L.m * L.m;
  hipStream_t st = T->prob->ctx->stream;
  if (hipMemcpyAsync(h, L.cst, 27 * v * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return GDX_ERR_HIP;
  return GDX_OK;
}

void twogrid_options(gdx_nn *nn, int sweeps, bool use_net) {
  if (TwoGrid *T = tg_of(nn)) {
    T->sweeps = sweeps;
    T->use_net = use_net;
  }
}

void twogrid_multigrid(gdx_nn *nn, bool on, int nu) {
  if (TwoGrid *T = tg_of(nn)) {
    T->mg = on;
    T->nu = nu;
  }
}

int twogrid_levels(gdx_nn *nn) {
  TwoGrid *T = tg_of(nn);
  return T ? (int)T->lv.size() : 0;
}

void twogrid_free(gdx_nn *nn) {
  TwoGrid *T = tg_of(nn);
  if (!T) return;
  mg_free(T);
  void *ptrs[] = {T->gid_node, T->flat, T->dlat, T->t1, T->t2, T->t3, T->rho, T->red, T->ec, T->ec2, T->tgt,
                  T->fst, T->cst, T->rc, T->ca, T->cb, T->lat};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  delete T;
  nn->tg = nullptr;
}

// the fine matrix's current values as a stencil on the lattice
static int fine_stencil(TwoGrid *T, hipStream_t st) {
  const long long *rs = nullptr;
  const int *rl = nullptr, *cg = nullptr;
  if (int rc = solve_csr_view(T->prob, &rs, &rl, &cg)) return rc;
  hipLaunchKernelGGL(k_fine_stencil, dim3((unsigned)std::max(1, (T->ng + kFsRows - 1) / kFsRows)), dim3(kB), 0, st,
                     T->ng, T->nf, rs, rl, cg, T->prob->dev.values, T->gid_node, T->fst);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

static int attach(gdx_nn *nn, gdx_problem *p) {
  nn::Net &N = nn->net;
  const int n = N.n;
  hipStream_t st = p->ctx->stream;
  TwoGrid *T = tg_of(nn);
  if (T && T->prob != p) {
    twogrid_free(nn);
    T = nullptr;
  }
  const int nf = 2 * n + 1;
  const int64_t v = (int64_t)n * n * n, nfl = (int64_t)nf * nf * nf;
  if (!T) {
    T = new TwoGrid;
    nn->tg = T;
    T->prob = p;
    T->n = n;
    T->nf = nf;
    T->ng = (int)p->ngdofs;
    // free global id -> fine lattice node (the problem's lattice: nf = 2n + 1
    // nodes per direction), built on the device when the numbering is there
    std::vector<long long> gid_node(p->dev_numbering ? 0 : std::max<int64_t>(p->ngdofs, 1), 0);
    for (const Part &P : p->P)
      for (int64_t i = 0; i < P.n_ldofs && !p->dev_numbering; ++i) {
        const int64_t l = P.ldof_lnode[i];
        const int64_t g0 = P.loc_lo[0] + l % P.lnn[0];
        const int64_t g1 = P.loc_lo[1] + (l / P.lnn[0]) % P.lnn[1];
        const int64_t g2 = P.loc_lo[2] + l / (P.lnn[0] * P.lnn[1]);
        gid_node[P.ldof_gid[i]] = g0 + (int64_t)nf * (g1 + (int64_t)nf * g2);
      }
    const size_t gsz = std::max<int64_t>(p->ngdofs, 1) * sizeof(double);
    bool ok = dev_malloc(reinterpret_cast<void **>(&T->gid_node), std::max<int64_t>(p->ngdofs, 1) * sizeof(long long)) ==
                  hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->flat), nfl * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->dlat), nfl * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->t1), gsz) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->t2), gsz) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->t3), gsz) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->rho), v * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->red), (kS + 16) * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->ec), v * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->ec2), v * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->tgt), v * sizeof(float)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->fst), 27 * nfl * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->cst), 27 * v * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->rc), v * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->ca), v * sizeof(double)) == hipSuccess &&
              dev_malloc(reinterpret_cast<void **>(&T->cb), v * sizeof(double)) == hipSuccess;
    if (!ok) return GDX_ERR_ALLOC;
    // the entries of absent neighbours stay zero: one matrix pattern for as long as the attachment lasts
    if (hipMemsetAsync(T->fst, 0, 27 * nfl * sizeof(double), st) != hipSuccess) return GDX_ERR_HIP;
    if (p->dev_numbering ? gid_node_device(p, T->gid_node) != GDX_OK
                         : hipMemcpy(T->gid_node, gid_node.data(), gid_node.size() * sizeof(long long),
                                     hipMemcpyHostToDevice) != hipSuccess)
      return GDX_ERR_HIP;
  }
  int ng = 0;
  int rc = solve_dinv(p, &T->dinv, &ng);
  if (rc) return rc;
  (void)hipMemsetAsync(T->dlat, 0, nfl * sizeof(double), st);
  hipLaunchKernelGGL(k_scatter, dim3(nb(T->ng)), dim3(kB), 0, st, T->ng, T->gid_node, T->dinv, T->dlat);
  hipLaunchKernelGGL(k_input1, dim3(nb(v)), dim3(kB), 0, st, n, nf, p->kp.h[0], T->dlat, N.inp_f + v);
  // fine stencil and the Galerkin coarse operator of the current matrix
  if ((rc = fine_stencil(T, st))) return rc;
  galerkin(n, nf, 0, nfl, T->fst, T->cst, st);
  if ((rc = mg_setup(T, st))) return rc;
  return hipStreamSynchronize(st) == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

// bind the network to a problem's current matrix: transfer maps, the fine
// inverse diagonal on the lattice and the network's diagonal feature.  A binding
// that fails half way is dropped: the next one to the same problem starts anew.
int twogrid_attach(gdx_nn *nn, gdx_problem *p) {
  if (p->D != 3 || p->K != 1) return GDX_ERR_UNSUPPORTED;
  if (p->desc.dir_kind != 1) return GDX_ERR_UNSUPPORTED;
  for (int d = 0; d < 3; ++d)
    if (p->kp.ncells[d] != 2 * nn->net.n) return GDX_ERR_ARG;
  const int rc = attach(nn, p);
  if (rc) {
    (void)hipStreamSynchronize(p->ctx->stream);
    (void)hipGetLastError();  // an allocation's, seen already
    twogrid_free(nn);
  }
  return rc;
}

// the coarse correction of the fine residual s (global-id order, or on the
// lattice): its prolongation in T->flat
static int coarse_correction(gdx_nn *nn, TwoGrid *T, const double *s, bool lattice, double *flat, hipStream_t st) {
  nn::Net &N = nn->net;
  const int64_t nfl = (int64_t)T->nf * T->nf * T->nf;
  const bool mg = T->mg && T->lv.size() > 1;
  make_input(nn, T, s, st, T->use_net, lattice, mg && !T->use_net ? T->lv[0].e : nullptr);
  if (T->use_net) {
    int rc = N.forward_dev();
    if (rc) return rc;
  }
  const int64_t v = (int64_t)T->n * T->n * T->n;
  if (mg && !T->use_net) {  // from the zero guess: the V-cycle on rc itself
    const double *d = vcycle(T, 0, T->rc, st);
    hipLaunchKernelGGL(k_prolong_d, dim3(nb(nfl)), dim3(kB), 0, st, T->n, T->nf, d, flat);
    return GDX_OK;
  }
  hipLaunchKernelGGL(k_out_to_coarse, dim3(nb(v)), dim3(kB), 0, st, T->n, N.out, T->red + kS, T->use_net ? 1 : 0,
                     T->ca);
  if (T->use_net) {
    // the network's direction, scaled to minimise the coarse energy error:
    // a1 = (ec.rc) / (ec.Ac ec)
    hipLaunchKernelGGL(k_coarse_apply, dim3(nb(v)), dim3(kB), 0, st, T->n, T->cst, T->ca, T->cb);
    hipLaunchKernelGGL(k_dot2p, dim3(kRed), dim3(kB), 0, st, (int)v, T->ca, T->rc, T->ca, T->cb, T->red);
    hipLaunchKernelGGL(k_alpha, dim3(1), dim3(kB), 0, st, T->red, T->red + kS + 6);
    hipLaunchKernelGGL(k_scale_by, dim3(nb(v)), dim3(kB), 0, st, v, T->red + kS + 6, T->ca);
  }
  double *ea = T->ca, *eb = T->cb;
  if (mg) {
    // V-cycle on the coarse residual of the network's guess
    const Level &L = T->lv[0];
    hipLaunchKernelGGL(k_resid, dim3(nb(v)), dim3(kB), 0, st, T->n, T->cst, T->rc, ea, L.rhs);
    hipLaunchKernelGGL(k_sweep0, dim3(nb(v)), dim3(kB), 0, st, T->n, kOmegaC, T->cst, L.rhs, L.e);
    const double *d = vcycle(T, 0, L.rhs, st);
    hipLaunchKernelGGL(k_add, dim3(nb(v)), dim3(kB), 0, st, (int)v, ea, d);
  } else {
    for (int k = 0; k < T->sweeps; ++k) {
      hipLaunchKernelGGL(k_coarse_sweep, dim3(nb(v)), dim3(kB), 0, st, T->n, kOmegaC, T->cst, T->rc, ea, eb);
      std::swap(ea, eb);
    }
  }
  hipLaunchKernelGGL(k_prolong_d, dim3(nb(nfl)), dim3(kB), 0, st, T->n, T->nf, ea, flat);
  return GDX_OK;
}

// z += alpha c + w D^-1 (s - alpha Ac), alpha the energy-optimal step along c
static void coarse_step(TwoGrid *T, int n, const double *dinv, const double *s, const double *c, const double *ac,
                        double *z, hipStream_t st) {
  hipLaunchKernelGGL(k_dot2p, dim3(kRed), dim3(kB), 0, st, n, c, s, c, ac, T->red);
  hipLaunchKernelGGL(k_alpha, dim3(1), dim3(kB), 0, st, T->red, T->red + kS + 5);
  hipLaunchKernelGGL(k_coarse_post, dim3(nb(n)), dim3(kB), 0, st, n, kOmega, T->red + kS + 5, dinv, s, c, ac, z);
}

// z = M r (device vectors in global-id order)
int twogrid_apply(void *ctx, const double *r, double *z, hipStream_t st) {
  gdx_nn *nn = reinterpret_cast<gdx_nn *>(ctx);
  TwoGrid *T = tg_of(nn);
  if (!T) return GDX_ERR_STATE;
  gdx_problem *p = T->prob;
  const int ng = T->ng;
  hipLaunchKernelGGL(k_jacobi0, dim3(nb(ng)), dim3(kB), 0, st, ng, kOmega, T->dinv, r, z);
  solve_spmv_dev(p, z, T->t1, st);
  hipLaunchKernelGGL(k_rminus, dim3(nb(ng)), dim3(kB), 0, st, ng, r, T->t1);
  if (int rc = coarse_correction(nn, T, T->t1, false, T->flat, st)) return rc;
  hipLaunchKernelGGL(k_gather, dim3(nb(ng)), dim3(kB), 0, st, ng, T->gid_node, T->flat, T->t2);  // c
  solve_spmv_dev(p, T->t2, T->t3, st);                                                             // A c
  coarse_step(T, ng, T->dinv, T->t1, T->t2, T->t3, z, st);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

// The flexible CG on the fine lattice: its vectors hold every lattice node
// (boundary nodes zero), so neither the transfers nor the products permute.
// lattice vectors in T->lat
enum { kLx, kLr, kLz, kLp, kLq, kLt1, kLt2, kLt3, kLdinv, kLcount };

struct LatticeView {
  gdx_nn *nn;
  TwoGrid *T;
  int n, nblk;
  double *v[kLcount], *part;
};

static LatticeView lattice_view(void *ctx) {
  LatticeView L{};
  L.nn = reinterpret_cast<gdx_nn *>(ctx);
  L.T = tg_of(L.nn);
  if (!L.T || !L.T->lat) return L;
  L.n = L.T->nf * L.T->nf * L.T->nf;
  L.nblk = (int)nb(L.n);
  for (int k = 0; k < kLcount; ++k) L.v[k] = L.T->lat + (size_t)k * L.n;
  L.part = L.T->lat + (size_t)kLcount * L.n;
  return L;
}

static int lattice_begin(void *ctx, const double *r, bool current, hipStream_t st) {
  const LatticeView L = lattice_view(ctx);
  if (!L.n) return GDX_ERR_STATE;
  TwoGrid *T = L.T;
  const size_t bytes = (size_t)L.n * sizeof(double);
  if (!current)
    if (int rc = fine_stencil(T, st)) return rc;
  // boundary nodes zero: x's, r's and D^-1's here, and with them every other vector's
  if (hipMemsetAsync(T->asym, 0, sizeof(int), st) != hipSuccess ||
      hipMemsetAsync(L.v[kLx], 0, bytes, st) != hipSuccess || hipMemsetAsync(L.v[kLr], 0, bytes, st) != hipSuccess ||
      hipMemsetAsync(L.v[kLdinv], 0, bytes, st) != hipSuccess)
    return GDX_ERR_HIP;
  hipLaunchKernelGGL(k_asymmetric, dim3(L.nblk), dim3(kB), 0, st, T->nf, T->fst, T->asym);
  hipLaunchKernelGGL(k_scatter, dim3(nb(T->ng)), dim3(kB), 0, st, T->ng, T->gid_node, T->dinv, L.v[kLdinv]);
  hipLaunchKernelGGL(k_scatter, dim3(nb(T->ng)), dim3(kB), 0, st, T->ng, T->gid_node, r, L.v[kLr]);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

// z = M r after z = w D^-1 r, with the partials of z.q and r.r
static int lattice_precondition(const LatticeView &L, hipStream_t st) {
  TwoGrid *T = L.T;
  double *t1 = L.v[kLt1], *t2 = L.v[kLt2], *t3 = L.v[kLt3], *alpha = T->red + kS + 5;
  const dim3 gp(8 * ((L.nblk + 7) / 8)), g(L.nblk), b(kB);
  hipLaunchKernelGGL(k_lattice_product<true>, gp, b, 0, st, T->nf, 1, T->fst, T->asym, L.v[kLz], L.v[kLr], t1, nullptr);
  if (int rc = coarse_correction(L.nn, T, t1, true, t2, st)) return rc;
  hipLaunchKernelGGL(k_lattice_product<false>, gp, b, 0, st, T->nf, 0, T->fst, T->asym, t2, t1, t3, L.part);
  hipLaunchKernelGGL(k_sum2<true>, dim3(1), dim3(1024), 0, st, L.part, L.nblk, alpha);
  hipLaunchKernelGGL(k_lattice_post, g, b, 0, st, L.n, kOmega, alpha, L.v[kLdinv], t1, t2, t3, L.v[kLq], L.v[kLr],
                     L.v[kLz], L.part);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

static int lattice_first(void *ctx, hipStream_t st) {
  const LatticeView L = lattice_view(ctx);
  if (!L.n) return GDX_ERR_STATE;
  hipLaunchKernelGGL(k_jacobi0, dim3(L.nblk), dim3(kB), 0, st, L.n, kOmega, L.v[kLdinv], L.v[kLr], L.v[kLz]);
  if (hipMemsetAsync(L.v[kLq], 0, (size_t)L.n * sizeof(double), st) != hipSuccess) return GDX_ERR_HIP;
  if (int rc = lattice_precondition(L, st)) return rc;
  return hipMemcpyAsync(L.v[kLp], L.v[kLz], (size_t)L.n * sizeof(double), hipMemcpyDeviceToDevice, st) == hipSuccess
             ? GDX_OK
             : GDX_ERR_HIP;
}

static int lattice_iterate(void *ctx, double *sc, hipStream_t st) {
  const LatticeView L = lattice_view(ctx);
  if (!L.n) return GDX_ERR_STATE;
  TwoGrid *T = L.T;
  const dim3 gp(8 * ((L.nblk + 7) / 8)), g(L.nblk), b(kB);
  hipLaunchKernelGGL(k_lattice_product<false>, gp, b, 0, st, T->nf, 0, T->fst, T->asym, L.v[kLp], L.v[kLr], L.v[kLq],
                     L.part);
  hipLaunchKernelGGL(k_sum2<false>, dim3(1), dim3(1024), 0, st, L.part, L.nblk, sc);
  hipLaunchKernelGGL(k_lattice_update, g, b, 0, st, L.n, kOmega, sc, L.v[kLdinv], L.v[kLp], L.v[kLq], L.v[kLx],
                     L.v[kLr], L.v[kLz]);
  if (int rc = lattice_precondition(L, st)) return rc;
  hipLaunchKernelGGL(k_sum2<false>, dim3(1), dim3(1024), 0, st, L.part, L.nblk, sc + 2);
  hipLaunchKernelGGL(k_lattice_dir, g, b, 0, st, L.n, sc, L.v[kLz], L.v[kLp]);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

static void lattice_end(void *ctx, double *x, hipStream_t st) {
  const LatticeView L = lattice_view(ctx);
  hipLaunchKernelGGL(k_gather, dim3(nb(L.T->ng)), dim3(kB), 0, st, L.T->ng, L.T->gid_node, L.v[kLx], x);
}

FpcgPrec twogrid_prec(gdx_nn *nn, bool current) {
  FpcgPrec p{};
  p.apply = twogrid_apply;
  p.ctx = nn;
  TwoGrid *T = tg_of(nn);
  const int64_t nfl = T ? (int64_t)T->nf * T->nf * T->nf : 0;
  if (!T || nfl >= (int64_t)1 << 30) return p;  // 32-bit node ids in the kernels
  if (!T->lat && dev_malloc(reinterpret_cast<void **>(&T->lat), (kLcount * nfl + 2 * nb(nfl) + 1) * sizeof(double)) !=
                     hipSuccess) {
    (void)hipGetLastError();
    T->lat = nullptr;  // no room: the products from the CSR rows, in global-id order
  }
  if (T->lat) {
    T->asym = reinterpret_cast<int *>(T->lat + kLcount * nfl + 2 * nb(nfl));
    p.begin = lattice_begin;
    p.first = lattice_first;
    p.iterate = lattice_iterate;
    p.end = lattice_end;
    p.current = current;
  }
  return p;
}

// one training step on a fresh sample; loss (relative squared error) to *loss
int twogrid_train_step(gdx_nn *nn, uint64_t seed, float lr, int smooth_passes, float *loss) {
  TwoGrid *T = tg_of(nn);
  if (!T) return GDX_ERR_STATE;
  nn::Net &N = nn->net;
  gdx_problem *p = T->prob;
  hipStream_t st = p->ctx->stream;
  const int n = T->n, ng = T->ng;
  const int64_t v = (int64_t)n * n * n, nfl = (int64_t)T->nf * T->nf * T->nf;
  // smooth random coarse error, unit rms
  hipLaunchKernelGGL(k_coarse_noise, dim3(nb(v)), dim3(kB), 0, st, n, seed, T->ec);
  const dim3 gbox((n + kBoxX - 1) / kBoxX, (n + kBoxY - 1) / kBoxY, (n + kBoxZ - 1) / kBoxZ);
  for (int k = 0; k < smooth_passes;) {
    const int left = smooth_passes - k, now = left < kBoxPasses ? left : kBoxPasses;
    hipLaunchKernelGGL(now == 3 ? k_box<3> : now == 2 ? k_box<2> : k_box<1>, gbox, dim3(kBoxThreads), 0, st, n, T->ec,
                       T->ec2);
    std::swap(T->ec, T->ec2);
    k += now;
  }
  // r = A P ec
  hipLaunchKernelGGL(k_ec_to_float, dim3(nb(v)), dim3(kB), 0, st, v, T->ec, N.out);
  hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, st, T->red + kS + 2, 1.0);  // unit scale: P ec itself
  hipLaunchKernelGGL(k_prolong, dim3(nb(nfl)), dim3(kB), 0, st, n, T->nf, N.out, T->red + kS + 2, T->flat);
  hipLaunchKernelGGL(k_gather, dim3(nb(ng)), dim3(kB), 0, st, ng, T->gid_node, T->flat, T->t2);
  solve_spmv_dev(p, T->t2, T->t1, st);
  // input from r, target ec / s
  make_input(nn, T, T->t1, st);
  hipLaunchKernelGGL(k_target, dim3(nb(v)), dim3(kB), 0, st, v, T->ec, T->red + kS, T->tgt);
  int rc = N.forward_dev();
  if (rc) return rc;
  // scale-free loss 1 - cos^2(N, ec): the preconditioner rescales the
  // network's output optimally, so only its direction matters
  hipLaunchKernelGGL(k_dot3f, dim3(kRed), dim3(kB), 0, st, v, N.out, T->tgt, T->red);
  hipLaunchKernelGGL(k_finish3, dim3(1), dim3(kB), 0, st, T->red, T->red + kS + 8);
  hipLaunchKernelGGL(k_cos_grad, dim3(nb(v)), dim3(kB), 0, st, v, N.out, T->tgt, T->red + kS + 8, N.dout);
  if ((rc = N.backward_dev(false))) return rc;
  if ((rc = N.adam_step(lr, 1.0f))) return rc;
  double h = 0.0;
  if (hipMemcpyAsync(&h, T->red + kS + 11, sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return GDX_ERR_HIP;
  if (loss) *loss = (float)h;
  return GDX_OK;
}

// per-device address of the no-alloc staging array, set once with that device current
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_noalloc_mu;
double *g_noalloc_ptr[kMaxDevices] = {};
}  // namespace

int noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return GDX_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (g_noalloc_ptr[device]) return GDX_OK;
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess || cur != device) return GDX_ERR_STATE;
  void *ptr = nullptr;
  if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return GDX_ERR_HIP;
  g_noalloc_ptr[device] = static_cast<double *>(ptr);
  return GDX_OK;
}

double *noalloc_scratch(int device) {
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  return device >= 0 && device < kMaxDevices ? g_noalloc_ptr[device] : nullptr;
}

}  // namespace gdx

// ---------------------------------------------------------------------------
// C ABI (include/gdx.h)
// ---------------------------------------------------------------------------
extern "C" {

int gdx_nn_attach(gdx_nn *nn, gdx_problem *prob) {
  if (!nn || !prob) {
    gdx::set_error("NULL argument");
    return GDX_ERR_ARG;
  }
  if (!nn->ctx) {
    gdx::set_error("the network's context was finalized");
    return GDX_ERR_STATE;
  }
  if (!prob->symbolic_done || !prob->ctx) {
    gdx::set_error("the problem needs gdx_symbolic and a device context");
    return GDX_ERR_STATE;
  }
  if (prob->ctx != nn->ctx) {  // the network's kernels run on its context's stream
    gdx::set_error("network and problem belong to different contexts");
    return GDX_ERR_ARG;
  }
  if (hipSetDevice(prob->ctx->device) != hipSuccess) return GDX_ERR_HIP;
  const gdx::FaultScope fault_scope;
  int rc = gdx::twogrid_attach(nn, prob);
  if (rc == GDX_ERR_UNSUPPORTED) gdx::set_error("the two-grid preconditioner is built for 3D Q1 with Dirichlet data on the whole boundary");
  else if (rc == GDX_ERR_ARG) gdx::set_error("the problem must have 2n x 2n x 2n cells for a network grid of n^3");
  else if (rc) gdx::set_error("attaching the network failed");
  return rc;
}

int gdx_nn_train_step(gdx_nn *nn, uint64_t seed, float lr, int32_t smooth_passes, float *loss) {
  if (!nn || !(lr > 0.0f) || smooth_passes < 0 || smooth_passes > 1000) {
    gdx::set_error("invalid argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg || !nn->ctx) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  if (hipSetDevice(nn->ctx->device) != hipSuccess) return GDX_ERR_HIP;
  return gdx::twogrid_train_step(nn, seed, lr, smooth_passes, loss);
}

int gdx_nn_set_options(gdx_nn *nn, int32_t coarse_sweeps, int32_t use_network) {
  if (!nn || coarse_sweeps < 0 || coarse_sweeps > 64) {
    gdx::set_error("invalid argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  gdx::twogrid_options(nn, coarse_sweeps, use_network != 0);
  return GDX_OK;
}

int gdx_nn_coarse_operator(gdx_nn *nn, double *stencil) {
  if (!nn || !stencil) {
    gdx::set_error("NULL argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg || !nn->ctx) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  if (hipSetDevice(nn->ctx->device) != hipSuccess) return GDX_ERR_HIP;
  return gdx::twogrid_export_coarse(nn, stencil);
}

int gdx_nn_set_multigrid(gdx_nn *nn, int32_t enable, int32_t nu, int32_t *levels) {
  if (!nn || nu < 1 || nu > 8) {
    gdx::set_error("invalid argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  gdx::twogrid_multigrid(nn, enable != 0, nu);
  if (levels) *levels = gdx::twogrid_levels(nn);
  return GDX_OK;
}

int gdx_nn_level_operator(gdx_nn *nn, int32_t level, int32_t *m, double *stencil) {
  if (!nn || !m) {
    gdx::set_error("NULL argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg || !nn->ctx) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  if (hipSetDevice(nn->ctx->device) != hipSuccess) return GDX_ERR_HIP;
  int mm = 0;
  const int rc = gdx::twogrid_export_level(nn, level, &mm, stencil);
  if (rc == GDX_ERR_ARG) gdx::set_error("no such level");
  *m = mm;
  return rc;
}

int gdx_nn_apply(gdx_nn *nn, const double *r, double *z) {
  if (!nn || !r || !z) {
    gdx::set_error("NULL argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg || !nn->ctx) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  if (hipSetDevice(nn->ctx->device) != hipSuccess) return GDX_ERR_HIP;
  gdx_problem *p = gdx::twogrid_problem(nn);
  const size_t bytes = std::max<int64_t>(p->ngdofs, 1) * sizeof(double);
  double *rd = nullptr, *zd = nullptr;
  hipStream_t st = p->ctx->stream;
  if (hipMalloc(reinterpret_cast<void **>(&rd), bytes) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&zd), bytes) != hipSuccess) {
    (void)hipFree(rd);
    return GDX_ERR_ALLOC;
  }
  int rc = hipMemcpyAsync(rd, r, p->ngdofs * sizeof(double), hipMemcpyHostToDevice, st) == hipSuccess ? GDX_OK
                                                                                                          : GDX_ERR_HIP;
  if (!rc) rc = gdx::twogrid_apply(nn, rd, zd, st);
  if (!rc && (hipMemcpyAsync(z, zd, p->ngdofs * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
              hipStreamSynchronize(st) != hipSuccess))
    rc = GDX_ERR_HIP;
  (void)hipFree(rd);
  (void)hipFree(zd);
  return rc;
}

int gdx_nn_apply_noalloc(gdx_nn *nn, const double *r, double *z) {
  if (!nn || !r || !z) {
    gdx::set_error("NULL argument");
    return GDX_ERR_ARG;
  }
  if (!nn->tg || !nn->ctx) {
    gdx::set_error("gdx_nn_attach has not run");
    return GDX_ERR_STATE;
  }
  const int dev = nn->ctx->device;
  if (hipSetDevice(dev) != hipSuccess) return GDX_ERR_HIP;
  gdx_problem *p = gdx::twogrid_problem(nn);
  const int64_t n = p->ngdofs;
  if (2 * n > (int64_t)kNoAllocDoubles) {
    gdx::set_error("gdx_nn_apply_noalloc: the problem has more than 2,097,152 free dofs (the staging limit)");
    return GDX_ERR_ARG;
  }
  int rc = gdx::noalloc_setup(dev);  // normally done by gdx_init on this device
  double *base = gdx::noalloc_scratch(dev);
  if (rc || !base) {
    gdx::set_error("gdx_nn_apply_noalloc: no device address for the staging array");
    return rc ? rc : GDX_ERR_HIP;
  }
  // r is copied in whole and z written in whole: nothing has to start at zero
  double *rd = base, *zd = base + n;
  hipStream_t st = p->ctx->stream;
  rc = n == 0 || hipMemcpyAsync(rd, r, n * sizeof(double), hipMemcpyHostToDevice, st) == hipSuccess ? GDX_OK
                                                                                                   : GDX_ERR_HIP;
  if (!rc) rc = gdx::twogrid_apply(nn, rd, zd, st);
  if (!rc && ((n > 0 && hipMemcpyAsync(z, zd, n * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess) ||
              hipStreamSynchronize(st) != hipSuccess))
    rc = GDX_ERR_HIP;
  if (rc) gdx::set_error("gdx_nn_apply_noalloc failed");
  return rc;
}

int gdx_fpcg(gdx_problem *prob, gdx_nn *nn, const double *rhs, double rtol, int32_t maxiter, double *xsol,
             int32_t *iters, double *relres, double *ms, int32_t *fellback) {
  if (!prob || !(rtol > 0.0) || maxiter < 1) {
    gdx::set_error("invalid argument");
    return GDX_ERR_ARG;
  }
  if (!prob->symbolic_done || !prob->ctx) {
    gdx::set_error("the problem needs gdx_symbolic and a device context");
    return GDX_ERR_STATE;
  }
  if (nn && (!nn->tg || gdx::twogrid_problem(nn) != prob)) {
    gdx::set_error("the network is not attached to this problem (gdx_nn_attach)");
    return GDX_ERR_STATE;
  }
  if (hipSetDevice(prob->ctx->device) != hipSuccess) return GDX_ERR_HIP;
  const gdx::FaultScope fault_scope;
  const gdx::FpcgPrec pr = nn ? gdx::twogrid_prec(nn, false) : gdx::FpcgPrec{};
  int it = 0, fb = 0;
  int rc = gdx::solve_fpcg(prob, nn ? &pr : nullptr, rhs, rtol, maxiter, xsol, &it, relres, ms, &fb);
  if (iters) *iters = it;
  if (fellback) *fellback = fb;
  if (rc) gdx::set_error("flexible PCG failed");
  return rc;
}

}  // extern "C"

