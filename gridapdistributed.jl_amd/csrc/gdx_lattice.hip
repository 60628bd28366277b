// Matrix and RHS kernel of the diffusion form on the uniform box (2D and 3D,
// Q1 and Q2): owner-computes-rows through the lattice of node pairs.
//
// On a Cartesian mesh the entry of row i and column j is a product form,
//   A_ij = sum_q kappa(q) [G1 M2 M3 + M1 G2 M3 + M1 M2 G3](q; i, j),
// and every 1D factor G_d, M_d is symmetric in (i_d, j_d).  So A_ij depends on
// the UNORDERED node pair {i_d, j_d} of each direction only: a Q2 cell has 5
// pairs per direction and 125 distinct values for its 512 stored entries, a Q1
// cell 8 for 27.  A workgroup takes a tile of C1 x C2 x C3 cells' rows:
//   1. kappa at the tile's quadrature points (one cell of halo below) to LDS;
//   2. one thread per (x pair, y pair) contracts the x-y points of each z
//      plane straight from LDS into registers, with the two combined weights
//      G1 M2 + M1 G2 and M1 M2, then contracts z for every z pair and leaves
//      the tile's distinct values in LDS (the pair lattice U);
//   3. each row is a gather: lane <-> position in the CSR row, one LDS read of
//      U at the row's base plus the position's offset (a 16-bit table per
//      position pattern), one store.  Every store instruction writes
//      consecutive doubles of one row.
// kappa constant on each cell (a constant or a cell-wise coefficient) takes the
// same path with one point per cell: the 1D factors are summed over the Gauss
// points first, which is the same quadrature.
//
// Measured against the z-marching kernel that was the default before, whole
// numeric phases: 3D Q2 64^3, Fourier kappa 0.86 -> 0.51 ms (the matrix kernel
// 790 -> 410 us); 3D Q1 131 x 97 x 75, kappa per cell 517 -> 69 us (453 -> 50);
// 2D Q1 256^2 95 -> 13 us (71 -> 9).  The Q2 kernel writes 2.4 TB/s of the 6.7
// that a fill reaches; what is left is latency: at two workgroups per CU the
// LDS contraction (about 40% of a tile's time) hides behind little else.
//
// Tiles are cut on the global node lattice, across part boundaries: the row
// table is laid out on that lattice once, so a row's entry is one load.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "gdx_device.h"
#include "gdx_lattice.h"

namespace gdx {

namespace {

// pairs of one direction: per cell {v,v}, {v,m}, {m,m}, {v,v'}, {m,v'} (Q2) or
// {v,v}, {v,v'} (Q1), preceded by the pairs that the first vertex shares with
// the previous cell.  base(u) + step(parity, s) is the index of {u, u + s}.
template <int K>
struct Pairs {
  static constexpr int PC = K == 2 ? 5 : 2, PRE = K == 2 ? 2 : 1;
  static constexpr int SING = PC - 1;  // single-cell pairs per cell
  __host__ __device__ static constexpr int count(int C) { return PC * C + PRE; }
  __host__ __device__ static constexpr int base(int u) { return PRE + PC * (u / K); }
};

__host__ __device__ inline int pair_step(int K, int par, int s) {
  if (K == 1) return s;
  if (par == 0) return s == 2 ? 3 : s;  // -2, -1 lie in the previous cell
  return s == 0 ? 2 : (s < 0 ? 1 : 4);
}

template <int D_, int K_, int NQ_, int C1_, int C2_, int C3_, int NT_, int L_, bool SPLIT_ = false>
struct LatShape {
  static constexpr int D = D_, K = K_, NQ = NQ_, C1 = C1_, C2 = C2_, C3 = C3_, NT = NT_, L = L_;
  static constexpr bool SPLIT = SPLIT_;
  static constexpr int NW = NT / 64;
  static constexpr int R1 = K * C1, R2 = K * C2, R3 = D == 3 ? K * C3 : 1;
  static constexpr int ROWS = R1 * R2 * R3;
  static constexpr int NP1 = Pairs<K>::count(C1), NP2 = Pairs<K>::count(C2), NP3 = D == 3 ? Pairs<K>::count(C3) : 1;
  static constexpr int NP12 = NP1 * NP2, NU = NP12 * NP3;
  static constexpr int Q1 = NQ * (C1 + 1), Q2 = NQ * (C2 + 1), Q3 = D == 3 ? NQ * (C3 + 1) : 1;
  static constexpr int NKAP = Q1 * Q2 * Q3;
  static constexpr int FPT = (NKAP + NT - 1) / NT;
  static constexpr int S = D == 3 ? (2 * K + 1) * (2 * K + 1) * (2 * K + 1) : (2 * K + 1) * (2 * K + 1);
  static constexpr int PSTR = D == 3 ? (K == 2 ? 128 : 32) : (K == 2 ? 32 : 16);  // pattern table stride
  static constexpr int WPS = D == 3 && NQ > 1 ? (SPLIT ? 6 : 4) : 6;  // waves per SIMD that the registers leave room for
  static_assert(ROWS <= NT, "one thread per row");
  static_assert(PSTR >= S, "one entry per position");
};

// row of the tile in LDS, written and read by the same wave
struct LatRowL {
  long long off;  // byte offset of its first value
  int meta;  // as LatRow
  int ub;    // base of the row in U
};

typedef unsigned UInt2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double quad_swap1(double v) {  // the value of lane ^ 1
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | (long long)hi << 32);
}
__device__ __forceinline__ double quad_swap2(double v) {  // the value of lane ^ 2
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0x4E, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x4E, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | (long long)hi << 32);
}

// index i of a direction's pair order "two-cell pairs first": pair index, its
// number of cells, first region cell and kind there
template <int K>
__device__ __forceinline__ void single_pair(int i, int &pi, int &lc, int &kind) {
  // i-th pair supported on one cell
  if (K == 1) {
    pi = 2 * i, lc = i, kind = 1;
  } else {
    // previous cell's {v,v'}, {m,v'}, then {v,m}, {m,m}, {v,v'}, {m,v'} of every cell
    const int t = i + 2, j = t >> 2, k = t & 3;  // j: region cell; k: 0 {v,m}, 1 {m,m}, 2 {v,v'}, 3 {m,v'}
    pi = 5 * j - 3 + 1 + k;
    lc = j, kind = 1 + k;
  }
}

// place of node (x, y, z) in the row table: x lines, Q2 lines by node parity
// (the rows of one parity that a wave stores together are consecutive)
template <int K, class A>
__device__ __forceinline__ size_t row_at(const A &a, int x, int y, int z) {
  const int n0 = a.pn[0], n1 = a.pn[1], i = K == 2 ? (x & 1) * (n0 >> 1) + (x >> 1) : x;
  return i + (size_t)n0 * (y + (size_t)n1 * z);
}

// cells of tile node u of one direction (region cells), and its local index in the c-th
template <int K>
__device__ __forceinline__ int node_cell(int u) { return K == 1 ? u : (u + 1) / 2; }
template <int K>
__device__ __forceinline__ int node_cells(int u) { return K == 1 ? 2 : ((u & 1) ? 1 : 2); }
template <int K>
__device__ __forceinline__ int node_local(int u, int c) { return K == 1 ? 1 - c : ((u & 1) ? 1 : 2 - 2 * c); }

// the kernel's arguments, read by scalar loads
typedef const __attribute__((address_space(4))) LatArgs *ArgsPtr;
typedef const __attribute__((address_space(4))) LatArgs &ArgsRef;

// z contraction of one (x pair, y pair) for every z pair, constant indices
template <class T, int PZ = 0>
__device__ __forceinline__ void z_pairs(const double (&Y1)[T::Q3], const double (&Y2)[T::Q3], ArgsRef a,
                                        double *__restrict__ u) {
  if constexpr (PZ < T::NP3) {
    constexpr int K = T::K, NQ = T::NQ, PC = Pairs<K>::PC, PRE = Pairs<K>::PRE;
    constexpr int t = PZ - PRE + PC, j = t / PC, k = t % PC;  // j: region cell
    double v = 0.0;
    if constexpr (k == 0) {
      constexpr int last = K == 2 ? 5 : 2;  // {v', v'} of the cell below
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        v = fma(Y1[(j - 1) * NQ + q], a.M[2][last][q], fma(Y2[(j - 1) * NQ + q], a.G[2][last][q], v));
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) v = fma(Y1[j * NQ + q], a.M[2][k][q], fma(Y2[j * NQ + q], a.G[2][k][q], v));
    u[PZ * T::NP12] = v;
    z_pairs<T, PZ + 1>(Y1, Y2, a, u);
  }
}

// One row per wave instruction (Q2, 3D): the rows of one node parity have one
// length; the x lines of four such rows are dealt to the waves in order of that
// length, about as many store instructions to each wave.
template <class T>
struct RowLines {
  static constexpr int LPC = T::C2 * (T::D == 3 ? T::C3 : 1), NL = 8 * LPC;  // lines per parity, lines
  static constexpr int COST = 4 * LPC * 2 + 4 * LPC;  // the first half's lines need two stores a row
  __device__ static int first(int w) {
    const int c = (w * COST + T::NW - 1) / T::NW;
    return c < 8 * LPC ? (c + 1) / 2 : c - 4 * LPC;
  }
  // tile rows 2 g + p1, v2, v3 (g = 0..3) of line l
  __device__ static void line(int l, int &p1, int &v2, int &v3) {
    constexpr unsigned ORDER = 0x76534210u;  // parities (x | y << 1 | z << 2) by number of odd directions
    const int c = (int)(ORDER >> (4 * (l / LPC))) & 7, j = l % LPC;
    p1 = c & 1;
    v2 = 2 * (j % T::C2) + ((c >> 1) & 1);
    v3 = 2 * (j / T::C2) + (c >> 2);
  }
};

// sum_j A_ij uD_j over the neighbours of tile row (u1, u2, u3), node (g0, g1,
// g2), on the mesh boundary: face by face, a node on several at its first
template <class T>
__device__ __forceinline__ double lifting(ArgsRef a, const double *__restrict__ U, int u1, int u2, int u3, int g0,
                                          int g1, int g2) {
  constexpr int K = T::K, D = T::D;
  const int ub = (D == 3 ? Pairs<K>::base(u3) * T::NP12 : 0) + Pairs<K>::base(u2) * T::NP1 + Pairs<K>::base(u1);
  const int g[3] = {g0, g1, g2}, u[3] = {u1, u2, u3}, stride[3] = {1, T::NP1, T::NP12};
  auto coupled = [](int v, int s) { return s >= -K && s <= K && (K == 1 || !(v & 1) || (s != 2 && s != -2)); };
  double acc = 0.0;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    constexpr int E[3][2] = {{1, 2}, {0, 2}, {0, 1}};
    const int e = E[d][0], f = E[d][1];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int s = side ? a.nn[d] - 1 - g[d] : -g[d];
      if (!coupled(u[d], s)) continue;
      const int off = ub + stride[d] * pair_step(K, u[d] & 1, s);
      const double ud = a.dir_coef[0] + a.dir_coef[1 + d] * (a.x0[d] + a.hK[d] * (double)(g[d] + s));
#pragma unroll 1
      for (int se = -K; se <= K; ++se) {
        const int xe = g[e] + se;
        if (!coupled(u[e], se) || xe < 0 || xe >= a.nn[e] || (e < d && (xe == 0 || xe == a.nn[e] - 1))) continue;
        const int offe = off + stride[e] * pair_step(K, u[e] & 1, se);
        const double ue = ud + a.dir_coef[1 + e] * (a.x0[e] + a.hK[e] * (double)xe);
        if constexpr (D == 2) {
          acc = fma(U[offe], ue, acc);
        } else {
#pragma unroll 1
          for (int sf = -K; sf <= K; ++sf) {
            const int xf = g[f] + sf;
            if (!coupled(u[f], sf) || xf < 0 || xf >= a.nn[f] || (f < d && (xf == 0 || xf == a.nn[f] - 1))) continue;
            const double uf = ue + a.dir_coef[1 + f] * (a.x0[f] + a.hK[f] * (double)xf);
            acc = fma(U[offe + stride[f] * pair_step(K, u[f] & 1, sf)], uf, acc);
          }
        }
      }
    }
  }
  return acc;
}

template <class T>
__device__ __forceinline__ void lattice_tile(ArgsRef a, int tile) {
  constexpr int D = T::D, K = T::K, NQ = T::NQ, NT = T::NT;
  constexpr bool LROWS = T::L < 64;  // several rows per wave instruction: their entries go through LDS
  __shared__ double U[T::NU];
  __shared__ double kap[T::NKAP];
  __shared__ double tab[2 * 6 * 3 * 2];  // 1D factors of x and y: [d][kind][q]{G, M}
  __shared__ LatRowL rows[LROWS ? T::ROWS : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int o0 = a.lo[0] + (tile % a.nt[0]) * T::R1, o1 = a.lo[1] + ((tile / a.nt[0]) % a.nt[1]) * T::R2;
  const int o2 = D == 3 ? a.lo[2] + (tile / (a.nt[0] * a.nt[1])) * T::R3 : 0;

  // kappa at the region's points (cells org/K - 1 .. org/K + C - 1, zero outside
  // the mesh) and the entry of the lane's row: every load goes out at once, at a
  // point of the mesh
  const int qs0 = (o0 / K - 1) * NQ, qs1 = (o1 / K - 1) * NQ, qs2 = D == 3 ? (o2 / K - 1) * NQ : 0;
  const int n0 = a.ncell[0] * NQ, n1 = a.ncell[1] * NQ, n2 = D == 3 ? a.ncell[2] * NQ : 1;
  auto clamp = [](int i, int n) { return i < 0 ? 0 : (i < n ? i : n - 1); };
  double kpre[T::FPT];
#pragma unroll
  for (int j = 0; j < T::FPT; ++j) {
    const int i = tid + j * NT;
    const int q0 = qs0 + i % T::Q1, q1 = qs1 + (i / T::Q1) % T::Q2, q2 = qs2 + i / (T::Q1 * T::Q2);
    const size_t qi = clamp(q0, n0) + (size_t)n0 * (clamp(q1, n1) + (size_t)n1 * clamp(q2, n2));
    const bool in = (q0 >= 0) & (q0 < n0) & (q1 >= 0) & (q1 < n1) & (q2 >= 0) & (q2 < n2);
    const double v = NQ == 1 ? (a.W ? a.kconst * a.W[qi] : a.kconst) : a.W[qi];
    kpre[j] = in ? v : 0.0;
  }
  const int l0 = RowLines<T>::first(wave), l1 = RowLines<T>::first(wave + 1);
  int u1, u2, u3;  // the lane's row: tile row (u1, u2, u3)
  bool mine;
  if constexpr (LROWS) {
    u1 = tid % T::R1, u2 = (tid / T::R1) % T::R2, u3 = tid / (T::R1 * T::R2);
    mine = tid < T::ROWS;
  } else {
    int p1;
    mine = lane < 4 * (l1 - l0);
    RowLines<T>::line(mine ? l0 + lane / 4 : l0, p1, u2, u3);
    u1 = 2 * (lane % 4) + p1;
  }
  // 1D factor tables: a per-lane index into the argument would be a memory load each time
  if (tid < 72) {
    const int e = tid & 1, q = (tid >> 1) % 3, k = (tid / 6) % 6, d = tid / 36;
    tab[tid] = e ? a.M[d][k][q] : a.G[d][k][q];
  }
#pragma unroll
  for (int j = 0; j < T::FPT; ++j)
    if (tid + j * NT < T::NKAP) kap[tid + j * NT] = kpre[j];
  __syncthreads();

  // the pair lattice.  Pairs are dealt in four classes (both directions on two
  // cells, one of them, none), so that the cell loops of most waves are uniform.
  // SPLIT: one lane per (pair, cell), the up to four cells of a pair summed
  // across neighbouring lanes: every wave contracts one cell
  constexpr int V1 = T::C1, V2 = T::C2, S1 = T::NP1 - V1, S2 = T::NP2 - V2;
  constexpr int M4 = T::SPLIT ? 4 : 1, M2 = T::SPLIT ? 2 : 1;
  constexpr int E0 = V1 * V2 * M4, E1 = E0 + V1 * S2 * M2, E2 = E1 + S1 * V2 * M2, E3 = E2 + S1 * S2;
  static_assert(!T::SPLIT || E3 <= NT, "one lane per (pair, cell)");
  for (int t = tid; t < E3; t += NT) {
    int i1, i2, c1 = 0, c2 = 0;  // index among the direction's two-cell or one-cell pairs; the lane's cell
    const bool d1 = t < E1, d2 = t < E0 || (t >= E1 && t < E2);
    if (t < E0) {
      const int p = t / M4;
      i1 = p % V1, i2 = p / V1;
      c1 = t & 1, c2 = (t >> 1) & 1;
    } else if (t < E1) {
      const int p = (t - E0) / M2;
      i1 = p % V1, i2 = p / V1;
      c1 = t & 1;
    } else if (t < E2) {
      const int p = (t - E1) / M2;
      i1 = p % S1, i2 = p / S1;
      c2 = t & 1;
    } else {
      i1 = (t - E2) % S1, i2 = (t - E2) / S1;
    }
    constexpr int LASTK = K == 2 ? 5 : 2;  // kind {v', v'}
    int pi1, pi2, lc1, lc2, kd1 = 0, kd2 = 0;
    if (d1) pi1 = Pairs<K>::PRE + Pairs<K>::PC * i1, lc1 = i1;
    else single_pair<K>(i1, pi1, lc1, kd1);
    if (d2) pi2 = Pairs<K>::PRE + Pairs<K>::PC * i2, lc2 = i2;
    else single_pair<K>(i2, pi2, lc2, kd2);
    double Y1[T::Q3], Y2[T::Q3];
#pragma unroll
    for (int q = 0; q < T::Q3; ++q) Y1[q] = Y2[q] = 0.0;
    auto cell = [&](int c1, int c2) {
      const double *t1 = tab + (d1 ? (c1 ? 0 : LASTK) : kd1) * 6;
      const double *t2 = tab + 36 + (d2 ? (c2 ? 0 : LASTK) : kd2) * 6;
      const double *kr = kap + (lc2 + c2) * NQ * T::Q1 + (lc1 + c1) * NQ;
      double G1[NQ], M1[NQ];
#pragma unroll
      for (int x = 0; x < NQ; ++x) G1[x] = t1[2 * x], M1[x] = t1[2 * x + 1];
#pragma unroll 1
      for (int y = 0; y < NQ; ++y, kr += T::Q1, t2 += 2) {
        const double G2 = t2[0], M2 = t2[1];
        double w1[NQ], w2[NQ];
#pragma unroll
        for (int x = 0; x < NQ; ++x) w1[x] = fma(G1[x], M2, M1[x] * G2), w2[x] = M1[x] * M2;
#pragma unroll
        for (int q3 = 0; q3 < T::Q3; ++q3)
#pragma unroll
          for (int x = 0; x < NQ; ++x) {
            const double k = kr[q3 * T::Q2 * T::Q1 + x];
            Y1[q3] = fma(k, w1[x], Y1[q3]);
            if constexpr (D == 3) Y2[q3] = fma(k, w2[x], Y2[q3]);
          }
      }
    };
    bool leader = true;
    if constexpr (T::SPLIT) {
      cell(c1, c2);
      if (wave * 64 < E2) {
        const bool two = t < E2, four = t < E0;
        leader = four ? (t & 3) == 0 : !two || !(t & 1);
#pragma unroll
        for (int q = 0; q < T::Q3; ++q) {
          const double a1 = quad_swap1(Y1[q]), a2 = quad_swap1(Y2[q]);
          Y1[q] += two ? a1 : 0.0;
          Y2[q] += two ? a2 : 0.0;
        }
        if (wave * 64 < E0) {
          static_assert(!T::SPLIT || E0 % 64 == 0, "whole waves of four-cell pairs");
#pragma unroll
          for (int q = 0; q < T::Q3; ++q) Y1[q] += quad_swap2(Y1[q]), Y2[q] += quad_swap2(Y2[q]);
        }
      }
    } else {
#pragma unroll 1
      for (c2 = 0; c2 < (d2 ? 2 : 1); ++c2)
#pragma unroll 1
        for (c1 = 0; c1 < (d1 ? 2 : 1); ++c1) cell(c1, c2);
    }
    double *u = U + pi2 * T::NP1 + pi1;
    if (leader) {
      if constexpr (D == 3) z_pairs<T>(Y1, Y2, a, u);
      else u[0] = Y1[0];
    }
  }
  LatRow row{0, 0, -1};
  if (mine) row = a.rows[row_at<K>(a, o0 + u1, o1 + u2, o2 + u3)];
  if constexpr (LROWS)
    if (mine)
      rows[tid] = LatRowL{row.off, row.meta,
                          Pairs<K>::base(u3) * (D == 3 ? T::NP12 : 0) + Pairs<K>::base(u2) * T::NP1 + Pairs<K>::base(u1)};
  __syncthreads();

  if constexpr (!LROWS) {
    static_assert(LROWS || (K == 2 && D == 3 && T::C1 == 4), "lines of four rows");
    constexpr int G = 4;
    const int off_lo = (int)row.off, off_hi = (int)(row.off >> 32);
    // Every row is stored through a buffer resource of exactly its length, so
    // the lanes beyond it need no branch (a chunk's offset is part of the vector
    // offset: the scalar offset does not count in the bounds check); the offset
    // tables of the next line go out before this line's stores, which they then
    // never wait for.
    auto lines = [&](int la, int lb, auto chunks) {
      constexpr int CH = decltype(chunks)::value;  // 64-entry chunks of the longest row
      if (la >= lb) return;
      int dl[G][CH], nx[G][CH];
      auto offsets = [&](int l, int (&d)[G][CH]) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int mt = __builtin_amdgcn_readlane(row.meta, 4 * (l - l0) + g);
          const uint16_t *dt = a.delta + (size_t)(mt >> 9) * T::PSTR + lane;
#pragma unroll
          for (int c = 0; c < CH; ++c) d[g][c] = (int16_t)dt[64 * c];
        }
      };
      offsets(la, nx);
#pragma unroll 1
      for (int l = la; l < lb; ++l) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int c = 0; c < CH; ++c) dl[g][c] = nx[g][c];
        offsets(l + 1 < lb ? l + 1 : l, nx);
        int p1, v2, v3;
        RowLines<T>::line(l, p1, v2, v3);
        const int ub = Pairs<K>::base(v3) * T::NP12 + Pairs<K>::base(v2) * T::NP1 + Pairs<K>::PRE;
        double v[G][CH];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int c = 0; c < CH; ++c) v[g][c] = U[ub + g * Pairs<K>::PC + dl[g][c]];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int at = 4 * (l - l0) + g, mt = __builtin_amdgcn_readlane(row.meta, at);
          const long long off = (long long)(unsigned)__builtin_amdgcn_readlane(off_lo, at) |
                                (long long)__builtin_amdgcn_readlane(off_hi, at) << 32;
          const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
              reinterpret_cast<char *>(a.values) + off, 0, 8 * (mt & 0xFF), 0x00020000);
#pragma unroll
          for (int c = 0; c < CH; ++c)
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(UInt2, v[g][c]), rs, 8 * lane + 512 * c, 0, 0);
        }
      }
    };
    constexpr int H = RowLines<T>::NL / 2;  // the first half's rows are longer than 64 entries
    lines(l0, l1 < H ? l1 : H, std::integral_constant<int, 2>{});
    lines(l0 > H ? l0 : H, l1, std::integral_constant<int, 1>{});
  } else {
    // 64 / L rows per wave instruction, four instructions at a time: their row
    // entries, then their values, then the stores
    constexpr int RPI = 64 / T::L, G = 4, STEP = T::NW * RPI;
    const int sub = lane / T::L, k = lane % T::L;
    int cur = -1, dl = 0;
#pragma unroll 1
    for (int r0 = wave * RPI; r0 < T::ROWS; r0 += G * STEP) {
      LatRowL e[G];
      bool other = false;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int r = r0 + g * STEP + sub;
        e[g] = rows[r < T::ROWS ? r : 0];
        if (r >= T::ROWS) e[g].meta = 0;
        other = other || ((e[g].meta & 0xFF) && e[g].meta != cur);
      }
      int d[G];
      if (__any(other)) {  // another position pattern: its offsets, one wait for the four rows
#pragma unroll
        for (int g = 0; g < G; ++g) d[g] = (int16_t)a.delta[(size_t)(e[g].meta >> 9) * T::PSTR + k];
        cur = e[G - 1].meta;
        dl = d[G - 1];
      } else {
#pragma unroll
        for (int g = 0; g < G; ++g) d[g] = dl;
      }
      double v[G];
#pragma unroll
      for (int g = 0; g < G; ++g) v[g] = U[e[g].ub + d[g]];
#pragma unroll
      for (int g = 0; g < G; ++g)
        if (k < (e[g].meta & 0xFF))
          *reinterpret_cast<double *>(reinterpret_cast<char *>(a.values) + e[g].off + 8 * k) = v[g];
    }
  }
  // b: one lane per row
  if (row.bidx >= 0) {
    const int g[3] = {o0 + u1, o1 + u2, o2 + u3};
    const bool flag = row.meta & 0x100;
    const double lf = flag ? lifting<T>(a, U, u1, u2, u3, g[0], g[1], g[2]) : 0.0;
    if (a.source) {  // the source integral is in b
      if (flag) a.b[row.bidx] -= lf;
    } else {  // f constant: the source integral in closed form
      double v = a.fconst;
#pragma unroll
      for (int d = 0; d < D; ++d)
        v *= K == 2 && (g[d] & 1) ? a.Sv[d][1]
                                  : (g[d] > 0 ? a.Sv[d][K] : 0.0) + (g[d] < a.nn[d] - 1 ? a.Sv[d][0] : 0.0);
      a.b[row.bidx] = v - lf;
    }
  }
}

template <class T>
__global__ __launch_bounds__(T::NT, T::WPS) void k_lattice(const LatArgs, int ntiles) {
  const ArgsPtr args = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();  // the first argument
  // Consecutive blocks are dealt round-robin over the 8 XCDs: each XCD takes
  // whole x lines of tiles (which share their halos in its L2) in turn, another
  // of every eight each time, so the tiles at the mesh boundary, which take
  // longer, spread over all of them
  const int nx = args->nt[0], i = (int)(blockIdx.x / 8), line = (i / nx) * 8 + (int)((blockIdx.x + i / nx) % 8);
  const int tile = line * nx + i % nx;
  if (tile < ntiles) lattice_tile<T>(*args, tile);
}

// The tiles of many problems in one launch: a block finds its problem and tile
// in a table.
struct LatBlock {
  int prob, tile;
};
template <class T>
__global__ __launch_bounds__(T::NT, T::WPS) void k_lattice_batch(const LatArgs *probs, const LatBlock *blocks) {
  typedef const __attribute__((address_space(4))) LatBlock *BlockPtr;
  const int prob = ((BlockPtr)blocks)[blockIdx.x].prob, tile = ((BlockPtr)blocks)[blockIdx.x].tile;
  lattice_tile<T>(((ArgsPtr)probs)[prob], tile);
}

// ---------------------------------------------------------------------------
// Source integrals b_i = sum_q f(x_q) prod_d w_q h_d phi_i(x_q), f at the
// quadrature points, one direction at a time; a workgroup takes a tile of rows.
// x straight from HBM (each point is read by up to three lanes, from L1), y and
// z from LDS; the node factors come from LDS tables.
// ---------------------------------------------------------------------------
template <int D, int K, int NQ>
__global__ __launch_bounds__(256) void k_source(const LatArgs a, const double *__restrict__ F) {
  constexpr int R1 = 16, R2 = D == 3 ? 8 : 16, R3 = D == 3 ? 4 : 1;
  constexpr int Q2 = NQ * (R2 / K + 1), Q3 = D == 3 ? NQ * (R3 / K + 1) : 1;
  __shared__ double Z1[R1 * Q2 * Q3], Z2[R1 * R2 * Q3], vt[27];
  const int tid = threadIdx.x;
  if (tid < 27) vt[tid] = a.V[tid / 9][(tid / 3) % 3][tid % 3];
  const int o0 = a.lo[0] + blockIdx.x * R1, o1 = a.lo[1] + blockIdx.y * R2, o2 = D == 3 ? a.lo[2] + blockIdx.z * R3 : 0;
  const int n0 = a.ncell[0] * NQ, n1 = a.ncell[1] * NQ, n2 = D == 3 ? a.ncell[2] * NQ : 1;
  __syncthreads();
#pragma unroll 2
  for (int i = tid; i < R1 * Q2 * Q3; i += 256) {
    const int v = i % R1, y = (o1 / K - 1) * NQ + (i / R1) % Q2, z = D == 3 ? (o2 / K - 1) * NQ + i / (R1 * Q2) : 0;
    const bool in = (y >= 0) & (y < n1) & (z >= 0) & (z < n2);
    const double *f = F + (in ? (size_t)n0 * (y + (size_t)n1 * z) : 0);
    double acc = 0.0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {  // all loads go out; a point outside takes weight 0
      const int x = (o0 / K - 1 + node_cell<K>(v) + c) * NQ;
      const bool ok = in & (c < node_cells<K>(v)) & (x >= 0) & (x < n0);
      const double *w = vt + (ok ? node_local<K>(v, c) : 0) * 3;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const double t = f[(ok ? x : 0) + q];
        acc = fma(ok ? t : 0.0, w[q], acc);
      }
    }
    Z1[i] = acc;
  }
  __syncthreads();
  for (int i = tid; i < R1 * R2 * Q3; i += 256) {
    const int v = (i / R1) % R2;
    const double *z = Z1 + i % R1 + (i / (R1 * R2) * Q2 + node_cell<K>(v) * NQ) * R1;
    double acc = 0.0;
    for (int c = 0; c < node_cells<K>(v); ++c)
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc = fma(z[(c * NQ + q) * R1], vt[9 + node_local<K>(v, c) * 3 + q], acc);
    Z2[i] = acc;
  }
  __syncthreads();
  for (int i = tid; i < R1 * R2 * R3; i += 256) {
    const int v = i / (R1 * R2), g0 = o0 + i % R1, g1 = o1 + (i / R1) % R2, g2 = o2 + v;
    if (g0 >= a.hi[0] || g1 >= a.hi[1] || g2 >= a.hi[2]) continue;
    const LatRow row = a.rows[row_at<K>(a, g0, g1, g2)];
    if (row.bidx < 0) continue;
    double acc = 0.0;
    if (D == 3) {
      const double *z = Z2 + i % (R1 * R2) + node_cell<K>(v) * NQ * R1 * R2;
      for (int c = 0; c < node_cells<K>(v); ++c)
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc = fma(z[(c * NQ + q) * R1 * R2], vt[18 + node_local<K>(v, c) * 3 + q], acc);
    } else {
      acc = Z2[i];
    }
    a.b[row.bidx] = acc;
  }
}

template <int D, int K, int NQ>
void launch_source(gdx_problem *p, const LatArgs &a, const double *F, hipStream_t st) {
  constexpr int R[3] = {16, D == 3 ? 8 : 16, D == 3 ? 4 : 1};
  dim3 g((a.hi[0] - a.lo[0] + R[0] - 1) / R[0], (a.hi[1] - a.lo[1] + R[1] - 1) / R[1],
         (a.hi[2] - a.lo[2] + R[2] - 1) / R[2]);
  if (g.x && g.y && g.z) hipLaunchKernelGGL((k_source<D, K, NQ>), g, dim3(256), 0, st, a, F);
}

template <int D, int K, int NQ>
struct ShapeOf;
// Q2: 4 x 4 x 2 cells: 676 (pair, cell) lanes in 12 waves, three per SIMD, and
// 62 KB of LDS, so two workgroups share a CU.  With one lane per pair looping
// over its cells (8 waves) the first wave did four cells while the others did
// one: 600 against 500 us at 64^3 with the rest the same.  kappa constant on
// cells needs one point per cell, and 8 waves without the split.
template <int NQ>
struct ShapeOf<3, 2, NQ> {
  using type = LatShape<3, 2, NQ, 4, 4, 2, 768, 64, true>;
};
template <>
struct ShapeOf<3, 2, 1> {
  using type = LatShape<3, 2, 1, 4, 4, 2, 512, 64>;
};
// Q1: 15 x 7 rows in x and y (465 pairs of 512 threads); 15 rows of an x line
// are 3.2 KB of consecutive values
template <int NQ>
struct ShapeOf<3, 1, NQ> {
  using type = LatShape<3, 1, NQ, 15, 7, NQ == 1 ? 4 : 3, 512, 32>;
};
template <int NQ>
struct ShapeOf<2, 2, NQ> {
  using type = LatShape<2, 2, NQ, 8, 8, 1, 256, 32>;
};
template <int NQ>
struct ShapeOf<2, 1, NQ> {
  using type = LatShape<2, 1, NQ, 16, 16, 1, 256, 16>;
};

// row table on the global lattice, padded to whole tiles, from the parts' tables.
// A grid holds 65535 blocks in y and in z (a long box has more lines): each takes
// every gridDim-th line there.
constexpr int kLatRowsGrid = 32768;
template <int K>
__global__ void k_lat_rows(LatArgs a, int parts0, int parts1, const int *__restrict__ node_part,
                           const LatPart *__restrict__ parts, const RowInfo *__restrict__ rowinfo,
                           LatRow *__restrict__ rows) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= a.pn[0]) return;
  for (int z = blockIdx.z; z < a.pn[2]; z += gridDim.z)
    for (int y = blockIdx.y; y < a.pn[1]; y += gridDim.y) {
      LatRow r{0, 0, -1};
      if (x < a.nn[0] && y < a.nn[1] && z < a.nn[2]) {
        const LatPart P =
            parts[node_part[x] + parts0 * (node_part[a.nn[0] + y] + parts1 * node_part[a.nn[0] + a.nn[1] + z])];
        const RowInfo ri =
            rowinfo[P.base + ((long long)(z - P.lo[2]) * P.n[1] + (y - P.lo[1])) * P.n[0] + (x - P.lo[0])];
        if (ri.pid >= 0)
          r = LatRow{8 * ri.rowstart, ri.pid << 9 | ((ri.lenf >> 16) & 1) << 8 | (ri.lenf & 0xFF), (int)ri.bidx};
      }
      rows[row_at<K>(a, x, y, z)] = r;
    }
}

struct LatData {
  LatRow *rows = nullptr;
  uint16_t *delta = nullptr;
};

LatData *ld(gdx_problem *p) { return reinterpret_cast<LatData *>(p->lattice); }

template <class V>
hipError_t put(V **dst, const std::vector<V> &src) {
  const size_t bytes = std::max<size_t>(src.size(), 1) * sizeof(V);
  hipError_t e = dev_malloc(dst, bytes);
  if (e == hipSuccess && !src.empty()) e = hipMemcpy(*dst, src.data(), src.size() * sizeof(V), hipMemcpyHostToDevice);
  return e;
}

template <int D, int K>
void shape_of(int R[3], int nqe) {
  using A = typename ShapeOf<D, K, 1>::type;
  using B = typename ShapeOf<D, K, 2>::type;
  R[0] = nqe == 1 ? A::R1 : B::R1;
  R[1] = nqe == 1 ? A::R2 : B::R2;
  R[2] = nqe == 1 ? A::R3 : B::R3;
}

// rows per tile
void lattice_shape(int dim, int K, int R[3], int nqe) {
  if (dim == 3 && K == 2) shape_of<3, 2>(R, nqe);
  else if (dim == 3) shape_of<3, 1>(R, nqe);
  else if (K == 2) shape_of<2, 2>(R, nqe);
  else shape_of<2, 1>(R, nqe);
}

// lattice extents, the nodes that may hold rows and the row table's extents
void geometry(const gdx_problem *p, LatArgs &a) {
  int R[3], Rq[3];
  lattice_shape(p->D, p->K, R, 1);
  lattice_shape(p->D, p->K, Rq, 2);
  for (int d = 0; d < 3; ++d) {
    a.nn[d] = p->kp.nn[d];
    a.ncell[d] = p->kp.ncells[d];
    // with Dirichlet data on the whole boundary the first and last node of a
    // direction hold no rows; Q2 tiles start at a vertex
    const bool dir = p->desc.dir_kind == 1 && d < p->D;
    a.lo[d] = dir && p->K == 1 ? 1 : 0;
    a.hi[d] = dir ? a.nn[d] - 1 : a.nn[d];
    a.pn[d] = 0;
    for (const int r : {R[d], Rq[d]}) {
      const int nt = std::max(1, (a.hi[d] - a.lo[d] + r - 1) / r);
      a.pn[d] = std::max(std::max(a.pn[d], a.nn[d]), a.lo[d] + nt * r);
    }
    if (d == 0 && p->K == 2) a.pn[d] = (a.pn[d] + 7) & ~7;  // whole groups of four rows of one parity
  }
}

template <class T>
int64_t cut_tiles(LatArgs &a) {
  const int R[3] = {T::R1, T::R2, T::R3};
  for (int d = 0; d < 3; ++d) a.nt[d] = std::max(1, (a.hi[d] - a.lo[d] + R[d] - 1) / R[d]);
  return (int64_t)a.nt[0] * a.nt[1] * a.nt[2];
}

template <class T>
int launch(gdx_problem *p, LatArgs &a, hipStream_t st) {
  const int64_t n = cut_tiles<T>(a), lines = n / a.nt[0];
  const int64_t grid = 8 * ((lines + 7) / 8) * a.nt[0];
  hipLaunchKernelGGL((k_lattice<T>), dim3((unsigned)grid), dim3(T::NT), 0, st, a, (int)n);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

template <class T>
int launch_batch(const LatArgs *probs, const LatBlock *blocks, unsigned n, hipStream_t st) {
  hipLaunchKernelGGL((k_lattice_batch<T>), dim3(n), dim3(T::NT), 0, st, probs, blocks);
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

// the instance of (dim, order, points per cell and direction) `key`
template <class F>
int with_shape(int key, F &&f) {
  switch (key) {
    case 321: return f(ShapeOf<3, 2, 1>::type{});
    case 322: return f(ShapeOf<3, 2, 2>::type{});
    case 323: return f(ShapeOf<3, 2, 3>::type{});
    case 311: return f(ShapeOf<3, 1, 1>::type{});
    case 312: return f(ShapeOf<3, 1, 2>::type{});
    case 221: return f(ShapeOf<2, 2, 1>::type{});
    case 222: return f(ShapeOf<2, 2, 2>::type{});
    case 223: return f(ShapeOf<2, 2, 3>::type{});
    case 211: return f(ShapeOf<2, 1, 1>::type{});
    case 212: return f(ShapeOf<2, 1, 2>::type{});
    case 213: return f(ShapeOf<2, 1, 3>::type{});
  }
  return GDX_ERR_UNSUPPORTED;
}

// arguments of the problem's numeric launch; nqe = points per cell and direction
// that the contraction takes (1 when kappa is constant on every cell)
int fill_args(gdx_problem *p, LatArgs &a, int &nqe) {
  const LatData *L = ld(p);
  const KParams &kp = p->kp;
  const int K = p->K;
  const bool points = !p->coef_cell && kp.nmodes > 0;
  nqe = points ? p->NQ : 1;
  geometry(p, a);
  for (int d = 0; d < 3; ++d) {
    a.x0[d] = kp.x0[d];
    a.hK[d] = kp.hK[d];
    // kinds of pairs in one cell: {v,v}, {v,m}, {m,m}, {v,v'}, {m,v'}, {v',v'}
    static const int k2[6][2] = {{0, 0}, {0, 1}, {1, 1}, {0, 2}, {1, 2}, {2, 2}}, k1[3][2] = {{0, 0}, {0, 1}, {1, 1}};
    for (int k = 0; k < (K == 2 ? 6 : 3); ++k) {
      const int *ab = K == 2 ? k2[k] : k1[k];
      double sg = 0.0, sm = 0.0;
      for (int q = 0; q < p->NQ; ++q) {
        const double G = kp.fG[d][ab[0]][ab[1]][q], M = kp.fM[d][ab[0]][ab[1]][q];
        if (points) a.G[d][k][q] = G, a.M[d][k][q] = M;
        sg += G;
        sm += M;
      }
      if (!points) a.G[d][k][0] = sg, a.M[d][k][0] = sm;
    }
    for (int b = 0; b <= K; ++b) {
      a.Sv[d][b] = 0.0;
      for (int q = 0; q < p->NQ; ++q) {
        const double v = kp.qw[q] * kp.h[d] * kp.phi[b][q];
        if (q < 3) a.V[d][b][q] = v;
        a.Sv[d][b] += v;
      }
    }
  }
  for (int k = 0; k < 4; ++k) a.dir_coef[k] = kp.dir_coef[k];
  a.rows = L->rows;
  a.delta = L->delta;
  a.values = p->dev.values;
  a.b = p->dev.b;
  a.kconst = kp.coef_const;
  a.W = points ? p->dev.W : (p->coef_cell ? p->dev.cellk : nullptr);
  // the manufactured source vanishes where kappa is constant
  const bool manu = kp.rhs_kind == GDX_RHS_MANUFACTURED;
  a.source = points && manu;
  a.fconst = manu ? 0.0 : kp.rhs_const;
  return GDX_OK;
}

}  // namespace

void lattice_free(gdx_problem *p) {
  LatData *L = ld(p);
  if (!L) return;
  void *ptrs[] = {L->rows, L->delta};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  delete L;
  p->lattice = nullptr;
}

// per-direction part tables and the pattern offset tables, after the symbolic phase
int lattice_setup(gdx_problem *p) {
  lattice_free(p);
  LatData *L = new (std::nothrow) LatData;
  if (!L) return GDX_ERR_ALLOC;
  p->lattice = L;
  const int D = p->D, K = p->K, W = 2 * K + 1, S = D == 3 ? W * W * W : W * W, SP = pattern_stride(S);
  std::vector<LatPart> parts(p->nparts);
  std::vector<int> np;
  for (int r = 0; r < p->nparts; ++r) {
    const Part &P = p->P[r];
    for (int d = 0; d < 3; ++d) parts[r].lo[d] = (int)P.onb_lo[d], parts[r].n[d] = (int)P.onb_n[d];
    parts[r].base = P.rowinfo_base;
  }
  for (int d = 0; d < 3; ++d) {
    const int step = d == 0 ? 1 : (d == 1 ? p->desc.parts[0] : p->desc.parts[0] * p->desc.parts[1]);
    for (int q = 0; q < p->desc.parts[d]; ++q)
      np.insert(np.end(), parts[(size_t)q * step].n[d], q);
  }
  // tile strides of U: the row's offsets depend on them
  const int NP1 = D == 3 ? (K == 2 ? ShapeOf<3, 2, 1>::type::NP1 : ShapeOf<3, 1, 1>::type::NP1)
                         : (K == 2 ? ShapeOf<2, 2, 1>::type::NP1 : ShapeOf<2, 1, 1>::type::NP1);
  const int NP12 = D == 3 ? (K == 2 ? ShapeOf<3, 2, 1>::type::NP12 : ShapeOf<3, 1, 1>::type::NP12) : 0;
  const int PSTR = D == 3 ? (K == 2 ? 128 : 32) : (K == 2 ? 32 : 16);
  std::vector<uint16_t> delta((size_t)p->npat * PSTR, 0);
  for (int i = 0; i < p->npat; ++i) {
    const uint8_t *fwd = &p->pat_fwd[(size_t)i * SP];
    int par[3] = {1, 1, 1};  // a row at a vertex of direction d reaches offset -2 or 2 there
    for (int s = 0; s < S && K == 2; ++s) {
      if (fwd[s] == kSlotAbsent) continue;
      const int sd[3] = {s % W - K, (s / W) % W - K, D == 3 ? s / (W * W) - K : 0};
      for (int d = 0; d < D; ++d)
        if (sd[d] == 2 || sd[d] == -2) par[d] = 0;
    }
    for (int s = 0; s < S; ++s) {
      if (fwd[s] == kSlotAbsent || fwd[s] == kSlotDirichlet) continue;
      const int sd[3] = {s % W - K, (s / W) % W - K, D == 3 ? s / (W * W) - K : 0};
      const int off = pair_step(K, par[0], sd[0]) + NP1 * pair_step(K, par[1], sd[1]) +
                      (D == 3 ? NP12 * pair_step(K, par[2], sd[2]) : 0);
      delta[(size_t)i * PSTR + fwd[s]] = (uint16_t)(int16_t)off;
    }
  }
  LatArgs a{};
  geometry(p, a);
  const size_t n = (size_t)a.pn[0] * a.pn[1] * a.pn[2];
  // one buffer and one copy: the position tables, then what the row table is made from
  const auto up16 = [](size_t bytes) { return (bytes + 15) / 16 * 16; };
  const size_t at_parts = up16(delta.size() * sizeof(uint16_t)), at_np = at_parts + up16(parts.size() * sizeof(LatPart));
  std::vector<char> tab(at_np + up16(np.size() * sizeof(int)), 0);
  std::copy_n(reinterpret_cast<const char *>(delta.data()), delta.size() * sizeof(uint16_t), tab.data());
  std::copy_n(reinterpret_cast<const char *>(parts.data()), parts.size() * sizeof(LatPart), tab.data() + at_parts);
  std::copy_n(reinterpret_cast<const char *>(np.data()), np.size() * sizeof(int), tab.data() + at_np);
  char *dtab = nullptr;
  int rc = GDX_OK;
  if (put(&dtab, tab) != hipSuccess || dev_malloc(&L->rows, n * sizeof(LatRow)) != hipSuccess) rc = GDX_ERR_ALLOC;
  L->delta = reinterpret_cast<uint16_t *>(dtab);
  const LatPart *dparts = reinterpret_cast<const LatPart *>(dtab + at_parts);
  const int *node_part = reinterpret_cast<const int *>(dtab + at_np);
  if (!rc) {
    hipStream_t st = p->ctx->stream;
    const dim3 g((a.pn[0] + 255) / 256, std::min(a.pn[1], kLatRowsGrid), std::min(a.pn[2], kLatRowsGrid));
    const auto kernel = K == 2 ? k_lat_rows<2> : k_lat_rows<1>;
    hipLaunchKernelGGL(kernel, g, dim3(256), 0, st, a, p->desc.parts[0], p->desc.parts[1], node_part, dparts,
                       p->dev.rowinfo, L->rows);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) rc = GDX_ERR_HIP;
  }
  if (rc) lattice_free(p);
  return rc;
}

void lattice_shape(int dim, int K, int R[3]) { lattice_shape(dim, K, R, 2); }

// b = source integrals from f at the quadrature points
int launch_source(gdx_problem *p, hipStream_t st) {
  if (!p->lattice) return GDX_ERR_STATE;
  LatArgs a{};
  int nqe = 1;
  fill_args(p, a, nqe);
  const double *F = p->dev.F;
  switch (p->D * 100 + p->K * 10 + p->NQ) {
    case 323: launch_source<3, 2, 3>(p, a, F, st); break;
    case 322: launch_source<3, 2, 2>(p, a, F, st); break;
    case 312: launch_source<3, 1, 2>(p, a, F, st); break;
    case 222: launch_source<2, 2, 2>(p, a, F, st); break;
    case 223: launch_source<2, 2, 3>(p, a, F, st); break;
    case 212: launch_source<2, 1, 2>(p, a, F, st); break;
    case 213: launch_source<2, 1, 3>(p, a, F, st); break;
    default: return GDX_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? GDX_OK : GDX_ERR_HIP;
}

int launch_lattice(gdx_problem *p, hipStream_t st) {
  if (!p->lattice) return GDX_ERR_STATE;
  LatArgs a{};
  int nqe = 1;
  fill_args(p, a, nqe);
  return with_shape(p->D * 100 + p->K * 10 + nqe, [&](auto shape) { return launch<decltype(shape)>(p, a, st); });
}

// Tiles of many problems, one launch per instance.  A small problem's own launch
// fills a few CUs: 32 Q1 cubes of 16..48 cells on four branches of a graph took
// 0.87 ms a refill, the single launch (with the coefficients' two) 0.30 ms, 0.18 of
// them in this kernel.
struct LatticeBatch {
  LatArgs *probs = nullptr;
  struct Group {
    int key;
    LatBlock *blocks;
    unsigned n;
  };
  std::vector<Group> groups;
};

void lattice_batch_free(LatticeBatch *b) {
  if (!b) return;
  if (b->probs) (void)hipFree(b->probs);
  for (LatticeBatch::Group &g : b->groups)
    if (g.blocks) (void)hipFree(g.blocks);
  delete b;
}

int lattice_batch_build(const std::vector<gdx_problem *> &ps, LatticeBatch **out) {
  *out = nullptr;
  std::vector<LatArgs> probs;
  std::vector<int> keys;
  std::vector<std::vector<LatBlock>> blocks;
  for (gdx_problem *p : ps) {
    if (!p->lattice) return GDX_ERR_STATE;
    LatArgs a{};
    int nqe = 1;
    fill_args(p, a, nqe);
    const int key = p->D * 100 + p->K * 10 + nqe;
    int64_t n = 0;
    const int rc = with_shape(key, [&](auto shape) {
      n = cut_tiles<decltype(shape)>(a);
      return GDX_OK;
    });
    if (rc) return rc;
    const size_t g = std::find(keys.begin(), keys.end(), key) - keys.begin();
    if (g == keys.size()) {
      keys.push_back(key);
      blocks.emplace_back();
    }
    for (int64_t t = 0; t < n; ++t) blocks[g].push_back({(int)probs.size(), (int)t});
    probs.push_back(a);
  }
  LatticeBatch *b = new (std::nothrow) LatticeBatch;
  if (!b) return GDX_ERR_ALLOC;
  bool ok = put(&b->probs, probs) == hipSuccess;
  for (size_t g = 0; g < keys.size(); ++g) {
    b->groups.push_back({keys[g], nullptr, (unsigned)blocks[g].size()});
    ok = ok && put(&b->groups.back().blocks, blocks[g]) == hipSuccess;
  }
  if (!ok) {
    lattice_batch_free(b);
    return GDX_ERR_ALLOC;
  }
  *out = b;
  return GDX_OK;
}

int lattice_batch_launch(const LatticeBatch *b, hipStream_t st) {
  for (const LatticeBatch::Group &g : b->groups) {
    const int rc = with_shape(g.key, [&](auto shape) {
      return launch_batch<decltype(shape)>(b->probs, g.blocks, g.n, st);
    });
    if (rc) return rc;
  }
  return GDX_OK;
}

}  // namespace gdx
