// Geometric multigrid preconditioner for structured hex8 operators: level
// planning, Galerkin coarsening, stencil assembly, coarsest dense inverse,
// smoother bounds and the V-cycle.  Every reduction runs in a fixed order,
// so a V-cycle is bit-reproducible.
//
// Element-matrix indexing inside this file: corner bits (bit 0 x, bit 1 y,
// bit 2 z), local DOF = NC * bits + component.  Vectors use the solver's
// column-blocked layout: value (dof, c) at ((c / kc) * ndof + dof) * kc + c % kc.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <cstdlib>

#include "mg.hpp"

namespace skt {

// skfem corner order of the operator's K_e^0 (see operators.hip)
static int corner_id_h(int cx, int cy, int cz) {
  return cz * 4 + (cy ? (cx ? 2 : 3) : (cx ? 1 : 0));
}

static int axis_factor(int64_t n) {
  for (int f : {2, 3, 5})
    if (n % f == 0 && n / f >= 1) return f;
  return 1;
}

// Whether the hierarchy's operator has a null space on the free DOFs: a scalar
// one without Dirichlet nodes and without mass (which the products of tets
// leave out), or supports that leave a rigid
// motion free (the rigid motions' Gram matrix over the fixed DOFs has no full
// rank; nodes of a tet grid at their places on the grid).
static int singular_operator(const skt_operator* op, int* singular) {
  *singular = op->n_fixed == 0 && (op->mass_a == 0.0 || op->mesh == SKT_MESH_TET4);
  if (op->ncomp != 3 || op->n_fixed == 0) return SKT_OK;
  std::vector<int32_t> dofs;
  if (op->fixed_list) {
    dofs.resize((size_t)op->n_fixed);
    SKT_HIP(hipMemcpy(dofs.data(), op->fixed_list, sizeof(int32_t) * dofs.size(),
                      hipMemcpyDeviceToHost));
  } else {  // tet4 operators keep the flags alone
    std::vector<uint8_t> flag((size_t)op->n_nodes * 3);
    SKT_HIP(hipMemcpy(flag.data(), op->fixed, flag.size(), hipMemcpyDeviceToHost));
    for (size_t i = 0; i < flag.size(); ++i)
      if (flag[i]) dofs.push_back((int32_t)i);
  }
  const int64_t nnx = op->nx + 1, nny = op->ny + 1;
  const double len[3] = {op->nx * op->h[0], op->ny * op->h[1], op->nz * op->h[2]};
  const double unit = std::max(len[0], std::max(len[1], len[2]));
  double G[6][6] = {};
  for (int32_t dof : dofs) {
    const int64_t n = dof / 3;
    const double x[3] = {(n % nnx * op->h[0] - 0.5 * len[0]) / unit,
                         (n / nnx % nny * op->h[1] - 0.5 * len[1]) / unit,
                         (n / (nnx * nny) * op->h[2] - 0.5 * len[2]) / unit};
    const int d = dof % 3, e = (d + 1) % 3, f = (d + 2) % 3;
    double m[6] = {};          // component d of the translations and of the
    m[d] = 1.0;                // rotations about each axis (axis x position)
    m[3 + e] = x[f];
    m[3 + f] = -x[e];
    for (int i = 0; i < 6; ++i)
      for (int j = 0; j < 6; ++j) G[i][j] += m[i] * m[j];
  }
  // elimination with diagonal pivoting
  bool done[6] = {};
  const double tiny = 1e-10 * op->n_fixed;
  for (int step = 0; step < 6; ++step) {
    int p = -1;
    for (int i = 0; i < 6; ++i)
      if (!done[i] && (p < 0 || G[i][i] > G[p][p])) p = i;
    if (G[p][p] <= tiny) {
      *singular = 1;
      return SKT_OK;
    }
    done[p] = true;
    for (int i = 0; i < 6; ++i)
      for (int j = 0; j < 6; ++j)
        if (!done[i] && !done[j]) G[i][j] -= G[i][p] * G[p][j] / G[p][p];
  }
  return SKT_OK;
}

// Coarsening factors of a level by factors 2, 3 or 5 that divide its axes; an
// axis is not collapsed to a single element while a longer axis (more than 5
// elements) still coarsens: e.g. 15x5x5 -> 5x5x5, not 5x1x1.
static bool divide_axes(const MGLevel& f, int (&fac)[3]) {
  const int64_t n3[3] = {f.nx, f.ny, f.nz};
  bool longer = false;
  for (int a = 0; a < 3; ++a) {
    fac[a] = axis_factor(n3[a]);
    longer = longer || (n3[a] > 5 && fac[a] > 1);
  }
  if (longer)
    for (int a = 0; a < 3; ++a)
      if (fac[a] > 1 && n3[a] / fac[a] == 1) fac[a] = 1;
  return fac[0] > 1 || fac[1] > 1 || fac[2] > 1;
}

// Factor 2 on every axis, whatever its length: the last coarse element of an
// odd axis holds one fine element.  The same rule against collapsing.
static bool halve_axes(const MGLevel& f, int (&fac)[3]) {
  const int64_t n3[3] = {f.nx, f.ny, f.nz};
  const bool longer = std::max(f.nx, std::max(f.ny, f.nz)) > 5;
  for (int a = 0; a < 3; ++a) fac[a] = n3[a] > (longer ? 2 : 1) ? 2 : 1;
  return fac[0] > 1 || fac[1] > 1 || fac[2] > 1;
}

static MGLevel coarser(const MGLevel& f, const int (&fac)[3], int NC) {
  MGLevel c;
  c.nx = (f.nx + fac[0] - 1) / fac[0];
  c.ny = (f.ny + fac[1] - 1) / fac[1];
  c.nz = (f.nz + fac[2] - 1) / fac[2];
  for (int a = 0; a < 3; ++a) c.f[a] = fac[a];
  c.nn = (c.nx + 1) * (c.ny + 1) * (c.nz + 1);
  c.ndof = c.nn * NC;
  return c;
}

static bool has_cell_grid(const skt_operator* op) {
  return op->mesh == SKT_MESH_HEX8 || (op->mesh == SKT_MESH_TET4 && op->tet_grid);
}

static MGLevel fine_level(const skt_operator* op) {
  MGLevel l0;
  l0.nx = op->nx; l0.ny = op->ny; l0.nz = op->nz;
  l0.nn = (l0.nx + 1) * (l0.ny + 1) * (l0.nz + 1);
  l0.ndof = l0.nn * op->ncomp;
  return l0;
}

bool mg_divides(const skt_operator* op, const MGConfig& cfg) {
  if (!has_cell_grid(op)) return false;
  MGLevel l = fine_level(op);
  int n = 1;
  for (; l.ndof > cfg.max_coarse; ++n) {
    int fac[3];
    if (!divide_axes(l, fac)) return false;
    l = coarser(l, fac, op->ncomp);
  }
  return n >= 2;
}

bool mg_plan(const skt_operator* op, const MGConfig& cfg, std::vector<MGLevel>* out) {
  out->clear();
  if (!has_cell_grid(op)) return false;
  out->push_back(fine_level(op));
  // Conduction and mass operators take 8 to 16 iterations whatever the factors:
  // they keep the fewest levels where factors 2, 3 and 5 divide the grid.
  const bool few = op->ncomp == 1 && mg_divides(op, cfg);
  while (out->back().ndof > cfg.max_coarse) {
    const MGLevel& f = out->back();
    int fac[3];
    // Levels above kDivideNodes nodes are halved on every axis.  Factors 3
    // and 5 leave the smoother error it cannot reach and stretch the coarse
    // elements where the axes take different factors; on smaller levels a
    // level less is worth more than that.
    const bool ok = few || f.nn <= kDivideNodes ? divide_axes(f, fac) || halve_axes(f, fac)
                                                : halve_axes(f, fac);
    if (!ok) return false;
    MGLevel c = coarser(f, fac, op->ncomp);
    // A coarsest level that fits with factor 3 on some axes, where halving
    // them all does not: the largest such level.  One more halved level would
    // leave a much smaller coarsest one, and the exact solve is what catches
    // the error of stiff members in voids: 120x60x60, 8 loads, mixed, with
    // 10x8x5 elements in place of 15x8x8 and 8x4x4 takes 23 PCG iterations
    // per solve instead of 28 (16.0 against 19.2 ms per OC iteration); 100x50x50
    // 7.9 against 9.6 ms, 33x17x13 3.0 against 4.0, 75x45x30 the same.
    if (c.ndof > cfg.max_coarse && f.nn > kDivideNodes && !few) {
      const int64_t n3[3] = {f.nx, f.ny, f.nz};
      int64_t best = 0;
      for (int m = 1; m < 8; ++m) {
        int g[3];
        for (int a = 0; a < 3; ++a) g[a] = ((m >> a) & 1) && fac[a] == 2 && n3[a] >= 5 ? 3 : fac[a];
        const MGLevel t = coarser(f, g, op->ncomp);
        if (t.ndof <= cfg.max_coarse && t.ndof > best) {
          best = t.ndof;
          c = t;
        }
      }
    }
    out->push_back(c);
  }
  return out->size() >= 2;
}

// ------------------------------------------------------------- Galerkin

// Trilinear weight of coarse corner Q (bits) at fine corner q of child
// (a, b, c) inside a coarse element divided by (fx, fy, fz).
__device__ __forceinline__ double tri_weight(int q, int Q, int a, int b, int c, int fx, int fy,
                                             int fz) {
  const double sx = (double)(a + (q & 1)) / fx;
  const double sy = (double)(b + ((q >> 1) & 1)) / fy;
  const double sz = (double)(c + ((q >> 2) & 1)) / fz;
  const double wx = (Q & 1) ? sx : 1.0 - sx;
  const double wy = (Q & 2) ? sy : 1.0 - sy;
  const double wz = (Q & 4) ? sz : 1.0 - sz;
  return wx * wy * wz;
}

// Fine elements of coarse element C along an axis of nf fine elements: f, or
// what is left at the end of the axis.
__host__ __device__ inline int children(int64_t nf, int64_t C, int f) {
  const int64_t left = nf - C * f;
  return left < f ? (int)left : f;
}

// acc += P_j^T sK P_j for child (a, b, c) of a coarse element divided by
// (fx, fy, fz); sK holds the child's ND x ND matrix, 64 threads, acc[k] is
// entry tid + 64 k.
template <int NC>
__device__ __forceinline__ void galerkin_child(const double* sK, double* sT, double* sP, int a,
                                               int b, int c, int fx, int fy, int fz,
                                               double* acc) {
  constexpr int ND = 8 * NC;
  constexpr int NN = ND * ND;
  constexpr int PER = (NN + 63) / 64;
  const int tid = threadIdx.x;
  sP[tid] = tri_weight(tid >> 3, tid & 7, a, b, c, fx, fy, fz);  // sP[q*8+Q]
  __syncthreads();
  // T[(q,d)][(R,e)] = sum_r K[(q,d)][(r,e)] P[r][R]
  for (int i = tid; i < NN; i += 64) {
    const int row = i / ND, col = i % ND;
    const int R = col / NC, e = col % NC;
    double t = 0.0;
#pragma unroll
    for (int r = 0; r < 8; ++r) t += sK[row * ND + r * NC + e] * sP[r * 8 + R];
    sT[i] = t;
  }
  __syncthreads();
  // Kc[(Q,d)][(R,e)] += sum_q P[q][Q] T[(q,d)][(R,e)]
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + 64 * k;
    if (i < NN) {
      const int row = i / ND, col = i % ND;
      const int Q = row / NC, d = row % NC;
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < 8; ++q) t += sP[q * 8 + Q] * sT[(q * NC + d) * ND + col];
      acc[k] += t;
    }
  }
  __syncthreads();
}

// One workgroup of 64 threads per coarse element:
//   Kc = sum_children P_j^T K_j P_j,
// K_j = E_j Z_j K0 Z_j on the finest level (Z_j removes Dirichlet DOFs), or
// the finer level's Galerkin element matrix.  With `only`, elements whose
// flag is 0 are left to k_galerkin_interior.
template <int NC>
__global__ void __launch_bounds__(64)
k_galerkin(int64_t ncx, int64_t ncy, int64_t ncz, int64_t nfx, int64_t nfy, int64_t nfz, int fx,
           int fy, int fz, const double* __restrict__ Kf, const double* __restrict__ K0b,
           const double* __restrict__ E, const uint8_t* __restrict__ fixed,
           const uint8_t* __restrict__ only, double* __restrict__ Kc) {
  constexpr int ND = 8 * NC;
  constexpr int NN = ND * ND;
  constexpr int PER = (NN + 63) / 64;
  __shared__ double sK[NN];
  __shared__ double sT[NN];
  __shared__ double sP[64];
  const int64_t ce = blockIdx.x;
  if (only && !only[ce]) return;
  const int64_t CX = ce % ncx, CY = (ce / ncx) % ncy, CZ = ce / (ncx * ncy);
  const int64_t nfnx = nfx + 1, nfny = nfy + 1;
  const int tid = threadIdx.x;
  const int cx = children(nfx, CX, fx), cy = children(nfy, CY, fy), cz = children(nfz, CZ, fz);
  double acc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) acc[i] = 0.0;
  for (int c = 0; c < cz; ++c)
    for (int b = 0; b < cy; ++b)
      for (int a = 0; a < cx; ++a) {
        const int64_t ex = CX * fx + a, ey = CY * fy + b, ez = CZ * fz + c;
        const int64_t fe = ex + nfx * (ey + nfy * ez);
        // child matrix
        if (Kf) {
          for (int i = tid; i < NN; i += 64) sK[i] = Kf[fe * NN + i];
        } else {
          const double Ee = E[fe];
          for (int i = tid; i < NN; i += 64) {
            const int r = i / ND, s = i % ND;
            double v = Ee * K0b[i];
            if (fixed) {
              const int qr = r / NC, qs = s / NC;
              const int64_t nr = (ex + (qr & 1)) + nfnx * ((ey + ((qr >> 1) & 1)) +
                                                           nfny * (ez + (qr >> 2)));
              const int64_t ns = (ex + (qs & 1)) + nfnx * ((ey + ((qs >> 1) & 1)) +
                                                           nfny * (ez + (qs >> 2)));
              if (fixed[nr * NC + r % NC] || fixed[ns * NC + s % NC]) v = 0.0;
            }
            sK[i] = v;
          }
        }
        galerkin_child<NC>(sK, sT, sP, a, b, c, cx, cy, cz, acc);
      }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + 64 * k;
    if (i < NN) Kc[ce * NN + i] = acc[k];
  }
}

// First coarse level of a tet4 operator whose mesh is a grid of nx*ny*nz
// cells, each split into six tets (element 6 c + s lies in cell c, nodes
// numbered as the cell corners of the grid).  One workgroup of 64 threads
// per coarse element: every child cell's 8-corner matrix
//   K_cell = sum_{s < 6} E_t Z_t K_t Z_t   (t = 6 cell + s, in order s)
// is gathered in LDS (each tet's K_t = V B^T D B from its barycentric
// gradients, Z removing Dirichlet DOFs) and projected as the hex children.
template <int NC>
__global__ void __launch_bounds__(64)
k_galerkin_tet(int64_t ncx, int64_t ncy, int64_t ncz, int64_t nfx, int64_t nfy, int64_t nfz,
               int fx, int fy, int fz,
               const int32_t* __restrict__ conn, const double* __restrict__ g,
               const double* __restrict__ vol, double lam0, double mu0, int64_t n_el,
               const double* __restrict__ E, const uint8_t* __restrict__ fixed,
               double* __restrict__ Kc) {
  constexpr int ND = 8 * NC;
  constexpr int NN = ND * ND;
  constexpr int PER = (NN + 63) / 64;
  __shared__ double sK[NN];
  __shared__ double sT[NN];
  __shared__ double sP[64];
  __shared__ double sg[6][12];    // barycentric gradients of the cell's six tets
  __shared__ int scor[6][4];      // per tet: local node -> cell corner bits, or -1
  __shared__ double sw[6];        // per tet: E_t V_t
  __shared__ int64_t snode[8];    // cell corner bits -> global node
  __shared__ uint8_t sfix[ND];    // the cell corners' Dirichlet flags
  const int64_t ce = blockIdx.x;
  const int64_t CX = ce % ncx, CY = (ce / ncx) % ncy, CZ = ce / (ncx * ncy);
  const int64_t nfnx = nfx + 1, nfny = nfy + 1;
  const int tid = threadIdx.x;
  const int cx = children(nfx, CX, fx), cy = children(nfy, CY, fy), cz = children(nfz, CZ, fz);
  double acc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) acc[i] = 0.0;
  for (int c = 0; c < cz; ++c)
    for (int b = 0; b < cy; ++b)
      for (int a = 0; a < cx; ++a) {
        const int64_t ex = CX * fx + a, ey = CY * fy + b, ez = CZ * fz + c;
        const int64_t cell = ex + nfx * (ey + nfy * ez);
        // (the previous child's projection ended with a barrier)
        if (tid < 8)
          snode[tid] = (ex + (tid & 1)) + nfnx * ((ey + ((tid >> 1) & 1)) + nfny * (ez + (tid >> 2)));
        for (int idx = tid; idx < 6 * 12; idx += 64)
          sg[idx / 12][idx % 12] = g[(int64_t)(idx % 12) * n_el + 6 * cell + idx / 12];
        if (tid < 6) sw[tid] = E[6 * cell + tid] * vol[6 * cell + tid];
        __syncthreads();
        if (tid < 24) {
          const int sidx = tid / 4, q = tid % 4;
          const int64_t node = conn[(int64_t)q * n_el + 6 * cell + sidx];
          int corner = -1;
          for (int c8 = 0; c8 < 8; ++c8)
            if (snode[c8] == node) corner = c8;
          scor[sidx][q] = corner;
        }
        if (tid < ND) sfix[tid] = fixed ? fixed[snode[tid / NC] * NC + tid % NC] : 0;
        for (int i = tid; i < NN; i += 64) sK[i] = 0.0;
        __syncthreads();
        // K_cell = sum_{s < 6} E_t V_t Z_t B^T D B Z_t: tet by tet (in order
        // s), each thread adding some of the tet's (4 NC)^2 entries; distinct
        // entries of a tet land on distinct cell entries
        constexpr int NL = 4 * NC;
        for (int sidx = 0; sidx < 6; ++sidx) {
          for (int e = tid; e < NL * NL; e += 64) {
            const int r = e / NL, col = e % NL;
            const int la = r / NC, ca = r % NC, lb = col / NC, cb = col % NC;
            const int qa = scor[sidx][la], qb = scor[sidx][lb];
            if (qa < 0 || qb < 0) continue;
            const int ia = qa * NC + ca, ib = qb * NC + cb;
            if (sfix[ia] || sfix[ib]) continue;
            const double* ga = sg[sidx] + 3 * la;
            const double* gb = sg[sidx] + 3 * lb;
            double v;
            if (NC == 1) {
              v = ga[0] * gb[0] + ga[1] * gb[1] + ga[2] * gb[2];
            } else {
              const double gg = ga[0] * gb[0] + ga[1] * gb[1] + ga[2] * gb[2];
              v = lam0 * ga[ca] * gb[cb] + mu0 * ((ca == cb ? gg : 0.0) + ga[cb] * gb[ca]);
            }
            sK[ia * ND + ib] += sw[sidx] * v;
          }
          __syncthreads();
        }
        galerkin_child<NC>(sK, sT, sP, a, b, c, cx, cy, cz, acc);
      }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + 64 * k;
    if (i < NN) Kc[ce * NN + i] = acc[k];
  }
}

// On the finest level K_j = E_j K0 wherever the child has no Dirichlet DOF,
// so P_j^T K_j P_j = E_j M_j with M_j = P_j^T K0 P_j fixed per child
// position j = a + fx (b + fy c).  One workgroup per position.
template <int NC>
__global__ void __launch_bounds__(64)
k_galerkin_children(int fx, int fy, int fz, const double* __restrict__ K0b,
                    double* __restrict__ M) {
  constexpr int ND = 8 * NC;
  constexpr int NN = ND * ND;
  constexpr int PER = (NN + 63) / 64;
  __shared__ double sK[NN];
  __shared__ double sT[NN];
  __shared__ double sP[64];
  const int j = blockIdx.x;
  const int a = j % fx, b = (j / fx) % fy, c = j / (fx * fy);
  const int tid = threadIdx.x;
  for (int i = tid; i < NN; i += 64) sK[i] = K0b[i];
  double acc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) acc[i] = 0.0;
  galerkin_child<NC>(sK, sT, sP, a, b, c, fx, fy, fz, acc);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + 64 * k;
    if (i < NN) M[(int64_t)j * NN + i] = acc[k];
  }
}

// 1 for the coarse elements of the first coarse level whose fine nodes hold
// a Dirichlet DOF (their children need the masked product; fixed may be null)
// or that hold fewer fine elements than the others, else 0.
template <int NC>
__global__ void k_galerkin_flags(int64_t ncx, int64_t ncy, int64_t ncz, int64_t nfx, int64_t nfy,
                                 int64_t nfz, int fx, int fy, int fz,
                                 const uint8_t* __restrict__ fixed, uint8_t* __restrict__ flag) {
  const int64_t nce = ncx * ncy * ncz;
  const int64_t nfnx = nfx + 1, nfny = nfy + 1;
  for (int64_t ce = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; ce < nce;
       ce += (int64_t)gridDim.x * blockDim.x) {
    const int64_t CX = ce % ncx, CY = (ce / ncx) % ncy, CZ = ce / (ncx * ncy);
    const int cx = children(nfx, CX, fx), cy = children(nfy, CY, fy), cz = children(nfz, CZ, fz);
    uint8_t any = cx < fx || cy < fy || cz < fz;
    for (int k = 0; k <= cz && fixed; ++k)
      for (int j = 0; j <= cy; ++j)
        for (int i = 0; i <= cx; ++i) {
          const int64_t n = (CX * fx + i) + nfnx * ((CY * fy + j) + nfny * (CZ * fz + k));
#pragma unroll
          for (int d = 0; d < NC; ++d) any |= fixed[n * NC + d];
        }
    flag[ce] = any ? 1 : 0;
  }
}

// Kc = sum_j E_j M_j for the coarse elements without Dirichlet DOFs and with
// all their fine elements (flag null: all of them).  A workgroup of NN threads (one per entry) walks over
// coarse elements, with the element's child moduli staged in LDS; the
// children are summed in the order k_galerkin takes them.
constexpr int kMaxChildren = 125;  // factor 5 on every axis
template <int NC>
__global__ void __launch_bounds__(64 * NC * NC)
k_galerkin_interior(int64_t ncx, int64_t ncy, int64_t ncz, int64_t nfx, int64_t nfy, int fx,
                    int fy, int fz,
                    const double* __restrict__ M, const double* __restrict__ E,
                    const uint8_t* __restrict__ flag, double* __restrict__ Kc) {
  constexpr int NN = 64 * NC * NC;
  __shared__ double sE[kMaxChildren];
  const int64_t nce = ncx * ncy * ncz;
  const int nch = fx * fy * fz;
  const int tid = threadIdx.x;
  for (int64_t ce = blockIdx.x; ce < nce; ce += gridDim.x) {
    if (flag && flag[ce]) continue;  // uniform over the workgroup
    const int64_t CX = ce % ncx, CY = (ce / ncx) % ncy, CZ = ce / (ncx * ncy);
    for (int j = tid; j < nch; j += NN) {
      const int a = j % fx, b = (j / fx) % fy, c = j / (fx * fy);
      sE[j] = E[(CX * fx + a) + nfx * ((CY * fy + b) + nfy * (CZ * fz + c))];
    }
    __syncthreads();
    double acc = 0.0;
    for (int j = 0; j < nch; ++j) acc += sE[j] * M[(int64_t)j * NN + tid];
    Kc[ce * NN + tid] = acc;
    __syncthreads();
  }
}

// Sum of the element-matrix entries coupling (node n, comp d) with (node
// n + o, comp e) over the elements that hold both, in a fixed order.
template <int NC>
__device__ __forceinline__ double couple(const double* __restrict__ Kel, int64_t nx, int64_t ny,
                                         int64_t nz, int64_t i, int64_t j, int64_t k, int ox,
                                         int oy, int oz, int d, int e) {
  constexpr int ND = 8 * NC;
  double v = 0.0;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int sx = s & 1, sy = (s >> 1) & 1, sz = s >> 2;
    const int64_t ex = i - 1 + sx, ey = j - 1 + sy, ez = k - 1 + sz;
    if (ex < 0 || ex >= nx || ey < 0 || ey >= ny || ez < 0 || ez >= nz) continue;
    const int ax = 1 - sx, ay = 1 - sy, az = 1 - sz;
    const int bx = ax + ox, by = ay + oy, bz = az + oz;
    if (bx < 0 || bx > 1 || by < 0 || by > 1 || bz < 0 || bz > 1) continue;
    const int A = ax | (ay << 1) | (az << 2), B = bx | (by << 1) | (bz << 2);
    v += Kel[(ex + nx * (ey + ny * ez)) * (ND * ND) + (A * NC + d) * ND + B * NC + e];
  }
  return v;
}

// Stencil storage.  Coefficient c = (o * NC + d) * NC + e of a node couples
// its component d to component e of the neighbour at offset
// o = (ox+1) + 3 (oy+1) + 9 (oz+1).
// * Node-major: st[c * nn + node].
// * Tile-major (levels applied by the LDS-tiled kernel): nodes are grouped
//   in tsx x tsy x tsz tiles (tile-major, x fastest in both) and
//   st[(tile * 27 NC^2 + c) * ts + local], ts = tsx tsy tsz, padding nodes
//   past the grid holding zeros.  A wavefront's nodes then read contiguous
//   bytes per coefficient instead of 64-byte pieces of separate node rows;
//   the 60x30x30 level's apply went from 28.6 to 13.9 us.
// Tile shapes: 16x4x4 for levels of at least kTiledNodes nodes, 16x2x2
// (more, smaller workgroups) below: the 30x15x15 level's apply takes 6.9 us
// with it, 11.4 us with 16x4x4 tiles and 17.5 us node-major.
struct TileShape {
  int x, y, z;
};
constexpr TileShape kTileBig = {16, 4, 4}, kTileSmall = {16, 2, 2};
enum { ST_NODE = 0, ST_TILE_BIG = 1, ST_TILE_SMALL = 2 };

__host__ __device__ inline TileShape tile_shape(int layout) {
  return layout == ST_TILE_BIG ? kTileBig : kTileSmall;
}

__host__ __device__ inline int64_t st_tiles(int64_t nx, int64_t ny, int64_t nz, TileShape t) {
  return ((nx + t.x) / t.x) * ((ny + t.y) / t.y) * ((nz + t.z) / t.z);
}

// nodes the storage holds (tile padding included)
__host__ __device__ inline int64_t st_nodes(int64_t nx, int64_t ny, int64_t nz, int layout) {
  if (layout == ST_NODE) return (nx + 1) * (ny + 1) * (nz + 1);
  const TileShape t = tile_shape(layout);
  return st_tiles(nx, ny, nz, t) * (t.x * t.y * t.z);
}

// offset of coefficient c of node (i, j, k)
template <int NC>
__device__ __forceinline__ int64_t st_index(int64_t nx, int64_t ny, int64_t nz, int layout,
                                            int64_t i, int64_t j, int64_t k, int c) {
  const int64_t nnx = nx + 1, nny = ny + 1;
  if (layout != ST_NODE) {
    const TileShape t = tile_shape(layout);
    const int ts = t.x * t.y * t.z;
    const int64_t bx = (nx + t.x) / t.x, by = (ny + t.y) / t.y;
    const int64_t tile = i / t.x + bx * (j / t.y + by * (k / t.z));
    const int local = (int)(i % t.x + t.x * (j % t.y + t.y * (k % t.z)));
    return (tile * (27 * NC * NC) + c) * ts + local;
  }
  return c * (nnx * nny * (nz + 1)) + i + nnx * (j + nny * k);
}

// One entry per thread over the whole storage (tile padding included).
template <typename T, int NC>
__global__ void k_stencil_asm(int64_t nx, int64_t ny, int64_t nz, int layout,
                              const double* __restrict__ Kel, T* __restrict__ st) {
  constexpr int NS = 27 * NC * NC;
  const int64_t nnx = nx + 1, nny = ny + 1, nnz = nz + 1;
  const int64_t nn = nnx * nny * nnz;
  const int64_t total = st_nodes(nx, ny, nz, layout) * NS;
  const TileShape ts = tile_shape(layout);
  const int tsn = ts.x * ts.y * ts.z;
  const int64_t bx = (nx + ts.x) / ts.x, by = (ny + ts.y) / ts.y;
  // Consecutive blocks of entries (consecutive components of a tile) read
  // the same element-matrix lines; workgroups go to the 8 XCDs (each with
  // its own L2) in turn, so XCD x takes the contiguous range of logical
  // blocks starting at x q + min(x, r) (q, r: quotient and remainder of the
  // grid by 8) and those reads meet in one L2.
  const int64_t nb = gridDim.x, q8 = nb / 8, r8 = nb % 8;
  const int64_t xcd = blockIdx.x % 8;
  const int64_t lb = xcd * q8 + (xcd < r8 ? xcd : r8) + blockIdx.x / 8;
  for (int64_t t = lb * blockDim.x + threadIdx.x; t < total; t += nb * blockDim.x) {
    int64_t i, j, k;
    int c;
    if (layout != ST_NODE) {
      const int local = (int)(t % tsn);
      c = (int)((t / tsn) % NS);
      const int64_t tile = t / ((int64_t)tsn * NS);
      i = (tile % bx) * ts.x + local % ts.x;
      j = ((tile / bx) % by) * ts.y + (local / ts.x) % ts.y;
      k = (tile / (bx * by)) * ts.z + local / (ts.x * ts.y);
      if (i >= nnx || j >= nny || k >= nnz) {
        st[t] = T(0);
        continue;
      }
    } else {
      const int64_t node = t % nn;
      c = (int)(t / nn);
      i = node % nnx;
      j = (node / nnx) % nny;
      k = node / (nnx * nny);
    }
    const int e = c % NC, d = (c / NC) % NC, o = c / (NC * NC);
    const int ox = o % 3 - 1, oy = (o / 3) % 3 - 1, oz = o / 9 - 1;
    st[t] = (T)couple<NC>(Kel, nx, ny, nz, i, j, k, ox, oy, oz, d, e);
  }
}

// Jacobi inverse of a stencil level; rows with no stiffness (DOFs that no
// free fine DOF depends on) get 0 and stay 0 through the cycle.
template <typename T, int NC>
__global__ void k_stencil_dinv(int64_t nx, int64_t ny, int64_t nz, int layout,
                               const T* __restrict__ st, T* __restrict__ dinv) {
  const int64_t nnx = nx + 1, nny = ny + 1, nn = nnx * nny * (nz + 1);
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nn * NC;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t node = t / NC;
    const int d = (int)(t % NC);
    const int64_t i = node % nnx, j = (node / nnx) % nny, k = node / (nnx * nny);
    const T v = st[st_index<NC>(nx, ny, nz, layout, i, j, k, (13 * NC + d) * NC + d)];
    dinv[t] = v > T(0) ? T(1) / v : T(0);
  }
}

// Dense coarsest matrix (fp64, row-major, n rows padded to np with the
// identity), its diagonal times `scale` (above 1 for a singular operator).
template <int NC>
__global__ void k_dense_asm(int64_t nx, int64_t ny, int64_t nz, const double* __restrict__ Kel,
                            int64_t np, double scale, double* __restrict__ A) {
  const int64_t nnx = nx + 1, nny = ny + 1;
  const int64_t n = nnx * nny * (nz + 1) * NC;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < np * np;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = t / np, c = t % np;
    if (r >= n || c >= n) {
      A[t] = r == c ? 1.0 : 0.0;
      continue;
    }
    const int64_t nr = r / NC, ncn = c / NC;
    const int d = (int)(r % NC), e = (int)(c % NC);
    const int64_t i = nr % nnx, j = (nr / nnx) % nny, k = nr / (nnx * nny);
    const int64_t i2 = ncn % nnx, j2 = (ncn / nnx) % nny, k2 = ncn / (nnx * nny);
    const int64_t ox = i2 - i, oy = j2 - j, oz = k2 - k;
    double v = 0.0;
    if (ox >= -1 && ox <= 1 && oy >= -1 && oy <= 1 && oz >= -1 && oz <= 1)
      v = couple<NC>(Kel, nx, ny, nz, i, j, k, (int)ox, (int)oy, (int)oz, d, e);
    // a DOF that no free fine DOF depends on gets the identity
    A[t] = r != c ? v : v > 0.0 ? scale * v : 1.0;
  }
}

// ------------------------------------------- blocked Gauss-Jordan inverse
// Inversion of an SPD matrix (no pivoting needed) of T x T blocks of kGJ rows,
// one pivot block per launch: with P the inverse of pivot block A_bb,
//   A_bb <- P, A_bJ <- P A_bJ, A_Ib <- -A_Ib P, A_IJ <- A_IJ - A_Ib P A_bJ.
// The launches alternate between two copies of the matrix, so every block of
// a launch is independent: a workgroup takes one, forms P A_bJ for itself
// (float64 matrix instructions; the product twice over costs less than a
// launch of its own) and applies A_Ib to it.  The first workgroup takes the
// next pivot block, and inverts it in LDS: that chain, the two products and
// 16 steps of 4 pivots, is what a launch lasts on small matrices.  Before, a
// step took three launches with LDS-tiled products on the vector unit and one
// pivot at a time: n = 1188, 61 us of kernels per step, now 33; n = 1782, 85
// us, now 42.
constexpr int kGJ = 64;
constexpr int kGJStride = kGJ + 16;  // LDS row pitch: two rows of 16 lanes on distinct banks
typedef double gj_vec4 __attribute__((ext_vector_type(4)));

// Inverse of the kGJ x kGJ matrix in LDS (row pitch kGJStride) into P.  Each
// thread keeps a 4 x 4 block in registers; per step the owners of four pivot
// rows and columns publish them through LDS (double-buffered, one barrier per
// step), and every thread inverts the 4 x 4 pivot for itself.
__device__ __forceinline__ void gj_block_inv(const double* sM, double* __restrict__ P) {
  static_assert(kGJ == 64, "4 x 4 register blocks of a 64 x 64 matrix");
  __shared__ double prow[2][4][kGJ], pcol[2][kGJ][4];
  const int tid = threadIdx.x;
  const int tr = tid / 16, tc = tid % 16;  // rows 4 tr.., columns 4 tc..
  double m[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) m[i][j] = sM[(4 * tr + i) * kGJStride + 4 * tc + j];
  for (int kb = 0; kb < kGJ / 4; ++kb) {
    const int buf = kb & 1;
    const bool own_row = tr == kb, own_col = tc == kb;
    if (own_row) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) prow[buf][i][4 * tc + j] = m[i][j];
    }
    if (own_col) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) pcol[buf][4 * tr + i][j] = m[i][j];
    }
    __syncthreads();
    double d[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) d[i][j] = prow[buf][i][4 * kb + j];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double ip = 1.0 / d[k][k];
      d[k][k] = 1.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) d[k][j] *= ip;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i == k) continue;
        const double f = d[i][k];
        d[i][k] = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) d[i][j] -= f * d[k][j];
      }
    }
    // the pivot rows' new values in this thread's columns
    double rk[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) x[q] = prow[buf][q][4 * tc + j];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) v += d[i][q] * x[q];
        rk[i][j] = own_col ? d[i][j] : v;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      double c[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = pcol[buf][4 * tr + i][q];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double v = own_col ? 0.0 : m[i][j];
#pragma unroll
        for (int q = 0; q < 4; ++q) v -= c[q] * rk[q][j];
        m[i][j] = own_row ? rk[i][j] : v;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) P[(4 * tr + i) * kGJ + 4 * tc + j] = m[i][j];
}

// the first pivot block's inverse
__global__ void __launch_bounds__(256) k_gj_first(int np, const double* __restrict__ A,
                                                  double* __restrict__ P) {
  __shared__ double sM[kGJ * kGJStride];
  for (int i = threadIdx.x; i < kGJ * kGJ; i += 256)
    sM[(i / kGJ) * kGJStride + i % kGJ] = A[(int64_t)(i / kGJ) * np + i % kGJ];
  __syncthreads();
  gj_block_inv(sM, P);
}

// Step of pivot block b (its inverse in P): A into Aout, the next pivot's
// inverse into Pn.  Lane l of v_mfma_f64_16x16x4 holds A[l % 16][l / 16],
// B[l / 16][l % 16] and D[l / 16 + 4 i][l % 16], i < 4; wavefront w takes
// rows 16 w .. 16 w + 15 of the workgroup's block.
__global__ void __launch_bounds__(256) k_gj_step(int np, int b, const double* __restrict__ A,
                                                 const double* __restrict__ P,
                                                 double* __restrict__ Aout,
                                                 double* __restrict__ Pn) {
  __shared__ double sR[kGJ * kGJStride];
  const int T = np / kGJ;
  const int first = b + 1 < T ? (b + 1) * (T + 1) : 0;
  const int id = ((int)blockIdx.x + first) % (T * T);
  const int I = id / T, J = id % T;
  const int tid = threadIdx.x;
  double* out = Aout + ((int64_t)I * np + J) * kGJ;
  if (I == b && J == b) {
    for (int i = tid; i < kGJ * kGJ; i += 256) out[(int64_t)(i / kGJ) * np + i % kGJ] = P[i];
    return;
  }
  const int w = tid / kWave, lr = tid % 16, lk = (tid % kWave) / 16;
  gj_vec4 acc[4];
  if (J != b) {
    // P A_bJ
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = gj_vec4{0.0, 0.0, 0.0, 0.0};
    const double* x = A + ((int64_t)b * np + J) * kGJ + lr;
    const double* p = P + (16 * w + lr) * kGJ + lk;
#pragma unroll 8
    for (int s = 0; s < kGJ / 4; ++s) {
      const double a = p[4 * s];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[(int64_t)(4 * s + lk) * np + 16 * j],
                                                      acc[j], 0, 0, 0);
    }
    if (I != b) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sR[(16 * w + lk + 4 * i) * kGJStride + 16 * j + lr] = acc[j][i];
      const double* y = A + ((int64_t)I * np + J) * kGJ + lr;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[j][i] = y[(int64_t)(16 * w + lk + 4 * i) * np + 16 * j];
    }
  } else {
    for (int i = tid; i < kGJ * kGJ; i += 256) sR[(i / kGJ) * kGJStride + i % kGJ] = P[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = gj_vec4{0.0, 0.0, 0.0, 0.0};
  }
  if (I != b) {  // uniform over the workgroup
    __syncthreads();
    const double* l = A + ((int64_t)I * np + b) * kGJ + (int64_t)(16 * w + lr) * np + lk;
#pragma unroll 8
    for (int s = 0; s < kGJ / 4; ++s) {
      const double a = -l[4 * s];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
            a, sR[(4 * s + lk) * kGJStride + 16 * j + lr], acc[j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[(int64_t)(16 * w + lk + 4 * i) * np + 16 * j + lr] = acc[j][i];
  if (blockIdx.x == 0 && b + 1 < T) {
    __syncthreads();  // every wavefront has read sR
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) sR[(16 * w + lk + 4 * i) * kGJStride + 16 * j + lr] = acc[j][i];
    __syncthreads();
    gj_block_inv(sR, Pn);
  }
}

// the n x n matrix out of its padded copy
template <typename T>
__global__ void k_cast(int64_t n, int64_t np, const double* __restrict__ a, T* __restrict__ b) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = (T)a[(i / n) * np + i % n];
}

// ------------------------------------------------------------ operators

// N consecutive values of a node (NC components x KC columns, contiguous in
// the blocked layout) with paired loads / stores when KC is even: the
// offset is then a multiple of 2 values, so 8-byte (float) or 16-byte
// (double) aligned.
template <typename T> struct Pair;
template <> struct Pair<float> { using type = float2; };
template <> struct Pair<double> { using type = double2; };

template <typename T, int N, int KC>
__device__ __forceinline__ void load_node(const T* __restrict__ p, T (&v)[N]) {
  if constexpr (KC % 2 == 0) {
    using V = typename Pair<T>::type;
    const V* q = reinterpret_cast<const V*>(p);
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const V w = q[i];
      v[2 * i] = w.x;
      v[2 * i + 1] = w.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = p[i];
  }
}

template <typename T, int N, int KC>
__device__ __forceinline__ void store_node(T* __restrict__ p, const T (&v)[N]) {
  if constexpr (KC % 2 == 0) {
    using V = typename Pair<T>::type;
    V* q = reinterpret_cast<V*>(p);
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      V w;
      w.x = v[2 * i];
      w.y = v[2 * i + 1];
      q[i] = w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = v[i];
  }
}

// Output of a stencil apply: mode 0 writes y = S x; mode 2 writes a fused
// Chebyshev-Jacobi step x_out = x + c1 (x - x_prev) + c2 dinv (b - S x),
// where x_prev is read from the output buffer itself (ping-pong iterates,
// so no direction vector exists) unless prev_zero, and (c1, c2) = coef[0..1].
enum { ST_APPLY = 0, ST_CHEB = 2 };

template <typename T>
struct StOut {
  const T* b = nullptr;
  const T* dinv = nullptr;
  const double* coef = nullptr;
  int prev_zero = 1;
  const double* stop = nullptr;  // column stop flags (tiled kernel: skip stopped workgroups)
};

// y = S x on a stencil level.  A thread takes one (node, component row) and
// up to GM column groups, so each stencil row is read once for all of them.
template <typename T, int NC, int KC, int GM, int MODE>
__global__ void k_stencil_apply(int64_t nx, int64_t ny, int64_t nz, int groups,
                                const T* __restrict__ st, const T* __restrict__ X,
                                T* __restrict__ Y, StOut<T> oa) {
  const int64_t nnx = nx + 1, nny = ny + 1, nnz = nz + 1;
  const int64_t nn = nnx * nny * nnz;
  const int chunks = (groups + GM - 1) / GM;
  const int64_t total = nn * NC * chunks;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t node = t % nn;
    const int d = (int)((t / nn) % NC);
    const int g0 = (int)(t / (nn * NC)) * GM;
    const int ng = groups - g0 < GM ? groups - g0 : GM;
    const int64_t i = node % nnx, j = (node / nnx) % nny, k = node / (nnx * nny);
    T acc[GM][KC];
#pragma unroll
    for (int q = 0; q < GM; ++q)
#pragma unroll
      for (int c = 0; c < KC; ++c) acc[q][c] = T(0);
    // unrolled and branch-free: a neighbour outside the grid has an exactly
    // zero stencil block, so its address is clamped to the node itself
#pragma unroll
    for (int o = 0; o < 27; ++o) {
      const int ox = o % 3 - 1, oy = (o / 3) % 3 - 1, oz = o / 9 - 1;
      const int64_t i2 = i + ox, j2 = j + oy, k2 = k + oz;
      const bool in = i2 >= 0 && i2 < nnx && j2 >= 0 && j2 < nny && k2 >= 0 && k2 < nnz;
      const int64_t m = in ? i2 + nnx * (j2 + nny * k2) : node;
      T a[NC];
#pragma unroll
      for (int e = 0; e < NC; ++e) a[e] = st[((o * NC + d) * NC + e) * nn + node];
#pragma unroll
      for (int q = 0; q < GM; ++q) {
        if (q >= ng) break;
        T xv[NC * KC];
        load_node<T, NC * KC, KC>(X + ((int64_t)(g0 + q) * nn + m) * NC * KC, xv);
#pragma unroll
        for (int e = 0; e < NC; ++e)
#pragma unroll
          for (int c = 0; c < KC; ++c) acc[q][c] += a[e] * xv[e * KC + c];
      }
    }
    T c1 = T(0), c2 = T(0), dv = T(0);
    if constexpr (MODE == ST_CHEB) {
      c1 = (T)oa.coef[0];
      c2 = (T)oa.coef[1];
      dv = oa.dinv[node * NC + d];
    }
#pragma unroll
    for (int q = 0; q < GM; ++q) {
      if (q >= ng) break;
      const int64_t off = (((int64_t)(g0 + q) * nn + node) * NC + d) * KC;
      if constexpr (MODE == ST_CHEB) {
        T xc[KC], bv[KC], xp[KC];
        load_node<T, KC, KC>(X + off, xc);
        load_node<T, KC, KC>(oa.b + off, bv);
        if (oa.prev_zero) {
#pragma unroll
          for (int c = 0; c < KC; ++c) xp[c] = T(0);
        } else {
          load_node<T, KC, KC>(Y + off, xp);
        }
#pragma unroll
        for (int c = 0; c < KC; ++c)
          acc[q][c] = xc[c] + c1 * (xc[c] - xp[c]) + c2 * dv * (bv[c] - acc[q][c]);
      }
      store_node<T, KC, KC>(Y + off, acc[q]);
    }
  }
}

// First Chebyshev step from a zero iterate on the fine level:
// x = c2 dinv b (blocked vectors, total = ndof * k)
template <typename T>
__global__ void k_cheb_first(int64_t total, int64_t ndof, int kc, const double* __restrict__ coef,
                             const T* __restrict__ b, const T* __restrict__ dinv,
                             T* __restrict__ x) {
  const T c2 = (T)coef[1];
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x)
    x[t] = c2 * dinv[(t / kc) % ndof] * b[t];
}

// y = S x on a stencil level, LDS-tiled: a workgroup owns a SX x SY x SZ
// block of nodes and stages x of the block and its one-node halo for GM
// column groups in LDS once.  NC threads share a node, one per component
// row, so a workgroup runs TS NC threads (TS = SX SY SZ): each sums its
// row's 27 stencil blocks for all GM groups.  Stencil rows are read once per
// node, from the tile-major storage of the same tile shape.
template <typename T, int NC, int KC, int GM, int MODE, int SX, int SY, int SZ>
__global__ void __launch_bounds__(SX * SY * SZ * NC)
k_stencil_apply_tiled(int64_t nx, int64_t ny, int64_t nz, int groups, const T* __restrict__ st,
                      const T* __restrict__ X, T* __restrict__ Y, StOut<T> oa) {
  constexpr int HX = SX + 2, HY = SY + 2, HZ = SZ + 2, TS = SX * SY * SZ;
  constexpr int V = NC * KC;          // values of one node and one group
  constexpr int W = V * GM;           // values of one node in LDS
  __shared__ T xs[HZ * HY * HX * W];
  const int64_t nnx = nx + 1, nny = ny + 1, nnz = nz + 1;
  const int64_t nn = nnx * nny * nnz;
  const int bx = (int)((nnx + SX - 1) / SX), by = (int)((nny + SY - 1) / SY),
            bz = (int)((nnz + SZ - 1) / SZ);
  int b = blockIdx.x;
  const int tbx = b % bx; b /= bx;
  const int tby = b % by; b /= by;
  const int tbz = b % bz; b /= bz;
  const int g0 = b * GM;
  const int ng = groups - g0 < GM ? groups - g0 : GM;
  if (oa.stop) {
    bool all = true;
    for (int c = g0 * KC; c < (g0 + ng) * KC; ++c) all = all && oa.stop[c * kStopStride] != 0.0;
    if (all) return;
  }
  const int64_t x0 = (int64_t)tbx * SX, y0 = (int64_t)tby * SY, z0 = (int64_t)tbz * SZ;
  // this tile's coefficients (tile-major storage)
  st += (int64_t)(tbx + bx * (tby + by * tbz)) * (27 * NC * NC) * TS;
  const int nt = threadIdx.x % TS, d = threadIdx.x / TS;
  // stage x (halo nodes outside the grid read as zero; their stencil
  // entries are zero as well).  A thread's NIT items are all loaded before
  // any is stored, with unpredicated loads (an item outside the grid reads
  // the first node of the vector and stores zero): a load in a branch of its
  // own is waited for inside it, one memory latency per item.
  constexpr int NH = HZ * HY * HX * GM, NIT = (NH + TS * NC - 1) / (TS * NC);
  {
    T v[NIT][V];
    bool ok[NIT];
#pragma unroll
    for (int u = 0; u < NIT; ++u) {
      const int it = threadIdx.x + u * TS * NC;
      const int q = it % GM, hn = it / GM;
      const int hx = hn % HX, hy = (hn / HX) % HY, hz = hn / (HX * HY);
      const int64_t gx = x0 - 1 + hx, gy = y0 - 1 + hy, gz = z0 - 1 + hz;
      ok[u] = it < NH && q < ng && gx >= 0 && gx < nnx && gy >= 0 && gy < nny && gz >= 0 &&
              gz < nnz;
      const int64_t off = ok[u] ? ((int64_t)(g0 + q) * nn + gx + nnx * (gy + nny * gz)) * V : 0;
      load_node<T, V, KC>(X + off, v[u]);
    }
#pragma unroll
    for (int u = 0; u < NIT; ++u) {
      const int it = threadIdx.x + u * TS * NC;
      if (it < NH) {
        const int q = it % GM, hn = it / GM;
#pragma unroll
        for (int i = 0; i < V; ++i) xs[hn * W + q * V + i] = ok[u] ? v[u][i] : T(0);
      }
    }
  }
  __syncthreads();
  const int tx = nt % SX, ty = (nt / SX) % SY, tz = nt / (SX * SY);
  const int64_t gx = x0 + tx, gy = y0 + ty, gz = z0 + tz;
  if (gx >= nnx || gy >= nny || gz >= nnz) return;
  const int64_t node = gx + nnx * (gy + nny * gz);
  T acc[GM][KC];
#pragma unroll
  for (int q = 0; q < GM; ++q)
#pragma unroll
    for (int c = 0; c < KC; ++c) acc[q][c] = T(0);
#pragma unroll 3
  for (int o = 0; o < 27; ++o) {
    const int ox = o % 3, oy = (o / 3) % 3, oz = o / 9;  // halo offsets 0..2
    const T* xn = xs + ((tz + oz) * HY * HX + (ty + oy) * HX + (tx + ox)) * W;
    T a[NC];
#pragma unroll
    for (int e = 0; e < NC; ++e) a[e] = st[((o * NC + d) * NC + e) * TS + nt];
#pragma unroll
    for (int q = 0; q < GM; ++q)
#pragma unroll
      for (int e = 0; e < NC; ++e)
#pragma unroll
        for (int c = 0; c < KC; ++c) acc[q][c] += a[e] * xn[q * V + e * KC + c];
  }
  const T* xcen = xs + ((tz + 1) * HY * HX + (ty + 1) * HX + (tx + 1)) * W;
  // The Chebyshev operands of every group are loaded together (unpredicated:
  // a group past the last, or x_prev when it is zero, reads offset 0).  With
  // every group present (nq = GM, a constant after inlining) no store is
  // predicated, so the compiler does not sink a group's loads into a branch
  // of its own, where each would be waited for in turn.
  auto finish = [&](const int nq) {
    T c1 = T(0), c2 = T(0), dv = T(0);
    T bv[GM][KC], xp[GM][KC];
    if constexpr (MODE == ST_CHEB) {
      c1 = (T)oa.coef[0];
      c2 = (T)oa.coef[1];
      dv = oa.dinv[node * NC + d];
#pragma unroll
      for (int q = 0; q < GM; ++q) {
        const int64_t off = ((int64_t)(g0 + (q < nq ? q : 0)) * nn + node) * V + d * KC;
        load_node<T, KC, KC>(oa.b + off, bv[q]);
        load_node<T, KC, KC>(Y + (oa.prev_zero ? 0 : off), xp[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < GM; ++q) {
      if (q >= nq) break;
      const int64_t off = ((int64_t)(g0 + q) * nn + node) * V + d * KC;
      if constexpr (MODE == ST_CHEB) {
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const T xc = xcen[q * V + d * KC + c];
          const T xpc = oa.prev_zero ? T(0) : xp[q][c];
          acc[q][c] = xc + c1 * (xc - xpc) + c2 * dv * (bv[q][c] - acc[q][c]);
        }
      }
      store_node<T, KC, KC>(Y + off, acc[q]);
    }
  };
  if (ng == GM)
    finish(GM);
  else
    finish(ng);
}

// Chebyshev step on a level (blocked vectors, total = ndof * k):
//   d <- c1 d + c2 dinv (b - w);  x <- x + d   (w null: the iterate is 0)
// coef holds (c1, c2) for this step.
template <typename T>
__global__ void k_cheb(int64_t total, int64_t ndof, int kc, const double* __restrict__ coef,
                       const T* __restrict__ b, const T* __restrict__ w,
                       const T* __restrict__ dinv, T* __restrict__ d, T* __restrict__ x,
                       int x_is_zero) {
  const T c1 = (T)coef[0], c2 = (T)coef[1];
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t dof = (t / kc) % ndof;
    const T r = w ? b[t] - w[t] : b[t];
    const T dn = ((x_is_zero || c1 == T(0)) ? T(0) : c1 * d[t]) + c2 * dinv[dof] * r;
    d[t] = dn;
    x[t] = x_is_zero ? dn : x[t] + dn;
  }
}

// w = b - w (the fine level's residual after a generic operator apply), zero at
// Dirichlet DOFs
template <typename T>
__global__ void k_rsub(int64_t total, int64_t ndof, int kc, const uint8_t* __restrict__ fixed,
                       const T* __restrict__ b, T* __restrict__ w) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x)
    w[t] = (fixed && fixed[(t / kc) % ndof]) ? T(0) : b[t] - w[t];
}

template <typename T>
__global__ void k_copy_vec(int64_t total, const T* __restrict__ a, T* __restrict__ b) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x)
    b[t] = a[t];
}

// Transfers run on row grids: blockIdx.x and threadIdx.x give the node along
// x, blockIdx.y (strided) the row (y, z, column group), so the index
// arithmetic is a few 32-bit divisions per row rather than 64-bit ones per
// value.  (Splitting a node's components over three lanes made the
// prolongation twice as slow: the row of 3 nx pieces fills 256-lane
// workgroups poorly and every lane repeats the weights.)  Row counts and row
// lengths fit in 32 bits.
struct RowGrid {
  dim3 grid, block;
};

static RowGrid row_grid(int64_t row_len, int64_t rows) {
  RowGrid g;
  const int bx = row_len >= 256 ? 256 : (int)((row_len + 63) / 64) * 64;
  g.block = dim3((unsigned)bx);
  g.grid = dim3((unsigned)((row_len + bx - 1) / bx), (unsigned)std::min<int64_t>(rows, 65535));
  return g;
}

// Restriction b_c = P^T Z (b - w), separable in two passes.
// Pass 1 (x, y): t[(I, J, k)] = sum_{dx,dy} w(dx) w(dy) r(f I + dx, f J + dy, k)
// on every fine z plane k, r = b - w with Dirichlet DOFs removed.  Thread:
// coarse I; row: (J, k, group).  The coarse node at the end of an axis lies
// on the axis' last fine node, wl fine elements from its neighbour.
__device__ __forceinline__ int interval(int fn, int I, int f) {
  // fine elements right of coarse node I, f past the last one
  const int left = fn - I * f;
  return left > 0 && left < f ? left : f;
}

struct Taps {
  int x, wl, wr;  // fine position, fine elements to the left and right neighbour
};

__device__ __forceinline__ Taps coarse_taps(int I, int f, int fn) {
  Taps t;
  t.x = I * f < fn ? I * f : fn;
  t.wl = I > 0 ? t.x - (I - 1) * f : 1;
  const int right = fn - t.x;
  t.wr = right < f ? (right > 0 ? right : 1) : f;
  return t;
}

template <typename T, int NC, int KC>
__global__ void k_restrict_xy(int fnx, int fny, int fnz, int fx, int fy, int groups,
                              const T* __restrict__ b, const T* __restrict__ w,
                              const uint8_t* __restrict__ fixed, T* __restrict__ tbuf) {
  const int fnnx = fnx + 1, fnny = fny + 1, fnnz = fnz + 1;
  const int cnnx = (fnx + fx - 1) / fx + 1, cnny = (fny + fy - 1) / fy + 1;
  const int64_t tn = (int64_t)cnnx * cnny * fnnz, fnn = (int64_t)fnnx * fnny * fnnz;
  const int I = blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= cnnx) return;
  const Taps tx = coarse_taps(I, fx, fnx);
  const int nrows = cnny * fnnz * groups;
  for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
    const int J = row % cnny, kg = row / cnny, k = kg % fnnz, g = kg / fnnz;
    const T* bg = b + g * fnn * NC * KC;
    const T* wg = w ? w + g * fnn * NC * KC : nullptr;
    T acc[NC][KC];
#pragma unroll
    for (int d = 0; d < NC; ++d)
#pragma unroll
      for (int c = 0; c < KC; ++c) acc[d][c] = T(0);
    const Taps ty = coarse_taps(J, fy, fny);
    for (int dy = 1 - ty.wl; dy <= ty.wr - 1; ++dy) {
      const int j = ty.x + dy;
      const T wy = T(1) - (dy < 0 ? (T)-dy / (T)ty.wl : (T)dy / (T)ty.wr);
      for (int dx = 1 - tx.wl; dx <= tx.wr - 1; ++dx) {
        const int i = tx.x + dx;
        const T wgt = (T(1) - (dx < 0 ? (T)-dx / (T)tx.wl : (T)dx / (T)tx.wr)) * wy;
        const int64_t fn = i + fnnx * (j + (int64_t)fnny * k);
        T bv[NC * KC], wv[NC * KC];
        load_node<T, NC * KC, KC>(bg + fn * NC * KC, bv);
        if (wg) load_node<T, NC * KC, KC>(wg + fn * NC * KC, wv);
#pragma unroll
        for (int d = 0; d < NC; ++d) {
          if (fixed && fixed[fn * NC + d]) continue;
#pragma unroll
          for (int c = 0; c < KC; ++c)
            acc[d][c] += wgt * (wg ? bv[d * KC + c] - wv[d * KC + c] : bv[d * KC + c]);
        }
      }
    }
    const int64_t tnode = I + cnnx * (J + (int64_t)cnny * k);
    T* out = tbuf + g * tn * NC * KC;
#pragma unroll
    for (int d = 0; d < NC; ++d)
#pragma unroll
      for (int c = 0; c < KC; ++c) out[(tnode * NC + d) * KC + c] = acc[d][c];
  }
}

// Pass 1 for factors of at most 3 where its rows are few: a thread per coarse
// column and component, its up to 5 x 5 fine nodes and their flags loaded
// unpredicated (clamped addresses) before any is used.  The kernel above waits
// for memory at each of its taps.  The same sums in the same order.  33x17x13
// elements, factor 3, 2 float64 columns: 15.0 to 8.2 us; 25x13x13, one float32
// column: 7.4 to 4.9 us.
template <typename T, int NC, int KC, bool HASW>
__global__ void __launch_bounds__(256)
k_restrict_xy_gather(int fnx, int fny, int fnz, int fx, int fy, int groups,
                     const T* __restrict__ b, const T* __restrict__ w,
                     const uint8_t* __restrict__ fixed, T* __restrict__ tbuf) {
  const int fnnx = fnx + 1, fnny = fny + 1, fnnz = fnz + 1;
  const int cnnx = (fnx + fx - 1) / fx + 1, cnny = (fny + fy - 1) / fy + 1;
  const int64_t tn = (int64_t)cnnx * cnny * fnnz, fnn = (int64_t)fnnx * fnny * fnnz;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;  // launched below 2^31
  if (t >= tn * NC * groups) return;
  const int d = t % NC, gn = t / NC, g = gn / (int)tn, node = gn - g * (int)tn;
  const int row = node / cnnx, I = node - row * cnnx, k = row / cnny, J = row - k * cnny;
  const Taps tx = coarse_taps(I, fx, fnx), ty = coarse_taps(J, fy, fny);
  const T* bg = b + g * fnn * NC * KC;
  const T* wg = HASW ? w + g * fnn * NC * KC : nullptr;
  T acc[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) acc[c] = T(0);
  T bv[25][KC], wv[HASW ? 25 : 1][KC];
  uint8_t fx_[25];
#pragma unroll
  for (int o = 0; o < 25; ++o) {
    const int i = min(max(tx.x + o % 5 - 2, 0), fnx), j = min(max(ty.x + o / 5 - 2, 0), fny);
    const int64_t dof = (i + fnnx * (j + (int64_t)fnny * k)) * NC + d;
    load_node<T, KC, KC>(bg + dof * KC, bv[o]);
    if constexpr (HASW) load_node<T, KC, KC>(wg + dof * KC, wv[o]);
    fx_[o] = fixed ? fixed[dof] : 0;
  }
#pragma unroll
  for (int o = 0; o < 25; ++o) {
    const int dx = o % 5 - 2, dy = o / 5 - 2;
    const bool in = dx > -tx.wl && dx < tx.wr && dy > -ty.wl && dy < ty.wr && !fx_[o];
    const T wy = T(1) - (dy < 0 ? (T)-dy / (T)ty.wl : (T)dy / (T)ty.wr);
    const T wgt = (T(1) - (dx < 0 ? (T)-dx / (T)tx.wl : (T)dx / (T)tx.wr)) * wy;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const T n = acc[c] + wgt * (HASW ? bv[o][c] - wv[HASW ? o : 0][c] : bv[o][c]);
      acc[c] = in ? n : acc[c];
    }
  }
  store_node<T, KC, KC>(tbuf + ((g * tn + node) * NC + d) * KC, acc);
}

// Pass 2 (z): b_c(I, J, K) = sum_dz w(dz) t(I, J, f K + dz).  Thread: (I, J);
// row: (K, group).
template <typename T, int NC, int KC>
__global__ void k_restrict_z(int cnnx, int cnny, int fnz, int fz, int groups,
                             const T* __restrict__ tbuf, T* __restrict__ bc) {
  const int fnnz = fnz + 1, cnnz = (fnz + fz - 1) / fz + 1;
  const int64_t plane = (int64_t)cnnx * cnny;
  const int64_t tn = plane * fnnz, cnn = plane * cnnz;
  const int64_t IJ = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (IJ >= plane) return;
  const int nrows = cnnz * groups;
  for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
    const int K = row % cnnz, g = row / cnnz;
    const T* tg = tbuf + g * tn * NC * KC;
    T acc[NC][KC];
#pragma unroll
    for (int d = 0; d < NC; ++d)
#pragma unroll
      for (int c = 0; c < KC; ++c) acc[d][c] = T(0);
    const Taps tz = coarse_taps(K, fz, fnz);
    for (int dz = 1 - tz.wl; dz <= tz.wr - 1; ++dz) {
      const int k = tz.x + dz;
      const T wz = T(1) - (dz < 0 ? (T)-dz / (T)tz.wl : (T)dz / (T)tz.wr);
      const int64_t tnode = IJ + plane * k;
#pragma unroll
      for (int d = 0; d < NC; ++d)
#pragma unroll
        for (int c = 0; c < KC; ++c) acc[d][c] += wz * tg[(tnode * NC + d) * KC + c];
    }
    const int64_t cnode = IJ + plane * K;
    T* out = bc + g * cnn * NC * KC;
#pragma unroll
    for (int d = 0; d < NC; ++d)
#pragma unroll
      for (int c = 0; c < KC; ++c) out[(cnode * NC + d) * KC + c] = acc[d][c];
  }
}

// Restriction for factor 2 on every axis in one pass, b_c = P^T (b - w)
// (HASW: w given).  A 256-thread workgroup owns kR2I x kR2J coarse nodes of
// one column group and a chunk of zlen coarse planes (one where that leaves
// too few workgroups to hide the planes' latency), and streams the fine planes
// 2 K0 - 1 .. 2 K1 - 1 through LDS: per plane, the tile's (2 kR2I + 1) x
// (2 kR2J + 1) fine nodes, each fine row a contiguous run of the blocked
// layout (coalesced), prefetched one plane ahead in registers.  Each thread
// sums its coarse node's 3 x 3 fine neighbourhood on a plane with the
// weights and in the order of k_restrict_xy, and the planes with those of
// k_restrict_z, so the result is the two-pass one bit for bit.  No Dirichlet
// mask is applied: b must be zero at Dirichlet DOFs (the fine residual is) or
// there are none (coarse levels).  With x0 the kernel also writes the coarse
// level's first smoothing iterate from zero, x0 = c2 dinv_c b_c (k_cheb_first
// with c2 = cf[1]).  On an axis of odd length the last coarse node lies on the
// last fine node, the dx = -1 neighbour of where it would be: it takes that
// node with weight 1, and the coarse node before it has no dx = +1 neighbour.
constexpr int kR2I = 32, kR2J = 8;

template <typename T, int NC, int KC, bool HASW>
__global__ void __launch_bounds__(256)
k_restrict222(int fnx, int fny, int fnz, int tiles_x, int tiles_y, int zchunks, int zlen,
              const T* __restrict__ b, const T* __restrict__ w, T* __restrict__ bc,
              const T* __restrict__ dinv_c, const double* __restrict__ cf, T* __restrict__ x0) {
  static_assert(kR2I * kR2J == 256, "one thread per coarse node of a tile");
  constexpr int NV = NC * KC;
  constexpr int kW = 2 * kR2I + 1, kH = 2 * kR2J + 1;  // staged fine nodes per row, rows
  constexpr int kRow = kW * NV;                          // values of one staged row
  constexpr int kM = (kRow + 63) / 64;                   // values per lane per row
  constexpr int kQ = (kH + 3) / 4;                       // rows per wavefront
  __shared__ T sv[NV * kH * kW];                         // [value][row][node]
  const int fnnx = fnx + 1, fnny = fny + 1, fnnz = fnz + 1;
  const int cnnx = (fnx + 1) / 2 + 1, cnny = (fny + 1) / 2 + 1, cnnz = (fnz + 1) / 2 + 1;
  const int64_t fnn = (int64_t)fnnx * fnny * fnnz, cnn = (int64_t)cnnx * cnny * cnnz;
  int blk = blockIdx.x;
  const int tx = blk % tiles_x;
  blk /= tiles_x;
  const int ty = blk % tiles_y;
  blk /= tiles_y;
  const int zc = blk % zchunks;
  const int g = blk / zchunks;
  const int K0 = zc * zlen, K1 = K0 + zlen < cnnz ? K0 + zlen : cnnz;
  const int gx0 = 2 * kR2I * tx - 1, gy0 = 2 * kR2J * ty - 1;
  const T* bg = b + g * fnn * NV;
  const T* wg = HASW ? w + g * fnn * NV : nullptr;
  const int tid = threadIdx.x, lane = tid % 64, wv = tid / 64;
  // staging: wavefront wv takes rows wv, wv + 4, ...; lane l takes values
  // l, l + 64, ... of a row (value e: fine node gx0 + e / NV, component and
  // column e % NV)
  int s_lds[kM];
  unsigned s_ok = 0;
#pragma unroll
  for (int m = 0; m < kM; ++m) {
    const int e = lane + 64 * m;
    const int xn = e / NV, v = e % NV;
    s_lds[m] = (v * kH) * kW + xn;
    if (e < kRow && gx0 + xn >= 0 && gx0 + xn < fnnx) s_ok |= 1u << m;
  }
  T pb[kQ][kM], pw[HASW ? kQ : 1][HASW ? kM : 1];
  auto fetch = [&](int gz) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int r = wv + 4 * q, gy = gy0 + r;
      const bool row_ok = r < kH && gy >= 0 && gy < fnny && gz >= 0 && gz < fnnz;
      const int64_t rowoff = (((int64_t)gz * fnny + gy) * fnnx + gx0) * NV;
#pragma unroll
      for (int m = 0; m < kM; ++m) {
        const bool ok = row_ok && ((s_ok >> m) & 1u);
        const int64_t o = rowoff + lane + 64 * m;
        pb[q][m] = ok ? bg[o] : T(0);
        if constexpr (HASW) pw[q][m] = ok ? wg[o] : T(0);
      }
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int r = wv + 4 * q;
      if (r >= kH) continue;
#pragma unroll
      for (int m = 0; m < kM; ++m) {
        if (lane + 64 * m >= kRow) continue;
        if constexpr (HASW)
          sv[s_lds[m] + r * kW] = pb[q][m] - pw[q][m];
        else
          sv[s_lds[m] + r * kW] = pb[q][m];
      }
    }
  };
  // compute: coarse node (I, J) of the tile, fine node (2 Il + 1, 2 Jl + 1)
  // of the staged plane at its centre
  const int Il = tid % kR2I, Jl = tid / kR2I;
  const int I = tx * kR2I + Il, J = ty * kR2J + Jl;
  const bool own = I < cnnx && J < cnny;
  const T xl = 2 * I > fnx ? T(1) : T(0.5), xr = 2 * I + 1 == fnx ? T(0) : T(0.5);
  const T yl = 2 * J > fny ? T(1) : T(0.5), yr = 2 * J + 1 == fny ? T(0) : T(0.5);
  T acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = T(0);
  const T c2 = x0 ? (T)cf[1] : T(0);
  auto write = [&](int K) {
    if (!own) return;
    const int64_t cn = I + cnnx * (J + (int64_t)cnny * K);
    T* out = bc + (g * cnn + cn) * NV;
#pragma unroll
    for (int v = 0; v < NV; ++v) out[v] = acc[v];
    if (x0) {
      T* xo = x0 + (g * cnn + cn) * NV;
#pragma unroll
      for (int v = 0; v < NV; ++v) xo[v] = c2 * dinv_c[cn * NC + v / KC] * acc[v];
    }
  };
  // planes 2 K0 - 1 .. 2 K1 - 1 that exist
  const int gz_lo = K0 > 0 ? 2 * K0 - 1 : 0, gz_hi = 2 * K1 - 1 < fnz ? 2 * K1 - 1 : fnz;
  fetch(gz_lo);
  for (int gz = gz_lo; gz <= gz_hi; ++gz) {
    stash();
    __syncthreads();
    if (gz < gz_hi) fetch(gz + 1);  // in flight while this plane is summed
    const bool have = gz >= 0 && gz < fnnz;
    T t[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) t[v] = T(0);
    if (have) {
#pragma unroll
      for (int dy = -1; dy <= 1; ++dy) {
        const T wy = dy < 0 ? yl : dy > 0 ? yr : T(1);
#pragma unroll
        for (int dx = -1; dx <= 1; ++dx) {
          const T wgt = (dx < 0 ? xl : dx > 0 ? xr : T(1)) * wy;
          const int node = (2 * Jl + 1 + dy) * kW + 2 * Il + 1 + dx;
#pragma unroll
          for (int v = 0; v < NV; ++v) t[v] += wgt * sv[v * kH * kW + node];
        }
      }
    }
    __syncthreads();  // the next stash overwrites the plane
    // plane gz = 2K + dz contributes wz t to coarse plane K (dz = -1, 0, 1 in
    // this order, as k_restrict_z sums them)
    if (gz & 1) {
      const int K = (gz - 1) >> 1;  // dz = +1 for K, -1 for K + 1
      const bool end = gz == fnz;   // the last coarse plane lies on this one
      if (K >= K0) {
        if (have && !end) {
#pragma unroll
          for (int v = 0; v < NV; ++v) acc[v] += T(0.5) * t[v];
        }
        write(K);
      }
#pragma unroll
      for (int v = 0; v < NV; ++v) acc[v] = T(0);
      if (have && K + 1 < K1) {
        const T wz = end ? T(1) : T(0.5);
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] += wz * t[v];
        if (end) write(K + 1);
      }
    } else {
      const int K = gz >> 1;
#pragma unroll
      for (int v = 0; v < NV; ++v) acc[v] += T(1) * t[v];
      if (gz + 1 >= fnnz) write(K);  // the last plane: no dz = +1 term
    }
  }
}

// The same restriction where its tiles leave CUs idle: a thread per coarse node,
// component and column group gathers its 27 fine nodes straight from memory, all
// loads unpredicated (clamped addresses, weight zero), with the weights and in
// the order of k_restrict222 and the two passes, so the result is theirs bit for
// bit.  One wait for memory in place of one per staged plane: 21x11x11 coarse
// nodes, 8 float32 columns, 8.8 to 5.0 us, and 8.3 to 5.8 us with w.
template <typename T, int NC, int KC, bool HASW>
__global__ void __launch_bounds__(256)
k_restrict_gather(int fnx, int fny, int fnz, int groups, const T* __restrict__ b,
                  const T* __restrict__ w, T* __restrict__ bc, const T* __restrict__ dinv_c,
                  const double* __restrict__ cf, T* __restrict__ x0) {
  const int fnnx = fnx + 1, fnny = fny + 1, fnnz = fnz + 1;
  const int cnnx = (fnx + 1) / 2 + 1, cnny = (fny + 1) / 2 + 1, cnnz = (fnz + 1) / 2 + 1;
  const int64_t fnn = (int64_t)fnnx * fnny * fnnz, cnn = (int64_t)cnnx * cnny * cnnz;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= cnn * NC * groups) return;
  const int d = (int)(t % NC);
  const int64_t cn = t / NC % cnn, g = t / (NC * cnn);
  const int I = (int)(cn % cnnx), J = (int)(cn / cnnx % cnny), K = (int)(cn / ((int64_t)cnnx * cnny));
  // weights of the neighbours -1, 0, 1 (0 where there is none)
  T wx[3], wy[3], wz[3];
  int ix[3], iy[3], iz[3];
  auto axis = [](int C, int fn, T(&wt)[3], int(&at)[3]) {
    wt[0] = C == 0 ? T(0) : 2 * C > fn ? T(1) : T(0.5);
    wt[1] = 2 * C > fn ? T(0) : T(1);
    wt[2] = 2 * C + 1 >= fn ? T(0) : T(0.5);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int f = 2 * C + k - 1;
      at[k] = f < 0 ? 0 : f > fn ? fn : f;
    }
  };
  axis(I, fnx, wx, ix);
  axis(J, fny, wy, iy);
  axis(K, fnz, wz, iz);
  const T* bg = b + (g * fnn * NC + d) * KC;
  const T* wg = HASW ? w + (g * fnn * NC + d) * KC : nullptr;
  T v[27][KC], r[HASW ? 27 : 1][KC];
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    const int64_t off =
        (ix[o % 3] + (int64_t)fnnx * (iy[o / 3 % 3] + (int64_t)fnny * iz[o / 9])) * NC * KC;
    load_node<T, KC, KC>(bg + off, v[o]);
    if constexpr (HASW) load_node<T, KC, KC>(wg + off, r[o]);
  }
  T acc[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) acc[c] = T(0);
#pragma unroll
  for (int dz = 0; dz < 3; ++dz) {
    T s[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) s[c] = T(0);
#pragma unroll
    for (int o = 0; o < 9; ++o) {
      const T wgt = wx[o % 3] * wy[o / 3];
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const T q = HASW ? v[9 * dz + o][c] - r[HASW ? 9 * dz + o : 0][c] : v[9 * dz + o][c];
        const T n = s[c] + wgt * q;
        s[c] = wgt != T(0) ? n : s[c];
      }
    }
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const T n = acc[c] + wz[dz] * s[c];
      acc[c] = wz[dz] != T(0) ? n : acc[c];
    }
  }
  const int64_t at = ((g * cnn + cn) * NC + d) * KC;
  store_node<T, KC, KC>(bc + at, acc);
  if (x0) {
    const T s = (T)cf[1] * dinv_c[cn * NC + d];
#pragma unroll
    for (int c = 0; c < KC; ++c) acc[c] = s * acc[c];
    store_node<T, KC, KC>(x0 + at, acc);
  }
}

// x_f += Z P x_c.  Thread: fine i; row: (j, k, group).  FIX: Dirichlet flags
// of the fine level (no correction on fixed DOFs).  Every load of a row (the
// 8 coarse corners, the fine node, its flags) is unpredicated and issued
// before any is used: a corner outside the interpolation (weight zero) reads
// a clamped node and is dropped by a select, so the sums are those of the
// loop that skips it.  Predicated loads compiled to one branch and one wait
// each.
template <typename T, int NC, int KC, bool FIX>
__global__ void k_prolong_add(int fnx, int fny, int fnz, int fx, int fy, int fz, int groups,
                              const T* __restrict__ xc, const uint8_t* __restrict__ fixed,
                              T* __restrict__ xf) {
  const int fnnx = fnx + 1, fnny = fny + 1, fnnz = fnz + 1;
  const int cnnx = (fnx + fx - 1) / fx + 1, cnny = (fny + fy - 1) / fy + 1,
            cnnz = (fnz + fz - 1) / fz + 1;
  const int64_t cnn = (int64_t)cnnx * cnny * cnnz, fnn = (int64_t)fnnx * fnny * fnnz;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= fnnx) return;
  // the coarse element at the end of an axis may hold fewer fine elements
  const int I = i / fx, ax = i - I * fx;
  const T sx = (T)ax / (T)interval(fnx, I, fx);
  const int nrows = fnny * fnnz * groups;
  for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
    const int j = row % fnny, kg = row / fnny, k = kg % fnnz, g = kg / fnnz;
    const int J = j / fy, ay = j - J * fy, K = k / fz, az = k - K * fz;
    const T sy = (T)ay / (T)interval(fny, J, fy), sz = (T)az / (T)interval(fnz, K, fz);
    const int64_t fnode = i + fnnx * (j + (int64_t)fnny * k);
    const T* xg = xc + g * cnn * NC * KC;
    T* xfn = xf + (g * fnn + fnode) * NC * KC;
    uint8_t fv[NC];
    if constexpr (FIX) {
#pragma unroll
      for (int d = 0; d < NC; ++d) fv[d] = fixed[fnode * NC + d];
    }
    T out[NC * KC];
    load_node<T, NC * KC, KC>(xfn, out);
    T xv[8][NC * KC];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      // the +1 corner exists wherever its weight is nonzero
      const int qx = (q & 1) && ax != 0, qy = ((q >> 1) & 1) && ay != 0, qz = (q >> 2) && az != 0;
      const int64_t cn = (I + qx) + cnnx * ((J + qy) + (int64_t)cnny * (K + qz));
      load_node<T, NC * KC, KC>(xg + cn * NC * KC, xv[q]);
    }
    T acc[NC][KC];
#pragma unroll
    for (int d = 0; d < NC; ++d)
#pragma unroll
      for (int c = 0; c < KC; ++c) acc[d][c] = T(0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int qx = q & 1, qy = (q >> 1) & 1, qz = q >> 2;
      const bool skip = (qx && ax == 0) || (qy && ay == 0) || (qz && az == 0);
      const T wgt = (qx ? sx : T(1) - sx) * (qy ? sy : T(1) - sy) * (qz ? sz : T(1) - sz);
#pragma unroll
      for (int d = 0; d < NC; ++d)
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const T a = acc[d][c] + wgt * xv[q][d * KC + c];
          acc[d][c] = skip ? acc[d][c] : a;
        }
    }
#pragma unroll
    for (int d = 0; d < NC; ++d) {
      const bool keep = FIX && fv[d] != 0;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const T a = out[d * KC + c] + acc[d][c];
        out[d * KC + c] = keep ? out[d * KC + c] : a;
      }
    }
    store_node<T, NC * KC, KC>(xfn, out);
  }
}

// x = Ainv b on the coarsest level: one wavefront per (row, column group),
// lanes stride the row, fixed-order wave reduction
template <typename T, int KC>
__global__ void __launch_bounds__(256) k_dense_apply(int64_t n, int groups,
                                                     const T* __restrict__ Ainv,
                                                     const T* __restrict__ b,
                                                     T* __restrict__ x) {
  const int lane = threadIdx.x % kWave;
  const int64_t wid = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / kWave;
  if (wid >= n * groups) return;
  const int64_t row = wid % n, g = wid / n;
  const T* bg = b + g * n * KC;
  double acc[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) acc[c] = 0.0;
  for (int64_t j = lane; j < n; j += kWave) {
    const double a = (double)Ainv[row * n + j];
#pragma unroll
    for (int c = 0; c < KC; ++c) acc[c] += a * (double)bg[j * KC + c];
  }
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    const double v = wave_sum(acc[c]);
    if (lane == 0) x[(g * n + row) * KC + c] = (T)v;
  }
}

// The same product with every column group in one pass over Ainv: b (all G
// groups, G * KC columns) is staged in LDS node-major, and each wavefront
// takes R consecutive rows, so a row of Ainv is read once rather than once
// per group, and each b value read from LDS feeds R rows.  A lane's NJ values
// of its rows (n <= 64 NJ) are loaded into registers before the staging, so
// that every load of the launch is in flight at once.  Per (row, column) the
// lane sums and the wave reduction run in k_dense_apply's order, so the
// results are bit-identical to it.
template <typename T, int KC, int G, int R, int NJ>
__global__ void __launch_bounds__(256) k_dense_apply_rows(int n, const T* __restrict__ Ainv,
                                                          const T* __restrict__ b,
                                                          T* __restrict__ x) {
  constexpr int GK = G * KC;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* bl = reinterpret_cast<T*>(smem_raw);  // [n][GK]
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int row0 = (blockIdx.x * (256 / kWave) + tid / kWave) * R;
  const bool live = row0 < n;
  // unpredicated loads (row and column clamped into the matrix; the clamped
  // values are never used), so that none waits for the one before
  T av[R][NJ];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const T* ar = Ainv + (int64_t)(row0 + r < n ? row0 + r : n - 1) * n;
#pragma unroll
    for (int t = 0; t < NJ; ++t) {
      const int j = lane + kWave * t;
      av[r][t] = ar[j < n ? j : n - 1];
    }
  }
  // b: a thread's NBG values of every group are loaded (again unpredicated,
  // clamped) before any is stored
  constexpr int NBG = (kWave * NJ * KC + 255) / 256;
  const int nk = n * KC;
  T sb[G][NBG];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int u = 0; u < NBG; ++u) {
      const int i = tid + 256 * u;
      sb[g][u] = b[(int64_t)g * nk + (i < nk ? i : nk - 1)];
    }
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int u = 0; u < NBG; ++u) {
      const int i = tid + 256 * u;
      if (i < nk) {
        const int j = i / KC, c = i - j * KC;
        bl[j * GK + g * KC + c] = sb[g][u];
      }
    }
  __syncthreads();
  if (!live) return;
  double acc[R][GK];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < GK; ++c) acc[r][c] = 0.0;
#pragma unroll
  for (int t = 0; t < NJ; ++t) {
    const int j = lane + kWave * t;
    if (j < n) {
      double bv[GK];
#pragma unroll
      for (int c = 0; c < GK; ++c) bv[c] = (double)bl[j * GK + c];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double a = (double)av[r][t];
#pragma unroll
        for (int c = 0; c < GK; ++c) acc[r][c] += a * bv[c];
      }
    }
  }
  // wave_sum's butterfly, one step for all R * GK sums at a time, so that
  // their exchanges are in flight together
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1)
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < GK; ++c) acc[r][c] += __shfl_xor(acc[r][c], off, kWave);
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = row0 + r;
      if (row >= n) continue;
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < KC; ++c) x[((int64_t)g * n + row) * KC + c] = (T)acc[r][g * KC + c];
    }
  }
}

template <typename T, int KC, int R, int NJ>
static bool launch_dense_rows(int n, int groups, const T* Ainv, const T* b, T* x,
                              hipStream_t s) {
  const size_t lds = (size_t)n * groups * KC * sizeof(T);
  const dim3 grid((unsigned)((n + 4 * R - 1) / (4 * R)));
  switch (groups) {
    case 1:
      hipLaunchKernelGGL((k_dense_apply_rows<T, KC, 1, R, NJ>), grid, dim3(256), lds, s, n,
                         Ainv, b, x);
      return true;
    case 2:
      hipLaunchKernelGGL((k_dense_apply_rows<T, KC, 2, R, NJ>), grid, dim3(256), lds, s, n,
                         Ainv, b, x);
      return true;
    case 4:
      hipLaunchKernelGGL((k_dense_apply_rows<T, KC, 4, R, NJ>), grid, dim3(256), lds, s, n,
                         Ainv, b, x);
      return true;
    default:
      return false;
  }
}

// SKT_MG_DENSE_APPLY=wave: one wavefront per (row, group) at every size
static bool dense_rows_enabled() {
  const char* v = std::getenv("SKT_MG_DENSE_APPLY");
  return !(v && std::strcmp(v, "wave") == 0);
}

// x = Ainv b for `groups` column groups of KC: the row-blocked kernel when b
// fits in 64 KB of LDS, n <= 2048 and the group count is 1, 2 or 4, else one
// wavefront per (row, group)
template <typename T, int KC>
static void launch_dense_apply(int64_t n, int groups, const T* Ainv, const T* b, T* x,
                               hipStream_t s) {
  const size_t lds = (size_t)n * groups * KC * sizeof(T);
  if (lds <= 65536 && n <= 64 * 32 && dense_rows_enabled()) {
    if (n <= 64 * 8 ? launch_dense_rows<T, KC, 2, 8>((int)n, groups, Ainv, b, x, s)
                    : launch_dense_rows<T, KC, 2, 32>((int)n, groups, Ainv, b, x, s))
      return;
  }
  const int64_t waves = n * groups;
  hipLaunchKernelGGL((k_dense_apply<T, KC>), dim3((unsigned)((waves * kWave + 255) / 256)),
                     dim3(256), 0, s, n, groups, Ainv, b, x);
}

// ------------------------------------------------- smoother bounds (power)

__device__ __forceinline__ double hash_unit(int64_t i) {
  uint64_t z = (uint64_t)i * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (double)(z >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
}

template <typename T>
__global__ void k_pow_init(int64_t n, const T* __restrict__ dinv, T* __restrict__ v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    v[i] = dinv[i] != T(0) ? (T)hash_unit(i) : T(0);
}

// y <- dinv y (if scale_by_dinv), partial sums of y^2 per block
template <typename T>
__global__ void k_pow_norm(int64_t n, const T* __restrict__ dinv, T* __restrict__ y,
                           int scale_by_dinv, double* __restrict__ part) {
  __shared__ double sh[kBlock / kWave];
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    T v = y[i];
    if (scale_by_dinv) { v *= dinv[i]; y[i] = v; }
    acc += (double)v * (double)v;
  }
  const double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// norm = sqrt(sum part); inv_out = 1 / norm.  With lam_out, lam = norm *
// inv_in (inv_in: 1 / the norm of the vector the operator was applied to).
__global__ void k_pow_finish(int nb, const double* __restrict__ part, double* __restrict__ lam_out,
                             const double* __restrict__ inv_in, double* __restrict__ inv_out) {
  __shared__ double sh[kBlock / kWave];
  double a = 0.0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) a += part[i];
  const double s = block_sum(a, sh);
  if (threadIdx.x == 0) {
    const double nrm = sqrt(s);
    if (lam_out) *lam_out = nrm * *inv_in;
    *inv_out = nrm > 0.0 ? 1.0 / nrm : 0.0;
  }
}

// v = dinv y (an unnormalised power step)
template <typename T>
__global__ void k_pow_dscale(int64_t n, const T* __restrict__ dinv, const T* __restrict__ y,
                             T* __restrict__ v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    v[i] = dinv[i] * y[i];
}

template <typename T>
__global__ void k_pow_scale(int64_t n, const double* __restrict__ inv, const T* __restrict__ y,
                            T* __restrict__ v) {
  const T s = (T)*inv;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    v[i] = y[i] * s;
}

// Chebyshev (c1, c2) per step for the interval [beta/ratio, beta]; the last
// level takes ratio_low.  The residual polynomial stays below 1 in magnitude,
// and the cycle positive definite, up to beta (1 + 1/ratio): beta is chosen so
// that this is `margin` times the power iteration's estimate for every ratio.
__global__ void k_cheb_coef(int nlev, int degree, double ratio, double ratio_low, double margin,
                            const double* __restrict__ lam, double* __restrict__ coef) {
  const int l = threadIdx.x;
  if (l >= nlev) return;
  const double r = l > 0 && l == nlev - 1 ? ratio_low : ratio;
  const double bmax = margin / (1.0 + 1.0 / r) * lam[l];
  const double amin = bmax / r;
  const double theta = 0.5 * (bmax + amin), delta = 0.5 * (bmax - amin);
  const double sigma = theta / delta;
  double* c = coef + (size_t)l * 2 * degree;
  double rho_old = 1.0 / sigma;
  c[0] = 0.0;
  c[1] = 1.0 / theta;
  for (int s = 1; s < degree; ++s) {
    const double rho = 1.0 / (2.0 * sigma - rho_old);
    c[2 * s] = rho * rho_old;
    c[2 * s + 1] = 2.0 * rho / delta;
    rho_old = rho;
  }
}

// ------------------------------------------------------------ host side

// Chebyshev steps whose coefficients are kept per level
static int coef_steps(const MGData* mg) { return mg->degree + kLowSteps; }

static int64_t gj_pad(int64_t n) { return (n + kGJ - 1) / kGJ * kGJ; }

static size_t tsize(int dtype) { return dtype == SKT_F64 ? sizeof(double) : sizeof(float); }

void mg_free(MGData* mg) {
  // the set-up's side work and any background inverse are done
  if (mg->side) (void)hipStreamSynchronize(mg->side);
  if (mg->side2) (void)hipStreamSynchronize(mg->side2);
  if (mg->gjs) {
    (void)hipStreamSynchronize(mg->gjs);
    (void)hipStreamDestroy(mg->gjs);
    (void)hipEventDestroy(mg->ev_asm);
    (void)hipEventDestroy(mg->ev_gj);
    mg->gjs = nullptr;
    mg->ev_asm = mg->ev_gj = nullptr;
  }
  mg->have_inv = 0;
  mg->inv_pending = 0;
  for (hipEvent_t& e : mg->tev)
    if (e) {
      (void)hipEventDestroy(e);
      e = nullptr;
    }
  mg->tcount = 0;
  mg->time_fine = 0;
  for (MGLevel& l : mg->lv) {
    (void)hipFree(l.Kel); (void)hipFree(l.st); (void)hipFree(l.dinv);
    (void)hipFree(l.b); (void)hipFree(l.x); (void)hipFree(l.w); (void)hipFree(l.d);
    (void)hipFree(l.rt);
    l.Kel = nullptr; l.st = l.dinv = l.b = l.x = l.w = l.d = l.rt = nullptr;
  }
  (void)hipFree(mg->Ad); (void)hipFree(mg->Ad2); (void)hipFree(mg->Ainv);
  (void)hipFree(mg->lam); (void)hipFree(mg->coef); (void)hipFree(mg->part); (void)hipFree(mg->pv);
  (void)hipFree(mg->pvw);
  (void)hipFree(mg->K0b);
  if (mg->side) {
    (void)hipStreamDestroy(mg->side);
    (void)hipStreamDestroy(mg->side2);
    (void)hipEventDestroy(mg->ev_fork);
    (void)hipEventDestroy(mg->ev_gal);
    (void)hipEventDestroy(mg->ev_st);
    (void)hipEventDestroy(mg->ev_join);
    mg->side = mg->side2 = nullptr;
    mg->ev_fork = mg->ev_gal = mg->ev_st = mg->ev_join = nullptr;
  }
  (void)hipFree(mg->Mch);
  (void)hipFree(mg->gflag);
  mg->Mch = nullptr;
  mg->gflag = nullptr;
  mg->Ad = mg->Ad2 = nullptr; mg->Ainv = nullptr; mg->lam = mg->coef = mg->part = nullptr;
  mg->K0b = nullptr;
  mg->pv = nullptr;
  mg->pvw = nullptr;
  mg->warm = 0;
  mg->lv.clear();
  mg->dtype = -1;
}

// Stencil layout of a level with nn nodes: big tiles from kTiledNodes
// nodes, small tiles below.  SKT_MG_STENCIL_LAYOUT=node|big|small forces one
// layout on every level (read when a hierarchy is allocated; the three sum
// in the same order, which a test checks).
static int stencil_layout(int64_t nn) {
  const char* v = std::getenv("SKT_MG_STENCIL_LAYOUT");
  if (v && std::strcmp(v, "node") == 0) return ST_NODE;
  if (v && std::strcmp(v, "big") == 0) return ST_TILE_BIG;
  if (v && std::strcmp(v, "small") == 0) return ST_TILE_SMALL;
  return nn >= kTiledNodes ? ST_TILE_BIG : ST_TILE_SMALL;
}

// Power-iteration steps from the previous set-up's vector;
// SKT_MG_POWER_WARM=n (1..64) overrides the default.
static int warm_power_steps(const MGData* mg) {
  const char* v = std::getenv("SKT_MG_POWER_WARM");
  if (v) {
    const int n = std::atoi(v);
    if (n >= 1 && n <= 64) return n;
  }
  return mg->power_iters_warm;
}

int mg_warm_steps(const MGData* mg) { return warm_power_steps(mg); }

// SKT_MG_CHEB0=0 runs a degree-2 fine-level smoothing as the separate first
// step plus one fused step instead of the single two-step pass (the same
// arithmetic; a test checks that the solves agree bit for bit).
static bool cheb0_enabled() {
  const char* v = std::getenv("SKT_MG_CHEB0");
  return !(v && v[0] == '0' && v[1] == 0);
}

// SKT_MG_COARSE_REFRESH=n (1..64): set-ups one coarsest inverse may serve.
int mg_coarse_refresh(const MGData* mg) {
  const char* v = std::getenv("SKT_MG_COARSE_REFRESH");
  if (v) {
    const int n = std::atoi(v);
    if (n >= 1 && n <= 64) return n;
  }
  return mg->coarse_refresh;
}

static int lag_enabled() {
  const char* v = std::getenv("SKT_MG_LAG");
  return (v && v[0] == '1' && v[1] == 0) ? 1 : 0;
}

int mg_alloc(MGData* mg, const skt_operator* op, const MGConfig& cfg, int dtype, int max_cols) {
  if (mg->dtype == dtype && mg->max_cols == max_cols) return SKT_OK;
  SKT_CHECK((op->nx + 1) * (op->ny + 1) < INT32_MAX &&
                (op->ny + 1) * (op->nz + 1) * (int64_t)max_cols < INT32_MAX,
            "grid too large for the multigrid transfers' 32-bit row indices");
  mg_free(mg);
  std::vector<MGLevel>& lv = mg->lv;  // mg_free returns what a failed call allocated
  if (!mg_plan(op, cfg, &lv)) {
    set_error("grid cannot be coarsened for multigrid");
    return SKT_EINVAL;
  }
  int singular = 0;
  if (int stt = singular_operator(op, &singular)) return stt;
  mg->shift = singular ? kNullShift : 0.0;
  const int NC = op->ncomp, ND = 8 * NC;
  const size_t ts = tsize(dtype);
  const int L = (int)lv.size() - 1;
  for (int l = 0; l <= L; ++l) {
    MGLevel& v = lv[l];
    const size_t nv = (size_t)v.ndof * max_cols;
    if (l == 0) {
      SKT_HIP(hipMalloc(&v.x, ts * nv));
      continue;
    }
    SKT_HIP(hipMalloc(&v.Kel, sizeof(double) * (size_t)(v.nx * v.ny * v.nz) * ND * ND));
    SKT_HIP(hipMalloc(&v.rt, ts * (size_t)(v.nx + 1) * (v.ny + 1) * (lv[l - 1].nz + 1) * NC *
                                 max_cols));
    SKT_HIP(hipMalloc(&v.b, ts * nv));
    SKT_HIP(hipMalloc(&v.x, ts * nv));
    if (l < L) {
      v.layout = stencil_layout(v.nn);
      SKT_HIP(hipMalloc(&v.st, ts * (size_t)st_nodes(v.nx, v.ny, v.nz, v.layout) * 27 * NC * NC));
      SKT_HIP(hipMalloc(&v.dinv, ts * v.ndof));
      SKT_HIP(hipMalloc(&v.w, ts * nv));
      SKT_HIP(hipMalloc(&v.d, ts * nv));
    }
  }
  const int64_t nc = lv[L].ndof;
  SKT_HIP(hipMalloc(&mg->Ad, sizeof(double) * 2 * gj_pad(nc) * gj_pad(nc)));
  SKT_HIP(hipMalloc(&mg->Ad2, sizeof(double) * 2 * kGJ * kGJ));
  SKT_HIP(hipMalloc(&mg->Ainv, ts * nc * nc));
  SKT_HIP(hipMalloc(&mg->lam, sizeof(double) * (L + 1) * 2));
  SKT_HIP(hipMalloc(&mg->coef, sizeof(double) * (L + 1) * 2 * (std::max(cfg.degree, 1) + kLowSteps)));
  SKT_HIP(hipMalloc(&mg->part, sizeof(double) * 1024));
  SKT_HIP(hipMalloc(&mg->pv, ts * 2 * lv[0].ndof));
  int64_t npw = 0;
  for (int l = 0; l < L; ++l) npw += lv[l].ndof;
  SKT_HIP(hipMalloc(&mg->pvw, ts * npw));
  mg->warm = 0;
  // unit element matrix in corner-bit order
  std::vector<double> K0b((size_t)ND * ND);
  for (int A = 0; A < 8; ++A)
    for (int B = 0; B < 8; ++B) {
      const int a = corner_id_h(A & 1, (A >> 1) & 1, A >> 2);
      const int b = corner_id_h(B & 1, (B >> 1) & 1, B >> 2);
      for (int d = 0; d < NC; ++d)
        for (int e = 0; e < NC; ++e)
          K0b[(A * NC + d) * ND + B * NC + e] = op->K0h[(a * NC + d) * ND + b * NC + e];
    }
  SKT_HIP(hipMalloc(&mg->K0b, sizeof(double) * K0b.size()));
  SKT_HIP(hipMemcpy(mg->K0b, K0b.data(), sizeof(double) * K0b.size(), hipMemcpyHostToDevice));
  mg->dtype = dtype;
  ++mg->gen;
  mg->max_cols = max_cols;
  mg->degree = std::max(cfg.degree, 1);
  mg->low_steps = NC == 3 ? kLowSteps : 0;
  mg->ratio = NC == 3 ? cfg.ratio : cfg.ratio_scalar;
  if (const char* rv = std::getenv("SKT_MG_RATIO")) {  // smoothing interval [lambda/r, lambda]
    const double r = std::atof(rv);
    if (r > 1.0 && r < 1000.0) mg->ratio = r;
  }
  mg->margin = kChebMargin;
  if (const char* mv = std::getenv("SKT_MG_MARGIN")) {  // below 1 the cycle is not definite
    const double m = std::atof(mv);
    if (m > 0.0 && m <= 4.0) mg->margin = m;
  }
  mg->power_iters = cfg.power_iters;
  mg->lag = lag_enabled();
  return SKT_OK;
}

// apply of level l (k columns, group kc) in T
template <typename T, int MODE = ST_APPLY>
static int level_apply(MGData* mg, const skt_operator* op, const void* E, int l, int k, int kc,
                       const T* x, T* y, hipStream_t s, StOut<T> oa = StOut<T>()) {
  if (l == 0) return op_apply(const_cast<skt_operator*>(op), mg->dtype, k, kc, E, x, y, s);
  const MGLevel& v = mg->lv[l];
  const int groups = k / kc;
  const T* st = (const T*)v.st;
  // tile-major levels: LDS-tiled kernel of the level's tile shape (x staged
  // once per tile); node-major: one (node, row, column group) per thread.
  // A workgroup takes up to GMT column groups, which read the tile's
  // coefficients once.  One group per workgroup where there is only one (the
  // kernel sums all GM groups it is compiled for; one float32 column, a
  // Chebyshev step: 9.7 to 8.9 us on 50x25x25 elements, 6.2 to 4.7 us on
  // 25x13x13), or where the tiles with GMT groups are fewer than the CUs
  // (20x10x10 elements, 8 float32 columns: 72 workgroups, 7.1 us; 288 with one
  // group each, 5.2 us).  40x20x20, 8 loads: 3.98 to 3.71 ms per OC iteration,
  // 75x45x30, 3 loads: 8.34 to 7.75 ms per solve.  With more workgroups the
  // coefficients' second and third read costs more: at a limit of 512, 120x60x60
  // with 8 loads takes 17.1 instead of 15.9 ms, 66x36x28 with 3 loads 5.82
  // instead of 5.59, though 75x45x30 takes 7.57.
  constexpr int GMT = sizeof(T) == 4 ? 4 : 2;  // <= 62 KB of LDS for NC * KC = 6
  const TileShape ts = tile_shape(v.layout);
  const int64_t tiles = v.layout == ST_NODE ? 0 : st_tiles(v.nx, v.ny, v.nz, ts);
  const unsigned gmb = (unsigned)((groups + GMT - 1) / GMT);
  const bool single = groups == 1 || tiles * gmb < 256;
  const unsigned gt = (unsigned)(tiles * (single ? groups : gmb));
  const unsigned g = grid_for(v.nn * op->ncomp * groups);
#define SKT_ST(NC_, KC_, GM_, S_)                                                                \
  hipLaunchKernelGGL((k_stencil_apply_tiled<T, NC_, KC_, GM_, MODE, S_.x, S_.y, S_.z>), dim3(gt), \
                     dim3(S_.x * S_.y * S_.z * NC_), 0, s, v.nx, v.ny, v.nz, groups, st, x, y, oa)
#define SKT_SA(NC_, KC_)                                                                         \
  do {                                                                                           \
    if (v.layout == ST_TILE_BIG) {                                                               \
      if (single) SKT_ST(NC_, KC_, 1, kTileBig);                                                 \
      else SKT_ST(NC_, KC_, GMT, kTileBig);                                                      \
    } else if (v.layout == ST_TILE_SMALL) {                                                      \
      if (single) SKT_ST(NC_, KC_, 1, kTileSmall);                                               \
      else SKT_ST(NC_, KC_, GMT, kTileSmall);                                                    \
    } else {                                                                                     \
      hipLaunchKernelGGL((k_stencil_apply<T, NC_, KC_, 1, MODE>), dim3(g), dim3(kBlock), 0, s,    \
                         v.nx, v.ny, v.nz, groups, st, x, y, oa);                                \
    }                                                                                            \
  } while (0)
  if (op->ncomp == 3) {
    if (kc == 1) SKT_SA(3, 1);
    else if (kc == 2) SKT_SA(3, 2);
    else { set_error("unsupported column block"); return SKT_EINVAL; }
  } else {
    if (kc == 1) SKT_SA(1, 1);
    else if (kc == 2) SKT_SA(1, 2);
    else if (kc == 4) SKT_SA(1, 4);
    else { set_error("unsupported column block"); return SKT_EINVAL; }
  }
#undef SKT_SA
#undef SKT_ST
  SKT_LAUNCH_CHECK();
  return SKT_OK;
}

// One fused Chebyshev-Jacobi step on a stencil level: x_out = x + c1 (x -
// x_out_before) + c2 dinv (b - S x).
template <typename T>
static int level_cheb(MGData* mg, const skt_operator* op, int l, int k, int kc, const T* x,
                      T* xout, const double* coef, int prev_zero, hipStream_t s,
                      const double* stop) {
  const MGLevel& v = mg->lv[l];
  StOut<T> oa;
  oa.b = (const T*)v.b;
  oa.dinv = (const T*)v.dinv;
  oa.coef = coef;
  oa.prev_zero = prev_zero;
  oa.stop = stop;
  return level_apply<T, ST_CHEB>(mg, op, nullptr, l, k, kc, x, xout, s, oa);
}

// Blocked Gauss-Jordan inverse of the coarsest matrix in Ad, on stream g; the
// result is at gj_result (pivot block inverses alternate between the two
// halves of Ad2).
static void queue_gj(MGData* mg, hipStream_t g) {
  const int np = (int)gj_pad(mg->lv.back().ndof), T = np / kGJ;
  double *in = mg->Ad, *out = mg->Ad + (int64_t)np * np;
  double *p = mg->Ad2, *pn = mg->Ad2 + kGJ * kGJ;
  hipLaunchKernelGGL(k_gj_first, dim3(1), dim3(256), 0, g, np, (const double*)in, p);
  for (int b = 0; b < T; ++b) {
    hipLaunchKernelGGL(k_gj_step, dim3((unsigned)(T * T)), dim3(256), 0, g, np, b,
                       (const double*)in, (const double*)p, out, pn);
    std::swap(in, out);
    std::swap(p, pn);
  }
}

static const double* gj_result(const MGData* mg) {
  const int64_t np = gj_pad(mg->lv.back().ndof);
  return mg->Ad + (np / kGJ % 2 ? np * np : 0);
}

// the inverse in the cycle's precision
template <typename T>
static void queue_cast(MGData* mg, hipStream_t g) {
  const int64_t n = mg->lv.back().ndof;
  hipLaunchKernelGGL(k_cast<T>, dim3(grid_for(n * n)), dim3(kBlock), 0, g, n, gj_pad(n),
                     gj_result(mg), (T*)mg->Ainv);
}

bool mg_lagged(const MGData* mg) { return mg->lag && mg->have_inv; }

int mg_set_timing(MGData* mg, int enable) {
  if (enable && !mg->tev[0])
    for (hipEvent_t& e : mg->tev) SKT_HIP(hipEventCreate(&e));
  mg->time_fine = enable ? 1 : 0;
  return SKT_OK;
}

int mg_collect_timing(MGData* mg) {
  for (int i = 0; i < mg->tcount; ++i) {
    if (mg->ttag[i] < 0) continue;
    float ms = 0.f;
    SKT_HIP(hipEventElapsedTime(&ms, mg->tev[2 * i], mg->tev[2 * i + 1]));
    mg->tms[mg->ttag[i]] += ms;
    mg->tn[mg->ttag[i]] += 1;
  }
  mg->tcount = 0;
  return SKT_OK;
}

// event pair around one fine-level launch when timing (at most kTimedMax
// between two collections; later launches go untimed)
static int fine_timer_begin(MGData* mg, int tag, hipStream_t) {
  if (!mg->time_fine || mg->tcount >= MGData::kTimedMax) return -1;
  const int i = mg->tcount++;
  mg->ttag[i] = tag;
  modal_time_next(mg->tev[2 * i], mg->tev[2 * i + 1]);
  return i;
}

// a request that no launch took leaves its events unrecorded: drop the slot
static void fine_timer_end(MGData* mg, int i, hipStream_t) {
  if (i >= 0 && modal_time_clear()) mg->ttag[i] = -1;
}

int mg_lag_pre(MGData* mg, hipStream_t s) {
  if (!mg->inv_pending) return SKT_OK;
  SKT_HIP(hipStreamWaitEvent(s, mg->ev_gj, 0));
  if (mg->dtype == SKT_F64) queue_cast<double>(mg, s);
  else queue_cast<float>(mg, s);
  SKT_LAUNCH_CHECK();
  mg->inv_pending = 0;
  return SKT_OK;
}

int mg_lag_post(MGData* mg, hipStream_t s) {
  if (!mg->gjs) {
    SKT_HIP(hipStreamCreateWithFlags(&mg->gjs, hipStreamNonBlocking));
    SKT_HIP(hipEventCreateWithFlags(&mg->ev_asm, hipEventDisableTiming));
    SKT_HIP(hipEventCreateWithFlags(&mg->ev_gj, hipEventDisableTiming));
  }
  SKT_HIP(hipEventRecord(mg->ev_asm, s));
  SKT_HIP(hipStreamWaitEvent(mg->gjs, mg->ev_asm, 0));
  queue_gj(mg, mg->gjs);
  SKT_LAUNCH_CHECK();
  SKT_HIP(hipEventRecord(mg->ev_gj, mg->gjs));
  mg->inv_pending = 1;
  return SKT_OK;
}

template <typename T>
static int setup_t(MGData* mg, const skt_operator* op, const double* E64, const void* E,
                   const void* dinv0, hipStream_t s) {
  const int NC = op->ncomp, ND = 8 * NC;
  const int L = (int)mg->lv.size() - 1;
  const double* dK0 = mg->K0b;
  // The hierarchy is built on side streams while the main stream runs the
  // power iterations: `side` takes the Galerkin products and then the
  // coarsest inverse, `side2` the stencils and Jacobi inverses once the
  // products they need are done (ev_gal).  The fine level's power iteration
  // needs only the fine operator, the coarse levels' wait for the stencils
  // (ev_st), and the set-up joins the coarsest inverse (ev_join) before
  // returning.  The side streams touch the level matrices, stencils, Jacobi
  // inverses and the coarsest buffers only.
  if (!mg->side) {
    SKT_HIP(hipStreamCreateWithFlags(&mg->side, hipStreamNonBlocking));
    SKT_HIP(hipStreamCreateWithFlags(&mg->side2, hipStreamNonBlocking));
    SKT_HIP(hipEventCreateWithFlags(&mg->ev_fork, hipEventDisableTiming));
    SKT_HIP(hipEventCreateWithFlags(&mg->ev_gal, hipEventDisableTiming));
    SKT_HIP(hipEventCreateWithFlags(&mg->ev_st, hipEventDisableTiming));
    SKT_HIP(hipEventCreateWithFlags(&mg->ev_join, hipEventDisableTiming));
  }
  SKT_HIP(hipEventRecord(mg->ev_fork, s));
  SKT_HIP(hipStreamWaitEvent(mg->side, mg->ev_fork, 0));
  hipStream_t g = mg->side;
  // Galerkin hierarchy.  The first coarse level takes E_j M_j for its
  // interior elements (M_j and the boundary flags depend on the operator
  // only, so they are built once) and the masked product for the rest.
  const uint8_t* fx0 = op->n_fixed > 0 ? op->fixed : nullptr;
  if (op->mesh == SKT_MESH_TET4) {
    const MGLevel& c = mg->lv[1];
    const int64_t nce = c.nx * c.ny * c.nz;
    if (NC == 3)
      hipLaunchKernelGGL((k_galerkin_tet<3>), dim3((unsigned)nce), dim3(64), 0, g, c.nx, c.ny,
                         c.nz, op->nx, op->ny, op->nz, c.f[0], c.f[1], c.f[2], op->conn, op->g64, op->vol64, op->lam0,
                         op->mu0, op->n_el, E64, fx0, c.Kel);
    else
      hipLaunchKernelGGL((k_galerkin_tet<1>), dim3((unsigned)nce), dim3(64), 0, g, c.nx, c.ny,
                         c.nz, op->nx, op->ny, op->nz, c.f[0], c.f[1], c.f[2], op->conn, op->g64, op->vol64, op->lam0,
                         op->mu0, op->n_el, E64, fx0, c.Kel);
    SKT_LAUNCH_CHECK();
  } else {
    const MGLevel& c = mg->lv[1];
    const int nch = c.f[0] * c.f[1] * c.f[2];
    const int64_t nce = c.nx * c.ny * c.nz;
    if (!mg->Mch) {
      SKT_HIP(hipMalloc(&mg->Mch, sizeof(double) * (size_t)nch * ND * ND));
      if (NC == 3)
        hipLaunchKernelGGL((k_galerkin_children<3>), dim3(nch), dim3(64), 0, g, c.f[0], c.f[1],
                           c.f[2], dK0, mg->Mch);
      else
        hipLaunchKernelGGL((k_galerkin_children<1>), dim3(nch), dim3(64), 0, g, c.f[0], c.f[1],
                           c.f[2], dK0, mg->Mch);
      const bool ragged = c.nx * c.f[0] != op->nx || c.ny * c.f[1] != op->ny ||
                          c.nz * c.f[2] != op->nz;
      if (op->n_fixed > 0 || ragged) {
        SKT_HIP(hipMalloc(&mg->gflag, (size_t)nce));
        if (NC == 3)
          hipLaunchKernelGGL((k_galerkin_flags<3>), dim3(grid_for(nce)), dim3(kBlock), 0, g,
                             c.nx, c.ny, c.nz, op->nx, op->ny, op->nz, c.f[0], c.f[1], c.f[2], fx0,
                             mg->gflag);
        else
          hipLaunchKernelGGL((k_galerkin_flags<1>), dim3(grid_for(nce)), dim3(kBlock), 0, g,
                             c.nx, c.ny, c.nz, op->nx, op->ny, op->nz, c.f[0], c.f[1], c.f[2], fx0,
                             mg->gflag);
      }
      SKT_LAUNCH_CHECK();
    }
    SKT_CHECK(nch <= kMaxChildren, "internal: coarsening factor above 5");
    const unsigned gi = (unsigned)std::min<int64_t>(nce, 8192);
    if (NC == 3)
      hipLaunchKernelGGL((k_galerkin_interior<3>), dim3(gi), dim3(64 * 9), 0, g, c.nx, c.ny, c.nz,
                         op->nx, op->ny, c.f[0], c.f[1], c.f[2], mg->Mch, E64, mg->gflag, c.Kel);
    else
      hipLaunchKernelGGL((k_galerkin_interior<1>), dim3(gi), dim3(64), 0, g, c.nx, c.ny, c.nz,
                         op->nx, op->ny, c.f[0], c.f[1], c.f[2], mg->Mch, E64, mg->gflag, c.Kel);
    if (mg->gflag) {
      if (NC == 3)
        hipLaunchKernelGGL((k_galerkin<3>), dim3((unsigned)nce), dim3(64), 0, g, c.nx, c.ny,
                           c.nz, op->nx, op->ny, op->nz, c.f[0], c.f[1], c.f[2], nullptr, dK0,
                           E64, fx0, mg->gflag, c.Kel);
      else
        hipLaunchKernelGGL((k_galerkin<1>), dim3((unsigned)nce), dim3(64), 0, g, c.nx, c.ny,
                           c.nz, op->nx, op->ny, op->nz, c.f[0], c.f[1], c.f[2], nullptr, dK0,
                           E64, fx0, mg->gflag, c.Kel);
    }
    SKT_LAUNCH_CHECK();
  }
  for (int l = 2; l <= L; ++l) {
    // the stencil levels' products are done: side2 may start
    if (l == L) SKT_HIP(hipEventRecord(mg->ev_gal, g));
    const MGLevel &c = mg->lv[l], &f = mg->lv[l - 1];
    const int64_t nce = c.nx * c.ny * c.nz;
    const double* Kf = f.Kel;
    if (NC == 3)
      hipLaunchKernelGGL((k_galerkin<3>), dim3((unsigned)nce), dim3(64), 0, g, c.nx, c.ny, c.nz,
                         f.nx, f.ny, f.nz, c.f[0], c.f[1], c.f[2], Kf, dK0, E64, nullptr, nullptr, c.Kel);
    else
      hipLaunchKernelGGL((k_galerkin<1>), dim3((unsigned)nce), dim3(64), 0, g, c.nx, c.ny, c.nz,
                         f.nx, f.ny, f.nz, c.f[0], c.f[1], c.f[2], Kf, dK0, E64, nullptr, nullptr, c.Kel);
    SKT_LAUNCH_CHECK();
  }
  if (L < 2) SKT_HIP(hipEventRecord(mg->ev_gal, g));
  // stencils and Jacobi inverses of the intermediate levels (side2)
  SKT_HIP(hipStreamWaitEvent(mg->side2, mg->ev_gal, 0));
  g = mg->side2;
  for (int l = 1; l < L; ++l) {
    const MGLevel& v = mg->lv[l];
    const int64_t tot = st_nodes(v.nx, v.ny, v.nz, v.layout) * 27 * NC * NC;
    if (NC == 3) {
      hipLaunchKernelGGL((k_stencil_asm<T, 3>), dim3(grid_for(tot)), dim3(kBlock), 0, g, v.nx,
                         v.ny, v.nz, v.layout, v.Kel, (T*)v.st);
      hipLaunchKernelGGL((k_stencil_dinv<T, 3>), dim3(grid_for(v.ndof)), dim3(kBlock), 0, g,
                         v.nx, v.ny, v.nz, v.layout, (const T*)v.st, (T*)v.dinv);
    } else {
      hipLaunchKernelGGL((k_stencil_asm<T, 1>), dim3(grid_for(tot)), dim3(kBlock), 0, g, v.nx,
                         v.ny, v.nz, v.layout, v.Kel, (T*)v.st);
      hipLaunchKernelGGL((k_stencil_dinv<T, 1>), dim3(grid_for(v.ndof)), dim3(kBlock), 0, g,
                         v.nx, v.ny, v.nz, v.layout, (const T*)v.st, (T*)v.dinv);
    }
    SKT_LAUNCH_CHECK();
  }
  SKT_HIP(hipEventRecord(mg->ev_st, g));
  g = mg->side;
  // coarsest: dense matrix, blocked Gauss-Jordan inverse, cast to T (side
  // stream).  Enqueued after the fine level's power iteration, so that the
  // host's many small launches for it do not hold back the main stream.
  // With a lagged inverse (mg_lagged) only the matrix is assembled here;
  // mg_lag_post inverts it in the background after the set-up.
  const bool lagged = mg_lagged(mg);
  const bool reuse = mg->reuse_inv && mg->have_inv && !lagged;
  bool coarsest_queued = false;
  auto queue_coarsest = [&]() -> int {
    coarsest_queued = true;
    const MGLevel& c = mg->lv[L];
    const int64_t n = c.ndof;
    if (reuse) {  // the previous inverse stays in Ainv
      SKT_HIP(hipEventRecord(mg->ev_join, g));
      return SKT_OK;
    }
    const int64_t np = gj_pad(n);
    if (NC == 3)
      hipLaunchKernelGGL((k_dense_asm<3>), dim3(grid_for(np * np)), dim3(kBlock), 0, g, c.nx,
                         c.ny, c.nz, c.Kel, np, 1.0 + mg->shift, mg->Ad);
    else
      hipLaunchKernelGGL((k_dense_asm<1>), dim3(grid_for(np * np)), dim3(kBlock), 0, g, c.nx,
                         c.ny, c.nz, c.Kel, np, 1.0 + mg->shift, mg->Ad);
    if (!lagged) {
      queue_gj(mg, g);
      queue_cast<T>(mg, g);
    }
    SKT_LAUNCH_CHECK();
    SKT_HIP(hipEventRecord(mg->ev_join, g));
    return SKT_OK;
  };
  // smoother bounds: power iteration on D^-1 A (one column) per level
  double* inv = mg->lam + (L + 1);  // scratch scalar slot
  int64_t off = 0;
  bool st_joined = false;
  for (int l = 0; l < L; ++l) {
    if (l == 1) {
      if (int stt = queue_coarsest()) return stt;
      SKT_HIP(hipStreamWaitEvent(s, mg->ev_st, 0));
      st_joined = true;
    }
    const MGLevel& v = mg->lv[l];
    const int64_t n = v.ndof;
    T* pv0 = (T*)mg->pvw + off;      // this level's vector, kept for the next set-up
    T* pv1 = (T*)mg->pv;
    off += n;
    const T* dinv = l == 0 ? (const T*)dinv0 : (const T*)v.dinv;
    const unsigned nb = std::min<unsigned>(grid_for(n), 1024u);
    if (!mg->warm)
      hipLaunchKernelGGL(k_pow_init<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, dinv, pv0);
    // The iterate is left unnormalised between steps (it grows by about
    // lambda per step, far from the float range over these few steps); the
    // last step's input and output norms give lambda, and the normalised
    // result is kept for the next set-up.
    const int steps = mg->warm ? warm_power_steps(mg) : mg->power_iters;
    for (int it = 0; it < steps; ++it) {
      const bool last = it + 1 == steps;
      if (last) {
        hipLaunchKernelGGL(k_pow_norm<T>, dim3(nb), dim3(kBlock), 0, s, n, dinv, pv0, 0,
                           mg->part);
        hipLaunchKernelGGL(k_pow_finish, dim3(1), dim3(kBlock), 0, s, (int)nb, mg->part,
                           (double*)nullptr, (const double*)nullptr, inv);
      }
      int stt = level_apply<T>(mg, op, E, l, 1, 1, pv0, pv1, s);
      if (stt) return stt;
      if (!last) {
        hipLaunchKernelGGL(k_pow_dscale<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, dinv, pv1,
                           pv0);
        continue;
      }
      hipLaunchKernelGGL(k_pow_norm<T>, dim3(nb), dim3(kBlock), 0, s, n, dinv, pv1, 1, mg->part);
      hipLaunchKernelGGL(k_pow_finish, dim3(1), dim3(kBlock), 0, s, (int)nb, mg->part,
                         mg->lam + l, (const double*)inv, inv);
      hipLaunchKernelGGL(k_pow_scale<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, inv, pv1,
                         pv0);
    }
    SKT_LAUNCH_CHECK();
  }
  if (!coarsest_queued) {
    if (int stt = queue_coarsest()) return stt;
  }
  mg->warm = 1;
  hipLaunchKernelGGL(k_cheb_coef, dim3(1), dim3(64), 0, s, L, coef_steps(mg), mg->ratio,
                     mg->low_steps ? std::max(mg->ratio, kLowRatio) : mg->ratio, mg->margin, mg->lam,
                     mg->coef);
  SKT_LAUNCH_CHECK();
  // every side-stream branch joins the main stream before the set-up
  // returns (a graph capture of the set-up requires it)
  if (!st_joined) SKT_HIP(hipStreamWaitEvent(s, mg->ev_st, 0));
  SKT_HIP(hipStreamWaitEvent(s, mg->ev_join, 0));
  if (!lagged) mg->have_inv = 1;
  return SKT_OK;
}

int mg_setup(MGData* mg, const skt_operator* op, const double* E64, const void* E,
             const void* dinv0, hipStream_t s) {
  SKT_CHECK(mg->dtype >= 0 && !mg->lv.empty(), "multigrid not allocated");
  if (mg->dtype == SKT_F64) return setup_t<double>(mg, op, E64, E, dinv0, s);
  return setup_t<float>(mg, op, E64, E, dinv0, s);
}

// SKT_MG_TRANSFERS=rowgrid forces the row-grid restriction on every level,
// =tiled the kernels of large levels (row grid, and k_restrict222 where all
// factors are 2).  All give the same sums; tests check that the solves agree
// bit for bit.
enum Transfers { kGathers, kTiled, kRowGrid };
static Transfers transfers() {
  const char* v = std::getenv("SKT_MG_TRANSFERS");
  return !v ? kGathers : !std::strcmp(v, "rowgrid") ? kRowGrid : !std::strcmp(v, "tiled") ? kTiled : kGathers;
}

// Largest coarse level (nodes times column groups) that k_restrict_gather
// takes.  Limits of 32768 and 262144 change the time of a design iteration or
// solve by less than 1% (40x20x20 to 120x60x60); kernel times near the limit,
// gather against tiles: 3 components, 2 columns, 125,000 nodes: 12.8 and 14.2 us
// in float32, 20.4 and 26.5 in float64; scalar, 69,000 nodes: 1 float32 column
// 5.0 and 6.0 us (36,000 nodes), 4 columns 6.8 and 8.3.
constexpr int64_t kGatherNodes = 131072;

// Four float64 columns are 32 bytes a load: with w a thread's 27 nodes no longer
// fit in registers (17,000 scalar nodes: 12.6 us, tiles 9.2; 800 nodes: 10.4 and
// 7.6), and without it they do better on small levels only (36,000 nodes: 8.0
// and 10.7 us; 69,000: 12.2 and 11.8).
template <typename T, int KC>
static bool gather_fits(int64_t nodes, bool has_w) {
  constexpr int bytes = (int)sizeof(T) * KC;
  return bytes <= 16 ? nodes <= kGatherNodes : !has_w && nodes <= kGatherNodes / 2;
}

template <typename T, int NC, int KC>
static void launch_restrict(const MGLevel& f, const MGLevel& c, int groups, const T* b,
                            const T* w, const uint8_t* fixed, T* bc, hipStream_t s) {
  T* tbuf = (T*)c.rt;
  const int64_t rows = (c.nx + 1) * (c.ny + 1) * (f.nz + 1) * groups;
  // 25 loads a thread pay while they wait for latency, not for bandwidth (the
  // limit of the gather for factor 2, whose threads load as much), and where
  // most of them are used: 28x28x82 scalar rows by factor 3, 7.0 us against
  // 12.8, 12x7x14 with 6 float64 values 8.8 and 14.9.  With factors of 2 and 1,
  // on plates, the fine level with its Dirichlet flags is faster by rows (400 x
  // 320 elements: 10.3 us against 8.0; 300 x 280 coarsened in x only: 10.8 and
  // 4.8), a level coarsened by 2 in x and y without flags slightly slower
  // (50 x 40 coarse elements: 4.7 and 5.4).
  const bool three = c.f[0] == 3 || c.f[1] == 3;
  const bool used = c.f[0] <= 3 && c.f[1] <= 3 &&
                    (three || (c.f[0] == 2 && c.f[1] == 2 && !fixed));
  if (used && gather_fits<T, KC>(rows, w != nullptr) && transfers() == kGathers) {
    const unsigned gg = (unsigned)((rows * NC + 255) / 256);
    if (w)
      hipLaunchKernelGGL((k_restrict_xy_gather<T, NC, KC, true>), dim3(gg), dim3(256), 0, s,
                         (int)f.nx, (int)f.ny, (int)f.nz, c.f[0], c.f[1], groups, b, w, fixed, tbuf);
    else
      hipLaunchKernelGGL((k_restrict_xy_gather<T, NC, KC, false>), dim3(gg), dim3(256), 0, s,
                         (int)f.nx, (int)f.ny, (int)f.nz, c.f[0], c.f[1], groups, b, w, fixed, tbuf);
  } else {
    const RowGrid gxy = row_grid(c.nx + 1, (c.ny + 1) * (f.nz + 1) * groups);
    hipLaunchKernelGGL((k_restrict_xy<T, NC, KC>), gxy.grid, gxy.block, 0, s, (int)f.nx, (int)f.ny,
                       (int)f.nz, c.f[0], c.f[1], groups, b, w, fixed, tbuf);
  }
  const RowGrid gz = row_grid((c.nx + 1) * (c.ny + 1), (c.nz + 1) * groups);
  hipLaunchKernelGGL((k_restrict_z<T, NC, KC>), gz.grid, gz.block, 0, s, (int)(c.nx + 1),
                     (int)(c.ny + 1), (int)f.nz, c.f[2], groups, (const T*)tbuf, bc);
}

// Fused restriction into level c when every factor is 2 (k_restrict222; b
// zero at Dirichlet DOFs); with x0, also the first smoothing iterate of c
// (coefficients cf).  Returns false, launching nothing, otherwise.
template <typename T, int NC, int KC>
static bool launch_restrict_fused(const MGLevel& f, const MGLevel& c, int groups, const T* b,
                                  const T* w, T* bc, const double* cf, T* x0, hipStream_t s) {
  const Transfers how = transfers();
  if (c.f[0] != 2 || c.f[1] != 2 || c.f[2] != 2 || how == kRowGrid) return false;
  const int tiles_x = (int)((c.nx + 1 + kR2I - 1) / kR2I);
  const int tiles_y = (int)((c.ny + 1 + kR2J - 1) / kR2J);
  const int cnnz = (int)(c.nz + 1);
  // planes per chunk: halved until there are >= 1024 workgroups (each chunk
  // streams its 2 zlen + 1 fine planes one after the other)
  int zlen = 4;
  const int64_t per = (int64_t)tiles_x * tiles_y * groups;
  while (zlen > 1 && per * ((cnnz + zlen - 1) / zlen) < 1024) zlen /= 2;
  const int zch = (cnnz + zlen - 1) / zlen;
  const int64_t nblk = per * zch;
  const T* dc = x0 ? (const T*)c.dinv : nullptr;
  if (how == kGathers && gather_fits<T, KC>(c.nn * groups, w != nullptr)) {
    const unsigned gg = (unsigned)((c.nn * NC * groups + 255) / 256);
    if (w)
      hipLaunchKernelGGL((k_restrict_gather<T, NC, KC, true>), dim3(gg), dim3(256), 0, s,
                         (int)f.nx, (int)f.ny, (int)f.nz, groups, b, w, bc, dc, cf, x0);
    else
      hipLaunchKernelGGL((k_restrict_gather<T, NC, KC, false>), dim3(gg), dim3(256), 0, s,
                         (int)f.nx, (int)f.ny, (int)f.nz, groups, b, w, bc, dc, cf, x0);
    return true;
  }
  if (w)
    hipLaunchKernelGGL((k_restrict222<T, NC, KC, true>), dim3((unsigned)nblk), dim3(256), 0, s,
                       (int)f.nx, (int)f.ny, (int)f.nz, tiles_x, tiles_y, zch, zlen, b, w, bc,
                       dc, cf, x0);
  else
    hipLaunchKernelGGL((k_restrict222<T, NC, KC, false>), dim3((unsigned)nblk), dim3(256), 0, s,
                       (int)f.nx, (int)f.ny, (int)f.nz, tiles_x, tiles_y, zch, zlen, b, w, bc,
                       dc, cf, x0);
  return true;
}

template <typename T, int NC, int KC>
static void launch_prolong(const MGLevel& f, const MGLevel& c, int groups, const T* xc,
                           const uint8_t* fixed, T* xf, hipStream_t s) {
  const RowGrid gp = row_grid(f.nx + 1, (f.ny + 1) * (f.nz + 1) * groups);
  if (fixed)
    hipLaunchKernelGGL((k_prolong_add<T, NC, KC, true>), gp.grid, gp.block, 0, s, (int)f.nx,
                       (int)f.ny, (int)f.nz, c.f[0], c.f[1], c.f[2], groups, xc, fixed, xf);
  else
    hipLaunchKernelGGL((k_prolong_add<T, NC, KC, false>), gp.grid, gp.block, 0, s, (int)f.nx,
                       (int)f.ny, (int)f.nz, c.f[0], c.f[1], c.f[2], groups, xc, fixed, xf);
}

template <typename T>
static const T* modal_coef(const skt_operator* op);
template <>
const double* modal_coef<double>(const skt_operator* op) { return op->modal_d; }
template <>
const float* modal_coef<float>(const skt_operator* op) { return op->modal_f; }

// V-cycle.  On the fine level the Chebyshev steps and the residual are fused
// into the matrix-free apply (hex_cheb_modal / hex_resid_modal); the
// iterate ping-pongs between z and lv[0].x, and the Chebyshev direction is
// the difference of the two buffers, so no direction vector is kept.  The
// number of fused steps, 2 * degree - 1, is odd: starting in lv[0].x the
// cycle ends in z.
// Smoothing steps of level l
static int level_steps(const MGData* mg, int l) {
  return mg->degree + (l > 0 && l + 2 == (int)mg->lv.size() ? mg->low_steps : 0);
}

template <typename T, int NC, int KC>
static int vcycle_t(MGData* mg, const skt_operator* op, const void* E, const void* dinv0, int k,
                    const T* r, T* z, T* w0, hipStream_t s, double* dot, int max_slots,
                    int* slots, const double* stop) {
  StOut<T> ost;
  ost.stop = stop;
  const int L = (int)mg->lv.size() - 1;
  const int groups = k / KC;
  const int deg = mg->degree, cs = coef_steps(mg);
  const uint8_t* fixed0 = op->n_fixed > 0 ? op->fixed : nullptr;
  const T* coef0 = modal_coef<T>(op);
  const T* E0 = (const T*)E;
  int stt;
  if (L >= 32) {
    set_error("internal: too many multigrid levels");
    return SKT_EINVAL;
  }
  // levels whose first smoothing iterate the restriction into them formed
  bool x0_done[32] = {};
  T* cur = (T*)mg->lv[0].x;  // fine iterate (ping-pong with z)
  T* oth = z;
  // Operators without the fused modal kernels (tet4 on a grid): the fine
  // level's Chebyshev steps as operator applies plus vector updates, with
  // the direction kept in z; the iterate lives in lv[0].x and is copied to z
  // at the end.
  const bool generic = !(op->mesh == SKT_MESH_HEX8 && op->modal_ok);
  if (generic) {
    MGLevel& v = mg->lv[0];
    const int64_t total = v.ndof * k;
    const unsigned ge = grid_for(total);
    const double* cf = mg->coef;
    T* x = (T*)v.x;
    T* d = z;
    for (int st = 0; st < deg; ++st) {
      T* w = st == 0 ? nullptr : w0;
      if (st > 0 && (stt = op_apply(const_cast<skt_operator*>(op), mg->dtype, k, KC, E, x, w0,
                                    s)))
        return stt;
      hipLaunchKernelGGL(k_cheb<T>, dim3(ge), dim3(kBlock), 0, s, total, v.ndof, KC,
                         cf + 2 * st, r, (const T*)w, (const T*)dinv0, d, x, st == 0 ? 1 : 0);
    }
    if ((stt = op_apply(const_cast<skt_operator*>(op), mg->dtype, k, KC, E, x, w0, s)))
      return stt;
    // zero at Dirichlet DOFs, as the fused restriction needs
    hipLaunchKernelGGL(k_rsub<T>, dim3(ge), dim3(kBlock), 0, s, total, v.ndof, KC, fixed0, r, w0);
    T* x01 = L > 1 ? (T*)mg->lv[1].x : nullptr;
    if (launch_restrict_fused<T, NC, KC>(v, mg->lv[1], groups, (const T*)w0, (const T*)nullptr,
                                         (T*)mg->lv[1].b, mg->coef + (size_t)2 * cs, x01, s))
      x0_done[1] = x01 != nullptr;
    else
      launch_restrict<T, NC, KC>(v, mg->lv[1], groups, (const T*)w0, (const T*)nullptr, fixed0,
                                 (T*)mg->lv[1].b, s);
    SKT_LAUNCH_CHECK();
    cur = x;
  } else {
    MGLevel& v = mg->lv[0];
    const int64_t total = v.ndof * k;
    const double* cf = mg->coef;
    if (deg == 2 && cheb0_enabled()) {
      // steps 0 and 1 in one pass (step 0's iterate is formed on the fly
      // and never stored, so this form serves degree 2 only: a third step
      // would need it as its previous iterate)
      const int ti = fine_timer_begin(mg, MG_T_CHEB0, s);
      if ((stt = hex_cheb0_modal<T>(op, k, KC, coef0, E0, r, oth, (const T*)dinv0, cf, cf + 2,
                                    s, stop)))
        return stt;
      fine_timer_end(mg, ti, s);
      std::swap(cur, oth);
    } else {
      hipLaunchKernelGGL(k_cheb_first<T>, dim3(grid_for(total)), dim3(kBlock), 0, s, total,
                         v.ndof, KC, cf, r, (const T*)dinv0, cur);
      // step st reads its previous iterate from the buffer it overwrites:
      // zero for step 1, the iterate of step st - 2 after that
      for (int st = 1; st < deg; ++st) {
        const int ti = fine_timer_begin(mg, MG_T_CHEB, s);
        if ((stt = hex_cheb_modal<T>(op, k, KC, coef0, E0, cur, oth, r, (const T*)dinv0,
                                     cf + 2 * st, st == 1 ? 1 : 0, s, nullptr, stop)))
          return stt;
        fine_timer_end(mg, ti, s);
        std::swap(cur, oth);
      }
    }
    const int tr = fine_timer_begin(mg, MG_T_RESID, s);
    if ((stt = hex_resid_modal<T>(op, k, KC, coef0, E0, cur, r, w0, s, stop))) return stt;
    fine_timer_end(mg, tr, s);
    // the residual is zero at Dirichlet DOFs, as the fused restriction needs;
    // it also forms level 1's first smoothing iterate unless level 1 is the
    // coarsest
    T* x01 = L > 1 ? (T*)mg->lv[1].x : nullptr;
    if (launch_restrict_fused<T, NC, KC>(v, mg->lv[1], groups, (const T*)w0, (const T*)nullptr,
                                         (T*)mg->lv[1].b, mg->coef + (size_t)2 * cs, x01, s))
      x0_done[1] = x01 != nullptr;
    else
      launch_restrict<T, NC, KC>(v, mg->lv[1], groups, (const T*)w0, (const T*)nullptr, fixed0,
                                 (T*)mg->lv[1].b, s);
    SKT_LAUNCH_CHECK();
  }
  // coarse levels: each level's iterate ping-pongs between its x and d
  // buffers through fused Chebyshev steps; it[l] holds the current one
  T* it[32];
  for (int l = 1; l < L; ++l) {
    MGLevel& v = mg->lv[l];
    const T* b = (const T*)v.b;
    T* A = (T*)v.x;
    T* B = (T*)v.d;
    T* w = (T*)v.w;
    const int64_t total = v.ndof * k;
    const double* cf = mg->coef + (size_t)l * 2 * cs;
    // step 0 from a zero iterate (formed by the fused restriction into this
    // level, or here), then fused steps (the iterate before step 0 is zero)
    if (!x0_done[l])
      hipLaunchKernelGGL(k_cheb_first<T>, dim3(grid_for(total)), dim3(kBlock), 0, s, total,
                         v.ndof, KC, cf, b, (const T*)v.dinv, A);
    for (int st = 1; st < level_steps(mg, l); ++st) {
      if ((stt = level_cheb<T>(mg, op, l, k, KC, A, B, cf + 2 * st, st == 1 ? 1 : 0, s, stop)))
        return stt;
      std::swap(A, B);
    }
    it[l] = A;
    if ((stt = level_apply<T>(mg, op, E, l, k, KC, A, w, s, ost))) return stt;
    T* x0n = l + 1 < L ? (T*)mg->lv[l + 1].x : nullptr;
    if (launch_restrict_fused<T, NC, KC>(v, mg->lv[l + 1], groups, b, w, (T*)mg->lv[l + 1].b,
                                         mg->coef + (size_t)(l + 1) * 2 * cs, x0n, s))
      x0_done[l + 1] = x0n != nullptr;
    else
      launch_restrict<T, NC, KC>(v, mg->lv[l + 1], groups, b, w, nullptr, (T*)mg->lv[l + 1].b,
                                 s);
    SKT_LAUNCH_CHECK();
  }
  // coarsest
  {
    const MGLevel& c = mg->lv[L];
    launch_dense_apply<T, KC>(c.ndof, groups, (const T*)mg->Ainv, (const T*)c.b, (T*)c.x, s);
    SKT_LAUNCH_CHECK();
    it[L] = (T*)c.x;
  }
  // coarse levels, upward
  for (int l = L - 1; l >= 1; --l) {
    MGLevel& v = mg->lv[l];
    T* A = it[l];
    T* B = (A == (T*)v.x) ? (T*)v.d : (T*)v.x;
    const double* cf = mg->coef + (size_t)l * 2 * cs;
    launch_prolong<T, NC, KC>(v, mg->lv[l + 1], groups, (const T*)it[l + 1], nullptr, A, s);
    for (int st = 0; st < level_steps(mg, l); ++st) {
      // step 0 has c1 = 0 and needs no previous iterate
      if ((stt = level_cheb<T>(mg, op, l, k, KC, A, B, cf + 2 * st, st == 0 ? 1 : 0, s, stop)))
        return stt;
      std::swap(A, B);
    }
    it[l] = A;
    SKT_LAUNCH_CHECK();
  }
  if (generic) {
    MGLevel& v = mg->lv[0];
    const int64_t total = v.ndof * k;
    const unsigned ge = grid_for(total);
    const double* cf = mg->coef;
    T* x = (T*)v.x;
    launch_prolong<T, NC, KC>(v, mg->lv[1], groups, (const T*)it[1], fixed0, x, s);
    // post-smoothing from the corrected iterate (step 0 has c1 = 0, so the
    // stale direction in z is not used)
    for (int st = 0; st < deg; ++st) {
      if ((stt = op_apply(const_cast<skt_operator*>(op), mg->dtype, k, KC, E, x, w0, s)))
        return stt;
      hipLaunchKernelGGL(k_cheb<T>, dim3(ge), dim3(kBlock), 0, s, total, v.ndof, KC,
                         cf + 2 * st, r, (const T*)w0, (const T*)dinv0, z, x, 0);
    }
    hipLaunchKernelGGL(k_copy_vec<T>, dim3(ge), dim3(kBlock), 0, s, total, (const T*)x, z);
    if (slots) *slots = 0;
    SKT_LAUNCH_CHECK();
    return SKT_OK;
  }
  // fine level, correction and post-smoothing
  {
    MGLevel& v = mg->lv[0];
    const double* cf = mg->coef;
    launch_prolong<T, NC, KC>(v, mg->lv[1], groups, (const T*)it[1], fixed0, cur, s);
    // the last step can leave the partials of r . z
    const int ns = hex_modal_dot_slots(op, k, KC);
    double* last_dot = (dot && slots && ns <= max_slots) ? dot : nullptr;
    for (int st = 0; st < deg; ++st) {
      // step 0 has c1 = 0 and needs no previous iterate
      double* sd = st == deg - 1 ? last_dot : nullptr;
      const int ti = fine_timer_begin(mg, sd ? MG_T_CHEB_DOT : MG_T_CHEB, s);
      if ((stt = hex_cheb_modal<T>(op, k, KC, coef0, E0, cur, oth, r, (const T*)dinv0,
                                   cf + 2 * st, 0, s, sd, stop)))
        return stt;
      fine_timer_end(mg, ti, s);
      std::swap(cur, oth);
    }
    if (slots) *slots = (last_dot && deg >= 1) ? ns : 0;
    SKT_LAUNCH_CHECK();
  }
  if (cur != z) {
    set_error("internal: multigrid iterate did not end in z");
    return SKT_EINVAL;
  }
  return SKT_OK;
}

int mg_vcycle(MGData* mg, const skt_operator* op, const void* E, const void* dinv0, int ncols,
              int kc, const void* r, void* z, void* w0, hipStream_t s, double* dot,
              int max_slots, int* slots, const double* stop) {
  SKT_CHECK(mg->dtype >= 0, "multigrid not set up");
  SKT_CHECK(ncols <= mg->max_cols && ncols % kc == 0, "bad column count for multigrid");
#define SKT_VC(T_, NC_, KC_)                                                               \
  return vcycle_t<T_, NC_, KC_>(mg, op, E, dinv0, ncols, (const T_*)r, (T_*)z, (T_*)w0, s, dot, \
                                max_slots, slots, stop)
  if (mg->dtype == SKT_F64) {
    if (op->ncomp == 3) {
      if (kc == 1) SKT_VC(double, 3, 1);
      if (kc == 2) SKT_VC(double, 3, 2);
    } else {
      if (kc == 1) SKT_VC(double, 1, 1);
      if (kc == 2) SKT_VC(double, 1, 2);
      if (kc == 4) SKT_VC(double, 1, 4);
    }
  } else {
    if (op->ncomp == 3) {
      if (kc == 1) SKT_VC(float, 3, 1);
      if (kc == 2) SKT_VC(float, 3, 2);
    } else {
      if (kc == 1) SKT_VC(float, 1, 1);
      if (kc == 2) SKT_VC(float, 1, 2);
      if (kc == 4) SKT_VC(float, 1, 4);
    }
  }
#undef SKT_VC
  set_error("unsupported column block for multigrid");
  return SKT_EINVAL;
}

}  // namespace skt
