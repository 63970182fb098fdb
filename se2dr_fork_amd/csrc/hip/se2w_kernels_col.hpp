// se2w_kernels_col.hpp -- column kernel: one lane per element column.
//
// The p + 1 lanes of an element each hold one column of its nodes and the
// quadrature points of that column (lane i: the points (i, qj) and the nodes
// (i, j)).  A wave holds 64 / (p + 1) neighbouring elements of one element
// row, a workgroup WX waves in x times EY element rows.  Sums along a column
// (d/dy of the displacement, the column terms of the forces) run in the lane's
// registers against a derivative table that is the same for the whole wave,
// in SGPRs; sums along a row read the element's other columns from LDS, where
// every lane of an element reads the same address.  An element's rows are
// exchanged three times inside its wave (displacement, row stresses, nodal
// forces, all in one buffer, without a barrier); one barrier lets the
// neighbours' edge forces through.
//
// What it is for: from p = 5 up a lane or lane pair per element (the register
// kernels) holds 2 (p+1)^2 values per component, which takes a SIMD's whole
// register file in FP64 (one wave, scratch traffic from p = 7 on), and small
// meshes give such a kernel too few waves.  Here a lane holds a few times
// p + 1 values (two to four waves per SIMD in FP64, four in FP32), and a mesh
// gives (p+1)/2 times the waves.  It is bound by VALU issue and by the latency of
// its phases.  us per step, fastest register or LDS kernel -> this one: FP64
// 24^2 p4 15.0 -> 9.2, 256^2 p4 26.1 -> 22.6, 800^2 p4 189 -> 211, 389^2 p5
// 93 -> 69, 64^2 p6 21.9 -> 12.0, 330^2 p6 152 -> 86, 300^2 p7 297 -> 97,
// 256^2 p8 239 -> 104; FP32 512^2 p4 32.0 -> 33.5, 320^2 p5 28.3 -> 23.6,
// 200^2 p6 24.0 -> 18.3, 500^2 p6 74 -> 74, 300^2 p7 51 -> 36, 512^2 p8 199 ->
// 167; FP32+Kahan 512^2 p8 260 -> 230.
//
// Every sum runs over the same terms in the same order, with the same
// roundings, as in reg64_body / reg_body, so the results have the same bits
// (FP64: those of the reference's loop).  In FP64 the diagonal term of a row
// sum (the node or point of the lane's own column) is added by a multiply-add
// with a factor 1 or 0, one instruction of the three of a term.  The factor 0
// makes a NaN of an infinite term, and a NaN of every force that this touches:
// a wave that finds a NaN among its forces forms them again without the factor
// (col_force_f64).  Adding the term through a select instead is exact too and
// takes 2 to 9 % longer (us per step, this form and the select: 300^2 p3 18.3,
// 19.0, 220^2 p6 39.8, 41.3, 64^2 p7 15.0, 16.4, 256^2 p8 95, 99); under an
// execution mask of the lane's column it takes 0 to 10 % longer.
//
// Tiling: as in the register kernels, a workgroup owns its elements except
// the left column and the bottom row, which only supply their edge forces;
// the waves of the bottom row form the top edge alone.  The owner lane of a
// node updates it: lanes run along the node rows, so the loads and stores are
// contiguous except for the column that neighbouring elements share.
#pragma once
#include "se2w_kernels.hpp"

namespace se2w {

// Schedules: waves in x, element rows.  Four rows (of which three are owned)
// leave the most workgroups per CU and are the fastest in FP64 at every degree
// and size (7 % ahead of eight rows at 256 x 256 p8, level at 330 x 330 p6);
// FP32 needs half the registers and LDS, and eight rows, seven of them owned,
// are ahead by up to 5 % on some large meshes (512 x 512 p8: 166 against 172).  Two waves in x and six rows measured
// slower than either (64 x 64 p6 FP64: 12.0, 15.8, 13.9 and 15.1 us for 1 x 4,
// 1 x 8, 2 x 4 and 1 x 6).
struct ColSchedule { int wx, ey; };
constexpr ColSchedule kColSchedules[] = {{1, 4}, {1, 8}};
constexpr int kNumColSchedules = sizeof(kColSchedules) / sizeof(kColSchedules[0]);
constexpr int col_epw(int p) { return 64 / (p + 1); }  // elements per wave
constexpr bool col_schedule_built(int P, int mode, int S, bool fused) {
  return fused && P >= 2 && P <= kMaxP && S >= 0 && S < (mode == MODE_F64 ? 1 : kNumColSchedules);
}

// Orders the LDS accesses of one wave: its LDS instructions execute in order,
// so only the compiler has to keep them in order.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The same uniform pointer, opaque to the compiler: a table read through it is
// loaded where it is used.  Hoisted out of the row loops the tables take more
// SGPRs than there are, and every use of a spilled one costs a VALU move.
template <typename T>
__device__ __forceinline__ T *here(T *p) {
  asm volatile("" : "+s"(p));
  return p;
}

// The value that lane t (uniform) holds.
__device__ __forceinline__ int lane_value(int v, int t) { return __builtin_amdgcn_readlane(v, t); }
__device__ __forceinline__ float lane_value(float v, int t) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), t));
}
__device__ __forceinline__ double lane_value(double v, int t) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, t);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), t);
  return __longlong_as_double((long long)hi << 32 | lo);
}

// FP64 force of the node (i, j) from the displacement of its element, which B
// holds: the terms, their order and their roundings as in col_body, each
// stress formed where it is used.  Only for waves with a NaN among their
// forces, so small and slow: rolled loops, in which no lane uses another's
// stresses.  A second copy of the unrolled operator makes the first one spill.
template <int P>
__device__ double2 col_force_f64(const double2 *B, const double *D, const double *w2, const double *dny, double iJ00,
                                 double detJ, double lam, double mu, int i, int j) {
#pragma clang fp contract(off)
  constexpr int NB = P + 1;
  const double c11 = 2.0 * mu + lam;
  struct Stress { double xx, xy, yy; };
  auto stress = [&](int k, int q) {  // at the point (k, q)
    double e0 = 0.0, e1 = 0.0, e2 = 0.0;
#pragma unroll 1
    for (int l = 0; l < NB; l++) {
      const double dy = dny[q * NB + l];
      const double2 ul = B[l * NB + k];
      e1 = e1 + dy * ul.y;
      if (l != q) {
        e2 = e2 + dy * ul.x;
        continue;
      }
#pragma unroll 1
      for (int m = 0; m < NB; m++) {
        const double dx = iJ00 * D[k * NB + m];
        const double2 um = B[q * NB + m];
        e0 = e0 + dx * um.x;
        e2 = e2 + (m == k ? dy * ul.x + dx * um.y : dx * um.y);
      }
    }
    return Stress{c11 * e0 + lam * e1, mu * e2, lam * e0 + c11 * e1};
  };
  double2 f = double2{0.0, 0.0};
#pragma unroll 1
  for (int q = 0; q < NB; q++) {
    const Stress s = stress(i, q);
    const double dy = dny[q * NB + j];
    if (q != j) {
      const double nfac = -(detJ * w2[i * NB + q]);
      f.x = f.x + nfac * (dy * s.xy);
      f.y = f.y + nfac * (dy * s.yy);
      continue;
    }
#pragma unroll 1
    for (int k = 0; k < NB; k++) {
      const Stress t = stress(k, j);
      const double nfac = -(detJ * w2[j * NB + k]), dx = iJ00 * D[k * NB + i];
      const double x = dx * t.xx, y = dx * t.xy;
      f.x = f.x + nfac * (k == i ? dy * s.xy + x : x);
      f.y = f.y + nfac * (k == i ? dy * s.yy + y : y);
    }
  }
  return f;
}

template <int P, int MODE, int WX, int EY, typename PRM>
__device__ __forceinline__ void col_body(PRM &prm, int tile, int step, int last) {
#pragma clang fp contract(off)
  using R = typename RealOf<MODE>::T;
  using R2 = typename V2<R>::T;
  using CR = const __attribute__((address_space(4))) R;
  constexpr int NB = P + 1, EPW = col_epw(P), EX = EPW * WX;
  constexpr int TEX = EX - 1, TEY = EY - 1;
  // An odd number of nodes per element: the elements of a wave read rows at
  // this stride, which then falls on different banks.
  constexpr int ES = (NB * NB) | 1;
  __shared__ R2 buf[EY][EX][ES];

  const int tx = tile % prm.tiles_x, ty = tile / prm.tiles_x;
  const int ex0 = tx * TEX, ey0 = ty * TEY;
  const int ex_end = min(ex0 + TEX, prm.mx), ey_end = min(ey0 + TEY, prm.my);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  // Lanes past the wave's last whole element repeat the last lane and store
  // nothing to memory.
  const int el = min(lane / NB, EPW - 1), i = min(lane - el * NB, P);
  const int ly = wave / WX, lx = (wave % WX) * EPW + el;
  const int ey = ey0 - 1 + ly, ex = ex0 - 1 + lx;
  const bool row_valid = ey >= 0 && ey < ey_end;  // uniform per wave
  const bool owner = row_valid && ly >= 1 && lx >= 1 && ex < ex_end && lane < EPW * NB;
  R2 *B = &buf[ly][lx][0];  // [j][i]

  // The update's loads.  Nodes that the lane does not own load an owned node
  // instead (in bounds, unused), so they carry no branch.  Where the registers
  // allow they go out between the two halves of the element operator, in place
  // of the displacement column, and the forces cover their latency (EARLY);
  // else before the barrier.
  constexpr bool EARLY = MODE != MODE_F64;
  const bool rb = ex == prm.mx - 1, tb = ey == prm.my - 1;  // domain right / top boundary
  const bool mine = owner && (i < P || rb);
  const int gx = mine ? ex * P + i : ex0 * P;
  const int gy0 = mine ? ey * P : ey0 * P;
  const long idx0 = (long)gy0 * prm.pitch + gx;
  R2 pu[NB], pv[NB], pc[NB];
  R pm[NB];
  auto node_loads = [&]() {
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const long idx = idx0 + (long)(j < P || (mine && tb) ? j : 0) * prm.pitch;
      pu[j] = prm.u_in[idx];
      pv[j] = prm.v[idx];
      pm[j] = prm.mass[idx];
      if constexpr (MODE == MODE_F32K) pc[j] = prm.c_in[idx];
      else pc[j] = R2{R(0), R(0)};
    }
  };

  R2 F[NB];  // forces of the nodes (i, j)
  if (row_valid) {
    // columns of elements outside the mesh repeat its first or last column of
    // elements; nobody uses their forces
    const int exc = min(max(ex, 0), prm.mx - 1);
    const long base = (long)(ey * P) * prm.pitch + exc * P + i;
    R2 u[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) u[j] = prm.u_in[base + (long)j * prm.pitch];
    const int e = exc + ey * prm.mx;
    const R J00 = R(0.5) * prm.elem_dx[exc], J11 = R(0.5) * prm.elem_dy[ey];
    const R iJ00 = R(1) / J00, iJ11 = R(1) / J11, detJ = J00 * J11;
    const R lam = prm.lambda[e], mu = prm.mu[e], c11 = R(2) * mu + lam;
    CR *D = (CR *)(uintptr_t)prm.D;
    CR *W = (CR *)(uintptr_t)prm.w2;
#pragma unroll
    for (int j = 0; j < NB; j++) B[j * NB + i] = u[j];
    // derivatives along a row: at the lane's points dr[k] (of node column k),
    // at the lane's nodes dc[k] (from point column k, a row of D's transpose);
    // weights of the lane's points (the table is symmetric).  Rows, so that a
    // lane's values come in few wide loads.
    R dr[NB], dc[NB], w[NB];
    auto load_force_tables = [&]() {
#pragma unroll
      for (int k = 0; k < NB; k++) {
        dc[k] = prm.D[NB * NB + i * NB + k];
        w[k] = prm.w2[i * NB + k];
      }
    };
#pragma unroll
    for (int k = 0; k < NB; k++) dr[k] = prm.D[i * NB + k];
    if constexpr (MODE != MODE_F64) load_force_tables();
    wave_lds_order();
    if constexpr (MODE == MODE_F64) {
      // dN_dy of the element row, iJ11 D[qj][j], formed once on the host
      CR *dny = (CR *)(uintptr_t)prm.dny + (long)ey * (NB * NB);
      R own[NB];  // 1 for the lane's own column
#pragma unroll
      for (int k = 0; k < NB; k++) {
        dr[k] = iJ00 * dr[k];
        own[k] = k == i ? R(1) : R(0);
      }
      R sxx[NB], sxy[NB], syy[NB];
#pragma unroll
      for (int qj = 0; qj < NB; qj++) {
        CR *dq = here(dny + qj * NB);
        R e0 = R(0), e1 = R(0), e2 = R(0);
#pragma unroll
        for (int j = 0; j < qj; j++) {
          e1 = e1 + dq[j] * u[j].y;
          e2 = e2 + dq[j] * u[j].x;
        }
        e1 = e1 + dq[qj] * u[qj].y;
        const R tq = dq[qj] * u[qj].x;
#pragma unroll
        for (int k = 0; k < NB; k++) {
          const R2 uk = B[qj * NB + k];
          e0 = e0 + dr[k] * uk.x;
          e2 = e2 + fma(own[k], tq, dr[k] * uk.y);
        }
#pragma unroll
        for (int j = qj + 1; j < NB; j++) {
          e1 = e1 + dq[j] * u[j].y;
          e2 = e2 + dq[j] * u[j].x;
        }
        sxx[qj] = c11 * e0 + lam * e1;
        syy[qj] = lam * e0 + c11 * e1;
        sxy[qj] = mu * e2;
      }
      // after the displacement's last use: the registers take the one or the
      // other
      wave_lds_order();
      load_force_tables();
#pragma unroll
      for (int k = 0; k < NB; k++) dc[k] = iJ00 * dc[k];
      if constexpr (EARLY) node_loads();
#pragma unroll
      for (int qj = 0; qj < NB; qj++) B[qj * NB + i] = R2{sxx[qj], sxy[qj]};
      wave_lds_order();
      // row terms of node row j: points (k, j), k ascending, the lane's own
      // point with its column term inside
      auto row_terms = [&](int j, CR *dq, R2 &f) {
        const R cx = dq[j] * sxy[j], cy = dq[j] * syy[j];
        CR *wq = here(W + j * NB);
#pragma unroll
        for (int k = 0; k < NB; k++) {
          const R2 s = B[j * NB + k];
          const R nfac = -(detJ * wq[k]);
          f.x = f.x + nfac * fma(own[k], cx, dc[k] * s.x);
          f.y = f.y + nfac * fma(own[k], cy, dc[k] * s.y);
        }
      };
      auto column_term = [&](int qj, int j, CR *dq, R2 &f) {
        const R nfac = -(detJ * w[qj]);
        f.x = f.x + nfac * (dq[j] * sxy[qj]);
        f.y = f.y + nfac * (dq[j] * syy[qj]);
      };
      if (ly == 0) {  // uniform per wave
        R2 f = R2{R(0), R(0)};
#pragma unroll
        for (int qj = 0; qj < P; qj++) column_term(qj, P, dny + qj * NB, f);
        row_terms(P, dny + P * NB, f);
        F[P] = f;
      } else {
#pragma unroll
        for (int j = 0; j < NB; j++) F[j] = R2{R(0), R(0)};
#pragma unroll
        for (int qj = 0; qj < NB; qj++) {
          CR *dq = here(dny + qj * NB);
          row_terms(qj, dq, F[qj]);
#pragma unroll
          for (int j = 0; j < NB; j++)
            if (j != qj) column_term(qj, j, dq, F[j]);
        }
      }
      // Infinite forces of both signs make a NaN of a sum too, which costs time
      // and changes nothing.
      R2 sum = F[P];
      if (ly != 0) {
#pragma unroll
        for (int j = 0; j < P; j++) sum = R2{sum.x + F[j].x, sum.y + F[j].y};
      }
      if (__builtin_expect(__any(__builtin_isunordered(sum.x, sum.y)), 0)) {  // uniform per wave
        // Element and column again from the thread's index: held from above
        // they take registers of the operator (300 x 300 p7: 94 -> 111 us).
        int l = threadIdx.x;
        asm volatile("" : "+v"(l));
        l &= 63;
        const int le = min(l / NB, EPW - 1), col = min(l - le * NB, P), bx = (wave % WX) * EPW + le;
        const int x = min(max(ex0 - 1 + bx, 0), prm.mx - 1), el = x + ey * prm.mx;
        R2 *E = &buf[ly][bx][0];
        const R hx = R(0.5) * prm.elem_dx[x], hy = R(0.5) * prm.elem_dy[ey];
        const R *tD = prm.D, *tw = prm.w2, *tdny = prm.dny + (long)ey * (NB * NB);
        asm volatile("" : "+v"(tD), "+v"(tw), "+v"(tdny));  // vector registers are free here, scalar ones are not
        wave_lds_order();
#pragma unroll 1
        for (int j = 0; j < NB; j++) E[j * NB + col] = prm.u_in[(long)(ey * P + j) * prm.pitch + x * P + col];
        wave_lds_order();
#pragma unroll 1
        for (int n = ly != 0 ? 0 : P; n < NB; n++) {
          const R2 f = col_force_f64<P>(E, tD, tw, tdny, R(1) / hx, hx * hy, prm.lambda[el], prm.mu[el], col, n);
#pragma unroll
          for (int j = 0; j < NB; j++)
            if (j == n) F[j] = f;
        }
      }
    } else {
      const R s = -detJ;
      const R a1 = s * c11 * iJ00 * iJ00, a2 = s * lam * iJ00 * iJ11, a3 = s * c11 * iJ11 * iJ11;
      const R b1 = s * mu * iJ11 * iJ11, b2 = s * mu * iJ00 * iJ11, b3 = s * mu * iJ00 * iJ00;
      // rows of D, held in SGPRs up to p = 6
      auto table_row = [&](int qj) { return P > 6 ? here(D + qj * NB) : D + qj * NB; };
      // row stresses (A, Cx) and column stresses (Bs, E), as in
      // RegOperator::row_stress
      R2 rs[NB], cs[NB];
#pragma unroll
      for (int qj = 0; qj < NB; qj++) {
        CR *dq = table_row(qj);
        R dxux = R(0), dxuy = R(0), dyux = R(0), dyuy = R(0);
#pragma unroll
        for (int k = 0; k < NB; k++) {
          const R2 uk = B[qj * NB + k];
          dxux = fma(dr[k], uk.x, dxux);
          dxuy = fma(dr[k], uk.y, dxuy);
          dyux = fma((R)dq[k], u[k].x, dyux);
          dyuy = fma((R)dq[k], u[k].y, dyuy);
        }
        rs[qj] = R2{w[qj] * fma(a1, dxux, a2 * dyuy), w[qj] * fma(b3, dxuy, b2 * dyux)};
        cs[qj] = R2{w[qj] * fma(b1, dyux, b2 * dxuy), w[qj] * fma(a3, dyuy, a2 * dxux)};
      }
      wave_lds_order();
      node_loads();
#pragma unroll
      for (int qj = 0; qj < NB; qj++) B[qj * NB + i] = rs[qj];
      wave_lds_order();
      auto row_terms = [&](int j, R2 &f) {
#pragma unroll
        for (int k = 0; k < NB; k++) {
          const R2 t = B[j * NB + k];
          f.x = fma(dc[k], t.x, f.x);
          f.y = fma(dc[k], t.y, f.y);
        }
      };
      auto column_term = [&](int qj, int j, CR *dq, R2 &f) {
        f.x = fma((R)dq[j], cs[qj].x, f.x);
        f.y = fma((R)dq[j], cs[qj].y, f.y);
      };
      if (ly == 0) {
        R2 f = R2{R(0), R(0)};
#pragma unroll
        for (int qj = 0; qj < P; qj++) column_term(qj, P, D + qj * NB, f);
        row_terms(P, f);
        column_term(P, P, D + P * NB, f);
        F[P] = f;
      } else {
#pragma unroll
        for (int j = 0; j < NB; j++) F[j] = R2{R(0), R(0)};
#pragma unroll
        for (int qj = 0; qj < NB; qj++) {
          CR *dq = table_row(qj);
          row_terms(qj, F[qj]);
#pragma unroll
          for (int j = 0; j < NB; j++) column_term(qj, j, dq, F[j]);
        }
      }
    }
    // The edges that the neighbours read: node column p (i = p) and node row
    // p, where the rows' stresses were.
    wave_lds_order();
    if (ly != 0) {
#pragma unroll
      for (int j = 0; j < P; j++)
        if (i == P) B[j * NB + P] = F[j];
    }
    B[P * NB + i] = F[P];
  }
  if constexpr (!EARLY) node_loads();
  const TileLists tl = tile_lists(prm, tile, step, last);
  __syncthreads();
  const bool left = ex > 0 && i == 0, below = ey > 0;
  if (mine) {  // own force and the neighbours' in ascending element order
    const R2 *L = &buf[ly][lx - 1][0], *Dn = &buf[ly - 1][lx][0], *Dg = &buf[ly - 1][lx - 1][0];
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if (j == 0 && below) {
        R2 f = Dn[P * NB + i];
        if (left) {  // (ex-1,ey-1), (ex,ey-1), (ex-1,ey), own
          const R2 d = Dg[P * NB + P], l = L[P];
          f = R2{(d.x + f.x) + l.x, (d.y + f.y) + l.y};
        }
        F[j] = R2{f.x + F[j].x, f.y + F[j].y};
      } else if (left) {
        const R2 l = L[j * NB + P];
        F[j] = R2{l.x + F[j].x, l.y + F[j].y};
      }
    }
  }
  auto update_node = [&](int j, int last_step) {
    const TileLists none{0, 0, 0, 0, 0, 0, step, last_step};
    node_update_core<P, MODE>(prm, none, gx, gy0 + j, idx0 + (long)j * prm.pitch, F[j].x, F[j].y, pu[j].x, pu[j].y, pv[j],
                              pm[j], pc[j]);
  };
  // Almost every tile and step has no source, no receiver and no last-step
  // stores: a copy of the update without them, p + 1 nodes of straight code.
  if (tl.empty() && !last) {
    if (mine) {
#pragma unroll
      for (int j = 0; j < NB; j++)
        if (j < P || tb) update_node(j, 0);
    }
    return;
  }
  // With sources and receivers: a lane holds one list entry (64 at a time) and
  // every lane tests its node against each in turn, so the lists cost no memory
  // latency per node (36 elements at p = 8 with 8 receivers: 29 -> 24 us a
  // step).  The loops are uniform and every lane takes part in them; an entry is
  // read from its lane before the branch on the node, in which that lane may be
  // idle and its registers are not kept.
  // The lane's entries of the tile's source and receiver lists, with the node
  // coordinates of their element's first node.
  struct ListItem { int id, x, y, gll; };
  auto list_item = [&](const int *idx, const int *elem, int t0, int t1) {
    ListItem it{0, 0, 0, 0};
    if (t0 + lane < t1) {
      it.id = idx[t0 + lane];
      const int e = elem[it.id];
      it.x = e % prm.mx * P;
      it.y = e / prm.mx * P;
    }
    return it;
  };
  R psi = R(0);  // the source's value at this step
  auto source = [&](int t0) {
    const ListItem it = list_item(prm.tile_src_idx, prm.src_elem, t0, tl.s1);
    psi = prm.psi[(long)step * prm.ns + it.id];
    return it;
  };
  auto receiver = [&](int t0) {
    ListItem it = list_item(prm.tile_rec_idx, prm.rec_elem, t0, tl.r1);
    it.gll = prm.rec_gll[it.id];
    return it;
  };
  ListItem src{0, 0, 0, 0}, rec{0, 0, 0, 0};
  if (tl.s0 < tl.s1) src = source(tl.s0);
  if (tl.r0 < tl.r1) rec = receiver(tl.r0);
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const bool node = mine && (j < P || tb);
    R2 sum{R(0), R(0)};
    bool hit = false;
    for (int t0 = tl.s0; t0 < tl.s1; t0 += 64) {
      if (tl.s1 - tl.s0 > 64) src = source(t0);
      const int n = min(64, tl.s1 - t0);
      for (int t = 0; t < n; t++) {
        const int li = gx - lane_value(src.x, t), lj = gy0 + j - lane_value(src.y, t), id = lane_value(src.id, t);
        const R ps = lane_value(psi, t);
        if (node && li >= 0 && li <= P && lj >= 0 && lj <= P) {
          const long k = ((long)id * NB * NB + li + lj * NB) * 2;
          sum.x = sum.x + ps * prm.src_vals[k];
          sum.y = sum.y + ps * prm.src_vals[k + 1];
          hit = true;
        }
      }
    }
    if (hit) F[j] = R2{F[j].x + sum.x, F[j].y + sum.y};
    // the corrected velocity and the acceleration, as the update forms them
    // (node_finish_f64 / _f32)
    auto corrected = [&](R2 &v, R2 &a) {
      if constexpr (MODE == MODE_F64) {
        a = R2{F[j].x / pm[j], F[j].y / pm[j]};
        v = R2{pv[j].x + prm.hdt * a.x, pv[j].y + prm.hdt * a.y};
      } else {
        a = R2{F[j].x * pm[j], F[j].y * pm[j]};
        v = R2{fma(prm.hdt, a.x, pv[j].x), fma(prm.hdt, a.y, pv[j].y)};
      }
    };
    for (int t0 = tl.r0; t0 < tl.r1; t0 += 64) {
      if (tl.r1 - tl.r0 > 64) rec = receiver(t0);
      const int n = min(64, tl.r1 - t0);
      for (int t = 0; t < n; t++) {
        const int li = gx - lane_value(rec.x, t), lj = gy0 + j - lane_value(rec.y, t), g = lane_value(rec.gll, t);
        const int id = lane_value(rec.id, t), gi = g % NB, gj = g / NB;
        const bool on_column = li == gi && lj >= 0 && lj <= P, on_row = lj == gj && li >= 0 && li <= P;
        if (node && (on_column || on_row)) {
          R2 v, a;
          corrected(v, a);
          R *o = prm.rec + ((long)step * prm.nr + id) * rec_stride(P);
          if (on_column) o[6 + lj] = v.x;
          if (on_row) o[6 + NB + li] = v.y;
          if (on_column && on_row) {
            o[0] = pu[j].x; o[1] = pu[j].y; o[2] = v.x; o[3] = v.y; o[4] = a.x; o[5] = a.y;
          }
        }
      }
    }
    for (int t0 = tl.q0; t0 < tl.q1; t0 += 64) {  // element receivers: every node of the element
      const ListItem er = list_item(prm.tile_erec_idx, prm.erec_elem, t0, tl.q1);
      const int n = min(64, tl.q1 - t0);
      for (int t = 0; t < n; t++) {
        const int li = gx - lane_value(er.x, t), lj = gy0 + j - lane_value(er.y, t), id = lane_value(er.id, t);
        if (node && li >= 0 && li <= P && lj >= 0 && lj <= P) {
          R2 v, a;
          corrected(v, a);
          R *q = prm.erec + (((long)step * prm.ner + id) * (NB * NB) + li + lj * NB) * 4;
          q[0] = pu[j].x; q[1] = pu[j].y; q[2] = v.x; q[3] = v.y;
        }
      }
    }
    if (node) update_node(j, last);
  }
}

// Minimum waves per SIMD, i.e. the registers per lane: the most at which the
// waves gain more than the spills cost.  FP64 p = 4 and 6 spill 6 registers, p =
// 7 spills 32 at three (300 x 300: 90-95 us, 100 at two, without spills), 512 x
// 512 p4 takes 74 us at four and 77 at three; at p = 8 three waves spill 50
// registers (256 x 256: 114 us, 95-104 at two), and FP32+Kahan p = 8 10 at four
// (512 x 512: 254 us, 230 at three).
constexpr int col_waves(int p, int mode) {
  return mode == MODE_F64 ? (p <= 4 ? 4 : p <= 7 ? 3 : 2) : mode == MODE_F32K && p == 8 ? 3 : 4;
}

template <int P, int MODE, int WX, int EY>
__global__ __launch_bounds__(64 * WX * EY) __attribute__((amdgpu_waves_per_eu(col_waves(P, MODE), 8)))
void col_kernel(StepParams<typename RealOf<MODE>::T> prm) {
  const int tile = tile_of_block(blockIdx.x, prm.tiles_per_xcd);
  if (tile >= prm.tiles_x * prm.tiles_y) return;  // uniform per workgroup
  col_body<P, MODE, WX, EY>(prm, tile, prm.step, prm.last);
}

}  // namespace se2w
