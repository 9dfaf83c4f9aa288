// cbm_stage.h -- the integrator-stage kernel body and the row/cell
// geometry helpers it needs.  Self-contained (with cbm_device.h and
// cbm_structs.h) so hipRTC can compile it around a user interaction body.
#ifndef CBM_STAGE_H
#define CBM_STAGE_H

#include "cbm_device.h"
#include "cbm_structs.h"

#ifndef CBM_LIST_CHUNK
#define CBM_LIST_CHUNK 2
#endif

namespace cbm {

// ------------------------------------------------------------ row geometry
struct RowIdx { int sim; int64_t local; int64_t row; };

// Blocks are dispatched round-robin over the 8 XCDs; remap so that each XCD
// (own L2) serves one contiguous range of rows, i.e. one compact region of
// the Morton-ordered agents, and neighbor gathers stay in that L2.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int q = nb >> 3, r = nb & 7;
  const int x = b & 7, idx = b >> 3;
  return x < r ? x * (q + 1) + idx : r * (q + 1) + (x - r) * q + idx;
}

// Row of this thread for block bx of a launch whose first nb blocks serve
// the rows.
__device__ __forceinline__ RowIdx row_index_of(const RowGeom& g, int bx, int nb) {
  RowIdx r;
  const int b = xcd_tile(bx, nb);
  r.sim = g.block_sim[b];
  r.local = (int64_t)(b - g.block_off[r.sim]) * blockDim.x + threadIdx.x;
  r.row = g.sims[r.sim].row_off + r.local;
  return r;
}

__device__ __forceinline__ RowIdx row_index(const RowGeom& g) {
  RowIdx r;
  const int b = xcd_tile((int)blockIdx.x, (int)gridDim.x);
  r.sim = g.block_sim[b];
  r.local = (int64_t)(b - g.block_off[r.sim]) * blockDim.x + threadIdx.x;
  r.row = g.sims[r.sim].row_off + r.local;
  return r;
}

__device__ __forceinline__ double min_image(double d, double L) {
  if (d > 0.5 * L) d -= L; else if (d < -0.5 * L) d += L;
  return d;
}

// k-th of the 3^D neighbor cells (cellPosNeigh order, x fastest) as a local
// cell index, or -1 outside a non-periodic grid.
template <int D>
__device__ __forceinline__ int32_t neigh_cell(const SimDev& sd, int32_t cx, int32_t cy, int32_t cz, int k, int periodic) {
  int32_t q[3] = {cx, cy, cz};
  const int off[3] = {k % 3 - 1, (k / 3) % 3 - 1, k / 9 - 1};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    int32_t v = q[a] + off[a];
    if (periodic) { v = v < 0 ? v + sd.gn[a] : (v >= sd.gn[a] ? v - sd.gn[a] : v); }
    else if (v < 0 || v >= sd.gn[a]) return -1;
    q[a] = v;
  }
  return q[0] + sd.gn[0] * (q[1] + sd.gn[1] * q[2]);
}

// Cell of x on the model's grid along axis a: cellPos (src/neighbors.jl:
// 636-638, 0-based) on the padded grid, clamped on the periodic one.
__device__ __forceinline__ int32_t cl_axis(const SimDev& sd, int a, double x, int periodic) {
  if (periodic) {
    int64_t c = floor_div(x - sd.lo[a], sd.cedge[a]);
    c = c < 0 ? 0 : (c > sd.cgn[a] - 1 ? sd.cgn[a] - 1 : c);
    return (int32_t)c;
  }
  if (x > sd.hi[a]) return sd.cgn[a] - 1;
  if (x < sd.lo[a]) return 0;
  return (int32_t)(floor_div(x - sd.lo[a], sd.cedge[a]) + 1);
}

// The cell packed as 10 bits per axis (grids of at most 1023 cells per axis).
template <int D>
__device__ __forceinline__ int32_t cl_pack(const SimDev& sd, const double* x, int periodic) {
  int32_t v = 0;
#pragma unroll
  for (int a = 0; a < D; ++a) v |= cl_axis(sd, a, x[a], periodic) << (10 * a);
  return v;
}

// Position of cell pj among the 3^D neighbor cells of pi (cellPosNeigh
// order), or 27 when pj is not one of them.
template <int D, int PER>
__device__ __forceinline__ int cl_key(const SimDev& sd, int32_t pi, int32_t pj) {
  int k = 0, w = 1;
  bool adj = true;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    int d = ((pj >> (10 * a)) & 1023) - ((pi >> (10 * a)) & 1023);
    if (PER) d = d == sd.cgn[a] - 1 ? -1 : (d == 1 - sd.cgn[a] ? 1 : d);
    adj = adj && d >= -1 && d <= 1;
    k += (d + 1) * w;
    w *= 3;
  }
  return adj ? k : 27;
}

__host__ __device__ constexpr int pow3(int d) { return d == 1 ? 3 : (d == 2 ? 9 : 27); }

// A law with a per-agent term: `void self(const double* x, double* f) const`
// adds f (D values, zeroed before the call) to dt(x) at the stage state x,
// the agentODE body's terms that are not pair forces.
template <class L, class = void> struct has_self { static constexpr bool value = false; };
template <class L> struct has_self<L, decltype((void)&L::self)> { static constexpr bool value = true; };
template <class L, class = void> struct has_de { static constexpr bool value = false; };
template <class L> struct has_de<L, decltype((void)&L::de)> { static constexpr bool value = true; };

// A program around a body with user DE variables defines CBM_USER_DE (their
// count) and CBM_DE_BASE (the DE index of the first: dims, + 1 with vol).
#ifndef CBM_USER_DE
#define CBM_USER_DE 0
#define CBM_DE_BASE 0
#endif

// A general agentODE body (src/AgentStructure/functionDE.jl:13-116): a
// UserLaw with
//   static constexpr int sums = K;     // neighbor sums, 1..8
//   __device__ void pair(const LawAgent& i, const LawAgent& j, const double* dx, double d, double* s) const;
//   __device__ void ode(const LawAgent& i, const double* s, double* dxdt, double* dudt) const;
// The skeleton zeroes s[0..K), calls pair for every neighbor candidate j of
// agent i in reference loop order (dx = x_i - x_j, minimum image in a
// periodic box; d = |dx|), each call adding its terms to s in whatever order
// the body writes, and then ode with the sums: dxdt[0..D) = dt of the
// positions, dudt[k] = dt of user DE variable k (both zeroed before the call).
// The agents are seen at the stage state.
template <class L, class = void> struct general_body { static constexpr bool value = false; };
template <class L> struct general_body<L, decltype((void)&L::ode)> { static constexpr bool value = true; };
template <class L, class = void> struct law_sums { static constexpr int value = 1; };
template <class L> struct law_sums<L, decltype((void)L::sums)> { static constexpr int value = L::sums; };
// the Aggregation wall push, for laws that declare it
template <class L, class = void> struct law_walls { static constexpr bool value = false; };
template <class L> struct law_walls<L, decltype((void)L::walls)> {
  static constexpr bool value = L::active && L::walls;
};

// One agent of a pair as a general agentODE body sees it.
struct LawAgent {
  int64_t row, id;
  double x[3];              // position at the stage state
  double uv[USER_PARAMS];   // user parameters U0..U7: DE variables at the stage state, others as stored
  double volv;              // vol at the stage state (1 without the vol variable)
  __device__ double u(int k) const { return uv[k]; }
  __device__ double vol() const { return volv; }
};

template <int D, class Args>
__device__ __forceinline__ LawAgent law_agent(const Args& a, int64_t row, const double* x) {
  LawAgent r;
  r.row = row;
  r.id = a.id[row];
#pragma unroll
  for (int c = 0; c < 3; ++c) r.x[c] = c < D ? x[c] : 0.0;
#pragma unroll
  for (int k = 0; k < USER_PARAMS; ++k)
    r.uv[k] = k < CBM_USER_DE ? a.S[CBM_DE_BASE + k][row] : (a.upar[k] ? a.upar[k][row] : 0.0);
  r.volv = a.growth ? a.S[D][row] : 1.0;
  return r;
}

// Walk the candidate neighbors of row i in reference loop order (Args: the
// stage or rule arguments, with the list and cell tables of the last
// neighbor update).
template <int D, int NB, class Args, class Fn>
__device__ __forceinline__ void for_candidates(const Args& a, const SimDev& sd, int64_t N, int64_t i, Fn&& fn) {
  if (NB == NB_LIST) {
    const int32_t cnt = a.list_n[i];
    for (int32_t q = 0; q < cnt; ++q) fn((int64_t)a.list[(int64_t)q * a.ldl + i]);
  } else if (NB == NB_FULL) {
    const int64_t j0 = sd.row_off, j1 = sd.row_off + N;
    for (int64_t j = j0; j < j1; ++j) if (j != i) fn(j);
  } else {
    const int32_t c = a.cell_row[i];
    const int32_t cx = c % sd.gn[0];
    const int32_t cy = (c / sd.gn[0]) % sd.gn[1];
    const int32_t cz = c / (sd.gn[0] * sd.gn[1]);
    const CellRange* __restrict__ cr = a.cell_range + sd.rank_off;
    for (int k = 0; k < pow3(D); ++k) {
      const int32_t nc = neigh_cell<D>(sd, cx, cy, cz, k, a.periodic);
      if (nc < 0) continue;
      const CellRange r = cr[nc];
      for (int32_t j = r.s; j < r.e; ++j) if (j != i) fn((int64_t)j);
    }
  }
}

// Periodic box: a coordinate brought back into [lo, lo + L) (one period at most).
__device__ __forceinline__ double wrap_box(double x, double lo, double L) {
  if (x >= lo + L) return x - L;
  if (x < lo) return x + L;
  return x;
}

// ----------------------------------------------------------- stage kernel
// Minimum image (periodic boxes): the same comparisons as the oracle, as selects.
__device__ __forceinline__ double wrap_dx(double d, double L, double hL) {
  return d > hL ? d - L : (d < -hL ? d + L : d);
}

// The library's terms of a pair: dx, d^2 -> the term the agentODE interaction
// body adds to the accumulator, in the reference's per-axis order; +0 for an
// inactive pair (the accumulator starts at +0 and a sum is -0 only when both
// terms are, so it is never -0 and adding +0 or -0 leaves it unchanged).
template <int D, class Law, bool SOFT>
__device__ __forceinline__ void pair_library(const Law& law, const double* dx, double s2, double rad_i, double rad_j,
                                             int64_t fate_i, int64_t fate_j, bool live, double* t) {
  const double d = sqrt(s2);
  double s;
  bool on;
  if constexpr (SOFT) on = law.pair(d, rad_i, rad_j, fate_i, fate_j, s) && live;
  else on = law(d, s) && live;
  if constexpr (SOFT) {
    // ((s dx) / d) per axis, the reference's order (softSpheres.jl:28-29)
#pragma unroll
    for (int c = 0; c < D; ++c) t[c] = on ? (s * dx[c]) / d : 0.0;
  } else if (Law::per_axis_division) {
#pragma unroll
    for (int c = 0; c < D; ++c) t[c] = on ? s * (dx[c] / d) : 0.0;
  } else {
    const double f = s / d;
    const double fe = on ? f : 0.0;
#pragma unroll
    for (int c = 0; c < D; ++c) t[c] = fe * dx[c];
  }
}

// The built-in laws with near() and plain(): their root and quotient in range
// (root_inv, quotient).  By type: a user's law may have members of any name.
template <class L> struct has_near { static constexpr bool value = false; };
template <> struct has_near<PairLaw<LAW_LINEAR>> { static constexpr bool value = true; };
template <> struct has_near<PairLaw<LAW_REP_ADH>> { static constexpr bool value = true; };
template <> struct has_near<PairLaw<LAW_SOFT_SPHERES>> { static constexpr bool value = true; };

// What a law's range test lets through: nothing unless its constants do.
template <class Law>
__device__ __forceinline__ uint32_t law_span(const Law& law) {
  if constexpr (has_near<Law>::value) return law.plain() ? ROOT_SPAN : 0u;
  else return 0u;
}

// The terms of U neighbors at positions xj (+0 for one that is not live: list
// padding, or the agent itself).  A wavefront whose pairs all lie in range
// takes the short root and quotient, any other the library's: the same bits.
template <int D, class Law, int PER, bool SOFT, int U>
__device__ __forceinline__ void pair_terms(const Law& law, uint32_t span, const double* xi, const double (*xj)[3],
                                           const double* L, const double* hL, double rad_i, const double* rad_j,
                                           int64_t fate_i, const int64_t* fate_j, const bool* live, double (*t)[3]) {
  double dx[U][3], s2[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int c = 0; c < D; ++c) {
      dx[u][c] = xi[c] - xj[u][c];
      if (PER) dx[u][c] = wrap_dx(dx[u][c], L[c], hL[c]);
    }
    s2[u] = dx[u][0] * dx[u][0];
    if (D > 1) s2[u] = s2[u] + dx[u][1] * dx[u][1];
    if (D > 2) s2[u] = s2[u] + dx[u][2] * dx[u][2];
  }
  if constexpr (has_near<Law>::value) {
    bool bad = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bool ok = root_range(s2[u], span);
      if constexpr (SOFT) {
        // the numerators r_ij and s dx: no tiny offsets
        ok = ok && plain_length(rad_i + rad_j[u]);
#pragma unroll
        for (int c = 0; c < D; ++c) ok = ok && plain_constant(dx[u][c]);
      }
      bad = bad || (live[u] && !ok);
    }
    if (!__any(bad)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const RootInv q = root_inv(s2[u]);
        double s;
        if constexpr (SOFT) {
          const bool on = law.near(q.d, q.r, rad_i + rad_j[u], fate_i, fate_j[u], s) && live[u];
#pragma unroll
          for (int c = 0; c < D; ++c) {
            const double v = quotient(s * dx[u][c], q.d, q.r);
            t[u][c] = on ? v : 0.0;
          }
        } else {
          const bool on = law.near(q.d, s) && live[u];
          const double f = quotient(s, q.d, q.r);
          const double fe = on ? f : 0.0;
#pragma unroll
          for (int c = 0; c < D; ++c) t[u][c] = fe * dx[u][c];
        }
      }
      return;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    pair_library<D, Law, SOFT>(law, dx[u], s2[u], rad_i, SOFT ? rad_j[u] : 0.0, fate_i, SOFT ? fate_j[u] : 0, live[u],
                               t[u]);
}

// One neighbor's term.
template <int D, class Law, int PER, bool SOFT = false>
__device__ __forceinline__ void pair_term(const Law& law, uint32_t span, const double* xi, const double* xj,
                                          const double* L, const double* hL, bool live, double* t, double rad_i = 0.0,
                                          double rad_j = 0.0, int64_t fate_i = 0, int64_t fate_j = 0) {
  double x[1][3] = {{0.0, 0.0, 0.0}}, o[1][3];
#pragma unroll
  for (int c = 0; c < D; ++c) x[0][c] = xj[c];
  pair_terms<D, Law, PER, SOFT, 1>(law, span, xi, x, L, hL, rad_i, &rad_j, fate_i, &fate_j, &live, o);
#pragma unroll
  for (int c = 0; c < D; ++c) t[c] = o[0][c];
}

template <int D, int PER>
__device__ __forceinline__ void box_halves(const SimDev& sd, double* L, double* hL) {
#pragma unroll
  for (int c = 0; c < 3; ++c) { L[c] = 0.0; hL[c] = 0.0; }
  if (PER) {
#pragma unroll
    for (int c = 0; c < D; ++c) { L[c] = sd.L[c]; hL[c] = 0.5 * sd.L[c]; }
  }
}

// Pair sum of row i over its candidates in global memory (Verlet list,
// all rows, or the cell-linked walk), in reference loop order.
template <int D, int NB, class Law, int PER>
__device__ __forceinline__ void gather_global(const StageArgs& a, const SimDev& sd, int64_t N, int64_t i,
                                              const double* xi, double* acc) {
  constexpr bool SOFT = same_type<Law, PairLaw<LAW_SOFT_SPHERES>>::value;
  const Law law(sd.p);
  const double rad_i = SOFT ? a.rad[i] : 0.0;
  const int64_t fate_i = SOFT ? a.fate[i] : 0;
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  const uint32_t span = law_span(law);
  if (NB == NB_LIST) {
    // Verlet list in chunks of LCH gathers issued together (memory-level
    // parallelism per lane), branch-free: slots past the count read the
    // agent itself and add nothing.  The list indices of the next chunk are
    // loaded before the current chunk's positions are used.
    constexpr int LCH = CBM_LIST_CHUNK;
    const int32_t cnt = a.list_n[i];
    const int64_t ldl = a.ldl;
    const int32_t* __restrict__ lp = a.list + i;     // entry q at lp[q * ldl]
    int32_t jn[LCH];
#pragma unroll
    for (int u = 0; u < LCH; ++u) jn[u] = (u < cnt) ? lp[(int64_t)u * ldl] : (int32_t)i;
    for (int32_t q0 = 0; q0 < cnt; q0 += LCH) {
      double px[LCH][3], t[LCH][3], rj[LCH];
      int32_t jc[LCH];
      int64_t fj[LCH];
      bool live[LCH];
#pragma unroll
      for (int u = 0; u < LCH; ++u) {
        jc[u] = jn[u];
        live[u] = q0 + u < cnt;
#pragma unroll
        for (int c = 0; c < D; ++c) px[u][c] = a.S[c][jc[u]];
        rj[u] = SOFT ? a.rad[jc[u]] : 0.0;
        fj[u] = SOFT ? a.fate[jc[u]] : 0;
      }
      lp += LCH * ldl;
#pragma unroll
      for (int u = 0; u < LCH; ++u) jn[u] = (q0 + LCH + u < cnt) ? lp[(int64_t)u * ldl] : (int32_t)i;
      if constexpr (has_near<Law>::value) {
        // one pair after the other: the first one's arithmetic covers the way
        // of the second one's position and of the indices, for which a range
        // test of both at once would wait (device time per step: 2,305 agents
        // in space, Euler, 17.4 -> 17.1 us; 4,001 in the plane, Heun, 23.1 ->
        // 22.1; 12,001 in space, RK4, 36.4 -> 35.4; a million, Heun, 92.0 -> 91.4)
#pragma unroll
        for (int u = 0; u < LCH; ++u) {
          pair_term<D, Law, PER, SOFT>(law, span, xi, px[u], L, hL, live[u], t[u], rad_i, rj[u], fate_i, fj[u]);
#pragma unroll
          for (int c = 0; c < D; ++c) acc[c] = acc[c] + t[u][c];
        }
      } else {
        pair_terms<D, Law, PER, SOFT, LCH>(law, span, xi, px, L, hL, rad_i, rj, fate_i, fj, live, t);
#pragma unroll
        for (int u = 0; u < LCH; ++u)
#pragma unroll
          for (int c = 0; c < D; ++c) acc[c] = acc[c] + t[u][c];
      }
    }
  } else {
    for_candidates<D, NB>(a, sd, N, i, [&](int64_t j) {
      double xj[3] = {0.0, 0.0, 0.0}, t[3];
#pragma unroll
      for (int c = 0; c < D; ++c) xj[c] = a.S[c][j];
      pair_term<D, Law, PER, SOFT>(law, span, xi, xj, L, hL, true, t, rad_i, SOFT ? a.rad[j] : 0.0, fate_i,
                                   SOFT ? a.fate[j] : 0);
#pragma unroll
      for (int c = 0; c < D; ++c) acc[c] = acc[c] + t[c];
    });
  }
}

// The rest of the stage for row i once the pair sum acc is known: walls,
// the derivative of every DE variable, the integrator update, periodic
// wrap, the output write and the displacement check.
// Noise amplitude of the agentSDE part.  ConstNoise is the model's constant g
// on the positions (StageArgs::noise).  A user body (hipRTC) defines
//   struct UserNoise {
//     __device__ explicit UserNoise(const double* p);          // the simulation's p[8]
//     __device__ double operator()(int var, const double* u) const;
//   };
// giving g of DE variable var at the agent's state u (positions, then the
// other DE variables), evaluated at the stage state as the reference's g
// (src/integrators.jl:709-727 EM, :775-803 EulerHeun).
struct ConstNoise {
  __device__ explicit ConstNoise(const double*) {}
  __device__ double operator()(int, const double*) const { return 0.0; }
};

// Row i changed its cell on the model's grid: its list and those that hold it
// (its own entries: skin lists are symmetric) are ordered anew next step.  The
// lists of a row at capacity may miss it, so then every list is.
__device__ __forceinline__ void clv_moved(const StageArgs& a, int64_t i) {
  const int32_t n = a.list_n[i];
  a.order_row_next[i] = 1;
  if (n >= a.lcap) *a.order_next = 1;
  else
    for (int32_t q = 0; q < n; ++q) a.order_row_next[a.list[(int64_t)q * a.ldl + i]] = 1;
}

template <int D, class Law, int NOISE, bool PRE = false, class Noise = ConstNoise>
__device__ __forceinline__ void stage_finish(const StageArgs& a, const SimDev& sd, int sim, int64_t i,
                                             const double* xi, double* acc, const double* upre,
                                             double disp2 = -1.0, double* e2_out = nullptr) {
  constexpr bool SOFT = same_type<Law, PairLaw<LAW_SOFT_SPHERES>>::value;
  constexpr bool RODS = same_type<Law, RodLaw>::value;
  // u of variable c (with PRE, the caller loaded the positions' u early into
  // upre), and the stage state, whose positions are xi
  const double u0 = upre[0], u1 = upre[1], u2 = upre[2];   // values, so no pointer is selected
  auto Uc = [&](int c) -> double {
    if (PRE && c < D) return c == 0 ? u0 : (c == 1 ? u1 : u2);
    return a.U[c][i];
  };
  auto Sc = [&](int c) { return c < D ? xi[c] : a.S[c][i]; };
  if (law_walls<Law>::value && a.walls && sd.p[4] != 0.0) {   // p[4]: the walls switch
    const double rRep = sd.p[0], fRep = sd.p[1];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      const double x = xi[c];
      if (x < sd.lo[c] + rRep / 2) acc[c] = acc[c] + fRep;
      else if (x > sd.hi[c] - rRep / 2) acc[c] = acc[c] - fRep;
    }
  }

  // derivative of each DE variable
  constexpr bool PAIRB = general_body<Law>::value;
  constexpr bool UDE = CBM_USER_DE > 0 && (has_de<Law>::value || PAIRB);
  constexpr int NS = (UDE || RODS) ? MAX_STATE : BUILTIN_STATE;
  double du[NS];
  double dudt[4] = {0.0, 0.0, 0.0, 0.0};
  if constexpr (PAIRB) {
    // a general agentODE body: its equations from the neighbor sums acc
    const LawAgent me = law_agent<D>(a, i, xi);
    double dxdt[3] = {0.0, 0.0, 0.0};
    const Law law(sd.p);
    law.ode(me, acc, dxdt, dudt);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      double v = dxdt[c];
      if (a.drift != 0.0) v = v - a.drift * xi[c];
      du[c] = v;
    }
  } else if constexpr (RODS) {
    // acc = {fx, fy, W, pressure}; the DE variables x, y, vx, vy, theta,
    // omega (src/models/rods.jl:111-116)
    const double beta = sd.p[5], bw = sd.p[6];
    const double m = a.mass[i], d = a.rod_d[i], l = (a.nvar == 7 ? a.S[6] : a.rod_l)[i];
    const double vx = a.S[2][i], vy = a.S[3][i], om = a.S[5][i];
    du[0] = vx;
    du[1] = vy;
    du[2] = -beta * vx + acc[0] / m;
    du[3] = -beta * vy + acc[1] / m;
    du[4] = om;
    du[5] = acc[2] / (m * ((d + l) * (d + l)) / 12 + m * (d * d)) - bw * om;
    // rods2dGrowth (src/models/rods.jl:137-139): the length grows, slowed by
    // this evaluation's pressure
    if (a.nvar == 7) du[6] = a.rod_growth / (1 + a.rod_alpha * acc[3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) a.rod_out[k][i] = acc[k];
  } else if constexpr (SOFT) {
    // dt(v) = -b*v/m + f/m, dt(x) = v (src/models/softSpheres.jl:32-35)
    const double b = sd.p[0], m = a.mass[i];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      const double f = a.lagged ? a.F[c][i] : acc[c];
      const double v = a.S[D + c][i];
      du[c] = v;
      du[D + c] = -b * v / m + f / m;
      if (a.write_fnew) a.Fnew[c][i] = acc[c];
    }
  } else {
    double fs[3] = {0.0, 0.0, 0.0};
    if constexpr (has_self<Law>::value) {
      double xs[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int c = 0; c < D; ++c) xs[c] = xi[c];
      const Law law(sd.p);
      law.self(xs, fs);
    }
#pragma unroll
    for (int c = 0; c < D; ++c) {
      double v = a.lagged ? a.F[c][i] : acc[c];
      if (a.drift != 0.0) v = v - a.drift * xi[c];
      if constexpr (has_self<Law>::value) v = v + fs[c];
      du[c] = v;
      if (a.write_fnew) a.Fnew[c][i] = acc[c];
    }
  }
  const bool grow = UDE ? CBM_DE_BASE > D : !SOFT && !RODS && a.nvar > D;
  if (grow) du[D] = a.growth[i] * a.S[D][i];
  if constexpr (UDE) {
    // dt of the user DE variables at the stage state
    if constexpr (PAIRB) {
#pragma unroll
      for (int k = 0; k < CBM_USER_DE; ++k) du[CBM_DE_BASE + k] = dudt[k];
    } else {
      double xs[3] = {0.0, 0.0, 0.0}, us[4] = {0.0, 0.0, 0.0, 0.0}, ds[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int c = 0; c < D; ++c) xs[c] = xi[c];
#pragma unroll
      for (int k = 0; k < CBM_USER_DE; ++k) us[k] = a.S[CBM_DE_BASE + k][i];
      const Law law(sd.p);
      law.de(xs, us, ds);
#pragma unroll
      for (int k = 0; k < CBM_USER_DE; ++k) du[CBM_DE_BASE + k] = ds[k];
    }
  }

  const double dt = a.dt;
  const int nv = UDE ? CBM_DE_BASE + CBM_USER_DE : (RODS ? a.nvar : (SOFT ? 2 * D : (grow ? D + 1 : D)));
  double res[NS];
  if (NOISE && !same_type<Noise, ConstNoise>::value) {
    // a user agentSDE body: g of every DE variable at the stage state, one
    // normal per variable (pairs keyed pur, pur + 1, pur + 2); the
    // EulerHeun corrector averages g of both stages, g of stage 1 kept in gacc
    const int64_t id = a.id[i];
    const int64_t step = *a.step_ptr;
    const uint32_t pur = a.kind == ST_EH2 ? 0x500u : 0x100u;
    double z[NS], us[NS];
#pragma unroll
    for (int k = 0; k < NS / 2; ++k) {
      z[2 * k] = 0.0;
      z[2 * k + 1] = 0.0;
      if (2 * k < nv) normal2(draw(a.seed, step, id, sim, pur + (uint32_t)k), z[2 * k], z[2 * k + 1]);
    }
#pragma unroll
    for (int v = 0; v < NS; ++v) us[v] = v < nv ? Sc(v) : 0.0;
    const Noise gfn(sd.p);
#pragma unroll
    for (int v = 0; v < NS; ++v) {
      if (v >= nv) continue;
      const double g = gfn(v, us);
      const double u = v < D ? Uc(v) : a.U[v][i];
      if (a.kind == ST_EH2) {
        res[v] = u + ((a.kacc[v][i] + du[v]) * dt + (a.gacc[v][i] + g) * z[v] * a.sqdt) / 2;
      } else {
        res[v] = (u + du[v] * dt) + g * z[v] * a.sqdt;
        if (a.kind == ST_EH1) { a.kacc[v][i] = du[v]; a.gacc[v][i] = g; }
      }
    }
  } else if (NOISE) {
    // EM and the EulerHeun predictor: (u + f dt) + (g xi) sqrt(dt), xi keyed
    // 0x100/0x101; the EulerHeun corrector draws fresh noise (0x500/0x501)
    double z[4] = {0.0, 0.0, 0.0, 0.0};
    const int64_t id = a.id[i];
    const int64_t step = *a.step_ptr;
    const uint32_t pur = a.kind == ST_EH2 ? 0x500u : 0x100u;
    normal2(draw(a.seed, step, id, sim, pur), z[0], z[1]);
    if (D > 2) normal2(draw(a.seed, step, id, sim, pur + 1u), z[2], z[3]);
    if (a.kind == ST_EH2) {
#pragma unroll
      for (int c = 0; c < D; ++c)
        res[c] = Uc(c) + ((a.kacc[c][i] + du[c]) * dt + (a.noise + a.noise) * z[c] * a.sqdt) / 2;
      for (int v = D; v < nv; ++v) res[v] = a.U[v][i] + ((a.kacc[v][i] + du[v]) * dt) / 2;
    } else {
#pragma unroll
      for (int c = 0; c < D; ++c) res[c] = (Uc(c) + du[c] * dt) + a.noise * z[c] * a.sqdt;
      for (int v = D; v < nv; ++v) res[v] = a.U[v][i] + du[v] * dt;   // no noise off the positions
      if (a.kind == ST_EH1)
        for (int c = 0; c < nv; ++c) a.kacc[c][i] = du[c];
    }
  } else {
    // variable c from its u; positions first (c known at compile time, so
    // an early-loaded u stays in registers), then the other DE variables
    auto upd = [&](int c, double u) -> double {
      switch (a.kind) {
        case ST_EULER:
        case ST_HEUN1:
          return u + du[c] * dt;
        case ST_HEUN2:
          return (Sc(c) + (u + du[c] * dt)) / 2;
        case ST_RK4_1:
          a.kacc[c][i] = du[c];
          return u + du[c] * dt / 2;
        case ST_RK4_2:
          a.kacc[c][i] = a.kacc[c][i] + 2 * du[c];
          return u + du[c] * dt / 2;
        case ST_RK4_3:
          a.kacc[c][i] = a.kacc[c][i] + 2 * du[c];
          return u + du[c] * dt;
        default:  // ST_RK4_4
          return u + (a.kacc[c][i] + du[c]) * dt / 6;
      }
    };
#pragma unroll
    for (int c = 0; c < D; ++c) res[c] = upd(c, Uc(c));
    for (int v = D; v < nv; ++v) res[v] = upd(v, a.U[v][i]);
  }

  const bool final_stage = a.kind == ST_EULER || a.kind == ST_EM || a.kind == ST_HEUN2 ||
                           a.kind == ST_RK4_4 || a.kind == ST_EH2;
  if (final_stage && a.periodic) {
#pragma unroll
    for (int c = 0; c < D; ++c) res[c] = wrap_box(res[c], sd.lo[c], sd.L[c]);
  }
  for (int c = 0; c < nv; ++c) a.out[c][i] = res[c];
  if (a.clv) {
    // CellLinked on a skin list: the next step's cells, or this stage's
    // distance from the list's reference positions
    if (final_stage && a.ccell_out) {
      const int32_t cell = cl_pack<D>(sd, res, a.periodic);
      a.ccell_out[i] = cell;
      if (cell != a.ccell[i]) clv_moved(a, i);
    }
    if (!final_stage && e2_out) {
      double dx[3];
#pragma unroll
      for (int c = 0; c < D; ++c) {
        dx[c] = res[c] - a.xref[c][i];
        if (a.periodic) dx[c] = min_image(dx[c], sd.L[c]);
      }
      double s2 = dx[0] * dx[0];
      if (D > 1) s2 = s2 + dx[1] * dx[1];
      if (D > 2) s2 = s2 + dx[2] * dx[2];
      *e2_out = s2;
    }
  }
  if (disp2 >= 0.0) {
    // the stage-2 lists stay exact while no agent moves more than half their margin
    double s2 = 0.0;
#pragma unroll
    for (int c = 0; c < D; ++c) { const double d = res[c] - Uc(c); s2 = s2 + d * d; }
    if (!(s2 <= disp2)) *a.lgate = 0;
  }

  if (final_stage && (a.disp_check || (a.clv && a.efin))) {
    double dx[3];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      dx[c] = res[c] - a.xref[c][i];
      if (a.periodic) dx[c] = min_image(dx[c], sd.L[c]);
    }
    double s2 = dx[0] * dx[0];
    if (D > 1) s2 = s2 + dx[1] * dx[1];
    if (D > 2) s2 = s2 + dx[2] * dx[2];
    double st = 0.0;   // this step's displacement, squared
    if (a.clv) {
#pragma unroll
      for (int c = 0; c < D; ++c) {
        double d = res[c] - Uc(c);
        if (a.periodic) d = min_image(d, sd.L[c]);
        st = st + d * d;
      }
    }
    if (a.disp_check) {
      if (s2 > a.thr2) *a.flag = 1;   // sqrt(s2) >= thr, src/neighbors.jl:403 (>= skin/2)
      // CellLinked on a skin list rebuilds one step early: when this step's
      // displacement, repeated 1.5 times, would carry the agent past the
      // threshold, so that the next step's stages rarely leave half the skin
      if (a.clv && !(sqrt(s2) + 1.5 * sqrt(st) <= a.clv_half)) *a.flag = 1;
    }
    if (a.clv && a.efin) {
      // the displacement bound of the next step's stage 1 (agents past half
      // the skin; a value at or below the running maximum adds nothing), and
      // the host's cue to schedule a build: an agent that clv_ahead more
      // displacements like this step's would carry past half the skin
      if (s2 > a.clv_half2) {
        const unsigned long long e = (unsigned long long)__double_as_longlong(s2);
        if (e > *(volatile unsigned long long*)a.efin) atomicMax(a.efin, e);
      }
      if (!(sqrt(s2) + a.clv_ahead * sqrt(st) <= a.clv_half)) a.efin[1] = 1ull;
    }
  }
}

// One integrator stage for every agent row: the agentODE body over the
// neighbor candidates (Law = the pair law functor) fused with the stage
// update.  Built-in laws instantiate it in libcbm_hip.so; user laws are
// compiled around it with hipRTC.
template <int D, int NB, class Law, int PER, int NOISE, class Noise = ConstNoise>
__device__ __forceinline__ void stage_body(const StageArgs& a) {
  if (a.gate && *a.gate != a.gate_run) return;
  if (NB == NB_CELL) {
    // cell-linked: only blocks holding rows of bricks too dense for LDS
    if (a.sub_list && blockIdx.x == 0 && threadIdx.x == 0) *a.sub_n = 0;   // the sub-brick launch is done
    const int b = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    if (!a.blk_flag[b]) return;
    __syncthreads();
    if (threadIdx.x == 0) a.blk_flag[b] = 0;
  }
  const RowIdx ri = row_index(a.g);
  const SimDev& sd = a.g.sims[ri.sim];
  const int64_t N = a.g.st[ri.sim].N;
  const int64_t i = ri.row;
  // cell-linked: the brick kernel has done every row of a brick that fit in
  // LDS; the others are marked, and the mark is cleared here
  if (NB == NB_CELL) {
    if (ri.local >= sd.n_max || !a.brick_skip[i]) return;
    a.brick_skip[i] = 0;
  }
  if (ri.local >= N) return;

  double xi[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < D; ++c) xi[c] = a.S[c][i];
  double acc[3] = {0.0, 0.0, 0.0};
  if (Law::active) gather_global<D, NB, Law, PER>(a, sd, N, i, xi, acc);
  stage_finish<D, Law, NOISE, false, Noise>(a, sd, ri.sim, i, xi, acc, xi);
}

// One integrator stage of the rod model for every agent row: the contact
// sums over the neighbor candidates in reference loop order (pairs out of
// contact add exactly nothing: the reference adds +0 to sums that start at
// +0), then the stage update.  2-D, no periodic box.
//
// A pair costs some 400 instructions (the closest points, sin and cos) and a
// rod has tens of candidates, few of them contacts, so a lane per rod left
// the chip to a few hundred wavefronts in long series.  G lanes share a rod:
// they take G consecutive candidates at once, and the terms of those in
// contact are added one after the other in candidate order by every lane.
// Setting up and finishing a rod by one lane of G costs what the shorter
// series saves where wavefronts abound, so there is no other form.  20,011
// rods of 45 candidates each: 161 us per stage with a lane per rod, 37 us now;
// steps of 200,003 (Heun) and 1,000,003 (Euler) rods 0.90 and 2.8 ms, now 0.66
// and 2.7.
template <int NB> struct rod_lanes { static constexpr int value = NB == NB_LIST ? 8 : 16; };   // lists are shorter

template <int NB>
__device__ __forceinline__ void rod_stage_body(const StageArgs& a) {
  constexpr int G = rod_lanes<NB>::value;
  __shared__ int32_t cell_s[NB == NB_CELL ? BRICK_MAX_BLOCK / G : 1][9];       // first row of the rod's neighbor cells
  __shared__ int32_t cell_e[NB == NB_CELL ? BRICK_MAX_BLOCK / G : 1][9];       // and the candidates up to their ends
  const int tid = threadIdx.x, lane = tid & 63, sub = lane & (G - 1), grp = tid / G;
  // G consecutive blocks serve the rows of one block of the row geometry
  const int tile = xcd_tile((int)blockIdx.x, (int)gridDim.x);
  const int sim = a.g.block_sim[tile / G];
  const SimDev& sd = a.g.sims[sim];
  const int64_t N = a.g.st[sim].N;
  const int64_t local = (int64_t)(tile / G - a.g.block_off[sim]) * blockDim.x + (tile % G) * (int)(blockDim.x / G) + grp;
  const int64_t i = sd.row_off + local;
  const bool row = local < N;
  int32_t total = 0;
  if (NB == NB_CELL) {
    if (row && sub < 9) {
      const int32_t c = a.cell_row[i];
      const int32_t nc = neigh_cell<2>(sd, c % sd.gn[0], c / sd.gn[0], 0, sub, a.periodic);
      const CellRange r = nc < 0 ? CellRange{0, 0} : a.cell_range[sd.rank_off + nc];
      cell_s[grp][sub] = r.s;
      cell_e[grp][sub] = r.e - r.s;
    }
    __syncthreads();
    if (row && sub == 0) {
      int32_t run = 0;
      for (int k = 0; k < 9; ++k) { run += cell_e[grp][k]; cell_e[grp][k] = run; }
    }
    __syncthreads();
    if (row) total = cell_e[grp][8];
  } else if (row) {
    total = NB == NB_LIST ? a.list_n[i] : (int32_t)N;
  }
  if (!row) return;
  const double kn = sd.p[0], gn = sd.p[1], gt = sd.p[2], mucc = sd.p[3];
  const double* __restrict__ lcol = a.nvar == 7 ? a.S[6] : a.rod_l;   // l is a DE variable with growth
  auto rod_at = [&](int64_t j) {
    RodState r;
    r.a.x = a.S[0][j];
    r.a.y = a.S[1][j];
    r.vx = a.S[2][j];
    r.vy = a.S[3][j];
    sincos(a.S[4][j], &r.a.s, &r.a.c);
    r.a.l = lcol[j];
    r.d = a.rod_d[j];
    r.m = a.mass[j];
    return r;
  };
  const RodState me = rod_at(i);
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  bool domain = false;
  int cell = 0;
  for (int32_t c0 = 0; c0 < total; c0 += G) {
    const int32_t c = c0 + sub;
    int64_t j = i;
    if (c < total) {
      if (NB == NB_LIST) j = a.list[(int64_t)c * a.ldl + i];
      else if (NB == NB_FULL) j = sd.row_off + c;
      else {
        while (c >= cell_e[grp][cell]) ++cell;
        j = (int64_t)cell_s[grp][cell] + (c - (cell ? cell_e[grp][cell - 1] : 0));
      }
    }
    double f[4] = {0.0, 0.0, 0.0, 0.0};
    bool touch = false;
    if (j != i) {
      const RodState other = rod_at(j);
      touch = rod_force(me, other, kn, gn, gt, mucc, f[0], f[1], f[2], domain);
      f[3] = sqrt(f[0] * f[0] + f[1] * f[1]);
    }
    uint32_t bits = (uint32_t)(__ballot(touch) >> (lane & (64 - G))) & ((1u << G) - 1u);
    while (bits) {
      const int from = (lane & (64 - G)) + __ffs(bits) - 1;
      bits &= bits - 1u;
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] = acc[k] + __shfl(f[k], from, 64);
    }
  }
  if (domain) *a.rod_err = 1;
  if (sub != 0) return;
  double xi[3] = {me.a.x, me.a.y, 0.0};
  stage_finish<2, RodLaw, 0>(a, sd, sim, i, xi, acc, xi);
}

// One integrator stage of a general agentODE body (UserLaw::ode) for every agent
// row: the body's neighbor sums over the candidates in reference loop order
// (Full, the cell-linked walk or the Verlet list), then its equations.
template <int D, int NB, class Law, int PER, int NOISE, class Noise>
__device__ __forceinline__ void pair_stage_body(const StageArgs& a) {
  const RowIdx ri = row_index(a.g);
  const SimDev& sd = a.g.sims[ri.sim];
  const int64_t N = a.g.st[ri.sim].N;
  const int64_t i = ri.row;
  if (ri.local >= N) return;
  double xi[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < D; ++c) xi[c] = a.S[c][i];
  const LawAgent me = law_agent<D>(a, i, xi);
  constexpr int K = law_sums<Law>::value;
  static_assert(K >= 1 && K <= 8, "UserLaw::sums is 1..8");
  double s[K];
#pragma unroll
  for (int k = 0; k < K; ++k) s[k] = 0.0;
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  const Law law(sd.p);
  for_candidates<D, NB>(a, sd, N, i, [&](int64_t j) {
    double xj[3] = {0.0, 0.0, 0.0}, dx[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < D; ++c) {
      xj[c] = a.S[c][j];
      dx[c] = xi[c] - xj[c];
      if (PER) dx[c] = wrap_dx(dx[c], L[c], hL[c]);
    }
    double s2 = dx[0] * dx[0];
    if (D > 1) s2 = s2 + dx[1] * dx[1];
    if (D > 2) s2 = s2 + dx[2] * dx[2];
    const LawAgent nb = law_agent<D>(a, j, xj);
    law.pair(me, nb, dx, sqrt(s2), s);
  });
  stage_finish<D, Law, NOISE, false, Noise>(a, sd, ri.sim, i, xi, s, xi);
}

// The stage and brick kernels of a hipRTC module: a general agentODE body
// walks its candidates row by row (no brick tiles: its brick kernel returns
// at once and the row kernel takes every row); a pair law takes the
// built-in skeletons.
template <int D, int NB, class Law, int PER, int NOISE, class Noise>
__device__ __forceinline__ void user_stage(const StageArgs& a) {
  if constexpr (general_body<Law>::value) pair_stage_body<D, NB, Law, PER, NOISE, Noise>(a);
  else stage_body<D, NB, Law, PER, NOISE, Noise>(a);
}

// ------------------------------------------------ flattened list stage
// Exclusive block scan of one int32 per thread; the total lands in *total.
__device__ __forceinline__ int32_t block_excl_scan(int32_t v, int32_t* wsum, int32_t* total) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = (blockDim.x + 63) >> 6;
  int32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t y = __shfl_up(incl, off, 64);
    if (lane >= off) incl += y;
  }
  if (lane == 63 || tid == (int)blockDim.x - 1) wsum[w] = incl;
  __syncthreads();
  int32_t before = 0, tot = 0;
  for (int q = 0; q < nw; ++q) {
    const int32_t ws = wsum[q];
    if (q < w) before += ws;
    tot += ws;
  }
  if (tid == 0) *total = tot;
  return before + incl - v;
}

// ------------------------------------------------ cell-linked brick tiles
// The cell-linked stage on LDS tiles.  Block b serves one brick of
// bdim[0] x bdim[1] x bdim[2] grid cells, a Morton-aligned block (its edges
// are powers of two with x >= y >= z >= x/2), so that the rows of its cells
// are one contiguous range.  The agents of the brick and of its one-cell
// halo are staged in LDS in halo-cell order (x fastest): the three
// x-adjacent cells of a neighbor column are then one contiguous LDS run, and
// each home agent walks its 3^D cells there in the reference order
// (cellPosNeigh, x fastest; the rows of a cell by slot).  A brick whose halo
// holds more than brick_cap agents marks its rows in brick_skip and leaves
// them to the row-parallel stage kernel launched after it, which walks
// global memory in the same order, so the result does not depend on the
// path.

// Reach of a built-in law: a pair can be active only when d < reach (all of
// them also need d > 0).  Laws without it are not filtered; user bodies never
// are, whatever members they have.
template <class L> struct has_reach { static constexpr bool value = false; };
template <> struct has_reach<PairLaw<LAW_LINEAR>> { static constexpr bool value = true; };
template <> struct has_reach<PairLaw<LAW_REP_ADH>> { static constexpr bool value = true; };
template <> struct has_reach<PairLaw<LAW_AGGREGATION>> { static constexpr bool value = true; };

// A bound on d^2 that keeps every pair with d = sqrt(d2) < reach: sqrt is
// correctly rounded, so d < reach implies d2 < reach^2 (1 + 2^-51), and the
// product below exceeds that.  A NaN or infinite reach keeps every pair.
__device__ __forceinline__ double reach2_bound(double reach) {
  const double r2 = (reach * reach) * (1.0 + 0x1p-44);
  return (r2 == r2) ? r2 : __builtin_inf();
}

// Order-preserving int64 key of a double (for LDS atomicMax).
__device__ __forceinline__ long long order_key(double x) {
  const long long b = __double_as_longlong(x);
  return b < 0 ? (long long)(~(unsigned long long)b | 0x8000000000000000ull) : b;
}
__device__ __forceinline__ double order_val(long long k) {
  return __longlong_as_double(k < 0 ? (long long)(~(unsigned long long)k | 0x8000000000000000ull) : k);
}


// One brick's LDS tile.  The caller points hdr, hs, hrow, owner and home_li
// into its LDS; brick_stage fills the rest.
struct BrickTile {
  int sim;
  int32_t o[3];                   // origin cell
  int B[3], HX, HY, H;            // brick edge, halo extent, halo cells
  int32_t r0, r1, T;              // home rows [r0, r1); staged agents
  int32_t* hdr;                   // BRICK_HDR int32 words of scratch
  int32_t* hs;                    // LDS offset of halo cell h's agents, hs[H] = T
  int32_t* hrow;                  // first global row of halo cell h
  uint16_t* owner;                // halo cell of each staged agent, | 0x8000 at its home cell
  uint16_t* home_li;              // LDS index of home row r0 + k
};

// What brick_stage copies per agent besides the positions: an optional
// double column (radius; its block maximum is returned, +inf if any is NaN)
// and an optional integer column read as int64 (fate) or int32 (slot).
enum { BX_NONE = 0, BX_I64 = 1, BX_I32 = 2 };
struct BrickCols {
  const double* S[3];       // positions, S[c][row]
  double* pos[3];           // their LDS arrays
  const double* xd;         // double column (or NULL)
  double* xd_lds;
  const void* xi;           // integer column
  int32_t* xi_lds;
  const int32_t* map;       // MAP: the row at each place of the cell order (rows that stay in place)
};

// Stages brick b: the rows and counts of its halo cells (wrapped on a
// periodic grid, empty outside a bounded one), their exclusive scan, then
// the columns of every halo agent, U4 agents per thread in flight, at its
// LDS index q (halo-cell order, x fastest).  Returns 0 for an empty brick, 2
// for one whose halo exceeds cap (its rows are then marked for the
// row-parallel kernel), 1 when staged.
template <int D, int PER, int U4, bool XD, int XI, bool MAP = false>
__device__ __forceinline__ int brick_stage(const BrickSrc& src, int b, BrickTile& t, const BrickCols& cols,
                                           double& xd_max) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int32_t* bt = src.brick + BRICK_WORDS * (int64_t)b;
  t.sim = bt[0];
  t.o[0] = bt[1]; t.o[1] = bt[2]; t.o[2] = bt[3];
  const SimDev& sd = src.sims[t.sim];
  // the brick's cells hold consecutive buckets [b0, b1): its rows are one range
  t.r0 = src.bucket_start[bt[4]];
  t.r1 = src.bucket_start[bt[5]];
  if (t.r0 >= t.r1) return 0;
  t.B[0] = src.bdim[0]; t.B[1] = D > 1 ? src.bdim[1] : 1; t.B[2] = D > 2 ? src.bdim[2] : 1;
  t.HX = t.B[0] + 2;
  t.HY = D > 1 ? t.B[1] + 2 : 1;
  t.H = brick_halo_cells(D, t.B[0], t.B[1], t.B[2]);
  const int HX = t.HX, HY = t.HY, H = t.H;
  int32_t* hs = t.hs;
  int32_t* hrow = t.hrow;
  const CellRange* __restrict__ cr = src.cell_range + sd.rank_off;

  // halo cell h -> (hx, hy, hz), x fastest.  h + 0.5 lies at least 0.5 from
  // a multiple of the divisor, far beyond the float product's rounding for
  // h < 2^16, so the truncated products are the exact quotients.
  const float rHX = 1.0f / (float)HX, rHXY = 1.0f / (float)(HX * HY);
  auto halo_cell = [&](int h, bool& home) {
    const int hz = (int)(((float)h + 0.5f) * rHXY);
    const int rem = h - hz * HX * HY;
    const int hy = (int)(((float)rem + 0.5f) * rHX);
    const int hh[3] = {rem - hy * HX, hy, hz};
    bool ok = true;
    home = true;
    int32_t q[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < D; ++e) {
      int32_t v = t.o[e] + hh[e] - 1;
      home = home && hh[e] >= 1 && hh[e] <= t.B[e] && v < sd.gn[e];
      if (PER) {
        if (v == -1) v = sd.gn[e] - 1;
        else if (v == sd.gn[e]) v = 0;
        else if (v > sd.gn[e]) ok = false;
      } else {
        ok = ok && v >= 0 && v < sd.gn[e];
      }
      q[e] = v;
    }
    return ok ? q[0] + sd.gn[0] * (q[1] + sd.gn[1] * q[2]) : -1;
  };
  // 1. rows and counts of the halo cells, U4 cells per thread in flight
  for (int h0 = tid; h0 < H; h0 += U4 * nt) {
    CellRange r[U4];
#pragma unroll
    for (int u = 0; u < U4; ++u) {
      bool home;
      const int h = h0 + u * nt;
      const int32_t lin = h < H ? halo_cell(h, home) : -1;
      r[u] = lin >= 0 ? cr[lin] : CellRange{0, 0};
    }
#pragma unroll
    for (int u = 0; u < U4; ++u) {
      const int h = h0 + u * nt;
      if (h < H) { hs[h] = r[u].e - r[u].s; hrow[h] = r[u].s; }
    }
  }
  __syncthreads();

  // 2. exclusive scan of the halo counts (a contiguous chunk per thread)
  {
    const int K = (H + nt - 1) / nt;
    const int c0 = min(tid * K, H), c1 = min(c0 + K, H);
    int32_t sum = 0;
    for (int h = c0; h < c1; ++h) sum += hs[h];
    const int lane = tid & 63, w = tid >> 6, nw = (nt + 63) >> 6;
    int32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(incl, off, 64);
      if (lane >= off) incl += y;
    }
    if (lane == 63) t.hdr[4 + w] = incl;
    __syncthreads();
    int32_t run = incl - sum, tot = 0;
    for (int q = 0; q < nw; ++q) {
      const int32_t ws = t.hdr[4 + q];
      if (q < w) run += ws;
      tot += ws;
    }
    for (int h = c0; h < c1; ++h) { const int32_t v = hs[h]; hs[h] = run; run += v; }
    if (tid == 0) { hs[H] = tot; t.hdr[2] = tot; }
  }
  __syncthreads();
  t.T = t.hdr[2];
  const int32_t r0 = t.r0, r1 = t.r1;
  if (t.T > src.cap) {
    // too dense for LDS: the row-parallel kernel launched after this one
    // takes the brick's rows
    if (tid == 0 && !src.sub) atomicAdd(src.brick_over, 1ull);
    if (MAP) {
      for (int64_t i = (int64_t)r0 + tid; i < (int64_t)r1; i += nt) {
        const int64_t r = cols.map[i];
        src.brick_skip[r] = 1;
        src.blk_flag[src.block_off[t.sim] + (r - sd.row_off) / nt] = 1;
      }
      return 2;
    }
    for (int64_t i = (int64_t)r0 + tid; i < (int64_t)r1; i += nt) src.brick_skip[i] = 1;
    // wake the row-kernel blocks holding these rows (same block size)
    const int64_t q0 = src.block_off[t.sim] + ((int64_t)r0 - sd.row_off) / nt;
    const int64_t q1 = src.block_off[t.sim] + ((int64_t)r1 - 1 - sd.row_off) / nt;
    for (int64_t q = q0 + tid; q <= q1; q += nt) src.blk_flag[q] = 1;
    if (src.sub_list) {   // or, before it, the sub-brick launch
      const int32_t e = src.sub_first[b + 1];
      for (int32_t k0 = src.sub_first[b]; k0 < e; k0 += nt) {
        const int32_t k = k0 + tid;
        const int32_t id = k < e ? src.sub_ids[k] : 0;
        const int32_t* sb = src.sub_brick + BRICK_WORDS * (int64_t)id;
        const bool rows = k < e && src.bucket_start[sb[4]] < src.bucket_start[sb[5]];
        const unsigned long long m = __ballot(rows);     // one atomic per wavefront
        int32_t at = 0;
        if (rows && (m & ((1ull << (tid & 63)) - 1ull)) == 0ull) at = atomicAdd(src.sub_n, (int32_t)__popcll(m));
        at = __shfl(at, m ? __ffsll(m) - 1 : 0, 64);
        if (rows) src.sub_list[at + __popcll(m & ((1ull << (tid & 63)) - 1ull))] = id;
      }
    }
    return 2;
  }

  // 3. stage the halo agents; each home row notes the LDS index of its copy
  //    at its home cell
  for (int h = tid; h < H; h += nt) {
    bool home;
    (void)halo_cell(h, home);
    const uint16_t tag = (uint16_t)(h | (home ? 0x8000 : 0));
    for (int32_t q = hs[h]; q < hs[h + 1]; ++q) t.owner[q] = tag;
  }
  __syncthreads();
  const int32_t T = t.T;
  double xm = -__builtin_inf();
  bool xnan = false;
  for (int32_t q0 = tid; q0 < T; q0 += U4 * nt) {
    int64_t row[U4];
    int tag[U4];
    double v[U4][3], vd[U4];
    int32_t vi[U4];
#pragma unroll
    for (int u = 0; u < U4; ++u) {
      const int32_t q = q0 + u * nt;
      tag[u] = q < T ? t.owner[q] : 0;
      const int h = tag[u] & 0x7FFF;
      row[u] = q < T ? (int64_t)hrow[h] + (q - hs[h]) : -1;
      int64_t rr = row[u] < 0 ? (int64_t)r0 : row[u];
      if (MAP) rr = cols.map[rr];
#pragma unroll
      for (int c = 0; c < D; ++c) v[u][c] = cols.S[c][rr];
      if (XD) vd[u] = cols.xd[rr];
      if (XI == BX_I64) vi[u] = (int32_t)((const int64_t*)cols.xi)[rr];
      if (XI == BX_I32) vi[u] = ((const int32_t*)cols.xi)[rr];
    }
#pragma unroll
    for (int u = 0; u < U4; ++u) {
      const int32_t q = q0 + u * nt;
      if (q >= T) continue;
#pragma unroll
      for (int c = 0; c < D; ++c) cols.pos[c][q] = v[u][c];
      if (XD) {
        cols.xd_lds[q] = vd[u];
        xm = vd[u] > xm ? vd[u] : xm;
        xnan = xnan || vd[u] != vd[u];
      }
      if (XI != BX_NONE) cols.xi_lds[q] = vi[u];
      if (tag[u] & 0x8000) t.home_li[row[u] - r0] = (uint16_t)q;
    }
  }
  if (XD) {
    // block maximum of the double column through an order-preserving key
    long long* key = (long long*)(t.hdr + 12);
    if (tid == 0) *key = order_key(-__builtin_inf());
    __syncthreads();
    atomicMax(key, xnan ? order_key(__builtin_inf()) : order_key(xm));
  }
  __syncthreads();
  if (XD) xd_max = order_val(*(const long long*)(t.hdr + 12));
  return 1;
}

// Candidates of a home agent in halo cell h: its 3^(D-1) runs of three
// x-adjacent cells (z outer, then y); run (ry, rz) covers cells hb .. hb + 2.
template <int D>
__device__ __forceinline__ int brick_run0(const BrickTile& t, int h) {
  return h - 1 - (D > 1 ? t.HX : 0) - (D > 2 ? t.HX * t.HY : 0);
}
template <int D>
__device__ __forceinline__ int32_t brick_ncand(const BrickTile& t, int h) {
  const int hb0 = brick_run0<D>(t, h);
  int32_t n = 0;
#pragma unroll
  for (int rz = 0; rz < (D > 2 ? 3 : 1); ++rz)
#pragma unroll
    for (int ry = 0; ry < (D > 1 ? 3 : 1); ++ry) {
      const int hb = hb0 + rz * t.HX * t.HY + ry * t.HX;
      n += t.hs[hb + 3] - t.hs[hb];
    }
  return n;
}
// Visits the candidates of a home agent in halo cell h in walk order, as one
// flattened sequence, so the lanes of a wavefront stay in step.
template <int D, class Visit>
__device__ __forceinline__ void brick_walk(const BrickTile& t, int h, Visit&& visit) {
  const int32_t ncand = brick_ncand<D>(t, h);
  int ry = 0;
  int hb = brick_run0<D>(t, h);
  int32_t q = t.hs[hb], qe = t.hs[hb + 3];
  for (int32_t k = 0; k < ncand; ++k) {
    while (q == qe) {   // the next non-empty run; one exists while k < ncand
      if (++ry == 3) { ry = 0; hb += t.HX * t.HY - 2 * t.HX; } else { hb += t.HX; }
      q = t.hs[hb];
      qe = t.hs[hb + 3];
    }
    visit(q);
    ++q;
  }
}

// The value of lane G of this lane's quad (four consecutive lanes, all active).
template <int G>
__device__ __forceinline__ double quad_lane(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), G * 0x55, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), G * 0x55, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// The candidates of a home agent in halo cell h in walk order, G at a time:
// lane sub of the agent's G lanes gets candidate k + sub of each round (not
// live past the last one).
template <int D, int G>
struct BrickWalk {
  int32_t ncand, k, q, qe;
  int ry, hb;
  __device__ __forceinline__ BrickWalk(const BrickTile& t, int h, int sub)
      : ncand(brick_ncand<D>(t, h)), k(0), ry(0), hb(brick_run0<D>(t, h)) {
    q = t.hs[hb] + sub;
    qe = t.hs[hb + 3];
  }
  __device__ __forceinline__ bool more() const { return k < ncand; }
  __device__ __forceinline__ int32_t next(const BrickTile& t, int sub, bool& live) {
    live = G == 1 || k + sub < ncand;
    if (live)
      while (q >= qe) {   // into the run that holds this candidate; there is one
        const int32_t past = q - qe;
        if (++ry == 3) { ry = 0; hb += t.HX * t.HY - 2 * t.HX; } else { hb += t.HX; }
        q = t.hs[hb] + past;
        qe = t.hs[hb + 3];
      }
    const int32_t at = live ? q : 0;
    q += G;
    k += G;
    return at;
  }
};

// The cell-linked stage of a brick.  Built-in laws filter the candidates: a
// cheap test queues the LDS indices of the pairs within the law's reach (in
// walk order), and the full pair body runs on those only.  Every pair left
// out is inactive, so the sum is unchanged.
//
// BRICK_ONE: a lane per agent walks once, and walks again for what its queue
// did not hold.  That is the shortest code for the usual handful of agents in
// reach (rep_adh in space, 4 of 27: 300,001 agents in a periodic box, RK4,
// 50 steps 16.6 ms, with the queue drained as it fills 17.3), but where the
// queue overflows in every wavefront the second walk costs as much as the
// first (50 in reach, 100,001 agents: 6.3 ms against 4.9).
//
// BRICK_DRAIN: a lane per agent; the queue is drained and refilled, so cells of
// any density are tested once.
//
// BRICK_FOUR: four lanes share an agent: they test four consecutive candidates
// at once and evaluate four queued pairs at once, whose terms the first lane
// adds in order (DPP moves), so the sums keep the reference's order.  A
// wavefront waits for the longest walk of 16 agents and not of 64, bricks of
// fewer agents than lanes keep the lanes busy, and neighboring lanes read
// neighboring LDS words; the moves and shared adds cost instructions.  The
// queue is drained as it fills (soft spheres, 15 of 132 candidates near
// enough: 172 us per stage for 120,001 of them with one lane and a second walk
// with the full body, 81 us so).
//
// setup_bricks says which bricks take which.
template <int D, class Law, int PER, int NOISE, int FORM, bool SUB, class Noise>
__device__ __forceinline__ void brick_one(const StageArgs& a, unsigned char* lds, int b) {
  constexpr int G = brick_lanes(FORM);
  constexpr bool SOFT = same_type<Law, PairLaw<LAW_SOFT_SPHERES>>::value;
  // on sub-bricks in the plane every candidate takes the pair body: a third
  // of them is in reach, and the filter costs as much as it saves
  constexpr bool FILTER = (SOFT || has_reach<Law>::value) && !(SUB && D < 3);
  constexpr int U4 = 4;               // loads issued together per thread while staging
  // stage-2 lists (built-in laws without per-agent radii)
  constexpr bool WL = FILTER && !SOFT;
  const bool wl = WL && a.wlist != nullptr;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int cap = a.brick_cap;
  BrickSrc src;
  src.sims = a.g.sims; src.block_off = a.g.block_off; src.brick = a.brick; src.bucket_start = a.bucket_start;
  src.cell_range = a.cell_range; src.cap = cap;
  for (int e = 0; e < 3; ++e) src.bdim[e] = a.bdim[e];
  src.brick_skip = a.brick_skip; src.blk_flag = a.blk_flag; src.brick_over = a.brick_over;
  src.sub = SUB ? 1 : 0;
  src.sub_first = a.sub_first; src.sub_ids = a.sub_ids; src.sub_brick = a.brick2;
  src.sub_list = SUB ? nullptr : a.sub_list; src.sub_n = a.sub_n;
  const int H = brick_halo_cells(D, a.bdim[0], D > 1 ? a.bdim[1] : 1, D > 2 ? a.bdim[2] : 1);

  BrickTile t;
  t.hdr = (int32_t*)lds;
  double* pos[3];
  unsigned char* p = lds + 4 * BRICK_HDR;
#pragma unroll
  for (int c = 0; c < D; ++c) { pos[c] = (double*)p; p += (size_t)8 * cap; }
  double* rad = (double*)p;
  if (SOFT) p += (size_t)8 * cap;
  int32_t* fate = (int32_t*)p;
  if (SOFT) p += (size_t)4 * cap;
  t.hs = (int32_t*)p;
  p += (size_t)4 * (H + 1);
  t.hrow = (int32_t*)p;
  p += (size_t)4 * H;
  uint16_t* lst = (uint16_t*)p;       // the agents' queues of kept candidates
  if (FILTER) p += (size_t)2 * brick_queue(FORM) * (BRICK_MAX_BLOCK / G);
  t.owner = (uint16_t*)p;
  p += (size_t)2 * cap;
  t.home_li = (uint16_t*)p;

  // staged columns: positions (and radius and fate for soft spheres)
  BrickCols cols;
#pragma unroll
  for (int c = 0; c < 3; ++c) { cols.S[c] = a.S[c]; cols.pos[c] = pos[c]; }
  cols.xd = a.rad;
  cols.xd_lds = rad;
  cols.xi = a.fate;
  cols.xi_lds = fate;
  double rmax = 0.0;
  const int staged = brick_stage<D, PER, U4, SOFT, SOFT ? BX_I64 : BX_NONE>(src, b, t, cols, rmax);
  if (staged == 2 && wl && tid == 0) *a.lgate = 0;   // its rows get no list
  if (staged != 1) return;
  const int sim = t.sim;
  const SimDev& sd = a.g.sims[sim];
  const int64_t N = a.g.st[sim].N;
  const int32_t* hs = t.hs;
  const int32_t* hrow = t.hrow;
  const uint16_t* owner = t.owner;
  const uint16_t* home_li = t.home_li;

  // 4. the home agents
  const int32_t nh = t.r1 - t.r0;
  const Law law(sd.p);
  const uint32_t span = law_span(law);
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  double reach2 = __builtin_inf();
  double disp2 = -1.0;
  if constexpr (FILTER && !SOFT) {
    reach2 = reach2_bound(law.reach());
    if (wl) {
      // lists to CL_LIST_GROW x reach: valid while displacements stay under
      // half the margin (with a little slack for rounding)
      reach2 = reach2_bound(law.reach() * CL_LIST_GROW);
      const double half = 0.5 * (CL_LIST_GROW - 1.0) * law.reach() * (1.0 - 1e-9);
      disp2 = half > 0.0 ? half * half : 0.0;
    }
  }
  auto row_of = [&](int32_t q) {
    const int hq = owner[q] & 0x7FFF;
    return (int64_t)hrow[hq] + (q - hs[hq]);
  };
  // Each wavefront takes consecutive home agents, 64 at most: it walks them
  // 16 at a time, four lanes per agent, and then finishes the stage of all of
  // them with one agent per lane.  `own` is this lane's agent of the finish.
  const int lane = tid & 63, sub = lane & (G - 1), wv = tid >> 6, nw = nt >> 6;
  for (int32_t k0 = 0; k0 < nh; k0 += nt) {
    const int32_t m = nh - k0 < nt ? nh - k0 : nt;
    // agents per wavefront: whole rounds of 64 / G
    const int32_t npw = ((m + nw - 1) / nw + 64 / G - 1) & ~(64 / G - 1);
    const int32_t w0 = k0 + wv * npw;
    const int32_t w1 = w0 + npw < k0 + m ? w0 + npw : k0 + m;
    const int32_t own = w0 + lane;
    int64_t i = -1;
    int32_t own_li = 0;
    double upre[3] = {0.0, 0.0, 0.0}, acc[3] = {0.0, 0.0, 0.0};
    if (own < w1) {
      own_li = home_li[own];
      i = row_of(own_li);
      if (SUB) a.brick_skip[i] = 0;   // done here, not by the row kernel
      if (i - sd.row_off >= N) i = -1;
    }
    if (i >= 0) {
#pragma unroll
      for (int c = 0; c < D; ++c) upre[c] = a.U[c][i];   // consumed after the walk
    }
    for (int32_t g0 = w0; g0 < w1; g0 += 64 / G) {
      const int32_t k = g0 + lane / G;
      double sum[3] = {0.0, 0.0, 0.0};
      if (k < w1) {
        const int32_t li = home_li[k];
        const int h = owner[li] & 0x7FFF;
        const int64_t row = row_of(li);
        double xi[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < D; ++c) xi[c] = pos[c][li];
        const double rad_i = SOFT ? rad[li] : 0.0;
        const int64_t fate_i = SOFT ? fate[li] : 0;
        double keep2 = reach2;
        if constexpr (SOFT) keep2 = law.mu >= 0.0 ? reach2_bound(law.mu * (rad_i + rmax)) : __builtin_inf();
        // G candidates' terms (this lane's is q's, nothing unless live) added
        // to the agent's sum, in their order, by its first lane
        auto add = [&](int32_t q, bool live) {
          double xj[3] = {0.0, 0.0, 0.0}, t[3];
#pragma unroll
          for (int c = 0; c < D; ++c) xj[c] = pos[c][q];
          pair_term<D, Law, PER, SOFT>(law, span, xi, xj, L, hL, live, t, rad_i, SOFT ? rad[q] : 0.0, fate_i,
                                       SOFT ? (int64_t)fate[q] : 0);
#pragma unroll
          for (int c = 0; c < D; ++c) {
            // a lane past the last candidate adds +0, whatever it read (0 times
            // the offset of an agent that ran off to infinity is NaN)
            const double v = live ? t[c] : 0.0;
            sum[c] = sum[c] + v;
            if constexpr (G == 4) {
              sum[c] = sum[c] + quad_lane<1>(v);
              sum[c] = sum[c] + quad_lane<2>(v);
              sum[c] = sum[c] + quad_lane<3>(v);
            }
          }
        };
        if constexpr (FILTER) {
          auto near = [&](int32_t q) {
            double dx[3];
#pragma unroll
            for (int c = 0; c < D; ++c) {
              dx[c] = xi[c] - pos[c][q];
              if (PER) dx[c] = wrap_dx(dx[c], L[c], hL[c]);
            }
            double s2 = dx[0] * dx[0];
            if (D > 1) s2 = s2 + dx[1] * dx[1];
            if (D > 2) s2 = s2 + dx[2] * dx[2];
            return s2 <= keep2 && q != li;
          };
          const int ng = nt / G;
          uint16_t* que = lst + (tid / G);      // entry u at que[u * ng]
          int32_t cnt = 0;
          auto keep = [&](int32_t u, int32_t q) {      // candidate u as an entry of the stage-2 list
            if (wl && u < a.wcap) a.wlist[(int64_t)u * a.ldl + row] = (int32_t)row_of(q);
          };
          if constexpr (FORM == BRICK_ONE) {
            // one walk fills the queue, and only a lane whose queue was too
            // short walks again for the candidates past it
            brick_walk<D>(t, h, [&](int32_t q) {
              if (near(q)) {
                if (cnt < brick_queue(FORM)) que[cnt * ng] = (uint16_t)q;
                ++cnt;
              }
            });
            const int32_t nq = cnt < brick_queue(FORM) ? cnt : brick_queue(FORM);
            for (int32_t u = 0; u < nq; ++u) {
              const int32_t q = que[u * ng];
              add(q, true);
              keep(u, q);
            }
            if (cnt > nq) {
              int32_t u = 0;
              brick_walk<D>(t, h, [&](int32_t q) {
                if (!near(q)) return;
                if (u >= nq) { add(q, true); keep(u, q); }
                ++u;
              });
            }
          } else {
            // the LDS indices of the agent's candidates within reach, in walk
            // order, in its queue; a full queue is drained: the pair bodies of
            // its entries, and their rows as the stage-2 list
            BrickWalk<D, G> w(t, h, sub);
            for (;;) {
              int32_t nq = 0;
              if constexpr (G == 1) {
                // room for four more between the looks at the queues
                while (w.more()) {
                  for (int e = 0; e < 4 && w.more(); ++e) {
                    bool live;
                    const int32_t q = w.next(t, sub, live);
                    if (near(q)) que[nq++ * ng] = (uint16_t)q;
                  }
                  if (__any(nq > brick_queue(FORM) - 4)) break;
                }
              } else {
                while (w.more()) {
                  bool live;
                  const int32_t q = w.next(t, sub, live);
                  const bool in = live && near(q);
                  const uint32_t bits = (uint32_t)(__ballot(in) >> (lane & (64 - G))) & ((1u << G) - 1u);
                  if (in) que[(nq + __popc(bits & ((1u << sub) - 1u))) * ng] = (uint16_t)q;
                  nq += __popc(bits);
                  if (__any(nq > brick_queue(FORM) - G)) break;
                }
              }
              __builtin_amdgcn_wave_barrier();   // the agent's other lanes wrote most entries
              for (int32_t u = sub; u - sub < nq; u += G) {
                const bool live = u < nq;
                const int32_t q = live ? que[u * ng] : li;
                add(q, live);
                if (live) keep(cnt + u, q);
              }
              cnt += nq;
              if (!w.more()) break;
            }
          }
          if (wl && sub == 0 && row - sd.row_off < N) {
            a.wlist_n[row] = cnt < a.wcap ? cnt : a.wcap;
            if (cnt > a.wcap) *a.lgate = 0;
          }
        } else if constexpr (G == 1) {
          brick_walk<D>(t, h, [&](int32_t q) { if (q != li) add(q, true); });
        } else {
          // a lane past the last candidate takes the agent itself: a user's law
          // is called with distances of candidates and 0 alone
          BrickWalk<D, G> w(t, h, sub);
          while (w.more()) {
            bool live;
            const int32_t q = w.next(t, sub, live);
            add(live ? q : li, live && q != li);
          }
        }
      }
      // agent k's sum to the lane that finishes it
#pragma unroll
      for (int c = 0; c < D; ++c) {
        if constexpr (G == 1) acc[c] = sum[c];
        else {
          const double v = __shfl(sum[c], ((lane - (g0 - w0)) & (64 / G - 1)) * G, 64);
          if (own >= g0 && own < g0 + 64 / G) acc[c] = v;
        }
      }
    }
    if (i >= 0) {
      double xi[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int c = 0; c < D; ++c) xi[c] = pos[c][own_li];
      stage_finish<D, Law, NOISE, true, Noise>(a, sd, sim, i, xi, acc, upre, disp2);
    }
  }
}

template <int D, class Law, int PER, int NOISE, int FORM, class Noise = ConstNoise>
__device__ __forceinline__ void brick_body(const StageArgs& a, unsigned char* lds) {
  if (a.gate && *a.gate != a.gate_run) return;
  brick_one<D, Law, PER, NOISE, FORM, false, Noise>(a, lds, xcd_tile((int)blockIdx.x, (int)gridDim.x));
}

// The sub-brick launch: the listed sub-bricks in turn.  A colony's core is a
// few of its many sub-bricks, and a block per sub-brick spent more on finding
// out that it had nothing to do than on the core (150,001 agents at 2 per unit
// area, 16,641 sub-bricks, 1,200 with agents: 104 us with a block for each,
// 67 us from the list).
template <int D, class Law, int PER, int NOISE>
__device__ __forceinline__ void sub_brick_body(const StageArgs& a, unsigned char* lds) {
  if (a.gate && *a.gate != a.gate_run) return;
  const int32_t n = *a.sub_n;
  for (int32_t k = blockIdx.x; k < n; k += gridDim.x) {
    brick_one<D, Law, PER, NOISE, BRICK_DRAIN, true, ConstNoise>(a, lds, a.sub_list[k]);
    __syncthreads();
  }
}

// The brick kernel of a hipRTC module: nothing for a general agentODE body
// (its row kernel walks every row).  The form is the context's; a user law
// has no reach, so every candidate takes its pair body and there is no queue,
// but in bricks cut small to fill the chip one lane per agent leaves most of
// a block idle (27,991 agents in the plane, Heun: 13.9 -> 11.9 ms for 200
// steps with four).
template <int D, class Law, int PER, int NOISE, class Noise, int FORM>
__device__ __forceinline__ void user_brick(const StageArgs& a, unsigned char* lds) {
  if constexpr (!general_body<Law>::value) brick_body<D, Law, PER, NOISE, FORM, Noise>(a, lds);
}

// An element at a 32-bit byte offset from a base that all lanes share (a
// kernel argument): the access takes the base from scalar registers and the
// offset from one vector register, with no 64-bit address arithmetic.
template <class T>
__device__ __forceinline__ T ld_b(const T* base, uint32_t off) {
  return *(const T*)((const char*)base + off);
}
template <class T>
__device__ __forceinline__ void st_b(T* base, uint32_t off, T v) {
  *(T*)((char*)base + off) = v;
}

// Batcher's odd-even merge sort of N keys held in registers (every index is
// a compile-time constant once the loops unroll).
template <int N, class T>
__device__ __forceinline__ void sort_net(T* k) {
#pragma unroll
  for (int p = 1; p < N; p <<= 1)
#pragma unroll
    for (int kk = p; kk >= 1; kk >>= 1)
#pragma unroll
      for (int j = kk % p; j + kk < N; j += 2 * kk)
#pragma unroll
        for (int i = 0; i < kk && i + j + kk < N; ++i)
          if ((i + j) / (2 * p) == (i + j + kk) / (2 * p)) {
            const T x = k[i + j], y = k[i + j + kk];
            k[i + j] = x < y ? x : y;
            k[i + j + kk] = x < y ? y : x;
          }
}

// ------------------------------------------ CellLinked on a skin list
// CellLinked (src/neighbors.jl:587-747) walks, for agent i, the 3^D cells
// around i's cell in cellPosNeigh order (x fastest) and each cell's agents by
// slot.  Its active pairs (d < the law's reach) therefore come in the order
// (k, slot j), k the position of j's cell among i's neighbor cells.  With a
// skin list (radius reach + skin, rebuilt when an agent has moved skin/2)
// holding every pair within reach, the step needs no cell sort: each agent's
// list entries are ordered by (k, slot) from the agents' packed cells of the
// step start.

// Every candidate j of row i in the reference's CellLinked order whose
// stage position lies within sqrt(bound2) of xi (fn(j, s2)), found without
// the skin list: repeated minimum selection of the key (k, slot) over the
// list-build grid cells within R of xi, where R bounds the distance of every
// such j's position at the last list build.  Exact for any displacement;
// used for the few agents whose list may miss a pair, and for exports.
template <int D, int PER, class Fn>
__device__ void clv_each(const StageArgs& a, const SimDev& sd, int64_t i, const double* xi, double bound2, double R,
                         Fn&& fn) {
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  const int32_t ci = a.ccell[i];
  int32_t c0[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
#pragma unroll
  for (int e = 0; e < D; ++e) {
    const double x = xi[e];
    int64_t c = x < sd.lo[e] ? 0 : floor_div(x - sd.lo[e], sd.gedge[e]) + (PER ? 0 : 1);
    c = c < 0 ? 0 : c;
    c0[e] = (int32_t)(c > sd.gn[e] - 1 ? sd.gn[e] - 1 : c);
    const double q = R / sd.gedge[e];
    const int32_t m = (q == q && q < (double)sd.gn[e]) ? (int32_t)ceil(q) : sd.gn[e];
    if (PER && 2 * m + 1 >= sd.gn[e]) { lo[e] = 0; hi[e] = sd.gn[e] - 1; c0[e] = 0; }
    else { lo[e] = -m; hi[e] = m; }
  }
  const CellRange* __restrict__ cr = a.cell_range + sd.rank_off;
  unsigned long long from = 0;
  for (;;) {
    unsigned long long best = ~0ull;
    int64_t bj = -1;
    double bs2 = 0.0;
    for (int32_t oz = D > 2 ? lo[2] : 0; oz <= (D > 2 ? hi[2] : 0); ++oz)
      for (int32_t oy = D > 1 ? lo[1] : 0; oy <= (D > 1 ? hi[1] : 0); ++oy)
        for (int32_t ox = lo[0]; ox <= hi[0]; ++ox) {
          const int32_t o[3] = {ox, oy, oz};
          int32_t q[3] = {0, 0, 0};
          bool ok = true;
#pragma unroll
          for (int e = 0; e < D; ++e) {
            int32_t v = c0[e] + o[e];
            if (PER) v = ((v % sd.gn[e]) + sd.gn[e]) % sd.gn[e];
            else ok = ok && v >= 0 && v < sd.gn[e];
            q[e] = v;
          }
          if (!ok) continue;
          const CellRange r = cr[q[0] + sd.gn[0] * (q[1] + sd.gn[1] * q[2])];
          for (int32_t j = r.s; j < r.e; ++j) {
            if (j == i) continue;
            const int k = cl_key<D, PER>(sd, ci, a.ccell[j]);
            if (k == 27) continue;
            double dx[3];
#pragma unroll
            for (int c = 0; c < D; ++c) {
              dx[c] = xi[c] - a.S[c][j];
              if (PER) dx[c] = wrap_dx(dx[c], L[c], hL[c]);
            }
            double s2 = dx[0] * dx[0];
            if (D > 1) s2 = s2 + dx[1] * dx[1];
            if (D > 2) s2 = s2 + dx[2] * dx[2];
            if (!(s2 <= bound2)) continue;
            const unsigned long long key = ((unsigned long long)k << 32) | (uint32_t)a.cslot[j];
            if (key >= from && key < best) { best = key; bj = j; bs2 = s2; }
          }
        }
    if (bj < 0) return;
    fn(bj, bs2);
    from = best + 1;
  }
}

// The pair sum of row i by clv_each within the law's reach.
template <int D, class Law, int PER>
__device__ void clv_walk(const StageArgs& a, const SimDev& sd, int64_t i, const double* xi, double E, double* acc) {
  const Law law(sd.p);
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  const double reach = law.reach();
  const uint32_t span = law_span(law);
  double s[3] = {0.0, 0.0, 0.0};
  clv_each<D, PER>(a, sd, i, xi, reach2_bound(reach), reach + E, [&](int64_t j, double) {
    double xj[3] = {0.0, 0.0, 0.0}, t[3];
#pragma unroll
    for (int c = 0; c < D; ++c) xj[c] = a.S[c][j];
    pair_term<D, Law, PER>(law, span, xi, xj, L, hL, true, t);
#pragma unroll
    for (int c = 0; c < D; ++c) s[c] = s[c] + t[c];
  });
#pragma unroll
  for (int c = 0; c < D; ++c) acc[c] = s[c];
}

// CellLinked on a skin list, one agent per lane.  Per step:
//   clv_order_row (inside the step's first stage): the skin-list entries
//     inside an agent's 3^D neighbor cells are put in CellLinked order --
//     cell k among the neighbor cells, then list position (= slot order) --
//     and written as its ordered list (a.wlist).  The order depends on the
//     cells alone, so it is kept until the agent or an entry changes cell
//     (clv_moved: under 1 % of the lists per step of a tissue; ordering them
//     all took both stages of 1,048,576 agents from 46 to 52 us on average)
//     or the lists are built: lists of at most 16 entries
//     by a sorting network over keys (k, position, row) in registers, longer
//     ones by insertion of the keys (k << 6 | position) into the lane's LDS
//     queue (stride blockDim, a.lcap entries); a list at capacity (possibly
//     truncated) is marked -1.
//   clv_stage_body: every stage walks that list.  An agent whose list may
//     miss a pair -- marked -1, or whose distance e from its reference
//     position plus the largest, E, over all agents exceeds the skin --
//     writes nothing and is queued for
//   clv_fix_body, which sums its pairs by clv_walk and finishes its stage.
// Stage 1 of a two-stage integrator records max e^2 for stage 2, the final
// stage for the next step's stage 1 (only agents past half the skin report;
// E is at least half the skin).

// One lane's queued agent (a.fix_rows), counted per queue in a.fix_n[fix_q].
__device__ __forceinline__ void clv_defer(const StageArgs& a, int64_t i) {
  const int32_t q = atomicAdd(a.fix_n + a.fix_q, 1);
  a.fix_rows[q] = (int32_t)i;
}

// e^2 of a stage-1 output past half the skin, into the device maximum.
__device__ __forceinline__ void clv_report(const StageArgs& a, double e2) {
  if (a.emax && !(e2 <= a.clv_half2)) atomicMax(a.emax, (unsigned long long)__double_as_longlong(e2));
}

// The ordered list of an agent with n <= W skin-list entries (see
// clv_order_row); returns its length.  The list holds lcap >= 16 entries
// per row, so all W loads are in bounds; entries past the length are
// replaced by the agent itself and sorted last.
template <int W, int D, int PER>
__device__ __forceinline__ int32_t clv_order_small(const StageArgs& a, const SimDev& sd, int64_t i, int32_t n,
                                                   int32_t ci) {
  uint32_t key[W];
  const uint32_t i4 = (uint32_t)i * 4u, l4 = (uint32_t)a.ldl * 4u;
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const int32_t raw = ld_b(a.list, i4 + (uint32_t)u * l4);
    key[u] = (uint32_t)(u < n ? raw : (int32_t)i);
  }
  // all W gathers are issued before the first key: the empty asm uses each
  // loaded value unconditionally, so the compiler cannot move a load into
  // the (u < n) branch behind its own wait
  int32_t cj[W];
#pragma unroll
  for (int u = 0; u < W; ++u) cj[u] = ld_b(a.ccell, key[u] * 4u);
#pragma unroll
  for (int u = 0; u < W; ++u) __asm__ volatile("" ::"v"(cj[u]));
  int32_t kept = 0;
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const int k = u < n ? cl_key<D, PER>(sd, ci, cj[u]) : 27;   // 27: outside the 3^D cells, sorts last
    key[u] |= ((uint32_t)k << 27) | ((uint32_t)u << 23);
    kept += k < 27 ? 1 : 0;
  }
  sort_net<W>(key);
#pragma unroll
  for (int v = 0; v < W; ++v)
    if (v < kept) st_b(a.wlist, i4 + (uint32_t)v * l4, (int32_t)(key[v] & 0x7FFFFFu));
  return kept;
}

// Row i's skin-list entries (a.list, a.list_n) in CellLinked order, written
// to a.wlist; returns their count, or -1 for a list at capacity (possibly
// truncated).  LDS: blockDim * a.lcap 16-bit keys (lists over 16 entries).
template <int D, int PER>
__device__ __forceinline__ int32_t clv_order_row(const StageArgs& a, const SimDev& sd, int64_t i,
                                                 unsigned char* lds) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int32_t* __restrict__ lp = a.list + i;       // entry q at lp[q * ldl]
  const int64_t ldl = a.ldl;
  const int32_t n = a.list_n[i];
  if (n >= a.lcap) return -1;
  const int32_t ci = a.ccell[i];
  // lists of at most 16 entries: every list read and cell gather in flight,
  // and the keys (k << 27 | position << 23 | row) sorted by a network in
  // registers; the row rides in the key (the set-up allows this form below
  // 2^23 rows), and 32-bit byte offsets address from the kernel-argument
  // bases.  (A form for 8 entries beside it gains nothing: the lanes of a
  // wave rarely all hold lists that short.)
  if (n <= 16) return clv_order_small<16, D, PER>(a, sd, i, n, ci);
  uint16_t* qk = (uint16_t*)lds + tid;                // this lane's queue, entry u at qk[u * nt]
  int32_t kept = 0;
  auto insert = [&](uint16_t key) {
    int32_t pos = kept;
    while (pos > 0) {
      const uint16_t prev = qk[(pos - 1) * nt];
      if (prev < key) break;
      qk[pos * nt] = prev;
      --pos;
    }
    qk[pos * nt] = key;
    ++kept;
  };
  for (int32_t q0 = 0; q0 < n; q0 += 4) {
    int32_t jj[4], cc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) jj[u] = q0 + u < n ? lp[(int64_t)(q0 + u) * ldl] : (int32_t)i;
#pragma unroll
    for (int u = 0; u < 4; ++u) cc[u] = a.ccell[jj[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (q0 + u >= n) continue;
      const int k = cl_key<D, PER>(sd, ci, cc[u]);
      if (k < 27) insert((uint16_t)((k << 6) | (q0 + u)));
    }
  }
  for (int32_t v0 = 0; v0 < kept; v0 += 4) {
    int32_t jj[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) jj[u] = v0 + u < kept ? lp[(int64_t)(qk[(v0 + u) * nt] & 63) * ldl] : 0;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (v0 + u < kept) a.wlist[(int64_t)(v0 + u) * ldl + i] = jj[u];
  }
  return kept;
}

template <int D, class Law, int PER, int NOISE>
__device__ __forceinline__ void clv_stage_body(const StageArgs& a, unsigned char* lds) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    // the step's bookkeeping, where no other kernel is using the words: the
    // other queue (its fix kernel is done, the next user is a later stage),
    // and in the first stage the next step's stage-1 maximum
    a.fix_n[1 - a.fix_q] = 0;
    if (a.clv_order) {
      *a.emax_next = 0ull;
      if (a.book) {
        // the record the host reads (system-scope stores into mapped host
        // memory, the step last)
        __hip_atomic_store(&a.rec->soon, a.efin[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&a.rec->e2max, a.efin[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&a.rec->step, a.step_no, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  const RowIdx ri = row_index(a.g);
  const SimDev& sd = a.g.sims[ri.sim];
  if (ri.local >= a.g.st[ri.sim].N) return;
  const int64_t i = ri.row;
  double xi[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < D; ++c) xi[c] = a.S[c][i];
  int32_t n;
  if (a.clv_order) {
    // the step's first stage: is the agent within reach of every pair its
    // list must hold?  Then its entries in CellLinked order, written for
    // the later stages and walked below
    if (a.efin) {
      // every agent is within E0 of its reference position, E0 the largest
      // reported displacement (agents past half the skin report) or a
      // little over half the skin; with no report all pairs are in the lists
      const unsigned long long e0 = *a.efin;
      if (e0 != 0ull) {
        const double E0 = fmax(sqrt(__longlong_as_double((long long)e0)), a.clv_e1);
        double s2 = 0.0;
#pragma unroll
        for (int c = 0; c < D; ++c) {
          double d = xi[c] - a.xref[c][i];
          if (PER) d = min_image(d, sd.L[c]);
          s2 = s2 + d * d;
        }
        if (!(sqrt(s2) + E0 <= a.clv_skin)) {
          a.wlist_n[i] = -1;
          a.order_row_next[i] = 1;
          clv_defer(a, i);
          return;
        }
      }
    }
    // the order of an earlier step holds while neither the agent nor an entry
    // has changed cell
    if (*a.order_now != 0 || a.order_row[i] != 0) {
      n = clv_order_row<D, PER>(a, sd, i, lds);
      a.wlist_n[i] = n;
      a.order_row[i] = 0;
    } else {
      n = a.wlist_n[i];
    }
  } else {
    n = a.wlist_n[i];
  }
  if (n < 0) { clv_defer(a, i); return; }
  if (a.fix_stage == 1 && *a.emax != 0ull) {
    // stage 2: could a pair active here lie outside the list?  (With no
    // stage-1 report every agent is within half the skin: none can.)
    double dx[3];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      dx[c] = xi[c] - a.xref[c][i];
      if (PER) dx[c] = min_image(dx[c], sd.L[c]);
    }
    double s2 = dx[0] * dx[0];
    if (D > 1) s2 = s2 + dx[1] * dx[1];
    if (D > 2) s2 = s2 + dx[2] * dx[2];
    const double E = fmax(sqrt(__longlong_as_double((long long)*a.emax)), a.clv_half);
    if (!(sqrt(s2) + E <= a.clv_skin)) { clv_defer(a, i); return; }
  }
  double upre[3] = {0.0, 0.0, 0.0}, acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < D; ++c) upre[c] = a.U[c][i];
  const Law law(sd.p);
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  const uint32_t span = law_span(law);
  const int32_t* __restrict__ lp = a.wlist + i;       // entry q at lp[q * ldl]
  const int64_t ldl = a.ldl;
  int32_t jn[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) jn[u] = u < n ? lp[(int64_t)u * ldl] : (int32_t)i;
  for (int32_t q0 = 0; q0 < n; q0 += 2) {
    int32_t jc[2];
    double xj[2][3];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      jc[u] = jn[u];
#pragma unroll
      for (int c = 0; c < D; ++c) xj[u][c] = a.S[c][jc[u]];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) jn[u] = q0 + 2 + u < n ? lp[(int64_t)(q0 + 2 + u) * ldl] : (int32_t)i;
    const bool live[2] = {q0 < n, q0 + 1 < n};
    double t[2][3];
    if constexpr (has_near<Law>::value) {      // as in gather_global
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        pair_term<D, Law, PER>(law, span, xi, xj[u], L, hL, live[u], t[u]);
#pragma unroll
        for (int c = 0; c < D; ++c) acc[c] = acc[c] + t[u][c];
      }
    } else {
      pair_terms<D, Law, PER, false, 2>(law, span, xi, xj, L, hL, 0.0, nullptr, 0, nullptr, live, t);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int c = 0; c < D; ++c) acc[c] = acc[c] + t[u][c];
    }
  }
  double e2 = 0.0;
  stage_finish<D, Law, NOISE, true>(a, sd, ri.sim, i, xi, acc, upre, -1.0, &e2);
  clv_report(a, e2);
}

template <int D, class Law, int PER, int NOISE>
__device__ void clv_fix_body(const StageArgs& a) {
  const int32_t cnt = a.fix_n[a.fix_q];
  for (int32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < cnt; q += gridDim.x * blockDim.x) {
    const int64_t i = a.fix_rows[q];
    int sim = 0;
    while (sim + 1 < a.nsims && a.g.sims[sim + 1].row_off <= i) ++sim;
    const SimDev& sd = a.g.sims[sim];
    double xi[3] = {0.0, 0.0, 0.0}, upre[3] = {0.0, 0.0, 0.0}, acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < D; ++c) { xi[c] = a.S[c][i]; upre[c] = a.U[c][i]; }
    const double E = a.fix_stage == 1 ? fmax(sqrt(__longlong_as_double((long long)*a.emax)), a.clv_half)
                                      : fmax(a.efin ? sqrt(__longlong_as_double((long long)*a.efin)) : 0.0, a.clv_e1);
    clv_walk<D, Law, PER>(a, sd, i, xi, E, acc);
    double e2 = 0.0;
    stage_finish<D, Law, NOISE, true>(a, sd, sim, i, xi, acc, upre, -1.0, &e2);
    clv_report(a, e2);
  }
}

// One integrator stage over the Verlet lists with the pair work spread
// evenly over the block's lanes.  The entries of the block's agents are
// numbered agent-major (a block-wide scan of the list lengths) and processed
// in rounds of whole agents holding about `fchunk` entries: every lane
// evaluates entries of the round -- gather, square root, division and law
// of one pair per lane step -- and stores the term in LDS; then each
// agent's thread adds its terms in list order (the order of the per-agent
// walk, so the sums are bit-identical) and finishes the stage.  A wavefront
// thus no longer runs to its longest list.  Lists are at most FLAT_MAX_CAP
// long.
template <int D, class Law, int PER, int NOISE>
__device__ __forceinline__ void flat_body(const StageArgs& a, unsigned char* lds) {
  if (a.gate && *a.gate != a.gate_run) return;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int chunk = a.fchunk;
  const int ch = chunk + a.fcap;
  double* term[3];
  unsigned char* p = lds;
#pragma unroll
  for (int c = 0; c < D; ++c) { term[c] = (double*)p; p += (size_t)8 * ch; }
  double* hx[3];
#pragma unroll
  for (int c = 0; c < D; ++c) { hx[c] = (double*)p; p += (size_t)8 * BRICK_MAX_BLOCK; }
  int32_t* offs = (int32_t*)p;
  p += (size_t)4 * (BRICK_MAX_BLOCK + 1);
  int32_t* rfirst = (int32_t*)p;
  p += (size_t)4 * (FLAT_MAX_ROUNDS + 1);
  int32_t* wsum = (int32_t*)p;
  p += 4 * 8;
  uint8_t* owner = (uint8_t*)p;

  const RowIdx ri = row_index(a.g);
  const SimDev& sd = a.g.sims[ri.sim];
  const int64_t N = a.g.st[ri.sim].N;
  const int64_t i = ri.row;
  const int64_t row0 = i - tid;                  // the block's rows are consecutive
  const bool live = ri.local < N;
  double xi[3] = {0.0, 0.0, 0.0}, upre[3] = {0.0, 0.0, 0.0};
  int32_t n = 0;
  if (live) {
#pragma unroll
    for (int c = 0; c < D; ++c) xi[c] = a.S[c][i];
    n = a.list_n[i];
#pragma unroll
    for (int c = 0; c < D; ++c) upre[c] = a.U[c][i];   // consumed by the stage update
  }
#pragma unroll
  for (int c = 0; c < D; ++c) hx[c][tid] = xi[c];
  for (int r = tid; r <= FLAT_MAX_ROUNDS; r += nt) rfirst[r] = 0x7FFFFFFF;
  const int32_t off = block_excl_scan(n, wsum, wsum + 7);
  offs[tid] = off;
  // round of an agent: the chunk its first entry falls in; a round's entries
  // run from its first agent's first entry to the next round's
  const int myr = n > 0 ? off / chunk : -1;
  __syncthreads();
  if (n > 0) atomicMin(&rfirst[myr], off);
  const int32_t P = wsum[7];
  __syncthreads();

  const Law law(sd.p);
  double L[3], hL[3];
  box_halves<D, PER>(sd, L, hL);
  const uint32_t span = law_span(law);
  const int32_t* __restrict__ list = a.list;
  const int64_t ldl = a.ldl;
  double acc[3] = {0.0, 0.0, 0.0};
  for (int r = 0; r < FLAT_MAX_ROUNDS; ++r) {
    const int32_t lo = rfirst[r];
    if (lo >= P) break;
    const int32_t nx = rfirst[r + 1];
    const int32_t hi = nx < P ? nx : P;
    if (myr == r)
      for (int32_t k = 0; k < n; ++k) owner[off - lo + k] = (uint8_t)tid;
    __syncthreads();
    // every lane evaluates entries of the round, two in flight
    for (int32_t p0 = lo + tid; p0 < hi; p0 += 2 * nt) {
      int32_t pp[2], jj[2], tt[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        pp[u] = p0 + u * nt;
        const bool v = pp[u] < hi;
        tt[u] = v ? owner[pp[u] - lo] : tid;
        const int32_t q = pp[u] - offs[tt[u]];
        jj[u] = v ? list[(int64_t)q * ldl + row0 + tt[u]] : (int32_t)i;
      }
      double xj[2][3];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int c = 0; c < D; ++c) xj[u][c] = a.S[c][jj[u]];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (pp[u] >= hi) continue;
        double xo[3] = {0.0, 0.0, 0.0}, t[3];
#pragma unroll
        for (int c = 0; c < D; ++c) xo[c] = hx[c][tt[u]];
        pair_term<D, Law, PER>(law, span, xo, xj[u], L, hL, true, t);
#pragma unroll
        for (int c = 0; c < D; ++c) term[c][pp[u] - lo] = t[c];
      }
    }
    __syncthreads();
    if (myr == r)
      for (int32_t k = off - lo; k < off - lo + n; ++k)
#pragma unroll
        for (int c = 0; c < D; ++c) acc[c] = acc[c] + term[c][k];
    __syncthreads();
  }
  if (!live) return;
  stage_finish<D, Law, NOISE, true>(a, sd, ri.sim, i, xi, acc, upre);
}

}  // namespace cbm

#endif  // CBM_STAGE_H
