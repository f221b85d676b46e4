// Candidate generation over a cell grid, shared by the neighbour-row,
// pair-list and Coulomb sweeps.
//
// The stencil of a centre is the set of x-rows (dy, dz) whose band of cells
// comes within the cutoff of the centre, each trimmed in x to the cells that
// can still hold a neighbour; with cells of about half the short cutoff this
// is a close cover of the cutoff sphere.  Every row is one contiguous
// range of the cell-ordered atom array (two when it wraps a periodic edge).
// The ranges of one centre are collected in LDS with a prefix sum of their
// lengths, so a wavefront sweeps the concatenated candidates 64 at a time
// whatever the cell occupancy.
//
// Minimum distances are computed from cell indices; for an open grid atoms
// outside it are clamped to edge cells, which only lowers index differences,
// so the bound stays a lower bound of the true distance.
#pragma once
#include <math.h>

#include "tm_common.h"

struct CellGrid {
  const int* cell_start;   // ncell+1, offsets into cell_atoms
  const int* cell_atoms;   // atoms sorted by cell (index order inside a cell)
  const int* cell_of;      // cell of each atom
  const int* cell_pos;     // position of each atom in cell_atoms
  const double* posc;      // positions in cell order (float64 [N,3])
  const int* molc;         // molecule of each cell-ordered atom (NULL: one system)
  int nc[3];               // cells per axis
  float cs[3];             // cell edges (A)
  float org[3];            // grid origin (A): cell k of an axis spans [org + k cs, org + (k+1) cs)
  int periodic;            // 1: wrap, 0: clamp
  // stencil of one cutoff (tm_set_stencil, on the host)
  int k[3];                // cells to either side of a centre's that can hold a neighbour
  int full[3];             // 1: they wrap the whole periodic axis
  int ny, nrow;            // stencil rows per z layer, and in all
  unsigned magic;          // ceil(2^32 / ny): t / ny = (t magic) >> 32 for the row numbers here (ny > 1)
  double len[3], inv_len[3];   // axis lengths nc cs and their reciprocals
  float flo[3], fhi[3];    // bounds of a centre's offset inside its cell (tm_centre)
  float rc2, inv_cs0;      // squared trimmed cutoff, 1 / cs[0]
};

// Margin (A) added to the cutoff when rows are trimmed with the centre's own
// position: it covers the FP32 rounding of positions and cell bounds, so the
// candidates stay a superset of the atoms inside the cutoff.
constexpr float TM_TRIM_MARGIN = 2e-3f;

// Stencil of cutoff rc over the grid.  Computed once per launch: with the
// integer divisions and the ceilings of a cutoff in cells it cost each wave
// about half of its instructions per 64 rows.  Without a grid its sizes mean
// nothing (callers may pass zeros) and are not looked at.
inline void tm_set_stencil(CellGrid& g, float rc) {
  if (g.cell_atoms == nullptr) return;
  for (int d = 0; d < 3; ++d) {
    // a band further out is at least ceil(rc / cs) cells away.  An axis counts
    // as wrapped two bands before it is, which decides the order of its rows
    // and is kept, since sums are formed in that order.
    g.k[d] = (int)ceilf((rc + TM_TRIM_MARGIN) / g.cs[d]);
    g.full[d] = g.periodic && (2 * ((int)ceilf(rc / g.cs[d]) + 1) + 1 >= g.nc[d]);
    g.len[d] = (double)g.nc[d] * (double)g.cs[d];
    g.inv_len[d] = 1.0 / g.len[d];
    g.flo[d] = g.periodic ? -g.cs[d] : 0.f;
    g.fhi[d] = !g.periodic ? g.cs[d] : (g.nc[d] < 3 ? 2.f : 1.5f) * g.cs[d];
  }
  g.ny = g.full[1] ? g.nc[1] : 2 * g.k[1] + 1;
  g.nrow = g.ny * (g.full[2] ? g.nc[2] : 2 * g.k[2] + 1);
  g.magic = g.ny > 1 ? (unsigned)((0x100000000ull + (unsigned)g.ny - 1) / (unsigned)g.ny) : 0u;
  const float rcm = rc + TM_TRIM_MARGIN;
  g.rc2 = rcm * rcm;
  g.inv_cs0 = 1.0f / g.cs[0];
}

// Distance along one axis from a centre at offset f inside its cell to the band
// of cells d cells away (0 for its own band).
__device__ __forceinline__ float tm_band_dist(int d, float f, float cs) {
  return fmaxf(fmaxf((float)d * cs - f, f - (float)(d + 1) * cs), 0.f);
}

// Lanes below this one whose bit is set in a wave-wide ballot.
__device__ __forceinline__ int tm_lanes_below(unsigned long long bal) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
}

// Ranges per centre (at most two per stencil row).  A sweep of cutoff rc over
// cells of edge cs has at most (2*ceil(rc/cs)+3)^2 rows.
template <int CAP>
struct RangeLds {
  static constexpr int cap = CAP;
  int lo[CAP];
  int pre[CAP + 1];
  int mark[64];   // range starts inside the current chunk, tagged with the chunk's base
};

// A centre's cell and its offset inside the cell.
//
// A centre outside an open grid sits in an edge cell and is taken to that
// cell's face.  Taking centre and candidate into the grid never makes them
// further apart, so with the centre there all distances to bands of cells and
// the range along x bound the true ones from below; its own band, for one, can
// hold atoms that are as far outside.
// PERIODIC 1 or 0: what the grid is, where the kernel knows it; -1: the bounds
// come with the grid, one instruction per axis (a branch on g.periodic cost the
// periodic rows 0.5 us).  A periodic grid's bounds lie outside every offset a
// coordinate has (which is off by a whole cell only on axes of one or two) and
// hold those that have lost their digits near the grid.
struct CellCentre {
  int c[3];
  float f[3];
};
template <int PERIODIC = -1>
__device__ __forceinline__ CellCentre tm_centre(const CellGrid& g, int cell, double px, double py,
                                                double pz) {
  CellCentre o;
  o.c[0] = cell % g.nc[0];
  o.c[1] = (cell / g.nc[0]) % g.nc[1];
  o.c[2] = cell / (g.nc[0] * g.nc[1]);
  const double p[3] = {px, py, pz};
  const bool periodic = PERIODIC < 0 ? g.periodic : PERIODIC;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    double u = p[d] - (double)g.org[d];
    if (periodic && g.nc[d] < 3) u -= g.len[d] * floor(u / g.len[d]);
    u -= (double)o.c[d] * (double)g.cs[d];
    // wrapped in FP64, so unwrapped coordinates keep their precision; the
    // offset lies within a cell of a multiple of the length, so the nearest one is it
    if (periodic && g.nc[d] >= 3) u -= g.len[d] * rint(u * g.inv_len[d]);
    o.f[d] = (float)u;   // offset inside the centre's cell
    if (PERIODIC == 0) o.f[d] = __builtin_amdgcn_fmed3f(o.f[d], 0.f, g.cs[d]);
    if (PERIODIC < 0) o.f[d] = __builtin_amdgcn_fmed3f(o.f[d], g.flo[d], g.fhi[d]);
  }
  return o;
}

// The candidates of stencil row t of a centre: [lo0, lo0 + n0) and, where the
// row wraps a periodic edge, [lo1, lo1 + n1) of the cell-ordered arrays.
// Rows are trimmed with the centre's position: along y and z the distance from
// the centre to a row's band of cells, along x the cells that [x - s, x + s]
// covers with s^2 = (rc + margin)^2 - dy^2 - dz^2.  On an axis whose stencil
// wraps the whole periodic box the cell-gap bound (|d| - 1) cs is used instead
// (two images of a band can be equally near there).
__device__ __forceinline__ void tm_row(const CellGrid& g, const CellCentre& o, int t, int& lo0,
                                       int& n0, int& lo1, int& n1) {
  lo0 = lo1 = n0 = n1 = 0;
  if (t >= g.nrow) return;
  const int tz = g.ny > 1 ? (int)__umulhi((unsigned)t, g.magic) : t, ty = t - tz * g.ny;
  // band index along one axis, its cell and its distance; false outside an open grid
  auto band = [&](int d, int off, int& cell, float& dist) {
    if (g.full[d]) {
      int dd = off - o.c[d];
      if (dd > g.nc[d] / 2) dd -= g.nc[d];
      if (dd < -g.nc[d] / 2) dd += g.nc[d];
      cell = off;
      dist = fmaxf(0.f, (float)(abs(dd) - 1)) * g.cs[d];
      return true;
    }
    const int dd = off - g.k[d];
    cell = o.c[d] + dd;
    dist = tm_band_dist(dd, o.f[d], g.cs[d]);
    if (!g.periodic) return cell >= 0 && cell < g.nc[d];
    if (cell < 0) cell += g.nc[d];           // 2 k + 1 < nc here, so one wrap is enough
    else if (cell >= g.nc[d]) cell -= g.nc[d];
    return true;
  };
  int y, z;
  float my, mz;
  const bool oky = band(1, ty, y, my), okz = band(2, tz, z, mz);
  const float rem = g.rc2 - my * my - mz * mz;
  if (!oky || !okz || !(rem > 0.f)) return;
  const float sx = __builtin_amdgcn_sqrtf(rem);   // its last digit is far inside the margin
  int xlo = o.c[0] + (int)floorf((o.f[0] - sx) * g.inv_cs0);
  int xhi = o.c[0] + (int)floorf((o.f[0] + sx) * g.inv_cs0);
  const int* start = g.cell_start + g.nc[0] * (y + g.nc[1] * z);
  if (g.periodic && xhi - xlo + 1 >= g.nc[0]) {
    xlo = 0;
    xhi = g.nc[0] - 1;
  }
  if (!g.periodic) {
    xlo = max(xlo, 0);
    xhi = min(xhi, g.nc[0] - 1);
    if (xlo > xhi) return;
  }
  // a wrapped row is its upper part, then its lower part
  const bool wl = xlo < 0, wr = xhi >= g.nc[0];
  if (wl) xlo += g.nc[0];
  if (wr) xhi -= g.nc[0];
  lo0 = start[xlo];
  n0 = start[wl || wr ? g.nc[0] : xhi + 1] - lo0;
  if (wl || wr) {
    lo1 = start[0];
    n1 = start[xhi + 1] - lo1;
  }
}

// Builds the candidate ranges of atom i for the grid's cutoff into R (one
// wavefront, all lanes participate).  Returns the number of candidates; *nrange
// gets the number of ranges (capped at CAP, overflow flagged).  Every range is
// non-empty, so the range starts pre[] increase strictly.
template <int CAP>
__device__ inline int tm_build_ranges(int i, const CellGrid& g, RangeLds<CAP>& R, int lane,
                                      int* flags, int* nrange, double px, double py, double pz) {
  const CellCentre o = tm_centre(g, g.cell_of[i], px, py, pz);
  R.mark[lane] = -1;   // no chunk base is negative; ordered by the wave barriers below
  int nr = 0;   // wave-uniform
  for (int base = 0; base < g.nrow; base += 64) {
    int lo0, n0, lo1, n1;
    tm_row(g, o, base + lane, lo0, n0, lo1, n1);
    // keep only non-empty ranges (both halves of a wrapped row can be empty)
    int cnt = (n0 > 0) + (n1 > 0);
    if (n0 <= 0) { lo0 = lo1; n0 = n1; }
    // compact the non-empty ranges of this round into R (lane order = row order)
    unsigned long long b1 = __ballot(cnt >= 1);
    unsigned long long b2 = __ballot(cnt >= 2);
    int before = tm_lanes_below(b1) + tm_lanes_below(b2);
    int slot = nr + before;
    if (cnt >= 1 && slot < CAP) { R.lo[slot] = lo0; R.pre[slot + 1] = n0; }
    if (cnt >= 2 && slot + 1 < CAP) { R.lo[slot + 1] = lo1; R.pre[slot + 2] = n1; }
    nr += __popcll(b1) + __popcll(b2);
  }
  if (nr > CAP) {
    if (lane == 0 && flags) atomicOr(&flags[TM_FLAG_NB_OVERFLOW], 4);
    nr = CAP;
  }
  __syncwarp();
  // inclusive scan of lengths into pre[1..nr] (sequential over 64-wide blocks)
  if (lane == 0) R.pre[0] = 0;
  int carry = 0;
  for (int base = 0; base < nr; base += 64) {
    int t = base + lane;
    int v = t < nr ? R.pre[t + 1] : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      int u = __shfl_up(v, o, 64);
      if (lane >= o) v += u;
    }
    if (t < nr) R.pre[t + 1] = carry + v;
    carry += __shfl(v, 63, 64);
  }
  __syncwarp();
  *nrange = nr;
  return __builtin_amdgcn_readfirstlane(carry);   // the same in every lane
}

// Cell-order position of candidate base + lane of a sweep over the ranges in R
// (0 for base + lane >= total), and r0 advanced from the range holding
// candidate base to the range holding base + 64.  Call with base = 0, 64,
// 128, ... in turn, r0 = 0 first (wave-uniform); needs nr >= 1.
//
// Lane k looks at range r0 + k.  Ranges r0 + 1 .. r0 + span - 1 start inside
// the chunk, at offsets pre - base in [1, 63], distinct because every range
// is non-empty.  Each such lane tags slot (pre - base) of the wave's mark array
// with the chunk's base; every lane reads its own slot, and a ballot gives the
// start positions, so lane L's range is r0 + (number of starts at or below L).
// mark[0] is never written and older tags are other chunks' bases, so only
// this chunk's starts match.
template <int CAP>
__device__ __forceinline__ int tm_locate(RangeLds<CAP>& R, int nr, int total, int lane, int base,
                                         int& r0) {
  const int rk = r0 + lane;
  const int pv = R.pre[min(rk, nr)];
  const int lo_k = R.lo[min(rk, nr - 1)];
  const int pre_k = rk < nr ? pv : 0x7fffffff;   // past the last range: never inside
  const int span = __popcll(__ballot(pre_k <= base + 63));   // >= 1: range r0 holds base
  if (lane >= 1 && lane < span) R.mark[pre_k - base] = base;
  __syncwarp();
  const unsigned long long starts = __ballot(R.mark[lane] == base);
  const int idx = __popcll(starts & ((2ull << lane) - 1ull));
  const int lo_r = __shfl(lo_k, idx, 64);
  const int pre_r = __shfl(pre_k, idx, 64);
  // start of range r0 + span, the first one past the chunk (lane span holds it)
  const int nxt = span < 64 ? __builtin_amdgcn_readlane(pre_k, span)
                            : (r0 + 64 < nr ? R.pre[r0 + 64] : 0x7fffffff);
  r0 += span - 1 + (nxt <= base + 64 ? 1 : 0);
  const int t = base + lane;
  return t < total ? lo_r + (t - pre_r) : 0;
}

// Sweep the candidates of centre i: calls f(p, valid, mapped) with all 64
// lanes in lockstep (so f may use ballots); p indexes the cell-ordered arrays
// when mapped, the atom arrays otherwise (molecule range, no grid).
template <int CAP, class F>
__device__ __forceinline__ void tm_sweep(int i, const int* __restrict__ mol,
                                         const int* __restrict__ mol_start, const CellGrid& g,
                                         RangeLds<CAP>& R, int lane, int* flags, double px,
                                         double py, double pz, F&& f) {
  if (g.cell_atoms == nullptr) {
    const int m = mol[i];
    const int lo = mol_start[m], hi = mol_start[m + 1];
    for (int base = lo; base < hi; base += 64) {
      int p = base + lane;
      f(p, p < hi, 0);
    }
    return;
  }
  int nr = 0;
  const int total = tm_build_ranges(i, g, R, lane, flags, &nr, px, py, pz);
  // Walk the concatenated ranges 64 candidates at a time.
  int r0 = 0;
  for (int base = 0; base < total; base += 64) {
    const int p = tm_locate(R, nr, total, lane, base, r0);
    f(p, base + lane < total, 1);
  }
}

// tm_sweep with the candidate loads of the next chunk in flight while the
// current chunk is processed: load(p, valid, mapped) fetches what f needs for
// one candidate and returns it by value; f(p, valid, mapped, payload) consumes
// it.  Same candidates in the same order as tm_sweep.
template <int CAP, class LD, class F>
__device__ __forceinline__ void tm_sweep_pf(int i, const int* __restrict__ mol,
                                            const int* __restrict__ mol_start, const CellGrid& g,
                                            RangeLds<CAP>& R, int lane, int* flags, double px,
                                            double py, double pz, LD&& load, F&& f) {
  if (g.cell_atoms == nullptr) {
    const int m = mol[i];
    const int lo = mol_start[m], hi = mol_start[m + 1];
    auto cur = load(lo + lane, lo + lane < hi, 0);
    for (int base = lo; base < hi; base += 64) {
      const int pn = base + 64 + lane;
      auto nxt = load(pn, pn < hi, 0);
      f(base + lane, base + lane < hi, 0, cur);
      cur = nxt;
    }
    return;
  }
  int nr = 0;
  const int total = tm_build_ranges(i, g, R, lane, flags, &nr, px, py, pz);
  int r0 = 0;
  auto locate = [&](int base) { return tm_locate(R, nr, total, lane, base, r0); };
  if (total <= 0) return;
  int p = locate(0);
  auto cur = load(p, lane < total, 1);
  for (int base = 0; base < total; base += 64) {
    const int pc = p;
    const bool vc = base + lane < total;
    // issued unconditionally (one chunk past the end on the last pass: r0
    // stays in [0, nr - 1] and every lane is invalid), so the loads in flight
    // are the same on every path
    p = locate(base + 64);
    auto nxt = load(p, base + 64 + lane < total, 1);
    f(pc, vc, 1, cur);
    cur = nxt;
  }
}

// Inclusive sum over the lanes of a wave (DPP row shifts and broadcasts).
__device__ __forceinline__ int tm_wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31
  return x;
}

// The candidates of one centre as a list in LDS.  Each round takes 64 stencil
// rows, one per lane, and writes their candidates behind those left over from
// the round before (fewer than 64), in row order and at most CAP at a time;
// whole chunks of 64 are then consumed.  load(p) fetches what f needs for
// candidate p, one chunk ahead of its use; f(p, valid, payload) runs with all
// lanes in lockstep.  Same candidates in the same order as tm_sweep: a lane
// reads its candidate from the list where tm_sweep finds it by a search over
// the ranges (35 vector instructions and a chain of three LDS round trips per
// chunk).
template <int CAP>
struct ListLds {
  int p[CAP];
};

template <int CAP, class LD, class F>
__device__ __forceinline__ void tm_sweep_list(const CellGrid& g, const CellCentre& o,
                                              ListLds<CAP>& L, int lane, LD&& load, F&& f) {
  static_assert(CAP >= 192, "room for a chunk and what is left of the one before");
  int have = 0;   // candidates in the list, from its start (wave-uniform)
  for (int base = 0; base < g.nrow; base += 64) {
    int lo0, n0, lo1, n1;
    tm_row(g, o, base + lane, lo0, n0, lo1, n1);
    const int n = n0 + n1, incl = tm_wave_scan(n), pre = incl - n;
    const int total = __builtin_amdgcn_readlane(incl, 63);
    for (int w0 = 0; w0 < total;) {   // the round's candidates [w0, w1)
      const int w1 = min(total, w0 + CAP - have);
      {
        int q = max(pre, w0);
        const int e0 = min(pre + n0, w1), e1 = min(incl, w1), to = have - w0;
        for (; q < e0; ++q) L.p[to + q] = lo0 + (q - pre);
        for (q = max(q, pre + n0); q < e1; ++q) L.p[to + q] = lo1 + (q - pre - n0);
      }
      have += w1 - w0;
      w0 = w1;
      __syncwarp();
      if (have < 64) continue;
      // two payloads in turn: one chunk is used while the next one's loads are
      // in flight
      int h = 64, p0 = L.p[lane], p1;
      auto c0 = load(p0), c1 = c0;
      for (;;) {
        const bool m1 = h + 64 <= have;   // another whole chunk: its loads go first
        p1 = m1 ? L.p[h + lane] : p0;
        c1 = load(p1);
        f(p0, true, c0);
        if (!m1) break;
        h += 64;
        const bool m0 = h + 64 <= have;
        p0 = m0 ? L.p[h + lane] : p1;
        c0 = load(p0);
        f(p1, true, c1);
        if (!m0) break;
        h += 64;
      }
      // what is left moves to the front
      const int left = have - h;
      const int v = lane < left ? L.p[h + lane] : 0;
      __syncwarp();
      if (lane < left) L.p[lane] = v;
      have = left;
      __syncwarp();
    }
  }
  if (have > 0) {
    const bool valid = lane < have;
    const int p = L.p[valid ? lane : 0];
    f(p, valid, load(p));
  }
}

// Upper bound of the candidate ranges one centre's sweep can need (the
// ranges tm_build_ranges keeps): stencil rows (dy, dz) whose cell-gap distance
// max(|d| - 1, 0) cs is within the trimmed cutoff (the band distance the sweep
// uses is never smaller), two ranges per row where a periodic row can wrap.
inline int tm_range_bound(double rc, const double cs[3], const int nc[3], int periodic) {
  const double r = rc + (double)TM_TRIM_MARGIN;
  int span[2];
  int full[2];
  for (int d = 1; d < 3; ++d) {
    int k = (int)ceil(rc / cs[d]) + 1;
    full[d - 1] = periodic && 2 * k + 1 >= nc[d];
    span[d - 1] = full[d - 1] ? nc[d] : 2 * k + 1;
  }
  auto gap = [&](int axis, int o) {
    int d = full[axis] ? (o <= nc[axis + 1] / 2 ? o : o - nc[axis + 1]) : o - span[axis] / 2;
    return fmax(0.0, (double)(abs(d) - 1)) * cs[axis + 1];
  };
  int rows = 0;
  for (int oz = 0; oz < span[1]; ++oz)
    for (int oy = 0; oy < span[0]; ++oy) {
      double gy = gap(0, oy), gz = gap(1, oz);
      rows += gy * gy + gz * gz < r * r;
    }
  return periodic ? 2 * rows : rows;
}
