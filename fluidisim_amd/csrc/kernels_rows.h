// Coarse levels held as row coefficients: the levels that are neither
// compact (kernels_coarse.h) nor in the compact tail, that is every level of
// the re-discretised operator and of the damped-Jacobi smoother, and levels
// whose rows do not split into quads.
//
// row_sums (delta3d_multigrid.rs:216-255) looks at a face's aperture, then at
// its neighbour's kind, then at the neighbour's value: a chain of three rounds
// of memory latency per row, which a coarse level has nothing to hide behind.
// Here the hierarchy turns each row into six coefficients once per projection
// (face order x-, x+, y-, y+, z-, z+): a > 0 couples to the neighbour with a,
// -2a < 0 is the Dirichlet term of air at a coarse half cell, 0 is nothing.
// Every load of a pass is then independent of the others, and the arithmetic
// is row_sums' term for term. On the levels of a 128x64x96 domain a sweep
// takes 4.5 us against 5.4, a restriction 4.4 against 24, the
// one-workgroup tail 22 against 48.
#pragma once
#include "kernels_fast.h"

namespace fsp {

// Coefficients and diagonals of a level (coarse_row's terms in its order).
__global__ void __launch_bounds__(BLOCK) k_r6_build(Level L) {
#pragma clang fp contract(off)
  FSP_FOR(c, L.n) {
    int i, j, k;
    ldecode(L, c, i, j, k);
    const size_t plane = (size_t)L.nx * L.ny;
    const bool gal = L.galerkin != 0, on = L.kind[c] > 0;
    float acc = 0.f;
    auto face = [&](int f, float a, bool has, size_t n, bool top) {
      float v = 0.f;
      const int8_t kn = has ? L.kind[n] : (int8_t)(top ? -1 : 0);
      if (on && a != 0.f) {
        if (kn > 0) v = a;
        else if (!gal && kn < 0) v = -(2.0f * a);
      }
      if (v != 0.f) acc += fabsf(v);
      L.c6[(size_t)f * L.n + c] = v;
    };
    face(0, L.ou[((size_t)k * L.ny + j) * (L.nx + 1) + i], i > 0, c - 1, false);
    face(1, L.ou[((size_t)k * L.ny + j) * (L.nx + 1) + i + 1], i + 1 < L.nx, c + 1, false);
    face(2, L.ov[((size_t)k * (L.ny + 1) + j) * L.nx + i], j > 0, c - L.nx, false);
    face(3, L.ov[((size_t)k * (L.ny + 1) + j + 1) * L.nx + i], j + 1 < L.ny, c + L.nx, false);
    face(4, L.ow[((size_t)k * L.ny + j) * L.nx + i], k > 0, c - plane, false);
    face(5, L.ow[((size_t)(k + 1) * L.ny + j) * L.nx + i], k + 1 < L.nz, c + plane, true);
    if (on && gal) acc += L.dd[c];
    L.diag[c] = on ? acc * L.inv : 0.f;
  }
}

__device__ __forceinline__ float r6_row(const float v[6], bool gal, float dd, float inv, float pc, const float nb[6]) {
#pragma clang fp contract(off)
  float acc = 0.f;
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const float t = v[f] > 0.f ? v[f] * (pc - nb[f]) : -v[f] * pc;
    acc = v[f] != 0.f ? acc + t : acc;
  }
  if (gal) acc += dd * pc;
  return acc * inv;
}

// A cell's six neighbours, indices clamped into the level (a clamped one has no coupling).
__device__ __forceinline__ void r6_neighbours(const Level& L, size_t c, int i, int j, int k, size_t nb[6]) {
  const size_t plane = (size_t)L.nx * L.ny;
  nb[0] = i > 0 ? c - 1 : c;
  nb[1] = i + 1 < L.nx ? c + 1 : c;
  nb[2] = j > 0 ? c - L.nx : c;
  nb[3] = j + 1 < L.ny ? c + L.nx : c;
  nb[4] = k > 0 ? c - plane : c;
  nb[5] = k + 1 < L.nz ? c + plane : c;
}
__device__ __forceinline__ void r6_load(const Level& L, size_t c, float v[6]) {
#pragma unroll
  for (int f = 0; f < 6; ++f) v[f] = L.c6[(size_t)f * L.n + c];
}

constexpr float R6_OMEGA = 6.0f / 7.0f;  // delta3d_multigrid.rs:28-34

// One damped-Jacobi sweep (delta3d_multigrid.rs:290-299) of x from zero.
__global__ void __launch_bounds__(BLOCK) k_r6_zero(Level L, float* xout, Ctl* ctl) {
#pragma clang fp contract(off)
  if (!ctl->active) return;
  FSP_FOR(c, L.n) {
    const float dg = L.diag[c];
    xout[c] = dg > 0.f ? R6_OMEGA * L.r[c] / dg : 0.f;
  }
}
// The first two sweeps from zero in one launch: the first is local, so its
// neighbours' values are formed from their r and diagonals.
__global__ void __launch_bounds__(BLOCK) k_r6_first(Level L, float* xout, Ctl* ctl) {
#pragma clang fp contract(off)
  if (!ctl->active) return;
  FSP_FOR(c, L.n) {
    int i, j, k;
    ldecode(L, c, i, j, k);
    size_t n[6];
    r6_neighbours(L, c, i, j, k, n);
    float v[6], rn[6], dn[6], nb[6];
    r6_load(L, c, v);
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      rn[f] = L.r[n[f]];
      dn[f] = L.diag[n[f]];
    }
    const float rc = L.r[c], dg = L.diag[c], dd = L.galerkin ? L.dd[c] : 0.f;
#pragma unroll
    for (int f = 0; f < 6; ++f) nb[f] = dn[f] > 0.f ? R6_OMEGA * rn[f] / dn[f] : 0.f;
    float xc = dg > 0.f ? R6_OMEGA * rc / dg : 0.f;
    if (dg > 0.f) xc += R6_OMEGA * (rc - r6_row(v, L.galerkin != 0, dd, L.inv, xc, nb)) / dg;
    xout[c] = xc;
  }
}
// A sweep xin -> xout; PROLONG: of xin + the parents xp on level C.
template <bool PROLONG>
__global__ void __launch_bounds__(BLOCK) k_r6_jacobi(Level L, Level C, const float* xp, const float* xin, float* xout,
                                                     Ctl* ctl) {
#pragma clang fp contract(off)
  if (!ctl->active) return;
  FSP_FOR(c, L.n) {
    int i, j, k;
    ldecode(L, c, i, j, k);
    size_t n[6];
    r6_neighbours(L, c, i, j, k, n);
    float v[6], nb[6];
    r6_load(L, c, v);
#pragma unroll
    for (int f = 0; f < 6; ++f) nb[f] = xin[n[f]];
    float xc = xin[c];
    const float rc = L.r[c], dg = L.diag[c], dd = L.galerkin ? L.dd[c] : 0.f;
    if (PROLONG) {
      // a clamped neighbour's parent may be another cell's: it has no coupling
      const int di[6] = {-1, 1, 0, 0, 0, 0}, dj[6] = {0, 0, -1, 1, 0, 0}, dk[6] = {0, 0, 0, 0, -1, 1};
      float p[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        const int ii = max(i + di[f], 0), jj = max(j + dj[f], 0), kk = max(k + dk[f], 0);
        p[f] = xp[lidx(C, min(ii, L.nx - 1) >> 1, min(jj, L.ny - 1) >> 1, min(kk, L.nz - 1) >> 1)];
      }
      xc = xc + xp[lidx(C, i >> 1, j >> 1, k >> 1)];
#pragma unroll
      for (int f = 0; f < 6; ++f) nb[f] = nb[f] + p[f];
    }
    if (dg > 0.f) xc += R6_OMEGA * (rc - r6_row(v, L.galerkin != 0, dd, L.inv, xc, nb)) / dg;
    xout[c] = xc;
  }
}
// One colour of red-black Gauss-Seidel, in place; x and L.r in storage ST;
// first: x starts at zero.
template <int ST>
__global__ void __launch_bounds__(BLOCK) k_r6_gs(Level L, typename Store<ST>::T* x, int colour, int first, Ctl* ctl) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  if (!ctl->active) return;
  const typename SV::T* lr = reinterpret_cast<const typename SV::T*>(L.r);
  FSP_FOR(c, L.n) {
    int i, j, k;
    ldecode(L, c, i, j, k);
    const bool mine = ((i + j + k) & 1) == colour;
    if (first) {
      const float dg = L.diag[c];
      SV::st(x, c, mine && dg > 0.f ? SV::ld(lr, c) / dg : 0.f);
      continue;
    }
    if (!mine) continue;
    size_t n[6];
    r6_neighbours(L, c, i, j, k, n);
    float v[6], nb[6];
    r6_load(L, c, v);
#pragma unroll
    for (int f = 0; f < 6; ++f) nb[f] = SV::ld(x, n[f]);
    const float xc = SV::ld(x, c), rc = SV::ld(lr, c), dg = L.diag[c], dd = L.galerkin ? L.dd[c] : 0.f;
    if (dg > 0.f) SV::st(x, c, xc + (rc - r6_row(v, L.galerkin != 0, dd, L.inv, xc, nb)) / dg);
  }
}
// Residual of level F restricted to L (delta3d_multigrid.rs:312-321, restrict3
// :258-272): eight consecutive lanes take the eight children of a coarse
// cell, and every lane of the group sums them in child order (z, y, x; x fastest).
template <int ST>
__global__ void __launch_bounds__(BLOCK) k_r6_restrict(Level F, Level L, const typename Store<ST>::T* xf, Ctl* ctl) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  if (!ctl->active) return;
  const typename SV::T* fr = reinterpret_cast<const typename SV::T*>(F.r);
  typename SV::T* lr = reinterpret_cast<typename SV::T*>(L.r);
  const int base = (int)(threadIdx.x & 63u) & ~7;
  // (BLOCK and 8 L.n are multiples of 8: a group is never split, and the loop ends for all of it)
  for (size_t q = (size_t)blockIdx.x * BLOCK + threadIdx.x; q < 8 * L.n; q += (size_t)gridDim.x * BLOCK) {
    const size_t cc = q >> 3;
    const int ch = (int)(q & 7);
    int i, j, k;
    ldecode(L, cc, i, j, k);
    const int fi = 2 * i + (ch & 1), fj = 2 * j + ((ch >> 1) & 1), fk = 2 * k + (ch >> 2);
    const size_t f = lidx(F, fi, fj, fk);
    size_t n[6];
    r6_neighbours(F, f, fi, fj, fk, n);
    float v[6], nb[6];
    r6_load(F, f, v);
#pragma unroll
    for (int g = 0; g < 6; ++g) nb[g] = SV::ld(xf, n[g]);
    const float t = SV::ld(fr, f) - r6_row(v, F.galerkin != 0, F.galerkin ? F.dd[f] : 0.f, F.inv, SV::ld(xf, f), nb);
    float s = 0.f;
#pragma unroll
    for (int m = 0; m < 8; ++m) s += __shfl(t, base + m);
    if (ch == 0) SV::st(lr, cc, 0.125f * s);
  }
}

// ---------------------------------------------------------------- tail
// Levels of at most TAIL_CELLS cells in one workgroup: two buffers of x and r
// per level in LDS (12 bytes a cell), each thread's cells (up to four) with
// their coefficients in registers for a level's whole sequence of sweeps.
// Jacobi sweeps go from one buffer to the other, red-black ones stay in the
// first; the buffer that is free takes the residual for the restriction.
template <int ST>
struct R6Cells {
  using SV = Store<ST>;
  static constexpr int S = (TAIL_CELLS + TAIL_THREADS - 1) / TAIL_THREADS;
  float v[S][6], dg[S], dd[S], r[S];
  int par[S];

  __device__ __forceinline__ void load(const Level& L, const float* r_lds) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int c = (int)threadIdx.x + s * TAIL_THREADS;
      dg[s] = dd[s] = r[s] = 0.f;
      par[s] = -1;  // no cell
      if (c >= (int)L.n) continue;
      r6_load(L, c, v[s]);
      dg[s] = L.diag[c];
      if (L.galerkin) dd[s] = L.dd[c];
      r[s] = r_lds[c];
      int i, j, k;
      ldecode(L, c, i, j, k);
      par[s] = (i + j + k) & 1;
    }
  }
  __device__ __forceinline__ float row(const Level& L, const float* x, int s, int c) const {
    const int plane = L.nx * L.ny;
    const int off[6] = {-1, 1, -L.nx, L.nx, -plane, plane};
    float nb[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) nb[f] = x[c + (v[s][f] > 0.f ? off[f] : 0)];
    return r6_row(v[s], L.galerkin != 0, dd[s], L.inv, x[c], nb);
  }
  __device__ __forceinline__ void jacobi(const Level& L, const float* x, float* out, bool first) const {
#pragma clang fp contract(off)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (par[s] < 0) continue;
      const int c = (int)threadIdx.x + s * TAIL_THREADS;
      float xc = first ? 0.f : x[c];
      if (dg[s] > 0.f) xc = SV::rnd(xc + R6_OMEGA * (r[s] - (first ? 0.f : row(L, x, s, c))) / dg[s]);
      out[c] = xc;
    }
    __syncthreads();
  }
  __device__ __forceinline__ void gs(const Level& L, float* x, int colour, bool first) const {
#pragma clang fp contract(off)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (par[s] < 0) continue;
      const int c = (int)threadIdx.x + s * TAIL_THREADS;
      if (first) x[c] = par[s] == colour && dg[s] > 0.f ? SV::rnd(r[s] / dg[s]) : 0.f;
      else if (par[s] == colour && dg[s] > 0.f) x[c] = SV::rnd(x[c] + (r[s] - row(L, x, s, c)) / dg[s]);
    }
    __syncthreads();
  }
  __device__ __forceinline__ void residual(const Level& L, const float* x, float* out) const {
#pragma clang fp contract(off)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (par[s] < 0) continue;
      const int c = (int)threadIdx.x + s * TAIL_THREADS;
      out[c] = r[s] - row(L, x, s, c);
    }
    __syncthreads();
  }
};

// coarse_cycle3 (delta3d_multigrid.rs:303-332) over the tail levels; the
// first level's r is restricted, its x is written back.
template <int ST>
__global__ void __launch_bounds__(TAIL_THREADS) k_r6_tail(TailSet T, Ctl* ctl) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  if (!ctl->active) return;
  extern __shared__ float lds[];
  const int tid = (int)threadIdx.x, last = T.count - 1;
  const bool jacobi = T.smoother == 0;
  // buffers of level l: x at 3 base, the other at 3 base + n, r at 3 base + 2 n
  for (int q = tid; q < (int)T.lv[0].n; q += TAIL_THREADS)
    lds[2 * (int)T.lv[0].n + q] = SV::ld(reinterpret_cast<const typename SV::T*>(T.lv[0].r), q);
  __syncthreads();
  float* xl = nullptr;  // the iterate of the level below (going up)
  int base = 0;         // cells of the levels above
  for (int step = 0; step <= 2 * last; ++step) {
    const bool down = step <= last;
    const int l = down ? step : 2 * last - step;
    const Level L = T.lv[l];
    const int n = (int)L.n;
    if (!down) base -= n;
    float* buf[2] = {lds + 3 * base, lds + 3 * base + n};
    float* r = lds + 3 * base + 2 * n;
    const int count = l == last ? T.coarse : down ? T.pre : T.post;
    // which buffer a level's iterate is in after its sweeps on the way down
    const int pre_at = jacobi && T.pre > 0 ? (T.pre - 1) & 1 : 0;
    int at = down ? 1 : pre_at;  // from zero, the first Jacobi sweep writes buffer 0
    R6Cells<ST> cells;
    cells.load(L, r);
    if (!down) {
      const Level C = T.lv[l + 1];
      for (int c = tid; c < n; c += TAIL_THREADS) {
        int i, j, k;
        ldecode(L, c, i, j, k);
        buf[at][c] = SV::rnd(buf[at][c] + xl[((k >> 1) * C.ny + (j >> 1)) * C.nx + (i >> 1)]);
      }
      __syncthreads();
    }
    if (jacobi) {
      for (int s = 0; s < count; ++s) {
        cells.jacobi(L, buf[at], buf[at ^ 1], down && s == 0);
        at ^= 1;
      }
    } else {
      at = 0;
      const int passes = sweep_passes(l == last, count);
      for (int p = 0; p < passes; ++p) cells.gs(L, buf[0], sweep_colour(l == last, down, count, p), down && p == 0);
    }
    if (down && count == 0) {
      at = 0;
      for (int c = tid; c < n; c += TAIL_THREADS) buf[0][c] = 0.f;
      __syncthreads();
    }
    xl = buf[at];
    if (down && l < last) {
      const Level C = T.lv[l + 1];
      float* res = buf[at ^ 1];
      cells.residual(L, buf[at], res);
      float* rc = lds + 3 * (base + n) + 2 * (int)C.n;
      for (int c = tid; c < (int)C.n; c += TAIL_THREADS) {
        int i, j, k;
        ldecode(C, c, i, j, k);
        float s = 0.f;
#pragma unroll
        for (int ch = 0; ch < 8; ++ch)
          s += res[((2 * k + (ch >> 2)) * L.ny + 2 * j + ((ch >> 1) & 1)) * L.nx + 2 * i + (ch & 1)];
        rc[c] = SV::rnd(0.125f * s);
      }
      __syncthreads();
      base += n;
    }
  }
  for (int q = tid; q < (int)T.lv[0].n; q += TAIL_THREADS)
    SV::st(reinterpret_cast<typename SV::T*>(T.lv[0].x), q, xl[q]);
}

// LDS bytes k_r6_tail needs for the given levels.
inline size_t r6_tail_lds_bytes(const Level* lv, int count) {
  size_t floats = 0;
  for (int l = 0; l < count; ++l) floats += 3 * lv[l].n;
  return floats * sizeof(float);
}

}  // namespace fsp
