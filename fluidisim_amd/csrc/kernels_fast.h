// Fast path of the fine level and of the small coarse levels.
//
// Fine level ("quad" kernels, nx % 4 == 0): one thread owns four consecutive
// cells along x, so every lane of a wavefront is busy in both colours of a
// red-black pass and every access is a 16-byte vector access; x neighbours
// across quads come from the adjacent lane by wavefront shuffle, y and z
// neighbours are vector loads served mostly by L2. The 1-D grid is mapped to
// (x-segment, y-block, z) tiles in dispatch order (see xcd_block). Per-cell arithmetic
// is the fine operator's (face order x-, x+, y-, y+, z-, z+, no contraction),
// so results equal the generic kernels bit for bit.
//
// Small coarse levels: one workgroup runs every level below a size threshold
// with the vectors and coefficients in LDS, replacing dozens of tiny launches
// per V-cycle by one.
#pragma once
#include "kernels.h"

namespace fsp {

constexpr int QBLOCK = 256;
// Minimum workgroups per CU the fine red-black kernel is compiled for (the
// register budget follows from it).
#ifndef FSP_QGS_MIN_BLOCKS
#define FSP_QGS_MIN_BLOCKS 1
#endif
// Widest x extent of a workgroup tile, in quads (tile shapes for tuning).
#ifndef FSP_QX_MAX
#define FSP_QX_MAX 64
#endif

struct QuadGrid {
  int nq;   // quads per row (nx / 4)
  int QX;   // threads along x per block (power of two, <= 64)
  int RY;   // rows per block (QBLOCK / QX)
  int nbx;  // blocks along x
  int nby;  // blocks along y (over `rows`)
  int rows; // rows covered (ny, or ny/2 for the restriction)
  int planes;
  int sx;                     // log2 QX
  unsigned long long mx, my;  // divisions by nbx and nby (block_divisor)
};
// a / d = a * block_divisor(d) >> 40 for a < 2^20, d <= 2^20 (a grid has
// 65536 blocks at most): the divisions of the block number cost every
// workgroup some 200 cycles before its first load.
inline unsigned long long block_divisor(int d) { return ((1ull << 40) + (unsigned)d - 1) / (unsigned)d; }
__host__ __device__ inline unsigned block_quotient(unsigned a, unsigned long long m) { return (unsigned)(a * m >> 40); }

// Workgroups of `threads` threads, QX of them along x.
inline QuadGrid quad_grid(int nq, int rows, int planes, int qx, int threads) {
  QuadGrid Q{};
  Q.nq = nq; Q.QX = qx; Q.RY = threads / qx;
  Q.nbx = (nq + qx - 1) / qx;
  Q.nby = (rows + Q.RY - 1) / Q.RY;
  Q.rows = rows; Q.planes = planes;
  while (1 << Q.sx < qx) ++Q.sx;
  Q.mx = block_divisor(Q.nbx > 0 ? Q.nbx : 1);
  Q.my = block_divisor(Q.nby > 0 ? Q.nby : 1);
  return Q;
}
// The widest workgroups that rows of nq quads fill.
inline QuadGrid quad_grid(int nq, int rows, int planes) {
  int qx = 1;
  while (qx < nq && qx < FSP_QX_MAX) qx <<= 1;
  return quad_grid(nq, rows, planes, qx, QBLOCK);
}
// The restriction's grid for 128-thread halves (k_q_restrict2, k_gc_restrict2).
inline QuadGrid half_grid(const QuadGrid& Q) { return quad_grid(Q.nq, Q.rows, Q.planes, Q.QX, QBLOCK / 2); }
// Block L of the grid: bx, by, plane.
__device__ __forceinline__ void quad_block(const QuadGrid& Q, unsigned L, unsigned& bx, unsigned& by, int& plane) {
  const unsigned t = block_quotient(L, Q.mx);
  const unsigned z = block_quotient(t, Q.my);
  bx = L - t * (unsigned)Q.nbx;
  by = t - z * (unsigned)Q.nby;
  plane = (int)z;
}

// Tile coordinates of this thread; returns false for lanes past the edge
// (they still take part in shuffles).
struct BrickGrid {
  int bx, by, bz;             // bricks along x, y, z
  unsigned long long mx, mz;  // divisions by bx and bz (block_divisor)
};

__device__ __forceinline__ bool quad_coords(const QuadGrid& Q, int& qx, int& y, int& z) {
  unsigned bx, by;
  quad_block(Q, xcd_block(blockIdx.x, gridDim.x), bx, by, z);
  qx = ((int)bx << Q.sx) + (int)(threadIdx.x & (unsigned)(Q.QX - 1));
  y = (int)by * Q.RY + (int)(threadIdx.x >> Q.sx);
  return qx < Q.nq && y < Q.rows && z < Q.planes;
}

// A wet cell among the block's quads (a load like that of ctl->active, in
// flight with it). Kernels that a dry block leaves at once skip the air over a
// free surface: the projection of a 256x256x128 tank half full takes 4.08 ms
// with every block at work, 3.41 without the dry ones.
__device__ __forceinline__ uint32_t block_wet(const Fine& G) { return G.wetq[xcd_block(blockIdx.x, gridDim.x)]; }
// ctl->active, read together with the flag (else the compiler reads one after the other).
__device__ __forceinline__ bool loop_active(const Ctl* ctl, uint32_t& wet) {
  int32_t active = ctl->active;
  asm volatile("" : "+s"(active), "+s"(wet));
  return active != 0;
}
__device__ __forceinline__ void zero_partial(int op, double* partials) {
  if (threadIdx.x != 0) return;
  double* part = partials + (size_t)op * MAX_PARTIALS * 2;
  part[2 * blockIdx.x] = 0.0;
  part[2 * blockIdx.x + 1] = 0.0;
}

__device__ __forceinline__ float q_get(const float4& v, int e) { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; }
__device__ __forceinline__ void q_set(float4& v, int e, float x) {
  if (e == 0) v.x = x; else if (e == 1) v.y = x; else if (e == 2) v.z = x; else v.w = x;
}
__device__ __forceinline__ float4 ld4(const float* p, size_t c) { return *reinterpret_cast<const float4*>(p + c); }
__device__ __forceinline__ void st4(float* p, size_t c, const float4& v) { *reinterpret_cast<float4*>(p + c) = v; }
__device__ __forceinline__ float4 f4zero() { return make_float4(0.f, 0.f, 0.f, 0.f); }

// The sum of a free-surface row (about one row in a hundred); FORM as ghost_row.
template <int FORM = FORM_GENERAL>
__device__ __forceinline__ float ghost_row_sum(const Fine& G, int i, int j, int k, uint8_t m, float pc, const float nb[6],
                                            float& prec) {
#pragma clang fp contract(off)
  uint8_t type[6];
  float it[6], a[6];
  ghost_row<FORM>(G, i, j, k, m, type, it, a);
  float acc = 0.f, diag = 0.f;
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    if (type[f] == 1) { acc += a[f] * (pc - nb[f]); diag += a[f]; }
    else if (type[f] == 2) { acc += a[f] * pc * it[f]; diag += a[f] * it[f]; }
  }
  prec = diag > 0.f ? 1.0f / (diag * G.inv) : 0.f;
  return acc;
}

// Row of the fine operator from neighbour values already in registers, in the
// reference's face order; prec as rhs_mobile3 computes it (FORM as ghost_row).
template <int FORM = FORM_GENERAL>
__device__ __forceinline__ float row_local(const Fine& G, int i, int j, int k, uint8_t m, float pc, const float nb[6],
                                          float& prec) {
#pragma clang fp contract(off)
  prec = 0.f;
  if (!(m & M_WET)) return 0.f;
  float acc = 0.f;
  if (!(m & M_GHOST)) {
#pragma unroll
    for (int f = 0; f < 6; ++f)
      if (m & (1u << f)) acc += pc - nb[f];
    prec = G.prec_tab[__popc(m & 0x3Fu)];
  } else {
    acc = ghost_row_sum<FORM>(G, i, j, k, m, pc, nb, prec);
  }
  return acc * G.inv;
}

// A plain row's sum over its coupled faces (row code m), branch-free.
__device__ __forceinline__ float plain_sum(uint32_t m, float pc, const float nb[6]) {
#pragma clang fp contract(off)
  float acc = 0.f;
#pragma unroll
  for (int f = 0; f < 6; ++f) acc = (m & (1u << f)) ? acc + (pc - nb[f]) : acc;
  return acc;
}
// ghost_row_sum from a ghost row's entry: of its column's table (column col,
// layer k; apertures 1) or of the index (entry n).
struct GhostEntry {
  float it[6], a[6];
};
template <int FORM>
__device__ __forceinline__ GhostEntry ghost_load(const Fine& G, size_t col, int k, uint32_t n) {
  GhostEntry g;
  const float4* e = reinterpret_cast<const float4*>(FORM == FORM_INDEX ? G.gent + (size_t)n * GE_FLOATS
                                                                       : ghost_entry(G, col, k));
  const float4 x = e[0];
  g.it[0] = x.x; g.it[1] = x.y; g.it[2] = x.z; g.it[3] = x.w;
  if (FORM == FORM_INDEX) {
    const float4 y = e[1], z = e[2];
    g.it[4] = y.x; g.it[5] = y.y;
    g.a[0] = y.z; g.a[1] = y.w; g.a[2] = z.x; g.a[3] = z.y; g.a[4] = z.z; g.a[5] = z.w;
  } else {
    const float2 y = *reinterpret_cast<const float2*>(e + 1);
    g.it[4] = y.x; g.it[5] = y.y;
#pragma unroll
    for (int f = 0; f < 6; ++f) g.a[f] = 1.0f;
  }
  return g;
}
__device__ __forceinline__ float ghost_sum(const GhostEntry& g, uint32_t m, float pc, const float nb[6], float inv,
                                           float& prec) {
#pragma clang fp contract(off)
  float acc = 0.f, diag = 0.f;
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const bool one = (m & (1u << f)) != 0, two = !one && g.it[f] > 0.f;
    const float t = one ? g.a[f] * (pc - nb[f]) : g.a[f] * pc * g.it[f], d = one ? g.a[f] : g.a[f] * g.it[f];
    acc = (one || two) ? acc + t : acc;
    diag = (one || two) ? diag + d : diag;
  }
  prec = diag > 0.f ? 1.0f / (diag * inv) : 0.f;
  return acc;
}

// The rows (A x)_c of a quad's four cells from values in registers: zc and
// its x neighbours left and right, ym .. zp the quads around it. The plain
// rows first, without branches; a quad with free-surface rows then loads the
// four cells' table entries in one round (a row at a time, each after a look
// at its column, held a wavefront for up to eight rounds of memory latency,
// which a small grid has nothing to hide behind).
template <int FORM>
__device__ __forceinline__ void quad_rows(const Fine& G, int x0, int y, int k, uint32_t mq, const float4& zc, float left,
                                          float right, const float4& ym, const float4& yp, const float4& zm,
                                          const float4& zp, float row[4]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t m = (mq >> (8 * e)) & 0xFFu;
    const float nb[6] = {e == 0 ? left : q_get(zc, e - 1), e == 3 ? right : q_get(zc, e + 1),
                         q_get(ym, e), q_get(yp, e), q_get(zm, e), q_get(zp, e)};
    row[e] = (m & M_WET) ? plain_sum(m, q_get(zc, e), nb) * G.inv : 0.f;
  }
  const uint32_t ghosts = mq & 0x80808080u;
  if (!ghosts) return;
  // (index entries hold apertures too: two cells at a time keep the registers)
  constexpr int W = FORM == FORM_INDEX ? 2 : 4;
  const size_t col = (size_t)y * G.nx + x0;
  const uint32_t first = FORM == FORM_INDEX ? G.gq[((size_t)k * G.nx * G.ny + col) >> 2] : 0u;
#pragma unroll
  for (int e0 = 0; e0 < 4; e0 += W) {
    GhostEntry g[W];
    if (FORM != FORM_GENERAL)
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (FORM == FORM_TABLE || (ghosts & (0x80u << (8 * (e0 + w)))))
          g[w] = ghost_load<FORM>(G, col + e0 + w, k, ghost_index(G, mq, first, e0 + w));
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int e = e0 + w;
      if (!(ghosts & (0x80u << (8 * e)))) continue;
      const uint32_t m = (mq >> (8 * e)) & 0xFFu;
      const float pc = q_get(zc, e);
      const float nb[6] = {e == 0 ? left : q_get(zc, e - 1), e == 3 ? right : q_get(zc, e + 1),
                           q_get(ym, e), q_get(yp, e), q_get(zm, e), q_get(zp, e)};
      float prec;
      row[e] = FORM == FORM_GENERAL ? row_local<FORM>(G, x0 + e, y, k, (uint8_t)m, pc, nb, prec)
                                    : ghost_sum(g[w], m, pc, nb, G.inv, prec) * G.inv;
    }
  }
}

// The four cells' x neighbours: within the quad, from the adjacent lanes, or
// (at the edge of a lane segment) from memory through `edge`.
// Every lane takes part in the shuffles; only valid lanes read memory.
template <class Edge>
__device__ __forceinline__ void x_neighbours(const QuadGrid& Q, bool valid, int qx, const float4& v, float& left,
                                             float& right, Edge edge) {
  const float l_sh = __shfl_up(v.w, 1, 64);
  const float r_sh = __shfl_down(v.x, 1, 64);
  const int lane_in_seg = (int)(threadIdx.x & (unsigned)(Q.QX - 1));
  left = 0.f;
  right = 0.f;
  if (!valid) return;
  if (qx > 0) left = lane_in_seg > 0 ? l_sh : edge(-1);
  if (qx + 1 < Q.nq) right = (lane_in_seg < Q.QX - 1) ? r_sh : edge(4);
}

// ---------------------------------------------------------------- red-black pass
// One colour of a red-black Gauss-Seidel sweep on quads, in place (the first
// pass from z = 0 is fused with the second in k_q_gs_first).
// MODE 2: z is first prolonged from the first coarse level (z += x_c of the
//         parent, 0 on rows with prec == 0), then the colour is updated;
//         neighbours are prolonged on the fly, so this mode reads z and
//         writes zout (a different buffer).
// dot_op >= 0: also reduce <r, z> over every cell into that slot.
// z, zout and the parents xc are held in storage ST (r is the f32 CG
// residual); every value entering the arithmetic is a stored value.
template <int MODE, int ST, int FORM = FORM_GENERAL>
__global__ void __launch_bounds__(QBLOCK, FSP_QGS_MIN_BLOCKS) k_q_gs(Fine G, QuadGrid Q, const typename Store<ST>::T* z,
                                                 typename Store<ST>::T* zout, const float* r, int colour, Level L0,
                                                 const typename Store<ST>::T* xc, int dot_op, Ctl* ctl,
                                                 double* partials) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  if (!ctl->active) return;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  const size_t plane = (size_t)G.nx * G.ny;
  const size_t c0 = valid ? ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx : 0;
  double s = 0.0, unused = 0.0;
  static_assert(MODE == 0 || MODE == 2, "in place, or prolongation then update");
  // parent values of the prolongation
  auto parent = [&](int yy, int kk, int xq) -> float2 { return SV::ld2(xc, lidx(L0, 2 * xq, yy >> 1, kk >> 1)); };
  // prolongation z + parent, rounded to storage (prolong_add3 stores it)
  auto prolong = [&](float4& v, float2 a) {
    v.x = SV::rnd(v.x + a.x); v.y = SV::rnd(v.y + a.x); v.z = SV::rnd(v.z + a.y); v.w = SV::rnd(v.w + a.y);
  };
  float4 zc = f4zero(), rq = f4zero();
  uint32_t mq = 0;
  float4 ym = f4zero(), yp = f4zero(), zm = f4zero(), zp = f4zero();
  if (valid) {
    mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    zc = SV::ld4(z, c0);
    rq = ld4(r, c0);
    if (y > 0) ym = SV::ld4(z, c0 - G.nx);
    if (y + 1 < G.ny) yp = SV::ld4(z, c0 + G.nx);
    if (k > 0) zm = SV::ld4(z, c0 - plane);
    if (k + 1 < G.nz) zp = SV::ld4(z, c0 + plane);
    if (MODE == 2) {
      prolong(zc, parent(y, k, qx));
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!prec_positive((uint8_t)(mq >> (8 * e)))) q_set(zc, e, 0.f);
      if (y > 0) prolong(ym, parent(y - 1, k, qx));
      if (y + 1 < G.ny) prolong(yp, parent(y + 1, k, qx));
      if (k > 0) prolong(zm, parent(y, k - 1, qx));
      if (k + 1 < G.nz) prolong(zp, parent(y, k + 1, qx));
    }
  }
  float left, right;
  x_neighbours(Q, valid, qx, zc, left, right, [&](int off) {
    float v = SV::ld(z, c0 + off);
    if (MODE == 2) {
      const int xx = 4 * qx + off;
      v = SV::rnd(v + SV::ld(xc, lidx(L0, xx >> 1, y >> 1, k >> 1)));
    }
    return v;
  });
  if (valid) {
    float4 out = zc;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (((e + y + k) & 1) != colour) continue;
      const uint8_t m = (uint8_t)(mq >> (8 * e));
      const float pc = q_get(zc, e);
      const float xl = e == 0 ? left : q_get(zc, e - 1);
      const float xr = e == 3 ? right : q_get(zc, e + 1);
      const float nb[6] = {xl, xr, q_get(ym, e), q_get(yp, e), q_get(zm, e), q_get(zp, e)};
      float prec;
      const float az = row_local<FORM>(G, 4 * qx + e, y, k, m, pc, nb, prec);
      if (prec > 0.f) q_set(out, e, SV::rnd(pc + prec * (q_get(rq, e) - az)));
    }
    SV::st4(zout, c0, out);
    if (dot_op >= 0) s = (double)rq.x * out.x + (double)rq.y * out.y + (double)rq.z * out.z + (double)rq.w * out.w;
  }
  if (dot_op >= 0) reduce_finish<false>(s, unused, dot_op, ctl, partials);
}

// The first two passes of the pre-smoothing from z = 0 in one launch: the
// colour-0 pass from zero is local (colour-0 cells row_prec * r, colour-1
// cells 0), so the colour-1 pass recomputes those values for its neighbours
// from r and the per-cell row_prec (k_prec) instead of reading them back.
// Every value is the one the two single passes store, so the result is
// theirs bit for bit, for one pass's traffic plus the row_prec reads (a
// variant deriving plain rows' factor from the row code ran slower).
template <int ST, int FORM = FORM_GENERAL>
__global__ void __launch_bounds__(QBLOCK, FSP_QGS_MIN_BLOCKS) k_q_gs_first(Fine G, QuadGrid Q,
                                                                         typename Store<ST>::T* zout, const float* r,
                                                                         Ctl* ctl) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  uint32_t wet = block_wet(G);
  if (!loop_active(ctl, wet)) return;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  const size_t plane = (size_t)G.nx * G.ny;
  const size_t c0 = valid ? ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx : 0;
  if (!wet) {
    if (valid) SV::st4(zout, c0, f4zero());
    return;
  }
  // the first pass's value of cell (x, yy, kk): row_prec * r on colour 0
  auto first = [&](int x, int yy, int kk, float prec, float rv) -> float {
    if (((x + yy + kk) & 1) != 0) return 0.f;
    return prec > 0.f ? SV::rnd(prec * rv) : 0.f;
  };
  auto first4 = [&](const float4& pq, const float4& rq4, int yy, int kk) {
    float4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) q_set(v, e, first(4 * qx + e, yy, kk, q_get(pq, e), q_get(rq4, e)));
    return v;
  };
  float4 rq = f4zero(), zc = f4zero(), ym = f4zero(), yp = f4zero(), zm = f4zero(), zp = f4zero();
  uint32_t mq = 0;
  if (valid) {
    // every load first, then the values
    mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    rq = ld4(r, c0);
    const float4 pc = ld4(G.precv, c0);
    const bool hym = y > 0, hyp = y + 1 < G.ny, hzm = k > 0, hzp = k + 1 < G.nz;
    const size_t cym = c0 - G.nx, cyp = c0 + G.nx, czm = c0 - plane, czp = c0 + plane;
    const float4 r_ym = hym ? ld4(r, cym) : f4zero(), p_ym = hym ? ld4(G.precv, cym) : f4zero();
    const float4 r_yp = hyp ? ld4(r, cyp) : f4zero(), p_yp = hyp ? ld4(G.precv, cyp) : f4zero();
    const float4 r_zm = hzm ? ld4(r, czm) : f4zero(), p_zm = hzm ? ld4(G.precv, czm) : f4zero();
    const float4 r_zp = hzp ? ld4(r, czp) : f4zero(), p_zp = hzp ? ld4(G.precv, czp) : f4zero();
    zc = first4(pc, rq, y, k);
    if (hym) ym = first4(p_ym, r_ym, y - 1, k);
    if (hyp) yp = first4(p_yp, r_yp, y + 1, k);
    if (hzm) zm = first4(p_zm, r_zm, y, k - 1);
    if (hzp) zp = first4(p_zp, r_zp, y, k + 1);
  }
  float left, right;
  x_neighbours(Q, valid, qx, zc, left, right, [&](int off) {
    const size_t c = c0 + off;
    return first(4 * qx + off, y, k, G.precv[c], r[c]);
  });
  if (!valid) return;
  // the colour-1 cells: x-cells par and par + 2, par = 1 on even rows
  const bool odd = ((y + k) & 1) == 0;
  auto sel = [odd](float o, float e) -> float { return odd ? o : e; };
  const uint32_t m2[2] = {(mq >> (odd ? 8 : 0)) & 0xFFu, (mq >> (odd ? 24 : 16)) & 0xFFu};
  const float pc2[2] = {sel(zc.y, zc.x), sel(zc.w, zc.z)}, r2[2] = {sel(rq.y, rq.x), sel(rq.w, rq.z)};
  const float nb2[2][6] = {{sel(zc.x, left), sel(zc.z, zc.y), sel(ym.y, ym.x), sel(yp.y, yp.x), sel(zm.y, zm.x), sel(zp.y, zp.x)},
                           {sel(zc.z, zc.y), sel(right, zc.w), sel(ym.w, ym.z), sel(yp.w, yp.z), sel(zm.w, zm.z), sel(zp.w, zp.z)}};
  float v2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float prec = (m2[h] & M_WET) ? G.prec_tab[__popc(m2[h] & 0x3Fu)] : 0.f;
    v2[h] = prec > 0.f ? SV::rnd(pc2[h] + prec * (r2[h] - plain_sum(m2[h], pc2[h], nb2[h]) * G.inv)) : pc2[h];
  }
  if ((m2[0] | m2[1]) & M_GHOST) {
    GhostEntry g[2];
    const size_t col = (size_t)y * G.nx + 4 * qx + (odd ? 1 : 0);
    const uint32_t first = FORM == FORM_INDEX ? G.gq[c0 >> 2] : 0u;
    if (FORM != FORM_GENERAL)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (FORM == FORM_TABLE || (m2[h] & M_GHOST))
          g[h] = ghost_load<FORM>(G, col + 2 * h, k, ghost_index(G, mq, first, (odd ? 1 : 0) + 2 * h));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!(m2[h] & M_GHOST)) continue;
      float prec, az;
      if (FORM == FORM_GENERAL)
        az = row_local<FORM>(G, 4 * qx + (odd ? 1 : 0) + 2 * h, y, k, (uint8_t)m2[h], pc2[h], nb2[h], prec);
      else az = ghost_sum(g[h], m2[h], pc2[h], nb2[h], G.inv, prec) * G.inv;
      v2[h] = prec > 0.f ? SV::rnd(pc2[h] + prec * (r2[h] - az)) : pc2[h];
    }
  }
  const float4 out = make_float4(sel(zc.x, v2[0]), sel(v2[0], zc.y), sel(zc.z, v2[1]), sel(v2[1], zc.w));
  SV::st4(zout, c0, out);
}

// ---------------------------------------------------------------- fused red-black sweep on bricks
// Both colour passes of a red-black sweep in one launch, one brick per
// workgroup: z of the brick (BR_QX quads x BR_Y rows x BR_Z planes) and a
// halo of one quad in x and two cells in y and z is loaded into LDS at once;
// pass c runs over the brick and a ring of one cell (its neighbours are
// colour 1 - c values, untouched by it) back into LDS; after a barrier pass
// 1 - c runs over the brick (its neighbours are the colour-c values, all
// updated) and is stored to zout. Bricks are independent (zout must not
// alias zin), so many of them per CU overlap their loads with each other's
// arithmetic. Every cell's update uses the operands the single-colour passes
// use, in the same order: the sweep equals k_q_gs twice bit for bit.
// MODE 2: every value read from zin is first prolonged from the first coarse
// level (z + parent, rounded to storage), rows with prec == 0 become 0
// (prolong_add3 then the dry reset), as k_q_gs<2> does before its pass.
// dot_op >= 0: <r, z> of the result over every cell into that slot.
// Traffic per cell: mask, z, r in, z out (13 B in f32 storage), against
// twice that for two single passes.
#ifndef FSP_BRICK_XCD
#define FSP_BRICK_XCD 1
#endif
#ifndef FSP_BRICK_QX
#define FSP_BRICK_QX 8
#endif
#ifndef FSP_BRICK_Y
#define FSP_BRICK_Y 8
#endif
#ifndef FSP_BRICK_Z
#define FSP_BRICK_Z 8
#endif
constexpr int BR_QX = FSP_BRICK_QX, BR_Y = FSP_BRICK_Y, BR_Z = FSP_BRICK_Z;
#ifndef FSP_BRICK_THREADS
#define FSP_BRICK_THREADS 512
#endif
constexpr int BR_THREADS = FSP_BRICK_THREADS;
constexpr int BR_LQ = BR_QX + 2;                   // quads per LDS row
constexpr int BR_LX = 4 * BR_LQ;                   // floats per LDS row
constexpr int BR_LY = BR_Y + 4, BR_LZ = BR_Z + 4;  // LDS rows, planes
constexpr int BR_PAD = 4;                          // floats before and after (halo cells' unused reads)
constexpr int BR_FLOATS = BR_LX * BR_LY * BR_LZ + 2 * BR_PAD;
constexpr int BR_NLOAD = BR_LQ * BR_LY * BR_LZ;
constexpr int BR_LOADS = (BR_NLOAD + BR_THREADS - 1) / BR_THREADS;
constexpr int BR_NA = BR_LQ * (BR_Y + 2) * (BR_Z + 2);  // first-pass quads
constexpr int BR_AITEMS = (BR_NA + BR_THREADS - 1) / BR_THREADS;
constexpr int BR_NB = BR_QX * BR_Y * BR_Z;  // second-pass quads
constexpr int BR_BITEMS = (BR_NB + BR_THREADS - 1) / BR_THREADS;


template <int MODE, int ST, int FORM = FORM_GENERAL>
__global__ void __launch_bounds__(BR_THREADS) k_q_brick(Fine G, BrickGrid B, const typename Store<ST>::T* zin,
                                                        typename Store<ST>::T* zout, const float* r, int colour,
                                                        Level L0, const typename Store<ST>::T* xc, int dot_op,
                                                        Ctl* ctl, double* partials) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  static_assert(MODE == 0 || MODE == 2, "in place, or prolongation then the sweep");
  __shared__ __attribute__((aligned(16))) float zs_all[BR_FLOATS];
  __shared__ float s_prec[8];
  __shared__ double s_red[BR_THREADS / 64];
  float* zs = zs_all + BR_PAD;
  const int nx = G.nx, ny = G.ny, nz = G.nz;
  const int tid = (int)threadIdx.x;
  // Bricks in x, then z, then y order, each XCD taking a contiguous range of
  // them (dispatch deals workgroups to the 8 XCDs in turn): bricks that share
  // halo planes and rows run on one XCD close in time, so their halos come
  // from that XCD's L2.
  const unsigned G8 = gridDim.x / 8u;
  const unsigned bl = (FSP_BRICK_XCD && gridDim.x % 8u == 0u) ? (blockIdx.x % 8u) * G8 + blockIdx.x / 8u : blockIdx.x;
  const int t = (int)block_quotient(bl, B.mx), bxi = (int)bl - t * B.bx;
  const int byi = (int)block_quotient((unsigned)t, B.mz), bzi = t - byi * B.bz;
  const int qx0 = bxi * BR_QX - 1, y0 = byi * BR_Y - 2, z0 = bzi * BR_Z - 2;  // LDS origin (quad, row, plane)
  const int nq = nx / 4;
  uint32_t wet = G.wetb[bl];
  if (!loop_active(ctl, wet)) return;
  if (!wet) {
    for (int idx = tid; idx < BR_NB; idx += BR_THREADS) {
      const int q = qx0 + 1 + idx % BR_QX, y = y0 + 2 + idx / BR_QX % BR_Y, k = z0 + 2 + idx / (BR_QX * BR_Y);
      if (q < nq && y < ny && k < nz) SV::st4(zout, ((size_t)k * ny + y) * nx + 4 * (size_t)q, f4zero());
    }
    if (dot_op >= 0) zero_partial(dot_op, partials);
    return;
  }
  if (tid < 8) s_prec[tid] = tid < 7 ? G.prec_tab[tid] : 0.f;
  // every load of the workgroup in flight first: z of the brick and its halo
  // (prolonged in MODE 2), then r and the row codes of both passes' quads
  float4 rqa[BR_AITEMS], rqb[BR_BITEMS];
  uint32_t mqa[BR_AITEMS], mqb[BR_BITEMS];
  bool ona[BR_AITEMS], onb[BR_BITEMS];
  {
    float4 v[BR_LOADS];
#pragma unroll
    for (int m = 0; m < BR_LOADS; ++m) {
      const int idx = tid + BR_THREADS * m;
      const int lq = idx % BR_LQ, rest = idx / BR_LQ, ly = rest % BR_LY, lz = rest / BR_LY;
      const int q = qx0 + lq, y = y0 + ly, k = z0 + lz;
      v[m] = f4zero();
      if (idx < BR_NLOAD && q >= 0 && q < nq && y >= 0 && y < ny && k >= 0 && k < nz) {
        const size_t c = ((size_t)k * ny + y) * nx + 4 * (size_t)q;
        v[m] = SV::ld4(zin, c);
        if (MODE == 2) {
          const float2 a = SV::ld2(xc, lidx(L0, 2 * q, y >> 1, k >> 1));
          v[m].x = SV::rnd(v[m].x + a.x); v[m].y = SV::rnd(v[m].y + a.x);
          v[m].z = SV::rnd(v[m].z + a.y); v[m].w = SV::rnd(v[m].w + a.y);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < BR_AITEMS; ++m) {
      const int idx = tid + BR_THREADS * m;
      const int lq = idx % BR_LQ, rest = idx / BR_LQ, ly = 1 + rest % (BR_Y + 2), lz = 1 + rest / (BR_Y + 2);
      const int q = qx0 + lq, y = y0 + ly, k = z0 + lz;
      ona[m] = idx < BR_NA && q >= 0 && q < nq && y >= 0 && y < ny && k >= 0 && k < nz;
      rqa[m] = f4zero();
      mqa[m] = 0;
      if (ona[m]) {
        const size_t c = ((size_t)k * ny + y) * nx + 4 * (size_t)q;
        rqa[m] = ld4(r, c);
        mqa[m] = *reinterpret_cast<const uint32_t*>(G.mask + c);
      }
    }
#pragma unroll
    for (int m = 0; m < BR_BITEMS; ++m) {
      const int idx = tid + BR_THREADS * m;
      const int lq = 1 + idx % BR_QX, rest = idx / BR_QX, ly = 2 + rest % BR_Y, lz = 2 + rest / BR_Y;
      const int q = qx0 + lq, y = y0 + ly, k = z0 + lz;
      onb[m] = idx < BR_NB && q < nq && y < ny && k < nz;
      rqb[m] = f4zero();
      mqb[m] = 0;
      if (onb[m]) {
        const size_t c = ((size_t)k * ny + y) * nx + 4 * (size_t)q;
        rqb[m] = ld4(r, c);
        mqb[m] = *reinterpret_cast<const uint32_t*>(G.mask + c);
      }
    }
#pragma unroll
    for (int m = 0; m < BR_LOADS; ++m) {
      const int idx = tid + BR_THREADS * m;
      if (idx < BR_NLOAD) *reinterpret_cast<float4*>(zs + 4 * idx) = v[m];
    }
  }
  // One colour on the quad at LDS (lq, ly, lz): the colour's two cells
  // (x-cells par and par + 2) without branches on plain rows; free-surface
  // cells are left as they are and flagged in `late` (bits e) for
  // relax_late. Returns the quad with the colour's plain cells updated.
  auto relax = [&](int lq, int ly, int lz, int col, const float4 rq, uint32_t mq, uint32_t& late) -> float4 {
    const int q = qx0 + lq, y = y0 + ly, k = z0 + lz;
    const float* sc = zs + ((lz * BR_LY + ly) * BR_LX + 4 * lq);
    const float4 zc = *reinterpret_cast<const float4*>(sc);
    const float4 ym = *reinterpret_cast<const float4*>(sc - BR_LX);
    const float4 yp = *reinterpret_cast<const float4*>(sc + BR_LX);
    const float4 zm = *reinterpret_cast<const float4*>(sc - BR_LX * BR_LY);
    const float4 zp = *reinterpret_cast<const float4*>(sc + BR_LX * BR_LY);
    // the x neighbours' quads as whole 16-byte reads (scalar reads 16 bytes
    // apart would conflict in the LDS banks)
    const float4 xl4 = *reinterpret_cast<const float4*>(sc - 4);
    const float4 xr4 = *reinterpret_cast<const float4*>(sc + 4);
    const float left = q > 0 ? xl4.w : 0.f, right = q + 1 < nq ? xr4.x : 0.f;
    const bool odd = ((col + y + k) & 1) != 0;
    auto sel = [odd](float o, float e) -> float { return odd ? o : e; };
    auto cell = [&](float pc, float xl, float xr, float vym, float vyp, float vzm, float vzp, float rc,
                    uint32_t mc) -> float {
      const float nb[6] = {xl, xr, vym, vyp, vzm, vzp};
      float acc = 0.f;
#pragma unroll
      for (int f = 0; f < 6; ++f) acc = (mc & (1u << f)) ? acc + (pc - nb[f]) : acc;
      const float prec = s_prec[(mc & M_WET) ? __popc(mc & 0x3Fu) : 0];
      const float v = prec > 0.f ? SV::rnd(pc + prec * (rc - acc * G.inv)) : (MODE == 2 ? 0.f : pc);
      return (mc & M_GHOST) ? pc : v;
    };
    const uint32_t ma = (mq >> (odd ? 8 : 0)) & 0xFFu, mb = (mq >> (odd ? 24 : 16)) & 0xFFu;
    const float a = cell(sel(zc.y, zc.x), sel(zc.x, left), sel(zc.z, zc.y), sel(ym.y, ym.x), sel(yp.y, yp.x),
                         sel(zm.y, zm.x), sel(zp.y, zp.x), sel(rq.y, rq.x), ma);
    const float b = cell(sel(zc.w, zc.z), sel(zc.z, zc.y), sel(right, zc.w), sel(ym.w, ym.z), sel(yp.w, yp.z),
                         sel(zm.w, zm.z), sel(zp.w, zp.z), sel(rq.w, rq.z), mb);
    late = ((ma & M_GHOST) ? (odd ? 2u : 1u) : 0u) | ((mb & M_GHOST) ? (odd ? 8u : 4u) : 0u);
    return make_float4(sel(zc.x, a), sel(a, zc.y), sel(zc.z, b), sel(b, zc.w));
  };
  // The free-surface cells of colour col in that quad (up to two, flagged in
  // `bits` as relax flags them): row_local's ghost form with neighbours from LDS, both
  // cells' r, row codes and table entries in one round of loads. v: the two
  // colour cells' values, changed where flagged.
  auto relax_late = [&](int lq, int ly, int lz, int col, uint32_t bits, float v[2]) {
    const int q = qx0 + lq, y = y0 + ly, k = z0 + lz;
    const int par = (col + y + k) & 1;
    const size_t c = ((size_t)k * ny + y) * nx + 4 * (size_t)q + par;
    const size_t column = (size_t)y * nx + 4 * (size_t)q + par;
    uint32_t m2[2];
    float r2[2];
    GhostEntry g[2];
    const uint32_t mq = *reinterpret_cast<const uint32_t*>(G.mask + (c - par));
    const uint32_t first = FORM == FORM_INDEX ? G.gq[c >> 2] : 0u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      m2[h] = (mq >> (8 * (par + 2 * h))) & 0xFFu;
      r2[h] = r[c + 2 * h];
      if (FORM == FORM_TABLE || (FORM == FORM_INDEX && (bits & (1u << (par + 2 * h)))))
        g[h] = ghost_load<FORM>(G, column + 2 * h, k, ghost_index(G, mq, first, par + 2 * h));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = par + 2 * h;
      const float* sc = zs + ((lz * BR_LY + ly) * BR_LX + 4 * lq + e);
      const float pc = sc[0];
      v[h] = pc;
      if (!(bits & (1u << e))) continue;
      const float nb[6] = {(q > 0 || e > 0) ? sc[-1] : 0.f, (q + 1 < nq || e < 3) ? sc[1] : 0.f, sc[-BR_LX],
                           sc[BR_LX], sc[-BR_LX * BR_LY], sc[BR_LX * BR_LY]};
      float prec, az;
      if (FORM == FORM_GENERAL) az = row_local<FORM>(G, 4 * q + e, y, k, (uint8_t)m2[h], pc, nb, prec);
      else az = ghost_sum(g[h], m2[h], pc, nb, G.inv, prec) * G.inv;
      v[h] = prec > 0.f ? SV::rnd(pc + prec * (r2[h] - az)) : (MODE == 2 ? 0.f : pc);
    }
  };
  __syncthreads();
  // pass c over the brick and its ring (LDS rows 1..BR_Y+2, planes 1..BR_Z+2, every LDS quad)
  {
    uint32_t late = 0;
#pragma unroll
    for (int m = 0; m < BR_AITEMS; ++m) {
      if (!ona[m]) continue;
      const int idx = tid + BR_THREADS * m;
      const int lq = idx % BR_LQ, rest = idx / BR_LQ, ly = 1 + rest % (BR_Y + 2), lz = 1 + rest / (BR_Y + 2);
      uint32_t lt;
      const float4 o = relax(lq, ly, lz, colour, rqa[m], mqa[m], lt);
      *reinterpret_cast<float4*>(zs + ((lz * BR_LY + ly) * BR_LX + 4 * lq)) = o;
      late |= lt << (4 * m);
    }
    while (late) {
      const int m = (__ffs(late) - 1) >> 2;
      const uint32_t bits = (late >> (4 * m)) & 0xFu;
      late &= ~(0xFu << (4 * m));
      const int idx = tid + BR_THREADS * m;
      const int lq = idx % BR_LQ, rest = idx / BR_LQ, ly = 1 + rest % (BR_Y + 2), lz = 1 + rest / (BR_Y + 2);
      float v[2];
      relax_late(lq, ly, lz, colour, bits, v);
      float* dst = zs + (lz * BR_LY + ly) * BR_LX + 4 * lq + ((colour + y0 + ly + z0 + lz) & 1);
      dst[0] = v[0];
      dst[2] = v[1];
    }
  }
  __syncthreads();
  // pass 1 - c over the brick (LDS quads 1..BR_QX, rows 2..BR_Y+1, planes 2..BR_Z+1), to zout:
  // the plain cells of every quad, then the free-surface cells (their
  // neighbours are colour c, final in LDS, and their own value before the
  // pass is still there), then the stores. Kept apart so that the rare
  // free-surface path is not scheduled into the items' registers.
  double s = 0.0;
  {
    float4 ob[BR_BITEMS];
    uint32_t late = 0;
#pragma unroll
    for (int m = 0; m < BR_BITEMS; ++m) {
      ob[m] = f4zero();
      if (!onb[m]) continue;
      const int idx = tid + BR_THREADS * m;
      const int lq = 1 + idx % BR_QX, rest = idx / BR_QX, ly = 2 + rest % BR_Y, lz = 2 + rest / BR_Y;
      uint32_t lt;
      ob[m] = relax(lq, ly, lz, 1 - colour, rqb[m], mqb[m], lt);
      late |= lt << (4 * m);
    }
    while (late) {
      const int m = (__ffs(late) - 1) >> 2;
      const uint32_t bits = (late >> (4 * m)) & 0xFu;
      late &= ~(0xFu << (4 * m));
      const int idx = tid + BR_THREADS * m;
      const int lq = 1 + idx % BR_QX, rest = idx / BR_QX, ly = 2 + rest % BR_Y, lz = 2 + rest / BR_Y;
      float v[2];
      relax_late(lq, ly, lz, 1 - colour, bits, v);
#pragma unroll
      for (int mm = 0; mm < BR_BITEMS; ++mm) {
        if (mm != m) continue;
        if (bits & 1u) ob[mm].x = v[0];
        if (bits & 2u) ob[mm].y = v[0];
        if (bits & 4u) ob[mm].z = v[1];
        if (bits & 8u) ob[mm].w = v[1];
      }
    }
#pragma unroll
    for (int m = 0; m < BR_BITEMS; ++m) {
      if (!onb[m]) continue;
      const int idx = tid + BR_THREADS * m;
      const int lq = 1 + idx % BR_QX, rest = idx / BR_QX, ly = 2 + rest % BR_Y, lz = 2 + rest / BR_Y;
      const int q = qx0 + lq, y = y0 + ly, k = z0 + lz;
      const size_t c = ((size_t)k * ny + y) * nx + 4 * (size_t)q;
      SV::st4(zout, c, ob[m]);
      if (dot_op >= 0)
        s += (double)rqb[m].x * ob[m].x + (double)rqb[m].y * ob[m].y + (double)rqb[m].z * ob[m].z +
             (double)rqb[m].w * ob[m].w;
    }
  }
  if (dot_op >= 0) {
    const int lane = tid & 63, wid = tid >> 6;
    s = wave_sum(s);
    if (lane == 0) s_red[wid] = s;
    __syncthreads();
    if (tid == 0) {
      double tt = s_red[0];
      for (int w = 1; w < BR_THREADS / 64; ++w) tt += s_red[w];
      double* part = partials + (size_t)dot_op * MAX_PARTIALS * 2;
      part[2 * blockIdx.x] = tt;
      part[2 * blockIdx.x + 1] = 0.0;
    }
  }
}

// The wet flags of a block's quads, mq the row codes of the thread's quad (0: none).
__device__ __forceinline__ void flag_wet(const Fine& G, const BrickGrid& B, int qx, int j, int k, uint32_t mq) {
  if (B.bx > 0 && mq) G.wetb[((size_t)(j / BR_Y) * B.bz + k / BR_Z) * B.bx + qx / BR_QX] = 1;
  const int any = __syncthreads_or(mq != 0);
  if (threadIdx.x == 0) G.wetq[xcd_block(blockIdx.x, gridDim.x)] = any != 0;
}

// The flags of a geometry whose row codes another grid has made.
__global__ void __launch_bounds__(QBLOCK) k_wet_flags(Fine G, QuadGrid Q, BrickGrid B) {
  int qx, j, k;
  const bool valid = quad_coords(Q, qx, j, k);
  const uint32_t mq = valid ? *reinterpret_cast<const uint32_t*>(G.mask + cidx(G, 4 * qx, j, k)) : 0u;
  flag_wet(G, B, qx, j, k, mq);
}

// Row codes on quads (k_mask with four x-cells per thread: one decode, and
// the solid flags, apertures and surface heights of the quad and of its y and
// z neighbours as 4-byte and 16-byte loads). Same row_code per cell.
__global__ void __launch_bounds__(QBLOCK) k_mask_q(Fine G, QuadGrid Q, BrickGrid B, uint8_t* mask, Ctl* ctl,
                                                   double* partials) {
  double wet = 0.0, ghosts = 0.0;
  int qx, j, k;
  const bool valid = quad_coords(Q, qx, j, k);
  uint32_t out = 0;
  if (valid) {
    const int nx = G.nx, ny = G.ny, nz = G.nz, i0 = 4 * qx;
    const int jm = j > 0 ? j - 1 : j, jp = j + 1 < ny ? j + 1 : j;
    const int km = k > 0 ? k - 1 : k, kp = k + 1 < nz ? k + 1 : k;
    const int im0 = i0 > 0 ? i0 - 1 : i0, ip3 = i0 + 4 < nx ? i0 + 4 : i0 + 3;
    auto u32 = [](const uint8_t* p, size_t c) { return *reinterpret_cast<const uint32_t*>(p + c); };
    const uint32_t sc = u32(G.solid, cidx(G, i0, j, k));
    const uint32_t sym = u32(G.solid, cidx(G, i0, jm, k)), syp = u32(G.solid, cidx(G, i0, jp, k));
    const uint32_t szm = u32(G.solid, cidx(G, i0, j, km)), szp = u32(G.solid, cidx(G, i0, j, kp));
    const uint8_t sxm = G.solid[cidx(G, im0, j, k)], sxp = G.solid[cidx(G, ip3, j, k)];
    const size_t fu = fuidx(G, i0, j, k);
    uint8_t au[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) au[e] = G.ou[fu + e];
    const uint32_t av0 = u32(G.ov, fvidx(G, i0, j, k)), av1 = u32(G.ov, fvidx(G, i0, j + 1, k));
    const uint32_t aw0 = u32(G.ow, fwidx(G, i0, j, k)), aw1 = u32(G.ow, fwidx(G, i0, j, k + 1));
    const float4 h4 = ld4(G.eta, (size_t)j * nx + i0);
    const float4 hym = ld4(G.eta, (size_t)jm * nx + i0), hyp = ld4(G.eta, (size_t)jp * nx + i0);
    const float hxm = G.eta[(size_t)j * nx + im0], hxp = G.eta[(size_t)j * nx + ip3];
    auto byte = [](uint32_t w, int e) { return (uint8_t)(w >> (8 * e)); };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint8_t ap[6] = {au[e], au[e + 1], byte(av0, e), byte(av1, e), byte(aw0, e), byte(aw1, e)};
      const uint8_t sn[6] = {e > 0 ? byte(sc, e - 1) : sxm, e < 3 ? byte(sc, e + 1) : sxp, byte(sym, e),
                             byte(syp, e), byte(szm, e), byte(szp, e)};
      const float hn[4] = {e > 0 ? q_get(h4, e - 1) : hxm, e < 3 ? q_get(h4, e + 1) : hxp, q_get(hym, e),
                           q_get(hyp, e)};
      out |= (uint32_t)row_code(G, i0 + e, j, k, byte(sc, e), sn, ap, q_get(h4, e), hn, wet, ghosts) << (8 * e);
    }
    *reinterpret_cast<uint32_t*>(mask + cidx(G, i0, j, k)) = out;
  }
  flag_wet(G, B, qx, j, k, out);
  reduce_finish<false>(wet, ghosts, OP_COUNT, ctl, partials);
}

// r = b - A p, |r|^2 on quads (k_residual with four x-cells per thread: the
// pressures of the quad and of its y and z neighbours as 16-byte loads with
// indices clamped into the grid, the row's case decided after; apply_row_t's
// arithmetic per cell).
// BACKWARD: the same pass also folds the backward error of the r it stores
// into OP_BACKWARD, k_backward_q's arithmetic from the same pressures (|A||p|
// beside A p), so that the wrap-up reads p once for both.
template <int FORM = FORM_GENERAL, bool BACKWARD = false>
__global__ void __launch_bounds__(QBLOCK) k_residual_q(Fine G, QuadGrid Q, const double* p, const float* b, float* r,
                                                       int op, Ctl* ctl, double* partials, int gated) {
#pragma clang fp contract(off)
  if (gated && !replacing(ctl)) return;
  double s = 0.0, unused = 0.0, worst = 0.0;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  if (valid) {
    const size_t plane = (size_t)G.nx * G.ny;
    const size_t c0 = ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx;
    const uint32_t mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    const float4 bq = ld4(b, c0);
    auto quad = [&](size_t c, double v[4]) {
      const double2 a = *reinterpret_cast<const double2*>(p + c), e = *reinterpret_cast<const double2*>(p + c + 2);
      v[0] = a.x; v[1] = a.y; v[2] = e.x; v[3] = e.y;
    };
    double pc[4], pym[4], pyp[4], pzm[4], pzp[4];
    quad(c0, pc);
    quad(y > 0 ? c0 - G.nx : c0, pym);
    quad(y + 1 < G.ny ? c0 + G.nx : c0, pyp);
    quad(k > 0 ? c0 - plane : c0, pzm);
    quad(k + 1 < G.nz ? c0 + plane : c0, pzp);
    const double pxm = p[qx > 0 ? c0 - 1 : c0], pxp = p[4 * qx + 4 < G.nx ? c0 + 4 : c0 + 3];
    float4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint8_t m = (uint8_t)(mq >> (8 * e));
      double acc = 0.0, aabs = 0.0;
      if (m & M_WET) {
        const double pe = pc[e], pa = fabs(pc[e]);
        const double nb[6] = {e > 0 ? pc[e - 1] : pxm, e < 3 ? pc[e + 1] : pxp, pym[e], pyp[e], pzm[e], pzp[e]};
        if (!(m & M_GHOST)) {
#pragma unroll
          for (int f = 0; f < 6; ++f)
            if (m & (1u << f)) {
              acc += pe - nb[f];
              if (BACKWARD) aabs += pa + fabs(nb[f]);
            }
        } else {
          uint8_t type[6];
          float it[6], a[6];
          ghost_row<FORM>(G, 4 * qx + e, y, k, m, type, it, a);
#pragma unroll
          for (int f = 0; f < 6; ++f) {
            if (type[f] == 1) {
              acc += (double)a[f] * (pe - nb[f]);
              if (BACKWARD) aabs += (double)a[f] * (pa + fabs(nb[f]));
            } else if (type[f] == 2) {
              acc += (double)a[f] * pe * (double)it[f];
              if (BACKWARD) aabs += (double)a[f] * pa * (double)it[f];
            }
          }
        }
        acc = acc * (double)G.inv;
      }
      const double rc = (double)q_get(bq, e) - acc;
      const float rf = (float)rc;
      q_set(out, e, rf);
      s += rc * rc;
      if (BACKWARD && (m & M_WET)) {
        const double scale = fabs((double)q_get(bq, e)) + aabs * (double)G.inv;
        if (scale > 0.0) worst = fmax(worst, fabs((double)rf) / scale);
      }
    }
    st4(r, c0, out);
  }
  if (op >= 0) reduce_finish<false>(s, unused, op, ctl, partials);
  if (BACKWARD) reduce_finish<true>(worst, unused, OP_BACKWARD, ctl, partials);
}

// The aperture codes and solid flags of a quad's faces and cells for the
// aperture-weighted divergence: the y and z faces and the solid flags as one
// 4-byte load each (rows of nx bytes, nx % 4 == 0), the five x faces as bytes.
struct ApQuad {
  uint8_t u[5];
  uint32_t v0, v1, w0, w1, solid;
};
__device__ __forceinline__ ApQuad ap_quad(const Fine& G, size_t c0, size_t fu, size_t fv0, size_t fv1, size_t fw0,
                                          size_t fw1) {
  auto u32 = [](const uint8_t* a, size_t c) { return *reinterpret_cast<const uint32_t*>(a + c); };
  ApQuad A;
#pragma unroll
  for (int e = 0; e < 5; ++e) A.u[e] = G.ou[fu + e];
  A.v0 = u32(G.ov, fv0); A.v1 = u32(G.ov, fv1); A.w0 = u32(G.ow, fw0); A.w1 = u32(G.ow, fw1);
  A.solid = u32(G.solid, c0);
  return A;
}
__device__ __forceinline__ uint8_t ap_byte(uint32_t word, int e) { return (uint8_t)(word >> (8 * e)); }

// b = scale * div + ghost terms, prec (optional) and |b|^2 on quads
// (k_assemble with four x-cells per thread: the faces of the quad as 16-byte
// loads, its x faces as five scalars, or the given divergence; the row's
// arithmetic is k_assemble's, dry cells get 0).
__global__ void __launch_bounds__(QBLOCK) k_assemble_q(Fine G, QuadGrid Q, const float* us, const float* vs,
                                                       const float* ws, const float* div_in, float scale, float* b,
                                                       float* prec_out, Ctl* ctl, double* partials) {
#pragma clang fp contract(off)
  double s2 = 0.0, unused = 0.0, sum = 0.0, active = 0.0;
  int qx, j, k;
  const bool valid = quad_coords(Q, qx, j, k);
  if (valid) {
    const int i0 = 4 * qx;
    const size_t c0 = cidx(G, i0, j, k);
    const uint32_t mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    const size_t fu = fuidx(G, i0, j, k), fv0 = fvidx(G, i0, j, k), fv1 = fvidx(G, i0, j + 1, k);
    const size_t fw0 = fwidx(G, i0, j, k), fw1 = fwidx(G, i0, j, k + 1);
    float u5[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    float4 v0 = f4zero(), v1 = f4zero(), w0 = f4zero(), w1 = f4zero(), dq = f4zero();
    ApQuad A{};
    if (div_in) {
      dq = ld4(div_in, c0);
    } else {
#pragma unroll
      for (int e = 0; e < 5; ++e) u5[e] = us[fu + e];
      v0 = ld4(vs, fv0); v1 = ld4(vs, fv1); w0 = ld4(ws, fw0); w1 = ld4(ws, fw1);
      if (G.cut) A = ap_quad(G, c0, fu, fv0, fv1, fw0, fw1);
    }
    float4 out, pout = f4zero();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint8_t m = (uint8_t)(mq >> (8 * e));
      float bb = 0.f;
      if (m & M_WET) {
        float div;
        if (div_in) {
          div = q_get(dq, e);
        } else if (G.cut && ap_byte(A.solid, e)) {
          div = 0.f;
        } else {
          float fl = u5[e], fr = u5[e + 1], ff = q_get(v0, e), fk = q_get(v1, e), fb = q_get(w0, e), ft = q_get(w1, e);
          if (G.cut) {
            fl = aperture(G, 0, fu + e, A.u[e]) * fl; fr = aperture(G, 0, fu + e + 1, A.u[e + 1]) * fr;
            ff = aperture(G, 1, fv0 + e, ap_byte(A.v0, e)) * ff; fk = aperture(G, 1, fv1 + e, ap_byte(A.v1, e)) * fk;
            fb = aperture(G, 2, fw0 + e, ap_byte(A.w0, e)) * fb; ft = aperture(G, 2, fw1 + e, ap_byte(A.w1, e)) * ft;
          }
          div = ((fr - fl + ft - fb) + (fk - ff)) / G.dx;
        }
        bb = scale * div;
        float diag = 0.f;
        if (!(m & M_GHOST)) {
          for (int f = 0; f < 6; ++f) if (m & (1u << f)) diag += 1.0f;
        } else {
          RowG R;
          full_row(G, i0 + e, j, k, R);
          for (int f = 0; f < 6; ++f) {
            if (R.type[f] == 1) diag += R.a[f];
            else if (R.type[f] == 2) {
              diag += R.a[f] * R.it[f];
              bb += R.a[f] * R.val[f] * R.it[f] * G.inv;
            }
          }
        }
        if (prec_out) q_set(pout, e, diag > 0.f ? 1.0f / (diag * G.inv) : 0.f);
      }
      q_set(out, e, bb);
      s2 += (double)bb * (double)bb;
      if (prec_positive(m)) { sum += (double)bb; active += 1.0; }
    }
    st4(b, c0, out);
    if (prec_out) st4(prec_out, c0, pout);
  }
  reduce_finish<false>(s2, unused, OP_B2, ctl, partials);
  if (!ctl->gauge) return;
  __syncthreads();
  reduce_finish<false>(sum, active, OP_MEAN_B, ctl, partials);
}

// Velocity correction on quads (k_correct with four x-cells per thread: the
// x-, y- and z- faces of the quad and the closing faces on the +x, +y, +z
// walls; the solid flags, row codes and pressures of the quad and of the cells
// below it in x, y and z as 4-, 16- and 32-byte loads with indices clamped into
// the grid). Each face's arithmetic is k_correct's (corrected_side, ghost_up).
__global__ void __launch_bounds__(QBLOCK) k_correct_q(Fine G, QuadGrid Q, const float* us, const float* vs,
                                                      const float* ws, const double* p, float k1, float* u, float* v,
                                                      float* w, Ctl* ctl, double* partials) {
#pragma clang fp contract(off)
  double mx = 0.0, unused = 0.0;
  int qx, j, k;
  const bool valid = quad_coords(Q, qx, j, k);
  if (valid) {
    const int nx = G.nx, ny = G.ny, nz = G.nz, i0 = 4 * qx;
    const size_t plane = (size_t)nx * ny;
    const size_t c0 = cidx(G, i0, j, k);
    const size_t cy = j > 0 ? c0 - nx : c0, cz = k > 0 ? c0 - plane : c0, cx = i0 > 0 ? c0 - 1 : c0;
    auto u32 = [](const uint8_t* a, size_t c) { return *reinterpret_cast<const uint32_t*>(a + c); };
    auto byte = [](uint32_t wv, int e) { return (uint8_t)(wv >> (8 * e)); };
    auto pquad = [&](size_t c, double o[4]) {
      const double2 a = *reinterpret_cast<const double2*>(p + c), b = *reinterpret_cast<const double2*>(p + c + 2);
      o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y;
    };
    const uint32_t sq = u32(G.solid, c0), mq = u32(G.mask, c0);
    const uint32_t sy = u32(G.solid, cy), my = u32(G.mask, cy), sz = u32(G.solid, cz), mz = u32(G.mask, cz);
    const uint8_t sx = G.solid[cx], mxl = G.mask[cx];
    double pq[4], py[4], pz[4];
    pquad(c0, pq);
    pquad(cy, py);
    pquad(cz, pz);
    const double px = p[cx];
    const size_t fu = fuidx(G, i0, j, k), fv = fvidx(G, i0, j, k), fw = fwidx(G, i0, j, k);
    float ux[5];
    uint8_t ax[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      ux[e] = e < 4 || i0 + 4 == nx ? us[fu + e] : 0.f;
      ax[e] = e < 4 || i0 + 4 == nx ? G.ou[fu + e] : 0;
    }
    const float4 vq = ld4(vs, fv), wq = ld4(ws, fw);
    const uint32_t avq = u32(G.ov, fv), awq = u32(G.ow, fw);
    const bool top_y = j == ny - 1, top_z = k == nz - 1;
    const size_t fvt = fvidx(G, i0, ny, k), fwt = fwidx(G, i0, j, nz);
    const float4 vt = top_y ? ld4(vs, fvt) : f4zero(), wt = top_z ? ld4(ws, fwt) : f4zero();
    const uint32_t awt = top_z ? u32(G.ow, fwt) : 0u;
    const double kk = (double)k1, dx = (double)G.dx;
    // x- faces of the four cells, and the closing +x face
    float uo[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = i0 + e;
      const uint8_t sl = e > 0 ? byte(sq, e - 1) : sx, ml = e > 0 ? byte(mq, e - 1) : mxl;
      const double pl = e > 0 ? pq[e - 1] : px;
      const bool inner = i > 0;  // i < nx holds inside the quad
      float val = ux[e];
      if (inner && ax[e] && !sl && !byte(sq, e))
        val = corrected_side(G, val, pl, pq[e], (ml & M_WET) != 0, (byte(mq, e) & M_WET) != 0, k1, i - 1, j, i, j, k);
      uo[e] = val;
      mx = fmax(mx, (double)fabsf(val));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) u[fu + e] = uo[e];
    if (i0 + 4 == nx) {
      u[fu + 4] = ux[4];
      mx = fmax(mx, (double)fabsf(ux[4]));
    }
    // y- faces, and the closing +y faces
    float4 vo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = i0 + e;
      float val = q_get(vq, e);
      if (j > 0 && byte(avq, e) && !byte(sy, e) && !byte(sq, e))
        val = corrected_side(G, val, py[e], pq[e], (byte(my, e) & M_WET) != 0, (byte(mq, e) & M_WET) != 0, k1, i,
                             j - 1, i, j, k);
      q_set(vo, e, val);
      mx = fmax(mx, (double)fabsf(val));
    }
    st4(v, fv, vo);
    if (top_y) {
      st4(v, fvt, vt);
      mx = fmax(mx, (double)fmaxf(fmaxf(fabsf(vt.x), fabsf(vt.y)), fmaxf(fabsf(vt.z), fabsf(vt.w))));
    }
    // z- faces, and the closing +z faces
    auto zface = [&](float val, uint8_t open, int kf, uint8_t mb, double pb, uint8_t ma, double pa, int i, bool sb,
                     bool sa) {
      if (G.phi) {
        // level set (apic3d.rs:1016-1048): a face next to a solid is not
        // corrected, and air may lie below water
        if (kf >= 1 && kf < nz && open && !sb && !sa) {
          const bool wb = (mb & M_WET) != 0, wa = (ma & M_WET) != 0;
          float a, b;
          if (wb && wa) val = (float)((double)val - kk * (pa - pb) / dx);
          else if (wb) { ghost_up(G, i, j, kf - 1, a, b); val = (float)((double)val - kk * ((double)b - pb) * (double)a / dx); }
          else if (wa) { ghost_phi(G, i, j, kf, i, j, kf - 1, a, b); val = (float)((double)val - kk * (pa - (double)b) * (double)a / dx); }
        }
        return val;
      }
      if (kf >= 1 && open && (mb & M_WET)) {
        if (kf < nz && (ma & M_WET)) {
          val = (float)((double)val - kk * (pa - pb) / dx);
        } else {
          float a, b;
          ghost_up(G, i, j, kf - 1, a, b);
          val = (float)((double)val - kk * ((double)b - pb) * (double)a / dx);
        }
      }
      return val;
    };
    float4 wo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float val = zface(q_get(wq, e), byte(awq, e), k, byte(mz, e), pz[e], byte(mq, e), pq[e], i0 + e,
                              byte(sz, e) != 0, byte(sq, e) != 0);
      q_set(wo, e, val);
      mx = fmax(mx, (double)fabsf(val));
    }
    st4(w, fw, wo);
    if (top_z) {
      float4 wt2;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // face nz: below and (clamped) above are the top cell itself
        const float val = zface(q_get(wt, e), byte(awt, e), nz, byte(mq, e), pq[e], byte(mq, e), pq[e], i0 + e,
                                byte(sq, e) != 0, byte(sq, e) != 0);
        q_set(wt2, e, val);
        mx = fmax(mx, (double)fabsf(val));
      }
      st4(w, fwt, wt2);
    }
  }
  reduce_finish<true>(mx, unused, OP_UMAX, ctl, partials);
}

// max |div u| over wet rows and over plain rows on quads (k_divmetric with
// four x-cells per thread; divergence_at's arithmetic per cell).
__global__ void __launch_bounds__(QBLOCK) k_divmetric_q(Fine G, QuadGrid Q, const float* u, const float* v,
                                                        const float* w, Ctl* ctl, double* partials) {
#pragma clang fp contract(off)
  double all = 0.0, plain = 0.0;
  int qx, j, k;
  const bool valid = quad_coords(Q, qx, j, k);
  if (valid) {
    const int i0 = 4 * qx;
    const size_t c0 = cidx(G, i0, j, k);
    const uint32_t mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    if (mq & 0x40404040u) {  // a wet cell in the quad
      const size_t fu = fuidx(G, i0, j, k), fv0 = fvidx(G, i0, j, k), fv1 = fvidx(G, i0, j + 1, k);
      const size_t fw0 = fwidx(G, i0, j, k), fw1 = fwidx(G, i0, j, k + 1);
      float u5[5];
#pragma unroll
      for (int e = 0; e < 5; ++e) u5[e] = u[fu + e];
      const float4 v0 = ld4(v, fv0), v1 = ld4(v, fv1), w0 = ld4(w, fw0), w1 = ld4(w, fw1);
      const ApQuad A = G.cut ? ap_quad(G, c0, fu, fv0, fv1, fw0, fw1) : ApQuad{};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint8_t m = (uint8_t)(mq >> (8 * e));
        if (!(m & M_WET)) continue;
        float div = 0.f;
        if (!(G.cut && ap_byte(A.solid, e))) {
          float fl = u5[e], fr = u5[e + 1], ff = q_get(v0, e), fk = q_get(v1, e), fb = q_get(w0, e), ft = q_get(w1, e);
          if (G.cut) {
            fl = aperture(G, 0, fu + e, A.u[e]) * fl; fr = aperture(G, 0, fu + e + 1, A.u[e + 1]) * fr;
            ff = aperture(G, 1, fv0 + e, ap_byte(A.v0, e)) * ff; fk = aperture(G, 1, fv1 + e, ap_byte(A.v1, e)) * fk;
            fb = aperture(G, 2, fw0 + e, ap_byte(A.w0, e)) * fb; ft = aperture(G, 2, fw1 + e, ap_byte(A.w1, e)) * ft;
          }
          div = ((fr - fl + ft - fb) + (fk - ff)) / G.dx;
        }
        const double d = (double)fabsf(div);
        all = fmax(all, d);
        // plain: no ghost face (a row flagged for a fractional aperture alone is plain)
        bool plain_row = !(m & M_GHOST);
        if (!plain_row && G.frac) {
          RowG R;
          full_row(G, i0 + e, j, k, R);
          plain_row = true;
          for (int f = 0; f < 6; ++f) plain_row = plain_row && R.type[f] != 2;
        }
        if (plain_row) plain = fmax(plain, d);
      }
    }
  }
  reduce_finish<true>(all, plain, OP_DIVMAX, ctl, partials);
}

// Oettli-Prager backward error on quads (k_backward with four x-cells per
// thread, the pressures of the quad and of its y and z neighbours as 32-byte
// loads with indices clamped into the grid; k_backward's arithmetic per cell).
template <int FORM = FORM_GENERAL>
__global__ void __launch_bounds__(QBLOCK) k_backward_q(Fine G, QuadGrid Q, const double* p, const float* b,
                                                       const float* r, Ctl* ctl, double* partials) {
#pragma clang fp contract(off)
  double worst = 0.0, unused = 0.0;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  if (valid) {
    const size_t plane = (size_t)G.nx * G.ny;
    const size_t c0 = ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx;
    const uint32_t mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    auto quad = [&](size_t c, double v[4]) {
      const double2 a = *reinterpret_cast<const double2*>(p + c), e = *reinterpret_cast<const double2*>(p + c + 2);
      v[0] = a.x; v[1] = a.y; v[2] = e.x; v[3] = e.y;
    };
    double pc[4], pym[4], pyp[4], pzm[4], pzp[4];
    quad(c0, pc);
    quad(y > 0 ? c0 - G.nx : c0, pym);
    quad(y + 1 < G.ny ? c0 + G.nx : c0, pyp);
    quad(k > 0 ? c0 - plane : c0, pzm);
    quad(k + 1 < G.nz ? c0 + plane : c0, pzp);
    const double pxm = p[qx > 0 ? c0 - 1 : c0], pxp = p[4 * qx + 4 < G.nx ? c0 + 4 : c0 + 3];
    const float4 bq = ld4(b, c0), rq = ld4(r, c0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint8_t m = (uint8_t)(mq >> (8 * e));
      if (!(m & M_WET)) continue;
      const double pe = fabs(pc[e]);
      const double pn[6] = {e > 0 ? pc[e - 1] : pxm, e < 3 ? pc[e + 1] : pxp, pym[e], pyp[e], pzm[e], pzp[e]};
      double acc = 0.0;
      if (!(m & M_GHOST)) {
        for (int f = 0; f < 6; ++f)
          if (m & (1u << f)) acc += pe + fabs(pn[f]);
      } else {
        uint8_t type[6];
        float it[6], a[6];
        ghost_row<FORM>(G, 4 * qx + e, y, k, m, type, it, a);
        for (int f = 0; f < 6; ++f) {
          if (type[f] == 1) acc += (double)a[f] * (pe + fabs(pn[f]));
          else if (type[f] == 2) acc += (double)a[f] * pe * (double)it[f];
        }
      }
      const double scale = fabs((double)q_get(bq, e)) + acc * (double)G.inv;
      if (scale > 0.0) worst = fmax(worst, fabs((double)q_get(rq, e)) / scale);
    }
  }
  reduce_finish<true>(worst, unused, OP_BACKWARD, ctl, partials);
}

// Cold start, p = 0: p64 = 0, r = b - A 0 = b exactly, |r|^2 into `op`
// (k_load_p and k_residual in one pass over b), b without its mean first where
// the problem is pure Neumann.
__global__ void __launch_bounds__(QBLOCK) k_start_cold(size_t nquads, const uint8_t* mask, float* b, double* p, float* r,
                                                       int op, Ctl* ctl, double* partials) {
  const bool pure = ctl->pure_neumann != 0;
  const float mean = (float)ctl->mean_b;
  double s = 0.0, unused = 0.0;
  const size_t t = (size_t)blockIdx.x * QBLOCK + threadIdx.x;
  if (t < nquads) {
    const size_t c = 4 * t;
    float4 bq = ld4(b, c);
    if (pure) {
      const uint32_t mq = *reinterpret_cast<const uint32_t*>(mask + c);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (prec_positive((uint8_t)(mq >> (8 * e)))) q_set(bq, e, q_get(bq, e) - mean);
      st4(b, c, bq);
    }
    double2* pp = reinterpret_cast<double2*>(p + c);
    pp[0] = make_double2(0.0, 0.0);
    pp[1] = make_double2(0.0, 0.0);
    st4(r, c, bq);
    s = (double)bq.x * bq.x + (double)bq.y * bq.y + (double)bq.z * bq.z + (double)bq.w * bq.w;
  }
  reduce_finish<false>(s, unused, op, ctl, partials);
  if (!pure) return;
  __syncthreads();
  reduce_finish<false>(s, unused, OP_B2, ctl, partials);
}

// ---------------------------------------------------------------- damped Jacobi
// Sweeps of the fine level on quads (k_fjacobi's arithmetic,
// delta3d_multigrid.rs:398-405; the rows' factors from G.precv): zout = zin + w prec (r - A zin). MODE 2:
// zin is first prolonged from the first coarse level (k_prolong_fine's arithmetic) on the fly. MODE 1: the
// first two sweeps from zero; the first is local (w prec r), so its neighbours'
// values are formed from their r and factors. At 128x64x96 with a cut bottom
// a sweep takes 6.6 us against 10.9 with a thread per cell, the first two 8.0 against 21.8.
template <int MODE, int FORM>
__global__ void __launch_bounds__(QBLOCK) k_q_jacobi(Fine G, QuadGrid Q, const float* zin, float* zout, const float* r,
                                                     Level L0, const float* xc, Ctl* ctl) {
#pragma clang fp contract(off)
  uint32_t wet = block_wet(G);
  if (!loop_active(ctl, wet)) return;
  const float omega = 6.0f / 7.0f;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  const size_t plane = (size_t)G.nx * G.ny;
  const size_t c0 = valid ? ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx : 0;
  if (!wet) {
    if (valid) st4(zout, c0, f4zero());
    return;
  }
  auto first = [&](float prec, float rv) { return prec > 0.f ? omega * prec * rv : 0.f; };
  // the iterate of quad c in row yy, plane kk (MODE 2: prolonged; rows that the
  // prolongation zeroes have no coupling and no factor)
  auto iterate = [&](size_t c, int yy, int kk) {
    if (MODE == 1) {
      const float4 p = ld4(G.precv, c), v = ld4(r, c);
      return make_float4(first(p.x, v.x), first(p.y, v.y), first(p.z, v.z), first(p.w, v.w));
    }
    float4 v = ld4(zin, c);
    if (MODE == 2) {
      const float2 a = *reinterpret_cast<const float2*>(xc + lidx(L0, 2 * qx, yy >> 1, kk >> 1));
      v.x = v.x + a.x; v.y = v.y + a.x; v.z = v.z + a.y; v.w = v.w + a.y;
    }
    return v;
  };
  float4 zc = f4zero(), ym = f4zero(), yp = f4zero(), zm = f4zero(), zp = f4zero(), rq = f4zero(), pq = f4zero();
  uint32_t mq = 0;
  if (valid) {
    mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    rq = ld4(r, c0);
    pq = ld4(G.precv, c0);
    zc = iterate(c0, y, k);
    if (y > 0) ym = iterate(c0 - G.nx, y - 1, k);
    if (y + 1 < G.ny) yp = iterate(c0 + G.nx, y + 1, k);
    if (k > 0) zm = iterate(c0 - plane, y, k - 1);
    if (k + 1 < G.nz) zp = iterate(c0 + plane, y, k + 1);
  }
  float left, right;
  x_neighbours(Q, valid, qx, zc, left, right, [&](int off) {
    const size_t c = c0 + off;
    if (MODE == 1) return first(G.precv[c], r[c]);
    float v = zin[c];
    if (MODE == 2) v = v + xc[lidx(L0, (4 * qx + off) >> 1, y >> 1, k >> 1)];
    return v;
  });
  if (!valid) return;
  float row[4];
  quad_rows<FORM>(G, 4 * qx, y, k, mq, zc, left, right, ym, yp, zm, zp, row);
  float4 out = zc;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float prec = q_get(pq, e);
    float z = q_get(zc, e);
    if (MODE == 2 && !prec_positive((uint8_t)(mq >> (8 * e)))) z = 0.f;
    if (prec > 0.f) z += omega * prec * (q_get(rq, e) - row[e]);
    q_set(out, e, z);
  }
  st4(zout, c0, out);
}

// ---------------------------------------------------------------- residual + restriction
// The residual t = r - A z of the 16 fine cells of (fine quad column qx,
// coarse row J, coarse plane K), summed per coarse cell in the reference's
// child order and scaled by 1/8 (restrict3, delta3d_multigrid.rs:258-272),
// with the work split over two threads: the first 128 threads of a
// workgroup take the fine plane 2K, the last 128 the plane 2K + 1. The first half's
// partial sums (children of plane 2K, in the reference's order) reach the
// second half through LDS, which adds its own children in order: the sum,
// and so the coarse r, is the one-thread sum bit for bit, with twice the
// waves in flight to overlap the loads with the arithmetic (38 -> 28 us at
// 256x256x128). H: the restriction's quad grid for 128-thread halves.
template <int ST, int FORM = FORM_GENERAL>
__global__ void __launch_bounds__(QBLOCK) k_q_restrict2(Fine G, QuadGrid H, const typename Store<ST>::T* z,
                                                        const float* r, Level L0, Ctl* ctl) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  __shared__ float2 carry[QBLOCK / 2];
  const int local = (int)(threadIdx.x & (QBLOCK / 2 - 1)), dz = (int)(threadIdx.x / (QBLOCK / 2));
  const unsigned Lb = xcd_block(blockIdx.x, gridDim.x);
  unsigned bx, by;
  int K;
  quad_block(H, Lb, bx, by, K);
  // the rows of this block's two planes are two blocks of the quad grid
  const unsigned lower = Lb + (unsigned)K * (unsigned)(H.nbx * H.nby), upper = lower + (unsigned)(H.nbx * H.nby);
  uint32_t wet = G.wetq[lower] | G.wetq[upper];
  if (!loop_active(ctl, wet)) return;
  const int qx = ((int)bx << H.sx) + (local & (H.QX - 1));
  const int J = (int)by * H.RY + (local >> H.sx);
  const bool valid = qx < H.nq && J < H.rows && K < H.planes;
  const size_t plane = (size_t)G.nx * G.ny;
  if (!wet) {
    if (valid && dz == 0)
      SV::st2(reinterpret_cast<typename SV::T*>(L0.r), lidx(L0, 2 * qx, J, K), make_float2(0.f, 0.f));
    return;
  }
  const int k = 2 * K + dz;
  float t[2][4];  // [dy][e]
#pragma unroll
  for (int dy = 0; dy < 2; ++dy) {
    const int y = 2 * J + dy;
    const size_t c0 = valid ? ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx : 0;
    float4 zc = f4zero(), rq = f4zero(), ym = f4zero(), yp = f4zero(), zm = f4zero(), zp = f4zero();
    uint32_t mq = 0;
    if (valid) {
      mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
      zc = SV::ld4(z, c0);
      rq = ld4(r, c0);
      if (y > 0) ym = SV::ld4(z, c0 - G.nx);
      if (y + 1 < G.ny) yp = SV::ld4(z, c0 + G.nx);
      if (k > 0) zm = SV::ld4(z, c0 - plane);
      if (k + 1 < G.nz) zp = SV::ld4(z, c0 + plane);
    }
    float left, right;
    x_neighbours(H, valid, qx, zc, left, right, [&](int off) { return SV::ld(z, c0 + off); });
    // (invalid lanes: mq = 0, every row 0)
    float row[4];
    quad_rows<FORM>(G, 4 * qx, y, k, mq, zc, left, right, ym, yp, zm, zp, row);
#pragma unroll
    for (int e = 0; e < 4; ++e) t[dy][e] = q_get(rq, e) - row[e];
  }
  float2 sum = make_float2(0.f, 0.f);
  if (dz == 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float s = 0.f;
      s += t[0][2 * h]; s += t[0][2 * h + 1];
      s += t[1][2 * h]; s += t[1][2 * h + 1];
      if (h == 0) sum.x = s; else sum.y = s;
    }
    carry[local] = sum;
  }
  __syncthreads();
  if (dz == 0 || !valid) return;
  sum = carry[local];
  float2 out;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float s = h == 0 ? sum.x : sum.y;
    s += t[0][2 * h]; s += t[0][2 * h + 1];
    s += t[1][2 * h]; s += t[1][2 * h + 1];
    if (h == 0) out.x = 0.125f * s; else out.y = 0.125f * s;
  }
  SV::st2(reinterpret_cast<typename SV::T*>(L0.r), lidx(L0, 2 * qx, J, K), out);
}

// A vector held in storage ST, widened to f32.
template <int ST>
__global__ void __launch_bounds__(BLOCK) k_unpack(size_t n, const typename Store<ST>::T* z, float* out) {
  FSP_FOR(c, n) out[c] = Store<ST>::ld(z, c);
}

// ---------------------------------------------------------------- CG steps on quads
// d = z (first) or z + beta d_old, q = A d, <d, q> (delta3d_mobile.rs:520-523, :460-465).
// z is held in storage ST.
template <int ST, int FORM = FORM_GENERAL>
__global__ void __launch_bounds__(QBLOCK) k_q_spmv_dir(Fine G, QuadGrid Q, const typename Store<ST>::T* z, float* d0,
                                                       float* d1, float* q, Ctl* ctl, double* partials) {
#pragma clang fp contract(off)
  using SV = Store<ST>;
  uint32_t wet = block_wet(G);
  if (!loop_active(ctl, wet)) return;
  const int sel = ctl->dsel, first = ctl->first_dir;
  const float beta = (float)ctl->beta;
  const float* dold = sel ? d1 : d0;
  float* dnew = sel ? d0 : d1;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  const size_t plane = (size_t)G.nx * G.ny;
  const size_t c0 = valid ? ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx : 0;
  if (!wet) {
    // (flexible CG folds <q, z> over every cell)
    if (ctl->flexible && valid) st4(q, c0, f4zero());
    zero_partial(OP_DQ, partials);
    return;
  }
  auto dir4 = [&](size_t c) {
    float4 a = SV::ld4(z, c);
    if (!first) {
      const float4 b = ld4(dold, c);
      a.x = a.x + beta * b.x; a.y = a.y + beta * b.y; a.z = a.z + beta * b.z; a.w = a.w + beta * b.w;
    }
    return a;
  };
  float4 dc = f4zero(), ym = f4zero(), yp = f4zero(), zm = f4zero(), zp = f4zero();
  uint32_t mq = 0;
  if (valid) {
    mq = *reinterpret_cast<const uint32_t*>(G.mask + c0);
    dc = dir4(c0);
    if (y > 0) ym = dir4(c0 - G.nx);
    if (y + 1 < G.ny) yp = dir4(c0 + G.nx);
    if (k > 0) zm = dir4(c0 - plane);
    if (k + 1 < G.nz) zp = dir4(c0 + plane);
  }
  float left, right;
  x_neighbours(Q, valid, qx, dc, left, right, [&](int off) {
    const size_t c = c0 + off;
    return first ? SV::ld(z, c) : SV::ld(z, c) + beta * dold[c];
  });
  double s = 0.0, unused = 0.0;
  if (valid) {
    float row[4];
    quad_rows<FORM>(G, 4 * qx, y, k, mq, dc, left, right, ym, yp, zm, zp, row);
    const float4 qo = make_float4(row[0], row[1], row[2], row[3]);
    st4(dnew, c0, dc);
    st4(q, c0, qo);
    s = (double)dc.x * qo.x + (double)dc.y * qo.y + (double)dc.z * qo.z + (double)dc.w * qo.w;
  }
  reduce_finish<false>(s, unused, OP_DQ, ctl, partials);
}

// Largest number of partials that k_q_update folds itself.
#ifndef FSP_FOLD_PARTIALS
#define FSP_FOLD_PARTIALS 2048
#endif

// Sum of the first components of `count` partials by a whole workgroup of
// QBLOCK threads, in k_finish's order, for every thread.
__device__ __forceinline__ double fold_partials(const double* partials, int slot, unsigned count) {
  constexpr int WAVES = FIN_THREADS / 64, PER = WAVES / (QBLOCK / 64);
  __shared__ double sums[WAVES];
  const double* part = partials + (size_t)slot * MAX_PARTIALS * 2;
  const int lane = threadIdx.x & 63, first = (int)(threadIdx.x >> 6) * PER;
  double a[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) a[u] = 0.0;
  for (unsigned base = 0; base < count; base += FIN_THREADS) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const unsigned q = base + (unsigned)((first + u) * 64 + lane);
      a[u] += q < count ? part[2 * (size_t)q] : 0.0;
    }
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    a[u] = wave_sum(a[u]);
    if (lane == 0) sums[first + u] = a[u];
  }
  __syncthreads();
  double t = sums[0];
  for (int w = 1; w < WAVES; ++w) t += sums[w];
  return t;
}

// p += alpha d (f64), r -= alpha q, |r|^2; four cells per thread. dq_parts: the
// number of partials of <d, q> that every workgroup folds itself (the
// iteration's k_finish records the sum, the step and the buffer switch), or 0
// where k_finish has run in between (above FSP_FOLD_PARTIALS the folds read
// more than that launch costs). Folded against not, projections of tanks from
// 32^3 cells up, by their number of partials: to 1024 1.2 to 1.5 % faster (64^3
// 0.901 -> 0.887 ms, 128x64x128 1.299 -> 1.280), 1536 0.6, 2048 0.2, 3072 to
// 4096 0.1 to 0.3 % slower (128x192x128 1.786 -> 1.792), 6144 1.4 (256x192x128
// 2.396 -> 2.429), 8192 3 (256x128x256 3.43 -> 3.53).
__global__ void __launch_bounds__(QBLOCK) k_q_update(Fine G, QuadGrid Q, double* p, float* r, const float* d0,
                                                     const float* d1, const float* q, Ctl* ctl, double* partials,
                                                     unsigned dq_parts) {
  uint32_t wet = block_wet(G);
  if (!loop_active(ctl, wet)) return;
  if (!wet) {
    zero_partial(OP_RN, partials);
    return;
  }
  double alpha64 = ctl->alpha;
  int sel = ctl->dsel;
  int qx, y, k;
  const bool valid = quad_coords(Q, qx, y, k);
  const size_t c = valid ? ((size_t)k * G.ny + y) * G.nx + 4 * (size_t)qx : 0;
  if (dq_parts) sel ^= 1;
  const float4 dv = ld4(sel ? d1 : d0, c), qv = ld4(q, c);
  float4 rv = ld4(r, c);
  double2* pp = reinterpret_cast<double2*>(p + c);
  double2 p0 = pp[0], p1 = pp[1];
  if (dq_parts) {
    const double dq = fold_partials(partials, OP_DQ, dq_parts);
    if (!(dq > 0.0)) return;
    alpha64 = ctl->rz / dq;
  }
  const float alpha = (float)alpha64;
  double s = 0.0, unused = 0.0;
  if (valid) {
    p0.x += alpha64 * (double)dv.x; p0.y += alpha64 * (double)dv.y;
    p1.x += alpha64 * (double)dv.z; p1.y += alpha64 * (double)dv.w;
    pp[0] = p0;
    pp[1] = p1;
    rv.x = rv.x - alpha * qv.x; rv.y = rv.y - alpha * qv.y; rv.z = rv.z - alpha * qv.z; rv.w = rv.w - alpha * qv.w;
    st4(r, c, rv);
    s = (double)rv.x * rv.x + (double)rv.y * rv.y + (double)rv.z * rv.z + (double)rv.w * rv.w;
  }
  reduce_finish<false>(s, unused, OP_RN, ctl, partials);
}

// ---------------------------------------------------------------- small coarse levels in one workgroup
constexpr int TAIL_THREADS = 1024;
constexpr int TAIL_MAX_LEVELS = 8;
constexpr int TAIL_CELLS = 4096;                // largest first level of the tail
// Largest dynamic LDS of a tail workgroup, in floats: the compact tail's with
// one level of odd rows, six floats a cell, 96 KiB. (With even rows the first
// level is in registers, its x and two guards in LDS: 46 KiB with the levels
// below. The row-coefficient tail takes three floats a cell, 55 KiB in all.)
// With a limit of 64 KiB on levels held in LDS a closed box of 64^3 ran the
// 16 colour passes of its coarsest level, 16^3, as launches of their own.
constexpr int TAIL_LDS_FLOATS = 6 * TAIL_CELLS;

struct TailSet {
  Level lv[TAIL_MAX_LEVELS];  // global arrays of the tail levels (first .. last)
  const float* pack;          // Galerkin tail: every level's couplings in LDS order (k_gct_pack)
  int count;
  int smoother;               // FSP_SMOOTH_*
  int pre, post, coarse;
};

// The colours of a level's red-black sweeps: red-black on the way down,
// black-red on the way up, and on the coarsest level the palindrome of both halves
// (count passes of each colour in all).
__host__ __device__ inline int sweep_passes(bool coarsest, int count) {
  return coarsest ? 4 * (count / 2) + (count & 1) : 2 * count;
}
__host__ __device__ inline int sweep_colour(bool coarsest, bool forward, int count, int p) {
  if (!coarsest) return forward ? (p & 1) : 1 - (p & 1);
  const int mid = 2 * (count / 2) + (count & 1);
  return p < mid ? (p & 1) : 1 - ((p - mid) & 1);
}

}  // namespace fsp
