// The SIPG Laplace operator on affine (Cartesian) boxes, see launch_sipg_cartesian.
//
// On an affine axis-parallel mesh the SIPG operator is exactly a sum of Kronecker products:
//   A = L_x (x) M_y (x) M_z + M_x (x) L_y (x) M_z + M_x (x) M_y (x) L_z
// with M_d = h_d * M (1D mass, exact with QGauss(k+1)) and L_d the 1D DG Laplacian along d:
// K/h_d plus, at each line end, the flux terms of laplace_operator.h:180-197 written with
// the exterior trace (value w and d/dx_d derivative dw at the shared face):
//   right end: o_i -= 1/2 d1_i [u], o_{n-1} += -1/2 (du + dw) + tau [u],  [u] = u_{n-1} - w
//   left end : o_i += 1/2 d0_i [u], o_0     +=  1/2 (du + dw) + tau [u],  [u] = u_0 - w
// For boundary faces (w, dw) come from the mirror principle (weak_boundary_conditions.h):
// Dirichlet w = -u, dw = du; Neumann w = u, dw = -du -- one branch-free code path.
// Evaluated as out = M_z (M_y a_x + M_x a_y) + M_y M_x a_z with a_d = L_d(u, traces).
//
// One group of n^2 lanes per cell, each lane holding one line of the cell at a time, and three LDS
// buffers per cell:
//   P0: the cell's values to LDS (U), what the neighbours' lines are needed for
//   P1: a_y from y-lines (to A), a_z from z-lines (to B), a_x from x-lines
//   P2: M_x A and M_x B along x-lines in place, a_x to U
//   P3: M_y U and M_y B along y-lines in place
//   P4: M_z (U + A) + B along z-lines, the epilogue
// with workgroup barriers between them. The 1D matrices are applied in even-odd form; a line's
// even and odd parts serve its stiffness, its end derivatives and its flux terms.
//
// Two kernels share this. The single-layer one takes the cells of a row and reads all six
// neighbours of each; the layered one (short lines, long vectors) walks a tile of cells through a
// segment of layers and reads each cell about 2.4 times instead of 5.2, at the price of more
// registers and a longer start. What bounds them are LDS passes, vector instructions and the
// vector-memory address unit together: FP64 k = 4 on 64^3 cells kept them busy for 76%, 60% and 73%
// of the cycles (SQ_LDS_IDX_ACTIVE, SQ_ACTIVE_INST_VALU, TA_BUSY) when 41% of the LDS passes were
// bank conflicts, hence strides and line assignments by bank and the shared even-odd parts (now 58%
// with 7% conflicts, 55% and 40%). Launches in turn in one process, before / single-layer / layered:
// FP64 k = 4 on 64^3 cells 183 / 173 / 165 us (2.9 -> 3.2 TB/s of src and dst; 202 / - / 174 with
// changing inputs), k = 3 on 64^3 90 / 86 / 77; FP32 k = 6 on 31 x 45 x 27 42.9 / 41.0; FP64 k = 7 on
// 40^3 217 / 182; FP32 k = 2 on 96^3 95 / 91 / 68.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <numeric>
#include <vector>

#include "../../include/exadg_amd.h"
#include "laplace_kernels.h"
#include "sipg_lines.h"

namespace ExaDG
{
namespace
{
constexpr int kMaxLayered = 5;  // longest lines of the layered kernel, see use_layers

// The layered kernel's tile of BX x BY cells per workgroup, the waves per SIMD that its registers
// are held to, and its LDS strides in entries: `plane` from one z-plane of a cell to the next (x-
// and y-neighbours are 1 and n apart) and `slot` from one cell's three buffers to the next one's.
// LDS serves a group of 16 FP64 or 32 FP32 lanes in one pass if their addresses differ modulo 16
// or 32 entries. With these strides z-lines in the order of the vector do, and x- and y-lines once
// dealt out by their banks (deal_lines): modeled passes per access 1.0 - 1.3, dense 1.7 - 3.5.
template<int N, typename Number>
struct CartTile
{
  static_assert(N >= 2 && N <= kMaxLayered);
  static constexpr bool dp      = sizeof(Number) == 8;
  static constexpr int  BX      = N == 2 ? 8 : N == 3 ? 7 : N == 4 ? 4 : 5;
  static constexpr int  BY      = N == 2 ? 8 : N == 5 ? 2 : 4;
  static constexpr int  cells   = BX * BY;
  static constexpr int  threads = 256;
  static constexpr int  waves   = dp ? (N == 2 ? 6 : N <= 4 ? 5 : 4) : (N <= 3 ? 8 : N == 4 ? 7 : 5);
  static constexpr int  plane   = N == 2 ? 4 : N == 3 ? (dp ? 10 : 11) : N == 4 ? 16 : 26;
  static constexpr int  slot    = N == 2 ? 25 : N == 3 ? (dp ? 89 : 105) : N == 4 ? 193 : dp ? 393 : 409;
  static_assert(cells * N * N <= threads);
};

// the layered kernel's LDS
template<int N, typename Number>
struct LdsLayout
{
  using Tile              = CartTile<N, Number>;
  static constexpr int PY = Tile::plane, PC = PY * (N - 1) + N * N, S = Tile::slot;
  static_assert(S >= 3 * PC && S * Tile::cells <= 65536, "three buffers per cell, 16-bit offsets");
  // the halo pairs follow the cells' buffers, aligned to a pair
  static constexpr int cells = (S * Tile::cells + 1) / 2 * 2;
  static constexpr int halo  = 2 * (Tile::BX + Tile::BY) * N * N;
  static constexpr int tau   = cells + 2 * halo;  // 6 per cell: x-, x+, y-, y+, z, (padding)
  static constexpr int size  = tau + 6 * Tile::cells;
  // then, as integers, per cell its index in the plane and flags, and per halo face the neighbour
  static constexpr int    n_faces = 2 * (Tile::BX + Tile::BY);
  static constexpr size_t bytes   = size * sizeof(Number) + (2 * Tile::cells + n_faces) * sizeof(int);
};

// A store of an output that no kernel of the same apply reads back: marked non-temporal, so
// that it does not displace from the caches the neighbour cells that other workgroups are
// still reading. Used for the vmult; the Chebyshev and residual outputs are read by the next
// kernel of a V-cycle and stay cached.
template<typename Number>
__device__ __forceinline__ void store_stream(Number * p, Number v)
{
  __builtin_nontemporal_store(v, p);
}

// The 1D tables as uniform (scalar) loads. Each phase of the layer loop
// takes its pointer anew through fresh(), opaque to the compiler, so that a table is loaded
// (scalar cache) where it is used: hoisted out of the loop, the tables exceed the scalar
// registers and are spilled into vector registers.
template<typename Number>
using Table = Number const __attribute__((address_space(4))) *;

template<typename Number>
__device__ __forceinline__ Table<Number> fresh(Table<Number> t)
{
  asm volatile("" : "+s"(t));
  return t;
}

// Brings the tables into the scalar cache while the vector loads are under way: the phases would
// otherwise wait for a cache line or two each, which shows where a launch is a single round of
// workgroups (8^3 cells replayed from a graph, FP64 k = 3 5.9 -> 5.6 us, V-cycles 1 - 3%).
template<int N, typename Number>
__device__ __forceinline__ void touch_tables(Table<Number> t)
{
  constexpr int step = 64 / sizeof(Number), lines = (CartTable<N>::line(3) + step - 1) / step;
  int           v[lines];
#pragma unroll
  for(int i = 0; i < lines; ++i)
    v[i] = ((int const __attribute__((address_space(4))) *)t)[16 * i];
#pragma unroll
  for(int i = 0; i < lines; ++i)
    asm volatile("" : : "s"(v[i]));
}

// (value, derivative) of a line at a face
template<typename Number>
struct alignas(2 * sizeof(Number)) Trace
{
  Number w, dw;
};

// sum_i a_i v_{n-1-i}
template<int N, typename Number>
__device__ __forceinline__ Number dot_reversed(Table<Number> const a, Number const (&v)[N])
{
  Number s = 0;
#pragma unroll
  for(int i = 0; i < N; ++i)
    s += a[i] * v[N - 1 - i];
  return s;
}

// A line split into its even part e (v_j + v_{n-1-j}, the middle value last for odd n) and odd part
// o (v_j - v_{n-1-j}), with its end derivatives du(0), du(1): on symmetric nodes they mirror each
// other (d1_i = -d0_{n-1-i}), so that du(0) = de + do and du(1) = do - de with the even-odd form
// of d0. FP64 at n = 7 takes them by plain products instead, which measured 2% faster (see CellLayout).
template<int N, typename Number>
struct SplitLine
{
  static constexpr int  m = N / 2, me = m + N % 2;
  static constexpr bool plain = sizeof(Number) == 8 && N == 7;
  Number                e[me], o[m], du0, du1;
  __device__ __forceinline__ SplitLine(Table<Number> const tab, Number const (&v)[N])
  {
    Table<Number> const DE = tab + CartTable<N>::DE, DO = tab + CartTable<N>::DO;
    Number              se = 0, so = 0;
#pragma unroll
    for(int j = 0; j < m; ++j)
    {
      e[j] = v[j] + v[N - 1 - j];
      o[j] = v[j] - v[N - 1 - j];
      if constexpr(!plain)
      {
        se += DE[j] * e[j];
        so += DO[j] * o[j];
      }
    }
    if constexpr(N % 2 == 1)
    {
      e[m] = v[m];
      if constexpr(!plain)
        se += DE[m] * e[m];
    }
    du0 = plain ? dot_line<N>(tab + CartTable<N>::D0, v) : se + so;
    du1 = plain ? -dot_reversed<N, Number>(tab + CartTable<N>::D0, v) : so - se;
  }
};

// out = c L_d u along one line (c the scale of the Kronecker term): K c/h_d and d0 c/(2 h_d) in
// even-odd form in L, half = c/(2 h_d), tau the penalties times c; u0 and u1 the line's end values
// and l and r the exterior traces, with unit-interval derivatives (same h_d on a uniform box).
// The flux terms of both ends, d0_i (u_0 - w_l)/2 - d1_i (u_{n-1} - w_r)/2, join the even and odd
// sums.
template<int N, typename Number>
__device__ __forceinline__ void line_laplacian(Table<Number> const L, Number half,
                                               SplitLine<N, Number> const & u, Number u0, Number u1,
                                               Trace<Number> const & l, Trace<Number> const & r,
                                               Number tau_l, Number tau_r, Number (&out)[N])
{
  constexpr int       m = N / 2, me = m + N % 2;
  Table<Number> const Ae = L, Ao = L + m * me, Am = Ao + m * m, DE = L + cs_size(N), DO = DE + me;
  Number const        jl = u0 - l.w, jr = u1 - r.w, js = jl + jr, jd = jl - jr;
#pragma unroll
  for(int i = 0; i < m; ++i)
  {
    Number E = DE[i] * js, O = DO[i] * jd;
#pragma unroll
    for(int j = 0; j < me; ++j)
      E += Ae[i * me + j] * u.e[j];
#pragma unroll
    for(int j = 0; j < m; ++j)
      O += Ao[i * m + j] * u.o[j];
    out[i]         = E + O;
    out[N - 1 - i] = E - O;
  }
  if constexpr(N % 2 == 1)
  {
    Number E = DE[m] * js;
#pragma unroll
    for(int j = 0; j < me; ++j)
      E += Am[j] * u.e[j];
    out[m] = E;
  }
  out[0] += half * (u.du0 + l.dw);
  out[0] += tau_l * jl;
  out[N - 1] -= half * (u.du1 + r.dw);
  out[N - 1] += tau_r * jr;
}

// the exterior trace of a boundary face from the line's own trace (weak_boundary_conditions.h)
template<typename Number>
__device__ __forceinline__ Trace<Number> mirrored(int type, Number u, Number du)
{
  return type == EXADG_BC_DIRICHLET ? Trace<Number>{-u, du} : Trace<Number>{u, -du};
}

// flags of a cell of the tile, for its x-faces and, << 4, its y-faces: the neighbour at the lower /
// upper (<< 1) end is in the tile; there is none (the mirror principle), else it is in the halo.
// Above them the numbers of boundary faces: of the cell along x (bits 8), y (10), and the larger
// ones of the cell and its neighbour at x- (12), x+ (14), y- (16), y+ (18)
enum : int
{
  kInside = 1,
  kMirror = 4
};

// keeps a per-lane value in its register: flags tested in the layer loop would otherwise be
// turned into wave masks before it, more than there are scalar registers
__device__ __forceinline__ int opaque(int v)
{
  asm volatile("" : "+v"(v));
  return v;
}

// The layered kernel: a workgroup owns a BX x BY tile of cells in the (x, y) plane and walks a
// segment of layers in z. In z the traces come from registers: the layer below has just been
// computed and the layer above is the next one to be computed, loaded a layer ahead. In x and y a
// lane reads the neighbour's line from U inside the tile; the lines of the cells around the tile
// are loaded during the sweeps of the layer before, by all lanes in turn, and reduced to (value,
// derivative) pairs. vmult and vmult_add only: the other epilogues' loads stay exposed here (the
// Chebyshev step measured slower than the single-layer one at every size).
template<int N, typename Number, ApplyMode mode>
__global__ void __launch_bounds__((CartTile<N, Number>::threads))
  __attribute__((amdgpu_waves_per_eu(CartTile<N, Number>::waves)))
  sipg_cartesian_layers_kernel(SipgArgs<Number> a)
{
  constexpr int N2 = N * N, N3 = N * N * N;
  using Tile       = CartTile<N, Number>;
  using L          = LdsLayout<N, Number>;
  using CT         = CartTable<N>;
  constexpr int BX = Tile::BX, BY = Tile::BY, T = Tile::threads;
  constexpr int R = (L::halo + T - 1) / T;  // halo lines per lane
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Number *        smem = reinterpret_cast<Number *>(smem_raw);
  Trace<Number> * halo = reinterpret_cast<Trace<Number> *>(smem + L::cells);
  Table<Number> const tables = (Table<Number>)a.tables;
  int const           tid = threadIdx.x, slot = tid / N2, lt = tid - slot * N2;
  int const           nx = a.topo.nc[0], ny = a.topo.nc[1], nz = a.topo.nc[2];
  int const           nxy = nx * ny;
  bool const          per2 = a.topo.periodic[2];

  // the tile: BX consecutive columns of the rows of BY cells, laid end to end (row_length
  // columns each, so that a tile may run over the end of a row)
  int const lb   = (int)xcd_logical_block(blockIdx.x, gridDim.x);
  int const seg  = lb / a.tiles;
  int const col0 = (lb - seg * a.tiles) * BX;
  int const row0 = col0 / a.row_length, x0 = col0 - row0 * a.row_length;
  int const z0 = seg * a.layers_per_segment, z1 = min(z0 + a.layers_per_segment, nz);
  bool const short_rows = a.row_length < BX;  // a tile spans several rows
  auto       column     = [&](int sx, int & x, int & y) {  // cell (x, y) of column sx, lowest row
    int row = row0;
    x       = x0 + sx;
    if(short_rows)
    {
      row += x / a.row_length;
      x %= a.row_length;
    }
    else if(x >= a.row_length)
    {
      x -= a.row_length;
      ++row;
    }
    y = row * BY;
    return x < nx && y < ny;
  };
  // z-lines, in the order of the vector: this lane's line of the layer and of the one above
  int           x, y;
  bool          active = column(slot % BX, x, y) && slot < Tile::cells;
  y += slot / BX;
  active               = active && y < ny;
  int const     line_map[2] = {a.line_map[tid], a.line_map[T + tid]};
  size_t const  plane       = (size_t)nxy * N3;
  size_t        g0          = (active ? (size_t)(x + nx * y) * N3 + lt : 0) + (size_t)z0 * plane;
  int const     bz          = (active ? slot : 0) * L::S + lt % N + N * (lt / N);
  Number        own[N], nxt[N];
  Trace<Number> below = {};  // of the layer below
  Number const * next = a.src + g0;
  if(active)
  {
    load_line<N>(next, N2, own);
    if(z0 > 0 || per2)
      load_line<N>(next + (z0 > 0 ? 0 : nz * plane) - plane, N2, nxt);
  }

  // The tile's tables in LDS, one lane per cell or halo face: where the exterior traces of its x-
  // and y-faces come from, and the penalties. tau_K is a sum over the directions
  // (interior_penalty_parameter.h:43-99) that grows with the cell's boundary faces, tau of a face
  // the larger one of its two cells, here times the scale c_d of the Kronecker term: with
  // M_d = h_d M (unit-interval mass M),
  //   out = M_z M_y (c_x L_x u) + M_z M_x (c_y L_y u) + M_y M_x (c_z L_z u),
  // c_x = h_y h_z, c_y = h_x h_z, c_z = h_x h_y, so that every mass sweep is a plain M.
  Number * const taus  = smem + L::tau;
  int * const    cells = reinterpret_cast<int *>(smem + L::size), *faces = cells + 2 * Tile::cells;
  auto face_tau = [&](int d, int n0, int n1, int n2) {
    return Number(a.tau_base + n0 * a.tau_step[0] + n1 * a.tau_step[1] + n2 * a.tau_step[2]) * a.scale[d];
  };
  // number of boundary faces of a cell along d; the larger one of the cell and its neighbour
  auto count = [&](int d, int c) {
    return a.topo.periodic[d] ? 0 : (c == 0) + (c == a.topo.nc[d] - 1);
  };
  auto face_count = [&](int d, int c, int side) {
    int const n = a.topo.nc[d], near = side ? c >= n - 2 || c == 0 : c <= 1 || c == n - 1;
    return a.topo.periodic[d] ? 0 : near + (n == 1);
  };
  if(tid < Tile::cells)
  {
    int const sy = tid / BX, sx = tid - sy * BX;
    int       cx, cy;
    bool      ok = column(sx, cx, cy);
    cy += sy;
    ok      = ok && cy < ny;
    int f   = 0;
    int c[2] = {cx, cy};
#pragma unroll
    for(int d = 0; d < 2; ++d)
    {
      int const s = d ? sy : sx, last = (d ? BY : BX) - 1, end = a.topo.periodic[d] ? 0 : kMirror;
      f |= (s > 0 && c[d] > 0 ? kInside : c[d] == 0 ? end : 0) << (4 * d);
      f |= (s < last && c[d] < a.topo.nc[d] - 1 ? kInside : c[d] == a.topo.nc[d] - 1 ? end : 0) << (4 * d + 1);
    }
    int const n0 = count(0, cx), n1 = count(1, cy);
    int       nf[4];
#pragma unroll
    for(int k = 0; k < 4; ++k)
    {
      nf[k] = face_count(k / 2, c[k / 2], k & 1);
      f |= nf[k] << (12 + 2 * k);
      taus[6 * tid + k] = k < 2 ? face_tau(0, nf[k], n1, 0) : face_tau(1, n0, nf[k], 0);
    }
    taus[6 * tid + 4] = face_tau(2, n0, n1, 0);
    cells[2 * tid]     = ok ? cx + nx * cy : -1;
    cells[2 * tid + 1] = f | n0 << 8 | n1 << 10;
  }
  else if(tid >= T - L::n_faces)
  {
    // the cell behind the face: x-faces (2 per row of the tile), then y-faces (2 per column). The
    // upper x-face belongs to the last column of the tile (tiles of periodic boxes end with the
    // row, the others may run on, where the end of a row is a boundary)
    int const  f = tid - (T - L::n_faces), side = f & 1;
    bool const is_x = f < 2 * BY;
    int const  last = a.topo.periodic[0] ? min(BX - 1, nx - 1 - x0) : BX - 1;
    int        cx, cy;
    bool       ok = column(is_x ? side * last : (f - 2 * BY) >> 1, cx, cy);
    if(is_x)
    {
      cy += f >> 1;
      ok = ok && cy < ny;
      cx += 2 * side - 1;
      if(cx < 0 || cx >= nx)
      {
        ok = ok && a.topo.periodic[0];
        cx = cx < 0 ? nx - 1 : 0;
      }
    }
    else
    {
      cy = side ? min(cy + BY, ny) : cy - 1;
      if(cy < 0 || cy >= ny)
      {
        ok = ok && a.topo.periodic[1];
        cy = cy < 0 ? ny - 1 : 0;
      }
    }
    faces[f] = ok ? cx + nx * cy : -1;
  }
  static_assert(Tile::cells + L::n_faces <= T, "one lane per cell and face of the tile");
  __syncthreads();

  // this lane's halo lines: the tile's faces with n^2 lines each
  Number const * hp[R];
  int            hkind[R];  // 0 none, 1 x-line, 2 y-line; + 4 at the upper side
  Number         hv[R][N];
#pragma unroll
  for(int k = 0; k < R; ++k)
  {
    int const  h = tid + k * T, f = h / N2, r = h - f * N2;
    bool const is_x = f < 2 * BY;
    int const  cell = h < L::halo ? faces[f] : -1;
    hkind[k]        = cell < 0 ? 0 : (is_x ? 1 : 2) + 4 * (f & 1);
    hp[k] = a.src + (cell < 0 ? 0 : (size_t)cell * N3 + (is_x ? N * r : r % N + N2 * (r / N)) + (size_t)z0 * plane);
  }
  auto load_halo = [&]() {
#pragma unroll
    for(int k = 0; k < R; ++k)
    {
      int const kind = opaque(hkind[k]);
      if(kind & 1)
        load_line<N>(hp[k], 1, hv[k]);
      if(kind & 2)
        load_line<N>(hp[k], N, hv[k]);
      hp[k] += plane;
    }
  };
  load_halo();

  // x- and y-lines: the lines of all cells of the tile are dealt out to the lanes by their LDS
  // banks (line_map), so that a group of lanes served together touches distinct banks
  int base[2], flags[2], hbase[2], tbase[2];  // flags < 0: no line
#pragma unroll
  for(int d = 0; d < 2; ++d)
  {
    int const  m = line_map[d], line = (m >> 16) & 127, sx = (m >> 23) & 7, sy = (m >> 26) & 7;
    int const  s  = sx + BX * sy;
    bool const ok = m >= 0 && cells[2 * s] >= 0;
    flags[d]      = ok ? cells[2 * s + 1] : -1;
    base[d]       = m & 0xffff;
    hbase[d]      = (d ? 2 * (BY + sx) : 2 * sy) * N2 + line;
    tbase[d]      = 6 * s + 2 * d;
  }

  if(active)
  {
    if(z0 > 0 || per2)
    {
      SplitLine<N, Number> const v(tables, nxt);
      below = {nxt[N - 1], v.du1};
    }
    if(z0 + 1 < nz || per2)
    {
      next += z0 + 1 < nz ? plane : plane - nz * plane;
      load_line<N>(next, N2, nxt);
    }
  }

  for(int z = z0; z < z1; ++z, g0 += plane)
  {
    // P0
    Table<Number> tab = fresh<Number>(tables);
    if(active)
      store_line<N>(smem + bz, L::PY, own);
#pragma unroll
    for(int k = 0; k < R; ++k)
    {
      int const kind = opaque(hkind[k]);
      if(kind)
      {
        SplitLine<N, Number> const v(tab, hv[k]);
        halo[tid + k * T] = kind & 4 ? Trace<Number>{hv[k][0], v.du0} : Trace<Number>{hv[k][N - 1], v.du1};
      }
    }
    __syncthreads();
    // P1
    tab = fresh<Number>(tables);
    Number rx[N];
    // the layers at the ends of the mesh have larger penalties
    bool const end_layer = !per2 && (z < 2 || z >= nz - 2);
    if(active)
    {
      SplitLine<N, Number> const u(tab, own);
      Number                     v[N], tl = taus[6 * slot + 4], tr = tl;
      Trace<Number>              l = below, r = {nxt[0], dot_line<N>(tab + CT::D0, nxt)};
      below = {own[N - 1], u.du1};
      if(end_layer)
      {
        int const n0 = (cells[2 * slot + 1] >> 8) & 3, n1 = (cells[2 * slot + 1] >> 10) & 3;
        if(z == 0)
          l = mirrored<Number>(a.topo.bc[4], own[0], u.du0);
        if(z == nz - 1)
          r = mirrored<Number>(a.topo.bc[5], own[N - 1], u.du1);
        tl = face_tau(2, n0, n1, face_count(2, z, 0));
        tr = face_tau(2, n0, n1, face_count(2, z, 1));
      }
      line_laplacian<N, Number>(tab + CT::line(2), a.half[2], u, own[0], own[N - 1], l, r, tl, tr, v);
      store_line<N>(smem + 2 * L::PC + bz, L::PY, v);
    }
#pragma unroll
    for(int d = 1; d >= 0; --d)
    {
      int const flag = opaque(flags[d]);
      if(flag >= 0)
      {
        constexpr int strides[2] = {1, N}, across[2] = {L::S, BX * L::S};
        Number *      U = smem + base[d];
        Number        u[N], v[N];
        Trace<Number> t[2] = {halo[hbase[d]], halo[hbase[d] + N2]};
        load_line<N>(U, strides[d], u);
        if(flag & (kInside << (4 * d)))
        {
          load_line<N>(U - across[d], strides[d], v);
          t[0] = {v[N - 1], -dot_reversed<N, Number>(tab + CT::D0, v)};
        }
        if(flag & (kInside << (4 * d + 1)))
        {
          load_line<N>(U + across[d], strides[d], v);
          t[1] = {v[0], dot_line<N>(tab + CT::D0, v)};
        }
        SplitLine<N, Number> const w(tab, u);
        if(flag & (kMirror << (4 * d)))
          t[0] = mirrored<Number>(a.topo.bc[2 * d], u[0], w.du0);
        if(flag & (kMirror << (4 * d + 1)))
          t[1] = mirrored<Number>(a.topo.bc[2 * d + 1], u[N - 1], w.du1);
        Number tl = taus[tbase[d]], tr = taus[tbase[d] + 1];
        if(end_layer)
        {
          int const lo = (flag >> (12 + 4 * d)) & 3, up = (flag >> (14 + 4 * d)) & 3;
          int const other = (flag >> (10 - 2 * d)) & 3, nz_ = count(2, z);
          tl = d ? face_tau(1, other, lo, nz_) : face_tau(0, lo, other, nz_);
          tr = d ? face_tau(1, other, up, nz_) : face_tau(0, up, other, nz_);
        }
        line_laplacian<N, Number>(tab + CT::line(d), a.half[d], w, u[0], u[N - 1], t[0], t[1], tl, tr, v);
        if(d == 1)
          store_line<N>(U + L::PC, N, v);
        else
#pragma unroll
          for(int i = 0; i < N; ++i)
            rx[i] = v[i];
      }
    }
    __syncthreads();
    // the layer above becomes the current one; the next layer's lines are loaded during the sweeps
#pragma unroll
    for(int m = 0; m < N; ++m)
      own[m] = nxt[m];
    if(z + 1 < z1)
    {
      load_halo();
      if(active && (z + 2 < nz || per2))
      {
        next += plane;
        if(z + 2 == nz)  // around the periodic box
          next -= nz * plane;
        load_line<N>(next, N2, nxt);
      }
    }
    // P2
    tab = fresh<Number>(tables);
    if(opaque(flags[0]) >= 0)
    {
      Number * U = smem + base[0];
      Number   v[N], w[N];
      store_line<N>(U, 1, rx);
      load_line<N>(U + L::PC, 1, v);
      cs_apply<N>(tab + CT::M, v, w);
      store_line<N>(U + L::PC, 1, w);
      load_line<N>(U + 2 * L::PC, 1, v);
      cs_apply<N>(tab + CT::M, v, w);
      store_line<N>(U + 2 * L::PC, 1, w);
    }
    __syncthreads();
    // P3
    tab = fresh<Number>(tables);
    if(opaque(flags[1]) >= 0)
    {
      Number * U = smem + base[1];
      Number   v[N], w[N];
      load_line<N>(U, N, v);
      cs_apply<N>(tab + CT::M, v, w);
      store_line<N>(U, N, w);
      load_line<N>(U + 2 * L::PC, N, v);
      cs_apply<N>(tab + CT::M, v, w);
      store_line<N>(U + 2 * L::PC, N, w);
    }
    __syncthreads();
    // P4: out = M_z (U + A) + B along z-lines
    tab = fresh<Number>(tables);
    Number out[N];
    if(active)
    {
      Number v[N], w[N];
      load_line<N>(smem + bz, L::PY, v);
      load_line<N>(smem + bz + L::PC, L::PY, w);
#pragma unroll
      for(int i = 0; i < N; ++i)
        v[i] += w[i];
      cs_apply<N>(tab + CT::M, v, out);
      load_line<N>(smem + bz + 2 * L::PC, L::PY, v);
#pragma unroll
      for(int i = 0; i < N; ++i)
        out[i] += v[i];
    }
    if(active)
#pragma unroll
      for(int k = 0; k < N; ++k)
      {
        if constexpr(mode == ApplyMode::vmult)
          store_stream(&a.dst[g0 + k * N2], out[k]);
        else
          a.dst[g0 + k * N2] += out[k];
      }
  }
}

// LDS strides of the single-layer kernel: along y (PX) and z (PY), from cell to cell (S, three
// buffers), and whether its lanes take the x- or y-lines with their upper coordinate fastest. A
// group of 16 FP64 (32 FP32) lanes is served in one pass if its addresses differ modulo 16 (32)
// entries; these are the strides with the fewest passes over the three directions that leave the
// number of workgroups per CU as it is (modeled passes per access 1.26 - 1.61 instead of 1.5 - 4.1
// dense). FP64 at n = 7 keeps wider strides with more modeled passes: with PY = 49, S = 1041, the
// x-lines swapped and even-odd end derivatives vmult and vmult_add took 2 - 6% longer on 16^3 to
// 32 x 31 x 30 cells (24 x 23 x 22: 32.4 / 31.4 us, vmult_add 34.9 / 33.8), most of it from the
// strides; both leave three workgroups per CU.
template<int N, typename Number>
struct CellLayout
{
  static constexpr bool dp = sizeof(Number) == 8;
  static constexpr int  PX = N == 2 ? 3 : N == 4 ? 5 : N;
  static constexpr int  PY = N == 2 ? 6 : N == 4 ? 20 : N == 6 ? (dp ? 41 : 37) : N == 7 ? 52 :
                             N == 8 ? (dp ? 65 : 67) : N * N;
  static constexpr int  PC = (N - 1) * (PX + PY) + N;
  static constexpr int  S  = N == 2 ? 36 : N == 3 ? 91 : N == 4 ? (dp ? 237 : 240) : N == 5 ? 381 :
                             N == 6 ? (dp ? 724 : 676) : N == 7 ? (dp ? 1107 : 1105) :
                             N == 8 ? (dp ? 1557 : 1599) : dp ? 2193 : 2201;
  static_assert(S >= 3 * PC, "three buffers per cell");
  static constexpr bool swap_x = dp ? N == 6 || N >= 8 : N == 7 || N == 8;
  static constexpr bool swap_y = !dp && (N == 6 || N == 8);
};

// The single-layer kernel: a workgroup takes 256 / n^2 consecutive cells of the traversal and reads
// their own and neighbour lines at its start. The phases are those above with one more barrier,
// since the y-neighbours' cells are staged through A and B.
template<int N, typename Number, ApplyMode mode>
__global__ void __launch_bounds__(256) sipg_cartesian_kernel(SipgArgs<Number> a)
{
  constexpr int N2 = N * N, N3 = N * N * N;
  constexpr int CPB = 256 / N2;
  using L           = CellLayout<N, Number>;
  using CT          = CartTable<N>;
  Table<Number> const tab = (Table<Number>)a.tables;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Number *      smem   = reinterpret_cast<Number *>(smem_raw);
  int const     slot   = threadIdx.x / N2;
  int const     lt     = threadIdx.x - slot * N2;
  int const     pos0   = (int)xcd_logical_block(blockIdx.x, gridDim.x) * CPB;
  bool const    active = slot < CPB && pos0 + slot < (int)a.n_cells;
  // three LDS buffers per cell: U (the cell's values), A and B; before the X phase A and B
  // stage the two y-neighbour cells
  Number *      U      = smem + (active ? slot : 0) * L::S;
  Number *      Abuf   = U + L::PC;
  Number *      Bbuf   = Abuf + L::PC;
  int const     p = lt % N, q = lt / N;
  // this lane's x-, y- and z-line: their two other coordinates, and their LDS bases
  int const     x_line = L::swap_x ? q + N * p : lt, y_line = L::swap_y ? q + N * p : lt;
  int const     bx = L::PX * (x_line % N) + L::PY * (x_line / N), by = y_line % N + L::PY * (y_line / N),
            bz = p + L::PX * q;

  int    type[3][2];
  Number tau[3][2];
  Trace<Number> t[3][2];
  Number own[N];  // this lane's z-line of the cell (lt + m N2), used by the Z phase
  int    cell       = 0;
  bool   in_block_l = false, in_block_r = false;
  if(active)
  {
    int cc[3];
    traversal_coords(a.topo, a.tile_rows, pos0, slot, cc);
    int const nx = a.topo.nc[0], ny = a.topo.nc[1];
    int const stride_c[3] = {1, nx, nx * ny};
    cell                  = cc[0] + nx * (cc[1] + ny * cc[2]);
    int nb[3][2];
#pragma unroll
    for(int d = 0; d < 3; ++d)
    {
      int const n_d = a.topo.nc[d], per = a.topo.periodic[d];
      int const t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
      int const fbase =
        (int)a.topo.face_base[d] + a.topo.layers[d] * (cc[t1] + a.topo.nc[t1] * cc[t2]);
      nb[d][0] = cc[d] > 0 ? cell - stride_c[d] : (per ? cell + (n_d - 1) * stride_c[d] : -1);
      nb[d][1] = cc[d] < n_d - 1 ? cell + stride_c[d] : (per ? cell - (n_d - 1) * stride_c[d] : -1);
      int const fr = (per && cc[d] + 1 == n_d) ? 0 : cc[d] + 1;
      tau[d][0]    = a.tau_face[fbase + cc[d]];
      tau[d][1]    = a.tau_face[fbase + fr];
#pragma unroll
      for(int s = 0; s < 2; ++s)
        type[d][s] = nb[d][s] >= 0 ? kInterior : a.topo.bc[2 * d + s];
    }
    {
      // All global loads up front. The own cell and the z- and y-neighbour cells are read in
      // the same pattern (lane lt reads DoFs lt + m N^2: consecutive lanes, consecutive
      // addresses); a lane then holds z-lines, so the z traces are lane-local and the
      // y-neighbour cells go through LDS (A, B) to be read as y-lines. Only x-neighbours at
      // the workgroup's ends are read as strided x-lines; the others come from U.
      Number const * own_p = a.src + (size_t)cell * N3 + lt;
      in_block_l = slot > 0 && cc[0] > 0;
      in_block_r = slot + 1 < CPB && cc[0] + 1 < a.topo.nc[0] && pos0 + slot + 1 < (int)a.n_cells;
      Number zl[N], zr[N], yl[N], yr[N], xl[N], xr[N];
      Number const * pz0 = a.src + (size_t)(nb[2][0] >= 0 ? nb[2][0] : cell) * N3 + lt;
      Number const * pz1 = a.src + (size_t)(nb[2][1] >= 0 ? nb[2][1] : cell) * N3 + lt;
      Number const * py0 = a.src + (size_t)(nb[1][0] >= 0 ? nb[1][0] : cell) * N3 + lt;
      Number const * py1 = a.src + (size_t)(nb[1][1] >= 0 ? nb[1][1] : cell) * N3 + lt;
#pragma unroll
      for(int m = 0; m < N; ++m)
      {
        own[m] = own_p[m * N2];
        zl[m]  = pz0[m * N2];
        zr[m]  = pz1[m * N2];
        yl[m]  = py0[m * N2];
        yr[m]  = py1[m * N2];
      }
      int const xbase = N * x_line;
      {
        Number const * px0 = a.src + (size_t)(nb[0][0] >= 0 ? nb[0][0] : cell) * N3 + xbase;
        Number const * px1 = a.src + (size_t)(nb[0][1] >= 0 ? nb[0][1] : cell) * N3 + xbase;
#pragma unroll
        for(int i = 0; i < N; ++i)
        {
          xl[i] = in_block_l ? Number(0) : px0[i];
          xr[i] = in_block_r ? Number(0) : px1[i];
        }
      }
      touch_tables<N, Number>(tab);
#pragma unroll
      for(int m = 0; m < N; ++m)
      {
        U[bz + L::PY * m]    = own[m];
        Abuf[bz + L::PY * m] = yl[m];
        Bbuf[bz + L::PY * m] = yr[m];
      }
      // lane-local traces (x ones are replaced from LDS for in-block neighbours)
      t[2][0] = {zl[N - 1], -dot_reversed<N, Number>(tab + CT::D0, zl)};
      t[2][1] = {zr[0], dot_line<N>(tab + CT::D0, zr)};
      t[0][0] = {xl[N - 1], -dot_reversed<N, Number>(tab + CT::D0, xl)};
      t[0][1] = {xr[0], dot_line<N>(tab + CT::D0, xr)};
    }
  }
  __syncthreads();
  // P1: the remaining neighbour traces, then the three line Laplacians into registers
  Number rx[N], ry[N], rz[N];
  if(active)
  {
    Number u[N], w[N];
    // y traces from the staged neighbour cells
    load_line<N>(Abuf + by, L::PX, w);
    t[1][0] = {w[N - 1], -dot_reversed<N, Number>(tab + CT::D0, w)};
    load_line<N>(Bbuf + by, L::PX, w);
    t[1][1] = {w[0], dot_line<N>(tab + CT::D0, w)};
    if(in_block_l)
    {
      load_line<N>(U - L::S + bx, 1, w);
      t[0][0] = {w[N - 1], -dot_reversed<N, Number>(tab + CT::D0, w)};
    }
    if(in_block_r)
    {
      load_line<N>(U + L::S + bx, 1, w);
      t[0][1] = {w[0], dot_line<N>(tab + CT::D0, w)};
    }
    auto laplacian = [&](int d, Number const(&v)[N], Number(&o)[N]) {
      SplitLine<N, Number> const s(tab, v);
      if(type[d][0] != kInterior)
        t[d][0] = mirrored<Number>(type[d][0], v[0], s.du0);
      if(type[d][1] != kInterior)
        t[d][1] = mirrored<Number>(type[d][1], v[N - 1], s.du1);
      line_laplacian<N, Number>(tab + CT::line(d), a.half[d], s, v[0], v[N - 1], t[d][0], t[d][1],
                                tau[d][0] * a.scale[d], tau[d][1] * a.scale[d], o);
    };
    load_line<N>(U + bx, 1, u);
    laplacian(0, u, rx);
    load_line<N>(U + by, L::PX, u);
    laplacian(1, u, ry);
    laplacian(2, own, rz);
  }
  __syncthreads();  // U, A and B are read across lanes up to here
  if(active)
  {
    store_line<N>(Abuf + bx, 1, rx);
    store_line<N>(Bbuf + by, L::PX, ry);
    store_line<N>(U + bz, L::PY, rz);
  }
  __syncthreads();
  // P2: B <- M_x B and U <- M_x U along x-lines, A <- M_y A along y-lines (each line in place:
  // in one phase every line of a buffer belongs to one lane)
  if(active)
  {
    Number v[N], w[N];
    load_line<N>(Bbuf + bx, 1, v);
    cs_apply<N>(tab + CT::M, v, w);
    store_line<N>(Bbuf + bx, 1, w);
    load_line<N>(U + bx, 1, v);
    cs_apply<N>(tab + CT::M, v, w);
    store_line<N>(U + bx, 1, w);
    load_line<N>(Abuf + by, L::PX, v);
    cs_apply<N>(tab + CT::M, v, w);
    store_line<N>(Abuf + by, L::PX, w);
  }
  __syncthreads();
  // P3: U <- M_y U along y-lines (the finished z-term); outp = M_z (A + B) along z-lines
  Number outp[N];
  if(active)
  {
    Number v[N], w[N];
    load_line<N>(U + by, L::PX, v);
    cs_apply<N>(tab + CT::M, v, w);
    store_line<N>(U + by, L::PX, w);
    load_line<N>(Abuf + bz, L::PY, v);
    load_line<N>(Bbuf + bz, L::PY, w);
#pragma unroll
    for(int i = 0; i < N; ++i)
      v[i] += w[i];
    cs_apply<N>(tab + CT::M, v, outp);
  }
  __syncthreads();
  if constexpr(mode == ApplyMode::residual_restrict)
  {
    // r = rhs - A u along the lane's z-line, restricted along z in registers, then along x and
    // y through A and B (free after the barrier above); the coarse cell is added to dst
    int const      nc = a.restrict_nc;
    Number const * P  = a.restrict_P;  // P[i nc + c]: fine node i, coarse node c
    if(active)
    {
      Number v[N], r[N];
      load_line<N>(U + bz, L::PY, v);
      size_t const g0 = (size_t)cell * N3 + lt;
#pragma unroll
      for(int k = 0; k < N; ++k)
        r[k] = a.rhs[g0 + k * N2] - (outp[k] + v[k]);
#pragma unroll
      for(int c = 0; c < N; ++c)
        if(c < nc)
        {
          Number s = 0;
#pragma unroll
          for(int k = 0; k < N; ++k)
            s += P[k * nc + c] * r[k];
          Abuf[lt + N2 * c] = s;  // (x, y, c_z)
        }
    }
    __syncthreads();
    if(active && lt < N * nc)
    {
      int const y = lt % N, cz = lt / N;
      for(int cx = 0; cx < nc; ++cx)
      {
        Number s = 0;
#pragma unroll
        for(int x = 0; x < N; ++x)
          s += P[x * nc + cx] * Abuf[x + N * y + N2 * cz];
        Bbuf[cx + nc * (y + N * cz)] = s;
      }
    }
    __syncthreads();
    if(active && lt < nc * nc)
    {
      int const     cx = lt % nc, cz = lt / nc;
      int64_t const nc3 = (int64_t)nc * nc * nc;
      for(int cy = 0; cy < nc; ++cy)
      {
        Number s = 0;
#pragma unroll
        for(int y = 0; y < N; ++y)
          s += P[y * nc + cy] * Bbuf[cx + nc * (y + N * cz)];
        a.dst[(int64_t)cell * nc3 + cx + nc * (cy + nc * cz)] += s;
      }
    }
    return;
  }
  // out = outp + the z-term held in U, along the z-lines
  if(active)
  {
    // direct per-lane stores: lane (p, q) owns the z-line of DoFs lt + k N2 (a workgroup-wide
    // LDS-staged store of the block's contiguous cells measured 10% slower)
    Number v[N];
    load_line<N>(U + bz, L::PY, v);
    size_t const g0 = (size_t)cell * N3 + lt;
#pragma unroll
    for(int k = 0; k < N; ++k)
    {
      Number const ax = outp[k] + v[k];
      size_t const g  = g0 + k * N2;
      if constexpr(mode == ApplyMode::vmult)
        store_stream(&a.dst[g], ax);
      else if constexpr(mode == ApplyMode::vmult_add)
        a.dst[g] += ax;
      else if constexpr(mode == ApplyMode::residual)
        a.dst[g] = a.rhs[g] - ax;
      else
      {
        Number r = (Number(1) + a.f1) * own[k] + a.f2 * a.dinv[g] * (a.rhs[g] - ax);
        if(a.has_old)
          r -= a.f1 * a.x_old[g];
        a.dst[g] = r;
      }
    }
  }
}

// How the layered kernel covers a box: tiles of BX columns of the rows of BY cells, laid end to end,
// and segments of layers
struct LayerTiling
{
  int row_length, tiles, segments, layers_per_segment;
};

template<int N, typename Number>
LayerTiling layer_tiling(BoxTopology const & t)
{
  using Tile   = CartTile<N, Number>;
  int const nx = t.nc[0], ny = t.nc[1], nz = t.nc[2];
  LayerTiling l;
  // a tile may run over the end of a row of tiles, except where the row's ends are neighbours
  l.row_length = t.periodic[0] ? (nx + Tile::BX - 1) / Tile::BX * Tile::BX : nx;
  l.tiles = (int)(((int64_t)((ny + Tile::BY - 1) / Tile::BY) * l.row_length + Tile::BX - 1) / Tile::BX);
  // 2 to 8 layers per segment, of nearly equal length, with some 4000 workgroups where there are
  // enough cells (longer segments leave the last round of workgroups uneven: 12 layers instead of 8
  // cost 9% at FP64 k = 4 on 64^3 cells)
  int const longest    = (int)std::max<int64_t>(2, std::min<int64_t>(8, (int64_t)nz * l.tiles / 4000));
  l.segments           = (nz + longest - 1) / longest;
  l.layers_per_segment = (nz + l.segments - 1) / l.segments;
  return l;
}

// Whether the layered kernel is the faster one: where its fewer reads count, as src and dst outgrow
// the 256 MB last-level cache, and with n <= 5 nodes per line, above which FP64 has too few waves
// (k = 5 on 48^3 cells 141 us against 131 single-layer, k = 7 on 40^3 207 against 183; FP32 was not
// tried there). The line lies between, layered against single-layer in us: FP64 k = 4 50^3 cells
// (125 MB) 94 / 87, 64^3 (262 MB) 165 / 177; k = 3 48^3 (57 MB) 44 / 43, 64^3 (134 MB) 85 / 94; k = 2
// 72^3 (81 MB) 60 / 60, 88^3 (147 MB) 100 / 104. FP32 k = 4 56^3 (88 MB) 69 / 74, k = 3 64^3 (67 MB)
// 51 / 54, k = 2 56^3 (19 MB) 21 / 23, k = 1 96^3 (28 MB) 30 / 34.
//
// It also takes a box that fills the tiles: lanes without a cell cost as much as the others. Layered
// against single-layer in us by the share of cells in the tiles: 1/50 (k = 1 on 1 x 1 x 480000)
// 327 / 33, 1/8 (690 x 1 x 690) 52 / 20, 1/4 (k = 3 on 420 x 1 x 420) 106 / 66, 1/2 (k = 1 on
// 350 x 4 x 350) 23 / 21, 0.6 (k = 4, 6 periodic cells along x) 161 / 134, 0.8 (8 along x) 143 / 135,
// 0.82 (k = 1, 33 along x) 18.9 / 18.3, 0.9 and more 0.75 - 0.97 times. One layer alone leaves n = 2
// with nothing to reuse (700 x 680 x 1 21.9 / 19.7; k = 2 on 400 x 400 x 1 20 / 21).
template<int N, typename Number>
bool use_layers(SipgArgs<Number> const & a)
{
  int64_t const bytes = a.n_cells * (N * N * N * sizeof(Number));
  if(bytes < 1000000 * (sizeof(Number) == 8 ? (N == 5 ? 180 : 90) : N >= 4 ? 60 : 15))
    return false;
  int const     nz    = a.topo.nc[2];
  int64_t const slots = (int64_t)layer_tiling<N, Number>(a.topo).tiles * CartTile<N, Number>::cells * nz;
  return 20 * a.n_cells >= 17 * slots && (N > 2 || nz > 1);
}

template<int N, typename Number, ApplyMode mode>
hipError_t launch_layers_n(SipgArgs<Number> a, hipStream_t stream)
{
  LayerTiling const l  = layer_tiling<N, Number>(a.topo);
  a.row_length         = l.row_length;
  a.tiles              = l.tiles;
  a.layers_per_segment = l.layers_per_segment;
  hipLaunchKernelGGL((sipg_cartesian_layers_kernel<N, Number, mode>), dim3((unsigned)l.tiles * l.segments),
                     dim3(CartTile<N, Number>::threads), (LdsLayout<N, Number>::bytes), stream, a);
  return hipGetLastError();
}

template<int N, typename Number, ApplyMode mode>
hipError_t launch_cartesian_n(SipgArgs<Number> const & a, hipStream_t stream)
{
  if constexpr(N <= kMaxLayered && (mode == ApplyMode::vmult || mode == ApplyMode::vmult_add))
    if(use_layers<N, Number>(a))
      return launch_layers_n<N, Number, mode>(a, stream);
  constexpr int CPB    = 256 / (N * N);
  int const     blocks = (int)((a.n_cells + CPB - 1) / CPB);
  size_t const  lds    = sizeof(Number) * CPB * CellLayout<N, Number>::S;
  hipLaunchKernelGGL((sipg_cartesian_kernel<N, Number, mode>), dim3(blocks), dim3(256), lds, stream, a);
  return hipGetLastError();
}

template<typename Number, ApplyMode mode>
hipError_t dispatch_cartesian(int degree, SipgArgs<Number> const & a, hipStream_t s)
{
  switch(degree)
  {
    case 1: return launch_cartesian_n<2, Number, mode>(a, s);
    case 2: return launch_cartesian_n<3, Number, mode>(a, s);
    case 3: return launch_cartesian_n<4, Number, mode>(a, s);
    case 4: return launch_cartesian_n<5, Number, mode>(a, s);
    case 5: return launch_cartesian_n<6, Number, mode>(a, s);
    case 6: return launch_cartesian_n<7, Number, mode>(a, s);
    case 7: return launch_cartesian_n<8, Number, mode>(a, s);
    case 8: return launch_cartesian_n<9, Number, mode>(a, s);
    default: return hipErrorInvalidValue;
  }
}

// Deals the lines of one direction (x: d = 0, y: d = 1) out to the lanes of a workgroup: `banks`
// consecutive lanes are served by LDS in one pass if their addresses differ modulo `banks`
// entries (16 for FP64, 32 for FP32), so each such group takes one line from every residue class,
// the fullest classes first
template<int N, typename Number>
void deal_lines(int d, int * map)
{
  using Tile = CartTile<N, Number>;
  using L    = LdsLayout<N, Number>;
  constexpr int                 banks = 128 / sizeof(Number), n_lines = Tile::cells * N * N;
  std::vector<std::vector<int>> left(banks);
  for(int i = n_lines - 1; i >= 0; --i)
  {
    int const line = i % (N * N);
    int const base = i / (N * N) * L::S + (d ? 1 : N) * (line % N) + L::PY * (line / N);
    left[base % banks].push_back(i);
  }
  std::fill(map, map + Tile::threads, -1);
  for(int done = 0; done < n_lines;)
  {
    int const        want = std::min(banks, n_lines - done);
    std::vector<int> order(banks);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int p, int q) { return left[p].size() > left[q].size(); });
    for(int k = 0; k < want; ++k)
    {
      int b = order[k];
      if(left[b].empty())  // no class unused in this group has a line left
        for(b = 0; b < banks; ++b)
          if(!left[b].empty())
            break;
      int const i = left[b].back(), cell = i / (N * N), line = i % (N * N);
      map[done++] = (cell * L::S + (d ? 1 : N) * (line % N) + L::PY * (line / N)) | line << 16 |
                    (cell % Tile::BX) << 23 | (cell / Tile::BX) << 26;
      left[b].pop_back();
    }
  }
}

template<int N, typename Number>
std::vector<int> line_map_n()
{
  std::vector<int> m(2 * CartTile<N, Number>::threads);
  for(int d = 0; d < 2; ++d)
    deal_lines<N, Number>(d, m.data() + d * CartTile<N, Number>::threads);
  return m;
}
}  // namespace

template<typename Number>
std::vector<int> cartesian_line_map(int degree)
{
  switch(degree)
  {
    case 1: return line_map_n<2, Number>();
    case 2: return line_map_n<3, Number>();
    case 3: return line_map_n<4, Number>();
    case 4: return line_map_n<5, Number>();
    default: return {};  // no layered kernel
  }
}

template<typename Number>
char const * cartesian_vmult_kernel(int degree, SipgArgs<Number> const & a)
{
  bool const layered = degree == 1 ? use_layers<2, Number>(a) : degree == 2 ? use_layers<3, Number>(a) :
                       degree == 3 ? use_layers<4, Number>(a) : degree == 4 && use_layers<5, Number>(a);
  return layered ? "sipg_cartesian_layers_kernel" : "sipg_cartesian_kernel";
}

template char const * cartesian_vmult_kernel<double>(int, SipgArgs<double> const &);
template char const * cartesian_vmult_kernel<float>(int, SipgArgs<float> const &);
template std::vector<int> cartesian_line_map<double>(int);
template std::vector<int> cartesian_line_map<float>(int);

template<typename Number>
hipError_t launch_sipg_cartesian(int degree, ApplyMode mode, SipgArgs<Number> const & a,
                                 hipStream_t s)
{
  switch(mode)
  {
    case ApplyMode::vmult: return dispatch_cartesian<Number, ApplyMode::vmult>(degree, a, s);
    case ApplyMode::vmult_add: return dispatch_cartesian<Number, ApplyMode::vmult_add>(degree, a, s);
    case ApplyMode::chebyshev:
      return dispatch_cartesian<Number, ApplyMode::chebyshev>(degree, a, s);
    case ApplyMode::residual: return dispatch_cartesian<Number, ApplyMode::residual>(degree, a, s);
    case ApplyMode::residual_restrict:
      if(a.restrict_P == nullptr || a.restrict_nc < 1 || a.restrict_nc > degree + 1)
        return hipErrorInvalidValue;
      return dispatch_cartesian<Number, ApplyMode::residual_restrict>(degree, a, s);
    case ApplyMode::diagonal: break;  // affine meshes have closed forms of the diagonal and the blocks
  }
  return hipErrorInvalidValue;
}

template hipError_t launch_sipg_cartesian<double>(int, ApplyMode, SipgArgs<double> const &, hipStream_t);
template hipError_t launch_sipg_cartesian<float>(int, ApplyMode, SipgArgs<float> const &, hipStream_t);
}  // namespace ExaDG
