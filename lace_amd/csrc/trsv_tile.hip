// trsv_tile.hip -- several Jacobi sweeps of a stencil's triangular factor
// in one launch.
//
// A one-sweep launch on the diagonal form reads the factor, r and the
// previous iterate and writes the next one: k sweeps move the factor and r
// k times and every intermediate iterate twice.  The factors of a 5- or
// 7-point stencil couple a row only to its grid neighbours one step back
// along each axis, so a workgroup that loads a box of the grid widened by C
// points on that side can run C sweeps on it alone: sweep s is right on the
// box widened by C - s.  The factor and r are read once (with the halo:
// mostly from the L2 of the XCD, whose workgroups hold the neighbouring
// boxes), the iterates stay in registers and LDS, and only the last one is
// written.  Five sweeps of L and U (two launches against eight, the first
// sweep being r or r / diag): 128^3 FP32 78 -> 30 us, FP64 136 -> 53 us,
// 64^3 FP32 24 -> 10 us, 64^2 FP64 21 -> 6.6 us.  What bounds a launch now is
// the load phase (L 12 us for 44 MB at 128^3 FP32, U 17 us for 52 MB, of
// which about 3 us are the launch's start and end): all resident boxes load,
// then all compute.  Multiplying by a reciprocal formed once per row (with
// corrections that round as the division does) instead of dividing in every
// sweep measured slower (U 17.8 -> 22 us): the exact test of each quotient
// and its registers cost more than the division's instructions, which run
// under the other workgroups' loads.
#include <type_traits>

#include "common.hpp"
#include "device.hpp"
#include "parilu.hpp"
#include "trsv_tile.hpp"

namespace lace {

namespace {

// V consecutive values at row i (a multiple of V): a uniform base and a
// 32-bit byte offset, the addressing mode that needs no 64-bit arithmetic
// per lane (the launcher keeps rows * element size under 2^31).
template <int V, typename T>
__device__ __forceinline__ void ldw(const T* __restrict__ base, unsigned i, T (&v)[V]) {
  const T* p = reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (unsigned)sizeof(T));
  if constexpr (V == 1) v[0] = *p;
  else wload<T, V>(p, v);
}

// Factor values of one unit: FP32 / FP64 as stored, 16-bit words decoded
// with the rows' scales.
template <typename T, typename TS, int V>
__device__ __forceinline__ void ldf(const TS* __restrict__ base, unsigned i, const T (&sc)[V], T (&v)[V]) {
  if constexpr (std::is_same<T, TS>::value) {
    ldw<V, T>(base, i, v);
  } else {
    uint16_t h[V];
    ldw<V, uint16_t>(reinterpret_cast<const uint16_t*>(base), i, h);
#pragma unroll
    for (int k = 0; k < V; k++) v[k] = dequant<T, TS>(__builtin_bit_cast(TS, h[k]), sc[k]);
  }
}

template <int V, typename T>
__device__ __forceinline__ void lds_get(const T* p, T (&v)[V]) {
  if constexpr (V == 1) v[0] = *p;
  else wload<T, V>(p, v);
}
template <int V, typename T>
__device__ __forceinline__ void lds_put(T* p, const T (&v)[V]) {
  if constexpr (V == 1) *p = v[0];
  else wstore<T, V>(p, v);
}

__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }

}  // namespace

// C coupled sweeps y <- D^-1 (r - N y) on one box.  A unit is V rows along
// x (a 16-byte word; V = 1 where the grid's lines do not keep that
// alignment); thread t owns units t, t + BS, ... of the widened box in
// lexicographic order, so unit u's rows sit at u V of the LDS image and its
// neighbours one line and one plane away.  A unit's values, r, diagonal and
// iterate stay in registers; each sweep reads the neighbours' previous
// iterate from one LDS image and writes the other.  Rows outside the grid
// hold zeros, which add nothing to a sum (a row has an entry for every
// neighbour inside the grid: TriPlan::grid); rows on the widened box's
// edges read unrelated LDS words and are never read in turn by a row that
// is still right.  Each row's sum runs in CSR order, so results are
// bit-identical to one-sweep launches.
template <typename T, typename TS, int V, bool UPPER, bool UNIT, int D, int BS, int U>
__global__ __launch_bounds__(BS, 4) void tri_jacobi_tile_kernel(
    TileShape g, const int8_t* __restrict__ dexp, const TS* __restrict__ dia, const TS* __restrict__ dval,
    const T* __restrict__ r, const T* __restrict__ yin, T* __restrict__ yout) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) T img[2][BS * U * V];
  const int tile = xcd_block(blockIdx.x, gridDim.x);
  const int tx = tile % g.tx, tyz = tile / g.tx;
  const int ty = tyz % g.ty, tz = tyz / g.ty;
  // corner of the widened box: the halo is on the side the factor reads from
  const int cx = tx * g.bx - (UPPER ? 0 : g.hx), cy = ty * g.by - (UPPER ? 0 : g.hy),
            cz = tz * g.bz - (UPPER ? 0 : g.hz);
  const int line = g.ex, plane = g.ex * g.ey, rows = plane * g.ez;
  T v[U][D][V], rr[U][V], dd[U][V], y[U][V];
  unsigned row[U];
  bool in[U], core[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    // (ux, uy, uz) of the unit by multiplication: exact for the at most
    // 4096 units of a box
    const unsigned e = threadIdx.x + BS * u;
    const unsigned l = (e * g.mx) >> 20;
    const int uz = (int)((l * g.my) >> 20);
    const int uy = (int)l - uz * g.ey, ux = ((int)e - (int)l * g.nux) * V;
    const int x = cx + ux, yy = cy + uy, z = cz + uz;
    in[u] = (unsigned)x < (unsigned)g.nx && (unsigned)yy < (unsigned)g.ny && (unsigned)z < (unsigned)g.nz &&
            uz < g.ez;
    core[u] = UPPER ? ux < g.bx && uy < g.by && uz < g.bz : ux >= g.hx && uy >= g.hy && uz >= g.hz;
    row[u] = (unsigned)(x + g.nx * (yy + g.ny * z));
    if (in[u]) {
      T sc[V];
      if constexpr (!std::is_same<T, TS>::value) {
        int8_t ex[V];
        ldw<V, int8_t>(dexp, row[u], ex);
#pragma unroll
        for (int k = 0; k < V; k++) sc[k] = ldexpf(1.0f, (int)ex[k]);
      }
      ldw<V, T>(r, row[u], rr[u]);
      if constexpr (!UNIT) ldf<T, TS, V>(dval, row[u], sc, dd[u]);
      if (yin) ldw<V, T>(yin, row[u], y[u]);
#pragma unroll
      for (int q = 0; q < D; q++) ldf<T, TS, V>(dia + (size_t)q * g.n, row[u], sc, v[u][q]);
    }
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int e0 = ((int)threadIdx.x + BS * u) * V;
    if (in[u]) {
      if (!yin) {
#pragma unroll
        for (int k = 0; k < V; k++) y[u][k] = UNIT ? rr[u][k] : rr[u][k] / dd[u][k];
      }
      lds_put<V, T>(&img[0][e0], y[u]);
    } else {
      const T zero[V] = {};
      lds_put<V, T>(&img[0][e0], zero);
      lds_put<V, T>(&img[1][e0], zero);
    }
  }
  __syncthreads();
  for (int s = 1; s <= g.c; s++) {
    const T* src = img[(s - 1) & 1];
    T* dst = img[s & 1];
    // the outermost s layers are no longer right and no longer needed (nor
    // would their neighbours lie inside the image)
    const int gone = s * (D == 3 ? plane : line);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int e0 = ((int)threadIdx.x + BS * u) * V;
      if (!in[u] || (UPPER ? e0 >= rows - gone : e0 < gone)) continue;
      T ny[V], nz[V], o[V];
      // along x the neighbours are the unit's own rows but for one
      const T edge = src[UPPER ? e0 + V : e0 - 1];
      lds_get<V, T>(src + (UPPER ? e0 + line : e0 - line), ny);
      if constexpr (D == 3) lds_get<V, T>(src + (UPPER ? e0 + plane : e0 - plane), nz);
#pragma unroll
      for (int k = 0; k < V; k++) {
        const T nx = UPPER ? (k + 1 < V ? y[u][(k + 1) % V] : edge) : (k > 0 ? y[u][(k + V - 1) % V] : edge);
        // the first term starts from +0 (a fused multiply-add with zero
        // rounds once, as the product does)
        T t;
        if constexpr (UPPER) {
          t = fma_t(v[u][0][k], nx, T(0));
          t = t + v[u][1][k] * ny[k];
          if constexpr (D == 3) t = t + v[u][2][k] * nz[k];
        } else if constexpr (D == 3) {
          t = fma_t(v[u][0][k], nz[k], T(0));
          t = t + v[u][1][k] * ny[k];
          t = t + v[u][2][k] * nx;
        } else {
          t = fma_t(v[u][0][k], ny[k], T(0));
          t = t + v[u][1][k] * nx;
        }
        o[k] = UNIT ? rr[u][k] - t : (rr[u][k] - t) / dd[u][k];
      }
#pragma unroll
      for (int k = 0; k < V; k++) y[u][k] = o[k];
      if (s < g.c) lds_put<V, T>(dst + e0, o);
      else if (core[u])
        lds_put<V, T>(reinterpret_cast<T*>(reinterpret_cast<char*>(yout) + row[u] * (unsigned)sizeof(T)), o);
    }
    if (s < g.c) __syncthreads();
  }
}

// Box sides, threads and units a thread of a form: V rows a unit along x, D
// couplings.  The widened box's units must fit BS * U for the C <= kTileC
// sweeps of one launch.  At 128^3 FP32 the boxes between 16 x 8 x 8 and
// 32 x 16 x 16 all take 12.1-12.9 (L) and 16.9-17.9 (U) us: what a larger
// box saves in halo it loses in workgroups per CU; two (FP64: three) units
// a thread leave room for several workgroups.  Lines that do not keep the
// word's alignment (V = 1) move single rows and take a larger box for it.
template <typename T, int V, int D>
struct TileForm {
  static constexpr int BS = 512;
  static constexpr int U = D == 2 ? (V == 1 ? 2 : 1) : V == 1 ? (sizeof(T) == 8 ? 6 : 8) : sizeof(T) == 8 ? 3 : 2;
  static constexpr int BX = D == 2 ? (V == 4 ? 64 : V == 2 ? 32 : 28) : V == 1 ? 12 : 16;
  static constexpr int BY = D == 2 ? (V == 1 ? 28 : 24) : V == 1 ? 12 : 8;
  static constexpr int BZ = D == 2 ? 1 : V == 1 && sizeof(T) == 4 ? 12 : 8;
  static constexpr int HX = (kTileC + V - 1) / V * V;
  static_assert((BX + HX) / V * (BY + kTileC) * (D == 2 ? 1 : BZ + kTileC) <= BS * U, "box too large");
};

template <typename T, typename TS, int V, bool UPPER, bool UNIT, int D>
static void tile_launch(const TriPlan& P, const TS* dia, const TS* dval, const T* r, const T* yin, T* yout, int c,
                        TimedRegion& tr) {
  using F = TileForm<T, V, D>;
  TileShape g;
  g.n = P.n;
  g.nx = P.grid[0], g.ny = P.grid[1], g.nz = P.grid[2];
  g.c = c;
  g.hx = ceil_div(c, V) * V, g.hy = c, g.hz = D == 3 ? c : 0;
  g.bx = F::BX, g.by = F::BY, g.bz = F::BZ;
  // FP32 grids with many boxes a CU: a higher box saves halo (128^3: 29.9
  // against 30.9 us for L and U; on 100 x 77 x 53, with two boxes a CU, the
  // smaller box is ahead, 12.9 against 13.6 us)
  if (D == 3 && V == 4 && P.n >= (1 << 20)) g.by = 12;
  g.ex = g.bx + g.hx, g.ey = g.by + g.hy, g.ez = g.bz + g.hz;
  g.tx = ceil_div(g.nx, g.bx), g.ty = ceil_div(g.ny, g.by), g.tz = ceil_div(g.nz, g.bz);
  g.nux = g.ex / V;
  g.mx = ((1u << 20) + g.nux - 1) / g.nux;
  g.my = ((1u << 20) + g.ey - 1) / g.ey;
  tr.launch(tri_jacobi_tile_kernel<T, TS, V, UPPER, UNIT, D, F::BS, F::U>, dim3(g.tx * g.ty * g.tz), dim3(F::BS), g,
            (const int8_t*)P.dexp.p, dia, dval, r, yin, yout);
}

template <typename T, typename TS, int V>
static void tile_dispatch(const TriPlan& P, const TS* dia, const TS* dval, const T* r, const T* yin, T* yout, int c,
                          TimedRegion& tr) {
#define LACE_TILE_CASE(UP, UN, D)                                              \
  if (P.upper == UP && P.unit_diag == UN && P.dia.nd == D)                     \
    return tile_launch<T, TS, V, UP, UN, D>(P, dia, dval, r, yin, yout, c, tr)
  LACE_TILE_CASE(false, true, 3);
  LACE_TILE_CASE(true, false, 3);
  LACE_TILE_CASE(false, true, 2);
  LACE_TILE_CASE(true, false, 2);
  if constexpr (std::is_same<T, TS>::value) {  // U^T and L^T hold no 16-bit form
    LACE_TILE_CASE(false, false, 3);
    LACE_TILE_CASE(true, true, 3);
    LACE_TILE_CASE(false, false, 2);
    LACE_TILE_CASE(true, true, 2);
  }
#undef LACE_TILE_CASE
}

static bool has16(const TriPlan& P) {
  return P.grid[0] > 0 && P.dia16_fmt != LACE_F32 && P.dia16_src != nullptr && P.dia16_src == P.strict_src &&
         P.upper != P.unit_diag && (double)P.n * sizeof(float) < 2147483648.0 &&
         get_option("jacobi_dia16", 1) != 0 && get_option("jacobi_dia", 1) != 0 &&
         get_option("jacobi_dia_vec", 1) != 0;
}

// Option "jacobi_tile": 1 where boxes are ahead of one-sweep launches, 2
// wherever there is such a form, 0 never.  They are ahead at two sweeps and
// more but on large 3-D grids whose lines do not keep the 16-byte word of four
// rows: there a unit is one row, whose loads, 2 bytes wide for 16-bit words,
// cost more than one coupled sweep saves, and in 16 bits more than two save;
// below these sizes the launches saved make up for it.  Two sweeps of L and U,
// one-sweep launches -> boxes: 77 x 53 x 100 FP32 9.4 -> 12.3 us, 61 x 60 x 61
// 12.4 -> 10.7, 127 x 129 x 128 FP32 24 -> 29, BF16 22 -> 35, FP64 41 -> 36;
// three: 127 x 129 x 128 BF16 32.7 -> 40.6, FP32 39 -> 35, 90^3 BF16 18.7 ->
// 15.8; four, BF16 there 55 -> 51.
static bool tile_pays(const TriPlan& P, int W, int sweeps, bool d16) {
  const int tile = get_option("jacobi_tile", 1);
  if (sweeps < 2 || tile != 1) return sweeps >= 2 && tile == 2;
  if (P.dia.nd != 3 || W != 4 || P.grid[0] % 4 == 0) return true;
  return sweeps == 2 ? P.n < (1 << 18) : sweeps > 3 || !d16 || P.n < (1 << 20);
}

bool jacobi_tile16(const TriPlan& P, int sweeps) { return has16(P) && tile_pays(P, 4, sweeps, true); }

template <typename T>
bool jacobi_tile_ready(const TriPlan& P, const T* val, int sweeps) {
  if (P.grid[0] == 0 || P.strict_src != (const void*)val) return false;
  const bool d16 = sizeof(T) == 4 && has16(P);
  if (!tile_pays(P, 16 / (int)sizeof(T), sweeps, d16)) return false;
  if (d16) return true;
  return !(P.stale & TriPlan::kFormDia) && (P.unit_diag || !(P.stale & TriPlan::kFormDiag)) &&
         (double)P.n * sizeof(T) < 2147483648.0 && get_option("jacobi_dia", 1) != 0 &&
         get_option("jacobi_dia_vec", 1) != 0;
}

template <typename T>
int jacobi_tile(const TriPlan& P, const T* r, const T* yin, T* yout, int c) {
  constexpr int W = 16 / (int)sizeof(T);
  const auto al16 = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
  const bool vec = P.grid[0] % W == 0 && al16(r) && al16(yin) && al16(yout);
  const bool d16 = sizeof(T) == 4 && has16(P);
  const double es = sizeof(T), n = P.n, fs = d16 ? 2.0 : es;
  TimedRegion tr(P.upper ? "trsv_jacobi_sweep_upper" : "trsv_jacobi_sweep_lower", 0.0,
                 (P.dia.nd + (P.unit_diag ? 0 : 1)) * fs * n + (d16 ? n : 0.0) + (yin ? 3.0 : 2.0) * es * n, true);
  if constexpr (sizeof(T) == 4) {
    if (d16 && P.dia16_fmt == LACE_BF16) {
      const uint16_t *dv = P.dia16.as<uint16_t>(), *dg = P.dval16.as<uint16_t>();
      if (vec) tile_dispatch<float, uint16_t, W>(P, dv, dg, r, yin, yout, c, tr);
      else tile_dispatch<float, uint16_t, 1>(P, dv, dg, r, yin, yout, c, tr);
      LACE_HIP(hipGetLastError());
      return DEV_SUCCESS;
    }
    if (d16) {
      const _Float16 *dv = P.dia16.as<_Float16>(), *dg = P.dval16.as<_Float16>();
      if (vec) tile_dispatch<float, _Float16, W>(P, dv, dg, r, yin, yout, c, tr);
      else tile_dispatch<float, _Float16, 1>(P, dv, dg, r, yin, yout, c, tr);
      LACE_HIP(hipGetLastError());
      return DEV_SUCCESS;
    }
  }
  const T *dv = P.dia.val.as<T>(), *dg = P.dval.as<T>();
  if (vec) tile_dispatch<T, T, W>(P, dv, dg, r, yin, yout, c, tr);
  else tile_dispatch<T, T, 1>(P, dv, dg, r, yin, yout, c, tr);
  LACE_HIP(hipGetLastError());
  return DEV_SUCCESS;
}

template bool jacobi_tile_ready<float>(const TriPlan&, const float*, int);
template bool jacobi_tile_ready<double>(const TriPlan&, const double*, int);
template int jacobi_tile<float>(const TriPlan&, const float*, const float*, float*, int);
template int jacobi_tile<double>(const TriPlan&, const double*, const double*, double*, int);

}  // namespace lace
