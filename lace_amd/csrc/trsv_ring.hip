// trsv_ring.hip -- exact triangular solve by one workgroup in level order.
//
// A solve spread over the chip pays a device-coherent store and load for
// every dependency that crosses workgroups.  Where the rows a level reads
// lie at most an LDS image's worth of rows back in level order, one
// workgroup keeps the last rows of the solution in a ring in LDS and steps
// level by level with a workgroup barrier: a level then costs an LDS round
// trip, the row sums, the division and the barrier (0.19 us together), and
// what bounds a large factor is the rate at which one CU streams its entries
// (110 GB/s measured).  L and U together, persistent kernel -> this one:
// 64 x 64 5-point FP64 130 -> 61 us, 20^3 7-point FP64 77 -> 41 us, ragged
// 24 x 25 x 23 mesh FP64 506 -> 152 us, 43 x 47 x 45 mesh FP32 1037 -> 336 us.
// Forming FP64 reciprocals ahead of the barrier and correcting the quotient
// by its remainder was slower than dividing (75 against 66 us on 64 x 64: the
// exponent test and its branch cost what the division's steps do).
#include <algorithm>
#include <new>
#include <system_error>

#include "common.hpp"
#include "device.hpp"
#include "parilu.hpp"

namespace lace {

namespace {

constexpr int kRingBytes = 128 * 1024;   // the solution's last rows
constexpr int kRingDescs = 4064;         // chunk descriptors beside them (32 KB)
constexpr int kRingWaves = 16;           // most waves of the workgroup
constexpr int kRingLevelBits = 17;

template <typename T>
constexpr int ring_rows() {
  return kRingBytes / (int)sizeof(T);
}

}  // namespace

// Chunk blockIdx.x's operands, four slots of every row to a group: their
// places in level order modulo 2^15 (0xFFFF: no operand).  The block past
// the last chunk fills the group no chunk owns.
__global__ __launch_bounds__(64) void ring_index_kernel(int nchunks, const uint2* __restrict__ desc,
                                                        const int* __restrict__ perm,
                                                        const int* __restrict__ row, const int* __restrict__ col,
                                                        const int* __restrict__ pos, bool upper, int groups,
                                                        uint16_t* __restrict__ idx) {
  const int c = blockIdx.x, t = threadIdx.x;
  const bool extra = c == nchunks;
  const unsigned x = extra ? (unsigned)groups << 11 | 1u : desc[c].x;
  const int i = extra ? -1 : perm[(size_t)c * 64 + t];
  const int k0 = i < 0 ? 0 : row[i] + (upper ? 1 : 0), len = i < 0 ? 0 : row[i + 1] - row[i] - 1;
  for (int q = 0; q < (int)(x & 15u) * 4; q++)
    idx[((size_t)(x >> 11) + q / 4) * 256 + t * 4 + q % 4] = q < len ? (uint16_t)(pos[col[k0 + q]] & 32767) : 0xFFFF;
}

// The factor's values and diagonal in the same order (no entry: 0, no row:
// 1).  A group's values are 16-byte words, lane by lane: FP32 one word a
// lane, FP64 the first two values of every lane, then the last two (a load
// then covers whole lines).
template <typename T>
__global__ __launch_bounds__(64) void ring_gather_kernel(int nchunks, const uint2* __restrict__ desc,
                                                         const int* __restrict__ perm,
                                                         const int* __restrict__ row, bool upper, size_t slots,
                                                         const T* __restrict__ val, T* __restrict__ out,
                                                         T* __restrict__ diag) {
  const int c = blockIdx.x, t = threadIdx.x;
  if (c == nchunks) {
    for (int q = 0; q < 4; q++) out[slots - 256 + t * 4 + q] = T(0);
    return;
  }
  const unsigned x = desc[c].x;
  const int i = perm[(size_t)c * 64 + t];
  const int r0 = i < 0 ? 0 : row[i], len = i < 0 ? 0 : row[i + 1] - r0 - 1;
  const int k0 = upper ? r0 + 1 : r0;
  for (int q = 0; q < (int)(x & 15u) * 4; q++) {
    const int w = sizeof(T) == 4 ? t * 4 + q % 4 : (q % 4) / 2 * 128 + t * 2 + q % 2;
    out[((size_t)(x >> 11) + q / 4) * 256 + w] = q < len ? val[k0 + q] : T(0);
  }
  diag[(size_t)c * 64 + t] = i < 0 ? T(1) : val[upper ? r0 : r0 + len];
}

// Levels of a factor (lev: each row's earliest one) with the rows that are
// needed long after it put off: a row whose last reader comes more than
// `reach` levels later moves to `reach` levels before that reader, but stays
// before its first one.  The number of levels does not change.
static void ring_levels(int n, const int* row, const int* col, bool upper, int reach, std::vector<int>& lev) {
  std::vector<int> first(n, INT32_MAX), last(n, -1);
  for (int t = 0; t < n; t++) {
    const int i = upper ? t : n - 1 - t;  // a row's readers come before it
    if (last[i] - lev[i] > reach) lev[i] = std::max(lev[i], std::min(first[i] - 1, last[i] - reach));
    for (int k = row[i]; k < row[i + 1]; k++) {
      const int j = col[k];
      if (j == i) continue;
      first[j] = std::min(first[j], lev[i]);
      last[j] = std::max(last[j], lev[i]);
    }
  }
}

static RingHost ring_plan(int n, const int* row, const int* col, bool upper, int maxoff, int nlev,
                          const std::vector<int>& perm, std::vector<int> lptr) {
  RingHost h;
  // whole rounds of two chunks a wave, the last ones empty
  const auto padded = [](long chunks) { return (chunks + 2 * kRingWaves - 1) / (2 * kRingWaves) * (2 * kRingWaves); };
  if (n < 1 || maxoff > 16 || nlev >= (1 << kRingLevelBits) - 1 || padded(((long)n + 63) / 64) > kRingDescs) return h;
  const auto len = [&](int i) { return row[i + 1] - row[i] - 1; };
  std::vector<int> lev(n), pos(n), order(n), at;
  for (int l = 0; l < nlev; l++)
    for (int t = lptr[l]; t < lptr[l + 1]; t++) lev[perm[t]] = l;
  int span = 0, widest = 0;
  for (int pass = 0;; pass++) {
    // rows by level and, in a level, by falling length, so that a chunk's
    // rows need the same number of slots
    at.assign((size_t)nlev * 17 + 1, 0);
    for (int i = 0; i < n; i++) {
      if (len(i) < 0) return h;
      at[(size_t)lev[i] * 17 + 16 - len(i) + 1]++;
    }
    for (size_t q = 1; q < at.size(); q++) at[q] += at[q - 1];
    for (int l = 0; l <= nlev; l++) lptr[l] = at[(size_t)l * 17];
    for (int i = 0; i < n; i++) pos[i] = at[(size_t)lev[i] * 17 + 16 - len(i)]++;
    for (int i = 0; i < n; i++) order[pos[i]] = i;
    span = widest = 0;
    for (int l = 0; l < nlev; l++) widest = std::max(widest, lptr[l + 1] - lptr[l]);
    for (int i = 0; i < n; i++)
      for (int k = row[i]; k < row[i + 1]; k++) {
        const int j = col[k];
        if (j == i) continue;
        if (lev[j] >= lev[i]) return h;  // not a triangular factor: no such form
        // a solved row must still be in the ring while its reader's level writes
        span = std::max(span, lptr[lev[i] + 1] - pos[j]);
      }
    // a few rows with few entries of their own often lie far before their
    // readers (ragged 47 x 45 x 46 mesh: 31 operands of 672 thousand more
    // than 16384 rows back, 31482 at most; 8139 after)
    if (span <= ring_rows<double>() || pass == 1) break;
    ring_levels(n, row, col, upper, std::max(1, ring_rows<double>() / (2 * widest)), lev);
  }
  if (span > ring_rows<float>()) return h;
  long chunks = 0;
  for (int l = 0; l < nlev; l++) chunks += (lptr[l + 1] - lptr[l] + 63) / 64;
  const int all = (int)padded(chunks);
  if (all > kRingDescs) return h;
  h.form.assign(66 * (size_t)all + 2 * (size_t)((n + 1) / 2 * 2), -1);
  uint2* desc = reinterpret_cast<uint2*>(h.form.data());
  int* rp = h.form.data() + 2 * (size_t)all;
  int* slot = rp + 64 * (size_t)all;
  std::copy(pos.begin(), pos.end(), slot + (n + 1) / 2 * 2);
  int c = 0, groups = 0, gmax = 1;
  for (int l = 0; l < nlev; l++)
    for (int p0 = lptr[l]; p0 < lptr[l + 1]; p0 += 64, c++) {
      const int rows = std::min(64, lptr[l + 1] - p0);
      const int ng = (len(order[p0]) + 3) / 4;
      desc[c].x = (unsigned)groups << 11 | (unsigned)rows << 4 | (unsigned)ng;
      desc[c].y = (unsigned)l << 15 | (unsigned)(p0 & 32767);
      for (int t = 0; t < rows; t++) {
        rp[(size_t)c * 64 + t] = order[p0 + t];
        slot[order[p0 + t]] = c * 64 + t;
      }
      groups += ng;
      gmax = std::max(gmax, ng);
    }
  for (; c < all; c++) {
    desc[c].x = (unsigned)groups << 11;
    desc[c].y = (unsigned)(nlev - 1) << 15;
  }
  h.chunks = all;
  h.groups = gmax;
  h.all_groups = groups;
  h.span = span;
  return h;
}

// One workgroup against the whole chip: 0.19 us a level plus the entries at
// 100 GB/s and 8 ns a chunk, against 0.5 us a level in boxes of a 2-D grid,
// 0.65 us in boxes of a 3-D grid and 1.6 us in runs of consecutive rows.
// Measured on either side for L and U (FP64): 32^3 85 against 118 us (here),
// 48^3 227 against 182 us (there), 400 x 300 397 against 704 us (here).
static double ring_us(int nlev, size_t slots, int chunks, size_t elem_size) {
  return 0.19 * nlev + 1e-5 * ((double)slots * (elem_size + 2.0) + 192.0 * chunks * elem_size) + 0.008 * chunks;
}
static double chip_us(const TriPlan& P) {
  return P.nlev * (P.tile_dims[0] == 0 ? 1.6 : P.tile_dims[2] > 1 ? 0.65 : 0.5);
}
static bool ring_pays(const TriPlan& P, size_t elem_size) {
  return ring_us(P.nlev, P.rslots, P.rchunks, elem_size) < 0.9 * chip_us(P);
}

// Making a handle of a 91000-row mesh took 42.7 ms without level orders, 47.5
// with their host parts in line, and takes 40.8 with them beside the other
// forms (and the transposes' level sets copied).  A thread costs about what
// planning 8000 rows takes; without one the host part runs in end_ring.
void TriPlan::levels(int n_, const int* row_, const int* col_, bool upper_, bool ring) {
  n = n_;
  nnz = row_[n_];
  upper = upper_;
  h_perm.resize(n);
  std::vector<int> lptr_h(n + 1);
  nlev = lace_level_sets(n, row_, col_, upper ? 1 : 0, h_perm.data(), lptr_h.data());
  h_lptr.assign(lptr_h.begin(), lptr_h.begin() + nlev + 1);
  maxoff = 0;
  for (int i = 0; i < n; i++) maxoff = std::max(maxoff, row_[i + 1] - row_[i] - 1);
  rval_src = nullptr;
  rchunks = 0;
  // not where it could not pay even with full chunks, against the slowest
  // blocks of the persistent kernel
  if (!ring || n == 0 ||
      (get_option("trsv_exact_ring", 1) != 2 && ring_us(nlev, std::max(0, nnz - n), ceil_div(n, 64), 4) >= 1.44 * nlev))
    return;
  auto task = [n = n, row_, col_, upper = upper, maxoff = maxoff, nlev = nlev, perm = h_perm, lptr = h_lptr] {
    return ring_plan(n, row_, col_, upper, maxoff, nlev, perm, lptr);
  };
  if (n >= 8000) {
    try {
      ring_host = std::async(std::launch::async, task);
      return;
    } catch (const std::system_error&) {  // no thread to be had
    }
  }
  ring_host = std::async(std::launch::deferred, std::move(task));
}

// The form is kept where it is expected to pay (option "trsv_exact_ring" 2:
// wherever there is one).  Without memory for it a plan has none, and its exact
// solves run the persistent kernel, which needs no more than the factor.
int TriPlan::end_ring(size_t elem_size, RingHost* host) {
  if (!ring_host.valid()) return DEV_SUCCESS;
  RingHost& h = *host;
  try {
    h = ring_host.get();
  } catch (const std::bad_alloc&) {
    return DEV_SUCCESS;
  }
  if (h.chunks == 0) return DEV_SUCCESS;
  // one more group: where a chunk without operands points
  rslots = ((size_t)h.all_groups + 1) * 256;
  rgroups = h.groups;
  rspan = h.span;
  rchunks = h.chunks;
  const bool fits = rspan <= kRingBytes / (int)elem_size;
  if (!fits || (get_option("trsv_exact_ring", 1) != 2 && !ring_pays(*this, elem_size)) ||
      rform.alloc(rform_bytes(elem_size)) != DEV_SUCCESS) {
    (void)hipGetLastError();
    rchunks = 0;
    return DEV_SUCCESS;
  }
  LACE_HIP(hipMemcpyAsync(rform.p, h.form.data(), sizeof(int) * h.form.size(), hipMemcpyHostToDevice, stream()));
  ring_index_kernel<<<rchunks + 1, 64, 0, stream()>>>(rchunks, reinterpret_cast<const uint2*>(rdesc()), rperm(),
                                                      row.as<int>(), col.as<int>(), rplace(), upper, h.all_groups,
                                                      ridx());
  LACE_HIP(hipGetLastError());
  return DEV_SUCCESS;
}

// A vector into chunk order (map: the row at each slot) or out of it (the
// slot of each row), so that the one workgroup moves whole words; with map2
// from one factor's chunk order into another's.
template <typename T>
__global__ __launch_bounds__(256) void ring_move_kernel(int m, const int* __restrict__ map,
                                                        const int* __restrict__ map2,
                                                        const T* __restrict__ in, T* __restrict__ out) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= m) return;
  const int i = map[k];
  out[k] = i < 0 ? T(0) : in[map2 ? map2[i] : i];
}

// The form of a plan with the same pattern and triangle (symmetric patterns:
// U^T has L's, L^T has U's).
int TriPlan::copy_ring(const TriPlan& o, size_t elem_size) {
  ring_copied = true;
  rval_src = nullptr;
  rchunks = o.rchunks;
  if (rchunks == 0) return DEV_SUCCESS;
  rslots = o.rslots;
  rgroups = o.rgroups;
  rspan = o.rspan;
  if (rform.alloc(rform_bytes(elem_size)) != DEV_SUCCESS) {
    (void)hipGetLastError();
    rchunks = 0;
    return DEV_SUCCESS;
  }
  LACE_HIP(hipMemcpyAsync(rform.p, o.rform.p, sizeof(int) * rform_words() + 2 * rslots, hipMemcpyDeviceToDevice,
                          stream()));
  return DEV_SUCCESS;
}

namespace {

// A chunk's data in flight: lane t holds row t's entries.
template <typename T, int NG>
struct RingStage {
  T v[NG][4];
  ushort4 id[NG];
  T r, d;
  int row;                   // of a direct solve
  unsigned cell[NG][4];      // operands' byte offsets in LDS
  bool unit;                 // wave-uniform, as are:
  int ng, rows, level, pos;
};

// Four values of lane `lane` of group `at` (see ring_gather_kernel).
__device__ __forceinline__ void load_group(const float* __restrict__ val, unsigned group, unsigned lane, float (&v)[4]) {
  vload<float, 4>(val + group * 256u + lane * 4, v);
}
__device__ __forceinline__ void load_group(const double* __restrict__ val, unsigned group, unsigned lane,
                                           double (&v)[4]) {
  double a[2], b[2];
  vload<double, 2>(val + group * 256u + lane * 2, a);
  vload<double, 2>(val + group * 256u + 128 + lane * 2, b);
  v[0] = a[0], v[1] = a[1], v[2] = b[0], v[3] = b[1];
}

}  // namespace

// Wave w takes chunks w, w + W, ...; each chunk's entries are loaded two of
// the wave's chunks ahead, so memory latency is off the chain of levels.  A
// chunk runs once every wave has passed the barrier of the level before.  A
// chunk's prefetch is issued after the barrier that ends its predecessor's
// level, so that the other waves do not wait for it, and always with the
// same number of loads (groups a chunk does not have read one word), so that
// waiting for one chunk's loads leaves the next one's in flight; what does
// not depend on the solution (the operands' places in LDS) is worked out
// before the last barrier a chunk waits at.  Padding entries are a zero
// times a cell that holds zero: a sum that starts from +0 is unchanged by
// adding +0.  Each row's sum runs in CSR order and then divides, as in
// substitution, and dividing by one is exact: results are bit-identical to
// the other exact solves.  Every wave passes exactly nlev barriers.  DIRECT:
// rhs and out are in the caller's row order (perm: the row at each slot),
// else in chunk order.
template <typename T, int NG, int W, bool DIRECT>
__global__ __launch_bounds__(W * 64) void tri_ring_kernel(int nlev, int nchunks,
                                                          const uint2* __restrict__ desc,
                                                          const T* __restrict__ val,
                                                          const ushort4* __restrict__ idx,
                                                          const T* __restrict__ rhs,
                                                          const T* __restrict__ diag,
                                                          const int* __restrict__ perm, T* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr unsigned MASK = ring_rows<T>() - 1;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  uint2* sd = reinterpret_cast<uint2*>(smem + kRingBytes + 16);
  for (int i = threadIdx.x; i < nchunks; i += W * 64) sd[i] = desc[i];
  if (threadIdx.x == 0) *reinterpret_cast<T*>(smem + kRingBytes) = T(0);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned lane = threadIdx.x & 63;
  using Stage = RingStage<T, NG>;
  // the rows of the chunk to be loaded next into each stage
  int nextA = DIRECT ? perm[wave * 64 + lane] : 0, nextB = DIRECT ? perm[(wave + W) * 64 + lane] : 0;
  const auto load = [&](Stage& s, int& next, uint2 w, int c) {
    const unsigned x = __builtin_amdgcn_readfirstlane(w.x), y = __builtin_amdgcn_readfirstlane(w.y);
    const unsigned base = x >> 11;
    s.ng = (int)(x & 15u);
    s.rows = (int)((x >> 4) & 127u);
    s.level = (int)(y >> 15);
    s.pos = (int)(y & 32767u);
#pragma unroll
    for (int g = 0; g < NG; g++) {
      const unsigned group = g < s.ng ? base + g : base, at = g < s.ng ? lane : 0u;
      load_group(val, group, at, s.v[g]);
      s.id[g] = idx[group * 64 + at];
    }
    const unsigned k = (unsigned)c * 64 + lane;
    s.d = diag[k];
    if constexpr (DIRECT) {
      s.row = next;
      s.r = rhs[next < 0 ? 0 : next];
      const int cn = c + 2 * W < nchunks ? c + 2 * W : c;
      next = perm[(unsigned)cn * 64 + lane];
    } else {
      s.r = rhs[k];
    }
  };
  int lev = 0;
  const auto reach = [&](int l) {
    for (; lev < l; lev++) lds_barrier();
  };
  const auto ready = [&](Stage& s) {
    reach(s.level - 1);
#pragma unroll
    for (int g = 0; g < NG; g++) {
      const unsigned e[4] = {s.id[g].x, s.id[g].y, s.id[g].z, s.id[g].w};
#pragma unroll
      for (int q = 0; q < 4; q++)
        s.cell[g][q] = e[q] == 0xFFFFu ? (unsigned)kRingBytes : (e[q] & MASK) * (unsigned)sizeof(T);
    }
    s.unit = __all(s.d == T(1));
    reach(s.level);
  };
  const auto solve = [&](const Stage& s, int c) {
    T sum = T(0);
#pragma unroll
    for (int g = 0; g < NG; g++)
      if (g < s.ng) {
        T x[4];
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = *reinterpret_cast<const T*>(smem + s.cell[g][q]);
#pragma unroll
        for (int q = 0; q < 4; q++) sum = sum + s.v[g][q] * x[q];
      }
    T y = s.r - sum;
    if (!s.unit) y = y / s.d;
    if ((int)lane < s.rows) {
      *reinterpret_cast<T*>(smem + ((unsigned)(s.pos + lane) & MASK) * sizeof(T)) = y;
      if constexpr (DIRECT) out[s.row] = y;
      else out[(unsigned)c * 64 + lane] = y;
    }
  };
  Stage A, B;
  load(A, nextA, sd[wave], wave);
  load(B, nextB, sd[wave + W], wave + W);
  for (int c = wave; c < nchunks; c += 2 * W) {
    const int ca = c + 2 * W < nchunks ? c + 2 * W : c;
    const uint2 da = sd[ca];
    ready(A);
    solve(A, c);
    if (lev < B.level) reach(lev + 1);
    load(A, nextA, da, ca);
    const uint2 db = sd[ca + W];
    ready(B);
    solve(B, c + W);
    if (lev < A.level) reach(lev + 1);
    load(B, nextB, db, ca + W);
  }
  reach(nlev);
}

template <typename T>
bool ring_ready(const TriPlan& P) {
  const int ring = get_option("trsv_exact_ring", 1);
  if (ring == 0 || P.rchunks == 0 || P.rspan > ring_rows<T>()) return false;
  // options that shape the persistent kernel ask for that kernel
  return ring == 2 || (ring_pays(P, sizeof(T)) && get_option("trsv_exact_tiles", 1) != 0 &&
                       get_option("trsv_exact_rows", 512) == 512);
}

// The kernels' LDS is past what a launch may ask for by itself: allowed for
// each of them, on the present device, when the library is initialised on it.
template <typename T, int NG, int W, bool DIRECT>
static int ring_allow() {
  LACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(tri_ring_kernel<T, NG, W, DIRECT>),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               kRingBytes + 16 + (int)sizeof(uint2) * kRingDescs));
  return DEV_SUCCESS;
}
template <typename T, int W, bool DIRECT>
static int ring_allow_groups() {
  LACE_TRY((ring_allow<T, 1, W, DIRECT>()));
  LACE_TRY((ring_allow<T, 2, W, DIRECT>()));
  return ring_allow<T, 4, W, DIRECT>();
}
template <typename T>
static int ring_allow_all() {
  LACE_TRY((ring_allow_groups<T, 8, false>()));
  LACE_TRY((ring_allow_groups<T, 8, true>()));
  LACE_TRY((ring_allow_groups<T, 16, false>()));
  return ring_allow_groups<T, 16, true>();
}
int ring_setup() {
  LACE_TRY(ring_allow_all<float>());
  return ring_allow_all<double>();
}

template <typename T, int NG, int W, bool DIRECT>
static int ring_launch(const TriPlan& P, const T* rhs, T* out) {
  const size_t lds = kRingBytes + 16 + sizeof(uint2) * P.rchunks;
  tri_ring_kernel<T, NG, W, DIRECT><<<1, W * 64, lds, stream()>>>(
      P.nlev, P.rchunks, reinterpret_cast<const uint2*>(P.rdesc()), P.rval<T>(), reinterpret_cast<const ushort4*>(P.ridx()), rhs, P.rdiag<T>(),
      P.rperm(), out);
  LACE_HIP(hipGetLastError());
  return DEV_SUCCESS;
}

template <typename T, bool DIRECT>
static int ring_solve(const TriPlan& P, const T* rhs, T* out) {
  const double es = sizeof(T), rows = 64.0 * P.rchunks;
  TimedRegion tr(P.upper ? "trsv_exact_upper" : "trsv_exact_lower", 0.0,
                 (double)P.rslots * (es + 2.0) + rows * 3.0 * es);
  // 16 waves where levels hold several chunks (32^3 FP64 L and U 85 against
  // 107 us), else 8, whose barrier is shorter (64 x 64: 66 against 69 us)
  if (2 * P.rchunks > 5 * P.nlev) {
    if (P.rgroups <= 1) return ring_launch<T, 1, 16, DIRECT>(P, rhs, out);
    if (P.rgroups <= 2) return ring_launch<T, 2, 16, DIRECT>(P, rhs, out);
    return ring_launch<T, 4, 16, DIRECT>(P, rhs, out);
  }
  if (P.rgroups <= 1) return ring_launch<T, 1, 8, DIRECT>(P, rhs, out);
  if (P.rgroups <= 2) return ring_launch<T, 2, 8, DIRECT>(P, rhs, out);
  return ring_launch<T, 4, 8, DIRECT>(P, rhs, out);
}

// Whether the workgroup reads the right-hand side and writes the solution in
// row order itself (38 ns a chunk to scatter 64 rows against 8 ns to store
// them in order) instead of leaving that to launches of their own (3 us
// each).  L and U, FP64: 64 x 64 (128 chunks) 61 against 66 us, 24 x 25 x 23
// mesh (290) 152 against 155 us, 200 x 200 (800) 254 against 209 us.
static bool ring_direct(const TriPlan& P) { return P.rchunks <= 320; }

// The values of val in chunk order.
template <typename T>
static int ring_values(const TriPlan& P, const T* val) {
  if (P.rval_src == (const void*)val) return DEV_SUCCESS;
  ring_gather_kernel<T><<<P.rchunks + 1, 64, 0, stream()>>>(P.rchunks, reinterpret_cast<const uint2*>(P.rdesc()), P.rperm(),
                                                            P.row.as<int>(), P.upper, P.rslots, val,
                                                            P.rval<T>(), P.rdiag<T>());
  LACE_HIP(hipGetLastError());
  P.rval_src = val;
  return DEV_SUCCESS;
}

template <typename T>
static int ring_move(int m, const int* map, const int* map2, const T* in, T* out) {
  ring_move_kernel<T><<<ceil_div(m, 256), 256, 0, stream()>>>(m, map, map2, in, out);
  LACE_HIP(hipGetLastError());
  return DEV_SUCCESS;
}

template <typename T>
int tri_solve_ring(const TriPlan& P, const T* val, const T* r, T* y) {
  LACE_REQUIRE((const void*)r != (const void*)y, DEV_ERR_ILLEGAL_VALUE, "exact solve needs distinct r and y");
  LACE_TRY(ring_values<T>(P, val));
  if (ring_direct(P)) return ring_solve<T, true>(P, r, y);
  LACE_TRY(ring_move<T>(P.rchunks * 64, P.rperm(), nullptr, r, P.rrhs<T>()));
  LACE_TRY((ring_solve<T, false>(P, P.rrhs<T>(), P.rsol<T>())));
  return ring_move<T>(P.n, P.rslot(), nullptr, P.rsol<T>(), y);
}

template <typename T>
int tri_solve_ring2(const TriPlan& P, const T* val, const TriPlan& Q, const T* val2, const T* r, T* y) {
  LACE_TRY(ring_values<T>(P, val));
  LACE_TRY(ring_values<T>(Q, val2));
  LACE_TRY(ring_move<T>(P.rchunks * 64, P.rperm(), nullptr, r, P.rrhs<T>()));
  LACE_TRY((ring_solve<T, false>(P, P.rrhs<T>(), P.rsol<T>())));
  LACE_TRY(ring_move<T>(Q.rchunks * 64, Q.rperm(), P.rslot(), P.rsol<T>(), Q.rrhs<T>()));
  LACE_TRY((ring_solve<T, false>(Q, Q.rrhs<T>(), Q.rsol<T>())));
  return ring_move<T>(Q.n, Q.rslot(), nullptr, Q.rsol<T>(), y);
}

template <typename T>
bool ring_pair(const TriPlan& P, const TriPlan& Q) {
  return ring_ready<T>(P) && ring_ready<T>(Q) && !ring_direct(P) && !ring_direct(Q);
}

template bool ring_pair<float>(const TriPlan&, const TriPlan&);
template bool ring_pair<double>(const TriPlan&, const TriPlan&);
template bool ring_ready<float>(const TriPlan&);
template bool ring_ready<double>(const TriPlan&);
template int tri_solve_ring<float>(const TriPlan&, const float*, const float*, float*);
template int tri_solve_ring<double>(const TriPlan&, const double*, const double*, double*);
template int tri_solve_ring2<float>(const TriPlan&, const float*, const TriPlan&, const float*, const float*, float*);
template int tri_solve_ring2<double>(const TriPlan&, const double*, const TriPlan&, const double*, const double*,
                                     double*);

}  // namespace lace
