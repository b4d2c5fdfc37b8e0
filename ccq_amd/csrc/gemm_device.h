// Device code of the GEMM kernels of the coupled-cluster amplitude engine
// (gfx950): operand / epilogue helpers shared with the other kernels, the
// LDS-tiled MFMA tile kernel (single, chained and grouped launches) and the
// register-direct kernel.  Templates: their instantiations live in the units
// that launch them (gemm_f64.hip, gemm_f32.hip, gemm_f32io.hip: one
// arithmetic / storage pair each, compiled in parallel).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include "kernels.h"

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

namespace ccqk {


// ---------------------------------------------------------------------------
// GEMM building blocks

// Offset of summed index k in an operand: an int32 table, or k * aff when the
// table is affine (aff >= 0), which saves the dependent table load.
__device__ __forceinline__ int64_t koff(const int* __restrict__ tab, int64_t aff, int64_t k) {
  return aff >= 0 ? k * aff : (int64_t)tab[k];
}

// Storage type IO of the tensors a kernel reads and writes: double, or float
// in the FP32-storage sweeps (the argument pointers then hold float arrays;
// arithmetic on loaded values is FP64 in the epilogues)
template <typename IO>
__device__ __forceinline__ double ldg(const double* p, int64_t i) {
  return (double)reinterpret_cast<const IO*>(p)[i];
}
template <typename IO>
__device__ __forceinline__ void stg(double* p, int64_t i, double v) {
  reinterpret_cast<IO*>(p)[i] = (IO)v;
}

template <typename IO>
__device__ __forceinline__ void put_c(double* base, int64_t off, double v, int accumulate) {
  if (accumulate) stg<IO>(base, off, ldg<IO>(base, off) + v); else stg<IO>(base, off, v);
}

// IOC: the stored type of C (GemmArgs::c64: double beside float operands)
template <typename IO, typename IOC = IO>
__device__ __forceinline__ void store_c(const GemmArgs& g, int64_t m, int64_t n, double s, double alpha) {
  const int64_t r = g.rowC[m], c = g.colC[n];
  double v = alpha * s;
  if (g.D) v += g.dcoef * ldg<IO>(g.D, (int64_t)g.rowD[m] + g.colD[n]);
  put_c<IOC>(g.C, r + c, v, g.accumulate);
  if (g.rowC2) {
    const int64_t r2 = g.rowC2[m];
    put_c<IOC>(g.C, r2 + c, -v, g.accumulate);
    if (g.colC2) put_c<IOC>(g.C, r2 + g.colC2[n], v, g.accumulate);
  }
  if (g.colC2) put_c<IOC>(g.C, r + g.colC2[n], -v, g.accumulate);
}

// sum_{i < cnt} q[i * stride] with four interleaved partial sums (fixed order)
__device__ __forceinline__ double sum_strided(const double* __restrict__ q, int64_t stride, int cnt) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  int i = 0;
  for (; i + 4 <= cnt; i += 4) {
    a0 += q[0];
    a1 += q[stride];
    a2 += q[2 * stride];
    a3 += q[3 * stride];
    q += 4 * stride;
  }
  for (; i < cnt; ++i) {
    a0 += q[0];
    q += stride;
  }
  return (a0 + a1) + (a2 + a3);
}

// Tile order.  Workgroups are dispatched round-robin over the 8 XCDs of
// MI355X, each with its own L2, in linear id order (x fastest, then y, z).
// The linear id is remapped so that every XCD receives a contiguous range of
// logical tiles, and logical tiles are ordered in groups of `group` tile rows
// (all of one split-K slice first), so the A row panels and B column panels a
// workgroup needs are mostly shared with the other workgroups on its XCD.
__device__ __forceinline__ int xcd_logical(int lin, int total) {
  const int q = total >> 3, r = total & 7;
  const int xcd = lin & 7, slot = lin >> 3;
  return xcd < r ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
}

// tile pid of tm x tn in groups of `group` tile rows
__device__ __forceinline__ void tile_in_group(int pid, int tm, int tn, int group, int& tx, int& ty) {
  const int gsize = group * tn;
  const int first = (pid / gsize) * group;
  const int gm = tm - first < group ? tm - first : group;
  const int in = pid - (pid / gsize) * gsize;
  tx = first + in % gm;
  ty = in / gm;
}

__device__ __forceinline__ void tile_coords(int group, int& tx, int& ty, int& tz) {
  const int tm = gridDim.x, tn = gridDim.y;
  const int total = tm * tn * (int)gridDim.z;
  const int lin = blockIdx.x + tm * (blockIdx.y + tn * blockIdx.z);
  const int logical = xcd_logical(lin, total);
  const int per_z = tm * tn;
  tz = logical / per_z;
  tile_in_group(logical - tz * per_z, tm, tn, group, tx, ty);
}

// Grouped launch (1-D grid over the tiles of every member): the member owning
// the workgroup's logical tile, and the tile inside that member in the order
// above.  Members occupy consecutive logical ranges, so an XCD's range covers
// the tiles of one or two members.
template <int BM, int BN>
__device__ __forceinline__ int group_tile(const GemmGroup& gg, int& tx, int& ty) {
  const int logical = xcd_logical((int)blockIdx.x, gg.start[gg.n]);
  int mem = 0;
#pragma unroll
  for (int i = 1; i < kMaxGroup; ++i)
    if (i < gg.n && logical >= gg.start[i]) mem = i;
  const GemmArgs& g = gg.g[mem];
  const int tm = (int)((g.M + BM - 1) / BM), tn = (int)((g.N + BN - 1) / BN);
  tile_in_group(logical - gg.start[mem], tm, tn, g.group, tx, ty);
  return mem;
}

// Split-K: workgroup z of a tile stores its partial product of K range
// [z*kchunk, (z+1)*kchunk) at ws[z][m][n] (M x N, row-major); gemm_splitk_reduce
// sums the nsplit partials of every element in a fixed order and writes C.
__device__ __forceinline__ void store_partial(const GemmArgs& g, int z, int64_t m, int64_t n, double v) {
  g.ws[((int64_t)z * g.M + m) * g.N + n] = v;
}

// LDS tile of an operand: R rows of BK values of type T, pitch BK + P, whatever
// the operand's layout in memory.  P keeps rows on pairs of values (the
// loader writes and the fragments read two consecutive k at a time) and
// spreads the 16 rows of a fragment read over all 64 banks: FP64 pitch
// 18 / 34 pairs of words 4 apart mod 64, FP32 pitch 20 / 36.
template <typename T, int R, int BK>
struct LdsTile {
  static constexpr int pitch = BK + (sizeof(T) == 8 ? 2 : 4);
  static constexpr int size = R * pitch;
};

// How an operand's summed indices lie in memory.  Vec: contiguous, two k per
// load.  Aff: a constant stride.  The others read a table: Pair, a k-contiguous
// operand in which k and k + 1 are neighbours for every even k (runs of even
// length), two k per load; TabK, any k-contiguous operand; Tab, any.  All of
// these address it with 32-bit byte offsets; Wide is Tab with 64-bit addresses,
// for operands that reach 4 GiB (GemmArgs::wide).
// 900 x 900 x 900, hot: Vec 42 us, Tab 54, TabK 52.6, Pair 46.
enum class KMode { Vec, Aff, Pair, TabK, Tab, Wide };

// Offsets of the summed indices of a table operand's K range, in LDS (bytes;
// Wide: elements), for at most kKCache indices; longer ranges are walked in runs
// of kKCache.
constexpr int kKCache = 1024;

// One operand's slabs (R rows x BK k-values), global memory -> registers ->
// LDS, 256 threads.  A thread owns L values: Vec and Pair: L / 2 rows, two
// consecutive k; else one k of L rows (kfast: neighbouring threads own neighbouring k) or L
// k of one row (neighbouring threads own neighbouring rows).  FP64 MFMAs share
// the vector ALUs with everything else (a pure loop of them runs at 77 TF/s,
// and every other vector instruction takes its time from it), so the loop over
// whole slabs has none of its own: Vec and Aff addresses are a scalar base that
// moves by a slab plus a 32-bit offset that does not, rows past the end are
// clamped to the last one (their products are never stored), and only the last
// slab is masked.
// The registers hold the stored type IO: a conversion right after the load
// would wait for it there.
template <typename T, typename IO, int R, int BK, KMode MODE>
struct Feed {
  static constexpr bool vec = MODE == KMode::Vec || MODE == KMode::Pair;
  static constexpr bool tab = MODE != KMode::Vec && MODE != KMode::Aff;
  // unit of off[] and of the offset table
  static constexpr uint32_t unit = MODE == KMode::Wide ? 1 : (uint32_t)sizeof(IO);
  static constexpr int L = R * BK / 256;
  static constexpr int NJ = vec ? L / 2 : L;
  static constexpr int pitch = LdsTile<T, R, BK>::pitch;
  typedef IO io2 __attribute__((ext_vector_type(2), aligned(sizeof(IO))));
  typedef T t2 __attribute__((ext_vector_type(2)));
  struct Slab {
    IO v[L];
  };
  const char* base;   // the operand, at the first summed index of the range (Vec, Aff)
  int64_t aff;
  uint32_t off[NJ];   // offset of each row (Vec, Aff: plus that of the value's k in the slab)
  int k0, ks;         // k of item j in a slab: k0 + j ks
  int lds0, ldss;     // its place in the LDS tile: lds0 + j ldss

  __device__ __forceinline__ void init(const double* X, const int* __restrict__ rowtab, int64_t r0, int64_t rows,
                                       int kfast, int64_t kaff, int64_t kr, int tid) {
    int r, rs;
    if constexpr (vec) {
      r = tid / (BK / 2), rs = 512 / BK;
      k0 = 2 * (tid % (BK / 2)), ks = 0;
    } else if constexpr (MODE == KMode::TabK) {
      r = tid / BK, rs = 256 / BK;
      k0 = tid % BK, ks = 0;
    } else {
      r = kfast ? tid / BK : tid % R, rs = kfast ? 256 / BK : 0;
      k0 = kfast ? tid % BK : tid / R, ks = kfast ? 0 : 256 / R;
    }
    lds0 = r * pitch + k0;
    ldss = rs * pitch + ks;
    aff = tab ? 0 : kaff;
    base = reinterpret_cast<const char*>(X) + kr * aff * (int64_t)sizeof(IO);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int64_t gr = r0 + r + j * rs;
      off[j] = (uint32_t)rowtab[gr < rows ? gr : rows - 1] * unit;
      if (!tab) off[j] += (uint32_t)((k0 + j * ks) * aff) * unit;
    }
  }
  __device__ __forceinline__ IO at(uint32_t row, uint32_t k) const {
    if constexpr (MODE == KMode::Wide) return reinterpret_cast<const IO*>(base)[(uint64_t)row + k];
    else return *reinterpret_cast<const IO*>(base + (row + k));
  }
  // whole slab at index i of the range; ko: the range's offset table
  __device__ __forceinline__ void fetch(Slab& s, int i, const uint32_t* ko) const {
    const char* p = base + i * aff * (int64_t)sizeof(IO);
    const uint32_t o = vec || MODE == KMode::TabK ? (tab ? ko[i + k0] : 0u) : 0u;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if constexpr (vec) {
        const io2 x = *reinterpret_cast<const io2*>(p + (off[j] + o));
        s.v[2 * j] = x.x;
        s.v[2 * j + 1] = x.y;
      } else if constexpr (MODE == KMode::Aff) {
        s.v[j] = *reinterpret_cast<const IO*>(p + off[j]);
      } else if constexpr (MODE == KMode::TabK) {
        s.v[j] = at(off[j], o);
      } else {
        s.v[j] = at(off[j], ko[i + k0 + j * ks]);
      }
    }
  }
  // the slab at index i with k past the end (klen) clamped to the last one
  __device__ __forceinline__ void fetch_tail(Slab& s, int i, int klen, const uint32_t* ko) const {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int q = vec ? j / 2 : j;
      const int kq = k0 + q * ks;
      const int k = i + (vec ? k0 + (j & 1) : kq);
      const int kc = k < klen ? k : klen - 1;
      if constexpr (tab)
        s.v[j] = at(off[q], ko[kc]);
      else
        s.v[j] = *reinterpret_cast<const IO*>(base + off[q] + (int64_t)(kc - kq) * aff * (int64_t)sizeof(IO));
    }
  }
  __device__ __forceinline__ void stash(T* to, const Slab& s) const {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if constexpr (vec) {
        t2 x;
        x.x = (T)s.v[2 * j];
        x.y = (T)s.v[2 * j + 1];
        *reinterpret_cast<t2*>(to + lds0 + j * ldss) = x;
      } else {
        to[lds0 + j * ldss] = (T)s.v[j];
      }
    }
  }
  // left: summed indices from the slab's first k to the end of the range
  __device__ __forceinline__ void stash_tail(T* to, const Slab& s, int left) const {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int q = vec ? j / 2 : j, e = vec ? j & 1 : 0;
      to[lds0 + q * ldss + e] = k0 + q * ks + e < left ? (T)s.v[j] : T(0);
    }
  }
};

// MFMA step and D-fragment row of one 16x16 tile, by arithmetic type.
// v_mfma_f64_16x16x4f64 and v_mfma_f32_16x16x4f32 read the same A / B
// fragments (lane l: row l%16, k = l/16); their D layouts differ (measured on
// gfx950): FP64 lane l, register v holds row (l/16) + 4v, FP32 row 4(l/16) + v;
// column l%16 in both.
template <typename T>
struct Mma;
template <>
struct Mma<double> {
  typedef d4 acc_t;
  __device__ static acc_t step(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Mma<float> {
  typedef f4 acc_t;
  __device__ static acc_t step(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// LDS-tiled GEMM C(M x N) (+)= alpha * A(M x K) B(K x N), for products with
// both output extents large (MFMA bound).  256 threads = 4 waves in a 2 x 2
// grid; each wave owns a (BM/2) x (BN/2) sub-tile of 16x16 MFMA tiles.
// Operands are gathered in their stored type IO (FP64; FP32 in the
// FP32-storage sweeps) through int32 row offset tables (rowA, colB) and their
// summed indices' stride or table (kA, kB), and staged into LDS as T.  T =
// double runs on v_mfma_f64_16x16x4f64; T = float rounds the operands to FP32
// and multiplies on v_mfma_f32_16x16x4f32 (the mixed-precision form): kF32Run
// summed indices at a time accumulate in FP32, the runs in FP64.
// FP64, against one slab of look-ahead with two barriers a slab, predicated
// loads and single-k fragment reads: 1225 x 4375 x 1225 303 -> 244 us (54 TF/s),
// 900^3 58.6 -> 42 us, 8100 x 100 x 8100 448 -> 328 us, 4096 x 4096 x 2048
// 53 -> 65 TF/s; without the loads and LDS writes the same loop runs at 73.
// blockIdx.z owns K range [z*kchunk, (z+1)*kchunk) (split-K, completed by
// gemm_splitk_reduce).  KS = 2 doubles the workgroup: two groups of 4 waves
// take alternate K slabs of the same tile (each with its own LDS slab) and
// combine their accumulators through LDS at the end in a fixed order -- the
// K split of a global split-K without its partial products in HBM and its
// reduction launch.
// Epilogue of one tile: C[rowC[m] + colC[n]] (+)= alpha val (+ dcoef D[..]).
// Each lane loads its row offsets once and, per column, all its old C and
// addend values in one batch before storing: the compiler has to assume a
// store through C may change the offset tables, so an element-by-element
// epilogue serialises a table load, a C load and the store for every
// element.  Outputs with mirrored images (packed pairs) take the
// element-by-element path.
template <typename IO, typename IOC, int TM, int TN, typename MM, typename V>
__device__ __forceinline__ void store_tile(const GemmArgs& g, int64_t m0, int64_t n0, int wm, int wn, int lane,
                                           double alpha, const V (&val)[TM][TN]) {
  if (g.rowC2 || g.colC2) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t gn = n0 + wn + 16 * j + (lane & 15);
      if (gn >= g.N) continue;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t gm = m0 + wm + 16 * i + MM::row(lane, v);
          if (gm < g.M) store_c<IO, IOC>(g, gm, gn, (double)val[i][j][v], alpha);
        }
    }
    return;
  }
  int rc[TM][4], rd[TM][4];   // int32 offsets as in the tables; -1: row out of range
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t gm = m0 + wm + 16 * i + MM::row(lane, v);
      const bool in = gm < g.M;
      rc[i][v] = in ? g.rowC[gm] : -1;
      rd[i][v] = (in && g.D) ? g.rowD[gm] : 0;
    }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t gn = n0 + wn + 16 * j + (lane & 15);
    if (gn >= g.N) continue;
    const int64_t cc = g.colC[gn];
    double out[TM][4];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) out[i][v] = alpha * (double)val[i][j][v];
    if (g.D) {
      const int64_t cd = g.colD[gn];
      double dv[TM][4];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) dv[i][v] = rc[i][v] >= 0 ? ldg<IO>(g.D, (int64_t)rd[i][v] + cd) : 0.0;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) out[i][v] += g.dcoef * dv[i][v];
    }
    if (g.accumulate) {
      double old[TM][4];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) old[i][v] = rc[i][v] >= 0 ? ldg<IOC>(g.C, (int64_t)rc[i][v] + cc) : 0.0;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) out[i][v] = old[i][v] + out[i][v];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (rc[i][v] >= 0) stg<IOC>(g.C, (int64_t)rc[i][v] + cc, out[i][v]);
  }
}

// Waves per SIMD the tile kernels are compiled for: three 64 x 64 workgroups a CU
// measured 8 % faster than two on operands that are not k-contiguous
// (1225 x 4375 x 1225: 287 -> 265 us).
template <int KS>
constexpr int kTileWaves = KS > 1 ? 1 : 3;

// LDS bytes of one tile-kernel variant (two slabs per group)
template <typename T, int BM, int BN, int BK, int KS>
struct TabLds {
  static constexpr int slab = LdsTile<T, BM, BK>::size + LdsTile<T, BN, BK>::size;
  static constexpr int tile = 2 * KS * slab * (int)sizeof(T);
  static constexpr int red = (KS - 1) * 256 * (BM / 32) * (BN / 32) * 4 * (int)sizeof(double);
  static constexpr int kts = (tile > red ? tile : red);   // offset of the K offsets
  static constexpr int bytes = kts + 2 * kKCache * (int)sizeof(int);
};

// Summed indices that FP32 products accumulate before they are added to the FP64
// sums.  The rounding of an FP32 accumulator grows with its length, so a bound of
// the kernel's own keeps it independent of tiles and K splits, which levels
// choose longer than a launch per product would.  The FP64 sums take 32 registers
// in a 64 x 64 tile, and some spill in the table modes (FP32-storage sweeps of CCSD
// 61 orbitals 362 -> 375 us, CCSDT 31 1131 -> 1160); two workgroups a CU without
// spills are slower (428, 1282), sums of runs in FP32 too (394, 1198), and runs
// of 128 no faster.
constexpr int kF32Run = 64;

// The K-slab loop of the tile kernel: acc += A(m0.., kbeg..kend) B(kbeg..kend, n0..)
// (the caller zeroes acc; group grp of KS takes slabs grp, grp + KS, ...).
// Slab s is multiplied out of one LDS buffer while slab s + 1 is written to
// the other and slabs s + 2, s + 3 are in flight to registers: one barrier a
// slab, and a load has two slabs' time to arrive.  A fragment read takes two
// consecutive k (the four 16-lane groups of an MFMA then hold k, k + 2, k + 4,
// k + 6: the same products, summed in another order).
template <typename T, typename IO, int BM, int BN, int BK, int KS, KMode MA, KMode MB>
__device__ __forceinline__ void tile_run(const GemmArgs& g, int64_t m0, int64_t n0, int64_t kbeg, int64_t kend,
                                         unsigned char* smem, d4 (&acc)[BM / 32][BN / 32]) {
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int TM = WM / 16, TN = WN / 16;
  using FA = Feed<T, IO, BM, BK, MA>;
  using FB = Feed<T, IO, BN, BK, MB>;
  using MM = Mma<T>;
  typedef T t2 __attribute__((ext_vector_type(2)));
  constexpr int slab = TabLds<T, BM, BN, BK, KS>::slab;
  constexpr bool tab = FA::tab || FB::tab;
  const int grp = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  T* lds = reinterpret_cast<T*>(smem) + grp * 2 * slab;
  uint32_t* kts = reinterpret_cast<uint32_t*>(smem + TabLds<T, BM, BN, BK, KS>::kts);
  const int tid = threadIdx.x & 255;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const T* fa = lds + ((wave & 1) * WM + (lane & 15)) * FA::pitch + 2 * (lane >> 4);
  const T* fb = lds + LdsTile<T, BM, BK>::size + ((wave >> 1) * WN + (lane & 15)) * FB::pitch + 2 * (lane >> 4);

  constexpr bool f32 = sizeof(T) == 4;
  f4 low[f32 ? TM : 1][f32 ? TN : 1];   // FP32 sums of the current run
  auto flush = [&] {
#pragma unroll
    for (int i = 0; f32 && i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] += __builtin_convertvector(low[i][j], d4);
        low[i][j] = f4{0, 0, 0, 0};
      }
  };
  auto fma = [&](T a, T b, int i, int j) {
    if constexpr (f32) low[i][j] = MM::step(a, b, low[i][j]);
    else acc[i][j] = MM::step(a, b, acc[i][j]);
  };
#pragma unroll
  for (int i = 0; f32 && i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) low[i][j] = f4{0, 0, 0, 0};
  auto mma = [&](int b) {
#pragma unroll
    for (int ks = 0; ks < BK; ks += 8) {
      t2 af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = *reinterpret_cast<const t2*>(fa + b * slab + 16 * i * FA::pitch + ks);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = *reinterpret_cast<const t2*>(fb + b * slab + 16 * j * FB::pitch + ks);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) fma(af[i].x, bf[j].x, i, j);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) fma(af[i].y, bf[j].y, i, j);
    }
  };
  const int64_t run = tab ? (int64_t)kKCache : kend - kbeg;
  for (int64_t kr = kbeg; kr < kend; kr += run) {
    const int klen = (int)(kend - kr < run ? kend - kr : run);
    const int nfull = klen / BK;   // whole slabs
    const int nsteps = ((klen + BK - 1) / BK + KS - 1) / KS;
    FA la;
    FB lb;
    la.init(g.A, g.rowA, m0, g.M, g.a_kfast, g.kA_aff, kr, tid);
    lb.init(g.B, g.colB, n0, g.N, g.b_kfast, g.kB_aff, kr, tid);
    typename FA::Slab ra[2];
    typename FB::Slab rb[2];
    if (tab) {
      if (kr > kbeg) __syncthreads();
      for (int i = (int)threadIdx.x; i < klen; i += 256 * KS) {
        if (FA::tab) kts[i] = (uint32_t)(g.kA_aff >= 0 ? (kr + i) * g.kA_aff : (int64_t)g.kA[kr + i]) * FA::unit;
        if (FB::tab)
          kts[kKCache + i] = (uint32_t)(g.kB_aff >= 0 ? (kr + i) * g.kB_aff : (int64_t)g.kB[kr + i]) * FB::unit;
      }
      __syncthreads();
    }
    auto first = [&](int s) { return (s * KS + grp) * BK; };
    // values of slab s to register set x, and from there to LDS buffer x; whole
    // slabs, and any slab (past the end: zeros, so both groups run the same barriers)
    auto fetch = [&](int x, int s) {
      la.fetch(ra[x], first(s), kts);
      lb.fetch(rb[x], first(s), kts + kKCache);
    };
    auto fetch_any = [&](int x, int s) {
      if (s * KS + grp < nfull) {
        fetch(x, s);
      } else {
        la.fetch_tail(ra[x], first(s), klen, kts);
        lb.fetch_tail(rb[x], first(s), klen, kts + kKCache);
      }
    };
    auto stash = [&](int x) {
      la.stash(lds + x * slab, ra[x]);
      lb.stash(lds + x * slab + LdsTile<T, BM, BK>::size, rb[x]);
    };
    auto stash_any = [&](int x, int s) {
      if (s * KS + grp < nfull) {
        stash(x);
      } else {
        la.stash_tail(lds + x * slab, ra[x], klen - first(s));
        lb.stash_tail(lds + x * slab + LdsTile<T, BM, BK>::size, rb[x], klen - first(s));
      }
    };
    // step s: slab s is in buffer x = s & 1; register set 1 - x holds slab s + 1
    auto step = [&](int x, int s) {
      __syncthreads();
      stash(1 - x);
      fetch(1 - x, s + 3);
      mma(x);
    };
    auto step_any = [&](int x, int s) {
      __syncthreads();
      if (s + 1 < nsteps) stash_any(1 - x, s + 1);
      if (s + 3 < nsteps) fetch_any(1 - x, s + 3);
      mma(x);
    };
    fetch_any(0, 0);
    if (nsteps > 1) fetch_any(1, 1);
    stash_any(0, 0);
    if (nsteps > 2) fetch_any(0, 2);
    // a run's slabs are counted per group; after slab s, s odd
    auto end_run = [&](int s) {
      if (f32 && (s + 1) % (kF32Run / BK) == 0) flush();
    };
    int s = 0;
    for (; s + 4 < nfull / KS; s += 2) {
      step(0, s);
      step(1, s + 1);
      end_run(s + 1);
    }
    for (; s + 2 <= nsteps; s += 2) {
      step_any(0, s);
      step_any(1, s + 1);
      end_run(s + 1);
    }
    if (s < nsteps) step_any(0, s);
    if (f32) flush();
  }
}

// FEW: k-contiguous tables and tables only, whatever the operands
template <typename T, typename IO, int BM, int BN, int BK, int KS, bool FEW = false>
__device__ __forceinline__ void tile_mma(const GemmArgs& g, int64_t m0, int64_t n0, int64_t kbeg, int64_t kend,
                                         unsigned char* smem, d4 (&acc)[BM / 32][BN / 32]) {
  // 0 contiguous, 1 strided, 2 pairs, 3 k-contiguous table, 4 table
  const int ma = g.kA_aff >= 0 ? (g.a_kfast && g.kA_aff == 1 ? 0 : 1) : g.a_kfast ? (g.a_pair ? 2 : 3) : 4;
  const int mb = g.kB_aff >= 0 ? (g.b_kfast && g.kB_aff == 1 ? 0 : 1) : g.b_kfast ? (g.b_pair ? 2 : 3) : 4;
  // two k per load (a chain may enter an operand at an odd index, between pairs)
  const bool even = !(kbeg & 1);
  const bool pa = ma == 0 || (ma == 2 && even), pb = mb == 0 || (mb == 2 && even);
#define CCQ_RUN(a, b) tile_run<T, IO, BM, BN, BK, KS, KMode::a, KMode::b>(g, m0, n0, kbeg, kend, smem, acc)
  if (g.wide) CCQ_RUN(Wide, Wide);
  else if (FEW && g.a_kfast && g.b_kfast) CCQ_RUN(TabK, TabK);
  else if (FEW) CCQ_RUN(Tab, Tab);
  else if (ma < 2 && mb < 2) {
    if (ma == 0 && mb == 0) CCQ_RUN(Vec, Vec);
    else if (ma == 0) CCQ_RUN(Vec, Aff);
    else if (mb == 0) CCQ_RUN(Aff, Vec);
    else CCQ_RUN(Aff, Aff);
  } else if (pa && pb) CCQ_RUN(Pair, Pair);
  else if (g.a_kfast && g.b_kfast) CCQ_RUN(TabK, TabK);
  else if (g.b_kfast) CCQ_RUN(Tab, TabK);
  else if (g.a_kfast) CCQ_RUN(TabK, Tab);
  else CCQ_RUN(Tab, Tab);
#undef CCQ_RUN
}

template <typename T, typename IO, int BM, int BN, int BK, int KS, bool FEW = false>
__device__ __forceinline__ void gemm_tab_tile(const GemmArgs& g, int tx, int ty, int tz, unsigned char* smem) {
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int TM = WM / 16, TN = WN / 16;
  using MM = Mma<T>;
  const int grp = threadIdx.x >> 8;
  const int tid = threadIdx.x & 255;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int64_t m0 = (int64_t)tx * BM;
  const int64_t n0 = (int64_t)ty * BN;
  const int64_t kbeg = (int64_t)tz * g.kchunk;
  const int64_t kend = (kbeg + g.kchunk < g.K) ? kbeg + g.kchunk : g.K;
  const int wm = (wave & 1) * WM;
  const int wn = (wave >> 1) * WN;

  d4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = d4{0, 0, 0, 0};
  tile_mma<T, IO, BM, BN, BK, KS, FEW>(g, m0, n0, kbeg, kend, smem, acc);

  if (KS > 1) {
    // group 1 hands its accumulators to group 0 (slab order: group 0's sum
    // plus group 1's sum, the same for every launch)
    double* red = reinterpret_cast<double*>(smem);
    __syncthreads();
    if (grp == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) red[(((i * TN + j) * 4 + v) << 8) + tid] = acc[i][j][v];
    }
    __syncthreads();
    if (grp == 1) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] += red[(((i * TN + j) * 4 + v) << 8) + tid];
  }

  if (g.nsplit == 1) {
    if (sizeof(IO) == 4 && g.c64)
      store_tile<IO, double, TM, TN, MM>(g, m0, n0, wm, wn, lane, g.alpha, acc);
    else
      store_tile<IO, IO, TM, TN, MM>(g, m0, n0, wm, wn, lane, g.alpha, acc);
    return;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t gn = n0 + wn + 16 * j + (lane & 15);
    if (gn >= g.N) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t gm = m0 + wm + 16 * i + MM::row(lane, v);
        if (gm >= g.M) continue;
        store_partial(g, tz, gm, gn, acc[i][j][v]);
      }
  }
}

template <typename T, typename IO, int BM, int BN, int BK, int KS>
__global__ __launch_bounds__(256 * KS, kTileWaves<KS>) void gemm_tab(GemmArgs g) {
  __shared__ __align__(16) unsigned char smem[TabLds<T, BM, BN, BK, KS>::bytes];
  int tx, ty, tz;
  tile_coords(g.group, tx, ty, tz);
  gemm_tab_tile<T, IO, BM, BN, BK, KS>(g, tx, ty, tz, smem);
}

// Entries e0 <= e < e1 of a chain accumulating into one output tile (tx, ty):
// the workgroup walks the concatenated K range [kbeg, kend) (kend < 0: all of
// it) entry by entry, each with its own operands and layouts, adds alpha_e
// times the entry's partial product to an FP64 sum, and stores once with the
// first entry's output arguments (split z of a split-K launch: into the
// workspace).
template <typename T, typename IO, int BM, int BN, int BK>
__device__ __forceinline__ void tile_entries(const GemmArgs* es, int e0, int e1, int tx, int ty, int tz,
                                             int64_t kbeg, int64_t kend, unsigned char* smem) {
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int TM = WM / 16, TN = WN / 16;
  using MM = Mma<T>;
  const GemmArgs& o = es[e0];
  const int lane = threadIdx.x & 63;
  const int wave = (threadIdx.x & 255) >> 6;
  const int64_t m0 = (int64_t)tx * BM;
  const int64_t n0 = (int64_t)ty * BN;
  const int wm = (wave & 1) * WM;
  const int wn = (wave >> 1) * WN;

  d4 sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  int64_t off = 0;
  for (int e = e0; e < e1; ++e) {
    const GemmArgs& g = es[e];
    const int64_t lo = kend < 0 ? off : (kbeg > off ? kbeg : off);
    const int64_t hi = kend < 0 ? off + g.K : (kend < off + g.K ? kend : off + g.K);
    const int64_t a = lo - off, b = hi - off;
    off += g.K;
    if (a >= b) continue;
    d4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = d4{0, 0, 0, 0};
    // the previous entry's waves are past their last LDS reads
    if (e > e0) __syncthreads();
    tile_mma<T, IO, BM, BN, BK, 1>(g, m0, n0, a, b, smem, acc);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[i][j][v] += g.alpha * acc[i][j][v];
  }

  if (kend < 0 || o.nsplit == 1) {
    store_tile<IO, IO, TM, TN, MM>(o, m0, n0, wm, wn, lane, 1.0, sum);
    return;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t gn = n0 + wn + 16 * j + (lane & 15);
    if (gn >= o.N) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t gm = m0 + wm + 16 * i + MM::row(lane, v);
        if (gm >= o.M) continue;
        store_partial(o, tz, gm, gn, sum[i][j][v]);
      }
  }
}

// A chain of GEMMs accumulating into one output with the same tile mapping
// and operand layouts (C (+)= sum_e alpha_e A_e B_e (+ dcoef D)), as one
// product over the concatenated K ranges, split along the concatenated K
// (split z of tile (tx, ty) covers [z kchunk, (z + 1) kchunk)).
template <typename T, typename IO, int BM, int BN, int BK>
__global__ __launch_bounds__(256, kTileWaves<1>) void gemm_tab_chain(GemmChain ch) {
  __shared__ __align__(16) unsigned char smem[TabLds<T, BM, BN, BK, 1>::bytes];
  int tx, ty, tz;
  tile_coords(ch.e[0].group, tx, ty, tz);
  const int64_t ktot = ch.koff[ch.n];
  const int64_t kbeg = (int64_t)tz * ch.e[0].kchunk;
  const int64_t kend = (kbeg + ch.e[0].kchunk < ktot) ? kbeg + ch.e[0].kchunk : ktot;
  tile_entries<T, IO, BM, BN, BK>(ch.e, 0, ch.n, tx, ty, tz, kbeg, kend, smem);
}

// The same tile kernel over the tiles of a group of independent GEMMs (full K
// each).
template <typename T, typename IO, int BM, int BN, int BK>
__global__ __launch_bounds__(256, kTileWaves<1>) void gemm_tab_group(GemmGroup gg) {
  __shared__ __align__(16) unsigned char smem[TabLds<T, BM, BN, BK, 1>::bytes];
  int tx, ty;
  const int mem = group_tile<BM, BN>(gg, tx, ty);
  gemm_tab_tile<T, IO, BM, BN, BK, 1>(gg.g[mem], tx, ty, 0, smem);
}

// One dependency level (launch_level).  Bodies of every task kind in one kernel:
// the operations of a level are a few microseconds each, most of it latency
// (descriptor, tables, operands), so a launch per operation costs 3 - 4 us of
// GPU time, or 4 us of host time each in a graph with parallel branches; side
// by side in one launch they share that latency.  CCSD 24 orbitals: 919 us a
// sweep as 176 launches, 185 us in 27 levels.
// The descriptors are read through the constant address space: nothing
// writes them while the kernel runs, so they stay scalar loads.
// Adds and sums move up to 2048 elements an item, all loads of a thread in
// flight before its first store: an item lasts as long as its latencies do, and beside
// large products it has one of a CU's three places (1024 elements an item, loads
// of 8 bytes: CCSD, 100 orbitals, 1900 us a sweep, this 1867).
template <typename IO>
struct Pair2 {
  typedef IO type __attribute__((ext_vector_type(2), aligned(sizeof(IO))));
};
template <typename IO>
__device__ __forceinline__ d2 ldg2(const double* p, int64_t i) {
  const auto v = *reinterpret_cast<const typename Pair2<IO>::type*>(reinterpret_cast<const IO*>(p) + i);
  return d2{(double)v.x, (double)v.y};
}
template <typename IO>
__device__ __forceinline__ void stg2(double* p, int64_t i, d2 v) {
  typename Pair2<IO>::type w;
  w.x = (IO)v.x;
  w.y = (IO)v.y;
  *reinterpret_cast<typename Pair2<IO>::type*>(reinterpret_cast<IO*>(p) + i) = w;
}

// (IOC: the stored type of C, as in store_c)
template <typename IO, typename IOC>
__device__ __forceinline__ void level_perm(const LevelTask& t, int idx) {
  const GemmArgs& g = t.g;
  const uint32_t N = (uint32_t)g.N, total = (uint32_t)(g.M * g.N);
  const uint32_t e0 = (uint32_t)idx * (uint32_t)t.chunk;
  const uint32_t e1 = total - e0 < (uint32_t)t.chunk ? total : e0 + (uint32_t)t.chunk;
  auto run = [&](uint32_t b, auto count) {   // count elements a thread, 256 apart
    constexpr int J = decltype(count)::value;
    int64_t ia[J], ic[J];
    double v[J], c[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint32_t e = b + 256u * j < e1 ? b + 256u * j : b;
      const uint32_t r = e / N, n = e - r * N;
      ia[j] = (int64_t)g.rowA[r] + g.kA[n];
      ic[j] = (int64_t)g.rowC[r] + g.colC[n];
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      v[j] = ldg<IO>(g.A, ia[j]);
      c[j] = g.accumulate ? ldg<IOC>(g.C, ic[j]) : 0.0;
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (b + 256u * j < e1) stg<IOC>(g.C, ic[j], g.accumulate ? c[j] + g.alpha * v[j] : g.alpha * v[j]);
  };
  uint32_t b = e0 + threadIdx.x;
  if (t.chunk > 512)
    for (; b < e1; b += 2048) run(b, std::integral_constant<int, 8>{});
  else
    for (; b < e1; b += 512) run(b, std::integral_constant<int, 2>{});
}

// C (+)= alpha A, or C += the sum of n arrays; whole pairs, then the last one.
// (IOC: the stored type of an add's C, of the arrays of a sum, whose C is IO)
template <typename IO, typename IOC>
__device__ __forceinline__ void level_flat(const LevelTask& t, int idx) {
  const GemmArgs& g = t.g;
  const int64_t total = t.kind == kLvSum ? g.M : g.M * g.N, e0 = (int64_t)idx * t.chunk;
  const int64_t e1 = e0 + t.chunk < total ? e0 + t.chunk : total;
  const bool add = t.kind != kLvSum;
  auto one = [&](int64_t e) {
    double s = add ? g.alpha * ldg<IO>(g.A, e) : 0.0;
    if (!add) {
      s = ldg<IO>(g.C, e);
      for (int k = 0; k < t.nsrc; ++k) s += ldg<IOC>(t.src[k], e);
    } else if (g.accumulate) {
      s = ldg<IOC>(g.C, e) + s;
    }
    if (add) stg<IOC>(g.C, e, s);
    else stg<IO>(g.C, e, s);
  };
  auto pairs = [&](int64_t e, auto count) {   // count pairs a thread, 512 elements apart
    constexpr int J = decltype(count)::value;
    d2 s[J];
    if (add) {
      d2 v[J];
#pragma unroll
      for (int j = 0; j < J; ++j) {
        v[j] = ldg2<IO>(g.A, e + 512 * j);
        s[j] = g.accumulate ? ldg2<IOC>(g.C, e + 512 * j) : d2{0.0, 0.0};
      }
#pragma unroll
      for (int j = 0; j < J; ++j)
        s[j] = g.accumulate ? s[j] + g.alpha * v[j] : g.alpha * v[j];
    } else {
      d2 v[kMaxLevelSrc - 1][J];
#pragma unroll
      for (int j = 0; j < J; ++j) s[j] = ldg2<IO>(g.C, e + 512 * j);
#pragma unroll
      for (int k = 0; k < kMaxLevelSrc - 1; ++k)
        if (k < t.nsrc)
#pragma unroll
          for (int j = 0; j < J; ++j) v[k][j] = ldg2<IOC>(t.src[k], e + 512 * j);
#pragma unroll
      for (int k = 0; k < kMaxLevelSrc - 1; ++k)
        if (k < t.nsrc)
#pragma unroll
          for (int j = 0; j < J; ++j) s[j] += v[k][j];
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (add) stg2<IOC>(g.C, e + 512 * j, s[j]);
      else stg2<IO>(g.C, e + 512 * j, s[j]);
  };
  int64_t e = e0 + 2 * threadIdx.x;
  for (; e - 2 * threadIdx.x + 1024 <= e1; e += 1024) pairs(e, std::integral_constant<int, 2>{});
  for (; e + 2 <= e1; e += 512) pairs(e, std::integral_constant<int, 1>{});
  if (e < e1) one(e);
}

// P = 2^pshift threads share an element (splits p, p + P, ...), combined in p
// order; 256 / P elements a pass
template <typename IO, typename IOC>
__device__ __forceinline__ void level_reduce(const LevelTask& t, int idx, double* red) {
  const GemmArgs& g = t.g;
  const int P = 1 << t.pshift, p = threadIdx.x & (P - 1);
  const uint32_t total = (uint32_t)(g.M * g.N), N = (uint32_t)g.N;
  const uint32_t e0 = (uint32_t)idx * (uint32_t)t.chunk;
  const uint32_t e1 = total - e0 < (uint32_t)t.chunk ? total : e0 + (uint32_t)t.chunk;
  for (uint32_t b = e0; b < e1; b += 256u >> t.pshift) {
    const uint32_t e = b + (threadIdx.x >> t.pshift);
    double s = 0.0;
    if (e < e1) s = sum_strided(g.ws + (int64_t)p * total + e, (int64_t)P * total, (g.nsplit - p + P - 1) >> t.pshift);
    if (P > 1) {
      if (b > e0) __syncthreads();
      red[threadIdx.x] = s;
      __syncthreads();
      if (p == 0)
        for (int x = 1; x < P; ++x) s += red[threadIdx.x + x];
    }
    if (e < e1 && p == 0) store_c<IO, IOC>(g, e / N, e % N, s, g.alpha);
  }
}

template <typename T, typename IO>
__global__ __launch_bounds__(256, kTileWaves<1>) void level_kernel(const LevelTask* __restrict__ tasks,
                                                                   const LevelItem* __restrict__ items) {
  // the FP64 tiles are in every arithmetic's kernel; theirs is the largest LDS
  constexpr int b1 = TabLds<double, 64, 64, tile_bk(64, 64), 1>::bytes, b2 = TabLds<double, 32, 32, tile_bk(32, 32), 1>::bytes;
  __shared__ __align__(16) unsigned char smem[b1 > b2 ? b1 : b2];
  typedef const __attribute__((address_space(4))) LevelTask* ConstTask;
  typedef const __attribute__((address_space(4))) LevelItem* ConstItem;
  const LevelItem& it = *(const LevelItem*)((ConstItem)items + blockIdx.x);
  if (it.task < 0) return;
  const LevelTask& t = *(const LevelTask*)((ConstTask)tasks + it.task);
  const int idx = it.idx;
  if (t.kind >= kLvPerm) {
    auto run = [&](auto c) {
      using IOC = decltype(c);
      switch (t.kind) {
        case kLvPerm: level_perm<IO, IOC>(t, idx); break;
        case kLvFlat:
        case kLvSum: level_flat<IO, IOC>(t, idx); break;
        case kLvReduce: level_reduce<IO, IOC>(t, idx, reinterpret_cast<double*>(smem)); break;
        default: {
          const int64_t e0 = (int64_t)idx * t.chunk;
          const int64_t e1 = e0 + t.chunk < t.g.M ? e0 + t.chunk : t.g.M;
          for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) stg<IOC>(t.g.C, e, 0.0);
        }
      }
    };
    if constexpr (sizeof(IO) == 4) {
      if (t.g.c64) {
        run(double());
        return;
      }
    }
    run(IO());
    return;
  }
  const GemmArgs& g = t.g;
  const int tm = (int)((g.M + g.bm - 1) / g.bm), tn = (int)((g.N + g.bn - 1) / g.bn);
  const int per_z = tm * tn;
  const int tz = idx / per_z;
  int tx, ty;
  tile_in_group(idx - tz * per_z, tm, tn, g.group, tx, ty);
#define CCQ_LV(A, FEW)                                                                         \
  switch ((t.kind - kLvTile6464) & 3) {                                                        \
    case 0: gemm_tab_tile<A, IO, 64, 64, tile_bk(64, 64), 1, FEW>(g, tx, ty, tz, smem); break; \
    case 1: gemm_tab_tile<A, IO, 64, 32, tile_bk(64, 32), 1, FEW>(g, tx, ty, tz, smem); break; \
    case 2: gemm_tab_tile<A, IO, 32, 64, tile_bk(32, 64), 1, FEW>(g, tx, ty, tz, smem); break; \
    default: gemm_tab_tile<A, IO, 32, 32, tile_bk(32, 32), 1, FEW>(g, tx, ty, tz, smem);       \
  }
  // FP64 products of the FP32 modes are small or bound by memory; on FP32 storage
  // three operand modes for them are faster than nine (CCSDTQ 14 orbitals 2534 ->
  // 2389 us a sweep, CCSDT 40 2298 -> 2276), on FP64 storage slower (2500 -> 2515)
  if constexpr (sizeof(T) == 4) {
    if (t.kind >= kLvTileF64) {
      CCQ_LV(double, sizeof(IO) == 4)
      return;
    }
  }
  CCQ_LV(T, false)
#undef CCQ_LV
}

// Register-direct GEMM for skinny and dot-shaped products (an output extent
// of at most a few MFMA tiles; HBM / latency bound).  No LDS staging: in a
// 16-deep k step, lane l loads row l%16 of each 16-row block at
// k = kb + 4*(l/16) + s, s = 0..3, and MFMA s contracts exactly those k
// (the A/B fragment layout of v_mfma_f64_16x16x4f64 with the 4 MFMAs of the
// step taking k in the order kb + 4q + s, q = 0..3).  The next step's values
// are loaded while the current step is multiplied.
// Workgroup = 4 waves: WK along K (same output tile, interleaved k steps,
// combined through LDS in wave order), 4/WK along M.  Wave tile (16 RM) x (16 RN).
// The step holds the stored type IO (converted at the MFMA, so a load in
// flight is not waited for before the current step's MFMAs).
template <typename IO, int RM, int RN, int WK>
struct RegStep {
  IO a[RM][4];
  IO b[RN][4];
};

template <typename IO, int RM, int RN, int WK>
__device__ __forceinline__ void reg_load(RegStep<IO, RM, RN, WK>& st, const GemmArgs& g, const int (&ra)[RM],
                                         const int (&cb)[RN], int q, int64_t kb, int64_t kend) {
  const IO* __restrict__ A = reinterpret_cast<const IO*>(g.A);
  const IO* __restrict__ B = reinterpret_cast<const IO*>(g.B);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int64_t gk = kb + 4 * q + s;
    const bool in = gk < kend;
    const int64_t oa = in ? koff(g.kA, g.kA_aff, gk) : 0;
    const int64_t ob = in ? koff(g.kB, g.kB_aff, gk) : 0;
#pragma unroll
    for (int i = 0; i < RM; ++i) st.a[i][s] = (in && ra[i] >= 0) ? A[(int64_t)ra[i] + oa] : IO(0);
#pragma unroll
    for (int j = 0; j < RN; ++j) st.b[j][s] = (in && cb[j] >= 0) ? B[ob + cb[j]] : IO(0);
  }
}

template <typename IO, int RM, int RN, int WK>
__device__ __forceinline__ void reg_mma(d4 (&acc)[RM][RN], const RegStep<IO, RM, RN, WK>& st) {
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)st.a[i][s], (double)st.b[j][s], acc[i][j], 0, 0, 0);
}

template <typename IO, int RM, int RN, int WK>
__global__ __launch_bounds__(256) void gemm_f64_reg(GemmArgs g) {
  constexpr int WMW = 4 / WK;
  constexpr int TBM = WMW * 16 * RM, TBN = 16 * RN;
  constexpr int WACC = 256 * RM * RN;   // doubles of one wave's accumulators
  constexpr int SMEM = WK > 1 ? (WK - 1) * WMW * WACC : 1;
  __shared__ double red[SMEM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wk = wave % WK, wmi = wave / WK;
  const int r = lane & 15, q = lane >> 4;
  int tx, ty, tz;
  tile_coords(g.group, tx, ty, tz);
  const int64_t m0 = (int64_t)tx * TBM, n0 = (int64_t)ty * TBN;
  const int64_t wm0 = m0 + wmi * 16 * RM;
  const int64_t kbeg = (int64_t)tz * g.kchunk;
  const int64_t kend = (kbeg + g.kchunk < g.K) ? kbeg + g.kchunk : g.K;
  int ra[RM], cb[RN];
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int64_t m = wm0 + 16 * i + r;
    ra[i] = m < g.M ? g.rowA[m] : -1;
  }
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    const int64_t n = n0 + 16 * j + r;
    cb[j] = n < g.N ? g.colB[n] : -1;
  }
  d4 acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = d4{0, 0, 0, 0};

  const int64_t nsteps = kend > kbeg ? (kend - kbeg + 15) / 16 : 0;
  RegStep<IO, RM, RN, WK> s0, s1;
  int64_t st = wk;
  if (st < nsteps) reg_load<IO>(s0, g, ra, cb, q, kbeg + 16 * st, kend);
  while (st < nsteps) {
    const int64_t n1 = st + WK;
    if (n1 < nsteps) reg_load<IO>(s1, g, ra, cb, q, kbeg + 16 * n1, kend);
    reg_mma(acc, s0);
    if (n1 >= nsteps) break;
    const int64_t n2 = n1 + WK;
    if (n2 < nsteps) reg_load<IO>(s0, g, ra, cb, q, kbeg + 16 * n2, kend);
    reg_mma(acc, s1);
    st = n2;
  }

  if (WK > 1) {
    // waves wk > 0 hand their accumulators to wave wk == 0 of the same M slot
    if (wk > 0) {
      double* dst = red + ((wk - 1) * WMW + wmi) * WACC;
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) dst[((i * RN + j) * 4 + v) * 64 + lane] = acc[i][j][v];
    }
    __syncthreads();
    if (wk == 0) {
      for (int w = 1; w < WK; ++w) {
        const double* src = red + ((w - 1) * WMW + wmi) * WACC;
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[i][j][v] += src[((i * RN + j) * 4 + v) * 64 + lane];
      }
    }
  }

  if (wk != 0) return;
  // lane l, register v of 16x16 block (i, j) holds row 16i + l/16 + 4v and
  // column 16j + l%16: the FP64 MFMA output layout of the tile epilogue
  if (g.nsplit == 1) {
    if (sizeof(IO) == 4 && g.c64)
      store_tile<IO, double, RM, RN, Mma<double>>(g, wm0, n0, 0, 0, lane, g.alpha, acc);
    else
      store_tile<IO, IO, RM, RN, Mma<double>>(g, wm0, n0, 0, 0, lane, g.alpha, acc);
    return;
  }
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    const int64_t gn = n0 + 16 * j + r;
    if (gn >= g.N) continue;
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t gm = wm0 + 16 * i + q + 4 * v;
        if (gm >= g.M) continue;
        store_partial(g, tz, gm, gn, acc[i][j][v]);
      }
  }
}


// Launchers of one arithmetic / storage pair (defined in the gemm_*.hip
// units); false when the plan names a shape that has no instantiation.
// f64: FP64 MFMA on FP64 storage; f32: FP32 MFMA on FP64 storage; f32io:
// FP32 MFMA on FP32 storage.  The register-direct kernel depends on the
// storage only (f64: FP64 storage, f32io: FP32 storage).
bool launch_tile_f64(hipStream_t s, dim3 grid, const GemmArgs& g);
bool launch_tile_f32(hipStream_t s, dim3 grid, const GemmArgs& g);
bool launch_tile_f32io(hipStream_t s, dim3 grid, const GemmArgs& g);
bool launch_chain_f64(hipStream_t s, dim3 grid, const GemmChain& ch);
bool launch_chain_f32(hipStream_t s, dim3 grid, const GemmChain& ch);
bool launch_chain_f32io(hipStream_t s, dim3 grid, const GemmChain& ch);
bool launch_group_f64(hipStream_t s, dim3 grid, const GemmGroup& gg);
bool launch_group_f32(hipStream_t s, dim3 grid, const GemmGroup& gg);
bool launch_group_f32io(hipStream_t s, dim3 grid, const GemmGroup& gg);
void launch_level_f64(hipStream_t s, const LevelTask* tasks, const LevelItem* items, int n);
void launch_level_f32(hipStream_t s, const LevelTask* tasks, const LevelItem* items, int n);
void launch_level_f32io(hipStream_t s, const LevelTask* tasks, const LevelItem* items, int n);
bool launch_reg_f64(hipStream_t s, dim3 grid, const GemmArgs& g);
bool launch_reg_f32io(hipStream_t s, dim3 grid, const GemmArgs& g);

}  // namespace ccqk
