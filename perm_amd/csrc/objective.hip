// PERM container objective on gfx950 (coldpress/perm/objective.py:17-49).
//
// tensor_err(x, ttype, qw, perm, wvec, rows) =
//     sum_c w[c] * sum_r (roundtrip(x[rows][:, perm])[r, c] - x[rows][r, perm[c]])^2
// with w = wvec[perm], qw[perm] or 1, evaluated for many tensors in one pass:
//   gather   x rows (a sorted sample) and permuted columns, f16 or f32 -> f32
//   encode   the container codec bodies of kq_blocks.h, one launch per type group, which
//            write the decoded weights (Q8_0: bytes, then its decoder)
//   colsum   per column, the float64 squared errors added row after row -- the
//            order of numpy's d2.sum(0) over a C-contiguous array, so the result is
//            bit-identical
//   final    +0.0 plus numpy's pairwise sum of colerr * w (the order of a
//            contiguous float64 .sum()), one workgroup per tensor
// col_log_rms(x, row_step) is the per-column float64 sum of squares in row chunks
// (a sequential chain per chunk, the chunk sums added in order), then
// log(sqrt(acc / nrow) + 1e-12).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "kq_blocks.h"
#include "np_sum.h"
#include "phase_clock.h"

namespace cp {

// Table-held pointers are generic to the compiler; reads through these global
// address-space types become global loads (a flat load also waits on LDS traffic
// and forces the loads ahead of it to drain).
typedef const float __attribute__((address_space(1)))* GF32;
typedef const uint16_t __attribute__((address_space(1)))* GU16;
typedef const int32_t __attribute__((address_space(1)))* GI32;

struct ErrDev {
  const void* x;
  const int32_t* rows;
  const int32_t* perm;
  const float* qw;
  const double* wvec;
  float* xs;       // [R, n] gathered targets
  float* qwp;      // [n] qw[perm] (or null)
  uint8_t* raw;    // Q8_0's bytes [R, n / 32 * 34] (the k-quants leave none)
  float* recon;    // [R, n]
  double* colerr;  // [n]
  int* bad;        // set when an index is out of range
  int64_t nrow_src;
  int R, n, ttype, x_f16;
  int slot;  // the caller's index of this tensor (its result slot)
  int gfirst;  // first workgroup of the gather that works on this tensor
  int by_rows; // table index of the tensor with the k-th most rows, k this entry's index
};

// --------------------------------------------------------------- gather
// Workgroups take tiles of kGatherRows rows x 1024 columns, tensor by tensor (gfirst), so a
// call of one large and many small tensors launches no idle ones. A thread keeps its four
// consecutive columns' indices in registers over the tile's rows, so an entry costs its
// gathered load and a quarter of a 16-byte store. (One thread per four entries of a
// (largest tensor, tensors) grid, reading and checking its indices for every row, took
// 238 us for 29 tensors of 1 M - 16.8 M entries; this takes 138, 3.5 TB/s of f16 in and f32
// out.) Negative indices count from the end, as numpy's do; indices still out of range read
// element 0 and flag the tensor, whose result becomes NaN.
constexpr int kGatherRows = 32, kGatherCols = 1024;

// Rows i0, i0 + steps, ... below i1, columns j .. j + 3. NARROW false: steps is 1 (its own code:
// a step in a register took the 1024-wide tiles 137 -> 142 us).
template <bool F16, bool NARROW>
__device__ __forceinline__ void gather_tile(const ErrDev& T, int i0, int i1, int steps, int j) {
  const int n = T.n, step = NARROW ? steps : 1;
  const GU16 x16 = (GU16)T.x;
  const GF32 x32 = (GF32)T.x;
  const GI32 perm = (GI32)T.perm, rows = (GI32)T.rows;
  bool bad = false;
  int c[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    c[q] = perm ? perm[j + q] : j + q;
    c[q] = c[q] < 0 ? c[q] + n : c[q];
    if (c[q] < 0 || c[q] >= n) {
      bad = true;
      c[q] = 0;
    }
  }
  const auto row_of = [&](int i) {
    int64_t src = rows ? rows[i] : i;
    src = src < 0 ? src + T.nrow_src : src;
    if (src < 0 || src >= T.nrow_src) {
      bad = true;
      src = 0;
    }
    return src * n;
  };
  float4* out = reinterpret_cast<float4*>(T.xs + j);
  constexpr int U = 8;  // rows in flight
  int i = i0;
  for (; i1 - i > (U - 1) * step; i += U * step) {
    float v[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t o = row_of(i + u * step);
#pragma unroll
      for (int q = 0; q < 4; ++q) v[u][q] = F16 ? half_value(x16[o + c[q]]) : x32[o + c[q]];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      out[(int64_t)(i + u * step) * (n / 4)] = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
  }
  for (; i < i1; i += step) {
    const int64_t o = row_of(i);
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = F16 ? half_value(x16[o + c[q]]) : x32[o + c[q]];
    out[(int64_t)i * (n / 4)] = make_float4(v[0], v[1], v[2], v[3]);
  }
  if (bad) *T.bad = 1;
}

__global__ __launch_bounds__(256) void err_gather_kernel(const ErrDev* __restrict__ tab, int count) {
  int lo = 0, hi = count - 1;  // the last tensor with gfirst <= blockIdx.x
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (tab[mid].gfirst <= (int)blockIdx.x)
      lo = mid;
    else
      hi = mid - 1;
  }
  const ErrDev& T = tab[lo];
  const int blk = (int)blockIdx.x - T.gfirst, n = T.n;
  if (blk == 0 && T.qwp) {
    for (int j = threadIdx.x; j < n; j += 256) {
      int c = T.perm ? T.perm[j] : j;
      c = c < 0 ? c + n : c;  // numpy's negative indices
      if (c < 0 || c >= n) {
        *T.bad = 1;
        c = 0;
      }
      T.qwp[j] = T.qw[c];
    }
  }
  const int ct = (n + kGatherCols - 1) / kGatherCols, rt = blk / ct;
  // up to 512 columns leave half the threads or more over: they take rows of their own (32
  // columns walked by 8 of 256 threads, [64, 32]: 6.4 us; 3.1 so)
  const int w = n / 4 < 256 ? n / 4 : 256, step = 256 / w, r = (int)threadIdx.x / w;
  const int j = (blk - rt * ct) * kGatherCols + 4 * ((int)threadIdx.x - r * w);
  if (r >= step || j >= n) return;  // n % 32 == 0: the four columns exist together
  const int64_t i0 = (int64_t)rt * kGatherRows;
  const int i1 = (int)(T.R - i0 < kGatherRows ? T.R : i0 + kGatherRows);
  const auto tile = [&](auto f16) {
    constexpr bool F16 = decltype(f16)::value;
    if (step > 1)
      gather_tile<F16, true>(T, (int)i0 + r, i1, step, j);
    else
      gather_tile<F16, false>(T, (int)i0, i1, 1, j);
  };
  if (T.x_f16)
    tile(std::true_type());
  else
    tile(std::false_type());
}

// Workgroups of one tensor's gather.
static int64_t gather_tiles(int64_t R, int64_t n) {
  return ((R + kGatherRows - 1) / kGatherRows) * ((n + kGatherCols - 1) / kGatherCols);
}

// --------------------------------------------------------------- codec
template <int TT, bool IMAT>
__global__ __launch_bounds__(256) void err_encode_kernel(const ErrDev* __restrict__ tab) {
  const ErrDev& T = tab[blockIdx.y];
  const int64_t w = (int64_t)T.R * T.n;
  if constexpr (TT == CP_Q8_0) {
    const int64_t nblk = w / 32;
    if ((int64_t)blockIdx.x * 8 * kWavesPerBlock >= nblk) return;
    q8_encode_block(T.xs, nblk, T.raw, blockIdx.x);
  } else {
    constexpr int S = 64 / Kq<TT>::G;
    const int64_t NB = w / 256;
    const int64_t blocks = ((NB + S - 1) / S + kWavesPerBlock - 1) / kWavesPerBlock;
    if ((int64_t)blockIdx.x >= blocks) return;
    kq_encode_block<TT, IMAT, KqOut::kRecon>(T.xs, T.qwp, NB, T.n / 256, nullptr, blockIdx.x, T.recon);
  }
}

// Q8_0: one thread per 4 weights.
__global__ __launch_bounds__(256) void err_decode_q8_kernel(const ErrDev* __restrict__ tab) {
  const ErrDev& T = tab[blockIdx.y];
  q8_decode_thread(T.raw, (int64_t)T.R * T.n / 32, T.recon, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// --------------------------------------------------------------- column sums
// The sequential chain of one column over rows [r0, r1), loads running one block
// of B rows ahead of the adds. The block after next is always loaded (clamped to
// the last full block), so no branch sits between a load and its use and the
// loads never have to drain early.
template <int B, class T, class Ld, class Use>
__device__ __forceinline__ void chain_rows(int64_t r0, int64_t r1, const Ld& ld, const Use& use) {
  const int64_t nfull = (r1 - r0) / B;
  T a[B], b[B];
  auto fill = [&](T (&v)[B], int64_t r) {
#pragma unroll
    for (int i = 0; i < B; ++i) v[i] = ld(r + i);
  };
  auto drain = [&](const T (&v)[B]) {
#pragma unroll
    for (int i = 0; i < B; ++i) use(v[i]);
  };
  if (nfull > 0) fill(a, r0);
  int64_t k = 0;
  for (; k + 1 < nfull; k += 2) {
    fill(b, r0 + (k + 1) * B);
    drain(a);
    const int64_t ra = r0 + (k + 2) * B;
    fill(a, ra < r1 - B ? ra : r1 - B);  // past the end: a valid block, never used
    drain(b);
  }
  if (k < nfull) drain(a);
  for (int64_t r = r0 + nfull * B; r < r1; ++r) {
    T v = ld(r);
    use(v);
  }
}

// colerr[c] = (((0 + d2[0,c]) + d2[1,c]) + ...), d2 the float64 square of the float64
// difference. The order makes each column one chain of R additions, so a column's time is
// that chain or the delivery of its values, whichever is longer. A workgroup takes 32 columns
// (128-byte row segments): seven waves load four tiles ahead and put the squares, which are off
// the chain, into a double-buffered LDS tile; the eighth only adds, one lane per column,
// reading 16 rows ahead of the adds. One wave doing it all for 64 columns, its loads one
// 16-row block ahead, took 741 us for 29 tensors (79.7 M entries, one of 16384 rows) where this
// takes 228, the tensors with the most rows first (269 in table order): 2.8 TB/s.
constexpr int kSumCols = 32, kSumWaves = 8, kSumPer = 8, kSumAhead = 4;
constexpr int kSumRows = (kSumWaves - 1) * 2 * kSumPer;  // 112 rows per tile

__global__ __launch_bounds__(64 * kSumWaves) void err_colsum_kernel(const ErrDev* __restrict__ tab) {
  const ErrDev& T = tab[tab[blockIdx.y].by_rows];  // longest chains first
  const int64_t n = T.n;
  const int c0 = (int)blockIdx.x * kSumCols;
  if (c0 >= n) return;  // n % 32 == 0: all 32 columns exist
  __shared__ double d2[2][kSumRows][kSumCols];
  const int R = T.R, tiles = (R + kSumRows - 1) / kSumRows;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), c = (int)threadIdx.x & 31;
  if (wv < kSumWaves - 1) {
    const GF32 xs = (GF32)T.xs + c0 + c;
    const GF32 rc = (GF32)T.recon + c0 + c;
    const int g = ((int)threadIdx.x >> 5) * kSumPer;  // this thread's first row of a tile
    float2 v[kSumAhead][kSumPer];
    auto fill = [&](float2 (&d)[kSumPer], int tile) {
#pragma unroll
      for (int i = 0; i < kSumPer; ++i) {  // past the last row: that row again, never added
        const int64_t r = (int64_t)tile * kSumRows + g + i, rr = r < R ? r : R - 1;
        d[i] = make_float2(xs[rr * n], rc[rr * n]);
      }
    };
#pragma unroll
    for (int a = 0; a < kSumAhead; ++a) fill(v[a], a);
    for (int k = 0; k < tiles; k += kSumAhead) {  // every wave passes the same ``tiles`` barriers
#pragma unroll
      for (int a = 0; a < kSumAhead; ++a) {
        if (k + a >= tiles) break;
#pragma unroll
        for (int i = 0; i < kSumPer; ++i) {
          const double d = (double)v[a][i].y - (double)v[a][i].x;
          d2[a & 1][g + i][c] = d * d;
        }
        __syncthreads();
        fill(v[a], k + a + kSumAhead);
      }
    }
  } else {
    // tile k is whole after barrier k; its buffer is written again only after barrier k + 1,
    // which this wave passes when it has added tile k
    double acc = 0.0;
    for (int k = 0; k < tiles; ++k) {
      __syncthreads();
      const double(*p)[kSumCols] = d2[k & 1];
      const int rows = R - k * kSumRows < kSumRows ? R - k * kSumRows : kSumRows;
      if (rows == kSumRows) {
        double v[2][16];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[0][i] = p[i][c];
#pragma unroll
        for (int q = 0; q < kSumRows / 16; ++q) {
          if (q + 1 < kSumRows / 16) {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[(q + 1) & 1][i] = p[16 * (q + 1) + i][c];
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) acc = acc + v[q & 1][i];
        }
      } else {
        for (int r = 0; r < rows; ++r) acc = acc + p[r][c];
      }
    }
    if (((int)threadIdx.x & 63) < kSumCols) T.colerr[c0 + c] = acc;
  }
}

// --------------------------------------------------------------- total
__global__ __launch_bounds__(256) void err_final_kernel(const ErrDev* __restrict__ tab,
                                                        double* __restrict__ out) {
  __shared__ NpSumLds lds;
  const ErrDev& T = tab[blockIdx.x];
  double s;
  const double* ce = T.colerr;
  if (*T.bad) {
    s = __builtin_nan("");
  } else if (T.wvec) {
    const int32_t* perm = T.perm;
    const double* wv = T.wvec;
    const int64_t n = T.n;
    s = np_sum_block([=](int64_t i) {
      const int64_t c = perm ? perm[i] : i;
      return ce[i] * wv[c < 0 ? c + n : c];
    }, T.n, lds);
  } else if (T.qwp) {
    const float* q = T.qwp;
    s = np_sum_block([=](int64_t i) { return ce[i] * (double)q[i]; }, T.n, lds);
  } else {
    s = np_sum_block([=](int64_t i) { return ce[i]; }, T.n, lds);
  }
  if (threadIdx.x == 0) out[T.slot] = s;
}

__global__ void err_clear_kernel(int* __restrict__ bad, int count) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < count) bad[t] = 0;
}

// --------------------------------------------------------------- col_log_rms
// One lane per (column, chunk of row_step rows): the chunk's float64 sum of
// squares row after row, for many tensors in one launch. A second pass adds the
// chunk sums in order (and takes log(sqrt(acc / nrow) + 1e-12) when asked).
struct ColDev {
  const void* x;
  double* part;  // [nchunk, n] chunk sums
  double* out;   // [n]
  int64_t nrow;
  int n, x_f16, nchunk, col_groups;
};

template <bool F16>
__global__ __launch_bounds__(64) void col_chunk_kernel(const ColDev* __restrict__ tab,
                                                       int64_t row_step) {
  const ColDev& T = tab[blockIdx.y];
  const int chunk = (int)(blockIdx.x / T.col_groups);
  if (chunk >= T.nchunk) return;
  const int c = (int)(blockIdx.x - chunk * T.col_groups) * 64 + threadIdx.x;
  if (c >= T.n) return;
  const int64_t n = T.n;
  const int64_t r0 = (int64_t)chunk * row_step;
  const int64_t r1 = r0 + row_step < T.nrow ? r0 + row_step : T.nrow;
  double acc = 0.0;
  if constexpr (F16) {
    const GU16 x = (GU16)T.x;
    chain_rows<32, uint16_t>(r0, r1, [&](int64_t r) { return (x + r * n)[c]; },
                             [&](uint16_t h) {
                               const double v = (double)half_value(h);
                               acc = acc + v * v;
                             });
  } else {
    const GF32 x = (GF32)T.x;
    chain_rows<32, float>(r0, r1, [&](int64_t r) { return (x + r * n)[c]; },
                          [&](float f) {
                            const double v = (double)f;
                            acc = acc + v * v;
                          });
  }
  T.part[(int64_t)chunk * n + c] = acc;
}

__global__ void col_combine_kernel(const ColDev* __restrict__ tab, int log_rms) {
  const ColDev& T = tab[blockIdx.y];
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= T.n) return;
  double acc = 0.0;
  for (int k = 0; k < T.nchunk; ++k) acc = acc + T.part[(int64_t)k * T.n + c];
  T.out[c] = log_rms ? log(sqrt(acc / (double)T.nrow) + 1e-12) : acc;
}

// --------------------------------------------------------------- host side

static size_t a256(size_t v) { return (v + 255) & ~(size_t)255; }

struct ErrLayout {
  size_t xs, qwp, raw, recon, colerr, end;
};

static ErrLayout err_layout(const cp_err_tensor& t, size_t o) {
  KqGeom g;
  kq_geom(t.ttype, &g);
  const int64_t R = t.rows ? t.rows_used : t.nrow;
  ErrLayout L;
  L.xs = o; o += a256((size_t)R * t.n * 4);
  L.qwp = o; o += a256((size_t)t.n * 4);
  L.raw = o; o += t.ttype == CP_Q8_0 ? a256((size_t)R * (t.n / g.block_weights) * g.block_bytes) : 0;
  L.recon = o; o += a256((size_t)R * t.n * 4);
  L.colerr = o; o += a256((size_t)t.n * 8);
  L.end = o;
  return L;
}

static size_t err_tables_bytes(int count) {
  return a256((size_t)count * sizeof(ErrDev)) + a256((size_t)count * sizeof(int));
}

size_t err_ws_bytes(const cp_err_tensor* ts, int count) {
  size_t o = err_tables_bytes(count);
  for (int i = 0; i < count; ++i) o = err_layout(ts[i], o).end;
  return o;
}

constexpr int kErrPerStore = 31;
struct ErrBatch {
  ErrDev t[kErrPerStore];
};
static_assert(sizeof(ErrBatch) <= 4000, "kernel argument block");
__global__ void err_store_kernel(ErrBatch b, int cn, ErrDev* __restrict__ dst) {
  // the table leaves through vector stores, one 8-byte word per lane
  const int words = cn * (int)(sizeof(ErrDev) / 8);
  const uint64_t* s = reinterpret_cast<const uint64_t*>(b.t);
  uint64_t* d = reinterpret_cast<uint64_t*>(dst);
  for (int w = threadIdx.x; w < words; w += blockDim.x) d[w] = s[w];
}
static_assert(sizeof(ErrDev) % 8 == 0, "table rows are whole 8-byte words");

struct ErrGroup {
  int first, count, ttype;
  bool imat;
  int64_t max_w;  // weights of the largest gathered tensor
};

// Optional per-phase timing (cp_err_profile / cp_err_phase_ms): gather, encode,
// decode, column sums, total.
static thread_local PhaseClock g_err_clock;

template <int TT>
static void launch_err_encode(const ErrDev* tab, const ErrGroup& g, hipStream_t st) {
  int64_t blocks;
  if constexpr (TT == CP_Q8_0) {
    blocks = (g.max_w / 32 + 8 * kWavesPerBlock - 1) / (8 * kWavesPerBlock);
  } else {
    constexpr int S = 64 / Kq<TT>::G;
    blocks = ((g.max_w / 256 + S - 1) / S + kWavesPerBlock - 1) / kWavesPerBlock;
  }
  const dim3 grid((unsigned)blocks, (unsigned)g.count);
  if constexpr (TT == CP_Q8_0)  // no weighted path
    err_encode_kernel<TT, false><<<grid, 256, 0, st>>>(tab + g.first);
  else if (g.imat)
    err_encode_kernel<TT, true><<<grid, 256, 0, st>>>(tab + g.first);
  else
    err_encode_kernel<TT, false><<<grid, 256, 0, st>>>(tab + g.first);
}

static void launch_err_group(const ErrDev* tab, const ErrGroup& g, hipStream_t st) {
  switch (g.ttype) {
    case CP_Q8_0: launch_err_encode<CP_Q8_0>(tab, g, st); break;
    case CP_Q2_K: launch_err_encode<CP_Q2_K>(tab, g, st); break;
    case CP_Q3_K: launch_err_encode<CP_Q3_K>(tab, g, st); break;
    case CP_Q4_K: launch_err_encode<CP_Q4_K>(tab, g, st); break;
    case CP_Q5_K: launch_err_encode<CP_Q5_K>(tab, g, st); break;
    default: launch_err_encode<CP_Q6_K>(tab, g, st); break;
  }
}

int err_batch(const cp_err_tensor* ts, int count, void* ws, size_t ws_bytes, double* out,
              hipStream_t st) {
  if (!ts || count <= 0) return set_error(CP_ERR_ARG, "no tensors");
  if (count > 65535) return set_error(CP_ERR_ARG, "at most 65535 tensors per call (got %d)", count);
  if (!out) return set_error(CP_ERR_ARG, "null out");
  for (int i = 0; i < count; ++i) {
    const cp_err_tensor& t = ts[i];
    KqGeom g;
    if (!kq_geom(t.ttype, &g)) return set_error(CP_ERR_TTYPE, "tensor %d: unsupported type %d", i, t.ttype);
    const int64_t R = t.rows ? t.rows_used : t.nrow;
    if (t.nrow <= 0 || t.n <= 0 || t.n % g.block_weights || t.n > (1 << 24) || R <= 0 ||
        R > 0x7FFFFFFF || R * t.n / 4 > (int64_t)0x7FFFFFFF * 256)
      return set_error(CP_ERR_SHAPE, "tensor %d: bad shape [%lld, %lld] (rows used %lld)", i,
                       (long long)t.nrow, (long long)t.n, (long long)R);
    if (t.x_dtype != 0 && t.x_dtype != 1) return set_error(CP_ERR_ARG, "tensor %d: x_dtype must be 0 or 1", i);
    if (!t.x) return set_error(CP_ERR_ARG, "tensor %d: null x", i);
    if (!aligned(t.x, t.x_dtype ? 2 : 4) || (t.qw && !aligned(t.qw, 4)) ||
        (t.wvec && !aligned(t.wvec, 8)))
      return set_error(CP_ERR_ALIGN, "tensor %d: misaligned buffer", i);
  }
  if (!ws || ws_bytes < err_ws_bytes(ts, count))
    return set_error(CP_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, err_ws_bytes(ts, count));
  if (!aligned(ws, 256)) return set_error(CP_ERR_ALIGN, "workspace needs 256-byte alignment");

  char* base = (char*)ws;
  ErrDev* dtab = (ErrDev*)base;
  int* bad = (int*)(base + a256((size_t)count * sizeof(ErrDev)));
  std::vector<ErrDev> devs(count);
  size_t o = err_tables_bytes(count);
  int max_n = 0;
  for (int i = 0; i < count; ++i) {
    const cp_err_tensor& t = ts[i];
    const ErrLayout L = err_layout(t, o);
    o = L.end;
    const int R = (int)(t.rows ? t.rows_used : t.nrow);
    devs[i] = ErrDev{t.x, t.rows, t.perm, t.qw, t.wvec,
                     (float*)(base + L.xs), t.qw ? (float*)(base + L.qwp) : nullptr,
                     (uint8_t*)(base + L.raw), (float*)(base + L.recon), (double*)(base + L.colerr),
                     bad + i, t.nrow, R, (int)t.n, t.ttype, t.x_dtype, i, 0, 0};
    max_n = (int)t.n > max_n ? (int)t.n : max_n;
  }
  // table ordered by (type, importance) so each codec group is one run of rows
  std::vector<int> order(count);
  for (int i = 0; i < count; ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    if (ts[a].ttype != ts[b].ttype) return ts[a].ttype < ts[b].ttype;
    return (ts[a].qw != nullptr) < (ts[b].qw != nullptr);
  });
  std::vector<ErrDev> sorted(count);
  int64_t gather_blocks = 0;
  for (int k = 0; k < count; ++k) {
    sorted[k] = devs[order[k]];
    sorted[k].gfirst = (int)gather_blocks;
    gather_blocks += gather_tiles(sorted[k].R, sorted[k].n);
    if (gather_blocks > 0x7FFFFFFF) return set_error(CP_ERR_SHAPE, "too many weights in one call");
  }
  std::vector<int> by_rows(count);
  for (int k = 0; k < count; ++k) by_rows[k] = k;
  std::stable_sort(by_rows.begin(), by_rows.end(), [&](int a, int b) { return sorted[a].R > sorted[b].R; });
  for (int k = 0; k < count; ++k) sorted[k].by_rows = by_rows[k];
  std::vector<ErrGroup> groups;
  for (int k = 0; k < count; ++k) {
    const ErrDev& d = sorted[k];
    const bool imat = d.qw != nullptr;
    const int64_t w = (int64_t)d.R * d.n;
    if (groups.empty() || groups.back().ttype != d.ttype || groups.back().imat != imat)
      groups.push_back(ErrGroup{k, 0, d.ttype, imat, 0});
    ErrGroup& g = groups.back();
    ++g.count;
    g.max_w = w > g.max_w ? w : g.max_w;
  }
  for (int c0 = 0; c0 < count; c0 += kErrPerStore) {
    const int cn = count - c0 < kErrPerStore ? count - c0 : kErrPerStore;
    ErrBatch b;
    for (int i = 0; i < cn; ++i) b.t[i] = sorted[c0 + i];
    err_store_kernel<<<1, 256, 0, st>>>(b, cn, dtab + c0);
  }
  CP_PHASE_MARK(g_err_clock, -1);
  err_clear_kernel<<<(count + 255) / 256, 256, 0, st>>>(bad, count);
  err_gather_kernel<<<(unsigned)gather_blocks, 256, 0, st>>>(dtab, count);
  CP_LAUNCHED("objective gather");
  CP_PHASE_MARK(g_err_clock, 0);
  for (const ErrGroup& g : groups) launch_err_group(dtab, g, st);
  CP_LAUNCHED("objective encode");
  CP_PHASE_MARK(g_err_clock, 1);
  for (const ErrGroup& g : groups)
    if (g.ttype == CP_Q8_0)
      err_decode_q8_kernel<<<dim3((unsigned)((g.max_w / 4 + 255) / 256), (unsigned)g.count), 256, 0, st>>>(
          dtab + g.first);
  CP_LAUNCHED("objective decode");
  CP_PHASE_MARK(g_err_clock, 2);
  err_colsum_kernel<<<dim3((unsigned)((max_n + kSumCols - 1) / kSumCols), (unsigned)count), 64 * kSumWaves, 0, st>>>(
      dtab);
  CP_LAUNCHED("objective column sums");
  CP_PHASE_MARK(g_err_clock, 3);
  err_final_kernel<<<count, 256, 0, st>>>(dtab, out);
  CP_LAUNCHED("objective total");
  CP_PHASE_MARK(g_err_clock, 4);
  return CP_OK;
}

constexpr int kColPerStore = 64;
struct ColBatch {
  ColDev t[kColPerStore];
};
static_assert(sizeof(ColBatch) <= 4000, "kernel argument block");
static_assert(sizeof(ColDev) % 8 == 0, "table rows are whole 8-byte words");
__global__ void col_store_kernel(ColBatch b, int cn, ColDev* __restrict__ dst) {
  const int words = cn * (int)(sizeof(ColDev) / 8);
  const uint64_t* s = reinterpret_cast<const uint64_t*>(b.t);
  uint64_t* d = reinterpret_cast<uint64_t*>(dst);
  for (int w = threadIdx.x; w < words; w += blockDim.x) d[w] = s[w];
}

size_t col_ws_bytes(const cp_col_tensor* ts, int count, int64_t row_step) {
  size_t o = a256((size_t)count * sizeof(ColDev));
  for (int i = 0; i < count; ++i)
    o += a256((size_t)((ts[i].nrow + row_step - 1) / row_step) * (size_t)ts[i].n * 8);
  return o;
}

int col_sums_batch(const cp_col_tensor* ts, int count, int64_t row_step, int log_rms, void* ws,
                   size_t ws_bytes, hipStream_t st) {
  if (!ts || count <= 0) return set_error(CP_ERR_ARG, "no tensors");
  if (count > 65535) return set_error(CP_ERR_ARG, "at most 65535 tensors per call (got %d)", count);
  if (row_step <= 0) return set_error(CP_ERR_SHAPE, "row_step %lld", (long long)row_step);
  int64_t max_blocks = 0;
  int max_n = 0;
  for (int i = 0; i < count; ++i) {
    const cp_col_tensor& t = ts[i];
    if (!t.x || !t.out) return set_error(CP_ERR_ARG, "tensor %d: null x/out", i);
    if (t.x_dtype != 0 && t.x_dtype != 1) return set_error(CP_ERR_ARG, "tensor %d: x_dtype must be 0 or 1", i);
    if (t.nrow <= 0 || t.n <= 0 || t.n > (1 << 24))
      return set_error(CP_ERR_SHAPE, "tensor %d: x is [%lld, %lld]", i, (long long)t.nrow, (long long)t.n);
    const int64_t nchunk = (t.nrow + row_step - 1) / row_step;
    const int64_t blocks = nchunk * ((t.n + 63) / 64);
    if (nchunk > 0x7FFFFFFF || blocks > 0x7FFFFFFF) return set_error(CP_ERR_SHAPE, "tensor %d: too many row chunks", i);
    if (!aligned(t.x, t.x_dtype ? 2 : 4) || !aligned(t.out, 8))
      return set_error(CP_ERR_ALIGN, "tensor %d: misaligned buffer", i);
    max_blocks = blocks > max_blocks ? blocks : max_blocks;
    max_n = (int)t.n > max_n ? (int)t.n : max_n;
  }
  if (!ws || ws_bytes < col_ws_bytes(ts, count, row_step))
    return set_error(CP_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, col_ws_bytes(ts, count, row_step));
  if (!aligned(ws, 256)) return set_error(CP_ERR_ALIGN, "workspace needs 256-byte alignment");
  char* base = (char*)ws;
  ColDev* dtab = (ColDev*)base;
  size_t o = a256((size_t)count * sizeof(ColDev));
  std::vector<ColDev> devs(count);
  bool any16 = false, any32 = false;
  for (int i = 0; i < count; ++i) {
    const cp_col_tensor& t = ts[i];
    const int nchunk = (int)((t.nrow + row_step - 1) / row_step);
    devs[i] = ColDev{t.x, (double*)(base + o), t.out, t.nrow, (int)t.n, t.x_dtype, nchunk,
                     (int)((t.n + 63) / 64)};
    o += a256((size_t)nchunk * (size_t)t.n * 8);
    (t.x_dtype ? any16 : any32) = true;
  }
  // one table per input dtype: f16 rows first, then f32
  std::stable_partition(devs.begin(), devs.end(), [](const ColDev& d) { return d.x_f16 != 0; });
  int n16 = 0;
  for (const ColDev& d : devs) n16 += d.x_f16 != 0;
  for (int c0 = 0; c0 < count; c0 += kColPerStore) {
    const int cn = count - c0 < kColPerStore ? count - c0 : kColPerStore;
    ColBatch b;
    for (int i = 0; i < cn; ++i) b.t[i] = devs[c0 + i];
    col_store_kernel<<<1, 256, 0, st>>>(b, cn, dtab + c0);
  }
  if (any16)
    col_chunk_kernel<true><<<dim3((unsigned)max_blocks, (unsigned)n16), 64, 0, st>>>(dtab, row_step);
  if (any32)
    col_chunk_kernel<false><<<dim3((unsigned)max_blocks, (unsigned)(count - n16)), 64, 0, st>>>(
        dtab + n16, row_step);
  col_combine_kernel<<<dim3((unsigned)((max_n + 255) / 256), (unsigned)count), 256, 0, st>>>(dtab, log_rms);
  CP_LAUNCHED("column sums");
  return CP_OK;
}

}  // namespace cp

extern "C" {

size_t cp_tensor_err_ws_bytes(const cp_err_tensor* tensors, int count) {
  if (!tensors || count <= 0) return 0;
  for (int i = 0; i < count; ++i) {
    cp::KqGeom g;
    if (!cp::kq_geom(tensors[i].ttype, &g)) return 0;
  }
  return cp::err_ws_bytes(tensors, count);
}

int cp_tensor_err_batch(const cp_err_tensor* tensors, int count, void* ws, size_t ws_bytes,
                        double* out, void* stream) {
  cp::clear_error();
  return cp::err_batch(tensors, count, ws, ws_bytes, out, (hipStream_t)stream);
}

void cp_err_profile(int enable) { cp::g_err_clock.on = enable != 0; }

int cp_err_phase_ms(float* out, int nphase) {
  cp::clear_error();
  if (!out || nphase <= 0) return cp::set_error(CP_ERR_ARG, "bad phase buffer");
  hipError_t r = cp::g_err_clock.read(out, nphase);
  if (r != hipSuccess) return cp::hip_fail(r, "phase events");
  return nphase < 5 ? nphase : 5;
}

size_t cp_col_sums_ws_bytes(int64_t nrow, int64_t n, int64_t row_step) {
  if (nrow <= 0 || n <= 0 || row_step <= 0) return 0;
  const cp_col_tensor t{nullptr, 0, nrow, n, nullptr};
  return cp::col_ws_bytes(&t, 1, row_step);
}

int cp_col_sq_sums(const void* x, int x_dtype, int64_t nrow, int64_t n, int64_t row_step,
                   double* acc, void* ws, size_t ws_bytes, void* stream) {
  cp::clear_error();
  const cp_col_tensor t{x, x_dtype, nrow, n, acc};
  return cp::col_sums_batch(&t, 1, row_step, 0, ws, ws_bytes, (hipStream_t)stream);
}

int cp_col_log_rms(const void* x, int x_dtype, int64_t nrow, int64_t n, int64_t row_step,
                   double* out, void* ws, size_t ws_bytes, void* stream) {
  cp::clear_error();
  const cp_col_tensor t{x, x_dtype, nrow, n, out};
  return cp::col_sums_batch(&t, 1, row_step, 1, ws, ws_bytes, (hipStream_t)stream);
}

size_t cp_col_sums_batch_ws_bytes(const cp_col_tensor* tensors, int count, int64_t row_step) {
  if (!tensors || count <= 0 || row_step <= 0) return 0;
  return cp::col_ws_bytes(tensors, count, row_step);
}

int cp_col_sq_sums_batch(const cp_col_tensor* tensors, int count, int64_t row_step, int log_rms,
                         void* ws, size_t ws_bytes, void* stream) {
  cp::clear_error();
  return cp::col_sums_batch(tensors, count, row_step, log_rms != 0, ws, ws_bytes,
                            (hipStream_t)stream);
}

}  // extern "C"
