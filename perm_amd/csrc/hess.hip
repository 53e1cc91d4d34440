// Input-Hessian accumulation H += X^T X on gfx950 MFMA (coldpress/hessians.py:137-154).
//
// X is [N, d] row-major activations (bf16 or f32), H is [d, d] float32 and is
// accumulated in place (beta = 1), so hook batches can stream in. Split-K over
// rows of X: N is 65536-131072 while d is 1024-14336, so the row dimension is
// what fills 256 CUs. The result does not depend on scheduling: with one row
// split a workgroup adds its finished tile into H itself (one writer per
// element); with several, each split stores its tile into a workspace slot of
// its own and one reduction pass adds the splits' tiles to H in split order
// (H + ((p0 + p1) + p2 ...), the f32 path in groups of 16 splits). The same X
// therefore gives the same H bit for bit, run after run.
//
//  bf16: lower-triangle 256 x 256 tiles on v_mfma_f32_32x32x16_bf16, operands
//        read transposed from LDS (hess_bf16_tri_kernel), then a pass that
//        reduces the splits and mirrors the lower triangle into the upper one;
//  f32:  lower-triangle 128 x 128 tiles on v_mfma_f32_32x32x2f32, which takes one row t
//        per lane, so the [t][i] panel is used as loaded.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <type_traits>

#include "cp_host.h"

namespace cp {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int HT = 128;  // f32 kernel: H tile edge
constexpr int KT = 32;   // f32 kernel: rows of X per step
constexpr int kFlush = 8;  // f32 and few-rows kernels: stages summed in one chain, 256 rows

// Row of the 32x32 MFMA result held by register v of lane l (column = l % 32).
__device__ __forceinline__ int mfma32_row(int v, int l) { return 8 * (v >> 2) + 4 * (l >> 5) + (v & 3); }

// ---------------------------------------------------------------- bf16 input
// Lower-triangle tiles of 256 x 256 (H is symmetric; hess_tri_reduce_kernel copies
// the lower triangle into the upper one afterwards), split-K over rows of X.
// A workgroup is 4 waves, each owning a 128 x 128 block as 4 x 4 MFMA 32x32
// tiles (256 float32 accumulators): the largest block a wave can hold, because
// the LDS traffic per MFMA, not the MFMAs, bounds this kernel.
//
// Rows of X are staged 32 at a time: both 32 x 256 panels (columns of the i-
// and j-tile; one panel on a diagonal tile) are fetched into registers two
// stages ahead of use, stored into a 4-slot LDS ring in X's own [t][c] layout,
// and read as MFMA operands with ds_read_b64_tr_b16, which returns 4
// consecutive rows t of one column per lane: v_mfma_f32_32x32x16_bf16 takes 8
// consecutive t per lane for both operands. Panel rows are padded from 512 to
// 576 bytes so the four rows of one transposed read fall 64 bytes apart in
// bank space (conflict-free), and every LDS address in the loop is a per-lane
// base plus an immediate: with one wave per SIMD, address arithmetic between
// the MFMAs is not hidden by anything.
//
// Work items (row split, tile) are ordered split-major and handed out
// XCD-contiguously: the hardware places workgroup w on XCD w % 8, so
// item = (w % 8) * per + w / 8 keeps the workgroups of one XCD on the same
// rows of X (shared in its L2).
constexpr int BT = 256;             // H tile edge
constexpr int KS = 32;              // rows of X per stage
constexpr int PROW = BT * 2 + 64;   // bytes per padded panel row
constexpr int PANEL = KS * PROW;    // 18 KB
constexpr int HNT = 256;            // threads per workgroup
constexpr int NSLOT = 4;            // LDS ring (stage s in slot s % 4)
constexpr int CPT = 2048 / HNT;     // 16-byte chunks per thread per stage (two panels)

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef short v8i16 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4i16* lds_v4p;

// Global side of the staging: raw buffer loads over the workgroup's row split
// (base X + r0 * d, num_records = its byte length). A load whose offset is at or
// past num_records returns zeros, so rows past the split's end and 8-column
// chunks past d (given an offset past the end) need no branch, and the loop
// has no control flow between loads: the compiler then waits only for the
// load a store needs, not for every load in flight.
//
// Chunk q of a stage (16 bytes per thread, q < 4 on the i-panel, q >= 4 on the
// j-panel): row (tid / 32) + 8 (q % 4), column chunk tid % 32.
constexpr uint32_t kOob = 0x80000000u;  // past any num_records the host allows

template <int NQ>
struct Stager {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[NQ];  // chunk q's byte offset at stage 0 (kOob when outside d)
  uint32_t sbytes;   // bytes per stage (KS rows)
};

template <int NQ>
__device__ __forceinline__ Stager<NQ> make_stager(const uint16_t* X, int64_t r0, int64_t nrows,
                                                  int d, int i0, int j0, int tid) {
  Stager<NQ> s;
  const uint32_t rowb = 2u * (uint32_t)d;
  s.rs = __builtin_amdgcn_make_buffer_rsrc((void*)(X + r0 * d), 0, (int)(nrows * rowb), 0x00020000);
  const int c8 = 8 * (tid & 31);
  const uint32_t row0 = (uint32_t)(tid >> 5) * rowb;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int c = (q >= 4 ? j0 : i0) + c8;  // d % 8 == 0: the 8 columns are all in or all out
    s.off[q] = c < d ? row0 + (uint32_t)(8 * (q & 3)) * rowb + 2u * (uint32_t)c : kOob;
  }
  s.sbytes = (uint32_t)KS * rowb;
  return s;
}

template <int NQ>
__device__ __forceinline__ void stage_load_one(const Stager<NQ>& st, int s, uint4 (&g)[CPT], int q) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(st.rs, (int)(st.off[q] + (uint32_t)s * st.sbytes),
                                                       0, 0);
  g[q] = make_uint4(v[0], v[1], v[2], v[3]);
}

// LDS byte offset of chunk q within a slot, relative to the thread's store base
// (tid / 32) * PROW + 16 * (tid % 32)
__device__ __forceinline__ constexpr int chunk_ofs(int q) { return (q >> 2) * PANEL + 8 * (q & 3) * PROW; }

struct Operands {
  bf16x8 a[4], b[4];
};

// Piece i (0..15) of one half of a stage's operands: the lo or hi four rows of
// one operand, in the order a0, b0, b1, b2, b3, a1, a2, a3 -- the order the
// MFMAs (x, y) = (i / 4, i % 4) first use them. ra / rb: this lane's read base
// in the A / B panel of the slot; the rest of the address is an immediate.
// Lane l gets column col + l % 32, rows 8 * (l / 32) + 0..7 of the half.
__device__ __forceinline__ void read_piece(const char* ra, const char* rb, int half, int i,
                                           Operands& f) {
  const int op = i >> 1, hi = i & 1;
  const bool isb = op >= 1 && op <= 4;
  const int idx = isb ? op - 1 : (op == 0 ? 0 : op - 4);
  const char* p = (isb ? rb : ra) + (16 * half + 4 * hi) * PROW + 64 * idx;
  const v4i16 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4p)p);
  const v8i16 w = __builtin_shufflevector(v, v, 0, 1, 2, 3, 0, 1, 2, 3);
  v8i16 cur = __builtin_bit_cast(v8i16, isb ? f.b[idx] : f.a[idx]);
  if (hi)
    cur = __builtin_shufflevector(cur, w, 0, 1, 2, 3, 12, 13, 14, 15);
  else
    cur = __builtin_shufflevector(w, cur, 0, 1, 2, 3, 12, 13, 14, 15);
  if (isb)
    f.b[idx] = __builtin_bit_cast(bf16x8, cur);
  else
    f.a[idx] = __builtin_bit_cast(bf16x8, cur);
}

// STAGE_ONLY: the wave stages its share of the panels and meets every barrier but
// reads no operands and issues no MFMAs -- the wave of a diagonal tile whose 128 x 128
// block lies wholly above the diagonal, whose sums would be discarded.
template <bool DIAG, bool STAGE_ONLY = false>
__device__ __forceinline__ void tile_rows(const uint16_t* X, int64_t r0, int64_t r1, int d, int i0,
                                          int j0, char* lds, f32x16 (&acc)[4][4]) {
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int wm = (w >> 1) * 128, wn = (w & 1) * 128;
  constexpr int NQ = DIAG ? CPT / 2 : CPT;  // 16-byte chunks per thread per stage
  constexpr int SLOT = DIAG ? PANEL : 2 * PANEL;
  // stages rounded up to a multiple of 4 (the unrolled loop body): stages past
  // the split's end load as zeros and add nothing
  const int ns = (int)((r1 - r0 + 4 * KS - 1) / (4 * KS)) * 4;
  const Stager<NQ> st = make_stager<NQ>(X, r0, r1 - r0, d, i0, j0, tid);
  // per-lane LDS bases: transposed reads (row 8 * (g / 2) + c / 4, column
  // 16 * (g % 2) + 4 * (c % 4) of the wave's block, g = l / 16, c = l % 16) and
  // stores (row tid / 32, 16-byte chunk tid % 32)
  const int g4 = l >> 4, c4 = l & 15;
  const int rlane = (8 * (g4 >> 1) + (c4 >> 2)) * PROW + 2 * (16 * (g4 & 1) + 4 * (c4 & 3));
  char* const ra0 = lds + rlane + 2 * wm;
  char* const rb0 = lds + rlane + 2 * wn + (DIAG ? 0 : PANEL);
  char* const wr0 = lds + (tid >> 5) * PROW + 16 * (tid & 31);
  uint4 g0[CPT], g1[CPT];
#pragma unroll
  for (int q = 0; q < NQ; ++q) stage_load_one(st, 0, g0, q);
#pragma unroll
  for (int q = 0; q < NQ; ++q) stage_load_one(st, 1, g1, q);
#pragma unroll
  for (int q = 0; q < NQ; ++q) *reinterpret_cast<uint4*>(wr0 + chunk_ofs(q)) = g0[q];
#pragma unroll
  for (int q = 0; q < NQ; ++q) *reinterpret_cast<uint4*>(wr0 + SLOT + chunk_ofs(q)) = g1[q];
#pragma unroll
  for (int q = 0; q < NQ; ++q) stage_load_one(st, 2, g0, q);
#pragma unroll
  for (int q = 0; q < NQ; ++q) stage_load_one(st, 3, g1, q);
  __syncthreads();
  Operands f0, f1;
  if constexpr (!STAGE_ONLY) {
#pragma unroll
    for (int i = 0; i < 16; ++i) read_piece(ra0, rb0, 0, i, f0);
  }
  // Stage s (K = s % 4): store stage s + 2 (fetched two stages ago) into slot
  // K + 2, fetch stage s + 4 into the same registers, and multiply stage s
  // while reading the next operands (its second half, then the first half of
  // stage s + 1). Past the end the same steps run on zero stages and slots no
  // stage reads, so the body has no branches.
  //
  // With one wave per SIMD nothing hides a wave's own LDS waits, so the step
  // is issued as one interleaved stream, pinned in place by scheduling
  // barriers: each of the 32 MFMAs is followed by one of the 32 transposed
  // reads of the next operands, and the stores are spread over the step, each
  // chunk's store followed by the load of the same chunk four stages ahead
  // (so every store waits only for the oldest load in flight), keeping the
  // LDS busy while the MFMAs run instead of the two taking turns.
  auto step = [&](auto kc, int s, uint4 (&g)[CPT]) {
    constexpr int K = decltype(kc)::value;
    __syncthreads();
    const char* ra = ra0 + K * SLOT;
    const char* rb = rb0 + K * SLOT;
    const char* na = ra0 + ((K + 1) % NSLOT) * SLOT;
    const char* nb = rb0 + ((K + 1) % NSLOT) * SLOT;
    char* dst = wr0 + ((K + 2) % NSLOT) * SLOT;
    constexpr int SE = 32 / NQ;  // MFMAs per store
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if constexpr (!STAGE_ONLY) {
        acc[i >> 2][i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f0.a[i >> 2], f0.b[i & 3],
                                                                     acc[i >> 2][i & 3], 0, 0, 0);
        read_piece(ra, rb, 1, i, f1);
      }
      if (i % SE == 0) {
        *reinterpret_cast<uint4*>(dst + chunk_ofs(i / SE)) = g[i / SE];
        stage_load_one(st, s + 4, g, i / SE);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if constexpr (!STAGE_ONLY) {
        acc[i >> 2][i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f1.a[i >> 2], f1.b[i & 3],
                                                                     acc[i >> 2][i & 3], 0, 0, 0);
        read_piece(na, nb, 0, i, f0);
      }
      if (i % SE == 0) {
        *reinterpret_cast<uint4*>(dst + chunk_ofs(NQ / 2 + i / SE)) = g[NQ / 2 + i / SE];
        stage_load_one(st, s + 4, g, NQ / 2 + i / SE);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0; s < ns; s += 4) {
    step(std::integral_constant<int, 0>(), s, g0);
    step(std::integral_constant<int, 1>(), s + 1, g1);
    step(std::integral_constant<int, 2>(), s + 2, g0);
    step(std::integral_constant<int, 3>(), s + 3, g1);
  }
}

// Up to kHessJobs Hessians of one shape per launch, by value in the kernel arguments.
constexpr int kHessJobs = 224;
struct HessJobs {
  const uint16_t* X[kHessJobs];
  float* H[kHessJobs];
};
static_assert(sizeof(HessJobs) <= 4000, "kernel argument block");

// part == nullptr (one row split): the workgroup adds its tile into H's lower
// triangle. Otherwise it stores the whole 256 x 256 tile, row-major, into slot
// (job, split, tile) of part, for hess_tri_reduce_kernel.
__global__ __launch_bounds__(HNT) void hess_bf16_tri_kernel(const HessJobs jobs, int njobs,
                                                            int64_t N, int d, int ntiles, int splits,
                                                            int64_t rows_per_split,
                                                            float* __restrict__ part) {
  __shared__ __align__(16) char lds[NSLOT * 2 * PANEL];
  // items run job by job, then split by split: the XCD-contiguous hand-out keeps one
  // XCD on the same rows of one X
  const int per_job = ntiles * splits;
  const int total = per_job * njobs;
  const int per = (total + 7) / 8;
  const int item = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (item >= total) return;
  const int job = item / per_job, rem = item - job * per_job;
  const int split = rem / ntiles, tile = rem - split * ntiles;
  const uint16_t* __restrict__ X = jobs.X[job];
  float* __restrict__ H = jobs.H[job];
  int ti = (int)((sqrtf(8.0f * (float)tile + 1.0f) - 1.0f) * 0.5f);
  while (ti * (ti + 1) / 2 > tile) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= tile) ++ti;
  const int tj = tile - ti * (ti + 1) / 2;
  const int i0 = ti * BT, j0 = tj * BT;
  const int64_t r0 = (int64_t)split * rows_per_split;
  const int64_t r1 = min(N, r0 + rows_per_split);
  if (r0 >= r1) return;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int wm = (w >> 1) * 128, wn = (w & 1) * 128;
  f32x16 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
  if (ti != tj)
    tile_rows<false>(X, r0, r1, d, i0, j0, lds, acc);
  else if (wn > wm)  // wave 1: its block is above the diagonal
    tile_rows<true, true>(X, r0, r1, d, i0, j0, lds, acc);
  else
    tile_rows<true>(X, r0, r1, d, i0, j0, lds, acc);
  // lane l holds, for register v of tile (x, y), row wm + 32x + mfma32_row(v, l)
  // and column wn + 32y + l % 32 of the workgroup tile
  if (part) {
    // every register stored (zeros where the wave skipped its block; rows and
    // columns past d hold sums of zero-filled loads): the reduction reads only
    // the lower-triangle entries inside d
    float* Pb = part + ((int64_t)(job * splits + split) * ntiles + tile) * (BT * BT) +
                (wm + 4 * (l >> 5)) * BT + wn + (l & 31);
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int v = 0; v < 16; ++v) Pb[(x * 32 + 8 * (v >> 2) + (v & 3)) * BT + y * 32] = acc[x][y][v];
    return;
  }
  float* Hb = H + (int64_t)(i0 + wm + 4 * (l >> 5)) * d + (j0 + wn + (l & 31));
  const bool full = ti != tj && i0 + BT <= d;  // interior tile strictly below the diagonal
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int i = i0 + wm + x * 32 + mfma32_row(v, l);
        const int j = j0 + wn + y * 32 + (l & 31);
        float* p = Hb + (int64_t)(x * 32 + 8 * (v >> 2) + (v & 3)) * d + y * 32;
        if (full || (i < d && j <= i)) *p = *p + acc[x][y][v];
      }
}

// Finishes a bf16 accumulation over the 64 x 64 blocks (bi, bj), bj <= bi, of the lower
// triangle, one workgroup each (blockIdx.x: the job's lower blocks in row order,
// blockIdx.y: the job). With part, each entry (i, j) becomes H + (p_0 + p_1 + ... +
// p_{splits-1}), the row splits' tiles summed in split order; then the block is written
// to the mirror position (j, i) as well, through LDS, so H leaves symmetric. Thread t
// covers 4 consecutive columns (16-byte accesses; d % 4 == 0, so a 4-column group is
// wholly inside or outside d) of rows t / 16 + 16 q. A diagonal block's entries above
// the diagonal are first written with the sums of their own (meaningless) positions and
// then overwritten by the mirror after the barrier, so its float4 stores need no mask;
// the mirror stores mask the entries on and below the diagonal. H's upper triangle is
// never used.
__global__ __launch_bounds__(256) void hess_tri_reduce_kernel(const HessJobs jobs, int d, int ntiles,
                                                              int splits,
                                                              const float* __restrict__ part) {
  float* __restrict__ H = jobs.H[blockIdx.y];
  __shared__ float tl[64][65];
  int bi = (int)((sqrtf(8.0f * (float)blockIdx.x + 1.0f) - 1.0f) * 0.5f);
  while (bi * (bi + 1) / 2 > (int)blockIdx.x) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= (int)blockIdx.x) ++bi;
  const int bj = (int)blockIdx.x - bi * (bi + 1) / 2;
  const int cg = threadIdx.x & 15, rt = threadIdx.x >> 4;
  const int j = bj * 64 + 4 * cg;
  const int tj = j / BT;
  const int64_t slot = (int64_t)ntiles * (BT * BT);  // floats between one split's tiles
  const float* pj = part ? part + (int64_t)blockIdx.y * splits * slot : nullptr;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = rt + 16 * q, i = bi * 64 + r;
    if (i >= d || j >= d) continue;
    float4 h = *reinterpret_cast<const float4*>(H + (int64_t)i * d + j);
    if (pj) {
      const int ti = i / BT;
      const float* p = pj + (int64_t)(ti * (ti + 1) / 2 + tj) * (BT * BT) + (i % BT) * BT + (j % BT);
      float4 s = *reinterpret_cast<const float4*>(p);
      for (int k = 1; k < splits; ++k) {
        const float4 v = *reinterpret_cast<const float4*>(p + k * slot);
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
      }
      h.x += s.x;
      h.y += s.y;
      h.z += s.z;
      h.w += s.w;
      *reinterpret_cast<float4*>(H + (int64_t)i * d + j) = h;
    }
    tl[r][4 * cg] = h.x;
    tl[r][4 * cg + 1] = h.y;
    tl[r][4 * cg + 2] = h.z;
    tl[r][4 * cg + 3] = h.w;
  }
  __syncthreads();
  // upper block: rows bj, columns bi; entry (bj*64 + r, bi*64 + c) = lower (bi*64 + c, bj*64 + r)
  const int jj = bi * 64 + 4 * cg;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = rt + 16 * q, i = bj * 64 + r;
    if (i >= d || jj >= d) continue;
    float* dst = H + (int64_t)i * d + jj;
    const float4 v = make_float4(tl[4 * cg][r], tl[4 * cg + 1][r], tl[4 * cg + 2][r], tl[4 * cg + 3][r]);
    if (bi != bj || jj > i) {
      *reinterpret_cast<float4*>(dst) = v;
    } else {
      if (jj + 1 > i) dst[1] = v.y;
      if (jj + 2 > i) dst[2] = v.z;
      if (jj + 3 > i) dst[3] = v.w;
    }
  }
}

// ---------------------------------------------------------------- bf16 input, few rows
// One hook call (a sequence of a few thousand rows, one H) gives the 256 x 256 tiles too
// little: [2048, 1024] is 10 tiles x 8 row splits, so 80 workgroups fill a pipeline for eight
// stages and store 21 MB of partial tiles that a second launch sums. Here a workgroup takes
// one 64 x 64 tile of the lower triangle over all rows: its eight waves take a row range each,
// stage their rows through LDS of their own (no barrier; rows of 192 bytes keep the
// transposed reads conflict-free), and their sums are added in wave order in LDS. At d = 1024 the
// kernel takes about 8 us whatever the rows (launch, the waves' sums through LDS, both triangles
// of H: [300, 1024] 8.1) and 0.86 per 256 rows ([2048, 1024] 15.0, [8192, 1024] 35.5), not for
// load latency (four stages in flight instead of two: 15.2 -> 16.0): [2048, 1024] 31.2 -> 15.5 us
// a call.
constexpr int SW = 8;                    // waves
constexpr int SROW = 64 * 2 + 64;        // bytes per padded panel row
constexpr int SPANEL = KS * SROW;        // 6 KB
constexpr int SPITCH = 64 + 1;           // floats per row of a wave's sums
static_assert(kFlush % 2 == 0, "the loop takes two stages at a time");

__global__ __launch_bounds__(64 * SW, 2) void hess_bf16_small_kernel(const HessJobs jobs, int64_t N, int d) {
  union Lds {
    char stage[SW][2 * SPANEL];
    float sum[SW][64][SPITCH];
  };
  __shared__ __align__(16) Lds lds;
  const uint16_t* __restrict__ X = jobs.X[blockIdx.y];
  float* __restrict__ H = jobs.H[blockIdx.y];
  int ti = (int)((sqrtf(8.0f * (float)blockIdx.x + 1.0f) - 1.0f) * 0.5f);
  while (ti * (ti + 1) / 2 > (int)blockIdx.x) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= (int)blockIdx.x) ++ti;
  const int tj = (int)blockIdx.x - ti * (ti + 1) / 2;
  const int i0 = 64 * ti, j0 = 64 * tj;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), l = (int)threadIdx.x & 63;
  // this wave's rows: whole stages, as even as they come
  const int64_t stages_all = (N + KS - 1) / KS, per = (stages_all + SW - 1) / SW;
  const int64_t r0 = min(N, wv * per * KS), r1 = min(N, (wv + 1) * per * KS);
  const int ns = (int)((r1 - r0 + KS - 1) / KS);
  // sums of kFlush stages, and their running total: one chain over all N / 8 rows is further from
  // the float64 sums than the 256 x 256 tiles' shorter splits ([12288, 1024] of unit normals
  // 1.22e-7 against 9.6e-8, 5.9e-8 with the totals; 51.3 us either way)
  f32x16 acc[2][2], tot[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[x][y][v] = tot[x][y][v] = 0.0f;
  if (ns > 0) {
    const uint32_t rowb = 2u * (uint32_t)d;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)(X + r0 * d), 0, (int)((r1 - r0) * rowb), 0x00020000);
    // chunk q < 4 of panel p: row l / 8 + 8 q, columns 8 (l % 8) .. + 7 (d % 8 == 0: all in or all out)
    const uint32_t row = (uint32_t)(l >> 3) * rowb;
    const int ci = i0 + 8 * (l & 7), cj = j0 + 8 * (l & 7);
    const uint32_t oi = ci < d ? row + 2u * (uint32_t)ci : kOob, oj = cj < d ? row + 2u * (uint32_t)cj : kOob;
    const auto fetch = [&](int s, uint4 (&g)[8]) {
      const uint32_t so = (uint32_t)s * KS * rowb;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(
            rs, (int)((q < 4 ? oi : oj) + so + (uint32_t)(8 * (q & 3)) * rowb), 0, 0);
        g[q] = make_uint4(v[0], v[1], v[2], v[3]);
      }
    };
    char* const base = lds.stage[wv];
    char* const wr = base + (l >> 3) * SROW + 16 * (l & 7);
    const int g4 = l >> 4, c4 = l & 15;
    const char* const rd = base + (8 * (g4 >> 1) + (c4 >> 2)) * SROW + 2 * (16 * (g4 & 1) + 4 * (c4 & 3));
    // lane l: column 32 x + l % 32 of the panel, rows 16 half + 8 (l / 32) + 0 .. 7
    const auto operand = [&](int panel, int half, int x) {
      const char* p = rd + panel * SPANEL + 16 * half * SROW + 64 * x;
      const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4p)p);
      const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4p)(p + 4 * SROW));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // one stage: into this wave's LDS, the stage after next into the registers, and its products
    // (the LDS serves a wave's accesses in order, so stage s + 1 overwrites what s has read)
    const auto stage = [&](int s, uint4 (&g)[8]) {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        *reinterpret_cast<uint4*>(wr + (q >> 2) * SPANEL + 8 * (q & 3) * SROW) = g[q];
      if (s + 2 < ns) fetch(s + 2, g);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        bf16x8 a[2], b[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          a[x] = operand(0, half, x);
          b[x] = operand(1, half, x);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[x], b[y], acc[x][y], 0, 0, 0);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    uint4 g0[8], g1[8];
    fetch(0, g0);
    if (ns > 1) fetch(1, g1);
    for (int s = 0; s < ns; s += 2) {
      stage(s, g0);
      if (s + 1 < ns) stage(s + 1, g1);
      if (s % kFlush == kFlush - 2 && s + 2 < ns) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            tot[x][y] += acc[x][y];
            acc[x][y] = 0.0f;
          }
      }
    }
  }
  __syncthreads();  // every wave is done with its staging area
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v) lds.sum[wv][32 * x + mfma32_row(v, l)][32 * y + (l & 31)] = tot[x][y][v] + acc[x][y][v];
  __syncthreads();
  // entry (r, c) of the tile: H plus the waves' sums in order, at (i, j) and, as H leaves
  // symmetric, at (j, i); a diagonal tile's entries above the diagonal are its mirror's
  float v[8];
  const int c = l;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = wv + SW * q;
    v[q] = lds.sum[0][r][c];
#pragma unroll
    for (int k = 1; k < SW; ++k) v[q] += lds.sum[k][r][c];
    const int i = i0 + r, j = j0 + c;
    if (i < d && j <= i) v[q] += H[(int64_t)i * d + j];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = wv + SW * q, i = i0 + r, j = j0 + c;
    lds.sum[0][r][c] = v[q];
    if (i < d && j <= i) H[(int64_t)i * d + j] = v[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = wv + SW * q, i = j0 + r, j = i0 + c;  // (i, j) above the diagonal
    if (j < d && i < j) H[(int64_t)i * d + j] = lds.sum[0][c][r];
  }
}

// ---------------------------------------------------------------- f32 input
// Lower-triangle 128 x 128 tiles on v_mfma_f32_32x32x2f32, split-K over rows of X; the
// products of the two triangles are equal bit for bit (the factors commute), so each tile
// serves both. Four waves of 64 x 64. Bound by the f32 matrix rate (64 cycles per 4096
// flops): rows come 32 at a time through raw buffer loads one stage ahead (rows past the
// split and columns past d read zeros, so any d takes the same loop) into a double-buffered
// LDS panel pair, one barrier per stage, two workgroups per CU. Full square tiles loaded with
// bounds branches and no stage in flight ran [8192, 1024] in 345 us (25 TFLOP/s of the
// triangle); this takes 88 us and 9 for the splits' sum (340 -> 97 us a call, 88 TFLOP/s).
//
// part: split s of tile k goes to slot (s, k) for hess_f32_reduce_kernel. part == nullptr
// (one split): the workgroup adds its tile into H, above the diagonal transposed.
constexpr int FCH = KT * HT / 256;  // floats per thread, panel and stage

__global__ __launch_bounds__(256, 2) void hess_f32_kernel(const float* __restrict__ X, int64_t N, int d,
                                                          int ntiles, int splits, int64_t rows_per_split,
                                                          float* __restrict__ H, float* __restrict__ part) {
  __shared__ float sP[2][2][KT][HT + 4];  // [buffer][panel]
  const int total = ntiles * splits, per = (total + 7) / 8;
  // an XCD's workgroups share rows of X (hess_bf16_tri_kernel)
  const int item = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (item >= total) return;
  const int split = item / ntiles, tile = item - split * ntiles;
  int ti = (int)((sqrtf(8.0f * (float)tile + 1.0f) - 1.0f) * 0.5f);
  while (ti * (ti + 1) / 2 > tile) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= tile) ++ti;
  const int tj = tile - ti * (ti + 1) / 2;
  const int i0 = ti * HT, j0 = tj * HT;
  const bool diag = ti == tj;
  const int64_t r0 = (int64_t)split * rows_per_split;
  const int nrows = (int)(min(N, r0 + rows_per_split) - r0);
  if (nrows <= 0) return;  // the host leaves no split without rows
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int wm = (w >> 1) * 64, wn = (w & 1) * 64;
  // thread: column tid % 128 of both panels, rows tid / 128 + 2 q
  const uint32_t rowb = 4u * (uint32_t)d;
  const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)(X + r0 * d), 0, (int)((uint32_t)nrows * rowb), 0x00020000);
  const int c = tid & (HT - 1), rr = tid >> 7;
  const uint32_t oi = i0 + c < d ? (uint32_t)rr * rowb + 4u * (uint32_t)(i0 + c) : kOob;
  const uint32_t oj = j0 + c < d ? (uint32_t)rr * rowb + 4u * (uint32_t)(j0 + c) : kOob;
  float gi[FCH], gj[FCH];
  // the whole offset in the lane's register: the range check is against it
  const auto fetch = [&](int st) {
    const uint32_t so = (uint32_t)st * KT * rowb;
#pragma unroll
    for (int q = 0; q < FCH; ++q)
      gi[q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(oi + so + 2u * q * rowb), 0, 0));
    if (!diag) {
#pragma unroll
      for (int q = 0; q < FCH; ++q)
        gj[q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(oj + so + 2u * q * rowb), 0, 0));
    }
  };
  const auto stash = [&](int b) {
#pragma unroll
    for (int q = 0; q < FCH; ++q) sP[b][0][rr + 2 * q][c] = gi[q];
    if (!diag) {
#pragma unroll
      for (int q = 0; q < FCH; ++q) sP[b][1][rr + 2 * q][c] = gj[q];
    }
  };
  // sums of kFlush stages, and their running total: rounding grows with the longer of the two
  f32x16 acc[2][2], tot[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = tot[a][b][v] = 0.0f;
  const int stages = (nrows + KT - 1) / KT;
  fetch(0);
  stash(0);
  __syncthreads();
  for (int st = 0; st < stages; ++st) {
    if (st + 1 < stages) fetch(st + 1);
    const float(*pa)[HT + 4] = sP[st & 1][0];
    const float(*pb)[HT + 4] = diag ? pa : sP[st & 1][1];
#pragma unroll 8
    for (int k = 0; k < KT; k += 2) {
      float a[2], b[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        a[x] = pa[k + (l >> 5)][wm + x * 32 + (l & 31)];
        b[x] = pb[k + (l >> 5)][wn + x * 32 + (l & 31)];
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[x], b[y], acc[x][y], 0, 0, 0);
    }
    if (st % kFlush == kFlush - 1 || st + 1 == stages) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          tot[x][y] += acc[x][y];
          acc[x][y] = 0.0f;
        }
    }
    if (st + 1 < stages) stash((st + 1) & 1);
    __syncthreads();
  }
  // the tile by rows: into its slot, or into LDS (the panels' 66 KB) on its way into H
  float* const slot = part ? part + (int64_t)(split * ntiles + tile) * (HT * HT) : &sP[0][0][0][0];
  const int pitch = part ? HT : HT + 4;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        slot[(wm + x * 32 + mfma32_row(v, l)) * pitch + wn + y * 32 + (l & 31)] = tot[x][y][v];
  if (part) return;
  static_assert(sizeof(sP) >= HT * (HT + 4) * sizeof(float), "a tile fits the panels");
  const float* tl = &sP[0][0][0][0];
  __syncthreads();
  // H's rows a0 .. + 127, columns b0 .. + 127 take t(r, c); 32 loads in flight (clamped, not
  // branched around)
  const auto add = [&](int a0, int b0, const auto& t) {
    const int cc = min(b0 + c, d - 1);
#pragma unroll
    for (int q0 = 0; q0 < HT / 2; q0 += 32) {
      float h[32];
#pragma unroll
      for (int q = 0; q < 32; ++q) h[q] = H[(int64_t)min(a0 + rr + 2 * (q0 + q), d - 1) * d + cc];
#pragma unroll
      for (int q = 0; q < 32; ++q) {
        const int r = rr + 2 * (q0 + q);
        if (a0 + r < d && b0 + c < d) H[(int64_t)(a0 + r) * d + b0 + c] = h[q] + t(r);
      }
    }
  };
  add(i0, j0, [&](int r) { return tl[r * (HT + 4) + c]; });
  if (!diag) add(j0, i0, [&](int r) { return tl[c * (HT + 4) + r]; });
}

// The row splits' tiles summed in split order, by groups (p_0 + ... + p_15) + (p_16 + ...) + ...,
// and added to H at (i, j) and (j, i), over 32 x 32 blocks of the lower triangle (blockIdx.x, row
// order; small blocks, so a narrow H with many splits still fills the chip); the mirror goes
// through LDS so both sides are coalesced.
constexpr int kSplitGroup = 16;

__global__ __launch_bounds__(256) void hess_f32_reduce_kernel(float* __restrict__ H, int d, int ntiles,
                                                              int splits, const float* __restrict__ part) {
  __shared__ float tl[32][33];
  int bi = (int)((sqrtf(8.0f * (float)blockIdx.x + 1.0f) - 1.0f) * 0.5f);
  while (bi * (bi + 1) / 2 > (int)blockIdx.x) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= (int)blockIdx.x) ++bi;
  const int bj = (int)blockIdx.x - bi * (bi + 1) / 2;
  const int c = threadIdx.x & 31, rt = threadIdx.x >> 5;
  const int ti = bi / 4, tj = bj / 4;
  const int64_t slot = (int64_t)ntiles * (HT * HT);  // floats between one split's tiles
  const float* p = part + (int64_t)(ti * (ti + 1) / 2 + tj) * (HT * HT) + ((bi % 4) * 32 + rt) * HT + (bj % 4) * 32 + c;
  // groups of kSplitGroup splits, and their running total: one chain over a narrow H's splits (up
  // to 512) is further from the float64 sums than fewer, longer splits ([16384, 200] of values
  // about 1: 9.4e-8 in 32 splits, 1.5e-7 in a chain of 128, 5.2e-8 so; [65536, 64] 1.5e-7, 3.0e-7,
  // 7.8e-8, and 85 -> 54 us a call with a group's loads in flight)
  float s[4];
  int k0 = 0;
  for (; k0 + kSplitGroup <= splits; k0 += kSplitGroup) {
    float v[kSplitGroup][4];  // a group's loads all in flight
#pragma unroll
    for (int k = 0; k < kSplitGroup; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[k][q] = p[(k0 + k) * slot + 8 * q * HT];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int k = 1; k < kSplitGroup; ++k) v[0][q] += v[k][q];
      s[q] = k0 ? s[q] + v[0][q] : v[0][q];
    }
  }
  if (k0 < splits) {
    float g[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) g[q] = p[k0 * slot + 8 * q * HT];
#pragma unroll 4
    for (int k = k0 + 1; k < splits; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q) g[q] += p[k * slot + 8 * q * HT];
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = k0 ? s[q] + g[q] : g[q];
  }
  const int j = bj * 32 + c;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = rt + 8 * q, i = bi * 32 + r;
    tl[r][c] = s[q];
    if (i < d && j < d) H[(int64_t)i * d + j] += s[q];
  }
  if (bi == bj) return;  // a diagonal block's tile is whole
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = rt + 8 * q, i = bj * 32 + r, jj = bi * 32 + c;
    if (i < d && jj < d) H[(int64_t)i * d + jj] += tl[c][r];
  }
}

// Row splits for the triangle kernel: one 144 KB-LDS workgroup per CU, so the
// main pass takes about rounds x (stages per split + epilogue), the epilogue (a
// 256 KB tile store) about 6 stages; with more than one split the reduction then
// reads every split's tile once, about 0.05 of a stage per tile and split
// spread over the GPU. A split spans at most 2^30 bytes of X, so the buffer
// offsets of its loads (up to eight stages past its end) stay below 2^31.
// Returns the split count (0 if none fits); *rows_per_split is a multiple of KS
// and every split has rows.
static int pick_splits(int ntiles, int64_t N, int64_t d, int64_t* rows_per_split) {
  int best_s = 0;
  double best = 1e30;
  for (int s = 1; s <= 4096; ++s) {
    const int64_t rows = (N + s - 1) / s;
    if ((rows + KS - 1) / KS * KS * 2 * d > (int64_t(1) << 30)) continue;
    if (best_s && rows < 256) break;
    const double stages = (double)((rows + KS - 1) / KS);
    const double rounds = (double)(((int64_t)ntiles * s + 255) / 256);
    const double cost = rounds * (stages + 6.0) + (s > 1 ? 0.05 * s * ntiles : 0.0);
    if (cost < best - 1e-9) {
      best = cost;
      best_s = s;
    }
  }
  if (const char* e = getenv("CP_HESS_SPLITS")) {  // tuning override (measurement only)
    const int s = atoi(e);
    if (s >= 1 && s <= 4096 && ((N + s - 1) / s + KS - 1) / KS * KS * 2 * d <= (int64_t(1) << 30)) best_s = s;
  }
  if (best_s == 0) return 0;
  int64_t rps = (N + best_s - 1) / best_s;
  rps = (rps + KS - 1) / KS * KS;
  *rows_per_split = rps;
  return (int)((N + rps - 1) / rps);  // rounding rps up may leave fewer splits with rows
}

static int f32_tiles(int64_t d) {
  const int64_t T = (d + HT - 1) / HT;
  return (int)(T * (T + 1) / 2);
}

// Row splits of the f32 kernel: two workgroups per CU, each at least 128 rows. A split spans
// at most 2^30 bytes of X, so its buffer offsets stay below 2^31.
static int f32_splits(int64_t N, int64_t d, int64_t* rows_per_split) {
  const int64_t tiles = f32_tiles(d);
  int64_t splits = 512 / tiles;
  if (splits < 1) splits = 1;
  int64_t rps = (N + splits - 1) / splits;
  if (rps < 128) rps = 128;
  rps = (rps + KT - 1) / KT * KT;
  const int64_t most = ((int64_t)1 << 30) / (4 * d) / KT * KT;  // d <= 2^20: at least 256 rows
  if (rps > most) rps = most;
  *rows_per_split = rps;
  return (int)((N + rps - 1) / rps);
}

constexpr size_t kTileBytes = (size_t)BT * BT * sizeof(float);

// Whether a launch of cn jobs takes the few-rows kernel: its 64 x 64 tiles run in one round (one
// workgroup per CU) and its predicted time is below the row splits'. In microseconds past the
// launches: a workgroup walks all N rows at 2.4 per 1024, more as tiles share the L2s (several
// jobs share no rows and wear on them sooner than one), and 0.7 more per unit where X is past one
// XCD's 4 MB L2 and its rows end inside a 128-byte line (a panel's 128-byte rows then take two;
// up to 128 columns the other panel of the workgroup uses the rest). The splits take their rounds
// of stages, their partial tiles' way through memory, and in the reduction a chain of one load
// per split for each 16 columns of a thread's 64. On 650 shapes (d = 8-1408, 64-131072 rows,
// 1-200 jobs) the line picks no kernel more than 2 % slower than the other; few-rows / splits, us:
// [2048, 1024] 17 / 31, [12288, 1024] 51 / 54, [16384, 1024] 66 / 61, [14000, 896] 52 / 58,
// [14000, 880] 70 / 58, [49152, 256] 138 / 218, [131072, 64] 332 / 314, [65536, 8] 160 / 71,
// 4 x [8192, 512] 47 / 51, 6 x 64 / 48, 5 x [49152, 256] 145 / 95, 64 x [32768, 64] 122 / 165.
static bool few_rows(int cn, int64_t N, int64_t d) {
  const int64_t t64 = (d + 63) / 64, tiles = t64 * (t64 + 1) / 2 * cn;
  if (tiles > 256 || N * d > (int64_t)1 << 29) return false;  // also: buffer offsets below 2^31
  const int64_t T = (d + BT - 1) / BT, units = T * (T + 1) / 2 * cn;
  int64_t rps = 0;
  const int s = pick_splits((int)units, N, d, &rps);
  const double load = cn == 1 ? (double)tiles / 600.0 : (double)(tiles * tiles) / (200.0 * 200.0);
  const bool torn = d > 128 && d % 64 && 2 * N * d * cn > (4 << 20);
  const double few = 0.0024 * (double)N * (1.0 + load + (torn ? 0.7 : 0.0));
  const double stages = (double)((units * s + 255) / 256) * ((double)(rps / KS) + 6.0);
  const int64_t chains = (d + 15) / 16 < 4 ? (d + 15) / 16 : 4;
  const double sums = s > 1 ? (double)s * (0.26 * (double)chains + 0.02 * (double)units) : 0.0;
  return few <= 1.0 + 0.5 * stages + sums;
}

// Workspace of one bf16 launch of cn jobs (0 when it runs as one split).
static size_t bf16_ws(int cn, int64_t N, int64_t d) {
  if (few_rows(cn, N, d)) return 0;
  const int T = (int)((d + BT - 1) / BT);
  const int ntiles = T * (T + 1) / 2;
  int64_t rps = 0;
  const int s = pick_splits(ntiles * cn, N, d, &rps);
  return s > 1 ? (size_t)cn * s * ntiles * kTileBytes : 0;
}

static size_t hess_ws_need(int count, int x_dtype, int64_t N, int64_t d) {
  if (N <= 0 || d <= 0 || count <= 0) return 0;
  if (x_dtype == 0) {
    int64_t rps = 0;
    const int s = f32_splits(N, d, &rps);
    return s > 1 ? (size_t)s * f32_tiles(d) * (HT * HT) * sizeof(float) : 0;  // jobs run one after another
  }
  size_t need = bf16_ws(count < kHessJobs ? count : kHessJobs, N, d);
  if (count > kHessJobs && count % kHessJobs) {
    const size_t tail = bf16_ws(count % kHessJobs, N, d);
    if (tail > need) need = tail;
  }
  return need;
}

}  // namespace cp

namespace cp {

// H_z += X_z^T X_z for count jobs of one shape, bf16 X.
static int hess_bf16_batch(const void* const* X, float* const* H, int count, int64_t N, int64_t d,
                           void* ws, size_t ws_bytes, hipStream_t st) {
  const int T = (int)((d + BT - 1) / BT);
  const int ntiles = T * (T + 1) / 2;
  for (int c0 = 0; c0 < count; c0 += kHessJobs) {
    const int cn = count - c0 < kHessJobs ? count - c0 : kHessJobs;
    HessJobs jobs;
    for (int i = 0; i < cn; ++i) {
      if (!X[c0 + i] || !H[c0 + i]) return set_error(CP_ERR_ARG, "job %d: null X/H", c0 + i);
      if (!aligned(X[c0 + i], 16) || !aligned(H[c0 + i], 4))
        return set_error(CP_ERR_ALIGN, "job %d: X needs 16-byte alignment", c0 + i);
      jobs.X[i] = (const uint16_t*)X[c0 + i];
      jobs.H[i] = H[c0 + i];
    }
    if (few_rows(cn, N, d)) {
      const int t64 = (int)((d + 63) / 64);
      hess_bf16_small_kernel<<<dim3(t64 * (t64 + 1) / 2, cn), 64 * SW, 0, st>>>(jobs, N, (int)d);
      CP_LAUNCHED("hessian launch");
      continue;
    }
    int64_t rps = 0;
    const int splits = pick_splits(ntiles * cn, N, d, &rps);
    if (splits == 0 || (int64_t)ntiles * cn * splits * 8 > INT32_MAX)
      return set_error(CP_ERR_SHAPE, "X [%lld, %lld] too large for one accumulation; pass fewer rows",
                       (long long)N, (long long)d);
    float* part = nullptr;
    if (splits > 1) {
      const size_t need = (size_t)cn * splits * ntiles * kTileBytes;
      if (!ws || ws_bytes < need)
        return set_error(CP_ERR_WORKSPACE, "Hessian workspace: need %zu bytes, have %zu", need, ws_bytes);
      if (!aligned(ws, 16)) return set_error(CP_ERR_ALIGN, "Hessian workspace needs 16-byte alignment");
      part = (float*)ws;
    }
    const int total = ntiles * splits * cn;
    const int per = (total + 7) / 8;
    hess_bf16_tri_kernel<<<dim3(8 * per), HNT, 0, st>>>(jobs, cn, N, (int)d, ntiles, splits, rps, part);
    CP_LAUNCHED("hessian launch");
    const int tb = (int)((d + 63) / 64);
    hess_tri_reduce_kernel<<<dim3(tb * (tb + 1) / 2, cn), 256, 0, st>>>(jobs, (int)d, ntiles, splits, part);
    CP_LAUNCHED("hessian reduce");
  }
  return CP_OK;
}

static int hess_f32(const float* X, int64_t N, int64_t d, float* H, void* ws, size_t ws_bytes,
                    hipStream_t st) {
  const int tiles = f32_tiles(d);
  int64_t rps = 0;
  const int splits = f32_splits(N, d, &rps);
  if ((int64_t)tiles * splits > INT32_MAX / 8)
    return set_error(CP_ERR_SHAPE, "X [%lld, %lld] too large for one accumulation; pass fewer rows",
                     (long long)N, (long long)d);
  float* part = nullptr;
  if (splits > 1) {
    const size_t need = (size_t)splits * tiles * (HT * HT) * sizeof(float);
    if (!ws || ws_bytes < need)
      return set_error(CP_ERR_WORKSPACE, "Hessian workspace: need %zu bytes, have %zu", need, ws_bytes);
    part = (float*)ws;
  }
  const int per = (tiles * splits + 7) / 8;
  hess_f32_kernel<<<dim3(8 * per), 256, 0, st>>>(X, N, (int)d, tiles, splits, rps, H, part);
  CP_LAUNCHED("hessian launch");
  if (part) {
    const int tb = (int)((d + 31) / 32);
    hess_f32_reduce_kernel<<<dim3(tb * (tb + 1) / 2), 256, 0, st>>>(H, (int)d, tiles, splits, part);
    CP_LAUNCHED("hessian reduce");
  }
  return CP_OK;
}

static int hess_check(int x_dtype, int64_t N, int64_t d) {
  if (N < 0 || d <= 0 || d > (1 << 20)) return set_error(CP_ERR_SHAPE, "bad X shape [%lld, %lld]", (long long)N, (long long)d);
  if (x_dtype != 0 && x_dtype != 1) return set_error(CP_ERR_ARG, "x_dtype must be 0 (f32) or 1 (bf16)");
  if (x_dtype == 1 && d % 8) return set_error(CP_ERR_SHAPE, "bf16 X needs d %% 8 == 0 (got %lld)", (long long)d);
  return CP_OK;
}

static int hess_run(const void* const* X, float* const* H, int count, int x_dtype, int64_t N,
                    int64_t d, void* ws, size_t ws_bytes, hipStream_t st) {
  if (x_dtype == 1) return hess_bf16_batch(X, H, count, N, d, ws, ws_bytes, st);
  for (int i = 0; i < count; ++i) {
    if (!X[i] || !H[i]) return set_error(CP_ERR_ARG, "job %d: null X/H", i);
    if (!aligned(X[i], 16) || !aligned(H[i], 4)) return set_error(CP_ERR_ALIGN, "job %d: misaligned", i);
    if (int s = hess_f32((const float*)X[i], N, d, H[i], ws, ws_bytes, st)) return s;
  }
  return CP_OK;
}

// hess_run with a stream-ordered workspace of its own, freed on the stream after
// the last launch that reads it.
static int hess_run_alloc(const void* const* X, float* const* H, int count, int x_dtype, int64_t N,
                          int64_t d, hipStream_t st) {
  const size_t need = hess_ws_need(count, x_dtype, N, d);
  void* ws = nullptr;
  if (need) CP_HIP(hipMallocAsync(&ws, need, st));
  const int s = hess_run(X, H, count, x_dtype, N, d, ws, need, st);
  if (ws) {
    const hipError_t e = hipFreeAsync(ws, st);
    if (s == CP_OK && e != hipSuccess) return hip_fail(e, "hipFreeAsync");
  }
  return s;
}

}  // namespace cp

extern "C" size_t cp_hess_ws_bytes(int count, int x_dtype, int64_t N, int64_t d) {
  return cp::hess_ws_need(count, x_dtype, N, d);
}

extern "C" int cp_hess_accum(const void* X, int x_dtype, int64_t N, int64_t d, float* H, void* stream) {
  cp::clear_error();
  if (int s = cp::hess_check(x_dtype, N, d)) return s;
  if (!H) return cp::set_error(CP_ERR_ARG, "null H");
  if (N == 0) return CP_OK;  // no rows: H += 0
  if (!X) return cp::set_error(CP_ERR_ARG, "null X");
  return cp::hess_run_alloc(&X, &H, 1, x_dtype, N, d, (hipStream_t)stream);
}

extern "C" int cp_hess_accum_batch(const void* const* X, float* const* H, int count, int x_dtype,
                                   int64_t N, int64_t d, void* stream) {
  cp::clear_error();
  if (!X || !H || count <= 0) return cp::set_error(CP_ERR_ARG, "no jobs");
  if (int s = cp::hess_check(x_dtype, N, d)) return s;
  if (N == 0) return CP_OK;  // no rows: every H += 0
  return cp::hess_run_alloc(X, H, count, x_dtype, N, d, (hipStream_t)stream);
}

extern "C" int cp_hess_accum_batch_ws(const void* const* X, float* const* H, int count, int x_dtype,
                                      int64_t N, int64_t d, void* ws, size_t ws_bytes, void* stream) {
  cp::clear_error();
  if (!X || !H || count <= 0) return cp::set_error(CP_ERR_ARG, "no jobs");
  if (int s = cp::hess_check(x_dtype, N, d)) return s;
  if (N == 0) return CP_OK;  // no rows: every H += 0
  return cp::hess_run(X, H, count, x_dtype, N, d, ws, ws_bytes, (hipStream_t)stream);
}
