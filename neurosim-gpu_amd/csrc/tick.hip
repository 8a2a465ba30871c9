// Fused dendritic matrix tick for gfx950: CSR gather-product over B columns,
// then the three-state update, with fp32 / fp16 / fp8 e4m3 / nvfp4 weights
// decoded in-register and accumulated in float32.
//
// Semantics follow the reference's fused kernel (csrc/compartmental.cu:121-140
// and :72-90) and its PyTorch twin (runtime.py:78-79, compartmental.py:152-183);
// the work decomposition is this library's own:
//
//  * Rows are cut on the host into row blocks of consecutive rows whose edges
//    fit one workgroup's edge capacity (ns_plan_row_blocks).  One 256-lane
//    workgroup owns one row block and one tile of BT batch columns.
//  * Phase 1 streams the block's contiguous edge range with aligned 16-byte
//    loads of col_idx (4 edges per lane per pass) and the matching weight
//    bytes, decodes, gathers s[col] for the BT columns and writes the products
//    to LDS ([column][edge] layout, padded).
//  * Phase 2 assigns a power-of-two group of lanes to every row (more lanes
//    to fewer, longer rows), reduces the row's products from LDS, finishes
//    with cross-lane xor shuffles and applies the update on one lane per
//    (row, column).
//  * A block that does not fit (a row longer than the capacity) is reduced
//    row by row by the whole workgroup.
//
// The summation order depends only on the plan, the batch tile and the
// weights' position, so results are bitwise repeatable and identical across
// weight encodings that decode to the same float32 values.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <type_traits>

#include "ns_common.h"
#include "ns_host.h"

namespace ns {

template <int BT>
struct TileCfg;
template <>
struct TileCfg<1> { static constexpr int passes = 2; };
template <>
struct TileCfg<2> { static constexpr int passes = 2; };
template <>
struct TileCfg<4> { static constexpr int passes = 1; };
template <>
struct TileCfg<8> { static constexpr int passes = 1; };

template <int BT>
constexpr int block_capacity() { return kThreads * 4 * TileCfg<BT>::passes; }

struct TickArgs {
  int64_t N, B, M;
  Plane s, d, a, u, v;
  Params p;
  const int32_t* rowptr;
  const int32_t* col;
  const void* weight;
  const uint8_t* scales;
  const float* gscale;
  const int32_t* bounds;
  int64_t n_blocks;
  OutPlane os, od, oa;
  OutPlane oj;          // optional: j as well (data null: not written)
  int32_t quad_loads;   // col/weight pointers aligned for one-quad vector loads
  int32_t s_rows;       // s is neuron-major: a source's columns are neighbours
  int32_t spmm_only;    // write j to `os` instead of advancing
  int32_t spmm_accumulate;  // with spmm_only: add j to `os` instead
};

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// Decode the four weights of the aligned quad [q, q+4) (q % 4 == 0).
// Lanes past the end of the arrays read nothing; those edges are masked later.
template <int FMT>
__device__ __forceinline__ void load_quad(const TickArgs& A, int64_t q, bool vec, int c[4],
                                          float w[4], float gscale) {
  if (vec) {
    const v4i cv = *reinterpret_cast<const v4i*>(A.col + q);
    c[0] = cv.x; c[1] = cv.y; c[2] = cv.z; c[3] = cv.w;
    if constexpr (FMT == NS_WEIGHT_F32) {
      const v4f wv = *reinterpret_cast<const v4f*>(static_cast<const float*>(A.weight) + q);
      w[0] = wv.x; w[1] = wv.y; w[2] = wv.z; w[3] = wv.w;
    } else if constexpr (FMT == NS_WEIGHT_F16) {
      const v4h hv = *reinterpret_cast<const v4h*>(static_cast<const _Float16*>(A.weight) + q);
      w[0] = static_cast<float>(hv.x); w[1] = static_cast<float>(hv.y);
      w[2] = static_cast<float>(hv.z); w[3] = static_cast<float>(hv.w);
    } else if constexpr (FMT == NS_WEIGHT_E4M3) {
      const uint32_t codes = *reinterpret_cast<const uint32_t*>(
          static_cast<const uint8_t*>(A.weight) + q);
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = e4m3_to_float((codes >> (8 * k)) & 0xFFu) * gscale;
    } else {
      const uint32_t nibbles = *reinterpret_cast<const uint16_t*>(
          static_cast<const uint8_t*>(A.weight) + (q >> 1));
      const float bs = e4m3_to_float(A.scales[q >> 4]) * gscale;
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = nvfp4_weight((nibbles >> (4 * k)) & 15u, bs);
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t e = q + k;
    c[k] = 0;
    w[k] = 0.0f;
    if (e < A.M) {
      c[k] = A.col[e];
      w[k] = csr_weight<FMT>(A.weight, A.scales, e, gscale);
    }
  }
}

__device__ __forceinline__ void finish(const TickArgs& A, int64_t n, int64_t b, float j) {
  if (A.spmm_only) {
    A.os.put(b, n, A.spmm_accumulate ? A.os.data[b * A.os.sb + n * A.os.sn] + j : j);
    return;
  }
  const NextState x = advance_one(A.p, n, j, A.s.get(b, n), A.d.get(b, n), A.a.get(b, n),
                                  A.u.get(b, n), A.v.get(b, n));
  A.os.put(b, n, x.soma);
  A.od.put(b, n, x.dendrite);
  A.oa.put(b, n, x.adaptation);
  if (A.oj.data) A.oj.put(b, n, j);
}

// Rows of a block that does not fit the LDS path: the whole workgroup reduces
// one row at a time (long rows, or a plan built for another capacity).
template <int BT, int FMT>
__device__ void rows_one_by_one(const TickArgs& A, int r0, int r1, int b0, float gscale,
                                float* red) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  for (int r = r0; r < r1; ++r) {
    const int64_t rs = A.rowptr[r], re = A.rowptr[r + 1];
    float acc[BT];
#pragma unroll
    for (int j = 0; j < BT; ++j) acc[j] = 0.0f;
    for (int64_t e = rs + tid; e < re; e += kThreads) {
      const float w = csr_weight<FMT>(A.weight, A.scales, e, gscale);
      const int64_t c = A.col[e];
#pragma unroll
      for (int j = 0; j < BT; ++j)
        if (b0 + j < A.B) acc[j] += w * A.s.data[(b0 + j) * A.s.sb + c * A.s.sn];
    }
#pragma unroll
    for (int j = 0; j < BT; ++j) {
      float x = acc[j];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
      if (lane == 0) red[wave * BT + j] = x;
    }
    __syncthreads();
    if (tid < BT && b0 + tid < A.B) {
      const float j = ((red[tid] + red[BT + tid]) + red[2 * BT + tid]) + red[3 * BT + tid];
      finish(A, r, b0 + tid, j);
    }
    __syncthreads();
  }
}

// Lanes that share a source's row, each loading up to four of the tile's columns.
template <int BT>
constexpr int kShare = BT > 4 ? BT / 4 : 1;

// Padded [column][edge] rows of a workgroup's products in LDS (16-byte aligned).
template <int BT>
constexpr int kProductStride = block_capacity<BT>() + 4;

// The value of the first (k = 0) or second lane of this lane's pair (kLanes 2).
template <int kLanes, int k>
__device__ __forceinline__ int shared_lane(int x) {
  if constexpr (kLanes == 1) return x;
  constexpr int control = k == 0 ? 0xA0 : 0xF5;   // quad_perm 0 0 2 2 or 1 1 3 3
  return __builtin_amdgcn_update_dpp(0, x, control, 0xF, 0xF, true);
}

// kCols neighbouring floats at any 4-byte aligned address, in one load.
template <int kCols>
__device__ __forceinline__ void load_columns(const float* at, float (&x)[4]) {
  if constexpr (kCols == 1) {
    x[0] = *at;
  } else {
    typedef float vec __attribute__((ext_vector_type(kCols)));
    struct __attribute__((packed, aligned(4))) words { vec v; };
    const vec y = reinterpret_cast<const words*>(at)->v;
#pragma unroll
    for (int k = 0; k < kCols; ++k) x[k] = y[k];
  }
}

template <int BT, int kCols>
__device__ __forceinline__ void gather_columns(const float* s, int64_t sn,
                                               const int (&c)[4 * kShare<BT>], int first, int e0,
                                               int e1, float (&g)[4 * kShare<BT>][4]) {
#pragma unroll
  for (int i = 0; i < 4 * kShare<BT>; ++i)
    if (first + i >= e0 && first + i < e1) load_columns<kCols>(s + c[i] * sn, g[i]);
}

// Phase 1 of one pass for a neuron-major state.  At eight columns the two lanes of
// a pair take their eight edges together, each loading four columns of every edge's
// source row, so that one load instruction reads 32 whole rows and the L2 sees one
// request per row rather than two (the lanes trade column indices and weights by
// DPP).  A row needs 4-byte alignment only, so odd batches load the same way, in
// one or two loads per edge where they took one per column.  The products and their
// LDS places are those of the per-lane path, so the sums are bitwise the same.  us
// per tick, N=50k, M=1M, fp32, before and after: B=2 10.5, 9.2; B=3 12.6, 10.0; B=5
// 18.8, 13.9; B=7 23.9, 14.7; B=4 and 8 unchanged (9.9, 13.8).
template <int BT, bool kWhole>
__device__ __forceinline__ void gather_rows(const TickArgs& A, const int (&c_own)[4],
                                            const float (&w_own)[4], bool have, int first, int e0,
                                            int e1, int b0, float* prod) {
  constexpr int kEdges = 4 * kShare<BT>;
  constexpr int kWidth = BT < 4 ? BT : 4;
  const int part = threadIdx.x & (kShare<BT> - 1);
  const int cols = kWhole ? kWidth
                          : static_cast<int>(min<int64_t>(kWidth, A.B - (b0 + kWidth * part)));
  int c[kEdges];
  float w[kEdges];
  const auto trade = [&](auto lane) {
    constexpr int k = decltype(lane)::value;
    if constexpr (k < kShare<BT>) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        c[4 * k + j] = shared_lane<kShare<BT>, k>(have ? c_own[j] : 0);
        w[4 * k + j] = __builtin_bit_cast(
            float, shared_lane<kShare<BT>, k>(__builtin_bit_cast(int, have ? w_own[j] : 0.0f)));
      }
    }
  };
  trade(std::integral_constant<int, 0>{});
  trade(std::integral_constant<int, 1>{});
  float g[kEdges][4];
#pragma unroll
  for (int i = 0; i < kEdges; ++i) g[i][0] = g[i][1] = g[i][2] = g[i][3] = 0.0f;
  const float* const s = A.s.data + (b0 + kWidth * part);
  // Where lanes of different column counts share rows, they load four floats all the
  // same, in one instruction, the ones past the batch being the next neuron's and
  // left unused; only a row at the plane's very end is loaded column by column.
  const int64_t end = kWhole || kShare<BT> == 1
                          ? 0 : (A.N - 1) * A.s.sn + A.B - (b0 + kWidth * part) - kWidth;
  if (kWhole || (kShare<BT> == 1 && cols >= kWidth)) {
    gather_columns<BT, kWidth>(s, A.s.sn, c, first, e0, e1, g);
  } else if (kShare<BT> == 1) {
    if (cols == 3) gather_columns<BT, 3>(s, A.s.sn, c, first, e0, e1, g);
    else if (cols == 2) gather_columns<BT, 2>(s, A.s.sn, c, first, e0, e1, g);
    else if (cols == 1) gather_columns<BT, 1>(s, A.s.sn, c, first, e0, e1, g);
  } else if (cols > 0) {
#pragma unroll
    for (int i = 0; i < kEdges; ++i) {
      const int64_t at = c[i] * A.s.sn;
      if (first + i < e0 || first + i >= e1) continue;
      if (at <= end) {
        load_columns<kWidth>(s + at, g[i]);
      } else {
        for (int k = 0; k < cols; ++k) g[i][k] = s[at + k];
      }
    }
  }
  if (first >= e1) return;
#pragma unroll
  for (int t = 0; t < kWidth; ++t) {
    if (!kWhole && t >= cols) break;   // nobody reads a column past the batch
    float* const at = prod + (kWidth * part + t) * kProductStride<BT>;
#pragma unroll
    for (int k = 0; k < kShare<BT>; ++k) {
      v4f pv;
      pv.x = w[4 * k] * g[4 * k][t];
      pv.y = w[4 * k + 1] * g[4 * k + 1][t];
      pv.z = w[4 * k + 2] * g[4 * k + 2][t];
      pv.w = w[4 * k + 3] * g[4 * k + 3][t];
      *reinterpret_cast<v4f*>(at + 4 * k) = pv;
    }
  }
}

// kWhole: the state is neuron-major and the batch a multiple of the tile, so that every
// workgroup takes whole rows and no lane tests its column against the batch.
// The one kernel for all forms kept 126 registers at 8 columns where this takes 102.
// us per 32 ticks, N=15k, M=900k, fp32, one kernel / this one: B=4 384 / 367, B=8 444 /
// 426, B=16 673 / 656; N=9k, M=700k, B=2 327 / 323.
template <int BT, int FMT, bool kWhole>
__global__ __launch_bounds__(kThreads) void tick_kernel(TickArgs A) {
  constexpr int kPasses = TileCfg<BT>::passes;
  constexpr int kCap = block_capacity<BT>();
  constexpr int kStride = kProductStride<BT>;
  __shared__ __attribute__((aligned(16))) float prod[BT * kStride];
  __shared__ int32_t srow[kMaxRows + 1];

  const int tid = threadIdx.x;
  const int64_t blk = blockIdx.x;
  const int b0 = blockIdx.y * BT;
  const float gscale = (FMT == NS_WEIGHT_E4M3 || FMT == NS_WEIGHT_NVFP4) ? *A.gscale : 1.0f;

  // The plan's boundary pairs carry each block's first row and first edge, so
  // the edge range needs no rowptr load (clamped into the edge arrays).
  const int32_t* bnd = A.bounds + 2 * blk;
  const int r0 = min(max(bnd[0], 0), static_cast<int>(A.N));
  const int r1 = min(max(bnd[2], r0), static_cast<int>(A.N));
  const int nrows = r1 - r0;
  if (nrows == 0) return;
  const int e0 = static_cast<int>(min<int64_t>(max(bnd[1], 0), A.M));
  const int e1 = static_cast<int>(min<int64_t>(max(bnd[3], e0), A.M));
  const int base = e0 & ~3;
  if (nrows > kMaxRows || e1 - base > kCap) {
    rows_one_by_one<BT, FMT>(A, r0, r1, b0, gscale, prod);
    return;
  }

  // Phase 1 loads first: the block's col/weight quads.
  int cq[kPasses][4];
  float wq[kPasses][4];
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int q = base + (p * kThreads + tid) * 4;
    if (q < e1) {
      const bool vec = A.quad_loads && (static_cast<int64_t>(q) + 4 <= A.M);
      load_quad<FMT>(A, q, vec, cq[p], wq[p], gscale);
    }
  }

  // Phase 2's geometry depends only on the row count, so each lane's update
  // operands (its row's parameters and its columns' five planes) load now,
  // alongside the quads, and the update at the end waits on nothing.
  int group = kThreads / nrows;                  // lanes per row, power of two, <= 64
  group = 1 << (31 - __builtin_clz(group));
  group = group > 64 ? 64 : group;
  const int cols_at_once = group < BT ? group : BT;
  const int slices = group / cols_at_once;
  const int col_rounds = BT / cols_at_once;
  const int i = tid / group;
  const int lane = tid & (group - 1);
  const int cpos = lane & (cols_at_once - 1);
  const int h = lane / cols_at_once;
  const bool row_ok = i < nrows;
  const bool updates = row_ok && h == 0 && !A.spmm_only;
  const int64_t n = r0 + i;
  NeuronParams prm{};
  float us[BT], ud[BT], ua[BT], uu[BT], uv[BT];
  if (updates) {
    prm = load_params(A.p, n);
#pragma unroll
    for (int round = 0; round < BT; ++round) {
      const int64_t b = b0 + cpos + round * cols_at_once;
      if (round < col_rounds && (kWhole || b < A.B)) {
        us[round] = A.s.get(b, n); ud[round] = A.d.get(b, n); ua[round] = A.a.get(b, n);
        uu[round] = A.u.get(b, n); uv[round] = A.v.get(b, n);
      }
    }
  }
  for (int r = tid; r <= nrows; r += kThreads) srow[r] = A.rowptr[r0 + r];

  // Phase 1: decode, gather, multiply, stage in LDS.
  bool staged = false;
  if constexpr (BT >= 2) {
    if (kWhole || A.s_rows) {
      staged = true;
      const bool whole = kWhole || b0 + BT <= A.B;
#pragma unroll
      for (int p = 0; p < kPasses; ++p) {
        const int q = base + (p * kThreads + tid) * 4;
        const bool have = q < e1;
        const int first = base + (p * kThreads + (tid & ~(kShare<BT> - 1))) * 4;
        if (whole)
          gather_rows<BT, true>(A, cq[p], wq[p], have, first, e0, e1, b0, prod + (first - base));
        else
          gather_rows<BT, false>(A, cq[p], wq[p], have, first, e0, e1, b0, prod + (first - base));
      }
    }
  }
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    if (kWhole || staged) break;
    const int q = base + (p * kThreads + tid) * 4;
    if (q < e1) {
      float g[4][BT];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int e = q + k;
        const bool valid = e >= e0 && e < e1;
        const int64_t c = cq[p][k];
#pragma unroll
        for (int j = 0; j < BT; ++j)
          g[k][j] = (valid && b0 + j < A.B) ? A.s.data[(b0 + j) * A.s.sb + c * A.s.sn] : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < BT; ++j) {
        v4f pv;
        pv.x = wq[p][0] * g[0][j];
        pv.y = wq[p][1] * g[1][j];
        pv.z = wq[p][2] * g[2][j];
        pv.w = wq[p][3] * g[3][j];
        *reinterpret_cast<v4f*>(prod + j * kStride + (q - base)) = pv;
      }
    }
  }
  __syncthreads();

  // Phase 2: per-row reduction from LDS, then the update.
  int rs = 0, re = 0;
  if (row_ok) {
    rs = max(srow[i], e0);
    re = min(srow[i + 1], e1);
  }
#pragma unroll
  for (int round = 0; round < BT; ++round) {
    if (round >= col_rounds) continue;   // (not break: the loop must fully unroll)
    const int j = cpos + round * cols_at_once;
    float acc = 0.0f;
    if (row_ok) {
      // Four running sums over interleaved products, so the LDS reads of a
      // row overlap instead of waiting on one add chain.
      const float* row = prod + j * kStride - base;
      float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
      int e = rs + h;
      for (; e + 3 * slices < re; e += 4 * slices) {
        a0 += row[e];
        a1 += row[e + slices];
        a2 += row[e + 2 * slices];
        a3 += row[e + 3 * slices];
      }
      for (; e < re; e += slices) a0 += row[e];
      acc = (a0 + a1) + (a2 + a3);
    }
    for (int off = cols_at_once; off < group; off <<= 1) acc += __shfl_xor(acc, off, 64);
    if (row_ok && h == 0 && (kWhole || b0 + j < A.B)) {
      if (A.spmm_only) {
        const int64_t b = b0 + j;
        A.os.put(b, n, A.spmm_accumulate ? A.os.data[b * A.os.sb + n * A.os.sn] + acc : acc);
      } else {
        const NextState x = advance_loaded(prm, acc, us[round], ud[round], ua[round], uu[round],
                                           uv[round]);
        A.os.put(b0 + j, n, x.soma);
        A.od.put(b0 + j, n, x.dendrite);
        A.oa.put(b0 + j, n, x.adaptation);
        if (A.oj.data) A.oj.put(b0 + j, n, acc);
      }
    }
  }
}

int column_tile(int64_t batch) {
  if (batch <= 1) return 1;
  if (batch <= 2) return 2;
  if (batch <= 4) return 4;
  // Wider batches run in tiles of 8 columns: a 16-column tile needs 67 KB of LDS and
  // 200 registers per lane, two workgroups per compute unit (us per tick at 16 / 8
  // columns per tile, N=50k, M=1M: B=12 25.4 / 23.2, B=16 27.0 / 25.7, B=24 50.3 /
  // 40.4; N=30k, M=3M, B=12 48.1 / 44.5).
  return 8;
}

int32_t capacity_for(int64_t batch) {
  switch (column_tile(batch)) {
    case 1: return block_capacity<1>();
    case 2: return block_capacity<2>();
    case 4: return block_capacity<4>();
    default: return block_capacity<8>();
  }
}

template <int BT, bool kWhole = false>
hipError_t launch_tile(const TickArgs& A, int fmt, hipStream_t stream) {
  if constexpr (BT > 1 && !kWhole) {
    if (A.s_rows && A.B % BT == 0) return launch_tile<BT, true>(A, fmt, stream);
  }
  const dim3 grid(static_cast<unsigned>(A.n_blocks),
                  static_cast<unsigned>((A.B + BT - 1) / BT));
  const dim3 block(kThreads);
  switch (fmt) {
    case NS_WEIGHT_F32:
      tick_kernel<BT, NS_WEIGHT_F32, kWhole><<<grid, block, 0, stream>>>(A);
      break;
    case NS_WEIGHT_F16:
      tick_kernel<BT, NS_WEIGHT_F16, kWhole><<<grid, block, 0, stream>>>(A);
      break;
    case NS_WEIGHT_E4M3:
      tick_kernel<BT, NS_WEIGHT_E4M3, kWhole><<<grid, block, 0, stream>>>(A);
      break;
    default:
      tick_kernel<BT, NS_WEIGHT_NVFP4, kWhole><<<grid, block, 0, stream>>>(A);
  }
  return hipGetLastError();
}

hipError_t launch_tick(const TickArgs& A, int fmt, hipStream_t stream) {
  switch (column_tile(A.B)) {
    case 1: return launch_tile<1>(A, fmt, stream);
    case 2: return launch_tile<2>(A, fmt, stream);
    case 4: return launch_tile<4>(A, fmt, stream);
    default: return launch_tile<8>(A, fmt, stream);
  }
}

int panel_step(const ns_step_args& a, hipStream_t stream, int product, bool launch);
int rollout_step(const ns_step_args& a, hipStream_t stream);

// Host-side validation shared by the tick and the plain product.
int check_csr(const ns_csr& m, int64_t n) {
  if (m.n_rows != n) return fail("CSR row count %lld does not match N=%lld",
                                 (long long)m.n_rows, (long long)n);
  if (m.n_edges < 0 || m.n_edges >= (int64_t{1} << 31))
    return fail("edge count must be in [0, 2^31)");
  if (!m.rowptr) return fail("CSR rowptr is required");
  if (m.n_edges > 0 && (!m.col || !m.weight)) return fail("CSR col and weight are required");
  switch (m.format) {
    case NS_WEIGHT_F32:
    case NS_WEIGHT_F16:
      if (m.block_scales || m.global_scale)
        return fail("floating-point CSR weights take no scales");
      break;
    case NS_WEIGHT_E4M3:
      if (!m.global_scale) return fail("quantized CSR weights require a global scale");
      if (m.block_scales) return fail("fp8 weights take no block scales");
      break;
    case NS_WEIGHT_NVFP4:
      if (!m.global_scale) return fail("quantized CSR weights require a global scale");
      if (m.n_edges > 0 && !m.block_scales) return fail("NVFP4 weights require block scales");
      break;
    default:
      return fail("unknown CSR weight format %d", m.format);
  }
  return NS_OK;
}

int check_matrix(const ns_csr& m, int64_t n, const ns_row_plan& plan, int64_t batch) {
  if (int rc = check_csr(m, n)) return rc;
  if (!plan.bounds || plan.n_blocks < 1) return fail("a row plan is required");
  if (plan.n_blocks > 0x7FFFFFFF) return fail("row plan has too many blocks");
  if (plan.block_edges < 8 || plan.block_edges % 4 || plan.block_edges > capacity_for(batch))
    return fail("row plan was built for %d edges per block, batch %lld takes a multiple of 4 "
                "from 8 to %d", plan.block_edges, (long long)batch, capacity_for(batch));
  return NS_OK;
}

int32_t quad_aligned(const ns_csr& m) {
  const uintptr_t col = reinterpret_cast<uintptr_t>(m.col);
  const uintptr_t w = reinterpret_cast<uintptr_t>(m.weight);
  uintptr_t need = 16;
  switch (m.format) {
    case NS_WEIGHT_F32: need = 16; break;
    case NS_WEIGHT_F16: need = 8; break;
    case NS_WEIGHT_E4M3: need = 4; break;
    default: need = 2; break;
  }
  return (col % 16 == 0) && (w % need == 0);
}

// Whether a source's columns are neighbours in memory (every tensor plane's
// address is a multiple of 4).
int32_t neuron_major(const ns_plane& s, int64_t batch) {
  return batch >= 2 && s.stride_b == 1 && reinterpret_cast<uintptr_t>(s.data) % 4 == 0;
}

}  // namespace ns

using namespace ns;

extern "C" int32_t ns_block_edges(int64_t batch) { return capacity_for(batch); }

namespace ns {

// Checks shared by every matrix-tick entry: sizes, parameters and the CSR's
// weight encoding (check_step_head), then the planes, which must be present
// and must not overlap where outputs are concerned (check_step_planes).
int check_step_head(const ns_step_args& a) {
  if (a.n_neurons <= 0) return fail("state must be [B,N], N > 0");
  if (a.batch < 0) return fail("batch must be non-negative");
  if (a.n_neurons >= (int64_t{1} << 31)) return fail("N must be below 2^31");
  for (int i = 0; i < 6; ++i)
    if (!a.params[i].data) return fail("six neuron parameter vectors are required");
  return check_csr(a.matrix, a.n_neurons);
}

int check_step_planes(const ns_step_args& a) {
  if (!a.state.data || !a.dendrite.data || !a.adaptation.data)
    return fail("state, dendrite and adaptation data are required");
  if (!a.out_state.data || !a.out_dendrite.data || !a.out_adaptation.data)
    return fail("three output planes are required");
  const Extent outs[4] = {extent(a.out_state, a.batch, a.n_neurons),
                          extent(a.out_dendrite, a.batch, a.n_neurons),
                          extent(a.out_adaptation, a.batch, a.n_neurons),
                          extent(a.out_current, a.batch, a.n_neurons)};
  const Extent ins[5] = {extent(a.state, a.batch, a.n_neurons),
                         extent(a.dendrite, a.batch, a.n_neurons),
                         extent(a.adaptation, a.batch, a.n_neurons),
                         extent(a.drive, a.batch, a.n_neurons),
                         extent(a.dendritic_drive, a.batch, a.n_neurons)};
  for (int o = 0; o < 4; ++o) {
    for (int i = 0; i < 5; ++i)
      if (overlaps(outs[o], ins[i])) return fail("output planes must not overlap inputs");
    for (int p = o + 1; p < 4; ++p)
      if (overlaps(outs[o], outs[p])) return fail("output planes must not overlap each other");
  }
  return NS_OK;
}

}  // namespace ns

extern "C" int ns_dendritic_step(const ns_step_args* args, void* stream) {
  clear_error();
  if (!args) return fail("arguments are required");
  const ns_step_args& a = *args;
  if (int rc = check_step_head(a)) return rc;
  if (a.rollout) return rollout_step(a, static_cast<hipStream_t>(stream));
  if (!a.panels)
    if (int rc = check_matrix(a.matrix, a.n_neurons, a.plan, a.batch)) return rc;
  if (a.batch == 0) return NS_OK;  // empty planes may carry null pointers
  if (int rc = check_step_planes(a)) return rc;
  if (a.panels) return panel_step(a, static_cast<hipStream_t>(stream), 0, true);

  TickArgs A{};
  A.N = a.n_neurons; A.B = a.batch; A.M = a.matrix.n_edges;
  A.s = plane(a.state, a.state.data); A.d = plane(a.dendrite, a.state.data);
  A.a = plane(a.adaptation, a.state.data);
  A.u = plane(a.drive, a.state.data); A.v = plane(a.dendritic_drive, a.state.data);
  for (int i = 0; i < 6; ++i) A.p.v[i] = Vec{a.params[i].data, a.params[i].stride};
  A.rowptr = a.matrix.rowptr; A.col = a.matrix.col; A.weight = a.matrix.weight;
  A.scales = a.matrix.block_scales; A.gscale = a.matrix.global_scale;
  A.bounds = a.plan.bounds; A.n_blocks = a.plan.n_blocks;
  A.os = out_plane(a.out_state); A.od = out_plane(a.out_dendrite);
  A.oa = out_plane(a.out_adaptation); A.oj = out_plane(a.out_current);
  A.quad_loads = quad_aligned(a.matrix);
  A.s_rows = neuron_major(a.state, a.batch);
  A.spmm_only = 0;
  const hipError_t err = launch_tick(A, a.matrix.format, static_cast<hipStream_t>(stream));
  if (err != hipSuccess) return fail_launch("dendritic tick", err);
  return NS_OK;
}

extern "C" int ns_csr_spmm(const ns_spmm_args* args, void* stream) {
  clear_error();
  if (!args) return fail("arguments are required");
  const ns_spmm_args& a = *args;
  if (a.n_neurons <= 0) return fail("source must be [B,N], N > 0");
  if (a.batch < 0) return fail("batch must be non-negative");
  if (a.n_neurons >= (int64_t{1} << 31)) return fail("N must be below 2^31");
  if (a.panels) {
    if (int rc = check_csr(a.matrix, a.n_neurons)) return rc;
  } else if (int rc = check_matrix(a.matrix, a.n_neurons, a.plan, a.batch)) {
    return rc;
  }
  if (a.batch == 0) return NS_OK;  // empty planes may carry null pointers
  if (!a.source.data) return fail("source data is required");
  if (!a.out.data) return fail("an output plane is required");
  if (overlaps(extent(a.out, a.batch, a.n_neurons), extent(a.source, a.batch, a.n_neurons)))
    return fail("output plane must not overlap the source");
  if (a.accumulate && !distinct_elements(a.out.stride_b, a.out.stride_n, a.batch, a.n_neurons))
    return fail("an accumulated output plane must not overlap itself (strides %lld, %lld)",
                (long long)a.out.stride_b, (long long)a.out.stride_n);
  if (a.panels) {
    // The panel kernel in product mode: per-panel sums, then the combine
    // kernel adds them in panel order and stores (1) or adds (2) them.
    ns_step_args step{};
    step.n_neurons = a.n_neurons; step.batch = a.batch;
    step.state = a.source; step.matrix = a.matrix; step.panels = a.panels;
    step.out_state = a.out;
    return panel_step(step, static_cast<hipStream_t>(stream), a.accumulate ? 2 : 1, true);
  }

  TickArgs A{};
  A.N = a.n_neurons; A.B = a.batch; A.M = a.matrix.n_edges;
  A.s = plane(a.source, a.source.data);
  A.rowptr = a.matrix.rowptr; A.col = a.matrix.col; A.weight = a.matrix.weight;
  A.scales = a.matrix.block_scales; A.gscale = a.matrix.global_scale;
  A.bounds = a.plan.bounds; A.n_blocks = a.plan.n_blocks;
  A.os = out_plane(a.out);
  A.quad_loads = quad_aligned(a.matrix);
  A.s_rows = neuron_major(a.source, a.batch);
  A.spmm_only = 1;
  A.spmm_accumulate = a.accumulate != 0;
  const hipError_t err = launch_tick(A, a.matrix.format, static_cast<hipStream_t>(stream));
  if (err != hipSuccess) return fail_launch("CSR product", err);
  return NS_OK;
}
