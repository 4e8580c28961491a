// bf16 dense softsign propagation without an edge matrix.
//
// The edges E = softsign(P_t diag(w_hat) P_s^T + b) are a product over at most
// 64 ranks: rebuilding a tile of them where it is used costs less than the
// N x N fp32 matrix costs to write and read (C4: 0.5 GB per eight batch
// elements, in each of six products).  Two kernels serve every N x N product of
// a layer, each with its rows and columns in either role:
//
//   dense_aggregate_kernel   out = E . V and E . x over the columns
//     rows = targets, V = projected values, x = projected state: the forward
//     rows = sources, V = grad delta_val, x = grad delta_state: E^T . gdv, E^T . gds
//   dense_score_grad_kernel  dP = G . P over the columns, with
//     G = (gdv . pv^T + gds ps^T) (1 - |E|)^2, never stored
//     rows = targets: the target projection's gradient (and the row sums of G)
//     rows = sources: the source projection's
//
// Arithmetic: the scores and G . P on three-term bf16 splits (x3_split: six
// exact products, fp32 accuracy); E . V and gdv . pv^T on bf16 operands, E
// rounded to bf16 as it enters the product; everything else in fp32.  Every sum
// has a fixed order.
//
// Measured at C4 sizes (16 x 4096 nodes, 512 values, rank 64, forward and
// backward) against the GEMMs over edge matrices in two batch chunks: step 5.48
// -> 2.85 ms; aggregate 0.42 and 0.41 ms (0.46 MFMA busy), score gradient 0.90
// and 0.89 ms (0.31 MFMA busy).
//
// The split operands are laid out by dense_planes_kernel and dense_pack_kernel
// before: rows of three 64-rank planes, their transposes in blocks of 32 rows,
// and value rows in MFMA fragment order.  Rows are padded to Npad (a multiple
// of 128) with zeros, which contribute nothing.
#include "jn_internal.hpp"

namespace jakal {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // (arrays of uint4 in flight go through scratch memory)

constexpr int kDfRows = 128;             // rows of an aggregate workgroup
constexpr int kDfThreads = 512;          // 8 waves of 16 rows (scores) or D / 8 columns (E . V)
constexpr int kDfGradRows = 64;          // rows of a score-gradient workgroup
constexpr int kDfGradThreads = 256;      // 4 waves: 2 row groups of 32 x 2 column groups of 16
constexpr int kDfRank = 64;              // ranks of a plane row (zeros past the rank)
constexpr int kDfPlaneRow = 3 * kDfRank; // elements of a row's planes: h, m, l
constexpr int kDfFrag = 512;             // elements of an MFMA fragment: 64 lanes of 8

// ---- operand layouts -----------------------------------------------------------

// Rows [b][j] of one projection (stride ld, r ranks) into three-term planes in
// MFMA fragment order, so that a wave's fragment is one contiguous kilobyte in
// global memory and in LDS (no bank conflicts):
//   planes [b][Npad / 16][2][3][64 lanes][8]: rows times scale (or 1); lane l of
//     a 16-row tile holds ranks 32 s + 8 (l / 16) .. + 7 of row l % 16;
//   blocks [b][Npad / 32][4][3][64 lanes][8]: transposed, unscaled; lane l of a
//     16-rank tile holds rows 8 (l / 16) .. + 7 of rank l % 16.
// A workgroup takes 32 rows; blockIdx.z picks the projection (0: targets, with
// the scale; 1: sources).
struct DensePlanesArgs {
  const float* proj[2];
  int64_t ld;
  const float* scale;  // of proj[0]'s planes
  bf16_t* planes[2];
  bf16_t* blocks[2];   // or null
  int N, Npad, r;
};

// eight values into one lane's piece of the h, m and l fragments at `to`
__device__ __forceinline__ void df_store_planes(const float (&x)[8], bf16_t* to) {
  uint32_t h[8], m[8], l[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x3_split(__float_as_uint(x[i]), h[i], m[i], l[i]);
  auto put = [&](int plane, const uint32_t(&v)[8]) {
    *reinterpret_cast<uint4*>(to + plane * kDfFrag) =
        make_uint4(x3_pair(v[0], v[1]), x3_pair(v[2], v[3]), x3_pair(v[4], v[5]), x3_pair(v[6], v[7]));
  };
  put(0, h);
  put(1, m);
  put(2, l);
}

__global__ __launch_bounds__(256) void dense_planes_kernel(DensePlanesArgs a) {
  __shared__ float tile[32][kDfRank + 1];
  const int z = blockIdx.z, b = blockIdx.y, j0 = blockIdx.x * 32, tid = threadIdx.x;
  const float* src = a.proj[z] + ((int64_t)b * a.N + j0) * a.ld;
  for (int e = tid; e < 32 * kDfRank; e += 256) {
    const int j = e / kDfRank, k = e % kDfRank;
    tile[j][k] = j0 + j < a.N && k < a.r ? src[(int64_t)j * a.ld + k] : 0.f;
  }
  __syncthreads();
  const int64_t base = ((int64_t)b * a.Npad + j0) * kDfPlaneRow;
  float x[8];
  {  // thread: row j, ranks k .. k + 7
    const int j = tid / 8, k = tid % 8 * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = tile[j][k + i];
      if (z == 0) x[i] *= k + i < a.r ? a.scale[k + i] : 0.f;
    }
    df_store_planes(x, a.planes[z] + base + ((j / 16 * 2 + k / 32) * 3 * 64 + j % 16 + k % 32 / 8 * 16) * 8);
  }
  if (!a.blocks[z]) return;
  {  // thread: rank k, rows j .. j + 7
    const int k = tid / 4, j = tid % 4 * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = tile[j + i][k];
    df_store_planes(x, a.blocks[z] + base + (k / 16 * 3 * 64 + k % 16 + j / 8 * 16) * 8);
  }
}

// Value rows [b][j][D] into [b][Npad / 32][D / 16][64 lanes][8]: lane l of a
// 16-column tile holds column l % 16 of rows 8 (l / 16) .. + 7 (the A fragment
// of v_mfma_f32_16x16x32_bf16 with k along the rows).  A workgroup takes 32
// rows x 128 columns.
__global__ __launch_bounds__(256) void dense_pack_kernel(const bf16_t* val, bf16_t* out, int N, int Npad, int D) {
  __shared__ uint16_t tile[32][128 + 2];
  const int d0 = blockIdx.x * 128, j0 = blockIdx.y * 32, b = blockIdx.z, tid = threadIdx.x;
  const uint16_t* src = reinterpret_cast<const uint16_t*>(val) + ((int64_t)b * N + j0) * D + d0;
  for (int e = tid; e < 32 * 16; e += 256) {
    const int j = e / 16, c = e % 16 * 8;
    uint4 x = make_uint4(0, 0, 0, 0);
    if (j0 + j < N) x = *reinterpret_cast<const uint4*>(src + (int64_t)j * D + c);
    uint32_t* to = reinterpret_cast<uint32_t*>(&tile[j][c]);
    to[0] = x.x; to[1] = x.y; to[2] = x.z; to[3] = x.w;
  }
  __syncthreads();
  bf16_t* dst = out + (((int64_t)b * (Npad / 32) + blockIdx.y) * (D / 16) + d0 / 16) * 512;
  for (int e = tid; e < 8 * 64; e += 256) {
    const int t = e / 64, l = e % 64, c = t * 16 + (l & 15), j = l / 16 * 8;
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = (uint32_t)tile[j + 2 * q][c] | (uint32_t)tile[j + 2 * q + 1][c] << 16;
    *reinterpret_cast<uint4*>(dst + (int64_t)e * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// ---- shared pieces ---------------------------------------------------------------

// 1 / y to within an ulp (y in [1, inf))
__device__ __forceinline__ float recip_f(float y) {
  const float r = __builtin_amdgcn_rcpf(y);
  return r * (2.0f - y * r);
}

// c += a . b over one 32-wide K step of three-plane operands, the small terms first
__device__ __forceinline__ floatx4 mfma_x3(const bf16x8v (&a)[3], const bf16x8v (&b)[3], floatx4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], c, 0, 0, 0);
}

// which columns j row i keeps: all, j <= i, j >= i.  Causal kernels test without
// a branch (a branch per element splits the schedule of a whole step).
constexpr int kDfAll = 0, kDfLower = 1, kDfUpper = 2;
__device__ __forceinline__ bool df_keep(int mode, int i, int j) {
  return (mode == kDfLower ? i - j : j - i) >= 0;
}

// the workgroup's batch element and first row (longest column ranges first)
__device__ __forceinline__ void df_tile(int Npad, int rows, int mode, int& b, int& i0) {
  const int id = xcd_swizzle(blockIdx.x, gridDim.x), per = Npad / rows;
  b = id / per;
  const int t = id - b * per;
  i0 = (mode == kDfLower ? per - 1 - t : t) * rows;
}

// ---- E . V and E . x ---------------------------------------------------------------
struct DenseAggregateArgs {
  const bf16_t* rows;    // planes of the row operand (dense_planes_kernel)
  const bf16_t* cols;    // planes of the column operand
  const bf16_t* values;  // packed values of the columns (dense_pack_kernel)
  const float* bias;     // scalar or null
  const float* x;        // [nb][N] of the columns
  bf16_t* out;           // [nb][N][D] or null
  float* out_state;      // [nb][N] or null
  int N, Npad, D, mode;
};

// 64 columns per step.  Scores are taken transposed (columns on M, rows on N),
// so that a lane holds four consecutive columns of one row: its edges go to LDS
// as 8-byte pieces of the aggregate's B fragments, whose A operand (the packed
// values: every wave owns D / 8 columns of V) loads straight into fragments.
// Two buffers each for the column planes and the edges: one barrier per step,
// and a wave may run its scores beside another's aggregate.
// Bound: MFMA (per 128 x 64 edges and SIMD 1536 cycles of scores, 2048 of
// aggregate at D = 512) plus the softsign's VALU work.
template <int NTW, int KS, bool CAUSAL>
__global__ __launch_bounds__(kDfThreads) void dense_aggregate_kernel(DenseAggregateArgs a) {
  constexpr int CT = 64;
  __shared__ __align__(16) bf16_t planes[2][CT * kDfPlaneRow];  // [4 tiles][2][3] fragments
  __shared__ __align__(16) bf16_t edges[2][16 * kDfFrag];       // [8 row tiles][2] fragments
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int col = lane & 15, kg = lane >> 4;
  int b, i0;
  df_tile(a.Npad, kDfRows, a.mode, b, i0);
  const int jbeg = a.mode == kDfUpper ? i0 : 0;
  const int jend = a.mode == kDfLower ? min(a.N, i0 + kDfRows) : a.N;
  const float bias = a.bias ? a.bias[0] : 0.f;

  const int row = wave * 16 + col;  // of the scores
  bf16x8v q[KS][3];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int p = 0; p < 3; ++p)
      q[s][p] = *reinterpret_cast<const bf16x8v*>(
          a.rows + ((int64_t)b * a.Npad + i0 + wave * 16) * kDfPlaneRow + (s * 3 + p) * kDfFrag + lane * 8);

  const u32x4* cols = reinterpret_cast<const u32x4*>(a.cols + (int64_t)b * a.Npad * kDfPlaneRow);
  const auto rs_x = make_rsrc(a.x + (int64_t)b * a.N, (uint32_t)a.N * 4u);
  u32x4 stage[3];
  auto load = [&](int j0) {  // the planes of 64 rows are 24 KB in one piece
#pragma unroll
    for (int u = 0; u < 3; ++u) stage[u] = cols[(int64_t)j0 * (kDfPlaneRow / 8) + tid + kDfThreads * u];
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 3; ++u) reinterpret_cast<u32x4*>(planes[buf])[tid + kDfThreads * u] = stage[u];
  };

  floatx4 acc[NTW][8];
#pragma unroll
  for (int d = 0; d < NTW; ++d)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[d][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float rsum = 0.f;

  load(jbeg);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int j0 = jbeg; j0 < jend; j0 += CT, buf ^= 1) {
    const bool more = j0 + CT < jend;
    if (more) load(j0 + CT);
    bf16x8v v[2][NTW];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int d = 0; d < NTW; ++d)
        v[s][d] = *reinterpret_cast<const bf16x8v*>(
            a.values + (((int64_t)b * (a.Npad / 32) + j0 / 32 + s) * (a.D / 16) + wave * NTW + d) * 512 + lane * 8);

#pragma unroll
    for (int t = 0; t < 4; ++t) {  // 16 columns
      const int j = t * 16 + kg * 4;
      const float4 x = buf_load4(rs_x, (uint32_t)(j0 + j) * 4u);
      floatx4 sc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8v c[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          c[p] = *reinterpret_cast<const bf16x8v*>(&planes[buf][((t * 2 + s) * 3 + p) * kDfFrag + lane * 8]);
        sc = mfma_x3(c, q[s], sc);
      }
      float e[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float s = sc[w] + bias;
        e[w] = s * recip_f(1.0f + fabsf(s));
        if constexpr (CAUSAL) e[w] = df_keep(a.mode, i0 + row, j0 + j + w) ? e[w] : 0.f;
      }
      rsum += (e[0] * x.x + e[1] * x.y) + (e[2] * x.z + e[3] * x.w);
      *reinterpret_cast<uint2*>(&edges[buf][(wave * 2 + t / 2) * kDfFrag + (col + (t % 2 * 2 + kg / 2) * 16) * 8 +
                                            kg % 2 * 4]) =
          make_uint2(pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3]));
    }
    if (more) store(buf ^ 1);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bf16x8v e = *reinterpret_cast<const bf16x8v*>(&edges[buf][(i * 2 + s) * kDfFrag + lane * 8]);
#pragma unroll
        for (int d = 0; d < NTW; ++d)
          acc[d][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[s][d], e, acc[d][i], 0, 0, 0);
      }
    }
  }

#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int m = i0 + i * 16 + col;
    if (m >= a.N || !a.out) continue;
    bf16_t* out = a.out + ((int64_t)b * a.N + m) * a.D + wave * NTW * 16 + kg * 4;
#pragma unroll
    for (int d = 0; d < NTW; ++d)
      *reinterpret_cast<uint2*>(out + d * 16) =
          make_uint2(pack_bf16x2(acc[d][i][0], acc[d][i][1]), pack_bf16x2(acc[d][i][2], acc[d][i][3]));
  }
  rsum += xor16_f(rsum);
  rsum += xor32_f(rsum);
  if (a.out_state && kg == 0 && i0 + row < a.N) a.out_state[(int64_t)b * a.N + i0 + row] = rsum;
}

// ---- G . P ---------------------------------------------------------------------------
struct DenseScoreGradArgs {
  const bf16_t* rows;     // planes of the row operand (dense_planes_kernel)
  const bf16_t* cols;     // planes of the column operand
  const bf16_t* blocks;   // transposed planes of the columns' raw projections
  const bf16_t* row_val;  // [nb][N][D]
  const bf16_t* col_val;  // [nb][N][D]
  const float* row_x;     // [nb][N]
  const float* col_x;     // [nb][N]
  const float* bias;      // scalar or null
  const float* out_scale; // [r] or null
  float* out;             // [nb][N] rows of stride ld: r values each
  int64_t ld;
  float* rowsum;          // [nb][N] or null: sums of G over the columns
  int N, Npad, r, mode;
};

// 32 columns per step, everything transposed as above.  The rows' value
// fragments stay in registers (2 x D / 32 of them), their score planes in LDS;
// the columns' values are staged in LDS (pieces of a row exchanged by its row
// number, so that 16 rows' pieces lie in distinct banks), the columns' planes
// and transposed planes load straight into fragments.  64 rows per workgroup:
// 70 KB of LDS, so that two share a CU and one's barriers and LDS phases run
// beside the other's MFMAs (128 rows in one workgroup of eight waves: 1.03 ms
// against 0.90 at C4; in one of four waves of 32 x 32: 1.6).
// Bound: MFMA (per 128 x 32 pairs and SIMD 768 cycles of scores, 1024 of
// gdv . pv^T at D = 512, 768 of G . P), the VALU work of the derivative and of
// splitting G, and LDS reads (2200 cycles).
template <int NK, int KS, bool CAUSAL>
__global__ __launch_bounds__(kDfGradThreads, 2) void dense_score_grad_kernel(DenseScoreGradArgs a) {
  constexpr int D = NK * 32, CT = 32;
  __shared__ __align__(16) bf16_t qs[kDfGradRows * kDfPlaneRow];   // rows' planes: [4 tiles][2][3] fragments
  __shared__ __align__(16) bf16_t vals[CT * D];                    // columns' values: rows of swizzled pieces
  __shared__ __align__(16) bf16_t gs[kDfGradRows / 16 * 3 * kDfFrag];  // G: [4 row tiles][3] fragments
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int wr = wave >> 1, wc = wave & 1, col = lane & 15, kg = lane >> 4;
  int b, i0;
  df_tile(a.Npad, kDfGradRows, a.mode, b, i0);
  const int jbeg = a.mode == kDfUpper ? i0 : 0;
  const int jend = a.mode == kDfLower ? min(a.N, i0 + kDfGradRows) : a.N;
  const float bias = a.bias ? a.bias[0] : 0.f;

  const auto rs_rv = make_rsrc(a.row_val + (int64_t)b * a.N * D, (uint32_t)a.N * (D * 2u));
  const auto rs_cv = make_rsrc(a.col_val + (int64_t)b * a.N * D, (uint32_t)a.N * (D * 2u));
  const auto rs_rx = make_rsrc(a.row_x + (int64_t)b * a.N, (uint32_t)a.N * 4u);
  const auto rs_cx = make_rsrc(a.col_x + (int64_t)b * a.N, (uint32_t)a.N * 4u);
  auto load16 = [](__amdgpu_buffer_rsrc_t rs, uint32_t off) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
  };

  bf16x8v rv[2][NK];  // this wave's 32 rows of values
  float rx[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int i = i0 + wr * 32 + n * 16 + col;
    rx[n] = buf_load1(rs_rx, (uint32_t)i * 4u);
#pragma unroll
    for (int s = 0; s < NK; ++s)
      rv[n][s] = __builtin_bit_cast(bf16x8v, load16(rs_rv, (uint32_t)i * (D * 2u) + s * 64u + kg * 16u));
  }
  {
    const uint4* src = reinterpret_cast<const uint4*>(a.rows + ((int64_t)b * a.Npad + i0) * kDfPlaneRow);
    for (int e = tid; e < kDfGradRows * kDfPlaneRow / 8; e += kDfGradThreads) reinterpret_cast<uint4*>(qs)[e] = src[e];
  }

  constexpr int VN = CT * D / 8 / kDfGradThreads, VP = D / 8;  // 16-byte pieces: per thread of a tile, of a row
  u32x4 sv[VN];
  auto load = [&](int j0) {
#pragma unroll
    for (int u = 0; u < VN; ++u)
      sv[u] = load16(rs_cv, (uint32_t)j0 * (D * 2u) + (uint32_t)(tid + kDfGradThreads * u) * 16u);
  };
  auto store = [&]() {
#pragma unroll
    for (int u = 0; u < VN; ++u) {
      const int e = tid + kDfGradThreads * u, j = e / VP, p = e % VP;
      reinterpret_cast<u32x4*>(vals)[j * VP + (p ^ (j & 15))] = sv[u];
    }
  };

  floatx4 acc[2][2];  // 32 ranks (wc) x 32 rows
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
  float rsum[2] = {0.f, 0.f}, rpart[2] = {0.f, 0.f};
  const bf16_t* cols = a.cols + (int64_t)b * a.Npad * kDfPlaneRow + lane * 8;
  const bf16_t* blocks = a.blocks + (int64_t)b * a.Npad * kDfPlaneRow + lane * 8;

  load(jbeg);
  int step = 0;
  for (int j0 = jbeg; j0 < jend; j0 += CT, ++step) {
    __syncthreads();  // the step before is consumed
    store();
    __syncthreads();
    if (j0 + CT < jend) load(j0 + CT);
    const float4 cx = buf_load4(rs_cx, (uint32_t)(j0 + wc * 16 + kg * 4) * 4u);
    bf16x8v c[KS][3];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        c[s][p] = *reinterpret_cast<const bf16x8v*>(cols + (int64_t)(j0 + wc * 16) * kDfPlaneRow +
                                                    (s * 3 + p) * kDfFrag);

    // gdv . pv^T and the scores: 16 columns (wc) x 32 rows
    floatx4 sc[2], gv[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) sc[n] = gv[n] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const bf16x8v v =
          reinterpret_cast<const bf16x8v*>(vals)[(wc * 16 + col) * VP + ((s * 4 + kg) ^ col)];
#pragma unroll
      for (int n = 0; n < 2; ++n) gv[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, rv[n][s], gv[n], 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        bf16x8v q[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          q[p] = *reinterpret_cast<const bf16x8v*>(&qs[(((wr * 2 + n) * 2 + s) * 3 + p) * kDfFrag + lane * 8]);
        sc[n] = mfma_x3(c[s], q, sc[n]);
      }
    bf16x8v t[2][3];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        t[m][p] = *reinterpret_cast<const bf16x8v*>(blocks + (int64_t)j0 * kDfPlaneRow +
                                                    ((wc * 2 + m) * 3 + p) * kDfFrag);
    const float cxv[4] = {cx.x, cx.y, cx.z, cx.w};
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      uint32_t h[4], mi[4], l[4];
      float g[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float d = recip_f(1.0f + fabsf(sc[n][w] + bias));  // 1 - |softsign|
        g[w] = (gv[n][w] + rx[n] * cxv[w]) * d * d;
        if constexpr (CAUSAL)
          g[w] = df_keep(a.mode, i0 + wr * 32 + n * 16 + col, j0 + wc * 16 + kg * 4 + w) ? g[w] : 0.f;
        x3_split(__float_as_uint(g[w]), h[w], mi[w], l[w]);
      }
      rpart[n] += (g[0] + g[1]) + (g[2] + g[3]);
      bf16_t* to = &gs[(wr * 2 + n) * 3 * kDfFrag + (col + (wc * 2 + kg / 2) * 16) * 8 + kg % 2 * 4];
      *reinterpret_cast<uint2*>(to) = make_uint2(x3_pair(h[0], h[1]), x3_pair(h[2], h[3]));
      *reinterpret_cast<uint2*>(to + kDfFrag) = make_uint2(x3_pair(mi[0], mi[1]), x3_pair(mi[2], mi[3]));
      *reinterpret_cast<uint2*>(to + 2 * kDfFrag) = make_uint2(x3_pair(l[0], l[1]), x3_pair(l[2], l[3]));
    }
    if ((step & 7) == 7) {  // short partial sums: their rounding does not grow with N
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        rsum[n] += rpart[n];
        rpart[n] = 0.f;
      }
    }
    __syncthreads();
    // G . P: 32 ranks (wc) x 32 rows (wr) over the 32 columns
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      bf16x8v g[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        g[p] = *reinterpret_cast<const bf16x8v*>(&gs[((wr * 2 + n) * 3 + p) * kDfFrag + lane * 8]);
#pragma unroll
      for (int m = 0; m < 2; ++m) acc[m][n] = mfma_x3(t[m], g, acc[m][n]);
    }
  }

#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int row = i0 + wr * 32 + n * 16 + col;
    if (row >= a.N) continue;
    float* out = a.out + ((int64_t)b * a.N + row) * a.ld;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int k = wc * 32 + m * 16 + kg * 4 + w;
        if (k < a.r) out[k] = a.out_scale ? acc[m][n][w] * a.out_scale[k] : acc[m][n][w];
      }
  }
  if (!a.rowsum) return;
  __syncthreads();  // the rows' planes are no longer read
  float* state = reinterpret_cast<float*>(qs);
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    float s = rsum[n] + rpart[n];
    s += xor16_f(s);
    s += xor32_f(s);
    if (kg == 0) state[wc * kDfGradRows + wr * 32 + n * 16 + col] = s;
  }
  __syncthreads();
  if (tid < kDfGradRows && i0 + tid < a.N) a.rowsum[(int64_t)b * a.N + i0 + tid] = state[tid] + state[kDfGradRows + tid];
}

// ---- host ------------------------------------------------------------------------------
static int64_t df_npad(int64_t N) { return (N + kDfRows - 1) / kDfRows * kDfRows; }

// bytes of the operand layouts of one batch element (each 256-byte aligned by Npad's size)
static size_t df_element_bytes(int64_t N, int64_t D) {
  return (size_t)df_npad(N) * (4 * kDfPlaneRow * sizeof(bf16_t) + (size_t)D * sizeof(bf16_t));
}

// Whole 128-column pieces of value rows (at most 512: a wave's accumulators),
// one plane of ranks, 32-bit offsets, and scratch for a batch element at least.
int64_t dense_fused_batch(int64_t batch, int64_t N, int64_t D, int64_t r, int compress_kind, size_t scratch_bytes) {
  if (compress_kind != 0 || r > kDfRank || D % 128 != 0 || D > 512 || N < 128 || N * D * 2 >= (1LL << 31)) return 0;
  const int64_t fit = (int64_t)(scratch_bytes / df_element_bytes(N, D));
  const int64_t nb = std::min(batch, fit);
  return std::min<int64_t>(nb, 65535);
}

struct DenseLayouts {
  bf16_t* planes[2];  // targets (scaled), sources
  bf16_t* blocks[2];
  bf16_t* packed;
};

static DenseLayouts df_carve(void* scratch, int nb, int64_t Npad) {
  DenseLayouts l{};
  bf16_t* p = static_cast<bf16_t*>(scratch);
  const int64_t one = (int64_t)nb * Npad * kDfPlaneRow;
  l.planes[0] = p;
  l.planes[1] = p + one;
  l.blocks[0] = p + 2 * one;
  l.blocks[1] = p + 3 * one;
  l.packed = p + 4 * one;
  return l;
}

static bool df_aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

static int df_prepare(const DenseFused& f, const DenseLayouts& l, int Npad, const void* values, bool transposed,
                      hipStream_t stream) {
  JN_REQUIRE(df_aligned(values) && df_aligned(f.projected_val) && df_aligned(f.scratch) && df_aligned(f.delta_val) &&
                 df_aligned(f.grad_projected_val),
             kUnsupported, "bf16 dense layers need 16-byte aligned operands");
  DensePlanesArgs a{};
  a.proj[0] = f.projections;
  a.proj[1] = f.projections + f.r;
  a.ld = 2 * f.r;
  a.scale = f.core_weight;
  for (int z = 0; z < 2; ++z) {
    a.planes[z] = l.planes[z];
    a.blocks[z] = transposed ? l.blocks[z] : nullptr;
  }
  a.N = f.N;
  a.Npad = Npad;
  a.r = f.r;
  {
    JN_PROFILE("dense_planes_kernel", stream);
    hipLaunchKernelGGL(dense_planes_kernel, dim3(Npad / 32, f.nb, 2), dim3(256), 0, stream, a);
    JN_LAUNCH_CHECK();
  }
  JN_PROFILE("dense_pack_kernel", stream);
  hipLaunchKernelGGL(dense_pack_kernel, dim3(f.D / 128, Npad / 32, f.nb), dim3(256), 0, stream,
                     static_cast<const bf16_t*>(values), l.packed, f.N, Npad, f.D);
  JN_LAUNCH_CHECK();
  return kOk;
}

template <int NTW>
static void df_launch_aggregate(const DenseAggregateArgs& a, int nb, int r, hipStream_t stream) {
  const dim3 grid(nb * (a.Npad / kDfRows)), block(kDfThreads);
  const bool causal = a.mode != kDfAll;
  if (r <= 32 && causal) hipLaunchKernelGGL((dense_aggregate_kernel<NTW, 1, true>), grid, block, 0, stream, a);
  else if (r <= 32) hipLaunchKernelGGL((dense_aggregate_kernel<NTW, 1, false>), grid, block, 0, stream, a);
  else if (causal) hipLaunchKernelGGL((dense_aggregate_kernel<NTW, 2, true>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((dense_aggregate_kernel<NTW, 2, false>), grid, block, 0, stream, a);
}

static int df_aggregate(const DenseAggregateArgs& a, int nb, int r, const char* name, hipStream_t stream) {
  JN_PROFILE(name, stream);
  switch (a.D / 128) {
    case 1: df_launch_aggregate<1>(a, nb, r, stream); break;
    case 2: df_launch_aggregate<2>(a, nb, r, stream); break;
    case 3: df_launch_aggregate<3>(a, nb, r, stream); break;
    default: df_launch_aggregate<4>(a, nb, r, stream); break;
  }
  JN_LAUNCH_CHECK();
  return kOk;
}

template <int NK, int KS>
static int df_launch_score_grad(const DenseScoreGradArgs& a, int nb, hipStream_t stream) {
  const dim3 grid(nb * (a.Npad / kDfGradRows)), block(kDfGradThreads);
  if (a.mode != kDfAll) hipLaunchKernelGGL((dense_score_grad_kernel<NK, KS, true>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((dense_score_grad_kernel<NK, KS, false>), grid, block, 0, stream, a);
  JN_LAUNCH_CHECK();
  return kOk;
}

static int df_score_grad(const DenseScoreGradArgs& a, int nb, int D, const char* name, hipStream_t stream) {
  JN_PROFILE(name, stream);
  const bool one = a.r <= 32;
  switch (D / 128) {
    case 1: return one ? df_launch_score_grad<4, 1>(a, nb, stream) : df_launch_score_grad<4, 2>(a, nb, stream);
    case 2: return one ? df_launch_score_grad<8, 1>(a, nb, stream) : df_launch_score_grad<8, 2>(a, nb, stream);
    case 3: return one ? df_launch_score_grad<12, 1>(a, nb, stream) : df_launch_score_grad<12, 2>(a, nb, stream);
    default: return one ? df_launch_score_grad<16, 1>(a, nb, stream) : df_launch_score_grad<16, 2>(a, nb, stream);
  }
}

int launch_dense_fused_forward(const DenseFused& f, hipStream_t stream) {
  const int Npad = (int)df_npad(f.N);
  const DenseLayouts l = df_carve(f.scratch, f.nb, Npad);
  int rc = df_prepare(f, l, Npad, f.projected_val, false, stream);
  if (rc) return rc;
  DenseAggregateArgs a{};
  a.rows = l.planes[0];
  a.cols = l.planes[1];
  a.values = l.packed;
  a.bias = f.bias;
  a.x = f.projected_state;
  a.out = static_cast<bf16_t*>(f.delta_val);
  a.out_state = f.delta_state;
  a.N = f.N;
  a.Npad = Npad;
  a.D = f.D;
  a.mode = f.causal ? kDfLower : kDfAll;
  return df_aggregate(a, f.nb, f.r, "dense_aggregate_kernel<forward>", stream);
}

int launch_dense_fused_backward(const DenseFused& f, hipStream_t stream) {
  const int Npad = (int)df_npad(f.N);
  const DenseLayouts l = df_carve(f.scratch, f.nb, Npad);
  int rc = df_prepare(f, l, Npad, f.grad_delta_val, true, stream);
  if (rc) return rc;
  if (f.grad_projected_val || f.grad_projected_state) {
    DenseAggregateArgs a{};  // rows: sources; columns: targets
    a.rows = l.planes[1];
    a.cols = l.planes[0];
    a.values = l.packed;
    a.bias = f.bias;
    a.x = f.grad_delta_state;
    a.out = static_cast<bf16_t*>(f.grad_projected_val);
    a.out_state = f.grad_projected_state;
    a.N = f.N;
    a.Npad = Npad;
    a.D = f.D;
    a.mode = f.causal ? kDfUpper : kDfAll;
    rc = df_aggregate(a, f.nb, f.r, "dense_aggregate_kernel<value_grad>", stream);
    if (rc) return rc;
  }
  DenseScoreGradArgs g{};
  g.rows = l.planes[0];
  g.cols = l.planes[1];
  g.blocks = l.blocks[1];
  g.row_val = static_cast<const bf16_t*>(f.grad_delta_val);
  g.col_val = static_cast<const bf16_t*>(f.projected_val);
  g.row_x = f.grad_delta_state;
  g.col_x = f.projected_state;
  g.bias = f.bias;
  g.out_scale = f.core_weight;
  g.out = f.dP;
  g.ld = 2 * f.r;
  g.rowsum = f.rowsum;
  g.N = f.N;
  g.Npad = Npad;
  g.r = f.r;
  g.mode = f.causal ? kDfLower : kDfAll;
  rc = df_score_grad(g, f.nb, f.D, "dense_score_grad_kernel<target>", stream);
  if (rc) return rc;
  g.rows = l.planes[1];
  g.cols = l.planes[0];
  g.blocks = l.blocks[0];
  g.row_val = static_cast<const bf16_t*>(f.projected_val);
  g.col_val = static_cast<const bf16_t*>(f.grad_delta_val);
  g.row_x = f.projected_state;
  g.col_x = f.grad_delta_state;
  g.out_scale = nullptr;
  g.out = f.dP + f.r;
  g.rowsum = nullptr;
  g.mode = f.causal ? kDfUpper : kDfAll;
  return df_score_grad(g, f.nb, f.D, "dense_score_grad_kernel<source>", stream);
}

}  // namespace jakal
