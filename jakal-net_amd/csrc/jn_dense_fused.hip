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
// Arithmetic: that of the GEMMs over an edge matrix (jn_gemm.hip), product for
// product and sum for sum, so a layer gives the same bits on either path (for
// ranks in multiples of 4; delta_state where N <= 16 D): the scores one chain of
// fp32 MFMAs over the ranks, E . V and gdv . pv^T on bf16 operands (E rounded
// to bf16 as it enters the product), G . P four chains of fp32 MFMAs, the row
// sums of E x and G in blocks of 32 columns, E^T . gds in sixteen chains.
//
// Measured at C4 sizes (16 x 4096 nodes, 512 values, rank 64, forward and
// backward) against the GEMMs over edge matrices in two batch chunks: step 5.48
// -> 3.19 ms; aggregate 0.62 and 0.60 ms, score gradient 0.97 and 0.95 ms.  An
// fp32 MFMA and vector instructions do not run side by side (33 cycles and 4.5
// for each of them, a bf16 MFMA 18 and little more for one or two), so vector
// work stands beside bf16 MFMAs or by itself.  The scores and G . P on
// three-term bf16 splits were faster (2.84 ms), but further from 64 bits on the
// same projections: delta_state 1.3 to 2.3 times as far as here, the projections'
// gradients 1.6 to 4.6 times, the score scale's 1.4 to 2.1 times.
//
// The operands are laid out by dense_ranks_kernel and dense_pack_kernel before:
// projections in fp32 MFMA fragment order, their transposes likewise, and value
// rows in bf16 fragment order.  Rows are padded to Npad (a multiple of 128) with
// zeros, which contribute nothing.
#include "jn_internal.hpp"

namespace jakal {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // (arrays of uint4 in flight go through scratch memory)

constexpr int kDfRows = 128;             // rows of an aggregate workgroup
constexpr int kDfThreads = 512;          // 8 waves of 16 rows (scores) or D / 8 columns (E . V)
constexpr int kDfGradRows = 64;          // rows of a score-gradient workgroup
constexpr int kDfGradThreads = 256;      // 4 waves of 16 rows
constexpr int kDfRank = 64;              // ranks of a laid-out row (zeros past the rank)
constexpr int kDfFrag = 512;             // elements of a bf16 MFMA fragment: 64 lanes of 8
constexpr int kDfFragF = 256;            // elements of four fp32 MFMA fragments: 64 lanes of 4
constexpr int kDfTile = 16 * kDfRank;    // elements of a 16-row tile of projections
constexpr int kDfBlock = 32;             // columns per partial row sum (dense_epi_parts)

// ---- operand layouts -----------------------------------------------------------

// Rows [b][j] of one projection (stride ld, r ranks) in fp32 MFMA fragment
// order, 16 rows at a time, so that a wave's load is one contiguous kilobyte in
// global memory and in LDS (no bank conflicts):
//   ranks [b][Npad / 16][4][64 lanes][4]: rows times scale (or 1); lane l holds
//     ranks 16 s + 4 (l / 16) .. + 3 of row l % 16;
//   cols [b][Npad / 16][4][64 lanes][4]: unscaled; lane l holds rows
//     4 (l / 16) .. + 3 of rank 16 s + l % 16.
// Element q of the lanes' four is the operand of the q-th MFMA (the k order of
// gemm_f32_kernel's fragments).  A workgroup takes 32 rows; blockIdx.z picks the
// projection (0: targets, with the scale; 1: sources).
struct DenseRanksArgs {
  const float* proj[2];
  int64_t ld;
  const float* scale;  // of proj[0]'s ranks
  float* ranks[2];
  float* cols[2];      // or null
  int N, Npad, r;
};

__global__ __launch_bounds__(256) void dense_ranks_kernel(DenseRanksArgs a) {
  __shared__ float tile[32][kDfRank + 1];
  const int z = blockIdx.z, b = blockIdx.y, j0 = blockIdx.x * 32, tid = threadIdx.x;
  const float* src = a.proj[z] + ((int64_t)b * a.N + j0) * a.ld;
  for (int e = tid; e < 32 * kDfRank; e += 256) {
    const int j = e / kDfRank, k = e % kDfRank;
    tile[j][k] = j0 + j < a.N && k < a.r ? src[(int64_t)j * a.ld + k] : 0.f;
  }
  __syncthreads();
  const int64_t base = ((int64_t)b * a.Npad + j0) * kDfRank;
#pragma unroll
  for (int u = 0; u < 2; ++u) {  // one 16-row tile each
    const int s = tid / 64, col = tid % 16, kg = tid % 64 / 16;
    const int64_t at = base + u * kDfTile + tid * 4;
    float x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = 16 * s + 4 * kg + q;
      x[q] = tile[u * 16 + col][k];
      if (z == 0) x[q] *= k < a.r ? a.scale[k] : 0.f;
    }
    *reinterpret_cast<float4*>(a.ranks[z] + at) = make_float4(x[0], x[1], x[2], x[3]);
    if (!a.cols[z]) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = tile[u * 16 + 4 * kg + q][16 * s + col];
    *reinterpret_cast<float4*>(a.cols[z] + at) = make_float4(x[0], x[1], x[2], x[3]);
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

// c += a . b over the 16 k of one laid-out piece (component q is MFMA q's)
__device__ __forceinline__ floatx4 mfma_f32x4(floatx4 a, floatx4 b, floatx4 c) {
#pragma unroll
  for (int q = 0; q < 4; ++q) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[q], c, 0, 0, 0);
  return c;
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

// a + b, never the tail of a fused multiply-add
__device__ __forceinline__ float df_add(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// the sum of v over the four lanes of a row (lanes l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ float df_row_sum(float v) {
  v += xor16_f(v);
  v += xor32_f(v);
  return v;
}

// ---- E . V and E . x ---------------------------------------------------------------
struct DenseAggregateArgs {
  const float* rows;     // ranks of the row operand (dense_ranks_kernel)
  const float* cols;     // ranks of the column operand
  const bf16_t* values;  // packed values of the columns (dense_pack_kernel)
  const float* bias;     // scalar or null
  const float* x;        // [nb][N] of the columns
  bf16_t* out;           // [nb][N][D] or null
  float* parts;          // forward: [nb][N][ceil(N / 32)], the sums of E x per 32 columns
  float* out_state;      // backward: [nb][N] or null
  int N, Npad, D, mode;
};

// 64 columns per step.  Scores are taken transposed (columns on M, rows on N),
// so that a lane holds four consecutive columns of one row: its edges go to LDS
// as 8-byte pieces of the aggregate's B fragments, whose A operand (the packed
// values: every wave owns D / 8 columns of V) loads straight into fragments.
// Two buffers each for the column ranks and the edges: one barrier per step,
// and a wave may run its scores beside another's aggregate.
// Bound: MFMA (per 128 x 64 edges and SIMD 4096 cycles of scores at rank 64,
// 2048 of aggregate at D = 512) plus the softsign's VALU work.
// KB: pieces of 16 ranks.  BWD: E . x in sixteen chains (colsum_rows_kernel's
// order), else in blocks of 32 columns (the order of the scores' epilogue).
template <int NTW, int KB, bool CAUSAL, bool BWD>
__global__ __launch_bounds__(kDfThreads) void dense_aggregate_kernel(DenseAggregateArgs a) {
  constexpr int CT = 64;
  __shared__ __align__(16) float ranks[2][4 * KB * kDfFragF];  // [4 tiles][KB] pieces
  __shared__ __align__(16) bf16_t edges[2][16 * kDfFrag];      // [8 row tiles][2] fragments
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int col = lane & 15, kg = lane >> 4;
  int b, i0;
  df_tile(a.Npad, kDfRows, a.mode, b, i0);
  const int jbeg = a.mode == kDfUpper ? i0 : 0;
  const int jend = a.mode == kDfLower ? min(a.N, i0 + kDfRows) : a.N;
  const float bias = a.bias ? a.bias[0] : 0.f;

  const int row = wave * 16 + col;  // of the scores
  floatx4 q[KB];
#pragma unroll
  for (int s = 0; s < KB; ++s)
    q[s] = *reinterpret_cast<const floatx4*>(a.rows + ((int64_t)b * a.Npad + i0 + wave * 16) * kDfRank +
                                             s * kDfFragF + lane * 4);

  // a step's column ranks: 4 tiles of 256 16-byte words, of which KB / 4 hold ranks
  constexpr int SN = 4 * KB * 64 / kDfThreads;
  const u32x4* cols = reinterpret_cast<const u32x4*>(a.cols + (int64_t)b * a.Npad * kDfRank);
  const auto rs_x = make_rsrc(a.x + (int64_t)b * a.N, (uint32_t)a.N * 4u);
  u32x4 stage[SN];
  auto load = [&](int j0) {
#pragma unroll
    for (int u = 0; u < SN; ++u) {
      const int e = tid + kDfThreads * u;
      stage[u] = cols[(int64_t)j0 * (kDfRank / 4) + e / (KB * 64) * (kDfTile / 4) + e % (KB * 64)];
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < SN; ++u) reinterpret_cast<u32x4*>(ranks[buf])[tid + kDfThreads * u] = stage[u];
  };

  floatx4 acc[NTW][8];
#pragma unroll
  for (int d = 0; d < NTW; ++d)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[d][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float chain[4] = {0.f, 0.f, 0.f, 0.f};  // BWD: columns 4 kg + w (mod 16)
  float hold = 0.f;                       // else: the sum of block 4 n + kg of the last four
  const int P = (a.N + kDfBlock - 1) / kDfBlock;

  __builtin_amdgcn_sched_barrier(0);  // the rows' ranks arrive before the loop
  load(jbeg);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int j0 = jbeg; j0 < jend; j0 += CT, buf ^= 1) {
    const bool more = j0 + CT < jend;
    float4 xs[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) xs[t] = buf_load4(rs_x, (uint32_t)(j0 + t * 16 + kg * 4) * 4u);
    bf16x8v v[2][NTW];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int d = 0; d < NTW; ++d)
        v[s][d] = *reinterpret_cast<const bf16x8v*>(
            a.values + (((int64_t)b * (a.Npad / 32) + j0 / 32 + s) * (a.D / 16) + wave * NTW + d) * 512 + lane * 8);

    load(more ? j0 + CT : j0);  // (the last step's again: a branch would make every wait one for all loads)
    __builtin_amdgcn_sched_barrier(0);
    float half = 0.f;
    auto scores = [&](int t) {  // 16 columns
      floatx4 c = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KB; ++s)
        c = mfma_f32x4(*reinterpret_cast<const floatx4*>(&ranks[buf][(t * KB + s) * kDfFragF + lane * 4]), q[s], c);
      return c;
    };
    floatx4 sc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) sc[t] = scores(t);
    __builtin_amdgcn_sched_barrier(0);  // (vector work among fp32 MFMAs runs beside none of them)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int j = t * 16 + kg * 4;
      const float4 x = xs[t];
      float e[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        e[w] = softsign_f(sc[t][w] + bias);
        if constexpr (CAUSAL) e[w] = df_keep(a.mode, i0 + row, j0 + j + w) ? e[w] : 0.f;
      }
      const float xv[4] = {x.x, x.y, x.z, x.w};
      if constexpr (BWD) {
#pragma unroll
        for (int w = 0; w < 4; ++w) chain[w] = fmaf(xv[w], e[w], chain[w]);
      } else {
        float p = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) p = fmaf(e[w], xv[w], p);
        p = df_row_sum(p);
        if (t % 2 == 0) {
          half = p;
        } else {
          const int blk = j0 / kDfBlock + t / 2;
          hold = (blk & 3) == kg ? half + p : hold;
        }
      }
      *reinterpret_cast<uint2*>(&edges[buf][(wave * 2 + t / 2) * kDfFrag + (col + (t % 2 * 2 + kg / 2) * 16) * 8 +
                                            kg % 2 * 4]) =
          make_uint2(pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3]));
    }
    if constexpr (!BWD) {
      if ((j0 & CT) != 0 || !more) {  // four blocks (or the last) are summed
        const int blk = (j0 / (2 * CT)) * 4 + kg;
        if (i0 + row < a.N && blk < P && blk * kDfBlock < j0 + CT)
          a.parts[((int64_t)b * a.N + i0 + row) * P + blk] = hold;
      }
    }
    store(buf ^ 1);
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
  if constexpr (BWD) {
    // the sixteen chains of a row in order: kg, then w
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float u = (((s + chain[0]) + chain[1]) + chain[2]) + chain[3];
      s = __shfl(u, col + 16 * g);
    }
    if (a.out_state && kg == 0 && i0 + row < a.N) a.out_state[(int64_t)b * a.N + i0 + row] = s;
  } else if constexpr (CAUSAL) {  // the blocks past the row's last column are empty
    if (i0 + row < a.N)
      for (int blk = (jend + kDfBlock - 1) / kDfBlock + kg; blk < P; blk += 4)
        a.parts[((int64_t)b * a.N + i0 + row) * P + blk] = 0.f;
  }
}

// ---- G . P ---------------------------------------------------------------------------
struct DenseScoreGradArgs {
  const float* rows;      // ranks of the row operand (dense_ranks_kernel)
  const float* cols;      // ranks of the column operand
  const float* proj;      // transposed raw projections of the columns (dense_ranks_kernel)
  const bf16_t* row_val;  // [nb][N][D]
  const bf16_t* col_val;  // [nb][N][D]
  const float* row_x;     // [nb][N]
  const float* col_x;     // [nb][N]
  const float* bias;      // scalar or null
  const float* out_scale; // [r] or null
  float* out;             // [nb][N] rows of stride ld: r values each
  int64_t ld;
  float* parts;           // [nb][N][ceil(N / 32)] or null: the sums of G per 32 columns
  int N, Npad, r, mode;
};

// 32 columns per step; a wave owns 16 rows and all of them.  Everything is taken
// transposed as above, so that the four columns of a row that a lane's G holds
// are component by component the operands of the four G . P chains: G never
// leaves its registers.  The rows' value fragments stay in registers; the
// columns' values (pieces of a row exchanged by its row number, so that 16 rows'
// pieces lie in distinct banks), ranks and transposed projections are staged in
// LDS.  64 rows per workgroup and 66 KB of LDS at D = 512: two share a CU, and
// one's barriers and LDS phases run beside the other's MFMAs.
// Bound: MFMA (per 64 x 32 pairs and SIMD 1024 cycles of scores and 1024 of
// G . P at rank 64, 512 of gdv . pv^T at D = 512) and LDS reads (1500 cycles).
template <int NK, int KB, bool CAUSAL>
__global__ __launch_bounds__(kDfGradThreads, 2) void dense_score_grad_kernel(DenseScoreGradArgs a) {
  constexpr int D = NK * 32, CT = 32;
  constexpr int VP = D / 8, VS = VP + 1;                       // 16-byte words of a row of values, and in LDS
  __shared__ __align__(16) u32x4 vals[CT * VS];                // columns' values (16 rows' words in distinct banks)
  __shared__ __align__(16) float ranks[2 * KB * kDfFragF];     // [2 tiles][KB] pieces
  __shared__ __align__(16) float proj[2 * KB * kDfFragF];
  // the rows' ranks: in registers, or in LDS where those would spill
  constexpr bool ROWS_LDS = NK == 16 && KB == 4;
  __shared__ __align__(16) float rows[ROWS_LDS ? kDfGradRows * kDfRank : 4];
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int col = lane & 15, kg = lane >> 4;
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

  const int row = i0 + wave * 16 + col;
  bf16x8v rv[NK];  // this lane's pieces of its row of values
#pragma unroll
  for (int s = 0; s < NK; ++s)
    rv[s] = __builtin_bit_cast(bf16x8v, load16(rs_rv, (uint32_t)row * (D * 2u) + s * 64u + kg * 16u));
  const float rx = buf_load1(rs_rx, (uint32_t)row * 4u);
  floatx4 qr[KB];
  floatx4* ql = reinterpret_cast<floatx4*>(rows) + (ROWS_LDS ? wave * KB * 64 : 0);  // this wave's, own to it
#pragma unroll
  for (int s = 0; s < KB; ++s) {
    qr[s] = *reinterpret_cast<const floatx4*>(a.rows + ((int64_t)b * a.Npad + i0 + wave * 16) * kDfRank +
                                              s * kDfFragF + lane * 4);
    if constexpr (ROWS_LDS) ql[s * 64 + lane] = qr[s];
  }

  // 16-byte words per thread of a step's values, and of its two tiles of 256
  // words of ranks and projections, of which KB / 4 are in use
  constexpr int VN = CT * VP / kDfGradThreads, RN = 2 * KB * 64 / kDfGradThreads;
  const uint32_t operand = (uint32_t)a.Npad * (kDfRank * 4u);
  const auto rs_c = make_rsrc(a.cols + (int64_t)b * a.Npad * kDfRank, operand);
  const auto rs_p = make_rsrc(a.proj + (int64_t)b * a.Npad * kDfRank, operand);
  u32x4 sv[VN], sc[RN], sp[RN];
  auto load = [&](int j0) {
#pragma unroll
    for (int u = 0; u < VN; ++u)
      sv[u] = load16(rs_cv, (uint32_t)j0 * (D * 2u) + (uint32_t)(tid + kDfGradThreads * u) * 16u);
#pragma unroll
    for (int u = 0; u < RN; ++u) {
      const int tile = kDfGradThreads * u / (KB * 64);  // (wave-uniform: KB is 4, or RN is 1 and the tile tid / 128)
      const uint32_t off = KB == 4 ? (uint32_t)tid * 16u : (uint32_t)(tid / 128 * 256 + tid % 128) * 16u;
      const uint32_t at = (uint32_t)j0 * (kDfRank * 4u) + (uint32_t)tile * (kDfTile * 4u);
      sc[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_c, off, at, 0));
      sp[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_p, off, at, 0));
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int u = 0; u < VN; ++u) {
      const int e = tid + kDfGradThreads * u;
      vals[e / VP * VS + e % VP] = sv[u];
    }
#pragma unroll
    for (int u = 0; u < RN; ++u) {
      reinterpret_cast<u32x4*>(ranks)[tid + kDfGradThreads * u] = sc[u];
      reinterpret_cast<u32x4*>(proj)[tid + kDfGradThreads * u] = sp[u];
    }
  };

  floatx4 acc[KB][4];  // 16 ranks x 16 rows, four chains
#pragma unroll
  for (int m = 0; m < KB; ++m)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[m][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  float hold = 0.f;  // the sum of block 4 n + kg of the last four
  const int P = (a.N + kDfBlock - 1) / kDfBlock;
  float* parts = a.parts && row < a.N ? a.parts + ((int64_t)b * a.N + row) * P : nullptr;

  load(jbeg);
  for (int j0 = jbeg; j0 < jend; j0 += CT) {
    __syncthreads();  // the step before is consumed
    store();
    __syncthreads();
    const bool more = j0 + CT < jend;
    float4 cx[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) cx[t] = buf_load4(rs_cx, (uint32_t)(j0 + t * 16 + kg * 4) * 4u);
    load(more ? j0 + CT : j0);  // (the last step's again: a branch would make every wait one for all loads)
    __builtin_amdgcn_sched_barrier(0);

    // the scores of 2 x 16 columns x 16 rows, and gdv . pv^T
    auto scores = [&](int t) {
      floatx4 c = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KB; ++s)
        c = mfma_f32x4(*reinterpret_cast<const floatx4*>(&ranks[(t * KB + s) * kDfFragF + lane * 4]),
                       ROWS_LDS ? ql[s * 64 + lane] : qr[s], c);
      return c;
    };
    auto slope = [&](floatx4 c) {  // 1 - |edge|
#pragma unroll
      for (int w = 0; w < 4; ++w) c[w] = 1.0f - fabsf(softsign_f(c[w] + bias));
      return c;
    };
    floatx4 g[2], d[2];
    d[0] = scores(0);
    d[1] = scores(1);
    __builtin_amdgcn_sched_barrier(0);
    g[0] = g[1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NK; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        g[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8v, vals[(t * 16 + col) * VS + s * 4 + kg]), rv[s], g[t], 0, 0, 0);
    d[0] = slope(d[0]);
    d[1] = slope(d[1]);
    // four reads ahead of the MFMAs, the slopes beside them
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // LDS reads
#pragma unroll
    for (int i = 0; i < 2 * NK - 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const float cxv[4] = {cx[t].x, cx[t].y, cx[t].z, cx[t].w};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float x = fmaf(rx, cxv[w], g[t][w]) * d[t][w] * d[t][w];
        if constexpr (CAUSAL) x = df_keep(a.mode, row, j0 + t * 16 + kg * 4 + w) ? x : 0.f;
        g[t][w] = x;
      }
    }
    if (a.parts) {  // the row's sum over the block, in the order of the score gradient's epilogue
      float s[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) s[w] = df_add(g[0][w], g[1][w]);
      const float sum = df_row_sum(df_add(df_add(s[0], s[1]), df_add(s[2], s[3])));
      const int blk = j0 / kDfBlock;
      hold = (blk & 3) == kg ? sum : hold;
      if (parts && ((blk & 3) == 3 || !more) && (blk & ~3) + kg <= blk) parts[(blk & ~3) + kg] = hold;
    }
    // G . P: all ranks x 16 rows over the 32 columns
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < KB; ++m) {
        const floatx4 p = *reinterpret_cast<const floatx4*>(&proj[(t * KB + m) * kDfFragF + lane * 4]);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[c], g[t][c], acc[m][c], 0, 0, 0);
      }
  }

  if (row < a.N) {
    float* out = a.out + ((int64_t)b * a.N + row) * a.ld;
#pragma unroll
    for (int m = 0; m < KB; ++m)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int k = m * 16 + kg * 4 + w;
        const float x = (acc[m][0][w] + acc[m][1][w]) + (acc[m][2][w] + acc[m][3][w]);
        if (k < a.r) out[k] = a.out_scale ? x * a.out_scale[k] : x;
      }
  }
  if constexpr (CAUSAL) {  // the blocks past the row's last column are empty
    if (parts)
      for (int blk = (jend + kDfBlock - 1) / kDfBlock + kg; blk < P; blk += 4) parts[blk] = 0.f;
  }
}

// ---- host ------------------------------------------------------------------------------
static int64_t df_npad(int64_t N) { return (N + kDfRows - 1) / kDfRows * kDfRows; }

// bytes of one batch element's layouts (a multiple of 256): the ranks of both
// projections, the packed values, and the transposed projections (backward) or
// the partial state sums (forward)
size_t dense_fused_element_bytes(int64_t N, int64_t D) {
  const size_t rows = (size_t)df_npad(N), ranks = 2 * kDfRank * sizeof(float);
  return rows * (ranks + (size_t)D * sizeof(bf16_t)) +
         std::max(rows * ranks, rows * dense_epi_parts((int)N) * sizeof(float));
}

// The layers these kernels serve: whole 128-column pieces of value rows (at most
// 512: a wave's accumulators), up to 64 ranks, 32-bit offsets, at least 512 nodes
// (the smallest measured), and layouts no larger than the edge matrix, whose
// buffer holds them.
bool dense_fused_serves(int64_t N, int64_t D, int64_t r, int compress_kind) {
  return compress_kind == 0 && r <= kDfRank && D % 128 == 0 && D <= 512 && N >= 512 && N * D * 2 < (1LL << 31) &&
         (size_t)N * N * sizeof(float) >= dense_fused_element_bytes(N, D);
}

// Whether a launch of that many aggregate workgroups (128 rows) is the faster
// path.  A workgroup walks all columns by itself, so a small grid takes as long
// as a full one, where the GEMMs over an edge matrix spread over the chip; they
// gain a little more from causal ranges.  Forward / step in us, without and with
// an edge matrix (rank 64; every width and rank measured on the line at 512 to
// 4096 nodes is the faster or within 2 % of it, but for the forward of 4 x 4096
// nodes with 256 values and rank 40, 302 against 278, whose step is 1102 against
// 1321):
//                          512 values                  128 values
//    4 x 1024   (32)  112 /  384,  68 /  282     89 /  312,  57 /  263
//   16 x 1024  (128)  125 /  422, 121 /  443     98 /  330,  81 /  336
//   24 x 1024  (192)  124 /  533, 161 /  593     98 /  412, 102 /  423
//     causal          126 /  558, 150 /  572    101 /  415,  95 /  411
//   64 x 512   (256)  102 /  393, 125 /  438     74 /  285,  82 /  312
//    1 x 4096   (32)  318 / 1196, 131 /  762    265 /  991, 130 /  726
//    4 x 4096  (128)  331 / 1234, 357 / 1488    268 / 1014, 316 / 1232
//     causal          339 / 1443, 300 / 1350    284 / 1046, 291 / 1157
//    6 x 4096  (192)  346 / 1603, 524 / 2121    284 / 1301, 459 / 1751
//     causal          346 / 1602, 406 / 1887    286 / 1188, 390 / 1607
static bool df_fills(int64_t blocks, int64_t N, int64_t D, bool causal) {
  if (blocks >= 256) return true;
  if (blocks >= 192) return D >= 256 || N >= 2560;
  return blocks >= 128 && N >= 3000 && !causal;
}

int64_t dense_fused_batch(int64_t batch, int64_t N, int64_t D, int64_t r, int compress_kind, bool causal,
                          size_t scratch_bytes) {
  if (batch < 1 || !dense_fused_serves(N, D, r, compress_kind)) return 0;
  const int64_t fit = std::min<int64_t>((int64_t)(scratch_bytes / dense_fused_element_bytes(N, D)), 65535);
  if (fit < 1) return 0;
  const int64_t launches = (batch + fit - 1) / fit;
  const int64_t nb = (batch + launches - 1) / launches;  // an even share each
  return df_fills(nb * (df_npad(N) / kDfRows), N, D, causal) ? nb : 0;
}

struct DenseLayouts {
  float* ranks[2];  // targets (scaled), sources
  float* cols[2];   // backward
  float* parts;     // forward: in the place of cols
  bf16_t* packed;
};

static DenseLayouts df_carve(void* scratch, int nb, int64_t Npad, int64_t D) {
  DenseLayouts l{};
  float* p = static_cast<float*>(scratch);
  const int64_t one = (int64_t)nb * Npad * kDfRank;
  l.ranks[0] = p;
  l.ranks[1] = p + one;
  l.packed = reinterpret_cast<bf16_t*>(p + 2 * one);
  l.parts = p + 2 * one + (int64_t)nb * Npad * D / 2;
  l.cols[0] = l.parts;
  l.cols[1] = l.parts + one;
  return l;
}

static bool df_aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

static int df_prepare(const DenseFused& f, const DenseLayouts& l, int Npad, const void* values, bool transposed,
                      hipStream_t stream) {
  JN_REQUIRE(df_aligned(values) && df_aligned(f.projected_val) && df_aligned(f.scratch) && df_aligned(f.delta_val) &&
                 df_aligned(f.grad_projected_val),
             kUnsupported, "bf16 dense layers need 16-byte aligned operands");
  DenseRanksArgs a{};
  a.proj[0] = f.projections;
  a.proj[1] = f.projections + f.r;
  a.ld = 2 * f.r;
  a.scale = f.core_weight;
  for (int z = 0; z < 2; ++z) {
    a.ranks[z] = l.ranks[z];
    a.cols[z] = transposed ? l.cols[z] : nullptr;
  }
  a.N = f.N;
  a.Npad = Npad;
  a.r = f.r;
  {
    JN_PROFILE("dense_ranks_kernel", stream);
    hipLaunchKernelGGL(dense_ranks_kernel, dim3(Npad / 32, f.nb, 2), dim3(256), 0, stream, a);
    JN_LAUNCH_CHECK();
  }
  JN_PROFILE("dense_pack_kernel", stream);
  hipLaunchKernelGGL(dense_pack_kernel, dim3(f.D / 128, Npad / 32, f.nb), dim3(256), 0, stream,
                     static_cast<const bf16_t*>(values), l.packed, f.N, Npad, f.D);
  JN_LAUNCH_CHECK();
  return kOk;
}

template <int NTW, int KB>
static void df_launch_aggregate(const DenseAggregateArgs& a, int nb, bool backward, hipStream_t stream) {
  const dim3 grid(nb * (a.Npad / kDfRows)), block(kDfThreads);
  const bool causal = a.mode != kDfAll;
  if (backward && causal) hipLaunchKernelGGL((dense_aggregate_kernel<NTW, KB, true, true>), grid, block, 0, stream, a);
  else if (backward) hipLaunchKernelGGL((dense_aggregate_kernel<NTW, KB, false, true>), grid, block, 0, stream, a);
  else if (causal) hipLaunchKernelGGL((dense_aggregate_kernel<NTW, KB, true, false>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((dense_aggregate_kernel<NTW, KB, false, false>), grid, block, 0, stream, a);
}

static int df_aggregate(const DenseAggregateArgs& a, int nb, int r, bool backward, const char* name,
                        hipStream_t stream) {
  JN_PROFILE(name, stream);
  const bool low = r <= 32;
  switch (a.D / 128) {
    case 1: (low ? df_launch_aggregate<1, 2> : df_launch_aggregate<1, 4>)(a, nb, backward, stream); break;
    case 2: (low ? df_launch_aggregate<2, 2> : df_launch_aggregate<2, 4>)(a, nb, backward, stream); break;
    case 3: (low ? df_launch_aggregate<3, 2> : df_launch_aggregate<3, 4>)(a, nb, backward, stream); break;
    default: (low ? df_launch_aggregate<4, 2> : df_launch_aggregate<4, 4>)(a, nb, backward, stream); break;
  }
  JN_LAUNCH_CHECK();
  return kOk;
}

template <int NK, int KB>
static int df_launch_score_grad(const DenseScoreGradArgs& a, int nb, hipStream_t stream) {
  const dim3 grid(nb * (a.Npad / kDfGradRows)), block(kDfGradThreads);
  if (a.mode != kDfAll) hipLaunchKernelGGL((dense_score_grad_kernel<NK, KB, true>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((dense_score_grad_kernel<NK, KB, false>), grid, block, 0, stream, a);
  JN_LAUNCH_CHECK();
  return kOk;
}

static int df_score_grad(const DenseScoreGradArgs& a, int nb, int D, const char* name, hipStream_t stream) {
  JN_PROFILE(name, stream);
  const bool low = a.r <= 32;
  switch (D / 128) {
    case 1: return low ? df_launch_score_grad<4, 2>(a, nb, stream) : df_launch_score_grad<4, 4>(a, nb, stream);
    case 2: return low ? df_launch_score_grad<8, 2>(a, nb, stream) : df_launch_score_grad<8, 4>(a, nb, stream);
    case 3: return low ? df_launch_score_grad<12, 2>(a, nb, stream) : df_launch_score_grad<12, 4>(a, nb, stream);
    default: return low ? df_launch_score_grad<16, 2>(a, nb, stream) : df_launch_score_grad<16, 4>(a, nb, stream);
  }
}

int launch_dense_fused_forward(const DenseFused& f, hipStream_t stream) {
  const int Npad = (int)df_npad(f.N);
  const DenseLayouts l = df_carve(f.scratch, f.nb, Npad, f.D);
  int rc = df_prepare(f, l, Npad, f.projected_val, false, stream);
  if (rc) return rc;
  DenseAggregateArgs a{};
  a.rows = l.ranks[0];
  a.cols = l.ranks[1];
  a.values = l.packed;
  a.bias = f.bias;
  a.x = f.projected_state;
  a.out = static_cast<bf16_t*>(f.delta_val);
  a.parts = l.parts;
  a.N = f.N;
  a.Npad = Npad;
  a.D = f.D;
  a.mode = f.causal ? kDfLower : kDfAll;
  rc = df_aggregate(a, f.nb, f.r, false, "dense_aggregate_kernel<forward>", stream);
  if (rc) return rc;
  return launch_dense_part_rowsum(l.parts, dense_epi_parts(f.N), (int64_t)f.nb * f.N, f.delta_state, stream);
}

int launch_dense_fused_backward(const DenseFused& f, hipStream_t stream) {
  const int Npad = (int)df_npad(f.N);
  const DenseLayouts l = df_carve(f.scratch, f.nb, Npad, f.D);
  int rc = df_prepare(f, l, Npad, f.grad_delta_val, true, stream);
  if (rc) return rc;
  if (f.grad_projected_val || f.grad_projected_state) {
    DenseAggregateArgs a{};  // rows: sources; columns: targets
    a.rows = l.ranks[1];
    a.cols = l.ranks[0];
    a.values = l.packed;
    a.bias = f.bias;
    a.x = f.grad_delta_state;
    a.out = static_cast<bf16_t*>(f.grad_projected_val);
    a.out_state = f.grad_projected_state;
    a.N = f.N;
    a.Npad = Npad;
    a.D = f.D;
    a.mode = f.causal ? kDfUpper : kDfAll;
    rc = df_aggregate(a, f.nb, f.r, true, "dense_aggregate_kernel<value_grad>", stream);
    if (rc) return rc;
  }
  DenseScoreGradArgs g{};
  g.rows = l.ranks[0];
  g.cols = l.ranks[1];
  g.proj = l.cols[1];
  g.row_val = static_cast<const bf16_t*>(f.grad_delta_val);
  g.col_val = static_cast<const bf16_t*>(f.projected_val);
  g.row_x = f.grad_delta_state;
  g.col_x = f.projected_state;
  g.bias = f.bias;
  g.out_scale = f.core_weight;
  g.out = f.dP;
  g.ld = 2 * f.r;
  g.parts = f.rowsum;
  g.N = f.N;
  g.Npad = Npad;
  g.r = f.r;
  g.mode = f.causal ? kDfLower : kDfAll;
  rc = df_score_grad(g, f.nb, f.D, "dense_score_grad_kernel<target>", stream);
  if (rc) return rc;
  g.rows = l.ranks[1];
  g.cols = l.ranks[0];
  g.proj = l.cols[0];
  g.row_val = static_cast<const bf16_t*>(f.projected_val);
  g.col_val = static_cast<const bf16_t*>(f.grad_delta_val);
  g.row_x = f.projected_state;
  g.col_x = f.grad_delta_state;
  g.out_scale = nullptr;
  g.out = f.dP + f.r;
  g.parts = nullptr;
  g.mode = f.causal ? kDfUpper : kDfAll;
  return df_score_grad(g, f.nb, f.D, "dense_score_grad_kernel<source>", stream);
}

}  // namespace jakal
