// Projections of few rows (transitions, slot and query layers, one graph at a
// time): C[M][N] = X[M][K] . [W0; W1]^T with N = the ranks (up to a few
// hundred) and few enough rows (gemm_rows_fits) that tiles of 128 x 128 or 64 x
// 64 leave many of the 256 CUs idle and walk K behind two barriers per slice
// with one slice's latency exposed each time.
//
// Every wave is a worker of its own: it owns an output tile of MT x NT MFMA
// tiles and walks all of K in 32-wide slices -- whole lines into registers,
// DEPTH slices ahead, then into its own LDS region, from which it reads its
// MFMA fragments -- so there is no workgroup barrier at all.  (Fragments
// loaded straight from global memory cost a cache lookup per 16 bytes: slower
// from 4096 rows on.)  The four waves of a workgroup take neighbouring column
// tiles of the same rows, which they share in L1.
//
// The arithmetic of an element is that of the tile kernel it replaces, product
// for product in the same order, so results are bit-identical to it: top-k
// selections downstream do not change.
//   kX3    gemm_x3_kernel: six bf16 MFMAs per slice over three-term splits
//   kC4    gemm_f32_kernel: fp32 MFMAs, four chains summed at the end
//   kBf    gemm_bf16_kernel: bf16 operands
//   kC4Bf  gemm_f32_kernel on widened bf16 rows and bf16-rounded weights
//
// Bound: below some 4096 rows the chain of 16 slices (K = 512), each a load's
// latency and a dependent run of MFMAs; above, the splits' VALU work and the
// MFMAs.  Measured with the events' own 5 us, K = 512, against the tile kernel
// of the same arithmetic (its 64 x 64 tiles where the grid is small):
//                      three-term           bf16              fp32 MFMA (N = 64)
//   1024 x 128      19.8 -> 13.4 us    11.2 ->  9.1 us    12.8 -> 10.3 us
//   4096 x 128      20.3 -> 17.8       11.3 -> 11.7       13.2 -> 10.5
//   8192 x 128      21.0 -> 22.8       12.1 -> 14.2       17.0 -> 14.4
//   1024 x 512      20.5 -> 18.1       12.0 -> 11.7       (32,768: 37.6 -> 33.1)
//   1300 x 512      20.8 -> 22.2       11.7 -> 13.0
//   4096 x 512      25.7 -> 30.0       14.2 -> 18.3
//   16,384 x 512    56.5 -> 99         27   -> 43
#include "jn_internal.hpp"

namespace jakal {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));

constexpr int kRowsSlice = 32;

struct RowsGemmArgs {
  RowsGemm p[2];
  int blocks0;     // workgroups of p[0]; the rest run p[1]
  int tiles_n[2];  // column tiles of each product
};

template <int ARITH, int MT, int NT, int DEPTH>
__global__ __launch_bounds__(256) void gemm_rows_kernel(RowsGemmArgs args) {
  constexpr bool A_BF = ARITH == kRowsBf || ARITH == kRowsC4Bf;
  constexpr bool X3 = ARITH == kRowsX3, C4 = ARITH == kRowsC4 || ARITH == kRowsC4Bf;
  constexpr int KS = kRowsSlice;
  // a staged row of a slice and 16 bytes of padding (the fragment reads of 16
  // rows then hit distinct banks); X3 keeps its three planes in a row each
  constexpr int SB = KS * (C4 ? 4 : 2) + 16;
  constexpr int ROWS = (MT + NT) * 16, PLANE = ROWS * SB;
  __shared__ __align__(16) char smem[4][PLANE * (X3 ? 3 : 1)];

  const int second = (int)blockIdx.x >= args.blocks0 ? 1 : 0;
  const RowsGemm& g = args.p[second];
  const int lane = lane_id(), wave = wave_id();
  const int row = lane & 15, kg = lane >> 4;
  const int t = ((int)blockIdx.x - (second ? args.blocks0 : 0)) * 4 + wave;
  const int tn = args.tiles_n[second];
  const int m0 = t / tn * (MT * 16), n0 = t % tn * (NT * 16);
  if (m0 >= g.M) return;
  char* stage = smem[wave];

  // One load instruction of a slice covers 8 fp32 rows (8 lanes of 16 bytes
  // each) or 16 bf16 rows (4 lanes each).  Rows past the end read the last one
  // (their results are not stored).
  constexpr int AL = A_BF ? 4 : 8, AR = 64 / AL, AN = MT * 16 / AR, BN = NT * 2;
  const char* pa[AN];
  const float* pb[BN];
#pragma unroll
  for (int i = 0; i < AN; ++i) {
    const int64_t m = min(m0 + i * AR + lane / AL, g.M - 1);
    pa[i] = static_cast<const char*>(g.X) + m * g.ldx * (A_BF ? 2 : 4) + lane % AL * 16;
  }
#pragma unroll
  for (int i = 0; i < BN; ++i) {
    const int n = min(n0 + i * 8 + (lane >> 3), g.N - 1);
    pb[i] = (n < g.split ? g.W0 + (int64_t)n * g.ldw : g.W1 + (int64_t)(n - g.split) * g.ldw) + (lane & 7) * 4;
  }

  uint4 ra[DEPTH][AN], rb[DEPTH][BN];
  auto load = [&](int d, int s) {
    const int k0 = s * KS;
    if (k0 + KS <= g.K) {
#pragma unroll
      for (int i = 0; i < AN; ++i) ra[d][i] = *reinterpret_cast<const uint4*>(pa[i] + (int64_t)k0 * (A_BF ? 2 : 4));
#pragma unroll
      for (int i = 0; i < BN; ++i) rb[d][i] = *reinterpret_cast<const uint4*>(pb[i] + k0);
    } else {  // the last, partial slice: K is whole 16-byte loads, so a load is all inside or all outside
      const bool ina = k0 + lane % AL * (A_BF ? 8 : 4) < g.K, inb = k0 + (lane & 7) * 4 < g.K;
#pragma unroll
      for (int i = 0; i < AN; ++i)
        ra[d][i] = ina ? *reinterpret_cast<const uint4*>(pa[i] + (int64_t)k0 * (A_BF ? 2 : 4)) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < BN; ++i)
        rb[d][i] = inb ? *reinterpret_cast<const uint4*>(pb[i] + k0) : make_uint4(0, 0, 0, 0);
    }
  };

  // four consecutive fp32 elements k4 * 4 .. + 3 of a staged row
  auto store_f32 = [&](int r, int k4, uint4 x, bool round) {
    char* to = stage + r * SB;
    if constexpr (X3) {
      uint32_t h[4], m[4], l[4];
      x3_split(x.x, h[0], m[0], l[0]);
      x3_split(x.y, h[1], m[1], l[1]);
      x3_split(x.z, h[2], m[2], l[2]);
      x3_split(x.w, h[3], m[3], l[3]);
      to += k4 * 8;
      *reinterpret_cast<uint2*>(to) = make_uint2(x3_pair(h[0], h[1]), x3_pair(h[2], h[3]));
      *reinterpret_cast<uint2*>(to + PLANE) = make_uint2(x3_pair(m[0], m[1]), x3_pair(m[2], m[3]));
      *reinterpret_cast<uint2*>(to + 2 * PLANE) = make_uint2(x3_pair(l[0], l[1]), x3_pair(l[2], l[3]));
    } else {
      const float f[4] = {__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z), __uint_as_float(x.w)};
      if constexpr (ARITH == kRowsBf) {
        *reinterpret_cast<uint2*>(to + k4 * 8) = make_uint2(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]));
      } else {
        *reinterpret_cast<float4*>(to + k4 * 16) =
            round ? make_float4((float)(bf16_t)f[0], (float)(bf16_t)f[1], (float)(bf16_t)f[2], (float)(bf16_t)f[3])
                  : make_float4(f[0], f[1], f[2], f[3]);
      }
    }
  };
  auto store = [&](int d) {
#pragma unroll
    for (int i = 0; i < AN; ++i) {
      const int r = i * AR + lane / AL, c = lane % AL;
      if constexpr (ARITH == kRowsBf) {
        *reinterpret_cast<uint4*>(stage + r * SB + c * 16) = ra[d][i];
      } else if constexpr (ARITH == kRowsC4Bf) {
        const Pack<8> x = unpack16<bf16_t, 8>(ra[d][i]);
        float4* to = reinterpret_cast<float4*>(stage + r * SB + c * 32);
        to[0] = make_float4(x.v[0], x.v[1], x.v[2], x.v[3]);
        to[1] = make_float4(x.v[4], x.v[5], x.v[6], x.v[7]);
      } else {
        store_f32(r, c, ra[d][i], false);
      }
    }
#pragma unroll
    for (int i = 0; i < BN; ++i) store_f32(MT * 16 + i * 8 + (lane >> 3), lane & 7, rb[d][i], ARITH == kRowsC4Bf);
  };

  constexpr int CHAINS = C4 ? 4 : 1;
  floatx4 acc[MT][NT][CHAINS];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int c = 0; c < CHAINS; ++c) acc[i][j][c] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto multiply = [&]() {
    const char* fa = stage + row * SB + kg * 16;
    const char* fb = fa + MT * 16 * SB;
    if constexpr (C4) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float4 a[MT], b[NT];
#pragma unroll
        for (int i = 0; i < MT; ++i) a[i] = *reinterpret_cast<const float4*>(fa + i * 16 * SB + h * 64);
#pragma unroll
        for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const float4*>(fb + j * 16 * SB + h * 64);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            acc[i][j][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[j].x, acc[i][j][0], 0, 0, 0);
            acc[i][j][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[j].y, acc[i][j][1], 0, 0, 0);
            acc[i][j][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].z, b[j].z, acc[i][j][2], 0, 0, 0);
            acc[i][j][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].w, b[j].w, acc[i][j][3], 0, 0, 0);
          }
      }
    } else {
      constexpr int P = X3 ? 3 : 1;
      bf16x8v a[MT][P], b[NT][P];
#pragma unroll
      for (int p = 0; p < P; ++p) {
#pragma unroll
        for (int i = 0; i < MT; ++i) a[i][p] = *reinterpret_cast<const bf16x8v*>(fa + i * 16 * SB + p * PLANE);
#pragma unroll
        for (int j = 0; j < NT; ++j) b[j][p] = *reinterpret_cast<const bf16x8v*>(fb + j * 16 * SB + p * PLANE);
      }
      // (a plane, b plane) of each product, the small terms first; step by step
      // over the tiles, so that their chains overlap
      constexpr int STEPS = X3 ? 6 : 1;
      constexpr int pa_of[6] = {X3 ? 2 : 0, 0, 1, 1, 0, 0}, pb_of[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int q = 0; q < STEPS; ++q)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa_of[q] % P], b[j][pb_of[q] % P], acc[i][j][0],
                                                                   0, 0, 0);
    }
  };

  const int slices = (g.K + KS - 1) / KS;
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (d < slices) load(d, d);
  for (int s = 0; s < slices; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (s + d < slices) {
        wave_lds_sync();  // the slice before is read
        store(d);
        wave_lds_sync();
        if (s + d + DEPTH < slices) load(d, s + d + DEPTH);
        multiply();
      }
    }
  }

#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = m0 + i * 16 + kg * 4 + v, n = n0 + j * 16 + row;
        float x = acc[i][j][0][v];
        if constexpr (C4) x = (x + acc[i][j][1 % CHAINS][v]) + (acc[i][j][2 % CHAINS][v] + acc[i][j][3 % CHAINS][v]);
        if (m < g.M && n < g.N) g.C[(int64_t)m * g.ldc + n] = x;
      }
}

static int64_t rows_tiles(const RowsGemm& g) { return (int64_t)((g.M + 15) / 16) * ((g.N + 15) / 16); }

// Whether this kernel is the faster one.  A wave loads (and splits) its rows of X
// again for every column tile, so against the MFMA tile kernels the outputs
// count: up to 2048 tiles of 16 x 16 on three-term products, fewer on bf16 ones
// (level there, 11.7 against 11.3 us, and slower beyond).  Against
// gemm_f32_kernel, at any number of columns, the rows: 32,768, or 16,384 from
// 128 columns on (the largest measured), but for fp32 products that fill about
// three of its 64 x 64 tiles per CU, which run at their best there (K = 512 /
// 200: 16,384 x 130 47 / 27 us against 51 / 30 here, 12,288 x 194 49 / 27
// against 54 / 31, 8192 x 322 49 / 27 against 54 / 31, 24,576 x 114 49 / 28
// against 55 / 32; 24,576 x 82 only half fills them, 49 / 28 against 44 / 27;
// at other counts 2 to 40 % faster here).
static bool rows_few(const RowsGemm& g) {
  if (g.arith == kRowsX3) return rows_tiles(g) <= 2048;
  if (g.arith == kRowsBf) return rows_tiles(g) < 2048;
  if (g.arith == kRowsC4) {
    const int64_t t64 = (int64_t)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (t64 > 640 && t64 <= 768 && (int64_t)g.M * g.N * 3 > t64 * 64 * 64 * 2) return false;
  }
  return g.M <= (g.N >= 128 ? kRowsMaxM / 2 : kRowsMaxM);
}

// Whole 16-byte loads (K and the row strides in whole vectors, 16-byte aligned
// operands), few rows.
bool gemm_rows_fits(const RowsGemm& g) {
  const bool bf = g.arith == kRowsBf || g.arith == kRowsC4Bf;
  const int kv = bf ? 8 : 4;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  return g.M >= 1 && g.N >= 1 && g.K >= 1 && g.N <= kRowsMaxN && rows_few(g) && g.K % kv == 0 && g.ldx % kv == 0 &&
         g.ldw % 4 == 0 && al16(g.X) && al16(g.W0) && al16(g.W1);
}

template <int ARITH, int MT, int NT, int DEPTH>
static void launch_rows(const RowsGemm* p, int n, hipStream_t stream) {
  RowsGemmArgs a{};
  int blocks = 0;
  for (int i = 0; i < n; ++i) {
    a.p[i] = p[i];
    a.tiles_n[i] = (p[i].N + NT * 16 - 1) / (NT * 16);
    if (i == 1) a.blocks0 = blocks;
    blocks += ((p[i].M + MT * 16 - 1) / (MT * 16) * a.tiles_n[i] + 3) / 4;
  }
  if (n == 1) a.blocks0 = blocks;
  hipLaunchKernelGGL((gemm_rows_kernel<ARITH, MT, NT, DEPTH>), dim3(blocks), dim3(256), 0, stream, a);
}

template <int ARITH>
static void launch_rows_tile(const RowsGemm* p, int n, hipStream_t stream) {
  int64_t tiles = 0, waves = 0;  // of 16 x 16, and of 16 x 32
  for (int i = 0; i < n; ++i) {
    tiles += rows_tiles(p[i]);
    waves += (int64_t)((p[i].M + 15) / 16) * ((p[i].N + 31) / 32);
  }
  // the largest tile that still gives every SIMD (1024) two waves, 32 x 32 also
  // where 16 x 32 would make a fourth (K = 512: 30 us at 16,384 x 128 against 38
  // on 16 x 32, 32 at 16,384 x 98 against 39; 24,576 x 66, of 4.5 waves of 16 x
  // 32 each, 43 against 40).  The MFMA tile kernels take over before those.
  if constexpr (ARITH == kRowsC4 || ARITH == kRowsC4Bf) {
    if (tiles >= 8192 || (waves > 3 * 1024 && waves <= 4 * 1024)) return launch_rows<ARITH, 2, 2, 2>(p, n, stream);
  }
  if (tiles >= 2048) launch_rows<ARITH, 1, 2, 3>(p, n, stream);
  else launch_rows<ARITH, 1, 1, 4>(p, n, stream);
}

int launch_gemm_rows(const RowsGemm* p, int n, hipStream_t stream) {
  JN_REQUIRE(n == 1 || (n == 2 && p[0].arith == p[1].arith), kInvalidArgument, "rows GEMM takes one or two products");
  for (int i = 0; i < n; ++i)
    JN_REQUIRE(gemm_rows_fits(p[i]), kInvalidArgument, "operands do not fit the rows GEMM");
  const int arith = p[0].arith;
  JN_PROFILE(arith == kRowsX3 || arith == kRowsC4 ? "gemm_rows_kernel<project>" : "gemm_rows_kernel<project_bf16>",
             stream);
  if (arith == kRowsX3) launch_rows_tile<kRowsX3>(p, n, stream);
  else if (arith == kRowsC4) launch_rows_tile<kRowsC4>(p, n, stream);
  else if (arith == kRowsBf) launch_rows_tile<kRowsBf>(p, n, stream);
  else launch_rows_tile<kRowsC4Bf>(p, n, stream);
  JN_LAUNCH_CHECK();
  return kOk;
}

}  // namespace jakal
