// The projections' GEMMs in fp32 (fp32 models), for small products:
//   NT  C = A B^T  (A [M, K], B [N, K]),  NN  C = A B  (B [K, N]),  TN  C = A^T B  (A [K, M], B [K, N])
// with an optional residual added to the result, on v_mfma_f32_16x16x4_f32 (fp32
// products and sums).  Replaces F.linear of the layer's projections
// (femtotron/parallel/tensor_parallel/linear.py:66-80, 194-214 at one rank) where
// the library's choice for a product of a few hundred rows is a tile of its whole
// output on one CU (97 us for 256 x 512 x 256).
//
// A workgroup takes one 32 x 32 tile of C, its four waves every fourth k chunk of
// 16 each, so a 256 x 512 output is 128 workgroups of four waves; their sums meet
// in LDS in wave order.  Operands go straight from global memory (L1 / L2) into
// registers, the next chunk's loads before this chunk's 16 MFMAs: lane (r, c) =
// (i%16, i/16) holds row / column r of its 16, k's 4c .. 4c+3 of the chunk (one
// 16-byte load where k is contiguous, four 4-byte ones where it is the outer
// index), and product e contracts k's 4c + e.
#include "fh_common.hpp"
#include "fh_mfma.hpp"

namespace fh {
namespace {

constexpr int kF32Tile = 32, kF32Waves = 4, kF32Chunk = 16;

struct GemmF32Args {
  const float* a;
  const float* b;
  float* c;
  const float* r;  // residual, nullable
  int64_t lda, ldb, ldc, ldr;
  int m, n, k;
};

// k's kk .. kk+3 of operand row (KC) or column (KO) `i`; zeros past k.
template <bool KO>
__device__ __forceinline__ f32x4 load_k4(const float* p, int64_t ld, int i, int kk, int k) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (KO) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (kk + e < k) v[e] = p[static_cast<int64_t>(kk + e) * ld + i];
  } else {
    if (kk < k) v = *reinterpret_cast<const f32x4*>(p + static_cast<int64_t>(i) * ld + kk);  // k % 4 == 0
  }
  return v;
}

template <bool A_KO, bool B_KO>
__global__ __launch_bounds__(64 * kF32Waves) void k_gemm_f32(GemmF32Args g) {
  __shared__ __align__(16) float4 part[kF32Waves][4][64];
  const int lane = threadIdx.x & 63, r = lane & 15, c = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = blockIdx.y * kF32Tile, n0 = blockIdx.x * kF32Tile;
  // Rows and columns past the end re-read the last one; they are not stored.
  const int ra[2] = {min(m0 + r, g.m - 1), min(m0 + 16 + r, g.m - 1)};
  const int rb[2] = {min(n0 + r, g.n - 1), min(n0 + 16 + r, g.n - 1)};
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 fa[2], fb[2];
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fa[i] = load_k4<A_KO>(g.a, g.lda, ra[i], k0 + 4 * c, g.k);
      fb[i] = load_k4<B_KO>(g.b, g.ldb, rb[i], k0 + 4 * c, g.k);
    }
  };
  constexpr int STEP = kF32Waves * kF32Chunk;
  load(wave * kF32Chunk);
  for (int k0 = wave * kF32Chunk; k0 < g.k; k0 += STEP) {
    const f32x4 ca[2] = {fa[0], fa[1]}, cb[2] = {fb[0], fb[1]};
    load(k0 + STEP);  // zeros past k
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[i][e], cb[j][e], acc[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      part[wave][2 * i + j][lane] = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  __syncthreads();
  // Wave q sums quadrant q: rows 16 (q/2) + 4c + e, column 16 (q%2) + r.
  float4 s = part[0][wave][lane];
#pragma unroll
  for (int w = 1; w < kF32Waves; ++w) {
    const float4 v = part[w][wave][lane];
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  const float o[4] = {s.x, s.y, s.z, s.w};
  const int col = n0 + 16 * (wave & 1) + r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = m0 + 16 * (wave >> 1) + 4 * c + e;
    if (row < g.m && col < g.n) {
      const float add = g.r != nullptr ? g.r[row * g.ldr + col] : 0.f;
      g.c[row * g.ldc + col] = g.r != nullptr ? add + o[e] : o[e];
    }
  }
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" int fh_gemm_f32(int op, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
                           const void* residual, int64_t ldr, int64_t m, int64_t n, int64_t k,
                           hipStream_t stream) {
  FH_REQUIRE(op == FH_GEMM_NT || op == FH_GEMM_NN || op == FH_GEMM_TN,
             "gemm_f32: op must be FH_GEMM_NT, FH_GEMM_NN or FH_GEMM_TN");
  FH_REQUIRE(m > 0 && n > 0 && k > 0, "gemm_f32: sizes must be positive");
  FH_REQUIRE(m < (int64_t(1) << 20) && n < (int64_t(1) << 24) && k < (int64_t(1) << 30), "gemm_f32: sizes too large");
  const bool a_ko = op == FH_GEMM_TN, b_ko = op != FH_GEMM_NT;
  FH_REQUIRE(lda >= (a_ko ? m : k) && ldb >= (b_ko ? n : k) && ldc >= n, "gemm_f32: leading dims must cover the rows");
  FH_REQUIRE(a && b && c, "gemm_f32: null pointer");
  FH_REQUIRE(a_ko || (k % 4 == 0 && lda % 4 == 0 && aligned16(a)),
             "gemm_f32: a with k contiguous needs k % 4 == 0 and 16-byte aligned rows");
  FH_REQUIRE(b_ko || (k % 4 == 0 && ldb % 4 == 0 && aligned16(b)),
             "gemm_f32: b with k contiguous needs k % 4 == 0 and 16-byte aligned rows");
  FH_REQUIRE(!residual || (ldr >= n && (residual != c || ldr == ldc)),
             "gemm_f32: the residual must have ldr >= n, and c's when it is c");
  const GemmF32Args g{static_cast<const float*>(a), static_cast<const float*>(b), static_cast<float*>(c),
                      static_cast<const float*>(residual), lda, ldb, ldc, ldr, static_cast<int>(m),
                      static_cast<int>(n), static_cast<int>(k)};
  const dim3 grid(static_cast<unsigned>((n + kF32Tile - 1) / kF32Tile),
                  static_cast<unsigned>((m + kF32Tile - 1) / kF32Tile));
  const dim3 block(64 * kF32Waves);
  if (op == FH_GEMM_NT) hipLaunchKernelGGL((k_gemm_f32<false, false>), grid, block, 0, stream, g);
  else if (op == FH_GEMM_NN) hipLaunchKernelGGL((k_gemm_f32<false, true>), grid, block, 0, stream, g);
  else hipLaunchKernelGGL((k_gemm_f32<true, true>), grid, block, 0, stream, g);
  return check_launch("fh_gemm_f32");
}
