// The layer's gate projections of a prefill (or any step that does not take
// the fused decode input side): b = x w_b^T and a = x w_a^T, 32 columns each.
//
// As two library GEMMs these take 10.4 us each at 2000 rows of 2048: 32
// columns give such a GEMM little to do, and each reads all of x.  Here one
// workgroup of 8 waves takes 16 RT rows and 16 CT of the 64 columns, its waves
// splitting K: a wave multiplies its K / 8 of the rows with its K / 8 of the
// weights on MFMA, operands straight from memory in the fragments' layout
// (16 bytes per lane), and the waves' partial products meet in LDS and are
// added in wave order, in fp32, and rounded once.  Bound: the bytes a CU
// brings in (64 CT KiB of weights, from L2, and 64 RT KiB of x).  A whole layer
// prefill, eager, 1 x 20 / 1 x 500 / 1 x 2000 / 1 x 4096 tokens with the modules and
// with this 165 / 170 / 238 / 399 and 124 / 127 / 226 / 389 us.
#include "gdn_common.h"
#include "gdn_gate_proj.h"

namespace gdn {
namespace {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int GP_WAVES = 8;

// KS: k-steps of 32 per wave (K = 256 KS); CT: column tiles of 16 per
// workgroup (of the 2 N / 16 of both weights, b's first); RT: row tiles of 16
template <int KS, int CT, int RT>
__global__ __launch_bounds__(64 * GP_WAVES) __attribute__((amdgpu_waves_per_eu(2, 2))) void gate_proj_kernel(const uint16_t *x, const uint16_t *wb,
                                                                  const uint16_t *wa, int M, int N, uint16_t *b, uint16_t *a) {
  constexpr int K = 32 * KS * GP_WAVES, TILES = RT * CT;
  __shared__ f32x4_t part[GP_WAVES][TILES][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int row0 = static_cast<int>(blockIdx.x) * 16 * RT;
  const int k0 = wave * 32 * KS + 8 * g;
  const uint16_t *xp[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)  // (rows past the end: the last one again, not stored)
    xp[t] = x + static_cast<int64_t>(min(row0 + 16 * t + r, M - 1)) * K + k0;
  const uint16_t *wp[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int col = 16 * (static_cast<int>(blockIdx.y) * CT + c);
    wp[c] = (col < N ? wb + col * K : wa + (col - N) * K) + r * K + k0;
  }
  f32x4_t acc[TILES];
#pragma unroll
  for (int i = 0; i < TILES; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // GS k-steps' operands at a time, two groups in flight (for 16 and 32 rows
  // all of the wave's)
  constexpr int GS = KS / (RT == 4 ? 4 : 2), NG = KS / GS;
  u32x4_t xv[2][GS][RT], wv[2][GS][CT];
  auto load = [&](int i) {
#pragma unroll
    for (int s = 0; s < GS; ++s) {
#pragma unroll
      for (int t = 0; t < RT; ++t) xv[i & 1][s][t] = *reinterpret_cast<const u32x4_t *>(xp[t] + 32 * (i * GS + s));
#pragma unroll
      for (int c = 0; c < CT; ++c)
        wv[i & 1][s][c] = *reinterpret_cast<const u32x4_t *>(wp[c] + 32 * (i * GS + s));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  load(0);
  load(1);
#pragma unroll
  for (int i = 0; i < NG; ++i) {
#pragma unroll
    for (int s = 0; s < GS; ++s)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          acc[t * CT + c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, wv[i & 1][s][c]), __builtin_bit_cast(bf16x8_t, xv[i & 1][s][t]),
              acc[t * CT + c], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (i + 2 < NG) load(i + 2);
  }
#pragma unroll
  for (int i = 0; i < TILES; ++i) part[wave][i][lane] = acc[i];
  __syncthreads();
  // lane (r, g) of a tile: columns 4 g .. + 3 of row r
  for (int i = wave; i < TILES; i += GP_WAVES) {
    f32x4_t sum = part[0][i][lane];
#pragma unroll
    for (int w = 1; w < GP_WAVES; ++w) sum += part[w][i][lane];
    const int row = row0 + 16 * (i / CT) + r, col = 16 * (static_cast<int>(blockIdx.y) * CT + i % CT);
    if (row < M)
      *reinterpret_cast<u32x2_t *>((col < N ? b + col : a + (col - N)) + static_cast<int64_t>(row) * N + 4 * g) =
          u32x2_t{f32_to_bf16_pair(sum[0], sum[1]), f32_to_bf16_pair(sum[2], sum[3])};
  }
}

// A workgroup's time is the bytes it reads (its columns' weights and its rows,
// 64 KiB per 16 of either at K = 2048), so the grid is one round over the CUs of the
// smallest ones: 16 rows, and of the 64 columns 16 up to 1,024 rows, 32 up to
// 2,048; then 32 and 64 rows.  From graphs, K = 2048, this against the two
// library products: 1 / 333 / 1,000 rows 4.4 / 6.2 / 6.6 against 11.6 / 12.2 /
// 12.3 us (all 64 columns to a workgroup 9.6 / 11.1 / 11.4); 2,000 rows 8.4
// against 14.7 (11.5); 4,096 12.0 / 15.8; 8,192 14.0 / 18.4; 16,384 18.6 / 26.6;
// 65,536 79 / 111.  K = 1024 and n = 16 take less of both (1 / 1,000 / 8,192 rows, K = 1024,
// n = 16: 3.4 / 4.6 / 6.8 against 8.3 / 9.2 / 12.2).
constexpr int GP_CUS = 256;

template <int KS>
void launch_gate_proj(const uint16_t *x, const uint16_t *wb, const uint16_t *wa, int M, int n, uint16_t *b, uint16_t *a,
                      hipStream_t s) {
  const int tiles = 2 * n / 16;
  auto grid = [&](int rows) { return static_cast<unsigned>((static_cast<int64_t>(M) + rows - 1) / rows); };
  auto launch = [&](auto kernel, int ct, int rt) {
    hipLaunchKernelGGL(kernel, dim3(grid(16 * rt), tiles / ct), dim3(64 * GP_WAVES), 0, s, x, wb, wa, M, n, b, a);
  };
  if (grid(16) <= GP_CUS) {
    if (grid(16) * tiles <= GP_CUS) return launch(gate_proj_kernel<KS, 1, 1>, 1, 1);
    if (grid(16) * tiles <= 2 * GP_CUS) return launch(gate_proj_kernel<KS, 2, 1>, 2, 1);
    return launch(gate_proj_kernel<KS, 4, 1>, 4, 1);
  }
  const bool two = grid(32) <= GP_CUS;
  if (tiles == 2) return two ? launch(gate_proj_kernel<KS, 2, 2>, 2, 2) : launch(gate_proj_kernel<KS, 2, 4>, 2, 4);
  return two ? launch(gate_proj_kernel<KS, 4, 2>, 4, 2) : launch(gate_proj_kernel<KS, 4, 4>, 4, 4);
}

}  // namespace
}  // namespace gdn

extern "C" int gdn_gate_proj(const void *x, const void *w_b, const void *w_a, int32_t M, int32_t K, int32_t n, void *b,
                             void *a, void *stream) {
  using namespace gdn;
  if (!x || !w_b || !w_a || !b || !a) return fail(GDN_ERR_INVALID_ARGUMENT, "gdn_gate_proj: null pointer argument");
  if (M < 0 || (K != 1024 && K != 2048) || (n != 16 && n != 32))
    return fail(GDN_ERR_UNSUPPORTED, "gdn_gate_proj: need K 1024 or 2048 and n 16 or 32 (got M=%d K=%d n=%d)", M, K, n);
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_b) | reinterpret_cast<uintptr_t>(w_a) |
       reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(a)) % 16)
    return fail(GDN_ERR_INVALID_ARGUMENT, "gdn_gate_proj: pointers must be 16-byte aligned");
  if (M == 0) return ok();
  const auto c = [](const void *p) { return static_cast<const uint16_t *>(p); };
  const auto m = [](void *p) { return static_cast<uint16_t *>(p); };
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (K == 2048)
    launch_gate_proj<8>(c(x), c(w_b), c(w_a), M, n, m(b), m(a), s);
  else
    launch_gate_proj<4>(c(x), c(w_b), c(w_a), M, n, m(b), m(a), s);
  return check_launch("gdn_gate_proj");
}
