// float32 projections on the matrix cores: C[M,N] = A[M,K] . B[N,K]^T (+ R).
//
// K is cut into chunks whose length depends on K alone (f32_chunk: at most 8 chunks of at least 32 k). A
// chunk is one chain of v_mfma_f32_16x16x4_f32, 16 k per four instructions: lane group g holds k = 4g..4g+3
// of a 16-k step (one 16-byte load per operand row, straight from global memory, no LDS), and instruction
// j takes element j of each group. The chunks' results are added in increasing order. Every tile shape
// below runs that same arithmetic, so an element does not depend on M, on the tile or on how the chunks
// are dealt to waves: a decode step, a verify window and a prefill give identical rows.
//
// What bounds it: a decode step (M of a few rows) is a stream of weights behind a chain of dependent
// matrix instructions, so the chunks of a 16 x 16 tile go to a workgroup's waves side by side and meet in
// LDS. A long batch is bound by the matrix cores (157 TFLOP/s in float32): there each wave walks the chunks
// of a 64 x 64 tile one after the other (no exchange), operands read through L1/L2 at 16 B per clock and CU.
//
// Measured (M x N x K, the one-fmaf-chain VALU kernel it replaces -> this): 1 x 512 x 256 23.2 -> 9.7 us a call
// (4.4 us of kernel), 1 x 4096 x 4096 420 -> 17 us (4.0 TB/s of weights), 64 x 6144 x 4096 531 -> 80 us,
// 640 x 1376 x 256 27 -> 12.7 us, 448 x 4096 x 4096 512 -> 253 us, 4096 x 28672 x 4096 16.6 -> 11.9 ms
// (81 TFLOP/s). Error against 64 bits: half (shorter chains), 7.5e-7 -> 4.2e-7 over a 4-layer model's logits.
#include "common.h"

namespace {

constexpr int kMaxChunks = 8;

int64_t f32_chunk(int64_t K) {
  const int64_t c = ((K + kMaxChunks - 1) / kMaxChunks + 15) / 16 * 16;
  return c < 32 ? 32 : c;
}

// SPLIT: the workgroup's waves take one K chunk each of one (16 TM) x (16 TN) tile and the chunk sums meet
// in LDS. Else the workgroup's 2 x 2 waves have a tile each and run its chunks one after the other.
// U: 16-k steps loaded together.
template <int TM, int TN, int U, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? 64 * kMaxChunks : 256)
    gemm_f32_mfma_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
                         float* __restrict__ C, int64_t ldc, const float* __restrict__ R, int64_t ldr, int64_t M,
                         int64_t N, int64_t K, int64_t chunk, int nchunks, int tiles_n) {
  constexpr int WM = SPLIT ? 1 : 2;   // waves along M and along N
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int64_t m0 = ((int64_t)(blockIdx.x / tiles_n) * WM + (SPLIT ? 0 : wave >> 1)) * (16 * TM);
  const int64_t n0 = ((int64_t)(blockIdx.x % tiles_n) * WM + (SPLIT ? 0 : wave & 1)) * (16 * TN);

  const float* pa[TM];
  const float* pb[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t r = m0 + 16 * i + l16;
    pa[i] = A + (r < M ? r : M - 1) * lda;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t r = n0 + 16 * j + l16;
    pb[j] = B + (r < N ? r : N - 1) * ldb;
  }

  float4_t acc[TM][TN], sum[TM][TN];
  float4_t a[2][U][TM], b[2][U][TN];

  // the chain of chunk c into acc
  auto run_chunk = [&](int c) {
    const int64_t kb = c * chunk, ke = kb + chunk < K ? kb + chunk : K;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    // U steps from k; a lane past the chunk's end (K % 4 == 0: a whole load) re-reads its last 16 bytes as zeros
    auto load = [&](int p, int64_t k) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t kk = k + 16 * u + 4 * g;
        const bool in = kk < ke;
        const int64_t ka = in ? kk : ke - 4;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const float4_t v = *reinterpret_cast<const float4_t*>(pa[i] + ka);
          a[p][u][i] = in ? v : float4_t{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const float4_t v = *reinterpret_cast<const float4_t*>(pb[j] + ka);
          b[p][u][j] = in ? v : float4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
    };
    auto step = [&](int p, int64_t k) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k + 16 * u >= ke) break;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[p][u][j][e], a[p][u][i][e], acc[i][j], 0, 0, 0);
      }
    };
    load(0, kb);
    for (int64_t k = kb; k < ke; k += 32 * U) {
      if (k + 16 * U < ke) load(1, k + 16 * U);
      step(0, k);
      if (k + 32 * U < ke) load(0, k + 32 * U);
      step(1, k + 16 * U);
    }
  };

  auto store = [&](int64_t row, int64_t col0, float4_t v) {   // C[row][col0 .. col0 + 3]
    if (row >= M) return;
    if (col0 + 3 < N && ((ldc | ldr | col0) & 3) == 0 && ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(R)) & 15) == 0) {
      if (R) {
        const float4_t r = *reinterpret_cast<const float4_t*>(R + row * ldr + col0);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] + r[e];
      }
      *reinterpret_cast<float4_t*>(C + row * ldc + col0) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col0 + e < N) C[row * ldc + col0 + e] = R ? v[e] + R[row * ldr + col0 + e] : v[e];
    }
  };

  if (SPLIT) {
    __shared__ float4_t part[kMaxChunks][TM * TN][64];
    run_chunk(wave);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) part[wave][i * TN + j][lane] = acc[i][j];
    __syncthreads();
    for (int t = wave; t < TM * TN; t += nchunks) {   // acc[i][j]: lane (l16, g) has C[16i + l16][16j + 4g + e]
      float4_t v = part[0][t][lane];
      for (int c = 1; c < nchunks; ++c) {
        const float4_t w = part[c][t][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] + w[e];
      }
      store(m0 + 16 * (t / TN) + l16, n0 + 16 * (t % TN) + 4 * g, v);
    }
  } else {
    for (int c = 0; c < nchunks; ++c) {
      run_chunk(c);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[i][j][e] = c ? sum[i][j][e] + acc[i][j][e] : acc[i][j][e];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) store(m0 + 16 * i + l16, n0 + 16 * j + 4 * g, sum[i][j]);
  }
}

}  // namespace

namespace fs {

bool gemm_f32_ok(const void* A, int64_t lda, const void* B, int64_t ldb, int64_t K) {
  return K % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 &&
         ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) == 0;
}

void gemm_f32(const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc, const float* R,
              int64_t ldr, int64_t M, int64_t N, int64_t K, hipStream_t s) {
  const int64_t chunk = f32_chunk(K);
  const int n = (int)((K + chunk - 1) / chunk);
  // 64 x 64 per wave once 128 x 128 tiles fill the CUs, 32 x 32 split over the chunks once those do, else 16 x 16:
  // a short batch wants workgroups more than reuse (the tile never changes a result)
  auto tiles = [&](int64_t t) { return ((M + t - 1) / t) * ((N + t - 1) / t); };
  if (tiles(128) >= 256)
    gemm_f32_mfma_kernel<4, 4, 1, false><<<dim3((unsigned)tiles(128)), 256, 0, s>>>(
        A, lda, B, ldb, C, ldc, R, R ? ldr : 0, M, N, K, chunk, n, (int)((N + 127) / 128));
  else if (tiles(32) >= 256)
    gemm_f32_mfma_kernel<2, 2, 2, true><<<dim3((unsigned)tiles(32)), 64 * n, 0, s>>>(
        A, lda, B, ldb, C, ldc, R, R ? ldr : 0, M, N, K, chunk, n, (int)((N + 31) / 32));
  else
    gemm_f32_mfma_kernel<1, 1, 4, true><<<dim3((unsigned)tiles(16)), 64 * n, 0, s>>>(
        A, lda, B, ldb, C, ldc, R, R ? ldr : 0, M, N, K, chunk, n, (int)((N + 15) / 16));
}

}  // namespace fs
