// Calibration kernels for gfx950: the packed weight candidates of a layer,
// the per-row loss of their outputs, and the choice of each row's clip.
//
// Restates actune/kernels/quantizers.py:23-94 (the codebooks, with torch's GPU
// division by a constant: a multiply by its fp32 reciprocal) and the candidate
// loop of actune/calibration.py:74-88.
//
// A calibration evaluates up to nine clip ratios of nine (W, A) pairs on one
// layer. As torch elementwise calls a candidate took about 45 launches over
// the fp32 weights (M = 512, 1024 x 1024: 20.1-22.5 ms a layer, the GPU 25% busy);
// here the codes of every ratio are one launch and the candidates stand one
// below the other as rows of one packed weight, so that one GEMM launch
// evaluates them all and one launch forms their losses (1.6 ms a layer).
#include <climits>

#include "../../include/actune_hip.h"
#include "common.hpp"
#include "launch.hpp"
#include "operands.hpp"

namespace actune {
namespace {

constexpr int kThreads = 256;
constexpr int kRowPass = kThreads * 8;  // elements of a row one pass of the workgroup reads

// Packed codes and scale of row n (blockIdx.x, + gridDim.x ...) under ratio
// blockIdx.y, written as row ratio * N + n. Each thread owns 8 consecutive codes per pass (W bytes).
// Bound by the division and rounding of each code (the row is read from L2
// for every ratio after the first); one workgroup per (row, ratio) keeps the
// chip full from a few hundred rows on.
template <int W, bool NESTED, int DT>
__global__ __launch_bounds__(kThreads) void weight_candidates_kernel(const void* __restrict__ w,
                                                                     const float* __restrict__ ratios, int N, int K,
                                                                     uint8_t* __restrict__ packed,
                                                                     float* __restrict__ scales) {
  __shared__ float red[kThreads / 64];
  const int tid = threadIdx.x;
  constexpr int ESZ = DT == kF32 ? 4 : 2;
  for (int n = blockIdx.x; n < N; n += (int)gridDim.x) {
    const char* row = static_cast<const char*>(w) + (size_t)n * K * ESZ;
    float amax = 0.0f;
    bool nan = false;  // torch's amax propagates NaN; fmaxf drops it
    for (int e = tid * 8; e < K; e += kRowPass) {
      float v[8];
      load8<DT>(row, e, v);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        amax = fmaxf(amax, fabsf(v[i]));
        nan = nan || v[i] != v[i];
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    const bool any_nan = __syncthreads_or(nan);
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i) amax = fmaxf(amax, red[i]);
    amax = any_nan ? __uint_as_float(0x7fc00000u) : fmaxf(amax, 1e-8f);
    constexpr bool CLIP = W != 8 || NESTED;  // plain W8 takes no clip
    if constexpr (CLIP) amax = amax * ratios[blockIdx.y];
    constexpr float R7 = 1.0f / 7.0f, R127 = 1.0f / 127.0f;
    const float s = W == 2 ? amax : W == 4 || NESTED ? amax * R7 : amax * R127;
    const size_t out = (size_t)blockIdx.y * N + n;
    if (tid == 0) scales[out] = NESTED ? s / 16.0f : s;
    constexpr float LO = W == 2 ? -2.0f : W == 4 ? -8.0f : -128.0f, HI = W == 2 ? 1.0f : W == 4 ? 7.0f : 127.0f;
    uint8_t* dst = packed + out * ((size_t)K * W / 8);
    for (int e = tid * 8; e < K; e += kRowPass) {
      float v[8];
      load8<DT>(row, e, v);
      uint32_t bits[2] = {0u, 0u};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float q = v[i] / s;
        int c;
        if constexpr (NESTED) {
          // q4 and a signed residual bounded so that 16 q4 + r4 stays an int8
          const float q4 = fminf(fmaxf(rintf(q), -8.0f), 7.0f);
          int r4 = (int)fminf(fmaxf(rintf(16.0f * (q - q4)), -8.0f), 7.0f);
          const int base = 16 * (int)q4;
          r4 = min(max(r4, max(-128 - base, -8)), min(127 - base, 7));
          c = base + r4;
        } else {
          c = (int)fminf(fmaxf(rintf(q), LO), HI);
        }
        const int bit = i * W;
        bits[bit >> 5] |= ((uint32_t)c & ((1u << W) - 1u)) << (bit & 31);
      }
      uint8_t* at = dst + (size_t)e * W / 8;
      if constexpr (W == 8) *reinterpret_cast<v2u*>(at) = v2u{bits[0], bits[1]};
      else if constexpr (W == 4) *reinterpret_cast<uint32_t*>(at) = bits[0];
      else *reinterpret_cast<uint16_t*>(at) = (uint16_t)bits[0];
    }
    __syncthreads();  // red is free for the next row
  }
}

// loss[r * N + n] = mean over m of (y[m, r * N + n] - ref[m, n])^2, the
// squares in fp32 and their sum in fp64. A workgroup takes 64 columns of one
// candidate: 16 waves a sixteenth of the rows each (whole 256-byte rows per
// load), added through LDS. HBM-bound on y.
__global__ __launch_bounds__(1024) void candidate_loss_kernel(const float* __restrict__ y, const float* __restrict__ ref,
                                                              int M, int N, int rows, float* __restrict__ loss) {
  __shared__ double part[16][64];
  const int c = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = (int)blockIdx.x * 64 + c, r = blockIdx.y;
  double sum = 0.0;
  if (n < N) {
    const float* yp = y + (size_t)r * N + n;
    for (int m0 = wave; m0 < M; m0 += 16 * 8) {
      float d[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = m0 + 16 * i;
        d[i] = m < M ? yp[(size_t)m * rows] - ref[(size_t)m * N + n] : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += (double)(d[i] * d[i]);
    }
  }
  part[wave][c] = sum;
  __syncthreads();
  if (wave == 0 && n < N) {
#pragma unroll
    for (int i = 1; i < 16; ++i) sum += part[i][c];
    loss[(size_t)r * N + n] = (float)(sum / (double)M);
  }
}

// The first candidate that lowers a row's loss strictly, in order of r;
// continues from the losses and ratios of earlier candidates.
__global__ __launch_bounds__(kThreads) void select_candidates_kernel(const float* __restrict__ loss,
                                                                     const float* __restrict__ ratios, int R, int N,
                                                                     float* __restrict__ best,
                                                                     float* __restrict__ chosen) {
  const int n = (int)blockIdx.x * kThreads + (int)threadIdx.x;
  if (n >= N) return;
  float b = best[n], c = chosen[n];
  for (int r = 0; r < R; ++r) {
    const float l = loss[(size_t)r * N + n];
    if (l < b) {
      b = l;
      c = ratios[r];
    }
  }
  best[n] = b;
  chosen[n] = c;
}

int fail(const char* msg) {
  set_last_error(msg);
  return ACTUNE_ERR_INVALID;
}

int status() {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return ACTUNE_OK;
  set_last_error(hipGetErrorString(e));
  return ACTUNE_ERR_DEVICE;
}

constexpr int64_t kMaxBytes = (int64_t)1 << 31;
constexpr int kMaxCandidates = 65535;  // grid y

template <int W, bool NESTED>
void launch_candidates(const void* w, int dt, const float* ratios, int R, int N, int K, uint8_t* packed, float* scales,
                       hipStream_t st) {
  const dim3 grid((unsigned)(N < (1 << 20) ? N : 1 << 20), (unsigned)R);
  if (dt == kBF16) weight_candidates_kernel<W, NESTED, kBF16><<<grid, kThreads, 0, st>>>(w, ratios, N, K, packed, scales);
  else if (dt == kF16) weight_candidates_kernel<W, NESTED, kF16><<<grid, kThreads, 0, st>>>(w, ratios, N, K, packed, scales);
  else weight_candidates_kernel<W, NESTED, kF32><<<grid, kThreads, 0, st>>>(w, ratios, N, K, packed, scales);
}

}  // namespace
}  // namespace actune

using namespace actune;

extern "C" {

int actune_weight_candidates(const void* w, int w_dtype, const float* ratios, int R, int64_t N, int64_t K, int W, int A,
                             uint8_t* packed, float* scales, void* stream) {
  set_last_error("");
  if ((W != 2 && W != 4 && W != 8) || (A != 2 && A != 4 && A != 8)) return fail("Unsupported integer width");
  if (w_dtype != kBF16 && w_dtype != kF16 && w_dtype != kF32) return fail("unsupported weight dtype");
  if (R < 0 || R > kMaxCandidates || N <= 0 || N > INT_MAX / 2 || K <= 0 || K % 64 || K > INT_MAX / 8)
    return fail("invalid dimensions");
  if (R > 0 && K * W / 8 > (kMaxBytes - 1) / (N * R))
    return fail("operand too large (the candidates must stay below 2 GiB)");
  if (R == 0) return ACTUNE_OK;
  if (!w || !ratios || !packed || !scales) return fail("null pointer");
  if ((uintptr_t)w % 16 || (uintptr_t)packed % 16 || (uintptr_t)ratios % 4 || (uintptr_t)scales % 4)
    return fail("misaligned operand (weights and packed data need 16 B)");
  hipStream_t st = (hipStream_t)stream;
  const int n = (int)N, k = (int)K;
  if (W == 2) launch_candidates<2, false>(w, w_dtype, ratios, R, n, k, packed, scales, st);
  else if (W == 4) launch_candidates<4, false>(w, w_dtype, ratios, R, n, k, packed, scales, st);
  else if (A == 4) launch_candidates<8, true>(w, w_dtype, ratios, R, n, k, packed, scales, st);
  else launch_candidates<8, false>(w, w_dtype, ratios, R, n, k, packed, scales, st);
  return status();
}

int actune_candidate_select(const float* y, const float* ref, const float* ratios, int R, int64_t M, int64_t N,
                            float* loss, float* best, float* chosen, void* stream) {
  set_last_error("");
  if (R < 0 || R > kMaxCandidates || M <= 0 || M > INT_MAX || N <= 0 || N > INT_MAX / 2)
    return fail("invalid dimensions");
  if (N * (R > 0 ? R : 1) > (kMaxBytes - 1) / 4 / M) return fail("operand too large (the outputs must stay below 2 GiB)");
  if (R == 0) return ACTUNE_OK;
  if (!y || !ref || !ratios || !loss || !best || !chosen) return fail("null pointer");
  if (((uintptr_t)y | (uintptr_t)ref | (uintptr_t)ratios | (uintptr_t)loss | (uintptr_t)best | (uintptr_t)chosen) % 4)
    return fail("misaligned operand");
  hipStream_t st = (hipStream_t)stream;
  const int n = (int)N;
  candidate_loss_kernel<<<dim3((unsigned)((n + 63) / 64), (unsigned)R), 1024, 0, st>>>(y, ref, (int)M, n, R * n, loss);
  select_candidates_kernel<<<dim3((unsigned)((n + kThreads - 1) / kThreads)), kThreads, 0, st>>>(loss, ratios, R, n,
                                                                                                best, chosen);
  return status();
}

}  // extern "C"
