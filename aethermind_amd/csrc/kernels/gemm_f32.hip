// fp32 Linear for two or more rows (prefill with fp32 activations and weights):
// out[M,N] = X[M,K] @ W[N,K]^T (+ residual) on v_mfma_f32_16x16x4_f32, fp32 products and
// sums throughout.
//
// What bounds it: fp32 models are small here (K of 512 to a few thousand), so the weights
// sit in L2 and a launch is latency: the block is one small output tile whose K range is
// dealt to its 4 waves in 16-value chunks, U chunks of loads in flight per wave, so a
// K of 512 is one or two round trips to memory.  Operands go from global memory straight
// to the MFMA's registers: a lane's 16-byte load of row (lane % 16), values 4 (lane / 16)
// to + 3 of a chunk, is its operand of four MFMAs (MFMA e takes value e of every lane,
// for X and W alike, so the chunk's 16 k values are summed in an order of their own).
// The waves' partial tiles meet in LDS and are summed in pairs.
//   Tiles: 16 x 16 while 32 x 32 tiles would leave CUs without a block (48 x 512 x 512:
//   96 blocks), 32 x 32 above (half the operand bytes per product).
// It replaces one GEMV launch per row: the prefill of 48 rows through the 4-layer 512-wide
// model took 1,344 launches of 2.5-3.3 us, now 28 of 5.0-8.3 us (a 48-token prompt and 32
// greedy tokens 7.8 -> 3.9 ms).

#include "am_gemv_common.h"
#include "am_launch_timing.h"

namespace am {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kWavesF = 4;  // waves of a block, each with its share of K

struct GemmF32Args {
  const float* x;
  const float* w;
  const float* residual;  // [M][N] or null; may alias out
  float* out;
  int32_t M, N, K, tiles_m;
};

// U: chunks of loads in flight per wave (a power of two).  Two blocks per CU at least, which
// keeps the MFMAs' results in registers that additions can read (without the bound they are
// copied there: 48 x 512 x 1376 9.1 us).
template <int MT, int NT, int U>
__global__ __launch_bounds__(kWavesF * 64, 2) void gemm_f32_kernel(GemmF32Args p) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int32_t tn = blockIdx.x / p.tiles_m, tm = blockIdx.x - tn * p.tiles_m;
  const int32_t m0 = tm * 16 * MT, n0 = tn * 16 * NT;
  const int r = lane & 15, kq = 4 * (lane >> 4);
  // rows past the edges read row 0 and are never stored
  const float* xr[MT];
  const float* wr[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int32_t row = m0 + 16 * i + r;
    xr[i] = p.x + static_cast<int64_t>(row < p.M ? row : 0) * p.K;
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int32_t row = n0 + 16 * i + r;
    wr[i] = p.w + static_cast<int64_t>(row < p.N ? row : 0) * p.K;
  }
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // chunk c holds k values 16 c .. 16 c + 15; K % 4 == 0, so a lane's four values are
  // all inside K or all past it (then zero on both sides)
  f32x4_t xa[U][MT], wb[U][NT];
  const f32x4_t zero = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto load = [&](int u, int32_t c) {
    const int32_t k = 16 * c + kq;
    const bool in = k < p.K;
    const int32_t kk = in ? k : 0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(xr[i] + kk);
      xa[u][i] = in ? v : zero;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(wr[j] + kk);
      wb[u][j] = in ? v : zero;
    }
  };
  const int32_t chunks = (p.K + 15) / 16;
  for (int32_t c0 = wave; c0 < chunks; c0 += kWavesF * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, c0 + kWavesF * u);
    // every load of the round goes out before the first product (left to itself the
    // compiler sinks each load to its use: 7.3 instead of 5.4 us for 48 x 512 x 512)
    __builtin_amdgcn_sched_barrier(0);
    // Sums of 4 products (one value of the chunk's 16-byte pieces), which meet in pairs over
    // the round, whose sum joins the running one: no more roundings on the way of a product
    // than in the GEMV, whose lanes keep sums of K / 256 products that meet in a tree.
    // (Four running sums over a wave's whole share of K left 1.4 times the GEMV's error at
    // K = 512, 1.9 times at 1376 and 2.7 times at 4096; 48 x 1376 x 512 took 5.9 us with them
    // and takes 6.1, 48 x 512 x 1376 7.8 and 8.3, 512 x 4096 x 4096 305 and 244.)
    f32x4_t t[U][4][MT][NT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            t[u][e][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[u][i][e], wb[u][j][e], zero, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        f32x4_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = (t[u][0][i][j] + t[u][1][i][j]) + (t[u][2][i][j] + t[u][3][i][j]);
#pragma unroll
        for (int n = U; n > 1; n /= 2)
#pragma unroll
          for (int u = 0; u < n / 2; ++u) v[u] = v[2 * u] + v[2 * u + 1];
        acc[i][j] += v[0];
      }
  }

  // lane holds D[4 (lane / 16) + e][lane % 16] of each 16 x 16 tile
  constexpr int TS = 16 * NT + 1;
  static_assert(kWavesF == 4, "summed in pairs below");
  __shared__ float part[kWavesF][16 * MT][TS];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[wave][16 * i + kq + e][16 * j + r] = acc[i][j][e];
  __syncthreads();
  constexpr int kOut = 16 * MT * 16 * NT;
#pragma unroll
  for (int o = 0; o < kOut / (kWavesF * 64); ++o) {
    const int t = tid + kWavesF * 64 * o, row = t / (16 * NT), col = t % (16 * NT);
    const int32_t gm = m0 + row, gn = n0 + col;
    if (gm >= p.M || gn >= p.N) continue;
    float v = (part[0][row][col] + part[1][row][col]) + (part[2][row][col] + part[3][row][col]);
    const int64_t idx = static_cast<int64_t>(gm) * p.N + gn;
    if (p.residual != nullptr) v = p.residual[idx] + v;
    p.out[idx] = v;
  }
}

bool Aligned16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; }

template <int MT, int NT, int U>
am_status_code LaunchF32(GemmF32Args p, hipStream_t s) {
  p.tiles_m = static_cast<int32_t>(CeilDiv(p.M, 16 * MT));
  const int64_t blocks = p.tiles_m * CeilDiv(p.N, 16 * NT);
  RecordLaunch(blocks, kWavesF * 64, 0, "gemm_f32<%dx%d>", 16 * MT, 16 * NT);
  hipLaunchKernelGGL((gemm_f32_kernel<MT, NT, U>), dim3(static_cast<unsigned>(blocks)), dim3(kWavesF * 64), 0, s, p);
  AM_RETURN_IF_LAUNCH_FAILED("gemm_f32");
  return AM_STATUS_OK;
}

}  // namespace

// fp32 rows and weights in 16-byte pieces, up to the row length the GEMV kernels take
// (longer rows and residuals that do not fit their LDS stay refused by them).
bool GemmF32Eligible(const am_gfx950_weight& w, int64_t m, const void* x, const void* residual) {
  constexpr int64_t kMaxK = 8192, kLdsLimit = 150 * 1024;
  return w.format == AM_WF_F32 && m >= 2 && w.k % 4 == 0 && w.k <= kMaxK && Aligned16(x) && Aligned16(w.data) &&
         w.k * 4 + (residual != nullptr ? w.n * 4 : 0) <= kLdsLimit && w.n < (int64_t{1} << 30) &&
         CeilDiv(m, 16) * CeilDiv(w.n, 16) < (int64_t{1} << 31);
}

am_status_code GemmF32(const void* x, int64_t m, const am_gfx950_weight& w, void* out, const void* residual,
                       hipStream_t s) {
  GemmF32Args p{};
  p.x = static_cast<const float*>(x);
  p.w = static_cast<const float*>(w.data);
  p.residual = static_cast<const float*>(residual);
  p.out = static_cast<float*>(out);
  p.M = static_cast<int32_t>(m);
  p.N = static_cast<int32_t>(w.n);
  p.K = static_cast<int32_t>(w.k);
  if (CeilDiv(m, 32) * CeilDiv(w.n, 32) >= DeviceCUs()) return LaunchF32<2, 2, 4>(p, s);
  return LaunchF32<1, 1, 8>(p, s);
}

}  // namespace am
