// y[M, N] = residual + x[M, K] @ dequant(W)^T for a few rows of x (M <= 32) in one launch: a short
// prompt, or several sequences decoded together (QLinear.forward at small M, scripts/llm/llama_q4.py:72).
//
// The weights are read once, so the floor is their HBM time; what the 64-row tiles of q4_linear lose
// here is rows padded to 64, too few workgroups and a serial chain of K steps. Instead:
//   * a workgroup owns 16 NT columns and ALL of K: its waves take 128-k steps in turn and
//     meet in LDS at the end, so the chip is filled by columns x waves with no partials in memory and no
//     second launch;
//   * each wave loads what it multiplies straight into registers: per step and 16 columns one 16-byte load
//     per lane (lane l: column l % 16, 32 k at 32 (l / 16)), whose four words four lane swaps turn into
//     the B operands of four v_mfma_f32_16x16x32_f16; and the fp32 x rows of the step, split in registers
//     into fp16 (hi, lo) as q4_linear does, so no plane is written and re-read. Each x value is split
//     once per workgroup; the rows come from L2;
//   * group scales multiply the fp32 sums of each group (kG128: one group per 128-k step; otherwise
//     every 32 k, so any group % 32 == 0 works).
// Products, splits and accumulation are those of q4_linear: y = sum_g s_g sum_k (hi + lo)(n - 8) in fp32.
// What bounds it is the latency of the loads (7x3072x3072: matrix cores busy 4% of the cycles, waves waiting 49%).
// M <= 16: a wave's next step is loaded before the present one is multiplied, but in a branch, after which the
// compiler waits for all loads, so in every other step the loads just issued too. M > 16: one step at a time, its
// x loads sunk to their uses, several memory round trips a step; the time then grows with K (32x3072x8192 36 us).
#include "q4_common.h"
#include "q4_internal.h"

#include <algorithm>

namespace q4 {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kOut = 0x80000000u;  // out of every buffer's range: the load returns zeros

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}

// w[i] of lane group c (16 lanes each) <- w[c] of lane group i: the upper 32 lanes of one word trade
// places with the lower 32 of another, then odd 16-lane rows with even ones.
__device__ __forceinline__ void transpose4(uint32_t (&w)[4]) {
  auto t = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
  w[0] = t[0], w[2] = t[1];
  t = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
  w[1] = t[0], w[3] = t[1];
  t = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);
  w[0] = t[0], w[1] = t[1];
  t = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
  w[2] = t[0], w[3] = t[1];
}

// transpose4 of four copies of one value: s[i] of every lane is v of lane group i. Inline asm, because
// this compiler folds the two results of a builtin swap whose operands are the same value into one; the
// s_nops cover the VALU hazards.
__device__ __forceinline__ void broadcast4(uint32_t v, uint32_t (&s)[4]) {
  uint32_t a = v, b = v;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  uint32_t a2 = a, b2 = b;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(a2));
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(b), "+v"(b2));
  s[0] = a, s[1] = a2, s[2] = b, s[3] = b2;
}

// Packed word of 8 nibbles -> fp16 (n - 8) in k order (0, 4, 1, 5, 2, 6, 3, 7), exact.
__device__ __forceinline__ half8 rows_nibbles(uint32_t w, const F16Magic& mg) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  const half2v b1024 = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-1032.0f)};
  const half2v b64 = {static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)};
  const uint32_t w8 = w >> 8;
  const half2v p0 = __builtin_bit_cast(half2v, (w & 0x000F000Fu) | mg.e1024) + b1024;
  const half2v p1 = __builtin_bit_cast(half2v, (w & 0x00F000F0u) | mg.e64) + b64;
  const half2v p2 = __builtin_bit_cast(half2v, (w8 & 0x000F000Fu) | mg.e1024) + b1024;
  const half2v p3 = __builtin_bit_cast(half2v, (w8 & 0x00F000F0u) | mg.e64) + b64;
  return half8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// Rows 16 MT, columns 16 NT per workgroup; blockDim.x / 64 waves share K. `magic`: the
// reciprocal 2^32 / d (rounded up) of d = 32-k blocks (kG128: 128-k steps) per group; 0 for d = 1.
template <int MT, int NT, bool kG128>
__global__ __launch_bounds__(MT == 1 && NT == 1 ? 1024 : 512) void q4_rows_kernel(const float* __restrict__ X, const int32_t* __restrict__ QW,
                                                      const uint16_t* __restrict__ SC, float* Y, const float* R, int M,
                                                      int N, int K, int spr, uint32_t magic) {
  extern __shared__ float red[];  // [waves][MT NT 4][64]
  const int lane = threadIdx.x & 63, col = lane & 15, c = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int n0 = blockIdx.x * (16 * NT);
  const __amdgpu_buffer_rsrc_t xr = rows_rsrc(X, static_cast<uint32_t>(M) * K * 4u);
  const __amdgpu_buffer_rsrc_t wr = rows_rsrc(QW, static_cast<uint32_t>(N) * (K / 2));
  const __amdgpu_buffer_rsrc_t sr = rows_rsrc(SC, static_cast<uint32_t>(N) * spr * 2u);
  const int steps = (K + 127) / 128;
  const F16Magic mg = f16_magic();
  const float m1 = minus_one();

  struct Step {
    i32x4 w[NT];
    uint32_t s[NT];  // fp16 scale bits of the lane's 32-k block (kG128: of the step)
    float4v x[MT][8];
  };
  // Per-lane offsets of step 0; a step adds a uniform one. Columns past N and rows past M read zeros.
  uint32_t wo[NT], so[NT], xo[MT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + 16 * j + col;
    wo[j] = n < N ? static_cast<uint32_t>(n) * (K / 2) + 16 * c : kOut;  // 32 k at 32 c
    so[j] = n < N ? static_cast<uint32_t>(n) * spr * 2u : kOut;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = 16 * i + col;
    xo[i] = m < M ? (static_cast<uint32_t>(m) * K + 8 * c) * 4u : kOut;  // 8 k at 32 q + 8 c
  }
  auto load = [&](int t, Step& b) {
    const bool half = 128 * t + 64 >= K;  // the step holds 64 k: lane groups 2 and 3, x blocks 2 and 3 are past K
    const bool w_in = !half || c < 2;
    const uint32_t idx = kG128 ? t : 4 * t + c;
    const uint32_t g = magic ? __umulhi(idx, magic) : idx;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      b.w[j] = __builtin_amdgcn_raw_buffer_load_b128(wr, w_in ? wo[j] : kOut, t * 64, 0);
      b.s[j] = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(sr, w_in ? so[j] + 2 * g : kOut, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const uint32_t xh = half ? kOut : xo[i];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t o = (q < 2 ? xo[i] : xh) + 128 * q;
        b.x[i][2 * q] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(xr, o, t * 512, 0));
        b.x[i][2 * q + 1] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(xr, o + 16, t * 512, 0));
      }
    }
  };

  float4v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](Step& b) {
    uint32_t w[NT][4], s[NT][4];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) w[j][q] = static_cast<uint32_t>(b.w[j][q]);
      transpose4(w[j]);
      const uint32_t f = __builtin_bit_cast(uint32_t, half_bits_to_float(static_cast<uint16_t>(b.s[j])));
      if constexpr (kG128) s[j][0] = s[j][1] = s[j][2] = s[j][3] = f;
      else broadcast4(f, s[j]);  // s[j][q]: the scale of 32-k block q in every lane
    }
    float4v part[MT][NT];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      half8 hi[MT], lo[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float4v a = b.x[i][2 * q], e = b.x[i][2 * q + 1];
        uint32_t h[4], l[4];  // k order 0, 4, 1, 5, 2, 6, 3, 7
        split_f16_pair(a.x, e.x, m1, h[0], l[0]);
        split_f16_pair(a.y, e.y, m1, h[1], l[1]);
        split_f16_pair(a.z, e.z, m1, h[2], l[2]);
        split_f16_pair(a.w, e.w, m1, h[3], l[3]);
        hi[i] = __builtin_bit_cast(half8, make_uint4(h[0], h[1], h[2], h[3]));
        lo[i] = __builtin_bit_cast(half8, make_uint4(l[0], l[1], l[2], l[3]));
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const half8 fb = rows_nibbles(w[j][q], mg);
        const float sc = __builtin_bit_cast(float, s[j][q]);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const float4v z = {0.0f, 0.0f, 0.0f, 0.0f};
          float4v p = kG128 && q > 0 ? part[i][j] : z;
          p = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[i], fb, p, 0, 0, 0);
          p = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[i], fb, p, 0, 0, 0);
          if (kG128 && q < 3) {
            part[i][j] = p;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(p[r], sc, acc[i][j][r]);
          }
        }
      }
    }
  };

  if constexpr (MT == 1) {  // two steps' operands: the next one's loads are issued before this one is multiplied
    Step a, b;
    if (wave < steps) load(wave, a);
    for (int t = wave; t < steps; t += 2 * waves) {
      if (t + waves < steps) load(t + waves, b);
      compute(a);
      if (t + waves < steps) {
        if (t + 2 * waves < steps) load(t + 2 * waves, a);
        compute(b);
      }
    }
  } else {
    Step a;
    for (int t = wave; t < steps; t += waves) {
      load(t, a);
      compute(a);
    }
  }

  // Sum over the waves in wave order. Accumulator r of lane l: row 4 (l / 16) + r, column l % 16.
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave * MT + i) * NT + j) * 256 + r * 64 + lane] = acc[i][j][r];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * NT * 256; e += blockDim.x) {
    float v = red[e];
    for (int w = 1; w < waves; ++w) v += red[w * (MT * NT * 256) + e];
    const int l = e & 63, r = (e >> 6) & 3, j = (e >> 8) % NT, i = (e >> 8) / NT;
    const int m = 16 * i + 4 * (l >> 4) + r, n = n0 + 16 * j + (l & 15);
    if (m < M && n < N) {
      const int64_t o = static_cast<int64_t>(m) * N + n;
      Y[o] = R ? R[o] + v : v;
    }
  }
}

template <int MT, int NT>
int rows_go(const float* x, int64_t M, const int32_t* qw, const uint16_t* sc, float* y, const float* res, int64_t N,
            int64_t K, int group, hipStream_t st) {
  constexpr int kWaves = MT == 1 && NT == 1 ? 16 : 8;
  const dim3 grid(static_cast<unsigned>((N + 16 * NT - 1) / (16 * NT)));
  const bool g128 = group % 128 == 0;
  const auto fn = g128 ? q4_rows_kernel<MT, NT, true> : q4_rows_kernel<MT, NT, false>;
  const uint32_t d = static_cast<uint32_t>(group / (g128 ? 128 : 32));
  const uint32_t magic = d > 1 ? static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d) : 0;
  hipLaunchKernelGGL(fn, grid, dim3(64 * kWaves), kWaves * MT * NT * 1024, st, x, qw, sc, y, res, (int)M, (int)N,
                     (int)K, (int)(K / group), magic);
  return launch_status();
}

}  // namespace

// Every workgroup reads and splits all of x, so the kernel's time grows with M K where the tiled path's
// (x planes, 64x256 tile, K-split partials: three launches) hardly does. Measured on one MI355X at group
// 128, graph replays over rotated weights, this kernel | that path (us):
//   M = 7:  3072x3072 7.0 | 14.1, 16384x3072 13.4 | 21.8, 3072x8192 15.0 | 20.8, 1024x2048 5.6 | 12.2
//   M = 16: 3072x3072 9.2 | 14.8, 16384x3072 15.6 | 23.3, 3072x8192 21.5 | 22.3, 1024x2048 7.1 | 12.8
//   M = 32: 3072x3072 15.1 | 17.2, 16384x3072 20.8 | 25.5, 3072x8192 36.0 | 25.1, 1024x2048 10.8 | 13.5
// (the one-tile-per-workgroup kernel before both: 70, 96, 186 and 48 us at every such M).
bool q4_rows_takes(int64_t M, int64_t K) { return M <= 16 || (M <= 32 && K <= 4096); }

// Columns per workgroup / 16: about one workgroup per CU, so 16 columns up to 4096, 32 up to 8192, else 64
// (M = 7: 5120 columns 8.6 us by 32 against 11.8 by 16, 16384 13.4 by 64 against 16.8 by 32).
static int rows_nt(int64_t N) { return N <= 4096 ? 1 : N <= 8192 ? 2 : 4; }

// Where a workspace makes the tiled path possible too, this kernel runs on its side of a line fitted to 2600
// shapes of M 2-32, N 64-131072, K 256-28672 at groups 128 and 32 (graph replays over rotated weights; at most
// 6% slower than the tiled path on any, and 0.5% off the faster one on average): M K below a limit that grows
// with how full the chip is of workgroups, since the tiled path's K splits fill it at any N; more for groups
// under 128, whose scales cost the tiles more; and up to a number of columns from where on both have work for
// every CU and the tiles read x less often. This kernel | tiled path, group 128 (us): 16x4096x8192 21.3 | 22.7,
// 16x4096x14336 34.3 | 28.5, 16x8192x14336 41.7 | 42.4, 12x8448x14336 54.1 | 47.4, 4x1536x28672 37.2 | 35.8,
// 32x64x4096 18.4 | 13.9, 32x4096x4096 19.1 | 20.9, 7x65536x8192 121 | 153, 24x131072x2048 85.3 | 74.3.
bool q4_rows_wins(int64_t M, int64_t N, int64_t K, int group) {
  if (!q4_rows_takes(M, K)) return false;
  const int nt = rows_nt(N);
  const double fill = std::min(1.0, static_cast<double>((N + 16 * nt - 1) / (16 * nt)) / 256.0), f2 = fill * fill;
  if (M <= 16) {
    if (N > 49152 && (N > 65536 || K < (group < 128 ? 1024 : M <= 8 ? 3072 : 5120))) return false;
    const double limit = (nt == 4 ? 65536.0 : 86016.0) + 81920.0 * nt * f2 * (nt == 1 ? 1.0 : nt == 2 ? fill : f2);
    // fewer rows than 2 nt cost the same: the loads of the weights
    return static_cast<double>(std::max<int64_t>(M, 2 * nt) * K) <= (group >= 128 ? limit : 1.5 * limit);
  }
  if (N > 16384) return N <= 32768 && group >= 128 && M * K <= 98304;
  const double limit = 79872.0 + 65536.0 * (nt == 4 ? f2 : fill);
  return static_cast<double>(M * K) <= (group >= 128 ? limit : 1.3 * limit);
}

int q4_rows_launch(const float* x, int64_t M, const int32_t* qw, const uint16_t* sc, float* y, const float* res,
                   int64_t N, int64_t K, int group, hipStream_t st) {
  const auto go = M <= 16 ? (rows_nt(N) == 1 ? rows_go<1, 1> : rows_nt(N) == 2 ? rows_go<1, 2> : rows_go<1, 4>)
                          : (rows_nt(N) == 1 ? rows_go<2, 1> : rows_nt(N) == 2 ? rows_go<2, 2> : rows_go<2, 4>);
  return go(x, M, qw, sc, y, res, N, K, group, st);
}

}  // namespace q4
