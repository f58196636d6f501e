// The m x m part of one Gram segment (start or restart to the next Q X) for matrices of at most
// 128 rows, in one launch: one workgroup per matrix keeps R, Z and Q in LDS.
//
// On the NT kernels such a product is a launch of 3-4 blocks that takes 5 us -- 2 us from launch to
// launch, 3 us of argument, first-slice and epilogue latency -- for 0.1 us of work, and a
// segment of three steps is nine of them. Here a product takes ~2.3 us, bound by the vector work of
// its epilogue and by two barriers on one CU, and nothing leaves the CU in between: 14 launches of
// one gram_newton_schulz become 2 of 14 and 21 us (128 x 512: 102 -> 67 us a call).
//
// 8 waves of 64 x 32 on v_mfma_f32_16x16x32_f16 with the NT kernels' arithmetic: the same K order
// (64-wide slices from 0: a matrix this small has one 256-block, so no rotation), the same
// epilogue operations in fp32 and one rounding, upper triangles mirrored -- the same bits.
// A 128-value row is 256 bytes, all 64 banks, so its sixteen 16-byte chunks sit under chunk ^
// (row % 16): a fragment read (16 rows at one chunk) covers every bank once.
#include "dmuon_amd_internal.h"

namespace dmuon {
namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

constexpr int N = 128, ROWB = 2 * N, MAT = N * ROWB;   // one matrix: 32 KiB

__device__ __forceinline__ uint16_t f2h(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
}
__device__ __forceinline__ float h2f(uint16_t h) {
  return static_cast<float>(__builtin_bit_cast(_Float16, h));
}
// byte offset of element (r, c) of a matrix in LDS
__device__ __forceinline__ int at(int r, int c) {
  return r * ROWB + (((c >> 3) ^ (r & 15)) << 4) + (c & 7) * 2;
}

// two values rounded to nearest even and packed, low half first
__device__ __forceinline__ unsigned pack2(float lo, float hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2_t{lo, hi}, f16x2_t));
}

// One matrix; KM (64 or 128): its rows rounded up to the 64-wide slice.
template <int KM>
__device__ __forceinline__ void gram_small(const GramSmallArgs& p, const GramSmallGroup& a,
                                           char* smem, int matrix) {
  constexpr int R = 0, Z = MAT, Q = 2 * MAT;       // LDS bytes
  const uint16_t* Rg = a.R + (long long)matrix * N * N;
  uint16_t* Qg = a.Q + (long long)matrix * N * N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this wave's values: 4 x 2 blocks of 16 x 16, or 2 x 1 of the 64 x 64
  constexpr int BI = KM / 32, BJ = KM / 64, KS = KM / 32;
  const int i0 = KM / 2 * (wave >> 2), j0 = KM / 4 * (wave & 3);
  // this lane's values of block (x, y): row i0 + 16 x + li, columns j0 + 16 y + lj .. + 3
  const int li = lane & 15, lj = 4 * (lane >> 4);

#pragma unroll
  for (int k = 0; k < KM * KM / 8 / 512; ++k) {
    const int q = k * 512 + tid, r = q / (KM / 8), c = q % (KM / 8) * 8;
    *reinterpret_cast<u32x4_t*>(smem + R + at(r, c)) = *reinterpret_cast<const u32x4_t*>(Rg + r * N + c);
  }
  __syncthreads();

  f32x4_t acc[BI][BJ];
  u32x2_t out[BI][BJ];
  // Byte offsets of this lane's accesses within a matrix, found once: a block 16 rows further is
  // 16 ROWB away at the same swizzle. (Found at each access the two segments take 15.4 and 23.7
  // us instead of 13.6 and 21.2; one body for all products, which fetches less code, 18 and 28.)
  int fa[KS], fb[KS], rc[BJ], mir[4][BI];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int c = (ks * 4 + (lane >> 4)) * 8;
    fa[ks] = at(i0 + li, c);
    fb[ks] = at(j0 + li, c);
  }
#pragma unroll
  for (int y = 0; y < BJ; ++y) rc[y] = at(i0 + li, j0 + 16 * y + lj);      // (i, j .. j + 3)
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int x = 0; x < BI; ++x) mir[e][x] = at(j0 + lj + e, i0 + 16 * x + li);   // (j + e, i)
  // blocks of a symmetric product below the diagonal are the mirror of those above
  auto needed = [&](int x, int y, bool sym) { return !sym || j0 + 16 * y >= i0 + 16 * x; };
  // acc = A B^T over this wave's values
  auto product = [&](int A, int B, bool sym) {
    if (sym && j0 + KM / 4 <= i0) return;           // wholly below the diagonal
    f16x8_t af[KS][BI], bf[KS][BJ];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int x = 0; x < BI; ++x)
        af[ks][x] = *reinterpret_cast<const f16x8_t*>(smem + A + 16 * ROWB * x + fa[ks]);
#pragma unroll
      for (int y = 0; y < BJ; ++y)
        bf[ks][y] = *reinterpret_cast<const f16x8_t*>(smem + B + 16 * ROWB * y + fb[ks]);
    }
#pragma unroll
    for (int x = 0; x < BI; ++x)
#pragma unroll
      for (int y = 0; y < BJ; ++y) acc[x][y] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int x = 0; x < BI; ++x)
#pragma unroll
        for (int y = 0; y < BJ; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[ks][y], af[ks][x], acc[x][y], 0, 0,
                                                             0);
  };
  // out = half(s * acc + beta * C (+ diag on the diagonal))
  auto finish = [&](int C, float s, float beta, float diag, bool sym) {
#pragma unroll
    for (int x = 0; x < BI; ++x)
#pragma unroll
      for (int y = 0; y < BJ; ++y) {
        if (!needed(x, y, sym)) continue;
        const u32x2_t c2 = *reinterpret_cast<const u32x2_t*>(smem + C + 16 * ROWB * x + rc[y]);
        float r[4] = {h2f(c2.x & 0xffff), h2f(c2.x >> 16), h2f(c2.y & 0xffff), h2f(c2.y >> 16)};
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = s * acc[x][y][e] + beta * r[e];
        if (sym && i0 + 16 * x == j0 + 16 * y) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (li == lj + e) r[e] += diag;
        }
        out[x][y] = u32x2_t{pack2(r[0], r[1]), pack2(r[2], r[3])};
      }
  };
  auto value = [&](int x, int y, int e) {
    const unsigned w = e < 2 ? out[x][y].x : out[x][y].y;
    return (uint16_t)(e & 1 ? w >> 16 : w & 0xffff);
  };
  auto put = [&](int byte, uint16_t h) { *reinterpret_cast<uint16_t*>(smem + byte) = h; };
  // The values on and above the diagonal to (i, j) and (j, i) of D; with `second`, to the matrix
  // that many bytes further too, there plus diag2 on the diagonal. Only the 16 x 16 blocks on the
  // diagonal need a look at each value.
  auto store_sym = [&](int D, int second, float diag2) {
#pragma unroll
    for (int x = 0; x < BI; ++x)
#pragma unroll
      for (int y = 0; y < BJ; ++y) {
        if (!needed(x, y, true)) continue;
        const int dr = D + 16 * ROWB * x + rc[y];
        if (i0 + 16 * x != j0 + 16 * y) {
          *reinterpret_cast<u32x2_t*>(smem + dr) = out[x][y];
          if (second) *reinterpret_cast<u32x2_t*>(smem + dr + second) = out[x][y];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int dm = D + 16 * ROWB * y + mir[e][x];
            put(dm, value(x, y, e));
            if (second) put(dm + second, value(x, y, e));
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint16_t h = value(x, y, e);
            const int dm = D + 16 * ROWB * y + mir[e][x];
            if (lj + e > li) {
              put(dm, h);
              if (second) put(dm + second, h);
            }
            if (lj + e >= li) {
              put(dr + 2 * e, h);
              if (second) put(dr + second + 2 * e, lj + e == li ? f2h(h2f(h) + diag2) : h);
            }
          }
        }
      }
  };
  auto store_full = [&](int D, bool transposed) {
#pragma unroll
    for (int x = 0; x < BI; ++x)
#pragma unroll
      for (int y = 0; y < BJ; ++y) {
        if (!transposed) {
          *reinterpret_cast<u32x2_t*>(smem + D + 16 * ROWB * x + rc[y]) = out[x][y];
          continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) put(D + 16 * ROWB * y + mir[e][x], value(x, y, e));
      }
  };

  float rs = a.rs;                                 // the stored R is rs times R
  for (int t = 0; t < p.steps; ++t) {
    const float ca = p.coeff[3 * t], cb = p.coeff[3 * t + 1], cc = p.coeff[3 * t + 2];
    const bool evolve = t + 1 < p.steps, fresh = t == 0;
    // Z = c R^2 + b R; at first also Q = Z + a I, or Q alone when the segment has one step
    product(R, R, true);
    finish(R, cc / (rs * rs), cb / rs, fresh && !evolve ? ca : 0.f, true);
    if (fresh && !evolve) store_sym(Q, 0, 0.f);
    else store_sym(Z, fresh ? Q - Z : 0, ca);
    __syncthreads();
    if (!fresh) {
      // Q^T <- Q^T Z + a Q^T; the last one leaves Q itself, which Q X reads
      product(Q, Z, false);
      finish(Q, 1.f, ca, 0.f, false);
      __syncthreads();
      store_full(Q, !evolve);
      if (!evolve) __syncthreads();
    }
    if (evolve) {
      // W = Z R + a R over R, then R = P R P = W Z + a W over W
      product(Z, R, true);
      finish(R, 1.f, ca, 0.f, true);
      __syncthreads();
      store_sym(R, 0, 0.f);
      __syncthreads();
      product(R, Z, true);
      finish(R, 1.f / rs, ca / rs, 0.f, true);
      __syncthreads();
      store_sym(R, 0, 0.f);
      __syncthreads();
      rs = 1.f;
    }
  }
#pragma unroll
  for (int k = 0; k < KM * KM / 8 / 512; ++k) {
    const int q = k * 512 + tid, r = q / (KM / 8), c = q % (KM / 8) * 8;
    *reinterpret_cast<u32x4_t*>(Qg + r * N + c) =
        *reinterpret_cast<const u32x4_t*>(smem + Q + at(r, c));
  }
}

__global__ __launch_bounds__(512) void gram_small_kernel(const GramSmallArgs p) {
  __shared__ __attribute__((aligned(16))) char smem[3 * MAT];
  int g = 0;
  while (g + 1 < p.n && (int)blockIdx.x >= p.g[g + 1].first) ++g;
  g = __builtin_amdgcn_readfirstlane(g);
  const int matrix = blockIdx.x - p.g[g].first;
  if (p.g[g].km == 64) gram_small<64>(p, p.g[g], smem, matrix);
  else gram_small<128>(p, p.g[g], smem, matrix);
}

}  // namespace

hipError_t launch_gram_small(const GramSmallArgs& a, int matrices, hipStream_t stream) {
  if (a.n < 1 || a.n > kMaxGroups || a.steps < 1 || a.steps > kGramSmallSteps || matrices < 1)
    return hipErrorInvalidValue;
  for (int g = 0; g < a.n; ++g)
    if (!a.g[g].R || !a.g[g].Q || (a.g[g].km != 64 && a.g[g].km != 128))
      return hipErrorInvalidValue;
  hipLaunchKernelGGL(gram_small_kernel, dim3((unsigned)matrices), dim3(512), 0, stream, a);
  return hipGetLastError();
}

}  // namespace dmuon
