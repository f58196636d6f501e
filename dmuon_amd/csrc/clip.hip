// Segmented gradient clipping on gfx950: the two device operations of the reference's fast
// clip path (dmuon/csrc/fast_clip_kernel.cu:34-107), over the same job table.
//
//   sumsq  local_sq[segments[t]] += sum over the job's elements of float(x)^2
//   scale  x <- T(float(x) * coefs[segments[t]])          in place
//
// A job is (tensor t = job_tensor_ids[j], elements [job_offsets[j], +chunk_size) clipped to
// numels[t]). The norm pass runs one 256-thread block per job (one atomic add per job, as in
// the reference); the scale pass, which has no reduction, splits each job into pieces of
// ClipArgs::piece elements (8192), one block per piece, consecutive blocks on consecutive
// pieces: on MI355X that moved the c5 gradients at 5.9 TB/s instead of 5.2 with one block per
// 262144-element job (the addresses the resident blocks touch stay close together). Tensor dtypes use the reference's codes
// (0 fp32, 1 fp16, 2 bf16; fast_clip.py:31-35). Where the reference walks a job with one
// scalar load per thread and reduces through a shared-memory tree, here the aligned middle of
// the job is read in 16-byte vectors (4 fp32 / 8 half-precision values per lane; the norm pass
// keeps four non-temporal loads in flight per lane, the scale pass two vectors), the partial
// sums are reduced across the wave with cross-lane shuffles and across the four waves through
// a 16-byte LDS array, and one lane per block adds the block's sum into local_sq with a
// global float atomic (so, as in the reference, the order of those additions -- and hence the
// last bits of local_sq -- may differ from run to run).
#include "dmuon_amd_internal.h"

namespace dmuon {
namespace {

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

constexpr int CF32 = 0, CF16 = 1, CBF16 = 2;

template <int D>
__device__ __forceinline__ float to_f(uint32_t bits16) {
  if constexpr (D == CF16) return static_cast<float>(__builtin_bit_cast(_Float16, (uint16_t)bits16));
  else return __uint_as_float(bits16 << 16);
}
template <int D>
__device__ __forceinline__ uint32_t from_f(float f) {
  if constexpr (D == CF16) return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
  else return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

template <int D>
__device__ __forceinline__ float load1(const void* p, long long i) {
  if constexpr (D == CF32) return static_cast<const float*>(p)[i];
  else return to_f<D>(static_cast<const uint16_t*>(p)[i]);
}
template <int D>
__device__ __forceinline__ void scale1(void* p, long long i, float c) {
  if constexpr (D == CF32) {
    float* q = static_cast<float*>(p) + i;
    *q = *q * c;
  } else {
    uint16_t* q = static_cast<uint16_t*>(p) + i;
    *q = (uint16_t)from_f<D>(to_f<D>(*q) * c);
  }
}

struct Job {
  int t;
  long long begin, end;
};
__device__ __forceinline__ Job job_of(const ClipArgs& a) {
  Job j;
  j.t = a.job_tensor_ids[blockIdx.x];
  j.begin = a.job_offsets[blockIdx.x];
  j.end = min(j.begin + a.chunk, (long long)a.numels[j.t]);
  return j;
}
// piece blockIdx.x % pieces of job blockIdx.x / pieces (empty past the end of its tensor)
__device__ __forceinline__ Job piece_of(const ClipArgs& a) {
  const long long pieces = (a.chunk + a.piece - 1) / a.piece;
  const long long b = blockIdx.x, job = b / pieces, k = b - job * pieces;
  Job j;
  j.t = a.job_tensor_ids[job];
  const long long end = min(a.job_offsets[job] + a.chunk, (long long)a.numels[j.t]);
  j.begin = min(a.job_offsets[job] + k * a.piece, end);
  j.end = min(j.begin + a.piece, end);
  return j;
}

// vector width in elements of a 16-byte access
template <int D>
constexpr int vw() { return D == CF32 ? 4 : 8; }

template <int D>
__device__ float job_sumsq(const void* p, long long begin, long long end) {
  constexpr int V = vw<D>();
  const bool aligned = (reinterpret_cast<uintptr_t>(p) & 15) == 0;
  long long vs = end, ve = end;
  if (aligned && begin < end) {
    vs = min((begin + V - 1) / V * V, end);
    ve = max(end / V * V, vs);
  }
  // four 16-byte loads in flight per thread, four partial sums
  float s4[4] = {0.f, 0.f, 0.f, 0.f};
  long long i = vs + (long long)V * threadIdx.x;
  for (; i + 3LL * V * 256 < ve; i += 4LL * V * 256) {
    u32x4_t w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (D == CF32) w[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p) + i + u * V * 256));
      else w[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(p) + i + u * V * 256));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (D == CF32) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float x = __uint_as_float(w[u][k]);
          s4[u] += x * x;
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float x0 = to_f<D>(w[u][k] & 0xffff), x1 = to_f<D>(w[u][k] >> 16);
          s4[u] += x0 * x0;
          s4[u] += x1 * x1;
        }
      }
    }
  }
  float s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  for (; i < ve; i += (long long)V * 256) {
    if constexpr (D == CF32) {
      const u32x4_t w = *reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p) + i);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float x = __uint_as_float(w[k]);
        s += x * x;
      }
    } else {
      const u32x4_t w = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(p) + i);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float x0 = to_f<D>(w[k] & 0xffff), x1 = to_f<D>(w[k] >> 16);
        s += x0 * x0;
        s += x1 * x1;
      }
    }
  }
  const long long nh = vs - begin, nt = end - ve;
  for (long long k = threadIdx.x; k < nh + nt; k += 256) {
    const float x = load1<D>(p, k < nh ? begin + k : ve + (k - nh));
    s += x * x;
  }
  return s;
}

template <int D>
__device__ void job_scale(void* p, long long begin, long long end, float c) {
  constexpr int V = vw<D>();
  const bool aligned = (reinterpret_cast<uintptr_t>(p) & 15) == 0;
  long long vs = end, ve = end;
  if (aligned && begin < end) {
    vs = min((begin + V - 1) / V * V, end);
    ve = max(end / V * V, vs);
  }
  auto sc = [&](u32x4_t w) {
    if constexpr (D == CF32) {
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = __float_as_uint(__uint_as_float(w[k]) * c);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = from_f<D>(to_f<D>(w[k] & 0xffff) * c) | (from_f<D>(to_f<D>(w[k] >> 16) * c) << 16);
    }
    return w;
  };
  u32x4_t* base = D == CF32 ? reinterpret_cast<u32x4_t*>(static_cast<float*>(p))
                            : reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(p));
  long long i = vs + (long long)V * threadIdx.x;
  // four vectors in flight per thread; the gradient is streamed once (non-temporal both ways)
  for (; i + 3LL * V * 256 < ve; i += 4LL * V * 256) {
    u32x4_t w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = __builtin_nontemporal_load(base + i / V + u * 256);
#pragma unroll
    for (int u = 0; u < 4; ++u) __builtin_nontemporal_store(sc(w[u]), base + i / V + u * 256);
  }
  for (; i < ve; i += (long long)V * 256) {
    u32x4_t* q = base + i / V;
    *q = sc(*q);
  }
  const long long nh = vs - begin, nt = end - ve;
  for (long long k = threadIdx.x; k < nh + nt; k += 256)
    scale1<D>(p, k < nh ? begin + k : ve + (k - nh), c);
}

__global__ __launch_bounds__(256) void seg_sumsq_kernel(const ClipArgs a) {
  __shared__ float part[4];
  const Job j = job_of(a);
  const void* p = reinterpret_cast<const void*>(a.ptrs[j.t]);
  const int dt = a.dtypes[j.t];
  float s;
  if (dt == CF32) s = job_sumsq<CF32>(p, j.begin, j.end);
  else if (dt == CF16) s = job_sumsq<CF16>(p, j.begin, j.end);
  else s = job_sumsq<CBF16>(p, j.begin, j.end);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) part[wave] = s;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(a.local_sq + a.segments[j.t], (part[0] + part[1]) + (part[2] + part[3]));
}

__global__ __launch_bounds__(256) void seg_scale_kernel(const ClipArgs a) {
  const Job j = piece_of(a);
  if (j.begin >= j.end) return;
  void* p = reinterpret_cast<void*>(a.ptrs[j.t]);
  const int dt = a.dtypes[j.t];
  const float c = a.coefs[a.segments[j.t]];
  if (dt == CF32) job_scale<CF32>(p, j.begin, j.end, c);
  else if (dt == CF16) job_scale<CF16>(p, j.begin, j.end, c);
  else job_scale<CBF16>(p, j.begin, j.end, c);
}

// Sum of squares of each piece, in order and without atomics (so the norms have the same bits on
// every call); an empty piece writes 0.
__global__ __launch_bounds__(256) void clip_partials_kernel(const ClipArgs a, float* partials) {
  __shared__ float part[4];
  const Job j = piece_of(a);
  float s = 0.f;
  if (j.begin < j.end) {
    const void* p = reinterpret_cast<const void*>(a.ptrs[j.t]);
    const int dt = a.dtypes[j.t];
    if (dt == CF32) s = job_sumsq<CF32>(p, j.begin, j.end);
    else if (dt == CF16) s = job_sumsq<CF16>(p, j.begin, j.end);
    else s = job_sumsq<CBF16>(p, j.begin, j.end);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ bool finite(float x) { return __builtin_isfinite(x); }
// min(max_norm / (norm + 1e-6), 1); NaN stays NaN, as torch.clamp keeps it
__device__ __forceinline__ float clip_coef(float norm, float max_norm) {
  const float c = max_norm / (norm + 1e-6f);
  return c > 1.f ? 1.f : c;
}

// From the pieces' sums to norms, coefficients and flags. A wave per tensor sums its pieces in fp64
// in a fixed order, then
//   global:    the tensor norms, each rounded to its tensor's dtype (as torch._foreach_norm
//              returns them), make one norm and one coefficient;
//   otherwise: one norm and coefficient per segment, and the norm of those.
// Few tensors and segments: one block of 16 waves does it all (FINISH_ALL), bounded by latency; it
// takes the place of ~20 torch operations on one-element tensors, about 4 us each on the device and
// more on the host: one transformer layer's gradients (218 M bf16 elements) 251 -> 218 us a call,
// three small ones 99 -> 37 us. That block's loops over tensors and segments are serial chains of
// loads (0.6 us for 16 tensors), so more than kFinishTensors of either take a launch per stage,
// spread over the device: FINISH_TENSORS (16 tensors a block), FINISH_SEGMENTS (a block per segment,
// or the one of the global norm) and FINISH_TOTAL. Norms of 1000 tensors of 16384 bf16 values 52 ->
// 14 us on the device, of 10000 of 4096 455 -> 30; 256 of 65536 would be 26 -> 17, but the host
// takes 4 us more for the two launches.
constexpr int kFinishWaves = 16, kFinishTensors = 256;
enum { FINISH_ALL, FINISH_TENSORS, FINISH_SEGMENTS, FINISH_TOTAL };

// sum over the block; the result is in thread 0
__device__ __forceinline__ double finish_sum(double v, double* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double all = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kFinishWaves; ++w) all += red[w];
  return all;
}
__device__ __forceinline__ void finish_segment(const ClipFinishArgs& a, int g, float norm) {
  a.norms[g] = norm;
  a.coefs[g] = a.has_max ? clip_coef(norm, a.max_norm) : 1.f;
  a.clipped[g] = a.has_max && finite(norm) && norm > a.max_norm;
  a.found_inf[g] = !finite(norm);
}

template <int PART>
__global__ __launch_bounds__(64 * kFinishWaves) void clip_finish_kernel(const ClipFinishArgs a) {
  __shared__ double red[kFinishWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if constexpr (PART == FINISH_ALL || PART == FINISH_TENSORS) {
    const int step = kFinishWaves * gridDim.x;
    for (int t = blockIdx.x * kFinishWaves + wave; t < a.n; t += step) {
      const long long k1 = (long long)a.first_job[t + 1] * a.pieces;
      double s = 0.0;
      for (long long k = (long long)a.first_job[t] * a.pieces + lane; k < k1; k += 64)
        s += (double)a.partials[k];
      s = wave_sum(s);
      if (lane == 0) a.tensor_sq[t] = s;
    }
    if constexpr (PART == FINISH_TENSORS) return;
    __syncthreads();
  }
  if (PART != FINISH_TOTAL && a.global) {
    double s = 0.0;
    for (int t = threadIdx.x; t < a.n; t += 64 * kFinishWaves) {
      float norm = sqrtf((float)a.tensor_sq[t]);
      if (a.dtypes[t] == CF16) norm = to_f<CF16>(from_f<CF16>(norm));
      else if (a.dtypes[t] == CBF16) norm = to_f<CBF16>(from_f<CBF16>(norm));
      s += (double)norm * (double)norm;
    }
    s = finish_sum(s, red);
    if (threadIdx.x == 0) {
      const float total = (float)sqrt(s);
      const float c = a.max_norm / (total + 1e-6f);
      a.norms[0] = total;
      a.coefs[0] = a.has_max ? clip_coef(total, a.max_norm) : 1.f;
      a.clipped[0] = a.has_max && finite(total) && c < 1.f;
      a.found_inf[0] = !finite(total);
    }
    return;
  }
  if constexpr (PART == FINISH_SEGMENTS) {
    double s = 0.0;
    for (int t = threadIdx.x; t < a.n; t += 64 * kFinishWaves)
      if (a.segments[t] == (int)blockIdx.x) s += a.tensor_sq[t];
    s = finish_sum(s, red);
    if (threadIdx.x == 0) finish_segment(a, blockIdx.x, sqrtf((float)s));
    return;
  }
  double all = 0.0;
  if constexpr (PART == FINISH_ALL) {     // of this wave's segments
    for (int g = wave; g < a.n_segments; g += kFinishWaves) {
      double s = 0.0;
      for (int t = lane; t < a.n; t += 64)
        if (a.segments[t] == g) s += a.tensor_sq[t];
      const float norm = sqrtf((float)wave_sum(s));
      if (lane == 0) {
        all += (double)norm * (double)norm;
        finish_segment(a, g, norm);
      }
    }
  } else {
    for (int g = threadIdx.x; g < a.n_segments; g += 64 * kFinishWaves)
      all += (double)a.norms[g] * (double)a.norms[g];
  }
  all = finish_sum(all, red);
  if (threadIdx.x == 0) a.norms[a.n_segments] = (float)sqrt(all);
}

}  // namespace

hipError_t launch_clip_norms(ClipArgs a, const ClipFinishArgs& f, hipStream_t stream) {
  if (f.n <= 0) return hipErrorInvalidValue;
  a.piece = (a.chunk + f.pieces - 1) / f.pieces;
  if (a.n_jobs > 0) {
    if (a.n_jobs > 0x7fffffffLL / f.pieces) return hipErrorInvalidValue;
    // piece_of() counts a job's pieces from chunk and piece: the same number as f.pieces
    if ((a.chunk + a.piece - 1) / a.piece != f.pieces) return hipErrorInvalidValue;
    hipLaunchKernelGGL(clip_partials_kernel, dim3((unsigned)(a.n_jobs * f.pieces)), dim3(256), 0,
                       stream, a, const_cast<float*>(f.partials));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const dim3 one(1), threads(64 * kFinishWaves);
  if (f.n <= kFinishTensors && f.n_segments <= kFinishTensors) {
    hipLaunchKernelGGL(clip_finish_kernel<FINISH_ALL>, one, threads, 0, stream, f);
    return hipGetLastError();
  }
  const unsigned blocks = (unsigned)((f.n + kFinishWaves - 1) / kFinishWaves);
  hipLaunchKernelGGL(clip_finish_kernel<FINISH_TENSORS>, dim3(blocks), threads, 0, stream, f);
  hipLaunchKernelGGL(clip_finish_kernel<FINISH_SEGMENTS>,
                     dim3(f.global ? 1u : (unsigned)f.n_segments), threads, 0, stream, f);
  if (!f.global) hipLaunchKernelGGL(clip_finish_kernel<FINISH_TOTAL>, one, threads, 0, stream, f);
  return hipGetLastError();
}

int clip_pieces(long long n_jobs, long long chunk) {
  // 4096 blocks or more of at least 8192 elements while the jobs allow it: a job of the default
  // 262144 elements is one block's work for 70 us, so a few small gradients left most of the
  // 256 CUs idle; with many jobs a piece is a whole job
  long long pieces = n_jobs > 0 ? (4096 + n_jobs - 1) / n_jobs : 1;
  const long long most = (chunk + 8191) / 8192;
  if (pieces > most) pieces = most;
  if (pieces < 1) pieces = 1;
  const long long piece = (chunk + pieces - 1) / pieces;
  return (int)((chunk + piece - 1) / piece);
}

hipError_t launch_clip_sumsq(const ClipArgs& a, hipStream_t stream) {
  if (a.n_jobs <= 0) return hipSuccess;
  hipLaunchKernelGGL(seg_sumsq_kernel, dim3((unsigned)a.n_jobs), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_clip_scale(ClipArgs a, hipStream_t stream) {
  if (a.n_jobs <= 0) return hipSuccess;
  // 8192-element pieces; longer ones when the grid would exceed 2^31 blocks
  a.piece = 8192;
  long long pieces = (a.chunk + a.piece - 1) / a.piece;
  if (pieces > 0x7fffffffLL / a.n_jobs) {
    pieces = 0x7fffffffLL / a.n_jobs;
    a.piece = (a.chunk + pieces - 1) / pieces;
    pieces = (a.chunk + a.piece - 1) / a.piece;
  }
  hipLaunchKernelGGL(seg_scale_kernel, dim3((unsigned)(a.n_jobs * pieces)), dim3(256), 0, stream,
                     a);
  return hipGetLastError();
}

}  // namespace dmuon
