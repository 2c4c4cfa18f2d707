// grxDNN softmax (over the last dimension) and GELU forward on gfx950.
//
// New: the reference plans both for grxDNN (ref
// docs/designs/grxcp_roadmap.md:864-877, grxcp_architecture.md:594) and ships
// neither. Both are HBM-bound streams: x is read once and y written once.
//
// Softmax, rows of up to 256 16-byte chunks: one row per wavefront, held
// packed in registers; the row max and the sum of exp(x - max) are in-register
// wave reductions (no LDS, no barrier). Up to 16384 chunks: one row per workgroup,
// two to sixteen chunks per thread in registers, one LDS combine per statistic.
// y = exp(x - max) / sum in fp32, rounded once (16-bit outputs use the
// hardware exp2, fp32 the library expf). Longer rows: one row per workgroup,
// three passes (max, sum, write) re-reading x.
// GELU: one 16-byte chunk per thread, over the tensor as one array when its
// rows are contiguous, else row by row; erf or tanh form in fp32, rounded once.
// Rows off 16-byte boundaries (an odd length or pitch) run the same kernels
// (AL = false) on chunks that lie on memory's 16-byte boundaries, the first and
// last of a row partial (RowChunks); where a kernel has no room for one chunk
// more, and for contiguous GELU, at element alignment with a partial end.

#include "../launch.h"
#include "device_common.h"
#include "row_io.h"

namespace grxk {
namespace {

// exp(d) for d <= 0. 16-bit outputs take the hardware exp2 of d*log2(e)
// (relative error well under their half ulp); fp32 keeps the library expf.
template <NormType T> __device__ __forceinline__ float exp_le0(float d) {
  if constexpr (T == NormType::F32) return expf(d);
  else return __builtin_amdgcn_exp2f(d * 1.4426950408889634f);
}

// Pairwise sum of N (a power of two) values: a few roundings deep instead of N.
template <int N> __device__ __forceinline__ float tree_sum(const float* v) {
  if constexpr (N == 1) return v[0];
  else return tree_sum<N / 2>(v) + tree_sum<N / 2>(v + N / 2);
}

// A chunk of -inf: adds nothing to a row's maximum or sum (a row whose
// maximum is -inf itself gives NaN either way).
template <NormType T> __device__ __forceinline__ u32x4 neg_inf() {
  constexpr uint32_t w = T == NormType::F32 ? 0xff800000u : T == NormType::BF16 ? 0xff80ff80u : 0xfc00fc00u;
  return u32x4{w, w, w, w};
}

struct RParams {
  const uint8_t* x;
  uint8_t* y;
  int64_t x_rs, y_rs;  // row strides, elements
  int64_t rows;
  int hidden;
  int align_mask;      // unaligned rows: RowChunks
};

template <NormType T, bool AL, int NC>
__global__ __launch_bounds__(256) void softmax_wave(RParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < p.rows; row += nwaves) {
    const uint8_t* xrow = p.x + row * p.x_rs * (int64_t)(16 / V);
    uint8_t* yrow = p.y + row * p.y_rs * (int64_t)(16 / V);
    const RowChunks<T, AL> rc(xrow, p.hidden, p.align_mask);
    u32x4 raw[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      raw[q] = rc.load(xrow, lane + 64 * q, neg_inf<T>());
    }
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      if (!rc.any(lane + 64 * q)) continue;
      float v[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) mx = fmaxf(mx, v[e]);
    }
    mx = wave_max(mx);
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      if (!rc.any(lane + 64 * q)) continue;
      float v[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = exp_le0<T>(v[e] - mx);
      if constexpr (T == NormType::F32) raw[q] = IO::pack(v);
      sum += tree_sum<V>(v);
    }
    // Keep only the packed row live between passes.
#pragma unroll
    for (int q = 0; q < NC; ++q) asm volatile("" : "+v"(raw[q]));
    const float inv = 1.0f / wave_sum(sum);
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int c = lane + 64 * q;
      if (!rc.any(c)) continue;
      float v[V], o[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = (T == NormType::F32 ? v[e] : exp_le0<T>(v[e] - mx)) * inv;
      rc.store(yrow, c, IO::pack(o));
    }
  }
}

// One row per NT-thread workgroup, NQ 16-byte chunks per thread (chunk
// tid + NT*q), held in registers: the streaming layout that measured fastest
// for rows of 2K-32K 16-bit elements (chunks/2 threads of two chunks each).
// The row max and the sum are each a wave butterfly plus one LDS combine of
// the waves' partials in a fixed order, identical in every thread.
template <NormType T, bool AL, int NT, int NQ>
__global__ __launch_bounds__(NT) void softmax_block(RParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  constexpr int NW = NT / 64;
  __shared__ float red[2][NW];
  const int tid = threadIdx.x;
  for (int64_t row = blockIdx.x; row < p.rows; row += gridDim.x) {
    const uint8_t* xrow = p.x + row * p.x_rs * (int64_t)(16 / V);
    uint8_t* yrow = p.y + row * p.y_rs * (int64_t)(16 / V);
    const RowChunks<T, AL> rc(xrow, p.hidden, p.align_mask);
    u32x4 raw[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      raw[q] = rc.load(xrow, tid + NT * q, neg_inf<T>());
    }
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (!rc.any(tid + NT * q)) continue;
      float v[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) mx = fmaxf(mx, v[e]);
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[0][tid >> 6] = mx;
    __syncthreads();
    mx = red[0][0];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, red[0][w]);
    // Long rows: only the packed row stays live between the passes (else the
    // compiler keeps the unpacked values, and spills).
    auto hold = [&]() __attribute__((always_inline)) {
      if constexpr (NQ >= 8)
#pragma unroll
        for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(raw[q]));
    };
    hold();
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (!rc.any(tid + NT * q)) continue;
      float v[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = exp_le0<T>(v[e] - mx);
      if constexpr (T == NormType::F32) raw[q] = IO::pack(v);
      sum += tree_sum<V>(v);
    }
    sum = wave_sum(sum);
    if ((tid & 63) == 0) red[1][tid >> 6] = sum;
    __syncthreads();
    sum = tree_sum<NW>(red[1]);
    const float inv = 1.0f / sum;
    hold();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = tid + NT * q;
      if (!rc.any(c)) continue;
      float v[V], o[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = (T == NormType::F32 ? v[e] : exp_le0<T>(v[e] - mx)) * inv;
      rc.store(yrow, c, IO::pack(o));
    }
    // Only a grid of fewer workgroups than rows (max_workgroups) loops: the
    // next row's partials must not land before every wave has read these.
    if (row + gridDim.x < p.rows) __syncthreads();
  }
}

// Rows of more than 16384 chunks: one row per 1024-thread workgroup, three
// passes (max, sum, write) re-reading x, four chunks in flight per thread.
template <NormType T, bool AL>
__global__ __launch_bounds__(1024) void softmax_rows(RParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  constexpr int NT = 1024, NW = NT / 64, U = 4;
  __shared__ float red[2][NW];
  const int tid = threadIdx.x;
  for (int64_t row = blockIdx.x; row < p.rows; row += gridDim.x) {
    const uint8_t* xrow = p.x + row * p.x_rs * (int64_t)(16 / V);
    uint8_t* yrow = p.y + row * p.y_rs * (int64_t)(16 / V);
    const RowChunks<T, AL> rc(xrow, p.hidden, p.align_mask);
    // f(chunk index, its values) for the thread's chunks of the row
    auto each = [&](auto f) __attribute__((always_inline)) {
      for (int c0 = tid; rc.any(c0); c0 += U * NT) {
        u32x4 raw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) raw[u] = rc.template load<false>(xrow, c0 + NT * u, neg_inf<T>());
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (!rc.any(c0 + NT * u)) continue;
          float v[V];
          IO::unpack(raw[u], v);
          f(c0 + NT * u, v);
        }
      }
    };
    float mx = -INFINITY;
    each([&](int, float* v) {
#pragma unroll
      for (int e = 0; e < V; ++e) mx = fmaxf(mx, v[e]);
    });
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[0][tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, red[0][w]);
    float sum = 0.0f;
    each([&](int, float* v) {
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = exp_le0<T>(v[e] - mx);
      sum += tree_sum<V>(v);
    });
    sum = wave_sum(sum);
    if ((tid & 63) == 0) red[1][tid >> 6] = sum;
    __syncthreads();
    sum = tree_sum<NW>(red[1]);
    const float inv = 1.0f / sum;
    each([&](int c, float* v) {
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = exp_le0<T>(v[e] - mx) * inv;
      rc.store(yrow, c, IO::pack(v));
    });
    __syncthreads();   // the next row's partials must not land before every wave has read these
  }
}

// Standard normal CDF, Phi(x) = erfc(-x / sqrt 2) / 2, through the Chebyshev
// fit of erfc in Press et al., Numerical Recipes in C (2nd ed., section 6.2,
// erfcc): erfc(z) = t exp(-z^2 + Q(t)), t = 1 / (1 + z/2), z >= 0, fractional
// error below 1.2e-7 for every z (1.05e-7 measured in float64 against scipy).
// The sign of x picks erfc(|z|)/2 or 1 - erfc(|z|)/2, so a small result is
// never the difference of two numbers near 1 (1 + erff(x / sqrt 2) is 0 in
// fp32 from x = -5.4 on), and no branch splits a wave. One reciprocal, one
// exp2 and 17 other VALU instructions (16384 x 8192 bf16: 5980 GB/s, against
// 5032 with the library erff and 3061 with the library erfcf, whose
// interval branches make it compute-bound).
__device__ __forceinline__ float normal_cdf(float x) {
  const float z = fabsf(x) * 0.7071067811865476f;
  const float t = __builtin_amdgcn_rcpf(fmaf(0.5f, z, 1.0f));
  float q = 0.17087277f;
  q = fmaf(t, q, -0.82215223f);
  q = fmaf(t, q, 1.48851587f);
  q = fmaf(t, q, -1.13520398f);
  q = fmaf(t, q, 0.27886807f);
  q = fmaf(t, q, -0.18628806f);
  q = fmaf(t, q, 0.09678418f);
  q = fmaf(t, q, 0.37409196f);
  q = fmaf(t, q, 1.00002368f);
  q = fmaf(t, q, -1.26551223f);
  const float a = fmaf(-z, z, q);                          // ln(erfc(z) / t)
  // erfc(z) / 2 = t * 2^(a log2(e) - 1)
  const float h = t * __builtin_amdgcn_exp2f(fmaf(a, 1.4426950408889634f, -1.0f));
  return x < 0.0f ? h : 1.0f - h;
}

// The tanh form uses x/2 (1 + tanh z) = x * sigmoid(2z) = x / (1 + exp(-2z)):
// one hardware exp2 and one reciprocal instead of a library tanh. The erf
// form is x * Phi(x) with Phi as above. Neither forms 1 + erf or 1 + tanh,
// which cancel in the negative tail, so small results keep their relative
// precision.
template <bool TANH> __device__ __forceinline__ float gelu(float x) {
  if (TANH) {
    const float z = 0.7978845608028654f * (x + 0.044715f * x * x * x);  // sqrt(2/pi)(x + 0.044715 x^3)
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.8853900817779268f * z));  // 2 log2(e)
  }
  return x * normal_cdf(x);
}

template <NormType T, bool TANH, bool AL>
__global__ __launch_bounds__(256) void gelu_vec(RParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  const int nchunks = (p.hidden + V - 1) / V + (AL ? 0 : 1);
  const int64_t total = p.rows * nchunks;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
    const int64_t row = i / nchunks;
    const int c = (int)(i - row * nchunks);
    const uint8_t* xrow = p.x + row * p.x_rs * (int64_t)(16 / V);
    const RowChunks<T, AL> rc(xrow, p.hidden, V - 1);
    if (!rc.any(c)) continue;
    float v[V];
    IO::unpack(rc.load(xrow, c, u32x4{0, 0, 0, 0}), v);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = gelu<TANH>(v[e]);
    rc.store(p.y + row * p.y_rs * (int64_t)(16 / V), c, IO::pack(v));
  }
}

// Contiguous rows (pitch == hidden): the tensor is one array of chunks, one
// chunk per thread, no row arithmetic. The elements past the last whole chunk
// of the array go one to a thread.
template <NormType T, bool TANH, bool AL>
__global__ __launch_bounds__(256) void gelu_flat(RParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  const int64_t elems = p.rows * p.hidden, total = elems / V;
  const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = first; i < total; i += stride) {
    float v[V];
    const RowChunks<T, AL> rc(p.x, V, 0);
    IO::unpack(rc.load(p.x + i * 16, 0, u32x4{0, 0, 0, 0}), v);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = gelu<TANH>(v[e]);
    rc.store(p.y + i * 16, 0, IO::pack(v));
  }
  if (first < elems - total * V) IO::st(p.y, total * V + first, gelu<TANH>(IO::ld(p.x, total * V + first)));
}

RParams make_params(const RowDesc& d) {
  RParams p{};
  p.x = (const uint8_t*)d.x;
  p.y = (uint8_t*)d.y;
  p.x_rs = d.x_row_stride;
  p.y_rs = d.y_row_stride;
  p.rows = d.rows;
  p.hidden = d.hidden;
  return p;
}

bool on16(const void* q) { return (uintptr_t)q % 16 == 0; }

template <NormType T>
bool vec_layout(const RowDesc& d) {
  constexpr int V = Io<T>::kVec;
  return d.hidden % V == 0 && d.x_row_stride % V == 0 && d.y_row_stride % V == 0 && on16(d.x) && on16(d.y);
}

template <NormType T, bool AL>
hipError_t run_softmax(const RowDesc& d, hipStream_t s) {
  constexpr int V = Io<T>::kVec;
  RParams p = make_params(d);
  const int nchunks = (d.hidden + V - 1) / V;
  const unsigned wgrid = (unsigned)std::min<int64_t>((d.rows + 3) / 4, 1 << 30);
  const unsigned bgrid = (unsigned)std::min<int64_t>(d.rows, 1 << 30);
  // Threads per row (each pair in one run): 4096 x 32000 bf16 86 us with 1024
  // threads of 4 chunks, 91 with 512 of 8, but 117 against 97 at 32001;
  // 2048 x 32000 fp32 107 us with 1024 of 8, 94 with 512 of 16, 104 at 32001
  // (264 in three element-wise passes); 1024 x 65536 fp32 112 us with 1024 of
  // 16, 117 with 512 of 32.
  // cap: chunks the kernel holds. A row off its boundaries takes one chunk
  // more (its first and last are partial) where a kernel has room for it.
  const int need = nchunks + (AL ? 0 : 1);
  auto go = [&](auto kern, int cap, unsigned grid, int threads) {
    grid = (unsigned)std::min<int64_t>(grid, max_workgroups(threads));   // the kernels loop over more rows
    p.align_mask = need <= cap ? V - 1 : 0;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), 0, s, p);
  };
  if (need <= 64) go(softmax_wave<T, AL, 1>, 64, wgrid, 256);
  else if (need <= 128) go(softmax_wave<T, AL, 2>, 128, wgrid, 256);
  else if (need <= 256) go(softmax_wave<T, AL, 4>, 256, wgrid, 256);
  else if (need <= 512) go(softmax_block<T, AL, 256, 2>, 512, bgrid, 256);
  else if (need <= 1024) go(softmax_block<T, AL, 512, 2>, 1024, bgrid, 512);
  else if (need <= 2048) go(softmax_block<T, AL, 1024, 2>, 2048, bgrid, 1024);
  else if (need <= 4096) go(softmax_block<T, AL, AL ? 1024 : 512, AL ? 4 : 8>, 4096, bgrid, AL ? 1024 : 512);
  else if (need <= 8192) go(softmax_block<T, AL, 512, 16>, 8192, bgrid, 512);
  else if (nchunks <= 16384) go(softmax_block<T, AL, 1024, 16>, 16384, bgrid, 1024);
  else go(softmax_rows<T, AL>, 1 << 30, bgrid, 1024);
  return hipGetLastError();
}

template <NormType T>
hipError_t run_softmax(const RowDesc& d, hipStream_t s) {
  return vec_layout<T>(d) ? run_softmax<T, true>(d, s) : run_softmax<T, false>(d, s);
}

template <NormType T, bool TANH>
hipError_t run_gelu(const RowDesc& d, hipStream_t s) {
  constexpr int V = Io<T>::kVec;
  const RParams p = make_params(d);
  const bool flat = d.rows == 1 || (d.x_row_stride == d.hidden && d.y_row_stride == d.hidden);
  const int64_t items = flat ? (d.rows * d.hidden + V - 1) / V : d.rows * ((d.hidden + V - 1) / V + 1);
  const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((items + 255) / 256, 1 << 20));
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, p); };
  if (flat && on16(d.x) && on16(d.y)) go(gelu_flat<T, TANH, true>);
  else if (flat) go(gelu_flat<T, TANH, false>);
  else if (vec_layout<T>(d)) go(gelu_vec<T, TANH, true>);
  else go(gelu_vec<T, TANH, false>);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_softmax(NormType t, const RowDesc& d, hipStream_t s) {
  switch (t) {
    case NormType::BF16: return run_softmax<NormType::BF16>(d, s);
    case NormType::F16:  return run_softmax<NormType::F16>(d, s);
    case NormType::F32:  return run_softmax<NormType::F32>(d, s);
  }
  return hipErrorNotSupported;
}

hipError_t launch_gelu(NormType t, bool tanh_form, const RowDesc& d, hipStream_t s) {
  switch (t) {
    case NormType::BF16: return tanh_form ? run_gelu<NormType::BF16, true>(d, s) : run_gelu<NormType::BF16, false>(d, s);
    case NormType::F16:  return tanh_form ? run_gelu<NormType::F16, true>(d, s) : run_gelu<NormType::F16, false>(d, s);
    case NormType::F32:  return tanh_form ? run_gelu<NormType::F32, true>(d, s) : run_gelu<NormType::F32, false>(d, s);
  }
  return hipErrorNotSupported;
}

}  // namespace grxk
