// grxDNN RMSNorm / LayerNorm forward on gfx950.
//
// New (the reference plans grxDNN normalisation but ships none:
// ref docs/designs/grxcp_roadmap.md:864-877). HBM-bound: every byte of x is
// read once and every byte of y written once, so the design goal is streaming
// bandwidth, not arithmetic.
//
//  * rows of up to 256 16-byte chunks (2048 bf16): one row per 64-lane
//    wavefront, held packed in registers between the statistics pass and the
//    output pass; both statistics are in-register wave reductions, so there
//    is no LDS and no barrier and every wave streams independently;
//  * longer rows (up to 16384 chunks, every length the entry points take):
//    one row per workgroup of chunks/2 threads (256, 512 or 1024), two
//    chunks per thread held in registers (four, eight or sixteen past 2048
//    chunks), one LDS combine per statistic; x is still read from HBM
//    exactly once;
//  * 16-byte non-temporal loads of x and stores of y, gamma/beta via the
//    normal cached path (every row reuses them);
//  * statistics in fp32: wavefront butterfly (DPP and row swaps) then an LDS
//    combine of the waves' partials, summed in a fixed order so every thread
//    sees the same value.
//    LayerNorm's variance is the two-pass (x - mean)^2 form over the cached
//    registers, which costs no extra memory traffic.
//  * rows whose length, pitch or base alignment rule out 16-byte boundaries
//    run the same kernels: those of a wavefront as whole chunks at element
//    alignment, of which the last ends with the row (WholeChunks), longer ones
//    on memory's 16-byte boundaries with a partial first and last chunk
//    (RowChunks, AL = false).

#include "../launch.h"
#include "device_common.h"
#include "row_io.h"

namespace grxk {
namespace {

constexpr u32x4 kZero = {0, 0, 0, 0};

struct NParams {
  const uint8_t* x;
  const uint8_t* gamma;
  const uint8_t* beta;
  uint8_t* y;
  int64_t x_rs, y_rs;  // row strides, elements
  int64_t rows;
  int rows_per_wg;     // norm_block: adjacent rows per workgroup
  int hidden;
  float eps;
  int align_mask;      // unaligned rows: RowChunks (before eps it split the aligned
                       // kernels' argument loads: 1-2 % slower)
};

// One row per NT-thread workgroup, NQ 16-byte chunks per thread (chunk
// tid + NT*q), for rows longer than a wavefront handles well. Measured on
// 268 MB of bf16 rows: two chunks per thread with NT = chunks/2 streams at
// 6.2-6.3 TB/s, against 5.6-5.8 TB/s for one row per wavefront at these
// lengths. Each statistic is one wave butterfly plus one barrier; the waves'
// partials are summed in a fixed order, so every thread sees the same value.
// On large inputs a workgroup takes two adjacent rows, with gamma and beta
// loaded once into registers (blocks of rows_per_wg rows, strided by the
// grid). Measured at 16384 x 8192 bf16, five interleaved repeats: one row per
// workgroup re-reads gamma (and beta) per row, and their per-workgroup read
// from L2 costs 3 % (a copy without gamma: 6460 against 6270 GB/s); two rows
// a grid stride apart took LayerNorm from 5960 to 6050 GB/s but RMSNorm
// down 0.8 %; two adjacent rows: RMSNorm 6250 -> 6310, LayerNorm 6050 ->
// 6120; four or eight rows per workgroup, sharing gamma through LDS between
// the halves of a 1024-thread workgroup, or prefetching the next row's x
// measured slower. The partials alternate between two LDS slots by row, so
// a wave still reading one row's partials cannot see the next row's writes,
// and the loop needs no barrier of its own.
template <NormType T, bool AL, bool LAYER, int NT, int NQ>
__global__ __launch_bounds__(NT) void norm_block(NParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  constexpr int NW = NT / 64;
  __shared__ float red[2][2][NW];   // [row parity][statistic][wave]
  const int tid = threadIdx.x;
  const float inv_h = 1.0f / (float)p.hidden;
  int parity = 0;
  auto combine = [&](float v, int slot) {
    v = wave_sum(v);
    if ((tid & 63) == 0) red[parity][slot][tid >> 6] = v;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += red[parity][slot][w];
    return t;
  };
  // gamma and beta are held beside the row (aligned rows: for all rows of
  // the workgroup; others have their chunks at offsets of their own). With
  // more than 4 chunks per thread the registers hold the row alone, and gamma
  // and beta are read when they are used (16 chunks of fp32, LayerNorm, still
  // spill 24 registers).
  constexpr bool HOLD = NQ <= 4;
  u32x4 graw[HOLD ? NQ : 1], braw[HOLD ? NQ : 1];
  auto weights = [&](const RowChunks<T, AL>& rc) __attribute__((always_inline)) {
    if constexpr (HOLD)
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int c = tid + NT * q;
        graw[q] = rc.template load<false>(p.gamma, c, kZero);
        braw[q] = LAYER ? rc.template load<false>(p.beta, c, kZero) : kZero;
      }
  };
  if constexpr (AL) weights(RowChunks<T, AL>(p.x, p.hidden, 0));

  const int64_t rb = p.rows_per_wg;
  for (int64_t base = (int64_t)blockIdx.x * rb; base < p.rows; base += (int64_t)gridDim.x * rb)
  for (int64_t row = base, rend = min(p.rows, base + rb); row < rend; ++row, parity ^= 1) {
    const uint8_t* xrow = p.x + row * p.x_rs * (int64_t)(16 / V);
    uint8_t* yrow = p.y + row * p.y_rs * (int64_t)(16 / V);
    const RowChunks<T, AL> rc(xrow, p.hidden, p.align_mask);
    u32x4 raw[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      raw[q] = rc.load(xrow, tid + NT * q, kZero);
    }
    if constexpr (!AL) weights(rc);
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      float v[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) s += LAYER ? v[e] : v[e] * v[e];
    }
    s = combine(s, 0);
    // Long rows: only the packed row stays live between the passes.
    if constexpr (NQ >= 8)
#pragma unroll
      for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(raw[q]));
    float mean = 0.0f, inv;
    if (LAYER) {
      mean = s * inv_h;
      float d2 = 0.0f;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int c = tid + NT * q;
        if (!rc.any(c)) continue;
        float v[V];
        IO::unpack(raw[q], v);
        if (AL || rc.whole(c)) {
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const float d = v[e] - mean;
            d2 += d * d;
          }
        } else {
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const float d = rc.has(c, e) ? v[e] - mean : 0.0f;
            d2 += d * d;
          }
        }
      }
      d2 = combine(d2, 1);
      if constexpr (NQ >= 8)
#pragma unroll
        for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(raw[q]));
      inv = 1.0f / sqrtf(d2 * inv_h + p.eps);
    } else {
      inv = 1.0f / sqrtf(s * inv_h + p.eps);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = tid + NT * q;
      if (!rc.any(c)) continue;
      float v[V], g[V], o[V];
      IO::unpack(raw[q], v);
      IO::unpack(HOLD ? graw[HOLD ? q : 0] : rc.template load<false>(p.gamma, c, kZero), g);
      if (LAYER) {
        float b[V];
        IO::unpack(HOLD ? braw[HOLD ? q : 0] : rc.template load<false>(p.beta, c, kZero), b);
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = (v[e] - mean) * inv * g[e] + b[e];
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = v[e] * inv * g[e];
      }
      rc.store(yrow, c, IO::pack(o));
    }
  }
}

// One row per 64-lane wavefront, for rows of up to NC x 64 16-byte chunks:
// the row lives in the wave's registers, both statistics are wave
// reductions (lane moves only: no LDS, no barrier), so every wave streams
// independently and a CU keeps ~20 rows of loads in flight. Rows off 16-byte
// boundaries take WholeChunks: with RowChunks a wave waits for its partial
// chunks one after the other and issues a load per element of them (LayerNorm,
// us, RowChunks / WholeChunks: bf16 2500 x 697 7.1 / 4.8, 2048 x 999 6.7 / 4.8,
// 16384 x 2047 56.9 / 28.1, 16384 x 511 20.5 / 9.0; fp32 2500 x 999 7.1 / 5.6,
// but 8192 x 777 11.6 / 12.7). Only rows shorter than a chunk keep RowChunks.
template <NormType T, class Chunks, bool LAYER, int NC>
__global__ __launch_bounds__(256) void norm_wave(NParams p) {
  using IO = Io<T>;
  constexpr int V = IO::kVec;
  const int lane = threadIdx.x & 63;
  const float inv_h = 1.0f / (float)p.hidden;
  const int64_t nwaves = (int64_t)gridDim.x * 4;

  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < p.rows; row += nwaves) {
    const uint8_t* xrow = p.x + row * p.x_rs * (int64_t)(16 / V);
    uint8_t* yrow = p.y + row * p.y_rs * (int64_t)(16 / V);
    const Chunks rc(xrow, p.hidden, p.align_mask);
    u32x4 raw[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      raw[q] = rc.load(xrow, lane + 64 * q, kZero);
    }
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      float v[V];
      IO::unpack(raw[q], v);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float x = !Chunks::kRepeats || rc.has(lane + 64 * q, e) ? v[e] : 0.0f;
        s += LAYER ? x : x * x;
      }
    }
    // Keep only the packed row live between passes (unpacking again is a
    // couple of ALU ops; holding 8*NC floats would halve the waves per CU).
#pragma unroll
    for (int q = 0; q < NC; ++q) asm volatile("" : "+v"(raw[q]));
    s = wave_sum(s);
    float mean = 0.0f, inv;
    if (LAYER) {
      mean = s * inv_h;
      float d2 = 0.0f;
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        const int c = lane + 64 * q;
        if (!rc.any(c)) continue;
        float v[V];
        IO::unpack(raw[q], v);
        if (rc.whole(c)) {
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const float d = v[e] - mean;
            d2 += d * d;
          }
        } else {
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const float d = rc.has(c, e) ? v[e] - mean : 0.0f;
            d2 += d * d;
          }
        }
      }
      d2 = wave_sum(d2);
#pragma unroll
      for (int q = 0; q < NC; ++q) asm volatile("" : "+v"(raw[q]));
      inv = 1.0f / sqrtf(d2 * inv_h + p.eps);
    } else {
      inv = 1.0f / sqrtf(s * inv_h + p.eps);
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int c = lane + 64 * q;
      if (!rc.any(c)) continue;
      float v[V], g[V], o[V];
      IO::unpack(raw[q], v);
      IO::unpack(rc.template load<false>(p.gamma, c, kZero), g);
      if (LAYER) {
        float b[V];
        IO::unpack(rc.template load<false>(p.beta, c, kZero), b);
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = (v[e] - mean) * inv * g[e] + b[e];
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = v[e] * inv * g[e];
      }
      rc.store(yrow, c, IO::pack(o));
    }
  }
}

template <NormType T, bool AL, bool LAYER>
hipError_t run_rows(NParams p, hipStream_t s) {
  constexpr int V = Io<T>::kVec;
  const int nchunks = (p.hidden + V - 1) / V;   // at most 65536 / V (the entry points' limit)
  if (p.hidden > 65536) return hipErrorNotSupported;
  const unsigned wgrid = (unsigned)std::min<int64_t>((p.rows + 3) / 4, 1 << 30);
  // norm_block: two adjacent rows per workgroup where that still leaves at
  // least four workgroups per CU
  p.rows_per_wg = p.rows >= 2048 ? 2 : 1;
  const unsigned bgrid =
      (unsigned)std::min<int64_t>((p.rows + p.rows_per_wg - 1) / p.rows_per_wg, 1 << 30);
  // Past 2048 chunks aligned rows run fastest on 1024 threads, others on 512
  // with twice the chunks (RMSNorm 4096 x 32000 bf16 92 us against 102;
  // LayerNorm 4096 x 32001 128 against 151). Element-wise passes re-reading
  // x, which such rows took before: 2 x 45008 73 us, now 7.
  // cap: chunks the kernel holds. A row off its boundaries takes one chunk
  // more (its first and last are partial) where a kernel has room for it.
  const int need = nchunks + (AL ? 0 : 1);
  auto go = [&](auto kern, int cap, unsigned grid, int threads) {
    grid = (unsigned)std::min<int64_t>(grid, max_workgroups(threads));   // the kernels loop over more rows
    p.align_mask = need <= cap ? V - 1 : 0;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), 0, s, p);
  };
  using Wave = std::conditional_t<AL, RowChunks<T, true>, WholeChunks<T>>;
  if (p.hidden < V) go(norm_wave<T, RowChunks<T, AL>, LAYER, 1>, 64, wgrid, 256);
  else if (nchunks <= 64) go(norm_wave<T, Wave, LAYER, 1>, 64, wgrid, 256);
  else if (nchunks <= 128) go(norm_wave<T, Wave, LAYER, 2>, 128, wgrid, 256);
  else if (nchunks <= 256) go(norm_wave<T, Wave, LAYER, 4>, 256, wgrid, 256);
  else if (need <= 512) go(norm_block<T, AL, LAYER, 256, 2>, 512, bgrid, 256);
  else if (need <= 1024) go(norm_block<T, AL, LAYER, 512, 2>, 1024, bgrid, 512);
  else if (need <= 2048) go(norm_block<T, AL, LAYER, 1024, 2>, 2048, bgrid, 1024);
  else if (need <= 4096) go(norm_block<T, AL, LAYER, AL ? 1024 : 512, AL ? 4 : 8>, 4096, bgrid, AL ? 1024 : 512);
  else if (V == 8 || need <= 8192) go(norm_block<T, AL, LAYER, 1024, 8>, 8192, bgrid, 1024);
  else if constexpr (V == 4) go(norm_block<T, AL, LAYER, 1024, 16>, 16384, bgrid, 1024);
  return hipGetLastError();
}

template <NormType T, bool LAYER>
hipError_t run(const NormDesc& d, hipStream_t s) {
  NParams p{};
  p.x = (const uint8_t*)d.x;
  p.gamma = (const uint8_t*)d.gamma;
  p.beta = (const uint8_t*)d.beta;
  p.y = (uint8_t*)d.y;
  p.x_rs = d.x_row_stride;
  p.y_rs = d.y_row_stride;
  p.rows = d.rows;
  p.hidden = d.hidden;
  p.eps = d.eps;
  constexpr int V = Io<T>::kVec;
  auto al = [](const void* q) { return ((uintptr_t)q % 16) == 0; };
  const bool vec = d.hidden % V == 0 && d.x_row_stride % V == 0 && d.y_row_stride % V == 0 &&
                   al(d.x) && al(d.y) && al(d.gamma) && (!LAYER || al(d.beta));
  return vec ? run_rows<T, true, LAYER>(p, s) : run_rows<T, false, LAYER>(p, s);
}

}  // namespace

hipError_t launch_rmsnorm(NormType t, const NormDesc& d, hipStream_t s) {
  switch (t) {
    case NormType::BF16: return run<NormType::BF16, false>(d, s);
    case NormType::F16:  return run<NormType::F16, false>(d, s);
    case NormType::F32:  return run<NormType::F32, false>(d, s);
  }
  return hipErrorNotSupported;
}

hipError_t launch_layernorm(NormType t, const NormDesc& d, hipStream_t s) {
  switch (t) {
    case NormType::BF16: return run<NormType::BF16, true>(d, s);
    case NormType::F16:  return run<NormType::F16, true>(d, s);
    case NormType::F32:  return run<NormType::F32, true>(d, s);
  }
  return hipErrorNotSupported;
}

}  // namespace grxk
