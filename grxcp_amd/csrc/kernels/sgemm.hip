// grxBLAS fp32 kernels on gfx950: Sgemm / SgemmStridedBatched, and the
// level-1/2 routines (saxpy, sscal, sgemv).
//
// Sgemm replaces the reference's one-thread-per-output kernel
// (ref: src/libs/grxblas/kernels/sgemm.cpp:22-89; 2 global loads per
// multiply-add) with an fp32 matrix-core kernel (v_mfma_f32_32x32x2_f32): a
// 128x128 (or, for problems too small to fill the chip, 64x64 or 32x32) tile
// of C per workgroup, 16- or 32-deep K stages double-buffered through LDS with
// loads that apply op() while staging (all four transposes, ragged shapes,
// any leading dimension). The batch is the grid's z dimension with
// signed element strides (a zero stride broadcasts an operand), exactly the
// reference's one-launch batching (ref: src/libs/grxblas/grxblas.cpp:936-938).
// beta == 0 never reads C (ref: kernels/sgemm.cpp:80-85). Problems that
// fill the GPU with 256x256 tiles run gemm_mfma.hip's TN kernel on fp32
// instead (grxblas.cpp sgemm_batched).
//
// Level 1/2 follow the reference's semantics (ref: kernels/blas12.cpp:41-132):
// BLAS increments (negative walks backwards), sgemv beta == 0 never reads y.

#include "../launch.h"
#include "device_common.h"

#include <algorithm>
#include <type_traits>

namespace grxk {
namespace {

// Four consecutive floats at any 4-byte aligned address: one
// global_load_dwordx4, which gfx950 takes on dword alignment, so columns of an
// odd leading dimension are read 16 bytes at a time too.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct SParams {
  const float* a; const float* b; float* c;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;
  int m, n, k;
  // (probe here keeps the sizes and what follows in separate argument loads:
  // one load of both made the kernel 1-2 % slower, 1970 x 177 x 526 T,T 10.8 ->
  // 11.0 us)
  grxCycleSlot* probe;
  int tiles_m;
  float alpha, beta;
};

// 4 waves (2 x 2) compute an MT x MT tile of C with
// v_mfma_f32_32x32x2_f32 (each wave MT/2 x MT/2, i.e. (MT/64)^2 .. 4 MFMA
// tiles). K advances KK at a time through double-buffered LDS tiles
// As[kk][i] = op(A)[row0+i][k0+kk] and Bs[kk][j] = op(B)[k0+kk][col0+j]; the
// next stage's loads (op() applied while loading, zeros outside the matrix)
// are issued before the current stage's MFMAs and stored after them, one
// barrier per stage. An MFMA k-step reads one float per lane per operand:
// lane l takes row/column l%32 at k = 2s + l/32.
// TA/TB are template parameters, so the staging code has no run-time
// transpose switch. 4 consecutive elements along an operand's contiguous
// dimension are one 16-byte load at float alignment, whatever the leading
// dimension; a stage wholly inside the matrices (decided once per stage,
// uniformly) takes those loads with no per-element guard, other stages the
// guarded path. (Measured at 4096^3:
// 91 -> 129 TFLOP/s against one kernel with run-time transposes and guards,
// 129 -> 134 with the fragment reads one k-step ahead. Slower, same output:
// a pitch that puts k-rows 2s and 2s+1 half the banks apart (3 %: 3 instead
// of 4 workgroups per CU), an XOR-swizzled unpadded layout (4 %), 32-deep
// stages (2 workgroups per CU, 5-9 %), 256x256 tiles (one wave per SIMD,
// 4 %), the next stage's LDS stores moved to mid-stage (no change).)
//
// KG K groups of 4 waves share a tile: group g takes stages g, g + KG, ...
// in LDS buffers of its own, and their accumulators meet pairwise in LDS at
// the end, in group 0, which stores C. It puts more waves on a CU where there
// are few tiles, whose stages would otherwise wait for one load each (1024^3,
// one 64x64 tile per CU: 29.8 us with KG = 1, 27 with 2, 25.7 with 4; two
// stages of loads in flight per group instead: no change).
//
// Tiles at the edge of C read their stages without guards too: rows past m
// (columns past n) of a group repeat the tile's first, and what a group reads
// past m or n along memory stays in its own rows of the product, none of which
// are stored. Guards remain where a stage passes k or the operand's end
// (1000^3 51.8 -> 29.8 us, 4095^3 1616 -> 1099; before, the waves of an edge
// tile took the guarded element loads, and waited for them, in every stage).
//
// MT = 32 (problems of few 64x64 tiles, 512^3 among them): each wave one
// 16x16 tile with v_mfma_f32_16x16x4_f32, K 32 deep per stage (so that the
// staging keeps one 4-element group per thread and operand), rows 33 floats
// apart: over 64 banks that keeps every access of the tile at most 2-way
// conflicted -- the fragment reads (four 16-lane groups at k = 4s .. 4s+3),
// the transposing stores of a K-contiguous operand (8-way at a pitch of 48)
// and the direct stores (4-way at 48); 512^3 30.7 -> 32.0 TFLOP/s, 39 with
// the K groups.
template <int MT, int KK, int KG, bool TA, bool TB>
__global__ __launch_bounds__(256 * KG) __attribute__((amdgpu_waves_per_eu(4, 8)))
void sgemm_mfma(SParams p) {
  constexpr int kK = KK;                // K per stage
  constexpr int WT = MT / 2;            // wave tile edge
  constexpr int NF = WT / 32;           // 32x32 MFMA tiles per wave edge (0 at MT = 32)
  constexpr int PITCH = MT == 32 ? 33 : MT + 4;  // MT + 4: 16-byte aligned rows, 4 workgroups fit a CU's LDS at MT=128
  constexpr int PER = MT * kK / 256;    // elements per thread per operand per stage
  constexpr int kAcc = MT * MT / 256;   // accumulators per thread
  constexpr int kStages = KG * 2 * kK * PITCH;
  constexpr int kMerge = KG > 1 ? KG / 2 * MT * MT : 0;
  // [operand][K group][stage parity][k][row], later the groups' partial sums
  __shared__ float smem[2 * kStages > kMerge ? 2 * kStages : kMerge];
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  float (*As)[kK][PITCH] = (float (*)[kK][PITCH])smem + 2 * kg;
  float (*Bs)[kK][PITCH] = (float (*)[kK][PITCH])smem + 2 * KG + 2 * kg;

  const uint64_t t0 = p.probe ? cycle_now() : 0;
  const int tid = threadIdx.x & 255;    // within the K group
  const int lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  const int tm = blockIdx.x % p.tiles_m;
  const int tn = blockIdx.x / p.tiles_m;
  const int row0 = tm * MT, col0 = tn * MT;
  const int64_t bz = blockIdx.z;
  const float* A = p.a + bz * p.sa;
  const float* B = p.b + bz * p.sb;
  float* C = p.c + bz * p.sc;
  const bool interior = row0 + MT <= p.m && col0 + MT <= p.n;

  // Staging: an operand stage is MT x kK elements read along its storage's
  // contiguous dimension (op(A): i for N, k for T; op(B): k for N, j for T)
  // in groups of 4 consecutive elements; thread t handles groups
  // t + 256*q. Element (cont, other) of a group maps to LDS [kk][i or j].
  constexpr int GPT = PER / 4;  // groups per thread per operand
  float ra[PER], rb[PER];
  // Element (c, o) of a group is X[o*ld + c], valid iff c < lim_cont, o < lim_other.
  auto load_group = [&](const float* X, int64_t ld, int lim_cont, int lim_other,
                        int cont, int other, float* out) {
    const float* q = X + (int64_t)other * ld + cont;
    if (other < lim_other && cont + 3 < lim_cont) {
      const f32x4 v = *(const f32x4u*)q;
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = (other < lim_other && cont + e < lim_cont) ? q[e] : 0.0f;
    }
  };
  // op(A) (m x k): N stores A[k*lda + i] (cont = i), T stores A[i*lda + k] (cont = k).
  // op(B) (k x n): N stores B[j*ldb + k] (cont = k), T stores B[k*ldb + j] (cont = j).
  // Where each group starts in the first stage, for stages read without
  // guards. Groups wholly past m (n) read the tile's first row (column)
  // instead: what they hold only reaches rows and columns of C that are not
  // stored.
  const float* ga[GPT];
  const float* gb[GPT];
#pragma unroll
  for (int q = 0; q < GPT; ++q) {
    const int e = 4 * (tid + 256 * q);
    const int ia = TA ? e / kK : e % MT, ka = TA ? e % kK : e / MT;
    const int ib = TB ? e % MT : e / kK, kb = TB ? e / MT : e % kK;
    const int64_t i = row0 + ia < p.m ? row0 + ia : row0, j = col0 + ib < p.n ? col0 + ib : col0;
    ga[q] = A + (TA ? i * p.lda + ka : ka * p.lda + i);
    gb[q] = B + (TB ? kb * p.ldb + j : j * p.ldb + kb);
  }
  // A group that straddles m (n) along memory reads up to 3 floats past it:
  // the next columns' (rows') values, inside the operand while at least 3
  // floats of later k follow.
  const int64_t slack_ld = !TA && TB ? min(p.lda, p.ldb) : TB ? p.ldb : p.lda;
  auto load = [&](int k0) {
    // One uniform decision per stage: the unguarded path is straight-line code.
    if (k0 + kK <= p.k && (interior || (TA && !TB) || (p.k - k0 - kK) * slack_ld >= 3)) {
#pragma unroll
      for (int q = 0; q < GPT; ++q) {
        const f32x4 va = *(const f32x4u*)(ga[q] + (TA ? (int64_t)k0 : k0 * p.lda));
        const f32x4 vb = *(const f32x4u*)(gb[q] + (TB ? k0 * p.ldb : (int64_t)k0));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ra[4 * q + e] = va[e];
          rb[4 * q + e] = vb[e];
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < GPT; ++q) {
        const int e = 4 * (tid + 256 * q);
        if (TA) load_group(A, p.lda, p.k, p.m, k0 + e % kK, row0 + e / kK, &ra[4 * q]);
        else load_group(A, p.lda, p.m, p.k, row0 + e % MT, k0 + e / MT, &ra[4 * q]);
        if (TB) load_group(B, p.ldb, p.n, p.k, col0 + e % MT, k0 + e / MT, &rb[4 * q]);
        else load_group(B, p.ldb, p.k, p.n, k0 + e % kK, col0 + e / kK, &rb[4 * q]);
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < GPT; ++q) {
      const int e = 4 * (tid + 256 * q);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (TA) As[buf][e % kK + v][e / kK] = ra[4 * q + v];
        else As[buf][e / MT][e % MT + v] = ra[4 * q + v];
        if (TB) Bs[buf][e / MT][e % MT + v] = rb[4 * q + v];
        else Bs[buf][e % kK + v][e / kK] = rb[4 * q + v];
      }
    }
  };

  auto first = [&]() __attribute__((always_inline)) {
    if (kg * kK < p.k || kg == 0) {
      load(kg * kK);
      store(0);
    }
    __syncthreads();
  };
  // Sum of the K groups' accumulators, at(0 .. kAcc-1) of each thread, in
  // group 0, pairwise; false in the groups that are done.
  auto merge = [&](auto at) __attribute__((always_inline)) {
#pragma unroll
    for (int half = KG / 2; half >= 1; half /= 2) {
      if (kg >= half && kg < 2 * half)
#pragma unroll
        for (int e = 0; e < kAcc; ++e) smem[((kg - half) * kAcc + e) * 256 + tid] = at(e);
      __syncthreads();
      if (kg < half)
#pragma unroll
        for (int e = 0; e < kAcc; ++e) at(e) += smem[(kg * kAcc + e) * 256 + tid];
      if (half > 1) __syncthreads();
    }
    return kg == 0;
  };

  // C = alpha*acc + beta*C (col-major) for a lane's run of 4 rows i0.. of
  // column gj: one 16-byte non-temporal store where the run lies inside C and
  // C's columns are 16-byte aligned, element by element otherwise (same
  // arithmetic).
  const bool vec = (p.ldc & 3) == 0 && ((uintptr_t)C & 15) == 0;
  auto run4 = [&](int i0, int gj, const float* v) __attribute__((always_inline)) {
    float* cp = C + (int64_t)gj * p.ldc + i0;
    if (vec && i0 + 4 <= p.m) {
      f32x4 o;
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = __fmul_rn(p.alpha, v[q]);
      if (p.beta != 0.0f) {
        const f32x4 old = *(const f32x4*)cp;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = __fadd_rn(o[q], __fmul_rn(p.beta, old[q]));
      }
      __builtin_nontemporal_store(o, (f32x4*)cp);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (i0 + q >= p.m) break;
        const float x = __fmul_rn(p.alpha, v[q]);
        cp[q] = (p.beta == 0.0f) ? x : __fadd_rn(x, __fmul_rn(p.beta, cp[q]));
      }
    }
  };

  if constexpr (MT == 32) {
    // One 16x16 tile per wave: lane l reads op(A) row 16*wm + l%16 and op(B)
    // column 16*wn + l%16 at k = 4s + l/16, and holds rows 4*(l/16) .. +3 of
    // column l%16 of the result.
    const int r16 = lane & 15, kq = lane >> 4;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    int buf = 0;
    first();
    for (int kb = 0; kb < p.k; kb += KG * kK) {
      const int k0 = kb + kg * kK;
      const bool more = k0 + KG * kK < p.k;
      if (more) load(k0 + KG * kK);
      float av[kK / 4], bv[kK / 4];
#pragma unroll
      for (int st = 0; st < kK / 4; ++st) {
        av[st] = As[buf][4 * st + kq][16 * wm + r16];
        bv[st] = Bs[buf][4 * st + kq][16 * wn + r16];
      }
      if (k0 < p.k)
#pragma unroll
        for (int st = 0; st < kK / 4; ++st)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[st], bv[st], acc, 0, 0, 0);
      if (more) store(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
    if (!merge([&](int e) -> float& { return ((float*)&acc)[e]; })) return;
    const int gj = col0 + 16 * wn + r16;
    const int i0 = row0 + 16 * wm + 4 * kq;
    if (gj < p.n && i0 < p.m) {
      const float v[4] = {acc[0], acc[1], acc[2], acc[3]};
      run4(i0, gj, v);
    }
  } else {
    f32x16 acc[NF][NF];
#pragma unroll
    for (int fm = 0; fm < NF; ++fm)
#pragma unroll
      for (int fn = 0; fn < NF; ++fn)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[fm][fn][r] = 0.0f;

    int buf = 0;
    first();
    for (int kb = 0; kb < p.k; kb += KG * kK) {
      const int k0 = kb + kg * kK;
      const bool more = k0 + KG * kK < p.k;
      if (more) load(k0 + KG * kK);
      // Fragments one k-step ahead: step s+1's LDS reads are issued before
      // step s's MFMAs (the scheduling barriers keep that order), so each
      // wait covers reads issued a whole step earlier.
      float av[2][NF], bv[2][NF];
      if (k0 < p.k) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          av[0][f] = As[buf][hh][WT * wm + 32 * f + l32];
          bv[0][f] = Bs[buf][hh][WT * wn + 32 * f + l32];
        }
#pragma unroll
        for (int s = 0; s < kK / 2; ++s) {
          if (s + 1 < kK / 2) {
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              av[(s + 1) & 1][f] = As[buf][2 * s + 2 + hh][WT * wm + 32 * f + l32];
              bv[(s + 1) & 1][f] = Bs[buf][2 * s + 2 + hh][WT * wn + 32 * f + l32];
            }
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int fm = 0; fm < NF; ++fm)
#pragma unroll
            for (int fn = 0; fn < NF; ++fn)
              acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[s & 1][fm], bv[s & 1][fn], acc[fm][fn],
                                                                 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (more) store(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
    if (!merge([&](int e) -> float& { return ((float*)acc)[e]; })) return;

    // A lane holds column l32 of each MFMA tile and rows 8*(r/4) + 4*hh +
    // r%4: runs of 4 rows.
#pragma unroll
    for (int fm = 0; fm < NF; ++fm)
#pragma unroll
      for (int fn = 0; fn < NF; ++fn) {
        const int gj = col0 + WT * wn + 32 * fn + l32;
        if (gj >= p.n) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int i0 = row0 + WT * wm + 32 * fm + 8 * g + 4 * hh;
          if (i0 >= p.m) continue;
          const float v[4] = {acc[fm][fn][4 * g], acc[fm][fn][4 * g + 1], acc[fm][fn][4 * g + 2],
                              acc[fm][fn][4 * g + 3]};
          run4(i0, gj, v);
        }
      }
  }
  cycle_record(p.probe, t0, (uint32_t)((bz * gridDim.x + blockIdx.x) * 4 + wave), wave);
}

__device__ __forceinline__ int64_t blas_index(int i, int n, int inc) {
  return inc > 0 ? (int64_t)i * inc : (int64_t)(n - 1 - i) * (int64_t)(-inc);
}

// Level-1/2 kernels run 256-thread workgroups; with a cycle probe attached
// every wave writes slot blockIdx*4 + wave, like the GEMM kernels.
__device__ __forceinline__ void l12_record(grxCycleSlot* probe, uint64_t t0) {
  cycle_record(probe, t0, blockIdx.x * 4 + (threadIdx.x >> 6), threadIdx.x >> 6);
}

__global__ void saxpy_kernel(int n, float alpha, const float* x, int incx, float* y, int incy,
                             grxCycleSlot* probe) {
  const uint64_t t0 = probe ? cycle_now() : 0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int64_t xi = blas_index((int)i, n, incx), yi = blas_index((int)i, n, incy);
    y[yi] = fmaf(alpha, x[xi], y[yi]);
  }
  l12_record(probe, t0);
}

__global__ void sscal_kernel(int n, float alpha, float* x, int incx, grxCycleSlot* probe) {
  const uint64_t t0 = probe ? cycle_now() : 0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    x[(int64_t)i * incx] *= alpha;
  l12_record(probe, t0);
}

// Element i of a BLAS vector of n elements lies at base + i * inc.
__device__ __forceinline__ int64_t blas_base(int n, int inc) {
  return inc > 0 ? 0 : (int64_t)(n - 1) * (-(int64_t)inc);
}

// y = alpha*A*x + beta*y (A m x n col-major). One workgroup per 4*lr rows:
// lr lanes cover them, 16 bytes each, and the NT/lr lane groups take every
// (NT/lr)-th column, U columns' loads in flight per thread; the groups' sums
// meet in LDS, in a fixed order. No partial result leaves the workgroup, so
// there is no workspace and no second launch. HBM-bound: 8192 x 4096 26 us,
// 5.2 TB/s; 16384 x 8192 84 us, 6.4 TB/s (one thread per row, a column per
// step, was bound by the latency of its one load in flight: 8192 x 4096
// 970 us). 512 threads with 4 columns in flight were the fastest at every
// size tried (256 or 1024 threads, 8 or 16 columns: equal to 30 % slower).
template <int NT, int U>
__global__ __launch_bounds__(NT) void sgemv_n_kernel(int m, int n, float alpha, const float* A,
                                                     int lda, const float* x, int incx, float beta,
                                                     float* y, int incy, int lr,
                                                     grxCycleSlot* probe) {
  const uint64_t t0 = probe ? cycle_now() : 0;
  __shared__ float part[NT * 4];       // [lane group][row]
  const int tid = threadIdx.x;
  // Neighbouring row blocks share cache lines of every column: give each XCD
  // (workgroups are dealt round-robin over the eight) a contiguous run.
  const int xcd = blockIdx.x & 7, each = gridDim.x >> 3, more = gridDim.x & 7;
  const int64_t row0 = (int64_t)(xcd * each + min(xcd, more) + (int)(blockIdx.x >> 3)) * 4 * lr;
  const int cg = tid / lr, ncg = NT / lr;
  const int64_t row = row0 + 4 * (tid - cg * lr);
  const float* a = A + row;
  const float* xb = x + blas_base(n, incx);
  const bool full = row + 4 <= m;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  if (cg < ncg && row < m) {
    for (int64_t j0 = cg; j0 < n; j0 += U * ncg) {
      f32x4 av[U];
      float xv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // Columns past n repeat the last one and are dropped below.
        const int64_t j = min(j0 + u * ncg, (int64_t)n - 1);
        xv[u] = xb[j * incx];
        if (full) {
          av[u] = *(const f32x4u*)(a + j * lda);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) av[u][e] = row + e < m ? a[j * lda + e] : 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u * ncg < n) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] = fmaf(av[u][e], xv[u], acc[e]);
        }
    }
  }
  *(f32x4*)&part[4 * tid] = acc;       // tid = cg * lr + lane, so rows of a group are adjacent
  // Halve the groups until one is left: group g takes group g + half.
  for (int groups = ncg; groups > 1;) {
    __syncthreads();
    const int half = (groups + 1) >> 1;
    if (cg < groups - half) {
      const f32x4 o = *(const f32x4*)&part[4 * (tid + half * lr)];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += o[e];
      *(f32x4*)&part[4 * tid] = acc;
    }
    groups = half;
  }
  __syncthreads();
  for (int r = tid; r < 4 * lr; r += NT) {
    const int64_t i = row0 + r;
    if (i >= m) break;
    const float t = part[r];
    float* yp = y + blas_index((int)i, m, incy);
    *yp = (beta == 0.0f) ? alpha * t : fmaf(beta, *yp, alpha * t);
  }
  l12_record(probe, t0);
}

// y = alpha*A^T*x + beta*y: WPC waves of a 256-thread workgroup take NC
// columns together, striding down them 16 bytes per lane with x read once for
// all of them; one reduction per column over the lanes, and for WPC = 4 over
// the waves through LDS in a fixed order. HBM-bound: 8192 x 4096 23.7 us, 5.7
// TB/s; 1000 x 8191 7.0 us (4-byte loads, a workgroup per column: 26.1 us
// at 8192 x 4096).
template <int WPC, int NC>
__global__ __launch_bounds__(256) void sgemv_t_kernel(int m, int n, float alpha, const float* A,
                                                      int lda, const float* x, int incx, float beta,
                                                      float* y, int incy, grxCycleSlot* probe) {
  static_assert(WPC == 1 || WPC == 4, "one wave or the whole workgroup per column group");
  const uint64_t t0 = probe ? cycle_now() : 0;
  __shared__ float part[4][NC];
  const int wave = threadIdx.x >> 6;
  const int t = WPC == 4 ? (int)threadIdx.x : (int)threadIdx.x & 63;
  const int j0 = (WPC == 4 ? (int)blockIdx.x : (int)blockIdx.x * 4 + wave) * NC;
  const float* xb = x + blas_base(m, incx);
  float acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0.0f;
  const float* a[NC];   // columns past n repeat the last one; their sums are not stored
#pragma unroll
  for (int c = 0; c < NC; ++c) a[c] = A + (int64_t)min(j0 + c, n - 1) * lda;
  const int m4 = m & ~3;
  constexpr int STEP = 4 * 64 * WPC;
  auto rows4 = [&](int64_t i) __attribute__((always_inline)) {
    f32x4 xv, av[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) av[c] = *(const f32x4u*)(a[c] + i);
    if (incx == 1) {
      xv = *(const f32x4u*)(xb + i);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[e] = xb[(i + e) * incx];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[c] = fmaf(av[c][e], xv[e], acc[c]);
  };
#pragma unroll 4
  for (int64_t i = 4 * t; i < m4; i += STEP) rows4(i);
  if (t < m - m4) {
    const float xv = xb[(int64_t)(m4 + t) * incx];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = fmaf(a[c][m4 + t], xv, acc[c]);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = wave_sum(acc[c]);
  if (WPC == 4) {
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int c = 0; c < NC; ++c) part[wave][c] = acc[c];
    __syncthreads();
  }
  if (t < NC && j0 + t < n) {
    float s = 0.0f;
    if (WPC == 4) {
      s = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c) s = c == t ? acc[c] : s;
    }
    float* yp = y + blas_index(j0 + t, n, incy);
    *yp = (beta == 0.0f) ? alpha * s : fmaf(beta, *yp, alpha * s);
  }
  l12_record(probe, t0);
}

}  // namespace

hipError_t launch_sgemm(const SgemmDesc& d, hipStream_t s) {
  SParams p{};
  p.a = d.a; p.b = d.b; p.c = d.c;
  p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.ldc;
  p.sa = d.stride_a; p.sb = d.stride_b; p.sc = d.stride_c;
  p.m = d.m; p.n = d.n; p.k = d.k;
  p.alpha = d.alpha; p.beta = d.beta;
  p.probe = d.probe;
  if (d.batch > 65535) return hipErrorInvalidValue;
  // Tile and K groups. 128-wide tiles (four workgroups share a CU) where they
  // are three or more per CU: 4095^3 1099 us, 1143 with 64-wide ones; below
  // that 64-wide tiles waste less of the last round (2047^2 x 500, 256 or 1024
  // tiles: 56 / 47 us), and where those are fewer than the CUs, 32-wide ones
  // (512^3 6.8 / 14.0 us, 700^3 13.4 / 18.9). Two K groups overlap one's loads
  // with the other's products; four where a CU has at most about one tile
  // (1000^3 28 -> 26 us, 256^2 x 2048 18.5 -> 16.4; 30.0 with one). A cycle
  // probe's slots are counted for 64-wide tiles and one group.
  const int64_t big = ((int64_t)(d.m + 127) / 128) * ((d.n + 127) / 128) * d.batch;
  const int64_t mid = ((int64_t)(d.m + 63) / 64) * ((d.n + 63) / 64) * d.batch;
  const int64_t small = ((int64_t)(d.m + 31) / 32) * ((d.n + 31) / 32) * d.batch;
  auto go = [&](auto mt_c, auto kg_c) {
    constexpr int MT = decltype(mt_c)::value, KG = decltype(kg_c)::value, KK = MT == 32 ? 32 : 16;
    p.tiles_m = (d.m + MT - 1) / MT;
    const int64_t tiles = (int64_t)p.tiles_m * ((d.n + MT - 1) / MT);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)tiles, 1, (unsigned)d.batch);
    auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256 * KG), 0, s, p); };
    if (d.ta && d.tb) launch(sgemm_mfma<MT, KK, KG, true, true>);
    else if (d.ta) launch(sgemm_mfma<MT, KK, KG, true, false>);
    else if (d.tb) launch(sgemm_mfma<MT, KK, KG, false, true>);
    else launch(sgemm_mfma<MT, KK, KG, false, false>);
    return hipGetLastError();
  };
  using std::integral_constant;
  constexpr integral_constant<int, 128> t128;
  constexpr integral_constant<int, 64> t64;
  constexpr integral_constant<int, 32> t32;
  constexpr integral_constant<int, 1> g1;
  constexpr integral_constant<int, 2> g2;
  constexpr integral_constant<int, 4> g4;
  if (d.probe) return big >= 256 ? go(t128, g1) : go(t64, g1);
  if (big >= 768) return go(t128, g1);
  if (mid >= 256) return mid <= 384 && d.k > 128 ? go(t64, g4) : go(t64, g2);
  return small <= 512 && d.k > 128 ? go(t32, g4) : go(t32, g2);
}

int64_t l1_blocks(int n) { return std::min<int64_t>(((int64_t)n + 255) / 256, 65536); }

int64_t sgemv_blocks(bool trans, int m, int n) { return trans ? n : ((int64_t)m + 255) / 256; }

hipError_t launch_saxpy(int n, float alpha, const float* x, int incx, float* y, int incy,
                        grxCycleSlot* probe, hipStream_t s) {
  hipLaunchKernelGGL(saxpy_kernel, dim3((unsigned)l1_blocks(n)), dim3(256), 0, s, n, alpha, x, incx,
                     y, incy, probe);
  return hipGetLastError();
}

hipError_t launch_sscal(int n, float alpha, float* x, int incx, grxCycleSlot* probe,
                        hipStream_t s) {
  hipLaunchKernelGGL(sscal_kernel, dim3((unsigned)l1_blocks(n)), dim3(256), 0, s, n, alpha, x, incx,
                     probe);
  return hipGetLastError();
}

hipError_t launch_sgemv(bool trans, int m, int n, float alpha, const float* A,
                        int lda, const float* x, int incx, float beta, float* y,
                        int incy, grxCycleSlot* probe, hipStream_t s) {
  // With a cycle probe the launch has the geometry its slots are counted for
  // (sgemv_blocks): a column per workgroup, or 256 rows.
  if (trans) {
    // Two columns per workgroup share each read of x; columns of up to 512
    // rows fit one wave, which then needs no LDS step (128 x 8192: 2.9
    // against 4.7 us; 2047 x 2000: 4.7 us with four waves, 5.9 with one).
    auto go = [&](auto kern, int64_t blocks) {
      hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, s, m, n, alpha, A, lda, x, incx,
                         beta, y, incy, probe);
    };
    if (probe) go(sgemv_t_kernel<4, 1>, sgemv_blocks(true, m, n));
    else if (m <= 512) go(sgemv_t_kernel<1, 2>, ((int64_t)n + 7) / 8);
    else go(sgemv_t_kernel<4, 2>, ((int64_t)n + 1) / 2);
    return hipGetLastError();
  }
  auto go = [&](auto kern, int threads, int lr) {
    hipLaunchKernelGGL(kern, dim3((unsigned)(((int64_t)m + 4 * lr - 1) / (4 * lr))), dim3(threads), 0, s,
                       m, n, alpha, A, lda, x, incx, beta, y, incy, lr, probe);
  };
  // Rows per workgroup: as many as leave one workgroup per CU in the fewest
  // passes over the 256 CUs, since a second workgroup on some CUs doubles the
  // call (9336 x 4451: 45.8 us as 584 workgroups of 16 rows, 62 as 292 of 32,
  // 29.4 as 234 of 40). At least 8, so that a wave's 16-byte loads of one
  // column are 32 bytes together (1000 x 8191: 13.6 us against 14.4 at 4).
  if (probe) {
    go(sgemv_n_kernel<256, 8>, 256, 64);
  } else {
    const int64_t passes = ((int64_t)m + 16383) / 16384;
    const int64_t lr = ((int64_t)m + 1024 * passes - 1) / (1024 * passes);
    go(sgemv_n_kernel<512, 4>, 512, lr < 2 ? 2 : (int)lr);
  }
  return hipGetLastError();
}

}  // namespace grxk
