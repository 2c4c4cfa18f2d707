// grxDNN fused scaled-dot-product attention (forward) on gfx950.
//
// New: the reference plans attention for grxDNN but ships no code
// (ref docs/designs/grxcp_roadmap.md:864-877). Single pass, online softmax,
// O(S) memory:
//
//  * persistent: one workgroup per CU (8 wavefronts, two per SIMD) loops
//    over work items of 256 query rows of one (batch, head); each wave owns
//    32 queries whose Q fragments stay in VGPRs for the item. The K/V loads
//    run across items (an item's last tiles load the next item's first),
//    the next item's Q loads behind the last tile, and O is stored while
//    the next item starts: no workgroup launch, prologue or drain between
//    items (measured ~30K idle cycles per CU between one-shot workgroups,
//    plus ~11K of prologue and epilogue);
//  * K and V stream through LDS in 64-key tiles by direct-to-LDS buffer loads
//    (no staging registers; rows past the sequence read as zero) into three
//    stages, each tile's loads issued two tiles ahead of its use (three
//    stages measured 0.7-2.7 % faster than two with the same waits);
//  * the K fragments of the score MFMAs are read four MFMAs ahead of their
//    use and the two 32-key accumulation chains alternate (pinned with
//    sched_group_barrier; +4 %);
//  * scores are computed TRANSPOSED, S^T = K Q^T (v_mfma_f32_32x32x16): per
//    lane the accumulator holds 32 keys of ONE query, so the softmax row
//    max/sum is an in-register reduction plus one exchange with lane^32;
//  * O^T += V^T P^T: P^T is already in the B-operand layout in the lanes
//    that computed it (no LDS round trip), and the V^T operand is read from
//    the row-major V tile with ds_read_b64_tr_b16 (gfx950's transposing LDS
//    read: 4 keys of one head-dim column per lane), so V is never rewritten;
//  * softmax in the exp2 domain with the running max m tracked in scaled
//    units: p = exp2(s*scale*log2e - m). m is only raised when a tile's max
//    exceeds it by more than 8 (p <= 2^8 otherwise, exact in bf16's relative
//    precision), so the O rescale (and its 128 multiplies) is rare. m starts at
//    the lowest finite float, so that -inf scores have weight 0 whichever tile
//    they fill, and a row of nothing else has l = 0 and comes out NaN;
//  * P is packed with v_cvt_pk_bf16_f32 (round to nearest even); O is
//    divided by the row sum once at the end, rounded once, and leaves
//    through a per-wave LDS region as whole rows (not 8-byte pieces of 32
//    rows per store instruction);
//  * registers: this file is compiled with MFMA results in VGPRs
//    (-amdgpu-mfma-vgpr-form), which keeps the scores, P and O out of
//    AGPR<->VGPR copies (226 VGPRs, two waves per SIMD);
//  * causal: key tiles past the query tile are never loaded; a 32-query block
//    skips tiles entirely above its diagonal; heads are split over the XCDs
//    (all query tiles of a head on one XCD: K/V shared in its L2), each
//    XCD's items are dealt a block of heads at a time, heaviest first, in a
//    snake order, so every CU gets the same number of key tiles (272 of
//    69632 at B4 H32 S4096) and an XCD's CUs share few heads' K/V at a time;
//  * problems whose 256-query items would leave CUs idle take attn_split:
//    items of 128 or 64 queries, a workgroup's waves split over the keys.

#include "../launch.h"
#include "device_common.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>

namespace grxk {
namespace {

constexpr int kNW = 8;          // wavefronts per workgroup (two per SIMD)
constexpr int kBQ = 32 * kNW;   // queries per workgroup, 32 per wave
constexpr int kBK = 64;   // keys per tile
constexpr int kNS = 3;    // K/V tile stages in LDS (96 KB at head dim 128)
constexpr int kQkAhead = 4;  // K fragments read ahead of the score MFMAs
static_assert(kNS == 3, "the tile loop below is unrolled for three stages");
constexpr uint32_t kRsrcWord3 = 0x00020000u;
constexpr float kLowest = -__FLT_MAX__;   // a row's maximum before its first key
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_t;
template <int N> struct Stage { static constexpr int value = N; };

// Buffer descriptor words: 48-bit base, stride 0, num_records bytes (reads
// past it return zero), raw-buffer format word.
__device__ __forceinline__ i32x4 rsrc_words(const void* base, uint32_t num_records) {
  const uint64_t a = (uint64_t)base;
  return i32x4{(int)(uint32_t)a, (int)(uint32_t)(a >> 32) & 0xffff, (int)num_records, (int)kRsrcWord3};
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(lds_ptr_t)p;
}
// 16 bytes per lane from global memory straight into LDS (lane L writes
// lds + 16*L). Issued as assembly so that the compiler does not see an LDS
// write: it would otherwise make every later transposing LDS read wait for
// ALL outstanding DMA, including the prefetch of the next tile. Ordering is
// explicit instead: each tile ends with s_waitcnt vmcnt(0) and a barrier
// before any wave reads the stage this DMA fills. M0 carries the LDS base:
// gfx950 needs one wait state between an M0 write and the LDS DMA that reads
// it (the s_nop; the compiler's hazard pass does not look inside inline
// assembly). M0 is a register the compiler reserves (a clobber naming it is
// ignored), so each DMA writes it itself; in the gfx950 code of this kernel
// and of gemm_tn128 no other instruction reads or writes M0.
// s_waitcnt vmcnt(0) through the builtin, so that the compiler's own wait
// bookkeeping also sees every earlier load as complete.
__device__ __forceinline__ void wait_vmem_all() {
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt 0, expcnt 7, lgkmcnt 15: wait on vmcnt only
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void dma16(i32x4 rsrc, uint32_t lds, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds), "v"(voff), "s"(rsrc) : "memory");
}
// The same with a wave-uniform byte offset in the instruction's soffset. The
// buffer's range check sees only the per-lane offset, so this form is for
// rows known to lie inside the tensor.
__device__ __forceinline__ void dma16_so(i32x4 rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

template <AttnType T> struct AIo;
template <> struct AIo<AttnType::BF16> {
  __device__ static f32x16 mma(i32x4 a, i32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  // two fp32 -> packed bf16 (RNE, v_cvt_pk_bf16_f32)
  __device__ static uint32_t pack2(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
  // acc + the two packed values (v_dot2_f32_bf16 against (1, 1))
  __device__ static float sum2(uint32_t packed, float acc) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, packed), one, acc, false);
  }
};
template <> struct AIo<AttnType::F16> {
  __device__ static f32x16 mma(i32x4 a, i32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  __device__ static uint32_t pack2(float a, float b) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 v = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
  __device__ static float sum2(uint32_t packed, float acc) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, packed), one, acc, false);
  }
};

struct AParams {
  const uint8_t* q; const uint8_t* k; const uint8_t* v; uint8_t* o;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t v_sb, v_sh, v_ss;
  int64_t o_sb, o_sh, o_ss;
  int B, H, S;
  int qtiles;
  int heads;      // B * H
  int hb;         // heads per block of an XCD's items (attn_fwd)
  int causal;
  float c;  // scale * log2(e)
  grxCycleSlot* probe;   // one slot per wave, or null
};

// K rows: ds_read_b128 of one logical chunk by 32 consecutive rows must hit
// distinct banks; V rows: the 8 keys x 4 chunks of one transposing read must
// spread evenly. Both are XOR swizzles of the 16-byte chunk index.
template <int D> __device__ __forceinline__ int kswz(int row) {
  if constexpr (D == 128) return row & 15;
  else return (row ^ (row >> 3)) & 7;
}
template <int D> __device__ __forceinline__ int vswz(int row) {
  if constexpr (D == 128) return 4 * (row & 3);
  else return 4 * ((row >> 1) & 1);
}

// Value from the other half of the wave (lane ^ 32): v_permlane32_swap
// exchanges the upper half of its first operand with the lower half of its
// second; with both operands = x, lane l of the two results holds x[l] and
// x[l ^ 32] in some order.
__device__ __forceinline__ float half_swap_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// A row's new maximum in scaled units, mx * c. From a magnitude on where the
// product's rounding alone would make exp2(mx * c - m) overflow T, it is rounded
// up instead: the weights of a group of hugely negative scores (a mask added to
// them) stay finite, so that group adds 0, not 0 * inf, where others dominate.
template <AttnType T> __device__ __forceinline__ float scaled_max(float mx, float c) {
  constexpr float kDeep = T == AttnType::BF16 ? 0x1p31f : 0x1p28f;   // half an ulp: 2^7, 2^4
  const float m = mx * c;
  const bool up = fabsf(m) >= kDeep && fmaf(mx, c, -m) > 0.0f;
  const int bits = __builtin_bit_cast(int, m);
  return up ? __builtin_bit_cast(float, bits + (m > 0.0f ? 1 : -1)) : m;
}
__device__ __forceinline__ float half_swap_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One work item = one (batch, head) and one tile of kBQ queries. Items are
// split over the 8 XCDs by head (head h on XCD h % 8, so one head's K/V stay
// in one L2). Inside an XCD, round r deals the items of the next block of
// heads (as many heads as one round has workgroups for their query tiles:
// 2 at 32 workgroups and 16 tiles), heaviest (causal: last) query tile
// first, to the XCD's workgroups in a snake order, left to right for even r
// and right to left for odd r: two rounds give every workgroup the same
// number of key tiles, and the workgroups of an XCD share few heads' K/V at
// a time (B4 H32 S4096: FETCH_SIZE 564 MB per launch, against 1420 MB when
// a round took the heaviest tiles of all 16 heads of the XCD). Where a few
// rounds do not come out even that way, all heads are one block (heads_per_block).
struct ItemMap {
  int xcd, wg, nwg;     // this workgroup's XCD, index within it, workgroups per XCD
  int hx;               // heads on this XCD
};
__device__ __forceinline__ bool item_at(const AParams& p, const ItemMap& m, int round,
                                        int* bh, int* qt) {
  const int nloc = m.hx * p.qtiles;
  const int k = (round & 1) ? (m.nwg - 1 - m.wg) : m.wg;
  const int j = round * m.nwg + k;
  if (j >= nloc || m.hx == 0) return false;
  const int hb = min(p.hb, m.hx);     // heads per block
  const int blk_items = hb * p.qtiles;
  const int blk = j / blk_items;
  const int r2 = j - blk * blk_items;
  const int hb_here = min(hb, m.hx - blk * hb);   // the last block may hold fewer
  const int rank = r2 / hb_here;                  // weight rank: 0 = heaviest
  const int hl = blk * hb + r2 % hb_here;
  *bh = m.xcd + 8 * hl;
  *qt = p.causal ? (p.qtiles - 1 - rank) : rank;
  return true;
}

// A lane's place in the fragments: query (and key row) l32, half hh, and the
// key and head-dim offsets of its transposing V reads.
struct LanePos {
  int l32, hh, tr_key, tr_d;
};
__device__ __forceinline__ LanePos lane_pos(int lane) {
  LanePos l;
  l.l32 = lane & 31;
  l.hh = lane >> 5;
  l.tr_key = 4 * l.hh + ((lane & 15) >> 2);
  l.tr_d = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  return l;
}

// One 64-key tile (keys kv0 .. kv0+63; K rows at kt, V rows at vt in LDS) for
// the wave's queries wq0 .. wq0+31: scores, online softmax, O^T += V^T P^T.
template <AttnType T, int D>
__device__ __forceinline__ void attend_tile(const AParams& p, const LanePos& l, const i32x4* kt,
                                            const uint8_t* vt, int kv0, int wq0,
                                            const i32x4 (&qf)[D / 16], f32x16 (&o_acc)[D / 32],
                                            float& m_run, float& l_run) {
  using IO = AIo<T>;
  constexpr int CH = D / 8, DSTEPS = D / 16, DT = D / 32;
    // S^T for keys 0-31 and 32-63: two independent accumulation chains,
    // issued alternately, with the K fragments read kQkAhead MFMAs ahead
    // of their use (the schedule is pinned below: left to itself the
    // compiler reads each fragment just before its MFMA and waits for it,
    // 4-5 % slower).
    f32x16 s[2];
    {
      i32x4 kf[DSTEPS][2];
#pragma unroll
      for (int d = 0; d < DSTEPS; ++d)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const int row = kb * 32 + l.l32;
          kf[d][kb] = kt[row * CH + ((2 * d + l.hh) ^ kswz<D>(row))];
        }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
#pragma unroll
      for (int d = 0; d < DSTEPS; ++d)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[kb] = IO::mma(kf[d][kb], qf[d], s[kb]);
    }
    // instruction groups, in order: kQkAhead LDS reads, then alternately
    // one MFMA and one read, then the last kQkAhead MFMAs
    __builtin_amdgcn_sched_group_barrier(0x100, kQkAhead, 0);
#pragma unroll
    for (int i = 0; i < 2 * DSTEPS - kQkAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kQkAhead, 0);
    const bool need_mask = (kv0 + kBK > p.S) || (p.causal && kv0 + kBK - 1 > wq0);
    if (need_mask) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kv0 + kb * 32 + 8 * (r >> 2) + 4 * l.hh + (r & 3);
          const bool masked = key >= p.S || (p.causal && key > wq0 + l.l32);
          s[kb][r] = masked ? -INFINITY : s[kb][r];
        }
    }
    uint32_t pk[2][8];
    {
      float mx0 = -INFINITY, mx1 = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        mx0 = fmaxf(mx0, s[0][r]);
        mx1 = fmaxf(mx1, s[1][r]);
      }
      const float mx = half_swap_max(fmaxf(mx0, mx1));
      // (>=: where 8 is lost in the rounding, equal maxima may still differ by
      // half an ulp, which scaled_max looks at. The difference as one fma
      // schedules the whole tile worse, 2 % at D = 64.)
      const bool raise = mx * p.c >= m_run + 8.0f;
      if (__builtin_amdgcn_ballot_w64(raise)) {
        float top = scaled_max<T>(mx, p.c);
        asm("" : "+v"(top));   // a select, not a branch of its own
        const float m_new = raise ? top : m_run;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o_acc[i][r] *= alpha;
      }
      const float m = m_run;
      float ps0 = 0.0f, ps1 = 0.0f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(s[kb][r], p.c, -m));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(s[kb][r + 1], p.c, -m));
          pk[kb][r >> 1] = IO::pack2(p0, p1);
          if (kb == 0) ps0 = IO::sum2(pk[kb][r >> 1], ps0);
          else ps1 = IO::sum2(pk[kb][r >> 1], ps1);
        }
      l_run += ps0 + ps1;
    }
#pragma unroll
    for (int st = 0; st < kBK / 16; ++st) {
      const int kb = st >> 1, half = st & 1;
      const i32x4 pf4 = i32x4{(int)pk[kb][4 * half + 0], (int)pk[kb][4 * half + 1],
                              (int)pk[kb][4 * half + 2], (int)pk[kb][4 * half + 3]};
      const int k1 = 16 * st + l.tr_key, k2 = k1 + 8;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int d = 32 * dt + l.tr_d;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4_t)(vt + k1 * (2 * D) + 16 * ((d >> 3) ^ vswz<D>(k1)) + 2 * (d & 7)));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4_t)(vt + k2 * (2 * D) + 16 * ((d >> 3) ^ vswz<D>(k2)) + 2 * (d & 7)));
        const u32x2 w0 = __builtin_bit_cast(u32x2, v0), w1 = __builtin_bit_cast(u32x2, v1);
        const i32x4 vf = i32x4{(int)w0.x, (int)w0.y, (int)w1.x, (int)w1.y};
        o_acc[dt] = IO::mma(vf, pf4, o_acc[dt]);
      }
    }
}

template <AttnType T, int D>
__global__ __launch_bounds__(64 * kNW, 1) void attn_fwd(AParams p) {
  using IO = AIo<T>;
  constexpr int CH = D / 8;
  constexpr int RPI = 64 / CH;
  constexpr int IPW = kBK / RPI / kNW;
  constexpr int DSTEPS = D / 16;
  constexpr int DT = D / 32;
  static_assert(IPW >= 1, "tile too small for the wave count");
  __shared__ __attribute__((aligned(1024))) i32x4 lds[kNS][2][kBK * CH];
  // Each wave's O tile (32 rows of D values) passes through here on its way
  // out, so that every global store writes whole rows (8 KB per wave at
  // D = 128; 160 KB of LDS in all).
  __shared__ __attribute__((aligned(1024))) i32x4 ost[kNW][32 * CH];

  const uint64_t t_start = cycle_now();
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  ItemMap map;
  map.xcd = blockIdx.x & 7;
  map.wg = blockIdx.x >> 3;
  map.nwg = gridDim.x >> 3;
  map.hx = p.heads / 8 + (map.xcd < (p.heads & 7) ? 1 : 0);

  const uint32_t q_rs = (uint32_t)(2 * p.q_ss), k_rs = (uint32_t)(2 * p.k_ss), v_rs = (uint32_t)(2 * p.v_ss);
  uint32_t kbase[IPW], vbase[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int blk = IPW * wave + i;
    const int row = RPI * blk + lane / CH;
    const int pc = lane % CH;
    kbase[i] = (uint32_t)row * k_rs + (uint32_t)(16 * (pc ^ kswz<D>(row)));
    vbase[i] = (uint32_t)row * v_rs + (uint32_t)(16 * (pc ^ vswz<D>(row)));
  }

  // Per-item state: head pointers, buffer descriptors, tile count.
  struct St {
    int q0, ntiles;
    const uint8_t* qg;
    uint8_t* og;
    i32x4 rk, rv;
  };
  auto setup = [&](int bh, int qt, St& s) {
    const int b = bh / p.H, h = bh % p.H;
    s.q0 = qt * kBQ;
    s.qg = p.q + 2 * (b * p.q_sb + h * p.q_sh);
    const uint8_t* kg = p.k + 2 * (b * p.k_sb + h * p.k_sh);
    const uint8_t* vg = p.v + 2 * (b * p.v_sb + h * p.v_sh);
    s.og = p.o + 2 * (b * p.o_sb + h * p.o_sh);
    s.rk = rsrc_words(kg, (uint32_t)(p.S - 1) * k_rs + 2 * D);
    s.rv = rsrc_words(vg, (uint32_t)(p.S - 1) * v_rs + 2 * D);
    const int kv_end = p.causal ? min(p.S, s.q0 + kBQ) : p.S;
    s.ntiles = (kv_end + kBK - 1) / kBK;
  };
  auto load_q = [&](const St& s, i32x4 (&qf)[DSTEPS]) {
    const int myq = s.q0 + 32 * wave + l32;
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void*)s.qg, (short)0, (int)((uint32_t)(p.S - 1) * q_rs + 2 * D), kRsrcWord3);
#pragma unroll
    for (int t = 0; t < DSTEPS; ++t)
      qf[t] = __builtin_amdgcn_raw_buffer_load_b128(
          rq, (uint32_t)myq * q_rs + (uint32_t)(2 * (16 * t + 8 * hh)), 0, 0);
  };
  // DMA of tile t of item s into LDS stage st (K and V).
  auto dma_tile = [&](const St& s, int t, int st) {
    const int kv0 = t * kBK;
    if (kv0 + kBK <= p.S) {
      const uint32_t ks = (uint32_t)kv0 * k_rs, vs = (uint32_t)kv0 * v_rs;
#pragma unroll
      for (int i = 0; i < IPW; ++i) {
        const int blk = IPW * wave + i;
        dma16_so(s.rk, lds_addr(&lds[st][0][blk * 64]), kbase[i], ks);
        dma16_so(s.rv, lds_addr(&lds[st][1][blk * 64]), vbase[i], vs);
      }
    } else {
#pragma unroll
      for (int i = 0; i < IPW; ++i) {
        const int blk = IPW * wave + i;
        dma16(s.rk, lds_addr(&lds[st][0][blk * 64]), (uint32_t)kv0 * k_rs + kbase[i]);
        dma16(s.rv, lds_addr(&lds[st][1][blk * 64]), (uint32_t)kv0 * v_rs + vbase[i]);
      }
    }
  };

  int round = 0, bh = 0, qt = 0;
  if (!item_at(p, map, round, &bh, &qt)) return;
  St cur;
  setup(bh, qt, cur);
  // DMA pointer: tile pft of item pround (state pf), kNS-1 tiles ahead of
  // the tile being computed, running on into the next items.
  int pround = 0, pft = 0;
  St pf = cur;
  bool pvalid = true;
  auto advance = [&]() {
    if (++pft == pf.ntiles) {
      int b2 = 0, q2 = 0;
      if (item_at(p, map, pround + 1, &b2, &q2)) {
        ++pround;
        setup(b2, q2, pf);
        pft = 0;
      } else {
        pvalid = false;
      }
    }
  };

  i32x4 qf[DSTEPS];
  load_q(cur, qf);
#pragma unroll
  for (int s0 = 0; s0 < kNS - 1; ++s0) {
    if (pvalid) {
      dma_tile(pf, pft, s0);
      advance();
    }
  }
  wait_vmem_all();
  __syncthreads();

  f32x16 o_acc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.0f;
  float m_run = kLowest;
  float l_run = 0.0f;

  const LanePos lp = lane_pos(lane);

  int t = 0;          // tile of the current item
  bool done = false;
  // One 64-key tile of the current item from LDS stage `stage`, while the
  // tile kNS-1 ahead (of this item or the next ones) loads into the stage
  // the previous tile used. After an item's last tile its O is written and
  // the next item's Q fragments are loaded.
  auto tile = [&](auto stage) {
    constexpr int cs = decltype(stage)::value;
    const bool last = (t + 1 == cur.ntiles);
    if (pvalid) {
      dma_tile(pf, pft, (cs + kNS - 1) % kNS);
      advance();
    }
    const int kv0 = t * kBK;
    const int wq0 = cur.q0 + 32 * wave;
    const i32x4* kt = &lds[cs][0][0];
    const uint8_t* vt = (const uint8_t*)&lds[cs][1][0];
    const bool wave_live = !p.causal || kv0 <= wq0 + 31;
    if (wave_live) {
      attend_tile<T, D>(p, lp, kt, vt, kv0, wq0, qf, o_acc, m_run, l_run);
    }
    if (last) {
      // O[q, d] = O^T[d, q] / l for this item; then start the next one.
      const float l_tot = half_swap_sum(l_run);
      const float inv_l = 1.0f / l_tot;   // l = 0 (every score -inf): 0 * inf is NaN
      // A lane holds 4-value pieces of its query's row, 16 of them spread
      // over the row; stored as they are, one instruction writes 8 bytes in
      // each of 32 rows. Instead the wave parks the rounded tile in its LDS
      // region ([row][16-byte chunk], chunk XOR row) and reads it back as
      // whole rows, RPI rows per instruction (+1.5-2.2 %; non-temporal
      // stores measured the same).
      {
        uint8_t* my = (uint8_t*)&ost[wave][0];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int c = (4 * dt + g) ^ (l32 & (CH - 1));
            u32x2 w;
            w.x = IO::pack2(o_acc[dt][4 * g + 0] * inv_l, o_acc[dt][4 * g + 1] * inv_l);
            w.y = IO::pack2(o_acc[dt][4 * g + 2] * inv_l, o_acc[dt][4 * g + 3] * inv_l);
            *(u32x2*)(my + 16 * (l32 * CH + c) + 8 * hh) = w;
          }
        // LDS operations of one wave complete in order; the compiler only
        // must not move the reads above the writes.
        asm volatile("" ::: "memory");
        const int rr = lane / CH, cc = lane % CH;
        // Rows at or past S lie outside the descriptor's range: the buffer
        // store drops them.
        const uint32_t o_rs = (uint32_t)(2 * p.o_ss);
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
            (void*)cur.og, (short)0, (int)((uint32_t)(p.S - 1) * o_rs + 2 * D), kRsrcWord3);
        const uint32_t vo = (uint32_t)(cur.q0 + 32 * wave + rr) * o_rs + 16 * cc;
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i) {
          const int r = RPI * i + rr;
          const i32x4 v = *(const i32x4*)(my + 16 * (r * CH + (cc ^ (r & (CH - 1)))));
          __builtin_amdgcn_raw_buffer_store_b128(v, ro, vo + (uint32_t)(RPI * i) * o_rs, 0, 0);
        }
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.0f;
      m_run = kLowest;
      l_run = 0.0f;
      int nbh = 0, nqt = 0;
      if (item_at(p, map, round + 1, &nbh, &nqt)) {
        setup(nbh, nqt, cur);
        load_q(cur, qf);   // waited for below, with the DMA
        ++round;
        t = 0;
      } else {
        done = true;
      }
    } else {
      ++t;
    }
    wait_vmem_all();
    __syncthreads();
  };
  while (true) {
    tile(Stage<0>{});
    if (done) break;
    tile(Stage<1>{});
    if (done) break;
    tile(Stage<2>{});
    if (done) break;
  }
  cycle_record(p.probe, t_start, blockIdx.x * kNW + wave, wave);
}

// Problems of few query tiles: one workgroup per item of 32*QW queries of one
// head, whose 8 waves are QW query blocks of 32 times KS = 8/QW key groups.
// Group g takes the 64-key tiles g, g + KS, ..., with the running maximum, sum
// and O of its own, and the groups' results meet in LDS at the end (O scaled
// by exp2(m_g - max m), fp32). So a head of S keys takes S/(64*KS) steps on
// ceil(S/(32*QW)) CUs instead of S/64 on ceil(S/256). NS LDS stages of KS
// tiles: with two, a step's loads are issued one step ahead; with one (the
// tiles of a step fill LDS) the next step's loads wait for this one's reads.
template <AttnType T, int D, int QW, int NS>
__global__ __launch_bounds__(64 * kNW, 1) void attn_split(AParams p) {
  using IO = AIo<T>;
  constexpr int KS = kNW / QW;
  constexpr int CH = D / 8, RPI = 64 / CH, DSTEPS = D / 16, DT = D / 32;
  constexpr int IPW = CH / QW;                     // 1 KB loads per wave, operand and tile
  constexpr int kTile = kBK * CH;                  // 16-byte chunks of one operand's tile
  constexpr int kPitch = D + 4;                    // floats per row of a wave's O in LDS
  constexpr int kStageBytes = NS * KS * 2 * kTile * 16;
  constexpr int kMergeBytes = kNW * 32 * kPitch * 4;
  static_assert((QW == 2 || QW == 4) && (NS == 1 || NS == 2), "query blocks, stages");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kStageBytes > kMergeBytes ? kStageBytes : kMergeBytes];
  __shared__ float ml[kNW][2][32];                 // running maximum and sum per query

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave / QW, qw = wave % QW;
  const LanePos lp = lane_pos(lane);

  // Items by weight (causal: the last query tiles first), heads inside: with
  // heads a multiple of 8 every item of a head runs on one XCD (workgroups are
  // dealt round-robin over the eight) and its K and V stay in that L2.
  const int r0 = blockIdx.x / p.heads, bh = blockIdx.x - r0 * p.heads;
  const int q0 = (p.causal ? p.qtiles - 1 - r0 : r0) * 32 * QW;
  const int b = bh / p.H, h = bh - b * p.H;
  const uint32_t q_rs = (uint32_t)(2 * p.q_ss), k_rs = (uint32_t)(2 * p.k_ss), v_rs = (uint32_t)(2 * p.v_ss);
  const uint32_t o_rs = (uint32_t)(2 * p.o_ss);
  const i32x4 rk = rsrc_words(p.k + 2 * (b * p.k_sb + h * p.k_sh), (uint32_t)(p.S - 1) * k_rs + 2 * D);
  const i32x4 rv = rsrc_words(p.v + 2 * (b * p.v_sb + h * p.v_sh), (uint32_t)(p.S - 1) * v_rs + 2 * D);
  const int kv_end = p.causal ? min(p.S, q0 + 32 * QW) : p.S;
  const int ntiles = (kv_end + kBK - 1) / kBK;
  const int steps = (ntiles + KS - 1) / KS;

  uint32_t kbase[IPW], vbase[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int row = RPI * (QW * i + qw) + lane / CH;
    const int pc = lane % CH;
    kbase[i] = (uint32_t)row * k_rs + (uint32_t)(16 * (pc ^ kswz<D>(row)));
    vbase[i] = (uint32_t)row * v_rs + (uint32_t)(16 * (pc ^ vswz<D>(row)));
  }
  auto tile_at = [&](int st, int operand) { return smem + (((st * KS + g) * 2 + operand) * kTile) * 16; };
  // The group's tile of step s into stage st.
  auto load = [&](int s, int st) __attribute__((always_inline)) {
    const int kv0 = (s * KS + g) * kBK;
    if (kv0 >= kv_end) return;
    const bool inside = kv0 + kBK <= p.S;          // rows past S read as zero
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const uint32_t lk = lds_addr(tile_at(st, 0) + 1024 * (QW * i + qw));
      const uint32_t lv = lds_addr(tile_at(st, 1) + 1024 * (QW * i + qw));
      if (inside) {
        dma16_so(rk, lk, kbase[i], (uint32_t)kv0 * k_rs);
        dma16_so(rv, lv, vbase[i], (uint32_t)kv0 * v_rs);
      } else {
        dma16(rk, lk, (uint32_t)kv0 * k_rs + kbase[i]);
        dma16(rv, lv, (uint32_t)kv0 * v_rs + vbase[i]);
      }
    }
  };
  auto landed = [&]() __attribute__((always_inline)) {
    wait_vmem_all();
    __syncthreads();
  };

  load(0, 0);
  const int wq0 = q0 + 32 * qw;
  i32x4 qf[DSTEPS];
  {
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.q + 2 * (b * p.q_sb + h * p.q_sh)), (short)0, (int)((uint32_t)(p.S - 1) * q_rs + 2 * D),
        kRsrcWord3);
#pragma unroll
    for (int t = 0; t < DSTEPS; ++t)
      qf[t] = __builtin_amdgcn_raw_buffer_load_b128(
          rq, (uint32_t)(wq0 + lp.l32) * q_rs + (uint32_t)(2 * (16 * t + 8 * lp.hh)), 0, 0);
  }
  f32x16 o_acc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.0f;
  float m_run = kLowest, l_run = 0.0f;
  landed();
  for (int s = 0; s < steps; ++s) {
    const int st = NS == 2 ? s & 1 : 0;
    if (NS == 2 && s + 1 < steps) load(s + 1, st ^ 1);
    const int kv0 = (s * KS + g) * kBK;
    if (kv0 < kv_end && (!p.causal || kv0 <= wq0 + 31))
      attend_tile<T, D>(p, lp, (const i32x4*)tile_at(st, 0), tile_at(st, 1), kv0, wq0, qf, o_acc, m_run, l_run);
    if (NS == 1 && s + 1 < steps) {
      // every read of this step's tiles is done before the next one's land
      __syncthreads();
      load(s + 1, 0);
    }
    if (s + 1 < steps) landed();
  }

  // The groups' O, maximum and sum to LDS, over the tiles.
  const float l_tot = half_swap_sum(l_run);
  wait_vmem_all();   // nothing is in flight here: stated for the check of the generated code
  __syncthreads();
  float* mo = (float*)smem;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4 v = {o_acc[dt][4 * r], o_acc[dt][4 * r + 1], o_acc[dt][4 * r + 2], o_acc[dt][4 * r + 3]};
      *(f32x4*)&mo[(wave * 32 + lp.l32) * kPitch + 32 * dt + 8 * r + 4 * lp.hh] = v;
    }
  if (lp.hh == 0) {
    ml[wave][0][lp.l32] = m_run;
    ml[wave][1][lp.l32] = l_tot;
  }
  __syncthreads();
  // Wave (g, qw) combines rows g*32/KS .. of query block qw, 8 values per lane.
  constexpr int ROWS = 32 / KS;
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.o + 2 * (b * p.o_sb + h * p.o_sh)), (short)0, (int)((uint32_t)(p.S - 1) * o_rs + 2 * D), kRsrcWord3);
  const int cc = lane % CH;
  for (int rr = lane / CH; rr < ROWS; rr += RPI) {
    const int row = g * ROWS + rr;
    float mx = ml[qw][0][row];
#pragma unroll
    for (int j = 1; j < KS; ++j) mx = fmaxf(mx, ml[j * QW + qw][0][row]);
    float l = 0.0f, o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      const int w = j * QW + qw;
      const float scale = __builtin_amdgcn_exp2f(ml[w][0][row] - mx);
      l = fmaf(scale, ml[w][1][row], l);
      const f32x4* src = (const f32x4*)&mo[(w * 32 + row) * kPitch + 8 * cc];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f32x4 v = src[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[4 * q + e] = fmaf(scale, v[e], o[4 * q + e]);
      }
    }
    const float inv_l = 1.0f / l;   // as in attn_fwd
    i32x4 out;
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] = (int)IO::pack2(o[2 * q] * inv_l, o[2 * q + 1] * inv_l);
    // rows at or past S lie outside the descriptor's range: dropped
    __builtin_amdgcn_raw_buffer_store_b128(out, ro, (uint32_t)(q0 + 32 * qw + row) * o_rs + 16 * cc, 0, 0);
  }
}

// CUs of the current device, a multiple of 8 (one share per XCD).
int compute_units() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return std::max(8, cus / 8 * 8);
}

// One workgroup per CU, no more than the items need.
int64_t workgroups(int cus, int B, int H, int S) {
  const int64_t qtiles = (S + kBQ - 1) / kBQ;
  int64_t wgs = cus;
  const int64_t per_xcd_items = ((int64_t)B * H + 7) / 8 * qtiles;
  if (wgs / 8 > per_xcd_items) wgs = 8 * per_xcd_items;
  if (wgs < 8) wgs = 8;
  return wgs;
}

// Heads per block of attn_fwd's item order: as many as one round of an XCD's
// workgroups has room for. Causal launches of at most 8 rounds whose rounds do
// not come out even (a block that is no whole share of a round, a last round
// that is odd or part empty) would leave a workgroup with two of the heaviest
// items: their heads are one block, whose snake pairs heavy with light (B2 H20
// S2500 D64 91 us in blocks of 3 heads).
int heads_per_block(int64_t hx, int qtiles, int nwg, bool causal) {
  const int hb = (int)std::max<int64_t>(1, std::min<int64_t>(nwg / qtiles, hx));
  const int64_t items = hx * qtiles;
  const bool even = nwg % (hb * qtiles) == 0 && items % (2 * nwg) == 0;
  return causal && !even && items > nwg && items <= 8 * nwg ? (int)hx : hb;
}

// Query blocks per workgroup of attn_split (4 or 2), or 0 for the persistent
// attn_fwd, whichever is modelled fastest (us; the constants fit bf16 times of
// 64 to 4000 keys on 4 to 256 heads). A CU runs one tile (or step of KS tiles)
// at a time, so a launch takes the steps of its busiest CU: the heaviest item
// while there is at most one per CU, the average CU's share beyond, plus a start
// and an end per item, which the persistent kernel hides. us, attn_fwd / QW 4 /
// QW 2: B2 H16 S1000 D64 24.0 / 16.9 / 21.9; B1 H8 S2048 D64 38.6 / 24.0 / 16.5
// and D128 49.9 / 33.6 / 27.0; B1 H24 S218 D128 12.3 / 9.8 / 8.5; B4 H16
// S1024 D64 23.5 / 24.1 / 36.2 and D128 36.5 / 43.1 / 63.6.
int split_blocks(int cus, int64_t heads, int S, int D, bool causal) {
  const double start = D == 64 ? 3.5 : 4.0;
  // Mean tiles of an item of `queries` over the heaviest item's.
  auto share = [&](int queries) {
    const int n = (S + queries - 1) / queries;
    return causal ? (n + 1.0) / (2.0 * n) : 1.0;
  };
  const double tiles = (S + kBK - 1) / kBK;
  // attn_fwd: the items of one XCD's heads over its workgroups
  const double items8 = (double)((heads + 7) / 8) * ((S + kBQ - 1) / kBQ) / (cus / 8);
  const double rounds = causal ? std::max(1.0, 1.1 * items8 * share(kBQ)) : std::ceil(items8);
  double best = 0.95 * (start + (D == 64 ? 1.25 : 1.8) * tiles * rounds);
  int qw = 0;
  for (int w = 4; w >= 2; w /= 2) {
    const double items = (double)heads * ((S + 32 * w - 1) / (32 * w)) / cus;   // per CU
    const double steps = std::ceil(tiles * w / kNW) * (items > 1.0 ? share(32 * w) : 1.0);
    const double step = D == 64 ? (w == 4 ? 1.55 : 1.65) : (w == 4 ? 2.2 : 3.0);
    double t;
    if (D == 64 && w == 4) {
      // Two workgroups share a CU. Items of one size leave some CUs a whole one
      // more than others, of which sharing hides a fifth (90 heads of 317 keys
      // 12.2 us, attn_fwd 10.5).
      const double busiest = causal || items <= 1.0 ? items : std::max(items, 0.82 * std::ceil(items));
      t = start + std::max(1.0, busiest) * (steps * step + 0.6);
      // Beside one round of attn_fwd the heaviest item counts: it shares its CU
      // with a light one, and a head's items lie on several XCDs where heads are
      // no multiple of 8 (causal, 110 heads of 307 keys 10.8 us, attn_fwd 10.3).
      if (causal && items > 1.0 && items8 <= 1.0 && heads % 8)
        t = std::max(t, start + std::ceil(tiles * w / kNW) * step + 1.4);
    } else {
      t = std::ceil(items) * (start + (D == 128 && w == 2 ? 0.8 : 0.2) + steps * step);
    }
    if (t < best) {
      best = t;
      qw = w;
    }
  }
  return qw;
}

// GRXDNN_LOG set (and not "0"): one line on stderr per attention call.
bool log_launches() {
  const char* v = std::getenv("GRXDNN_LOG");
  return v && *v && !(v[0] == '0' && v[1] == 0);
}

template <AttnType T, int D>
hipError_t run(const AttnDesc& d, hipStream_t s) {
  AParams p{};
  p.q = (const uint8_t*)d.q; p.k = (const uint8_t*)d.k; p.v = (const uint8_t*)d.v;
  p.o = (uint8_t*)d.o;
  p.q_sb = d.q_sb; p.q_sh = d.q_sh; p.q_ss = d.q_ss;
  p.k_sb = d.k_sb; p.k_sh = d.k_sh; p.k_ss = d.k_ss;
  p.v_sb = d.v_sb; p.v_sh = d.v_sh; p.v_ss = d.v_ss;
  p.o_sb = d.o_sb; p.o_sh = d.o_sh; p.o_ss = d.o_ss;
  p.B = d.B; p.H = d.H; p.S = d.S;
  p.qtiles = (d.S + kBQ - 1) / kBQ;
  p.heads = d.B * d.H;
  p.causal = d.causal ? 1 : 0;
  p.c = d.scale * 1.4426950408889634f;
  p.probe = d.probe;
  // Every buffer offset (Q, K and V loads, O stores) is 32-bit.
  int64_t pitch = d.q_ss > d.k_ss ? d.q_ss : d.k_ss;
  pitch = pitch > d.v_ss ? pitch : d.v_ss;
  pitch = pitch > d.o_ss ? pitch : d.o_ss;
  const int64_t span = ((int64_t)d.S + kBQ) * 2 * pitch + 2 * d.D;
  if (span >= (1ll << 31)) return hipErrorNotSupported;
  // item indices are 32-bit in the kernel
  if ((int64_t)d.B * d.H * p.qtiles > 0x7fffffff) return hipErrorInvalidValue;
  const int cus = compute_units();
  // (a cycle probe's slots are counted for attn_fwd)
  int qw = d.probe ? 0 : split_blocks(cus, (int64_t)d.B * d.H, d.S, D, p.causal);
  const int64_t items = qw ? (int64_t)p.heads * ((d.S + 32 * qw - 1) / (32 * qw)) : 0;
  if (items > max_workgroups(64 * kNW)) qw = 0;
  if (log_launches())
    std::fprintf(stderr, "grxdnn: attention %s b=%d h=%d s=%d d=%d causal=%d kernel=%s\n",
                 T == AttnType::BF16 ? "bf16" : "f16", d.B, d.H, d.S, D, (int)p.causal,
                 qw == 4 ? "split4" : qw == 2 ? "split2" : "fwd");
  if (qw) {
    p.qtiles = (d.S + 32 * qw - 1) / (32 * qw);
    const dim3 grid((unsigned)items);
    if (qw == 4) hipLaunchKernelGGL((attn_split<T, D, 4, 2>), grid, dim3(64 * kNW), 0, s, p);
    else hipLaunchKernelGGL((attn_split<T, D, 2, D == 64 ? 2 : 1>), grid, dim3(64 * kNW), 0, s, p);
    return hipGetLastError();
  }
  const int64_t wgs = workgroups(cus, d.B, d.H, d.S);
  p.hb = heads_per_block((p.heads + 7) / 8, p.qtiles, (int)(wgs / 8), p.causal);
  hipLaunchKernelGGL((attn_fwd<T, D>), dim3((unsigned)wgs), dim3(64 * kNW), 0, s, p);
  return hipGetLastError();
}

}  // namespace

int64_t attention_probe_slots(int B, int H, int S) { return workgroups(compute_units(), B, H, S) * kNW; }

hipError_t launch_attention(AttnType t, const AttnDesc& d, hipStream_t s) {
  if (t == AttnType::BF16) {
    if (d.D == 128) return run<AttnType::BF16, 128>(d, s);
    if (d.D == 64) return run<AttnType::BF16, 64>(d, s);
  } else {
    if (d.D == 128) return run<AttnType::F16, 128>(d, s);
    if (d.D == 64) return run<AttnType::F16, 64>(d, s);
  }
  return hipErrorNotSupported;
}

}  // namespace grxk
