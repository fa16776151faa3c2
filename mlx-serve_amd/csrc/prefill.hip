// Prefill (large-M) 4-bit affine quantized GEMM for gfx950:
//   y[M,N] (bf16) = x[M,K] (bf16) @ dequant(w)[N,K]^T, fp32 accumulation.
// Replaces the reference's prefill route of qmatmulBits / prefillDqGemm
// (src/transformer.zig:20894-20983, :20987-21011), which expands the whole weight to a bf16
// copy in memory before a dense GEMM; here each weight tile is dequantized in registers on
// its way into the matrix cores and never exists in bf16 outside them.
//
// Block: 256 (M) x 256 (N) outputs, 8 waves (two per SIMD), v_mfma_f32_16x16x32_bf16 with
// D[n][m] = W[n][k] x[m][k]. In a 64-wide step a lane (row lane % 16, quarter q = lane / 16)
// holds the 16 values k = 16q .. 16q+15 of its weight rows, dequantized as bf16(s*q + b): q
// from a scaled fp8 conversion, fma(s, q, b), one rounding to bf16 by v_cvt_pk_bf16_f32, as
// MLX's GPU qmm rounds the weights it stages; k-step e takes values 8e..8e+7 of each quarter,
// and the x fragment the 16-byte slot 2q+e of the row. All staging is buffer_load ... lds DMA
// (no VGPR round trip); the schedule is described at prefill_pp_kernel.
//
// What bounds it: the matrix cores at a power-limited clock. On random bf16 operands
// 16x16x32 sustains 1.96 PF and 32x32x16 1.70 PF (registers only, all CUs; 2.4 and 2.3 PF on
// zeros), so the smaller shape is taken; with the accumulators in plain VGPRs, since in AGPRs
// the compiler copied them around these MFMAs (4 moves each). 8192 rows 4-bit, 32x32x16 ->
// 16x16x32: [14336,4096] 889 -> 805 us, [4096,14336] 822 -> 759 (matrix cores busy 59% / 62% of the
// cycles, before 59% / 64% at a lower clock).
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "mi_common.h"
#include "mi_internal.h"
#include "qmv_common.h"
#include "dequant_bf16.h"
#include "prefill_tiles.h"

namespace mi {
namespace {

using qmv_detail::vmcnt_imm;
using dq::dequant8;
using dq::pack_bf16x2;

constexpr int kBM = 256, kBN = 256, kBK = 64, kRing = 3;
constexpr int kXBytes = kBM * kBK * 2;  // x tile: 256 rows x 128 B
constexpr int kBufFlags = 0x00020000;   // raw dword access

#define MI_DMA_LDS(SIZE, rsrc, lds, voff, soff)                                            \
  __builtin_amdgcn_raw_ptr_buffer_load_lds((rsrc), (__attribute__((address_space(3))) void*)(lds), \
                                           SIZE, (voff), (soff), 0, 0)

// Ping-pong variant: 8 waves, two per SIMD. Wave w owns weight rows [32w, 32w + 32) (two
// 16-row tiles) against all 256 x rows (sixteen tiles): 32 accumulators (128
// registers), so two waves fit a SIMD, and every weight of the block is dequantized by
// exactly one wave. (VALU work issued beside another wave's MFMAs delays them, so the
// dequantize count per MFMA is what this layout minimizes; the price is one 1 KB x
// fragment read per two MFMAs, half the LDS read bandwidth of a CU.) Each wave's work on a
// 64-wide step is two units: "mem" (its packed weights, scales and biases from LDS,
// dequantized to the 16 bf16 operand registers of the whole step, and the first x
// fragments) and "mfma" (the step's 64 MFMAs, the remaining x fragments read as they go).
// The two groups run the same units half a step apart on staggered barriers: while group
// 0 issues the matrix ops of step t, group 1 dequantizes step t, then the roles swap, so
// each SIMD always has one wave feeding the matrix core and one doing the VALU/LDS work.
// Timeline of half-steps h (a block barrier after each):
//   h = 2t:    group 0 mem(t),     group 1 mfma(t-1)
//   h = 2t+1:  group 0 mfma(t),    group 1 mem(t);  every wave issues the DMA of step t+2
//
// Staging is shaped by the number of memory requests, not bytes: the DMA path serves a
// bounded number of requests per CU per cycle, and a request per 4-byte scale was the
// largest cost. So LDS holds
//   - x: a 3-stage ring of 256 x 64 tiles (32 KB each; 128-byte rows, one request each),
//   - packed weights: 2 buffers of 2-step chunks (256 rows x 64 B: one request per row
//     per two steps, against one per step for 32-byte rows),
//   - scales and biases: 2 buffers of 8-group chunks (256 rows x 16 B each, moved as
//     4 dwords per row: one request per row per 8 groups).
// A chunk goes out with the x tile of its first step and lands one step ahead of use.
// Step t's x stage is last read in half 2t+2; the DMA that reuses it (step t+3) goes out
// in half 2t+3. Each wave waits (exact vmcnt) at the end of half 2t+1 for everything
// issued before the DMA of step t+2, so the barrier publishes step t+1 before group 0
// reads it in half 2t+2. The weight and scale buffers are reused two chunks later, after
// the last read of the chunk they held.
// 8-bit weights (BITS = 8) take the same path with one step per weight chunk (64 B of a row
// is one step's 64 codes), in 3 buffers: a 1-step chunk is last read in the half after its
// successor's DMA would go out, so two buffers would not do.
constexpr int kPPThreads = 512;
constexpr int kPPXStage = kXBytes;                   // 32 KB
constexpr int kPPWChunk = kBN * 64;                  // 256 rows x 64 B
constexpr int kPPSChunk = kBN * 16;                  // 256 rows x 16 B (scales or biases)
constexpr int kPPWOff = kRing * kPPXStage;           // 96 KB
// BITS = 16: weights already dequantized to bf16 (the other formats' large-M route). A
// lane's 64 bytes of its row per step are read straight into registers (a 3-step ring), so
// LDS holds only the x ring and the mem unit does no dequantize work.
template <int BITS>
constexpr int pp_wbufs() { return BITS == 4 ? 2 : BITS == 8 ? 3 : 0; }
template <int BITS>
constexpr int pp_soff() { return kPPWOff + pp_wbufs<BITS>() * kPPWChunk; }  // 128 / 144 KB
template <int BITS>
constexpr int pp_lds() { return BITS == 16 ? kPPWOff : pp_soff<BITS>() + 4 * kPPSChunk; }

// 8 bytes (codes q0..q7, k order) -> four bf16 pairs of s*q + b: each byte converts exactly
// (v_cvt_f32_ubyte), fma(s, q, b), one rounding to bf16.
MI_DEV u32x4_t dequant8_b8(uint32_t w0, uint32_t w1, float s, float b) {
  u32x4_t o;
  o.x = pack_bf16x2(fmaf(s, (float)(w0 & 0xFFu), b), fmaf(s, (float)((w0 >> 8) & 0xFFu), b));
  o.y = pack_bf16x2(fmaf(s, (float)((w0 >> 16) & 0xFFu), b), fmaf(s, (float)(w0 >> 24), b));
  o.z = pack_bf16x2(fmaf(s, (float)(w1 & 0xFFu), b), fmaf(s, (float)((w1 >> 8) & 0xFFu), b));
  o.w = pack_bf16x2(fmaf(s, (float)((w1 >> 16) & 0xFFu), b), fmaf(s, (float)(w1 >> 24), b));
  return o;
}

// XOR swizzles of the 16-byte LDS slots by row. A ds_read_b128 pass serves lanes 0-3, 12-15,
// 20-23 and 24-27 of a half together, so with the MFMA's lane layout (16 rows, quarter
// q = lane / 16) rows 0-3 and 12-15 of quarter q meet rows 4-11 of quarter q + 1: these keep
// their slots distinct (x: 8 slots of a 128-byte row, lane slot 2q + e; w: 4 of 64 bytes).
MI_DEV int xswz(int r) { return (r & 2) | ((r >> 2) & 1) | ((r >> 1) & 4); }
template <int BITS>
MI_DEV int wswz(int r) { return BITS == 8 ? 3 * ((r >> 2) & 1) : (r >> 2) & 3; }

MI_DEV f32x4_t mfma16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return mfma16x16x32(as_bf16x8(a), as_bf16x8(b), c);
}

MI_DEV void wait_vm(int n) {  // s_waitcnt vmcnt(n) for the counts one step can issue
  switch (n) {
    case 0: __builtin_amdgcn_s_waitcnt(vmcnt_imm(0)); break;
    case 4: __builtin_amdgcn_s_waitcnt(vmcnt_imm(4)); break;
    case 6: __builtin_amdgcn_s_waitcnt(vmcnt_imm(6)); break;
    case 8: __builtin_amdgcn_s_waitcnt(vmcnt_imm(8)); break;
    default: __builtin_amdgcn_s_waitcnt(vmcnt_imm(10)); break;
  }
}

template <int BITS, int GS, bool SPLIT>
__global__ void __launch_bounds__(kPPThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
prefill_pp_kernel(PrefillParams P) {
  constexpr int RB = BITS * kBK / 8;  // bytes of a weight row per step: 32, 64 or 128
  constexpr bool W16 = BITS == 16;
  constexpr int kSOff = pp_soff<BITS>();
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // steps per scale chunk (8 groups): 4, 8 or 16
  constexpr int kSP = GS / 8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, nq = wave & 3;
  const int fr = lane & 15, q = lane >> 4;
  const int M = P.M, N = P.N, K = P.K, G = K / GS;
  const TileOf at = tile_of_block((M + kBM - 1) / kBM, (N + kBN - 1) / kBN);
  const int m0 = at.mt * kBM, n0 = at.nt * kBN, split = at.split;
  const int s0 = split * P.sps;
  const int nsteps = min(P.sps, K / kBK - s0);
  const int mrows = min(kBM, M - m0), nrows = min(kBN, N - n0);

  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(P.x + (size_t)m0 * K), 0, mrows * K * 2, kBufFlags);
  const int rowb = K * BITS / 8;  // bytes of a weight row
  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const unsigned char*)P.w + (size_t)n0 * rowb), 0, nrows * rowb, kBufFlags);
  // group 0 moves the scales, group 1 the biases
  const __amdgpu_buffer_rsrc_t sbres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((grp ? P.biases : P.scales) + (size_t)n0 * G), 0, nrows * G * 2, kBufFlags);
  // x: wave w moves tile rows 32w..32w+31 as 4 instructions of 8 rows x 128 B; LDS slot p
  // of row r holds k-slot p ^ xswz(r).
  uint32_t xo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 32 * wave + 8 * i + (lane >> 3);
    const int c = (lane & 7) ^ xswz(r);
    xo[i] = (uint32_t)(min(r, mrows - 1) * K + 8 * c) * 2;
  }
  // packed-weight chunk (2 steps at 4 bits, 1 at 8): wave w moves rows 32w..32w+31 as 2
  // instructions of 16 rows x 64 B; LDS part p (16 B) of row r holds part p ^ wswz(r)
  // of the row's 64 bytes.
  uint32_t wo[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 32 * wave + 16 * i + (lane >> 2);
    const int c = (lane & 3) ^ wswz<BITS>(r);
    wo[i] = (uint32_t)(min(r, nrows - 1) * rowb + 16 * c);
  }
  // scale (group 0) or bias (group 1) chunk: wave moves rows 64nq..64nq+63 as 4
  // instructions of 16 rows x 4 dwords; row-major 16 B per row in LDS.
  uint32_t so[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 64 * nq + 16 * i + (lane >> 2);
    so[i] = (uint32_t)(min(r, nrows - 1) * G * 2 + 4 * (lane & 3));
  }
  // bf16 weights: lane (fr, q) reads bytes 32q .. 32q+31 of its two rows' 128 per step
  u32x4_t wreg[W16 ? 3 : 1][4];
  uint32_t w16o[2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
    w16o[a] = (uint32_t)min(32 * wave + 16 * a + fr, nrows - 1) * (uint32_t)rowb + 32 * q;
  // DMA of local step st (x; the weight chunk when st is even; the scale chunk when st
  // starts one; bf16 weights into register slot `slot`). Returns the instructions issued
  // (0 past the last step).
  auto issue = [&](int st, auto slot_c) -> int {
    constexpr int slot = decltype(slot_c)::value;
    if (st >= nsteps) return 0;
    const int k = s0 + st;
    unsigned char* xb = smem + (st % kRing) * kPPXStage;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      MI_DMA_LDS(16, xres, xb + wave * 4096 + i * 1024, xo[i], k * kBK * 2);
    int n = 4;
    if constexpr (W16) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        wreg[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(wres, w16o[i / 2] + 16 * (i % 2), k * RB, 0);
      return n + 4;
    }
    if (BITS == 8 || (st & 1) == 0) {
      unsigned char* wb = smem + kPPWOff + (BITS == 4 ? (st >> 1) & 1 : st % 3) * kPPWChunk;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        MI_DMA_LDS(16, wres, wb + wave * 2048 + i * 1024, wo[i], k * RB);
      n += 2;
    }
    if (st == 0 || k % kSP == 0) {
      const int c = k / kSP;
      unsigned char* sb = smem + kSOff + (c & 1) * 2 * kPPSChunk + grp * kPPSChunk;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        MI_DMA_LDS(4, sbres, sb + nq * 1024 + i * 256, so[i], c * 16);
      n += 4;
    }
    return n;
  };

  f32x4_t acc[2][16];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[a][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // x fragment of tile i, k-step e: row 16 i + fr, k-slot 2q + e.
  auto xfrag = [&](int stg, int i, int e) -> u32x4_t {
    const int r = 16 * i + fr, c = 2 * q + e;
    return *reinterpret_cast<const u32x4_t*>(smem + stg * kPPXStage + r * 128 +
                                             ((c ^ xswz(r)) << 4));
  };
  u32x4_t A[2][2], X[2][8];  // weight operands [row tile][k-step]; x tiles 8 at a time
  auto mem = [&](int st, auto slot_c) {
    constexpr int slot = decltype(slot_c)::value;
#pragma unroll
    for (int i = 0; i < 8; ++i) X[0][i] = xfrag(st % kRing, i, 0);
    if constexpr (W16) return;  // the MFMAs read the weight registers in place
    const int k = s0 + st;
    const unsigned char* wb =
        smem + kPPWOff + (BITS == 4 ? (st >> 1) & 1 : st % 3) * kPPWChunk;
    const unsigned char* sb = smem + kSOff + ((k / kSP) & 1) * 2 * kPPSChunk;
    // group of this lane's 16 k within the chunk's 8
    const int gi = GS == 32 ? 2 * (k % 4) + (q >> 1) : GS == 64 ? k % 8 : (k >> 1) % 8;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int r = 32 * wave + 16 * a + fr;
      const uint16_t sv = *reinterpret_cast<const uint16_t*>(sb + r * 16 + 2 * gi);
      const uint16_t bv = *reinterpret_cast<const uint16_t*>(sb + kPPSChunk + r * 16 + 2 * gi);
      const float sc = __uint_as_float((uint32_t)sv << 16);
      const float bp = __uint_as_float((uint32_t)bv << 16);
      if constexpr (BITS == 4) {
        // the lane's 16 codes: 8 B, half q % 2 of part 2(st%2) + q/2 of the row's 64 bytes
        const int part = 2 * (st & 1) + (q >> 1);
        const u32x2_t v = *reinterpret_cast<const u32x2_t*>(
            wb + r * 64 + ((part ^ wswz<BITS>(r)) << 4) + 8 * (q & 1));
        A[a][0] = dequant8(v.x, sc, bp);
        A[a][1] = dequant8(v.y, sc, bp);
      } else {
        const u32x4_t v =
            *reinterpret_cast<const u32x4_t*>(wb + r * 64 + ((q ^ wswz<BITS>(r)) << 4));
        A[a][0] = dequant8_b8(v.x, v.y, sc, bp);
        A[a][1] = dequant8_b8(v.z, v.w, sc, bp);
      }
    }
  };
  auto mfma = [&](int st, auto slot_c) {
    constexpr int slot = decltype(slot_c)::value;
    const int stg = st % kRing;
    // four parts: k-step u / 2 against x tiles 8(u%2) .. +7
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (u < 3) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          X[(u + 1) & 1][i] = xfrag(stg, 8 * ((u + 1) & 1) + i, (u + 1) / 2);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          f32x4_t& c = acc[a][8 * (u & 1) + i];
          c = mfma16(W16 ? wreg[slot][2 * a + u / 2] : A[a][u / 2], X[u & 1][i], c);
        }
      // the next part's fragment reads go out ahead of this part's MFMAs, one read per two
      // MFMAs, so their latency hides under the matrix work
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        if (u < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Both groups run the same unit sequence mem(t), mfma(t) with a barrier after each unit;
  // group 1 starts one half later (an extra barrier first), group 0 ends with an extra
  // barrier, so the barrier counts match. The DMA of step t+2 goes out in half 2t+1 for
  // both groups: after group 0's mfma(t) unit and after group 1's mem(t) unit.
  using c0 = std::integral_constant<int, 0>;
  using c1 = std::integral_constant<int, 1>;
  using c2 = std::integral_constant<int, 2>;
  issue(0, c0{});
  wait_vm(issue(1, c1{}));
  __builtin_amdgcn_s_barrier();
  if (grp) __builtin_amdgcn_s_barrier();
  // (ws: the register slot of step t's bf16 weights, wn: that of step t + 2)
  auto step = [&](int t, auto ws, auto wn) {
    mem(t, ws);
    __builtin_amdgcn_sched_barrier(0);
    if (grp) wait_vm(issue(t + 2, wn));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    mfma(t, ws);
    __builtin_amdgcn_sched_barrier(0);
    if (!grp) wait_vm(issue(t + 2, wn));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (W16) {
    // unrolled by 3 so the weight registers of steps t, t+1, t+2 sit in static slots
    for (int t0 = 0; t0 < nsteps; t0 += 3) {
      step(t0, c0{}, c2{});
      if (t0 + 1 < nsteps) step(t0 + 1, c1{}, c0{});
      if (t0 + 2 < nsteps) step(t0 + 2, c2{}, c1{});
    }
  } else {
    for (int t = 0; t < nsteps; ++t) step(t, c0{}, c0{});
  }
  if (!grp) __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // no DMA may outlive the block

  // epilogue: acc[a][i] register r is D[n = 32 wave + 16a + 4q + r][m = 16 i + fr]
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int m = m0 + 16 * i + fr;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int n = n0 + 32 * wave + 16 * a + 4 * q;
      if (n >= N) continue;
      const f32x4_t v = acc[a][i];
      if constexpr (SPLIT)
        *reinterpret_cast<f32x4_t*>(P.part + ((size_t)split * M + m) * N + n) = v;
      else
        *reinterpret_cast<u32x2_t*>(P.y + (size_t)m * N + n) =
            u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
}

// y = bf16(sum over splits in split order of part[split]); 4 outputs per thread.
__global__ void prefill_reduce_kernel(const float* __restrict__ part, uint16_t* __restrict__ y,
                                      int64_t mn4, int ks) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < mn4;
       i += (int64_t)gridDim.x * blockDim.x) {
    const f32x4_t* p4 = reinterpret_cast<const f32x4_t*>(part) + i;
    const f32x4_t acc = add_splits<8>(p4[0], p4, mn4, 1, ks);
    u32x2_t o;
    o.x = pack_bf16x2(acc[0], acc[1]);
    o.y = pack_bf16x2(acc[2], acc[3]);
    reinterpret_cast<u32x2_t*>(y)[i] = o;
  }
}

template <typename Kern>
hipError_t set_lds(Kern k, size_t lds) {
  return hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

template <int BITS, int GS>
hipError_t launch_gs(const PrefillParams& P, hipStream_t s) {
  const int mtiles = (P.M + kBM - 1) / kBM, ntiles = (P.N + kBN - 1) / kBN;
  constexpr int lds = pp_lds<BITS>();
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipSuccess;
    for (auto k : {prefill_pp_kernel<BITS, GS, true>, prefill_pp_kernel<BITS, GS, false>})
      if (e == hipSuccess) e = set_lds(k, lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  const dim3 grid((unsigned)(mtiles * ntiles), (unsigned)P.ks);
  if (P.ks > 1)
    hipLaunchKernelGGL((prefill_pp_kernel<BITS, GS, true>), grid, dim3(kPPThreads), lds, s, P);
  else
    hipLaunchKernelGGL((prefill_pp_kernel<BITS, GS, false>), grid, dim3(kPPThreads), lds, s, P);
  return hipGetLastError();
}

template <int BITS>
hipError_t launch_bits(const PrefillParams& P, hipStream_t s) {
  if constexpr (BITS == 16)
    return launch_gs<16, 64>(P, s);  // no groups
  else
    return P.group_size == 32   ? launch_gs<BITS, 32>(P, s)
           : P.group_size == 64 ? launch_gs<BITS, 64>(P, s)
                                : launch_gs<BITS, 128>(P, s);
}

}  // namespace

bool prefill_supported(int64_t M, int64_t N, int64_t K, int bits, int gs) {
  if (bits == 16)  // bf16 weights: no groups, no scale chunks
    return M >= 1 && N >= 4 && N % 4 == 0 && K % kBK == 0 &&
           (int64_t)kBM * K * 2 < ((int64_t)1 << 31) && (int64_t)kBN * K * 2 < ((int64_t)1 << 31) &&
           M < ((int64_t)1 << 30) && N < ((int64_t)1 << 30);
  if ((bits != 4 && bits != 8) || (gs != 32 && gs != 64 && gs != 128)) return false;
  // 32-bit buffer offsets per block; 4-output stores; whole 64-wide steps and groups; an
  // even group count, so every row's scales and biases start on a dword (the staging
  // moves them as dwords)
  return M >= 1 && N >= 4 && N % 4 == 0 && K % kBK == 0 && K % gs == 0 && (K / gs) % 2 == 0 &&
         (int64_t)kBM * K * 2 < ((int64_t)1 << 31) && (int64_t)kBN * K * bits / 8 < ((int64_t)1 << 31) &&
         M < ((int64_t)1 << 30) && N < ((int64_t)1 << 30);
}

size_t prefill_plan(PrefillParams& P) {
  static const int forced_ks = [] {
    const char* v = std::getenv("MI_QMM_PREFILL_KS");
    return v ? std::atoi(v) : 0;
  }();
  const int steps = P.K / kBK;
  // Tile height and K splits: the fewest estimated microseconds, over rounds of 256 blocks
  // (one per CU) x 64-wide steps a split, plus, for a split, its fp32 partials written and
  // read back once (~6 TB/s) and the reduce launch. At least 8 steps a split; those of 128-row
  // tiles are whole 4-step units. Time a step, full grid: 256 x 256 tiles 1.65 us (4 bits and
  // bf16) and 1.75 (8 bits), 128 x 256 tiles 1.0 (4 bits), 1.15 (8 bits) and 1.3 (bf16). So a
  // product that fills the chip several times over takes the 256-row tiles, and the 128-row
  // ones pay where they need fewer splits. Measured, us, 256-row / 128-row tiles, 4 bits:
  //   [14336,4096]  256 rows 53 / 48   512 81 / 72   700 105 / 116  2003 217 / 245
  //   [4096,14336]  256 rows 52 / 45   512 72 / 70   700  94 / 110  1024 117 / 123
  //   [4096,4096]   256 rows 33 / 27   512 40 / 33   1024 52 / 50   2003  80 / 70
  // 8 bits: [4096,4096] 512 rows 40 / 35, [14336,4096] 700 rows 109 / 139; bf16 weights (with
  // the dequantize of 6-bit ones): [4096,4096] 256 rows 44 / 37, [14336,4096] 700 143 / 171.
  double best = 1e30;
  for (const int bm : {256, 128}) {
    const int64_t tiles = (int64_t)((P.M + bm - 1) / bm) * ((P.N + kBN - 1) / kBN);
    const int unit = bm == 128 ? 4 : 1;
    const double step_us = bm == 128 ? (P.bits == 4 ? 1.0 : P.bits == 8 ? 1.15 : 1.3)
                                     : (P.bits == 8 ? 1.75 : 1.65);
    const int k0 = forced_ks > 0 ? std::min(forced_ks, steps) : 1;
    const int k1 = forced_ks > 0 ? k0 : std::max(1, steps / 8);
    for (int k = k0; k <= k1; ++k) {
      const int sps = (steps + k * unit - 1) / (k * unit) * unit;
      const int ks = (steps + sps - 1) / sps;
      const double part_us = ks > 1 ? (double)ks * P.M * P.N * 8 / 6e6 + 3.0 : 0.0;
      const double cost = (double)((tiles * ks + 255) / 256) * sps * step_us + part_us;
      if (cost < best - 1e-9) {
        best = cost;
        P.bm = bm;
        P.ks = ks;
        P.sps = sps;
      }
    }
  }
  return P.ks > 1 ? (size_t)P.ks * P.M * P.N * sizeof(float) : 0;
}

hipError_t launch_prefill(const PrefillParams& P, hipStream_t s) {
  if (!prefill_supported(P.M, P.N, P.K, P.bits, P.group_size)) return hipErrorNotSupported;
  if (P.ks > 1 && !P.part) return hipErrorInvalidValue;
  hipError_t e = P.bm == 128    ? launch_prefill128(P, s)
                 : P.bits == 16 ? launch_bits<16>(P, s)
                 : P.bits == 8 ? launch_bits<8>(P, s)
                               : launch_bits<4>(P, s);
  if (e != hipSuccess || P.ks == 1) return e;
  return launch_split_reduce(P.part, P.y, (int64_t)P.M * P.N, P.ks, s);
}

hipError_t launch_split_reduce(const float* part, uint16_t* y, int64_t n, int ks, hipStream_t s) {
  const int64_t n4 = n / 4;
  int64_t g = (n4 + 255) / 256;
  if (g > 8192) g = 8192;
  hipLaunchKernelGGL(prefill_reduce_kernel, dim3((unsigned)g), dim3(256), 0, s, part, y, n4, ks);
  return hipGetLastError();
}

}  // namespace mi
