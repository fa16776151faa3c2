// Prefill GEMM on 128 (M) x 256 (N) tiles: 4- and 8-bit affine weights (groups of 32, 64, 128)
// and weights already expanded to bf16,
//   y[M,N] (bf16) = x[M,K] (bf16) @ dequant(w)[N,K]^T, fp32 accumulation,
// for the row counts where 256 x 256 tiles (prefill.hip) leave the chip idle or split K into
// more fp32 partials: [14336,4096] at 512 rows is 224 of these tiles, against 112 of those in
// two K halves (59 MB of partials written and read back).
//
// Block: 8 waves, two per SIMD; wave w owns weight rows 32w..32w+31 (two 16-row tiles of
// v_mfma_f32_16x16x32_bf16) against all 128 x rows (eight tiles): 16 accumulators of 4
// registers. Every weight of the block is dequantized once, as bf16(s*q + b).
//
// No ping-pong between wave groups (prefill.hip): with half the matrix work a step, its two
// barriers a step cost more than they hide (a 128-row tile there took 1.36 us a step). All
// waves run one stream in which each group of 8 MFMAs carries the LDS reads of the next group
// and a fourth of the next step's dequantize (sched_group_barrier: 1 MFMA, 4 VALU, an LDS read
// every second MFMA), and one barrier a step. 0.93 us a step measured (4-bit).
//
// Weights, scales and biases come straight into registers (4 steps and one 4-step unit ahead):
// one instruction reads 16 rows x 64 contiguous bytes. At 4 bits that is two steps; one
// v_permlane32_swap per dword pair gives each lane two dwords of either step, the 8-value runs
// sb, sb + 1 of the step's eight (sb = 4 (q % 2) + 2 (q / 2) for quarter q = lane / 16). x comes
// by LDS DMA into a ring of four 16 KB stages, issued one instruction per group of MFMAs; the
// barrier of a step sits before its last group, which reads the next step's first fragments.
// Vector memory operations return in order, so "x stage t + 1 has arrived" is an exact vmcnt.
//
// Measured, us a call, 256-row tiles -> these: 4-bit [14336,4096] 512 rows 81 -> 72, 256 rows
// 53 -> 48; [4096,4096] 256 rows 33 -> 27, 2003 rows 80 -> 70; [7168,2048] 700 rows 45 -> 34;
// 8-bit [4096,4096] 512 rows 40 -> 35. Which tile a call takes: prefill_plan.
#include "mi_common.h"
#include "mi_internal.h"
#include "qmv_common.h"
#include "dequant_bf16.h"
#include "prefill_tiles.h"

namespace mi {
namespace {

using dq::pack_bf16x2;
using qmv_detail::vmcnt_imm;

constexpr int kBufFlags = 0x00020000;   // raw dword access
constexpr uint32_t kOOB = 0x7FFFFFF0u;  // past any resource: the load returns 0
constexpr int kBM = 128, kBN = 256, kMT = 8, kRing = 4, kU = 4;
constexpr int kXStage = kBM * 128;  // 128 rows x 64 values
constexpr int kXI = 2;              // x DMA instructions of a wave per step

MI_DEV float lo_f(uint32_t v) { return __uint_as_float(v << 16); }
MI_DEV float hi_f(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }

template <int k>
MI_DEV float byte_f(uint32_t w) { return (float)((w >> (8 * k)) & 0xFFu); }
MI_DEV u32x4_t dequant8_bytes(uint32_t w0, uint32_t w1, float s, float b) {
  return u32x4_t{pack_bf16x2(fmaf(s, byte_f<0>(w0), b), fmaf(s, byte_f<1>(w0), b)),
                 pack_bf16x2(fmaf(s, byte_f<2>(w0), b), fmaf(s, byte_f<3>(w0), b)),
                 pack_bf16x2(fmaf(s, byte_f<0>(w1), b), fmaf(s, byte_f<1>(w1), b)),
                 pack_bf16x2(fmaf(s, byte_f<2>(w1), b), fmaf(s, byte_f<3>(w1), b))};
}

MI_DEV f32x4_t mfma16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return mfma16x16x32(as_bf16x8(a), as_bf16x8(b), c);
}

// 64 lanes x 16 bytes into 1 KB of LDS (lane order)
MI_DEV void dma16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)lds, 16,
                                           voff, soff, 0, 0);
}

// s_waitcnt vmcnt(n); n is a constant after unrolling
MI_DEV void wait_vm(int n) {
  switch (n) {
#define C(n) case n: __builtin_amdgcn_s_waitcnt(vmcnt_imm(n)); break;
    C(1) C(2) C(3) C(4) C(5) C(6) C(7) C(8) C(9) C(10) C(11) C(12) C(13) C(14) C(15) C(16)
    default: __builtin_amdgcn_s_waitcnt(vmcnt_imm(0)); break;
#undef C
  }
}

// XOR swizzle of the 16-byte slots of a 128-byte x row. A ds_read_b128 pass serves lanes 0-3,
// 12-15, 20-23 and 24-27 of a half together: rows 0-3 and 12-15 of quarter q meet rows 4-11 of
// quarter q + 1, whose slots differ by 4 (4 bits) or 2; the bit of r that separates 0-3 from
// its pair is put where that difference maps the pair onto itself.
template <int BITS>
MI_DEV int xswz(int r) {
  return BITS == 4 ? ((r & 2) << 1) | ((r >> 2) & 1) | ((r >> 2) & 2)
                   : (r & 2) | ((r >> 2) & 1) | ((r >> 1) & 4);
}

// Memory operations of a step by group u of 8 MFMAs (0..3): x at 0 (the second half of stage
// t + 2) and 3 (the first of t + 3); weights at 1 and 2 (4 bits: odd steps only; bf16: one in
// each group); the unit's 4 scale loads at 0 of its first step. Operations younger than x
// stage t + 1 (complete at group 0 of step t - 1) at the wait in group 3 of step t:
template <int BITS>
constexpr int younger(int t) {
  const int w = BITS == 4 ? 2 : BITS == 8 ? 4 : 6;
  return kXI + w + (BITS != 16 && t % kU == 0 ? 4 : 0);
}

template <int BITS, int GS, bool SPLIT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
prefill128_kernel(PrefillParams P) {
  constexpr bool W16 = BITS == 16;
  constexpr int CS = BITS == 4 ? 2 : 1, DC = kU / CS;  // steps a chunk, chunks held
  constexpr int H = 256 / GS;                          // scale halves of a unit
  constexpr int RB = BITS * 8;                         // bytes of a weight row per step
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, q = lane >> 4;
  const int M = P.M, N = P.N, K = P.K, G = K / GS;
  const TileOf at = tile_of_block((M + kBM - 1) / kBM, (N + kBN - 1) / kBN);
  const int mt = at.mt, nt = at.nt, split = at.split;
  const int m0 = mt * kBM, n0 = nt * kBN;
  const int s0 = split * P.sps;
  const int ns = min(P.sps, K / 64 - s0);  // steps that hold data; sps is a multiple of kU
  const uint32_t rowb = (uint32_t)(K / 8 * BITS);
  const int mrows = min(kBM, M - m0), nrows = min(kBN, N - n0);
  const uint32_t xrec = (uint32_t)mrows * (uint32_t)K * 2, wrec = (uint32_t)nrows * rowb;
  const uint16_t* xb = P.x + (size_t)m0 * K;
  const unsigned char* wb = (const unsigned char*)P.w + (size_t)n0 * rowb;
  const int sb = BITS == 4 ? 4 * (q & 1) + 2 * (q >> 1) : 2 * q;

  uint32_t xo[kXI];
#pragma unroll
  for (int j = 0; j < kXI; ++j) {
    const int r = 8 * (wave * kXI + j) + (lane >> 3), c = (lane & 7) ^ xswz<BITS>(r);
    xo[j] = r < mrows ? (uint32_t)(r * K + 64 * s0 + 8 * c) * 2 : kOOB;
  }
  uint32_t wo[2], so[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const uint32_t r = (uint32_t)min(32 * wave + 16 * a + fr, nrows - 1);
    wo[a] = r * rowb + (uint32_t)(s0 * RB) + (W16 ? 32 : 16) * q;
    so[a] = (r * (uint32_t)G + (uint32_t)s0 * 64 / GS) * 2;  // on a dword: G is even
  }
  const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(P.scales + (W16 ? 0 : (size_t)n0 * G)), (short)0,
      W16 ? 0u : (uint32_t)nrows * (uint32_t)G * 2, kBufFlags);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(P.biases + (W16 ? 0 : (size_t)n0 * G)), (short)0,
      W16 ? 0u : (uint32_t)nrows * (uint32_t)G * 2, kBufFlags);

  // t0: first step of a unit (a multiple of kU, so ring slots are constants). Steps past the
  // range load through a resource of zero records (zeros, no traffic).
  u32x4_t W[DC][W16 ? 4 : 2];  // chunk: two row tiles; bf16: [2a + e], the operands themselves
  auto load_w = [&](int t0, int c, int o) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)wb, (short)0, t0 + CS * c < ns ? wrec : 0u, kBufFlags);
    W[c % DC][o] = W16 ? __builtin_amdgcn_raw_buffer_load_b128(rs, wo[o / 2] + 16 * (o % 2),
                                                               (t0 + c) * RB, 0)
                       : __builtin_amdgcn_raw_buffer_load_b128(rs, wo[o % 2], (t0 / CS + c) * 64, 0);
  };
  auto load_x = [&](int t0, int t, int j) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)xb, (short)0, t0 + t < ns ? xrec : 0u, kBufFlags);
    dma16(rs, smem + (t % kRing) * kXStage + (wave * kXI + j) * 1024, xo[j], (t0 + t) * 128);
  };
  uint32_t ts[2][H / 2], tb[2][H / 2], sd[2][H / 2], bd[2][H / 2];
  auto load_half = [&](__amdgpu_buffer_rsrc_t rs, uint32_t (&d)[H / 2], int a, int off)
      __attribute__((always_inline)) {
    if constexpr (H == 8) {
      const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, so[a], off, 0);
      d[0] = v.x, d[1] = v.y, d[2] = v.z, d[3] = v.w;
    } else if constexpr (H == 4) {
      const u32x2_t v =
          __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rs, so[a], off, 0));
      d[0] = v.x, d[1] = v.y;
    } else {
      d[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, so[a], off, 0);
    }
  };
  auto load_s = [&](int t0) __attribute__((always_inline)) {
    if constexpr (!W16) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        load_half(sres, ts[a], a, t0 / kU * H * 2);
        load_half(bres, tb[a], a, t0 / kU * H * 2);
      }
    }
  };
  auto take_s = [&](int t0) __attribute__((always_inline)) {
    if constexpr (!W16) {
#pragma unroll
      for (int d = 0; d < H / 2; ++d) {
        // halves of steps past the range belong to another row: masked out
        const int g0 = t0 + 2 * d * GS / 64, g1 = t0 + (2 * d + 1) * GS / 64;
        const uint32_t mask = (g0 < ns ? 0xFFFFu : 0u) | (g1 < ns ? 0xFFFF0000u : 0u);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          sd[a][d] = ts[a][d] & mask;
          bd[a][d] = tb[a][d] & mask;
        }
      }
    }
  };
  // a 4-bit chunk's dwords to step order: {step 0: 2, step 1: 2}
  auto prep_w = [&](int t) __attribute__((always_inline)) {
    if constexpr (BITS == 4) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        u32x4_t& v = W[(t / CS) % DC][a];
        const auto p = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
        const auto r = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
        v = u32x4_t{p[0], r[0], p[1], r[1]};
      }
    }
  };
  // operand of row tile a, k-step e in step t of the unit
  auto dq_w = [&](int t, int a, int e) -> u32x4_t {
    const u32x4_t v = W[(t / CS) % DC][a];
    const int hf = GS == 32 ? 2 * t : GS == 64 ? t : t / 2;  // (32: the lane's half of a pair)
    const bool up = GS == 32 ? sb >= 4 : hf % 2;
    const float s = up ? hi_f(sd[a][hf / 2]) : lo_f(sd[a][hf / 2]);
    const float b = up ? hi_f(bd[a][hf / 2]) : lo_f(bd[a][hf / 2]);
    if constexpr (BITS == 4) return dq::dequant8(v[2 * (t % 2) + e], s, b);
    return dequant8_bytes(v[2 * e], v[2 * e + 1], s, b);
  };
  auto xfrag = [&](int t, int i, int e) -> u32x4_t {
    const int r = 16 * i + fr, c = sb + e;
    return *reinterpret_cast<const u32x4_t*>(smem + (t % kRing) * kXStage + r * 128 +
                                             ((c ^ xswz<BITS>(fr)) << 4));
  };

  f32x4_t acc[2][kMT];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < kMT; ++i) acc[a][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Prologue, in the order that `younger` counts: the last weight loads and the first half of
  // x stage 2 come after stage 1, as in the loop. (bf16: chunk 3 goes out in step 0, and the
  // three loads counted in step -1 are those of chunk 2 here.)
  load_s(0);
  constexpr int kLate = W16 ? 2 : DC - 1;  // chunk whose loads the loop would issue in step -1
#pragma unroll
  for (int c = 0; c < kLate; ++c)
#pragma unroll
    for (int o = 0; o < (W16 ? 4 : 2); ++o) load_w(0, c, o);
  if constexpr (W16) load_w(0, kLate, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < kXI; ++j) load_x(0, t, j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int o = W16 ? 1 : 0; o < (W16 ? 4 : 2); ++o) load_w(0, kLate, o);
  __builtin_amdgcn_sched_barrier(0);
  load_x(0, 2, 0);
  __builtin_amdgcn_sched_barrier(0);
  wait_vm(kXI + (W16 ? 3 : 2) + 1);  // stage 0 has landed
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);

  u32x4_t X[2][4], A[2][2][2];  // x tiles 4 at a time; operands of this step and the next
#pragma unroll
  for (int i = 0; i < 4; ++i) X[0][i] = xfrag(0, i, 0);
  take_s(0);
  prep_w(0);
  if constexpr (!W16) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int e = 0; e < 2; ++e) A[0][a][e] = dq_w(0, a, e);
  }
#pragma unroll 1
  for (int t0 = 0; t0 < P.sps; t0 += kU) {
#pragma unroll
    for (int t = 0; t < kU; ++t) {
      const int tn = t + 1;  // next step
      if (tn % kU == 0) take_s(t0 + tn);
      if (tn % CS == 0) prep_w(tn % kU);
      // four groups: k-step u / 2 against x tiles 4(u%2) .. +3
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (u == 3) {
          wait_vm(younger<BITS>(t));  // this wave's part of x stage t + 1
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
        if (u == 3) load_x(t0, t + 3, 0);  // stage t - 1: every wave is past its last read
        if (u == 0) load_x(t0, t + 2, 1);
        if (u == 0 && t == 0) load_s(t0 + kU);
        if constexpr (W16) {
          load_w(t0, t + 3, u);  // into the slot of step t - 1
        } else {
          if (u >= 1 && u <= 2 && (BITS == 8 || t % 2 == 1)) load_w(t0, t / CS + DC, u - 1);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          X[(u + 1) & 1][i] = xfrag(u < 3 ? t : tn, 4 * ((u + 1) & 1) + i, u < 3 ? (u + 1) / 2 : 0);
        if constexpr (!W16) A[tn & 1][u & 1][u >> 1] = dq_w(tn % kU, u & 1, u >> 1);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            f32x4_t& c = acc[a][4 * (u & 1) + i];
            c = mfma16(W16 ? W[t % DC][(W16 ? 2 * a : 0) + u / 2] : A[t & 1][a][u / 2],
                       X[u & 1][i], c);
          }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (m % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          if (m == 3 || m == 5) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // no DMA may outlive the block

  // acc[a][i] register r is D[n = 32 wave + 16a + 4q + r][m = 16 i + fr]
#pragma unroll
  for (int i = 0; i < kMT; ++i) {
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

template <int BITS, int GS>
hipError_t launch_gs(const PrefillParams& P, hipStream_t s) {
  constexpr int lds = kRing * kXStage;
  const dim3 grid((unsigned)(((P.M + kBM - 1) / kBM) * ((P.N + kBN - 1) / kBN)), (unsigned)P.ks);
  if (P.ks > 1)
    hipLaunchKernelGGL((prefill128_kernel<BITS, GS, true>), grid, dim3(512), lds, s, P);
  else
    hipLaunchKernelGGL((prefill128_kernel<BITS, GS, false>), grid, dim3(512), lds, s, P);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_prefill128(const PrefillParams& P, hipStream_t s) {
  if (P.bits == 16) return launch_gs<16, 64>(P, s);
  if (P.bits == 8)
    return P.group_size == 32   ? launch_gs<8, 32>(P, s)
           : P.group_size == 64 ? launch_gs<8, 64>(P, s)
                                : launch_gs<8, 128>(P, s);
  return P.group_size == 32   ? launch_gs<4, 32>(P, s)
         : P.group_size == 64 ? launch_gs<4, 64>(P, s)
                              : launch_gs<4, 128>(P, s);
}

}  // namespace mi
