// Mid-row quantized GEMM, 17..128 activation rows, affine weights in groups of 64 (4 and 8 bits;
// 2, 3, 5 and 6 bits from 33 rows) and nvfp4 / mxfp4 / mxfp8 (from 33 rows):
//   y[M,N] (bf16) = x[M,K] (bf16) @ dequant(w)[N,K]^T, fp32 accumulation,
// on v_mfma_f32_32x32x16_bf16 with D[m][n] = x[m][k] W[n][k], so a lane's accumulators all
// belong to one weight row n = lane % 32 and its scale is one register.
//
// What bounds it: at 32 rows the weight stream (33 MB for [14336,4096] at 4 bits), at 128 rows
// the x traffic from L2 (every block reads all its x rows: about 42 B/clk a CU measured for
// LDS DMA, 1 MB a block at 128 rows) and the LDS fragment reads, both near the matrix time.
//
// Block: WN x WK waves. Wave (wn, kp) owns 32 weight rows and every WK-th part of the K range
// against all the rows (MT tiles of 32); the WN waves of a K part share its x tiles. K is
// split inside the block first (the parts are added through LDS at the end, in order), so a
// wide matrix needs no fp32 partials in memory: 64-row blocks give [14336,4096] 224 blocks.
//
// Step: 64 values of K, one group. x comes by LDS DMA into a ring of R tiles (128-byte rows,
// 16-byte slots XOR-swizzled by row), R - 1 steps ahead. Weights come straight into
// registers, D steps ahead, in chunks of 64 bytes of each row (2 steps at 4 bits, 1 at 8):
// one instruction reads 16 rows x 64 contiguous bytes (reading a lane's own 16 bytes of 32
// rows instead re-fetched each line: 17.7 against 15.1 us at 32 rows), and one
// v_permlane16_swap per dword pair puts a row's quarters into its own two lanes. Vector
// memory operations return in order, so "x tile t has arrived" is an exact vmcnt.
//
// EX (up to 64 rows): the codes enter the matrix product as exact bf16 integers; a group's
// sum is scaled in fp32 (s * sum, one FMA a value) and the bias term b_g * X_g (X_g = sum of
// x over the group, v_dot2 against ones) is added as one more matrix product per unit of U
// groups, X_g split into three bf16 parts (24 bits): no rounding of the weight. Otherwise
// (more rows, where the kernels below already round) operands are bf16(s q + b), as the
// prefill kernel's: 76 VALU a step and row tile whatever the rows, against 52 + 32 a tile.
//
// The bias-less modes use the 4- and 8-bit layouts; code x scale is exact in bf16
// (code_runs.h), so they need neither epilogue nor rounding. The conversions are exact at every
// scale byte but e8m0 255 (infinity; they give NaN): a wave that met one sums its range again
// after the loop, straight from memory, with such groups decoded by hand (a second copy of the
// pipelined steps spilled). The other widths are one
// bitstream a row: a lane loads the 4 * bits bytes of its own 32 codes.
//
// Steps past a wave's range load through a resource of zero records (zeros, no traffic) and
// their scales are masked to zero, so any K that is a multiple of 64 runs.
//
// Measured (us a call, distinct weights, before -> after): [14336,4096] 4-bit 32 rows
// 19.5 -> 15.5, 64 rows 37 -> 20.5, 77 rows 54 -> 23, 128 rows 42.3 -> 26.7; 8-bit 64 rows
// 45 -> 27, 128 rows 42.9 -> 30.1. At 77 rows the matrix cores are busy 16% and the VALU 17%.
#pragma once
#include "mi_common.h"
#include "qmv_common.h"
#include "dequant_bf16.h"
#include "code_runs.h"

namespace mi {
namespace midm {

using qmv_detail::mfma32;
using qmv_detail::vmcnt_imm;

constexpr int kBufFlags = 0x00020000;   // raw dword access
constexpr uint32_t kOOB = 0x7FFFFFF0u;  // past any resource: the load returns 0

using dq::pack_bf16x2;
typedef __bf16 bf16x2m __attribute__((ext_vector_type(2)));

MI_DEV float lo_f(uint32_t v) { return __uint_as_float(v << 16); }
MI_DEV float hi_f(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }
MI_DEV uint32_t cvt8(uint32_t v, bool hi) {
  return hi ? __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.f, true))
            : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.f, false));
}
// 8 nibbles -> exact bf16 pairs (q0, q1) .. (q6, q7): a byte 0..15 read as an e4m3 code is
// q * 2^-9 (dequant_bf16.h).
MI_DEV u32x4_t codes4(uint32_t w) {
  const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
  const uint32_t a = perm_b32(hi, lo, 0x05010400u), b = perm_b32(hi, lo, 0x07030602u);
  return u32x4_t{cvt8(a, false), cvt8(a, true), cvt8(b, false), cvt8(b, true)};
}
// 8 bytes -> exact bf16 pairs of the codes, or of s q + b with one rounding.
template <int k>
MI_DEV float byte_f(uint32_t w) { return (float)((w >> (8 * k)) & 0xFFu); }
MI_DEV u32x4_t codes8(uint32_t w0, uint32_t w1) {
  return u32x4_t{pack_bf16x2(byte_f<0>(w0), byte_f<1>(w0)), pack_bf16x2(byte_f<2>(w0), byte_f<3>(w0)),
                 pack_bf16x2(byte_f<0>(w1), byte_f<1>(w1)), pack_bf16x2(byte_f<2>(w1), byte_f<3>(w1))};
}
MI_DEV u32x4_t dequant8_bytes(uint32_t w0, uint32_t w1, float s, float b) {
  return u32x4_t{pack_bf16x2(fmaf(s, byte_f<0>(w0), b), fmaf(s, byte_f<1>(w0), b)),
                 pack_bf16x2(fmaf(s, byte_f<2>(w0), b), fmaf(s, byte_f<3>(w0), b)),
                 pack_bf16x2(fmaf(s, byte_f<0>(w1), b), fmaf(s, byte_f<1>(w1), b)),
                 pack_bf16x2(fmaf(s, byte_f<2>(w1), b), fmaf(s, byte_f<3>(w1), b))};
}

// Exchange the odd 16-lane rows of a with the even ones of b.
MI_DEV void swap16(u32x4_t& a, u32x4_t& b) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const auto r = __builtin_amdgcn_permlane16_swap(a[d], b[d], false, false);
    a[d] = r[0];
    b[d] = r[1];
  }
}
// v plus the value of lane ^ 32.
MI_DEV float add_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v - its bf16 part; 0 when that part is infinite (inf - inf would turn the sum to NaN).
MI_DEV float rest(float v, float part) {
  return __builtin_fabsf(part) == __builtin_inff() ? 0.f : v - part;
}

// 64 lanes x 16 bytes into 1 KB of LDS (lane order)
MI_DEV void dma16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)lds, 16,
                                           voff, soff, 0, 0);
}
// s_waitcnt vmcnt(n); n is a constant after unrolling
MI_DEV void wait_vm(int n) {
  switch (n > 31 ? 31 : n) {
#define C(n) case n: __builtin_amdgcn_s_waitcnt(vmcnt_imm(n)); break;
    C(0) C(1) C(2) C(3) C(4) C(5) C(6) C(7) C(8) C(9) C(10) C(11) C(12) C(13) C(14) C(15)
    C(16) C(17) C(18) C(19) C(20) C(21) C(22) C(23) C(24) C(25) C(26) C(27) C(28) C(29) C(30)
    default: __builtin_amdgcn_s_waitcnt(vmcnt_imm(31)); break;
#undef C
  }
}

// acc + the sum of the two bf16 values of v
MI_DEV float sum2(uint32_t v, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2m, v),
                                         __builtin_bit_cast(bf16x2m, 0x3F803F80u), acc, false);
}

template <int MT, int WN, int WK, int R>
constexpr int midm_lds() {
  const int a = WK * R * MT * 4096, b = WN * WK * MT * 4096;  // x rings; the waves' partial tiles
  return a > b ? a : b;
}

// Vector-memory operations that are certainly younger than X(t) when step t waits for it.
template <int CS, int R, int D, int U, int WOPS, int XOPS, int SOPS>
constexpr int midm_younger(int t) {
  // X(u) goes out in step u - R + 1 after that step's wait (in step 0 with the next unit's
  // scales, in either order); at the end of a step that ends a chunk, the weights D steps on
  int n = 0;
  for (int v = t - R + 1; v < t; ++v) {
    const int m = ((v % U) + U) % U;
    if (v > t - R + 1) n += XOPS + (m == 0 ? SOPS : 0);
    if (m % CS == CS - 1) n += WOPS;
  }
  if (t < R - 1) {  // in the first unit X(t) came from the prologue: W X(0) X(1) W X(2) ..
    int p = 0;
    for (int u = t + 1; u < (D > R - 1 ? D : R - 1); ++u) {
      if (u % CS == 0 && u < D) p += WOPS;
      if (u < R - 1) p += XOPS;
    }
    for (int v = 0; v < t; ++v) {
      p += XOPS + (v == 0 ? SOPS : 0);
      if (v % CS == CS - 1) p += WOPS;
    }
    n = p < n ? p : n;
  }
  return n;
}

// Storage bits of a format: affine bits, or 100 nvfp4, 101 mxfp4, 102 mxfp8.
constexpr int fmt_bits(int fmt) { return fmt < 100 ? fmt : fmt == 102 ? 8 : 4; }

// 8 codes of OB bits starting `byte` bytes into the lane's dwords -> bf16 pairs of s q + b.
template <int OB, int byte>
MI_DEV u32x4_t dequant8_odd(const uint32_t (&d)[OB], float s, float b) {
  constexpr int i = byte / 4, sh = byte % 4 * 8;
  const uint64_t v = ((((uint64_t)(i + 1 < OB ? d[i + 1 < OB ? i + 1 : i] : 0u)) << 32) | d[i]) >> sh;
  auto val = [&](int c) { return fmaf(s, (float)((uint32_t)(v >> (c * OB)) & ((1u << OB) - 1u)), b); };
  return u32x4_t{pack_bf16x2(val(0), val(1)), pack_bf16x2(val(2), val(3)),
                 pack_bf16x2(val(4), val(5)), pack_bf16x2(val(6), val(7))};
}

template <int FMT, bool EX, int MT, int WN, int WK, int R, int D>
__global__ void __launch_bounds__(64 * WN * WK) midm_kernel(MidmParams P) {
  constexpr bool FP = FMT >= 100;
  constexpr int BITS = fmt_bits(FMT);
  constexpr bool ODD = BITS != 4 && BITS != 8;
  constexpr bool E8M0 = FMT == 101 || FMT == 102;
  static_assert(!EX || (!FP && !ODD), "exact codes: affine 4 and 8 bits");
  constexpr int U = 4;  // steps of a unit: the loop body, one load of scales and biases
  constexpr int CS = BITS == 4 ? 2 : 1, DC = D / CS;
  constexpr int XI = 4 * MT / WN;  // x DMA instructions of a wave per step
  static_assert(4 * MT % WN == 0 && U % R == 0 && U % D == 0 && D % CS == 0, "rings");
  constexpr int WOPS = ODD ? (BITS > 4 ? 2 : 1) : 2, SOPS = !FP ? 4 : FMT == 100 ? 1 : 2;
  constexpr int BN = 32 * WN, BM = 32 * MT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, kp = wave / WN;
  const int fr = lane & 31, h = lane >> 5;
  const int M = P.M, N = P.N, K = P.K, G = K / 64;
  const int n0 = blockIdx.x * BN + wn * 32;
  const int s0 = (blockIdx.y * WK + kp) * P.steps;
  const int ns = min(P.steps, G - s0);  // steps of this wave that hold data, may be <= 0

  const uint32_t xrec = (uint32_t)M * (uint32_t)K * 2, rowb = (uint32_t)(K / 8 * BITS);
  const uint32_t wrec = (uint32_t)N * rowb;
  uint32_t xo[XI];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int r = 8 * (wn * XI + j) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    xo[j] = r < M ? (uint32_t)(r * K + 64 * s0 + 8 * c) * 2 : kOOB;
  }
  // instruction e of a chunk: rows 16e .. 16e+15, lane l row l % 16, quarter l/32 + 2 ((l/16) % 2)
  uint32_t wo[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int r = min(n0 + 16 * e + (lane & 15), N - 1);
    wo[e] = (uint32_t)r * rowb + (uint32_t)(s0 * 8 * BITS) + 16 * (h + 2 * ((lane >> 4) & 1));
  }
  // bitstream widths: the lane's own 4 * BITS bytes of row fr
  const uint32_t wodd =
      (uint32_t)min(n0 + fr, N - 1) * rowb + (uint32_t)(s0 * 8 * BITS) + (uint32_t)(4 * BITS * h);
  // A step's scales are one half of the row's run of G halves (one bf16 scale, or two e8m0
  // bytes; nvfp4: one dword). The run starts at any half: dwords from the one that holds the
  // first, shifted
  const uint32_t sa = ((uint32_t)min(n0 + fr, N - 1) * (uint32_t)G + (uint32_t)s0) * 2;
  const uint32_t so = FMT == 100 ? sa * 2 : sa & ~3u, ssh = FMT == 100 ? 0u : (sa & 2u) * 8u;
  const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)P.scales, (short)0, (uint32_t)N * (uint32_t)G * (FMT == 100 ? 4 : 2), kBufFlags);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)P.biases, (short)0, (uint32_t)N * (uint32_t)G * 2, kBufFlags);
  unsigned char* ring = smem + kp * (R * MT * 4096);

  // t0: first step of a unit (a multiple of U, so ring slots are constants), t: step in it
  u32x4_t W[ODD ? 1 : DC][2];
  uint32_t WO[ODD ? D : 1][ODD ? BITS : 1];
  auto load_w = [&](int t0, int c) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)P.w, (short)0, t0 + CS * c < ns ? wrec : 0u, kBufFlags);
    if constexpr (ODD) {
      uint32_t(&d)[BITS] = WO[c % D];
      const int off = (t0 + c) * 8 * BITS;
      if constexpr (BITS == 2) {
        const u32x2_t a = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rs, wodd, off, 0));
        d[0] = a.x, d[1] = a.y;
      } else if constexpr (BITS == 3) {
        const auto a = __builtin_amdgcn_raw_buffer_load_b96(rs, wodd, off, 0);
        d[0] = a[0], d[1] = a[1], d[2] = a[2];
      } else {
        const u32x4_t a = __builtin_amdgcn_raw_buffer_load_b128(rs, wodd, off, 0);
        d[0] = a.x, d[1] = a.y, d[2] = a.z, d[3] = a.w;
        if constexpr (BITS == 5) {
          d[4] = __builtin_amdgcn_raw_buffer_load_b32(rs, wodd + 16, off, 0);
        } else {
          const u32x2_t e = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rs, wodd + 16, off, 0));
          d[4] = e.x, d[5] = e.y;
        }
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
      W[ODD ? 0 : c % DC][e] = __builtin_amdgcn_raw_buffer_load_b128(rs, wo[e], (t0 / CS + c) * 64, 0);
  };
  auto load_x = [&](int t0, int t) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)P.x, (short)0, t0 + t < ns ? xrec : 0u, kBufFlags);
#pragma unroll
    for (int j = 0; j < XI; ++j)
      dma16(rs, ring + (t % R) * (MT * 4096) + (wn * XI + j) * 1024, xo[j], (t0 + t) * 128);
  };
  uint32_t ts[FMT == 100 ? 4 : 3], tb[3];
  auto load_s = [&](int t0) __attribute__((always_inline)) {
    if constexpr (FMT == 100) {
      const u32x4_t a = __builtin_amdgcn_raw_buffer_load_b128(sres, so, t0 * 4, 0);
      ts[0] = a.x, ts[1] = a.y, ts[2] = a.z, ts[3] = a.w;
    } else {
      const uint32_t last = ssh ? so + 8 : kOOB;
      const u32x2_t a = __builtin_bit_cast(
          u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(sres, so, t0 * 2, 0));
      ts[0] = a.x, ts[1] = a.y;
      ts[2] = __builtin_amdgcn_raw_buffer_load_b32(sres, last, t0 * 2, 0);
      if constexpr (!FP) {
        const u32x2_t b = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(bres, so, t0 * 2, 0));
        tb[0] = b.x, tb[1] = b.y;
        tb[2] = __builtin_amdgcn_raw_buffer_load_b32(bres, last, t0 * 2, 0);
      }
    }
  };

  load_s(0);
#pragma unroll
  for (int t = 0; t < (D > R - 1 ? D : R - 1); ++t) {
    // (the fences keep the order that midm_younger counts)
    __builtin_amdgcn_sched_barrier(0);
    if (t % CS == 0 && t < D) load_w(0, t / CS);
    __builtin_amdgcn_sched_barrier(0);
    if (t < R - 1) load_x(0, t);
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x16_t zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;
  f32x16_t acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = zero;

  // x fragment of rows 32j.., k-step ks: the 8 values the weight operand of ks covers
  auto xfrag = [&](int t, int j, int ks) -> u32x4_t {
    const int r = 32 * j + fr;
    const int c = BITS != 8 ? 4 * h + ks : 4 * (ks / 2) + 2 * h + ks % 2;
    return *reinterpret_cast<const u32x4_t*>(ring + (t % R) * (MT * 4096) + r * 128 +
                                             ((c ^ ((r >> 1) & 7)) << 4));
  };
  uint32_t ff = 0;  // non-zero: a scale byte of the lane's row is 255
#pragma unroll 1
  for (int t0 = 0; t0 < P.steps; t0 += U) {
    uint32_t sd[FMT == 100 ? 4 : 2], bd[2] = {0u, 0u};
    if constexpr (FMT == 100) {
#pragma unroll
      for (int d = 0; d < 4; ++d) sd[d] = t0 + d < ns ? ts[d] : 0u;
    } else {
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int g = t0 + 2 * d;  // steps past the range: another row's values, masked out
        const uint32_t mask = (g < ns ? 0xFFFFu : 0u) | (g + 1 < ns ? 0xFFFF0000u : 0u);
        sd[d] = __builtin_amdgcn_alignbit(ts[d + 1], ts[d], ssh) & mask;
        if constexpr (!FP) bd[d] = __builtin_amdgcn_alignbit(tb[d + 1], tb[d], ssh) & mask;
        if constexpr (E8M0) ff |= code_runs::ff_bytes(sd[d]);
      }
    }
    float xs[EX ? MT : 1][U];
    if constexpr (EX) {
#pragma unroll
      for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int t = 0; t < U; ++t) xs[j][t] = 0.f;
    }
#pragma unroll
    for (int t = 0; t < U; ++t) {
      if (t % 2 == 0 && t && t0 + t >= P.steps) break;  // steps is even
      wait_vm(midm_younger<CS, R, D, U, WOPS, XI, SOPS>(t));
      if constexpr (WN > 1) __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (t == 0) load_s(t0 + U);
      load_x(t0, t + R - 1);
      __builtin_amdgcn_sched_barrier(0);
      u32x4_t xf[MT][4];
#pragma unroll
      for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) xf[j][ks] = xfrag(t, j, ks);
      if constexpr (EX) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          float a = 0.f, b = 0.f;
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            a = sum2(xf[j][ks].x, a);
            b = sum2(xf[j][ks].y, b);
            a = sum2(xf[j][ks].z, a);
            b = sum2(xf[j][ks].w, b);
          }
          xs[j][t] = a + b;
        }
      }
      u32x4_t& w0 = W[ODD ? 0 : (t / CS) % DC][0];
      u32x4_t& w1 = W[ODD ? 0 : (t / CS) % DC][1];
      if (!ODD && t % CS == 0) swap16(w0, w1);
      const uint32_t sw = FMT == 100 ? sd[t] : sd[t / 2] >> (16 * (t % 2)) & 0xFFFFu;
      const float s = FP ? 0.f : __uint_as_float(sw << 16);
      const float b = FP ? 0.f : t % 2 ? hi_f(bd[t / 2]) : lo_f(bd[t / 2]);
      // e8m0 byte `i` of the step's two as the exponent field of a float
      auto e8m0 = [&](int i) { return __uint_as_float((sw >> (8 * i) & 0xFFu) << 23); };
      u32x4_t wq[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        if constexpr (ODD) {
          wq[ks] = ks == 0   ? dequant8_odd<BITS, 0>(WO[t % D], s, b)
                   : ks == 1 ? dequant8_odd<BITS, BITS>(WO[t % D], s, b)
                   : ks == 2 ? dequant8_odd<BITS, 2 * BITS>(WO[t % D], s, b)
                             : dequant8_odd<BITS, 3 * BITS>(WO[t % D], s, b);
        } else if constexpr (BITS == 4) {
          const uint32_t v = t % 2 ? w1[ks] : w0[ks];
          if constexpr (FMT == 100)  // 16-code groups: bytes 2h and 2h + 1 of the step's four
            wq[ks] = code_runs::fp4_run_e4m3(
                v, code_runs::fp_e4m3(sw >> (16 * h + 8 * (ks / 2)) & 0xFFu));
          else if constexpr (FMT == 101)  // 32-code groups: the lane half's byte
            wq[ks] = code_runs::fp4_run(v, e8m0(h));
          else
            wq[ks] = EX ? codes4(v) : dq::dequant8(v, s, b);
        } else {
          const u32x4_t v = ks / 2 ? w1 : w0;
          const uint32_t d0 = ks % 2 ? v.z : v.x, d1 = ks % 2 ? v.w : v.y;
          if constexpr (FMT == 102)  // 32-code groups: the first two k-steps, the last two
            wq[ks] = code_runs::fp8_run(d0, d1, e8m0(ks / 2));
          else
            wq[ks] = EX ? codes8(d0, d1) : dequant8_bytes(d0, d1, s, b);
        }
        if constexpr (!EX) {
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[j] = mfma32(xf[j][ks], wq[ks], acc[j]);
        }
      }
      if constexpr (EX) {
        // one tile's group sum at a time (two in flight spilled at 256 registers)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          f32x16_t c = zero;
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) c = mfma32(xf[j][ks], wq[ks], c);
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[j][r] = fmaf(s, c[r], acc[j][r]);
        }
      }
      if (t % CS == CS - 1) load_w(t0, (t + 1 - CS + D) / CS);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EX) {
      // bias term of the unit's 4 groups: k slots of lanes h = 0 take the high and middle
      // parts of the X_g, lanes h = 1 the low parts
      const u32x4_t B = {bd[0], bd[1], bd[0], bd[1]};
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        uint32_t hi[2], mi[2], lo[2];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const float X0 = add_halves(xs[j][2 * d]), X1 = add_halves(xs[j][2 * d + 1]);
          hi[d] = pack_bf16x2(X0, X1);
          const float r0 = rest(X0, lo_f(hi[d])), r1 = rest(X1, hi_f(hi[d]));
          mi[d] = pack_bf16x2(r0, r1);
          lo[d] = pack_bf16x2(r0 - lo_f(mi[d]), r1 - hi_f(mi[d]));
        }
        const u32x4_t A = h ? u32x4_t{lo[0], lo[1], 0, 0} : u32x4_t{hi[0], hi[1], mi[0], mi[1]};
        acc[j] = mfma32(A, B, acc[j]);
      }
    }
  }
  if constexpr (E8M0) {
    if (__builtin_amdgcn_ballot_w64(ff != 0u)) {
      const __amdgpu_buffer_rsrc_t xrs =
          __builtin_amdgcn_make_buffer_rsrc((void*)P.x, (short)0, xrec, kBufFlags);
      const __amdgpu_buffer_rsrc_t wrs =
          __builtin_amdgcn_make_buffer_rsrc((void*)P.w, (short)0, wrec, kBufFlags);
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] = zero;
#pragma unroll 1
      for (int t = 0; t < ns; ++t) {
        const uint32_t sw = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(sres, sa + 2 * t, 0, 0);
#pragma unroll 1
        for (int ks = 0; ks < 4; ++ks) {
          // the 8 values that operand ks holds in the loop above
          const int c = BITS == 4 ? 4 * h + ks : 4 * (ks / 2) + 2 * h + ks % 2;
          const uint32_t wb = (uint32_t)min(n0 + fr, N - 1) * rowb + (uint32_t)((s0 + t) * 8 + c) * BITS;
          const uint32_t sc = sw >> (8 * (c / 4)) & 0xFFu;  // 32-code groups
          u32x2_t q = {0u, 0u};
          if constexpr (BITS == 4)
            q.x = __builtin_amdgcn_raw_buffer_load_b32(wrs, wb, 0, 0);
          else
            q = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(wrs, wb, 0, 0));
          const float f = __uint_as_float(sc << 23);
          const u32x4_t w = sc == 0xFFu ? code_runs::inf_run<BITS>(q.x, q.y)
                            : BITS == 4 ? code_runs::fp4_run(q.x, f)
                                        : code_runs::fp8_run(q.x, q.y, f);
#pragma unroll
          for (int j = 0; j < MT; ++j) {
            const int r = 32 * j + fr;
            const uint32_t xb = r < M ? (uint32_t)(r * K + 64 * (s0 + t) + 8 * c) * 2 : kOOB;
            acc[j] = mfma32(__builtin_amdgcn_raw_buffer_load_b128(xrs, xb, 0, 0), w, acc[j]);
          }
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // no DMA may land on the sums below
  __syncthreads();
  // sums of the K parts, in order: red[kp][m][n of the block]
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      red[(kp * BM + 32 * j + 8 * (r / 4) + 4 * h + r % 4) * BN + 32 * wn + fr] = acc[j][r];
  __syncthreads();
  constexpr int C4 = BN / 4;
  for (int o = tid; o < M * C4; o += 64 * WN * WK) {
    const int m = o / C4, c = o % C4;
    const int n = blockIdx.x * BN + 4 * c;
    if (n >= N) continue;
    const f32x4_t* p = reinterpret_cast<const f32x4_t*>(red) + m * C4 + c;
    f32x4_t v = p[0];
#pragma unroll
    for (int k = 1; k < WK; ++k) v += p[k * BM * C4];
    if (gridDim.y > 1)
      *reinterpret_cast<f32x4_t*>(P.part + ((size_t)blockIdx.y * M + m) * N + n) = v;
    else
      *reinterpret_cast<u32x2_t*>(P.y + (size_t)m * N + n) =
          u32x2_t{pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)};
  }
}

template <int FMT, bool EX, int MT, int WN, int WK, int R>
hipError_t launch_one(const MidmParams& P, hipStream_t s) {
  // two chunks in flight (8-bit: 20.5 us at 2, 21.6 at 4 steps)
  constexpr int D = fmt_bits(FMT) == 8 ? 2 : 4;
  constexpr int lds = midm_lds<MT, WN, WK, R>();
  auto k = midm_kernel<FMT, EX, MT, WN, WK, R, D>;
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  hipLaunchKernelGGL(k, dim3((unsigned)((P.N + 32 * WN - 1) / (32 * WN)), (unsigned)P.ks),
                     dim3(64 * WN * WK), lds, s, P);
  return hipGetLastError();
}

// The instances of one format; block shapes as midm_plan counts them. The other widths and
// the bias-less modes start at 33 rows (fewer take the few-row kernel).
template <int FMT>
hipError_t launch_fmt(const MidmParams& P, bool wide, hipStream_t s) {
  constexpr bool EX = FMT == 4 || FMT == 8;
  const int mt = (P.M + 31) / 32;
  if constexpr (EX)
    if (mt == 1)
      return wide ? launch_one<FMT, true, 1, 2, 4, 4>(P, s) : launch_one<FMT, true, 1, 1, 4, 4>(P, s);
  if (wide)
    return mt <= 2   ? launch_one<FMT, EX, 2, 2, 4, 4>(P, s)
           : mt == 3 ? launch_one<FMT, false, 3, 2, 4, 2>(P, s)
                     : launch_one<FMT, false, 4, 2, 4, 2>(P, s);
  return mt <= 2   ? launch_one<FMT, EX, 2, 1, 4, 4>(P, s)
         : mt == 3 ? launch_one<FMT, false, 3, 1, 4, 2>(P, s)
                   : launch_one<FMT, false, 4, 1, 4, 2>(P, s);
}

}  // namespace midm
}  // namespace mi
