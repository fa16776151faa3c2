// Grouped quantized GEMM over expert-sorted work items: the sorted gather_qmm of an MoE
// prefill (reference: the three gather_qmm(sorted_indices = true) calls over expert
// segments in src/transformer.zig:14961-15043, gather at :15011), 4-bit affine weights,
// group size 64, bf16 activations.
//
// A work item is a run of sorted pairs with one expert, cut at 32 or 64 rows (build_items in
// quant.hip). One block = one item x NS tiles of 128 weight rows of its expert (gate + up: 64
// of either): it streams those weights from HBM exactly once and multiplies them by all the
// item's rows.
//
// What bounds it: the weight stream (226 MB a gate + up call of 128 experts, [768,2048]) as far
// as the arithmetic keeps up: 3.0 TB/s, where a timing build with the loads alone reached 5.8. When
// each wave ran barrier, LDS reads, MFMAs and dequantize one after another, the matrix cores
// were busy 25% and the VALU 46%, at 2.7 TB/s.
//
// Block: 4 waves, three blocks a CU; wave w owns 32 weight rows (two 16-row tiles of
// v_mfma_f32_16x16x32_bf16) against MT 16-row tiles of x. An item that holds at most half of
// its rows runs as one of half the tiles. Weights, dequantized once as bf16(s*q + b), scales
// and biases come straight into registers, one 4-step unit ahead: one instruction reads 16
// rows x 64 contiguous bytes, two steps; one v_permlane32_swap per dword pair gives each lane
// two dwords of either step, the 8-value runs sb, sb + 1 of the step's eight (sb = 4 (q % 2) +
// 2 (q / 2) for quarter q = lane / 16). The gathered x rows come by LDS DMA into a ring of
// four stages (rows past the item's end read past the end of x: zeros, no memory traffic).
// One barrier a step, before its second k-step, whose MFMAs carry the LDS reads of the next
// step's first fragments; every MFMA group carries half of the next step's dequantize. Vector
// memory operations return in order, so "x stage t + 1 has arrived" is an exact vmcnt. A block
// with two passes runs them as one stream of steps, so the rings never drain.
//
// Measured, us a call, 4 bits, before -> after: gate + up of 128 experts [768,2048], top 8, 64
// tokens 84.5 -> 74.6, 512 tokens 100 -> 90; 256 experts [2048,7168], 512 tokens 1765 -> 1471;
// down projections [2048,768] 64 tokens 42.9 -> 37.9, 600 tokens 51.9 -> 51.6 (64 x rows held in
// LDS then), [2048,1536] (64 experts, top 6) 500 tokens 58 -> 50, [7168,2048] 690 -> 602.
#include <algorithm>

#include "dequant_bf16.h"
#include "mi_common.h"
#include "mi_internal.h"
#include "qmv_common.h"

namespace mi {
namespace {

using dq::dequant8;
using dq::pack_bf16x2;
using qmv_detail::decode_item;
using qmv_detail::Item;
using qmv_detail::item_x_row;
using qmv_detail::vmcnt_imm;

constexpr uint32_t kOOB = 0x7FFFFFF0u;  // past any x: the load returns 0, no traffic
constexpr int kRing = 4, kU = 4;         // LDS stages of x; steps of the unrolled unit
constexpr int kWaves = 4;
constexpr int kBufFlags = 0x00020000;

// 64 lanes x 16 bytes into 1 KB of LDS (lane order)
MI_DEV void dma16(__amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16,
                                           voff, soff, 0, 0);
}
MI_DEV f32x4_t mfma16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return mfma16x16x32(as_bf16x8(a), as_bf16x8(b), c);
}
// XOR swizzle of the 16-byte slots of a 128-byte x row: the lanes that one pass of a
// ds_read_b128 serves (rows 0-3 and 12-15 of quarter q, 4-11 of quarter q + 1) fall in
// distinct banks with the slots of `sb` below.
MI_DEV int xswz(int r) { return ((r & 2) << 1) | ((r >> 2) & 1) | ((r >> 2) & 2); }

MI_DEV float half_f(uint32_t d, bool up) {
  return __uint_as_float(up ? d & 0xFFFF0000u : d << 16);
}

// MODE 0: plain products. 1: y = SwiGLU(P.swiglu_gate, product). 2 (P.dual): the first two waves run the gate bank (w, scales, biases) and the others
// the up bank (w2, scales2, biases2) on the same rows of both and the same x tiles; the
// epilogue writes y = SwiGLU(gate, up) through LDS (each product rounded to bf16 first).
// One item of up to 16 * MT rows.
template <int MT, int MODE>
MI_DEV void gmm_item(const QmvParams& P, const Item& it, int NS, unsigned char* smem,
                     const int64_t* rowtab) {
  constexpr bool DUAL = MODE == 2, staged = MODE != 0;  // staged: results leave through LDS
  constexpr int kWT = DUAL ? kWaves / 2 : kWaves;  // waves per weight bank
  constexpr int R = 16 * MT, kNT = 32 * kWT, kThreads = 64 * kWaves;
  constexpr int XI = MT / 2;  // x DMA instructions of a wave per step
  constexpr int kStage = R * 128;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, q = lane >> 4;
  const int N = P.N, K = P.K, G = K / 64, nsteps = K / 64;
  const int slice0 = blockIdx.x * kNT * NS;
  const int npass = min(NS, (N - slice0 + kNT - 1) / kNT), total = npass * nsteps;
  const int mw = DUAL ? wave % kWT : wave;  // the wave's 32 rows in its bank
  const bool up = DUAL && wave >= kWT;       // wave-uniform
  const int sb = 4 * (q & 1) + 2 * (q >> 1);
  const uint32_t rowb = (uint32_t)K / 2;
  const uint32_t xrec = (uint32_t)(P.x_batch * P.M * (int64_t)K * 2);

  const uint32_t e = __builtin_amdgcn_readfirstlane(it.expert_ok ? it.expert : 0u);
  const bool eok = it.expert_ok;
  // acc[a][i] register r is D[n = 32 mw + 16 a + 4 q + r][m = 16 i + fr]
  f32x4_t acc[2][MT];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[a][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  auto store = [&](int p) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = 16 * i + fr;
      const int64_t ro = rowtab[m];
      if (ro == -1) continue;
      const int64_t pos = it.pos0 + m;
      const bool nan = ro == -2 || !eok;
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int n = slice0 + p * kNT + 32 * mw + 16 * a + 4 * q;
        if (n >= N) continue;
        u32x2_t o = {pack_bf16x2(acc[a][i][0], acc[a][i][1]),
                     pack_bf16x2(acc[a][i][2], acc[a][i][3])};
        if (nan) o = u32x2_t{0x7FC07FC0u, 0x7FC07FC0u};
        *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(P.y) + pos * N + n) = o;
      }
    }
  };
  if (!eok) {
    if (!staged)
      for (int p = 0; p < npass; ++p) store(p);
  } else {
    const size_t mat = (size_t)e * (uint32_t)N;
    const unsigned char* wb = (const unsigned char*)(up ? P.w2 : P.w) + mat * rowb;
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((up ? P.scales2 : P.scales) + mat * (uint32_t)G), (short)0, N * G * 2, kBufFlags);
    const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((up ? P.biases2 : P.biases) + mat * (uint32_t)G), (short)0, N * G * 2, kBufFlags);
    // x: instruction j of wave w moves rows 8 (XI w + j) .. +7. Rows outside the item read
    // past the end of x (zeros, no memory traffic).
    uint32_t xo[XI];
#pragma unroll
    for (int j = 0; j < XI; ++j) {
      const int r = 8 * (XI * wave + j) + (lane >> 3), c = (lane & 7) ^ xswz(r);
      const int64_t ro = rowtab[r];
      xo[j] = ro >= 0 ? (uint32_t)ro * 2u + 16u * c : kOOB;
    }
    // flat steps 0 .. total - 1, pass p = step / nsteps (a unit lies in one pass)
    auto load_w = [&](int p, int t, bool in, int a, u32x4_t& d) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)wb, (short)0, in ? N * rowb : 0u, kBufFlags);
      const uint32_t r = (uint32_t)min(slice0 + p * kNT + 32 * mw + 16 * a + fr, N - 1);
      d = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, r * rowb + 16 * q, t * 32, 0));
    };
    auto load_x = [&](int t, bool in, int slot, int j) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)P.x, (short)0, in ? xrec : 0u, kBufFlags);
      dma16(rs, smem + slot * kStage + (wave * XI + j) * 1024, xo[j], t * 128);
    };
    u32x2_t ts[2], tb[2], sd[2], bd[2];
    auto load_s = [&](int p, int t) __attribute__((always_inline)) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const uint32_t r = (uint32_t)min(slice0 + p * kNT + 32 * mw + 16 * a + fr, N - 1);
        ts[a] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(sres, r * G * 2, t * 2, 0));
        tb[a] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(bres, r * G * 2, t * 2, 0));
      }
    };
    u32x4_t W[2][2];  // chunk of two steps, row tile
    // a chunk's dwords to step order: {even step: 2, odd step: 2}
    auto prep_w = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        u32x4_t& v = W[c][a];
        const auto x = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
        v = u32x4_t{x[0], y[0], x[1], y[1]};
      }
    };
    auto dq_w = [&](int t, int a, int k) __attribute__((always_inline)) {
      return dequant8(W[(t / 2) % 2][a][2 * (t % 2) + k], half_f(sd[a][t / 2], t % 2),
                      half_f(bd[a][t / 2], t % 2));
    };
    auto xfrag = [&](int t, int i, int k) -> u32x4_t {
      return *reinterpret_cast<const u32x4_t*>(smem + (t % kRing) * kStage + (16 * i + fr) * 128 +
                                               (((sb + k) ^ xswz(fr)) << 4));
    };
    // Prologue in the order that the loop's wait counts: the second chunk comes after the
    // first half of stage 1, as in the loop's step -1.
    load_s(0, 0);
#pragma unroll
    for (int a = 0; a < 2; ++a) load_w(0, 0, true, a, W[0][a]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < XI; ++j) load_x(t, true, t, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < 2; ++a) load_w(0, 2, true, a, W[1][a]);
    __builtin_amdgcn_sched_barrier(0);
    load_x(2, true, 2, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(XI + 2 + 1));  // stage 0 has landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    u32x4_t X[2][MT], A[2][2][2];  // fragments of a k-step; operands of this step and the next
#pragma unroll
    for (int i = 0; i < MT; ++i) X[0][i] = xfrag(0, i, 0);
#pragma unroll
    for (int a = 0; a < 2; ++a) sd[a] = ts[a], bd[a] = tb[a];
    prep_w(0);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int k = 0; k < 2; ++k) A[0][a][k] = dq_w(0, a, k);
    int pass = 0, tc = 0;  // of the unit
#pragma unroll 1
    for (int t0 = 0; t0 < total; t0 += kU) {
      const bool wrap = tc + kU == nsteps, in = t0 + kU < total;
      const int pn = in && wrap ? pass + 1 : pass, tn0 = wrap ? 0 : tc + kU;  // next unit
#pragma unroll
      for (int t = 0; t < kU; ++t) {
        const int tn = t + 1;
        if (tn == kU) {
#pragma unroll
          for (int a = 0; a < 2; ++a) sd[a] = ts[a], bd[a] = tb[a];
        }
        if (tn % 2 == 0) prep_w((tn / 2) % 2);
        auto stage = [&](int st, int j) __attribute__((always_inline)) {
          if (st < kU)
            load_x(tc + st, true, st % kRing, j);
          else
            load_x(tn0 + st - kU, in, st % kRing, j);
        };
        // two groups, one k-step each
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if (u == 1) {
            // this wave's part of x stage t + 1 is in: younger are the x DMA since (XI),
            // two weight loads every second step and four scale loads every fourth
            if (t < 2)
              __builtin_amdgcn_s_waitcnt(vmcnt_imm(XI + 6));
            else
              __builtin_amdgcn_s_waitcnt(vmcnt_imm(XI + 2));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            stage(t + 3, 0);  // slot of stage t - 1: every wave is past its last read
          } else {
            if constexpr (XI > 1) stage(t + 2, 1);
            __builtin_amdgcn_sched_barrier(0);
            if (t == 0) load_s(pn, tn0);
            if (t % 2 == 1) {
#pragma unroll
              for (int a = 0; a < 2; ++a) load_w(pn, tn0 + t - 1, in, a, W[t / 2][a]);
            }
          }
#pragma unroll
          for (int i = 0; i < MT; ++i) X[(u + 1) & 1][i] = xfrag(u ? tn : t, i, (u + 1) & 1);
#pragma unroll
          for (int a = 0; a < 2; ++a) A[tn & 1][a][u] = dq_w(tn % kU, a, u);
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int a = 0; a < 2; ++a) acc[a][i] = mfma16(A[t & 1][a][u], X[u][i], acc[a][i]);
#pragma unroll
          for (int m = 0; m < 2 * MT; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (m % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 48 / (2 * MT), 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (wrap && !staged) {
        store(pass);
        clear();
      }
      pass = pn;
      tc = tn0;
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // no DMA may outlive its stage
  }
  const int n0 = slice0;

  // results through LDS (the x ring's memory), then every thread takes 4 adjacent outputs of
  // a row: coalesced gate reads and output writes
  if constexpr (staged) {
    // DUAL: gate products in columns [0, kNT), up products in [kNT, 2 kNT); row stride
    // padded by 4 halves
    constexpr int kTS = (DUAL ? 2 : 1) * kNT + 4;
    uint16_t* tile = reinterpret_cast<uint16_t*>(smem);
    __syncthreads();  // every wave is done reading the x ring
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int a = 0; a < 2; ++a)
        *reinterpret_cast<u32x2_t*>(tile + (16 * i + fr) * kTS + (up ? kNT : 0) + 32 * mw + 16 * a +
                                    4 * q) =
            u32x2_t{pack_bf16x2(acc[a][i][0], acc[a][i][1]), pack_bf16x2(acc[a][i][2], acc[a][i][3])};
    __syncthreads();
    constexpr int kPerRow = kNT / 4, kRowsPerPass = kThreads / kPerRow;
    const int c4 = tid % kPerRow;
    const int n = n0 + 4 * c4;
#pragma unroll 1
    for (int m = tid / kPerRow; m < R; m += kRowsPerPass) {
      const int64_t ro = rowtab[m];
      if (ro == -1 || n >= N) continue;
      const int64_t pos = it.pos0 + m;
      u32x2_t pv = *reinterpret_cast<const u32x2_t*>(tile + m * kTS + 4 * c4), gv = pv;
      if constexpr (DUAL)
        pv = *reinterpret_cast<const u32x2_t*>(tile + m * kTS + kNT + 4 * c4);
      else
        gv = *reinterpret_cast<const u32x2_t*>(P.swiglu_gate + pos * N + n);
      if (ro == -2 || !eok) {  // NaN rows
        pv.x = pv.y = 0x7FC07FC0u;
        if constexpr (DUAL) gv = pv;
      }
      uint32_t o[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const uint32_t lo = swiglu_bf16((uint16_t)(gv[d] & 0xFFFFu), (uint16_t)(pv[d] & 0xFFFFu));
        const uint32_t hi = swiglu_bf16((uint16_t)(gv[d] >> 16), (uint16_t)(pv[d] >> 16));
        o[d] = lo | (hi << 16);
      }
      *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(P.y) + pos * N + n) = u32x2_t{o[0], o[1]};
    }
  }
  __syncthreads();  // the row table and the x ring are reused by the next item
}

// Items of 16 * MT rows; one that holds at most half of them runs as such.
template <int MT, int MODE>
__global__ void __launch_bounds__(64 * kWaves, 3) gmm_kernel(QmvParams P, int NS) {
  // Dynamic LDS: the x ring, then the row table. (With a static array the compiler would
  // drain every load before each LDS read that may alias an LDS DMA; the waits here are
  // exact and explicit.)
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int64_t* rowtab = reinterpret_cast<int64_t*>(smem + kRing * 16 * MT * 128);
  const int n_items = (int)*P.item_count;
  for (int it_i = blockIdx.y; it_i < n_items; it_i += gridDim.y) {
    const Item it = decode_item(P, it_i);
    if (it.cnt <= 0) continue;  // block-uniform
    if (threadIdx.x < 16 * MT) rowtab[threadIdx.x] = item_x_row(P, it, threadIdx.x);  // -1 skip, -2 NaN
    __syncthreads();
    // (a run's rows come first: the item ends where its expert does)
    if (MT > 2 && __builtin_amdgcn_readfirstlane((int)rowtab[8 * MT]) == -1)
      gmm_item<MT == 2 ? 2 : MT / 2, MODE>(P, it, NS, smem, rowtab);
    else
      gmm_item<MT, MODE>(P, it, NS, smem, rowtab);
  }
}

}  // namespace

bool gmm_supported(int64_t N, int64_t K, int bits, int gs, int x_f32, int64_t x_bytes) {
  // whole 64-wide steps; scale chunks of 4 groups on an 8-byte boundary; 4-output stores;
  // 32-bit buffer offsets
  return bits == 4 && gs == 64 && !x_f32 && K % 256 == 0 && N % 4 == 0 && N >= 4 &&
         N * (K / 2) < ((int64_t)1 << 31) && x_bytes + 2 * K < ((int64_t)1 << 31);
}

template <int MT, int MODE>
hipError_t launch_mt(const QmvParams& P, int ns, int grid_items, hipStream_t s) {
  constexpr size_t lds = (size_t)kRing * 16 * MT * 128 + 16 * MT * sizeof(int64_t);
  constexpr int kNT = 32 * (MODE == 2 ? kWaves / 2 : kWaves);
  const dim3 grid((unsigned)((P.N + kNT * ns - 1) / (kNT * ns)), (unsigned)std::max(1, grid_items));
  hipLaunchKernelGGL((gmm_kernel<MT, MODE>), grid, dim3(64 * kWaves), lds, s, P, ns);
  return hipGetLastError();
}

hipError_t launch_gmm(const QmvParams& P, int mt, double items, int grid_items, hipStream_t s) {
  if (!P.items || !P.item_count) return hipErrorInvalidValue;
  if (P.dual && (!P.w2 || !P.scales2 || !P.biases2)) return hipErrorInvalidValue;
  const int mode = P.dual ? 2 : P.swiglu_gate ? 1 : 0;
  // Passes of a block: one, since more blocks than a round (three a CU) even out items of
  // different rows. us a call, as many passes as one round takes (2 or 3) -> 1: [2048,768] of 128
  // experts, 500 tokens 52.9 -> 47.3, 900 tokens 87.0 -> 61.1; [2048,1536] of 64, 600 tokens 69.3
  // -> 54.6; [1536,2048] of 64, 500 tokens 51.9 -> 46.2. Two where one leaves a second round with
  // few blocks: [1536,2048] of 64 experts, 600 tokens (1.14 rounds) 59.0 -> 54.7, of K = 1024 39.3
  // -> 37.9, 4096 123 -> 106; [768,2048] of 128, 950 tokens (1.25) 67.3 -> 61.1. At 1.33 rounds one
  // pass is ahead again ([2048,1536] of 64, 450 tokens 47.2 against 52.6; 1.74 rounds 10-30%).
  const double rounds = (double)((P.N + 127) / 128) * items / 768.0;
  const int ns = mode == 0 && rounds > 1.03 && rounds < 1.33 ? 2 : 1;
  switch (mt * 4 + mode) {
    case 4: return launch_mt<2, 0>(P, ns, grid_items, s);
    case 5: return launch_mt<2, 1>(P, 1, grid_items, s);
    case 6: return launch_mt<2, 2>(P, 1, grid_items, s);
    case 8: return launch_mt<4, 0>(P, ns, grid_items, s);
    case 9: return launch_mt<4, 1>(P, 1, grid_items, s);
    case 10: return launch_mt<4, 2>(P, 1, grid_items, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mi
