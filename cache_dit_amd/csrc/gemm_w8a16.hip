// Weight-only FP8 GEMM (w8a16) for gfx950: bf16 activations x e4m3 weights,
// the weights dequantized to bf16 inside the mainloop, fp32 accumulate,
// per-output-channel scale + bias + optional GELU-tanh + bf16 in the epilogue.
//
//   out[m,n] = epi((sum_k x[m,k] float(b[n,k])) * b_scale[n] + bias[n])
//
// Every e4m3 value is exactly representable in bf16, so the in-loop conversion
// (v_cvt_scalef32_pk_bf16_fp8 with scale 1) is lossless and the weight never
// exists in HBM at 16 bits: B costs 1 byte per element of traffic instead of
// the 1 (read) + 2 (write) + 2 (read) of dequantize-then-GEMM.
//
// MFMA: v_mfma_f32_32x32x16_bf16; per lane 8 consecutive K elements of row
// (lane&31), K-group h = lane>>5. The K order inside a 32-element block is
// free as long as A and B agree, so lane group h takes elements [16h, 16h+16)
// of the block: one 16-byte read of B (two MFMA steps of 8 bytes) and one
// 32-byte read of A.
//
// Tile: BM x BN outputs, BK = 64 elements per pipeline step: A panel rows are
// 128 bytes (8 chunks, chunk c of row r at position c ^ ((r>>1)&7)), B panel
// rows are 64 bytes (4 chunks, chunk c of row r at position c ^ ((r>>2)&3)):
// with 64 LDS banks of 4 B and 16 lanes served per pass, both are conflict free
// for the 16-byte operand reads. Panels
// are staged with 128-bit LDS-DMA loads, double buffered.
//
// Replaces F.linear(x, W.dequantize(), bias) of the reference's
// float8_weight_only mode (src/cache_dit/quantization/torchao/quantize_ao.py:604-610).
#include <type_traits>

#include "gemm_common.h"
#include "quant_device.h"

namespace cdit {
namespace {

constexpr int BKE = 64;  // K elements per pipeline step

template <int BM_, int BN_, int WGM_, int WGN_, bool EPI_LDS_, int GROUP_M_>
struct CfgW {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
  static constexpr bool EPI_LDS = EPI_LDS_;
  static constexpr int GROUP_M = GROUP_M_;
  static constexpr int WAVES = WGM * WGN;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int WM = BM / WGM, WN = BN / WGN;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int A_ROW = BKE * 2, B_ROW = BKE;  // bytes per panel row
  static constexpr int A_BYTES = BM * A_ROW, B_BYTES = BN * B_ROW;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int EPI_PITCH = WN * 2 + 16;
  static constexpr int EPI_BYTES = EPI_LDS ? WAVES * 32 * EPI_PITCH : 0;
  static constexpr int LDS_BYTES = (2 * STAGE_BYTES > EPI_BYTES) ? 2 * STAGE_BYTES : EPI_BYTES;
  // LDS-DMA instructions per wave and stage (1 KiB each)
  static constexpr int A_DMA = A_BYTES / 1024 / WAVES, B_DMA = B_BYTES / 1024 / WAVES;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be a multiple of 32x32");
  static_assert(A_BYTES % (1024 * WAVES) == 0 && B_BYTES % (1024 * WAVES) == 0,
                "panel/waves mismatch");
};

template <class C>
__global__ __launch_bounds__(C::THREADS) void gemm_w8a16_tiled(GemmArgs g, int tiles_m,
                                                               int tiles_n) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C::WGN, wn = wave % C::WGN;

  int tm, tn;
  tile_of_block<C::GROUP_M>(blockIdx.x, gridDim.x, tiles_m, tiles_n, &tm, &tn);
  const int m0 = tm * C::BM, n0 = tn * C::BN;
  const uint8_t* __restrict__ A =
      static_cast<const uint8_t*>(g.a) + (int64_t)m0 * g.lda * 2;  // bf16: 2 bytes/element
  const uint8_t* __restrict__ B = g.b + (int64_t)n0 * g.ldb;
  const int rows_a = g.M - m0, rows_b = g.N - n0;

  // ---- LDS-DMA maps: a wave instruction fills 1 KiB = 8 A rows or 16 B rows;
  // lane l lands on (row l/8, position l%8) resp. (row l/4, position l%4) and
  // fetches the logical chunk that the swizzle puts there.
  uint32_t a_off[C::A_DMA], b_off[C::B_DMA];
#pragma unroll
  for (int p = 0; p < C::A_DMA; ++p) {
    const int row = (wave * C::A_DMA + p) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    a_off[p] = (uint32_t)min(row, rows_a - 1) * (uint32_t)(g.lda * 2) + c * 16;
  }
#pragma unroll
  for (int p = 0; p < C::B_DMA; ++p) {
    const int row = (wave * C::B_DMA + p) * 16 + (lane >> 2);
    const int c = (lane & 3) ^ ((row >> 2) & 3);
    b_off[p] = (uint32_t)min(row, rows_b - 1) * (uint32_t)g.ldb + c * 16;
  }

  // ---- operand read maps; kb = 32-element K block inside the step (0..1)
  const int h = lane >> 5;
  uint32_t rd_a[2][2], rd_b[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const int ra_row = wm * C::WM + (lane & 31);
#pragma unroll
    for (int e = 0; e < 2; ++e)
      rd_a[kb][e] = ra_row * C::A_ROW + (((4 * kb + 2 * h + e) ^ ((lane >> 1) & 7)) << 4);
    const int rb_row = wn * C::WN + (lane & 31);
    rd_b[kb] = C::A_BYTES + rb_row * C::B_ROW + (((2 * kb + h) ^ ((lane >> 2) & 3)) << 4);
  }

  v16f acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int KT = g.K / BKE;

  auto fetch = [&](int kt, int stage) {
    const uint8_t* Ak = A + (int64_t)kt * C::A_ROW;
    const uint8_t* Bk = B + (int64_t)kt * C::B_ROW;
    uint8_t* st = smem + stage * C::STAGE_BYTES;
#pragma unroll
    for (int p = 0; p < C::A_DMA; ++p)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(Ak + a_off[p]),
          (__attribute__((address_space(3))) void*)(st + (wave * C::A_DMA + p) * 1024), 16, 0, 0);
#pragma unroll
    for (int p = 0; p < C::B_DMA; ++p)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(Bk + b_off[p]),
          (__attribute__((address_space(3))) void*)(st + C::A_BYTES +
                                                    (wave * C::B_DMA + p) * 1024),
          16, 0, 0);
  };

  auto compute = [&](int stage) {
    const uint8_t* st = smem + stage * C::STAGE_BYTES;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      v8bf a_lo[C::TM], a_hi[C::TM];  // MFMA steps 0 and 1 of this block
#pragma unroll
      for (int i = 0; i < C::TM; ++i) {
        a_lo[i] = *reinterpret_cast<const v8bf*>(st + rd_a[kb][0] + i * 32 * C::A_ROW);
        a_hi[i] = *reinterpret_cast<const v8bf*>(st + rd_a[kb][1] + i * 32 * C::A_ROW);
      }
#pragma unroll
      for (int j = 0; j < C::TN; ++j) {
        const uint4 w = *reinterpret_cast<const uint4*>(st + rd_b[kb] + j * 32 * C::B_ROW);
        // 16 e4m3 bytes -> 16 bf16 (exact), two at a time
        v2bf c0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.x, 1.0f, false);
        v2bf c1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.x, 1.0f, true);
        v2bf c2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.y, 1.0f, false);
        v2bf c3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.y, 1.0f, true);
        v2bf c4 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.z, 1.0f, false);
        v2bf c5 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.z, 1.0f, true);
        v2bf c6 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.w, 1.0f, false);
        v2bf c7 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.w, 1.0f, true);
        const v8bf b_lo = {c0[0], c0[1], c1[0], c1[1], c2[0], c2[1], c3[0], c3[1]};
        const v8bf b_hi = {c4[0], c4[1], c5[0], c5[1], c6[0], c6[1], c7[0], c7[1]};
#pragma unroll
        for (int i = 0; i < C::TM; ++i) {
          // operands swapped: result rows follow B (n), result columns follow A (m)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b_lo, a_lo[i], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b_hi, a_hi[i], acc[i][j], 0, 0, 0);
        }
      }
    }
  };

  fetch(0, 0);
  for (int kt = 0; kt < KT; ++kt) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of step kt is in LDS
    __syncthreads();                     // ... and everyone's; stage (kt+1)&1 is free again
    if (kt + 1 < KT) fetch(kt + 1, (kt + 1) & 1);
    compute(kt & 1);
  }

  if constexpr (C::EPI_LDS) __syncthreads();  // all waves are done with the stage buffers
  tile_epilogue<C>(acc, g, smem + wave * (32 * C::EPI_PITCH), m0, n0, wm, wn, lane);
}

// ---------------------------------------------------------------------------
// Wide kernel: the schedule of the wide w8a8 kernel (one persistent workgroup of 4
// waves per CU, one wave per SIMD with all 256 AGPRs as accumulators, LDS-DMA by
// buffer loads spread over the MFMA stream DEPTH steps ahead, A panel in DEPTH + 1 LDS
// stages and B panel in DEPTH, one barrier per K step, the DMA stream running across
// tiles) with bf16 MFMAs:
// v_mfma_f32_32x32x16_bf16 (8 passes), K steps of 64 elements, wave tile
// (BM/2) x (BN/2) as TM x TN blocks of 32x32, four MFMAs per block and step.
//
// Panels: A rows 128 B (bf16), chunk c of row r at c ^ ((r>>1)&7); B rows 64 B
// (e4m3), chunk c at c ^ ((r>>2)&3). A lane reads, per 32-row block, the four A
// chunks 4t+2h+s (h = lane>>5) and the two B chunks 2t+h: the 16 B bytes of one
// chunk are the weights of MFMA steps 2t and 2t+1 (K order permuted identically on
// both sides). The weights are converted to bf16 once per step, two conversion
// instructions (half an operand) at a time on a compile-time schedule that ends two
// MFMAs ahead of the first use, and kept for all row blocks.
//
// The B fragments take their 32 rows in a permuted order, operand row p reads
// panel row 16 ((p>>2)&1) + 4 (p>>3) + (p&3) of its block: with the operands
// swapped (weights first) a lane then ends with 16 consecutive output columns per
// block, n = 32j + 16h + r for accumulator register r, and stores them with two
// 16-byte stores, no transpose.
template <int BM_, int BN_, int GROUP_M_, int DEPTH_ = 2>
struct CfgWW {
  static constexpr int BM = BM_, BN = BN_, GROUP_M = GROUP_M_;
  // K steps the DMA stream runs ahead of the MFMAs (A panel in DEPTH + 1 LDS stages,
  // B panel in DEPTH): 2 for the large tiles, more for small tiles with short steps
  static constexpr int DEPTH = DEPTH_;
  static constexpr int WAVES = 4, THREADS = 256;
  static constexpr int WM = BM / 2, WN = BN / 2;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int H = TM / 2;
  static constexpr int A_ROW = BKE * 2, B_ROW = BKE;
  static constexpr int A_BYTES = BM * A_ROW, B_BYTES = BN * B_ROW;
  static constexpr int A_STAGES = DEPTH + 1, B_STAGES = DEPTH;
  static constexpr int B_BASE = A_STAGES * A_BYTES;
  static constexpr int PANEL_BYTES = A_STAGES * A_BYTES + B_STAGES * B_BYTES;
  // b_scale and bias of a tile's BN columns are staged behind the panels (1 KiB each)
  static constexpr int EPI_BS = PANEL_BYTES, EPI_BI = PANEL_BYTES + 1024;
  static constexpr int LDS_BYTES = PANEL_BYTES + 2048;
  static_assert(BN * 4 <= 1024, "one LDS-DMA instruction per staged operand");
  // DMA instructions (1 KiB: 8 A rows or 16 B rows) per wave and step
  static constexpr int NDA = BM / 8 / WAVES, NDB = BN / 16 / WAVES, ND = NDA + NDB;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be a multiple of 32x32");
  static_assert(BM % 32 == 0 && BN % 64 == 0, "panels are dealt 1 KiB x 4 waves at a time");
  static_assert(TM * TN <= 16, "accumulators: at most 256 registers");
  static_assert(TM >= 2, "two halves per step");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
  static_assert(DEPTH >= 2 && (DEPTH - 2) * ND + NDA < 63, "DMA instructions in flight: vmcnt has 6 bits");

  // Issue schedule of a K step. Between two MFMAs (8 passes, 32 cycles) the wave issues
  // in order; one LDS read or DMA instruction and two conversions (8 cycles each) fit,
  // more delays the next MFMA, and the matrix core never makes that up. So everything is
  // spread: all slot numbers below are compile-time constants.
  //
  // First half: S1 MFMAs over the rows 0..H-1, MFMA step q of all their blocks before step
  // q+1: slot s = (q*H + i)*TN + j. A new weight operand (j, q) is then needed every
  // H slots only, which leaves room to convert it in pieces (below). Items: the
  // 4 (TM-1) single LDS reads of the fragments A_1 .. A_{TM-1} in the order of their first
  // use, and the NDA DMA instructions of the A panel, merged evenly, a read first, and
  // spread evenly over the slots.
  static constexpr int S1 = H * 4 * TN, NR1 = 4 * (TM - 1), T1 = NR1 + NDA;
  static constexpr int R = TM - H, S2 = R * 4 * TN, NR2 = 4 + 2 * TN;
  static constexpr int i_of_slot1(int s) { return s / TN % H; }
  static constexpr int q_of_slot1(int s) { return s / (H * TN); }
  // first use of A_i, MFMA step q, counted in slots from the start of the step
  static constexpr int use_a(int i, int q) {
    return i < H ? (q * H + i) * TN : S1 + (q * R + i - H) * TN;
  }
  static constexpr int H1 = H > 1 ? H - 1 : 1;
  static constexpr int read1_row(int r) {  // read r of the first half: fragment A_i ...
    return r < 4 * (H - 1) ? 1 + r % H1 : H + (r - 4 * (H - 1)) % R;
  }
  static constexpr int read1_step(int r) {  // ... MFMA step q
    return r < 4 * (H - 1) ? r / H1 : (r - 4 * (H - 1)) / R;
  }
  static constexpr int item_of_read1(int r) { return r * T1 / NR1; }
  static constexpr bool is_read1(int t) {
    for (int r = 0; r < NR1; ++r)
      if (item_of_read1(r) == t) return true;
    return false;
  }
  static constexpr int read1_index(int t) {  // reads before item t
    int n = 0;
    for (int r = 0; r < NR1; ++r) n += item_of_read1(r) < t;
    return n;
  }
  static constexpr int dma1_index(int t) { return t - read1_index(t); }
  static constexpr int slot1(int t) { return t * S1 / T1; }
  static constexpr bool first_half_reads_in_time() {
    for (int r = 0; r < NR1; ++r)
      if (slot1(item_of_read1(r)) + 3 > use_a(read1_row(r), read1_step(r))) return false;
    return true;
  }
  static_assert(first_half_reads_in_time(), "A fragment read too late for its first use");
  // Second half: S2 MFMAs over the rows H..TM-1 in the same order, slot s =
  // (q*R + i-H)*TN + j. The LDS reads of the next step (its raw weights, 2 per column, and
  // A_0, 4) are spread evenly over the slots from 1 on: first halves of the weights, A_0 of
  // MFMA step 0, second halves, rest of A_0. The NDB DMA instructions of the B panel go in
  // the middle of their share of the slots.
  static constexpr int key_w(int j, int t) { return t == 0 ? j : TN + 1 + j; }
  static constexpr int key_a0(int q) { return q == 0 ? TN : 2 * TN + 1 + q; }
  static constexpr int rank2(int key) {  // reads of the second half with a smaller key
    int n = 0;
    for (int j = 0; j < TN; ++j)
      for (int t = 0; t < 2; ++t) n += key_w(j, t) < key;
    for (int q = 0; q < 4; ++q) n += key_a0(q) < key;
    return n;
  }
  static constexpr int slot2(int key) { return 1 + rank2(key) * (S2 - 1) / NR2; }
  static constexpr int slot_w(int j, int t) { return slot2(key_w(j, t)); }  // read t (0/1) of column j
  static constexpr int slot_a0(int q) { return slot2(key_a0(q)); }
  // Conversions. Weight operand (j, q) (8 e4m3 bytes -> 8 bf16, four conversion
  // instructions) is converted as two half operands. Time t counts first-half slots of the
  // step the operand belongs to; t < 0 is second-half slot S2 + t of the step before (the
  // raw weights of a step are read during the step before it). A half operand must be
  // converted in front of slot use - CONVERT_AHEAD at the latest (an MFMA operand written
  // by a VALU instruction just before the inline-assembly MFMA reads stale data), and not
  // before the registers it goes to have been read for the last time (plus one MFMA) and
  // the LDS read it comes from has had three slots to land. Operands are placed latest
  // deadline first, each half in the latest slot with room for it; the smallest number of
  // half operands per slot that works is taken. Tiles too small for any of that convert
  // each operand whole in front of slot use - CONVERT_AHEAD, the first ones at the top of
  // the step (kConvTop).
  static constexpr int CONVERT_AHEAD = 2;
  static constexpr int kConvTop = -1000;
  static constexpr bool PIN_CONVERT = TM * TN >= 12;  // see convert_half() in the kernel
  static constexpr int last_use2(int j, int q) { return (q * R + R - 1) * TN + j; }
  static constexpr int conv_deadline(int j, int q) { return q * H * TN + j - CONVERT_AHEAD; }
  static constexpr int conv_release(int j, int q) {
    const int a = last_use2(j, q) + 2, b = slot_w(j, q >> 1) + 3;
    return (a > b ? a : b) - S2;
  }
  struct ConvSched {
    int t[TN][4][2];
    bool ok;
  };
  static constexpr ConvSched conv_sched_with(int cap) {
    ConvSched c{};
    c.ok = true;
    int load[S1 + S2] = {};  // half operands in slot t, at index t + S2
    for (int o = 4 * TN - 1; o >= 0; --o) {
      const int q = o / TN, j = o % TN;
      for (int h = 1; h >= 0; --h) {
        int t = conv_deadline(j, q);
        while (t >= conv_release(j, q) && load[t + S2] >= cap) --t;
        if (t < conv_release(j, q)) {
          c.ok = false;
          return c;
        }
        ++load[t + S2];
        c.t[j][q][h] = t;
      }
    }
    return c;
  }
  static constexpr ConvSched conv_sched() {
    for (int cap = 1; cap <= 2; ++cap) {
      const ConvSched c = conv_sched_with(cap);
      if (c.ok) return c;
    }
    ConvSched c{};
    c.ok = true;
    for (int j = 0; j < TN; ++j)
      for (int q = 0; q < 4; ++q)
        for (int h = 0; h < 2; ++h)
          c.t[j][q][h] = conv_deadline(j, q) < 0 ? kConvTop : conv_deadline(j, q);
    return c;
  }
  static constexpr ConvSched CONV = conv_sched();
  static constexpr int slot_dma2(int p) { return (2 * p + 1) * S2 / (2 * NDB); }
};

struct AFrag {
  v8bf k[4];  // operands of MFMA steps 0..3 of a K step (one 32-row block)
};
struct WRaw {
  uint4 t[2];  // weights as read from LDS: 2 x 16 e4m3 bytes
};

// acc (+)= W-fragment x A-fragment, accumulator tied to an AGPR tuple (see the wide
// w8a8 kernel for why this is inline assembly and what that obliges the code to do).
template <bool FIRST>
__device__ __forceinline__ void mfma_32x32x16_bf16(v16f& acc, const v8bf& w, const v8bf& a) {
  if constexpr (FIRST) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(w), "v"(a));
  } else {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(a));
  }
}

struct NoGroup {};

// GROUPED: the launch walks the tiles of a GemmGroup as one tile stream, as the w8a8
// kernel's grouped form does (gemm_fp8.hip): sibling Linears on one activation are members
// stacked along N, the Linears of the same stage on other activations follow; every member
// has its own weight, scale, bias, output and epilogue flag, K and the row strides are
// common (the B-side fields of `g` and grp.a_scale are unused). The instances without it are
// unchanged by its existence.
// KTAIL: K is any multiple of 16, as in the w8a8 kernel: the 16-byte chunks of a panel row
// beyond K go to an offset beyond the DMA descriptor, for which zeros land in the LDS, and a
// K shorter than the prefetch depth is padded with steps of zeros. The chunk a lane fetches
// is the same for every DMA instruction of a panel.
template <class C, bool GROUPED = false, bool KTAIL = false>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void
gemm_w8a16_wide(GemmArgs g, int tiles_m, int tiles_n,
                std::conditional_t<GROUPED, GemmGroup, NoGroup> grp) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: M0 from scalar code
  const int wm = wave >> 1, wn = wave & 1;
  // local copies: a template-dependent expression as a builtin argument inside a
  // lambda makes the host pass drop the kernel stub without a diagnostic
  constexpr int TM = C::TM, TN = C::TN, H = C::H, A_ROW = C::A_ROW, B_ROW = C::B_ROW;
  constexpr int D = C::DEPTH;
  // >= max(D, 3) (checked by the launcher, or padded here)
  const int KT = KTAIL ? max((g.K + BKE - 1) / BKE, D > 3 ? D : 3) : g.K / BKE;
  int ntiles = tiles_m * tiles_n;
  if constexpr (GROUPED) ntiles = grp.tile_begin[grp.acts];

  // Where a tile lives: for a batch, activation and member are looked up from the linear
  // tile id (the table sits in the kernel arguments: scalar loads with uniform indices).
  struct Where {
    int act, member, m0, n0;
  };
  auto locate = [&](int t) -> Where {
    Where w;
    if constexpr (GROUPED) {
      constexpr int kXcd = 8;
      int id = t;  // ids that run on one XCD are made consecutive, as tile_of_block does
      if (ntiles % kXcd == 0) id = (t % kXcd) * (ntiles / kXcd) + t / kXcd;
      int s = 0;
#pragma unroll
      for (int i = 1; i < kMaxActs; ++i)
        if (i < grp.acts && id >= grp.tile_begin[i]) s = i;
      int tm, tn;
      tile_of_linear<C::GROUP_M>(id - grp.tile_begin[s], grp.tiles_m[s], grp.tiles_n[s], &tm, &tn);
      int p = grp.first_member[s];
      const int p_end = grp.first_member[s + 1];
#pragma unroll
      for (int i = 1; i < kMaxGroup; ++i)
        if (i > p && i < p_end && tn >= grp.col_begin[i]) p = i;
      w.act = s;
      w.member = p;
      w.m0 = tm * C::BM;
      w.n0 = (tn - grp.col_begin[p]) * C::BN;
    } else {
      int tm, tn;
      tile_of_block<C::GROUP_M>(t, ntiles, tiles_m, tiles_n, &tm, &tn);
      w.act = 0;
      w.member = 0;
      w.m0 = tm * C::BM;
      w.n0 = tn * C::BN;
    }
    return w;
  };
  auto a_of = [&](int s) -> const uint8_t* {
    if constexpr (GROUPED) return static_cast<const uint8_t*>(grp.a[s]);
    return static_cast<const uint8_t*>(g.a);
  };
  auto m_of = [&](int s) -> int {
    if constexpr (GROUPED) return grp.M[s];
    return g.M;
  };
  auto b_of = [&](int p) -> const uint8_t* {
    if constexpr (GROUPED) return grp.b[p];
    return g.b;
  };
  auto n_of = [&](int p) -> int {
    if constexpr (GROUPED) return grp.N[p];
    return g.N;
  };
  int m0, n0;       // tile being computed
  int cur = 0;      // member it belongs to
  int cur_act = 0;  // and its activation
  {
    const Where w = locate(blockIdx.x);
    cur = w.member;
    cur_act = w.act;
    m0 = w.m0;
    n0 = w.n0;
  }

  // DMA source: the tile whose panels the DMA stream currently fetches
  const uint8_t* A;
  const uint8_t* B;
  uint32_t off[C::ND];
  int nrec = 0x7fffffff;  // 0: the stream has run past the last tile, fetch nothing
  // The lane offsets only depend on the tile through the clamps at the last rows of A
  // and B: between two tiles without partial panels they are not recomputed.
  bool off_clamped = true;  // the first call computes them
  auto set_source = [&](int sm0, int sn0, int member, int act) {
    A = a_of(act) + (int64_t)sm0 * g.lda * 2;
    B = b_of(member) + (int64_t)sn0 * g.ldb;
    const int rows_a = m_of(act) - sm0, rows_b = n_of(member) - sn0;
    const bool clamped = rows_a < C::BM || rows_b < C::BN;
    if (!clamped && !off_clamped) return;
    off_clamped = clamped;
    int l = lane;  // opaque: keeps the row indices out of registers across the K loop
    asm volatile("" : "+v"(l));
#pragma unroll
    for (int p = 0; p < C::NDA; ++p) {  // 8 rows of 128 B per instruction
      const int row = (wave + 4 * p) * 8 + (l >> 3);
      const int c = (l & 7) ^ ((row >> 1) & 7);
      off[p] = (uint32_t)min(row, rows_a - 1) * (uint32_t)(g.lda * 2) + c * 16;
    }
#pragma unroll
    for (int p = 0; p < C::NDB; ++p) {  // 16 rows of 64 B per instruction
      const int row = (wave + 4 * p) * 16 + (l >> 2);
      const int c = (l & 3) ^ ((row >> 2) & 3);
      off[C::NDA + p] = (uint32_t)min(row, rows_b - 1) * (uint32_t)g.ldb + c * 16;
    }
  };
  set_source(m0, n0, cur, cur_act);
  // KTAIL: a chunk of a panel row beyond K goes to an offset beyond the descriptor. (Kept out of
  // the other instances altogether: an `| 0` that the optimiser folds still changed their
  // register allocation, 1 % on the 256 x 192 tile.)
  auto dma_a = [&](int kt, int a_lds, int p) {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(A), 0, nrec, 0x00020000);
    if constexpr (KTAIL) {
      const int chunk = (lane & 7) ^ (((wave * 8 + (lane >> 3)) >> 1) & 7);  // of every row it fetches
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(smem + a_lds + (wave + 4 * p) * 1024), 16,
          (int)(off[p] | (kt * BKE + chunk * 8 < g.K ? 0u : 0x80000000u)), kt * A_ROW, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(smem + a_lds + (wave + 4 * p) * 1024), 16,
          (int)off[p], kt * A_ROW, 0, 0);
    }
  };
  auto dma_b = [&](int kt, int b_lds, int p) {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(B), 0, nrec, 0x00020000);
    if constexpr (KTAIL) {
      const int chunk = (lane & 3) ^ ((lane >> 4) & 3);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(smem + b_lds + (wave + 4 * p) * 1024), 16,
          (int)(off[C::NDA + p] | (kt * BKE + chunk * 16 < g.K ? 0u : 0x80000000u)), kt * B_ROW, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(smem + b_lds + (wave + 4 * p) * 1024), 16,
          (int)off[C::NDA + p], kt * B_ROW, 0, 0);
    }
  };

  // operand read map: A row lane&31 of its block, chunks 4t+2h+s; W operand row
  // p = lane&31 reads panel row 16((p>>2)&1) + 4(p>>3) + (p&3), chunks 2t+h
  const int h = lane >> 5, r32 = lane & 31;
  const int wrow = 16 * ((r32 >> 2) & 1) + 4 * (r32 >> 3) + (r32 & 3);
  uint32_t rd_a[4], rd_b[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      rd_a[2 * t + e] =
          (wm * C::WM + r32) * C::A_ROW + (((4 * t + 2 * h + e) ^ ((r32 >> 1) & 7)) << 4);
    rd_b[t] = (wn * C::WN + wrow) * C::B_ROW + (((2 * t + h) ^ ((wrow >> 2) & 3)) << 4);
  }
  // __restrict__: loads through a restrict-qualified pointer carry alias scope
  // information. Without it the compiler assumes that an LDS read may alias any
  // LDS-DMA write in flight and puts s_waitcnt vmcnt(0) in front of the read, which
  // drains the DMA stream at every step. The stages read in a step are never the
  // ones its DMA fills; the explicit waits before the barriers order the two.
  auto read_a = [&](const uint8_t* __restrict__ st, int i) -> AFrag {
    AFrag f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      f.k[q] = *reinterpret_cast<const v8bf*>(st + rd_a[q] + i * 32 * C::A_ROW);
    return f;
  };
  auto read_a1 = [&](const uint8_t* __restrict__ st, int i, int q) -> v8bf {
    return *reinterpret_cast<const v8bf*>(st + rd_a[q] + i * 32 * C::A_ROW);
  };
  auto read_w1 = [&](const uint8_t* __restrict__ st, int j, int t) -> uint4 {
    return *reinterpret_cast<const uint4*>(st + rd_b[t] + j * 32 * C::B_ROW);
  };
  auto read_w = [&](const uint8_t* __restrict__ st, int j) -> WRaw {
    WRaw f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
      f.t[t] = *reinterpret_cast<const uint4*>(st + rd_b[t] + j * 32 * C::B_ROW);
    return f;
  };

  v16f acc[TM][TN];
  AFrag af[TM];
  AFrag wf[TN];  // converted weights
  WRaw wr[TN];   // weights as read from LDS (next step's, until converted)

  // step s lives in A stage s mod (D+1) and B stage s mod D
  int a_prev = D * C::A_BYTES, a_cur = 0, a_next = C::A_BYTES;
  int b_cur = C::B_BASE, b_next = C::B_BASE + C::B_BYTES;
  // prologue: steps 0 .. D-1 in flight, step 0 landed
#pragma unroll
  for (int s = 0; s < D; ++s) {
#pragma unroll
    for (int p = 0; p < C::NDA; ++p) dma_a(s, s * C::A_BYTES, p);
#pragma unroll
    for (int p = 0; p < C::NDB; ++p) dma_b(s, C::B_BASE + s * C::B_BYTES, p);
  }
  wait_and_barrier<(D - 1) * C::ND>();

  for (int tile = blockIdx.x;; tile += gridDim.x) {
    const int next_tile = tile + gridDim.x;
    int nm0 = 0, nn0 = 0, next_member = 0, next_act = 0;
    // fragments of step 0 (in LDS since the prologue, or since the barrier of the
    // previous tile's last step)
#pragma unroll
    for (int j = 0; j < TN; ++j) wr[j] = read_w(smem + b_cur, j);
    af[0] = read_a(smem + a_cur, 0);

    // One K step; FIRST: step 0 of the tile (the accumulators start from zero).
    // EVENTS: the step may be one of the last max(D, 2) of the tile, where the DMA stream
    // moves on to the next tile and the epilogue operands are staged. The steps before
    // them run in a loop of their own without these tests: what stands between the last
    // MFMA of a step and the first of the next (tests, taken branches) is time the matrix
    // core waits.
    auto step = [&](int kt, auto first_tag, auto events_tag) {
      constexpr bool FIRST = decltype(first_tag)::value;
      constexpr bool EVENTS = decltype(events_tag)::value;
      if (EVENTS && kt == KT - D) {
        // every DMA of this tile has been issued: the stream moves on
        if (next_tile < ntiles) {
          const Where w = locate(next_tile);
          next_member = w.member;
          next_act = w.act;
          nm0 = w.m0;
          nn0 = w.n0;
          set_source(nm0, nn0, next_member, next_act);
        } else {
          nrec = 0;
        }
      }
      if (EVENTS && kt == KT - 2) {
        // b_scale and bias of this tile's columns go to the LDS with two DMA instructions
        // (every wave issues both: equal instruction counts; the same bytes land four
        // times) instead of 6 TN loads per lane at the start of the epilogue. What lies
        // beyond N reads as zero, a null bias is an empty buffer.
        const float* cur_b_scale = g.b_scale;
        const uint16_t* cur_bias = g.bias;
        if constexpr (GROUPED) {
          cur_b_scale = grp.b_scale[cur];
          cur_bias = grp.bias[cur];
        }
        const int cur_n = n_of(cur);
        const __amdgpu_buffer_rsrc_t bs_buf = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(cur_b_scale), 0, cur_n * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t bi_buf = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(cur_bias), 0, cur_bias ? cur_n * 2 : 0, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            bs_buf, (__attribute__((address_space(3))) void*)(smem + C::EPI_BS), 16,
            n0 * 4 + 16 * lane, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            bi_buf, (__attribute__((address_space(3))) void*)(smem + C::EPI_BI), 16,
            n0 * 2 + 16 * lane, 0, 0, 0);
      }
      // step (of its tile) to fetch
      const int kd = !EVENTS || kt + D < KT ? kt + D : kt + D - KT;
      const uint8_t* st = smem + a_cur;
      // half h of the weight operand of column j, MFMA step q: 4 e4m3 bytes -> 4 bf16
      auto convert_half = [&](int j, int q, int h) {
        const uint4& w = wr[j].t[q >> 1];
        const uint32_t src = (q & 1) ? (h ? w.w : w.z) : (h ? w.y : w.x);
        uint4 o = __builtin_bit_cast(uint4, wf[j].k[q]);
        uint32_t c0, c1;
        if constexpr (C::PIN_CONVERT) {
          // Inline assembly (volatile): the conversions stay in the MFMA slot they are
          // written in. As builtins they are pure functions of loaded values, and with the
          // large wave tiles the compiler gathered most of a step's conversions at the top
          // of the loop, where the matrix core then waited for them (with the small wave
          // tiles its own placement is the better one).
          asm volatile("v_cvt_scalef32_pk_bf16_fp8 %0, %1, 1.0" : "=v"(c0) : "v"(src));
          asm volatile("v_cvt_scalef32_pk_bf16_fp8 %0, %1, 1.0 op_sel:[1,0,0]" : "=v"(c1) : "v"(src));
        } else {
          c0 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(src, 1.0f, false));
          c1 = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(src, 1.0f, true));
        }
        if (h) {
          o.z = c0;
          o.w = c1;
        } else {
          o.x = c0;
          o.y = c1;
        }
        wf[j].k[q] = __builtin_bit_cast(v8bf, o);
      };
      // the half operands the schedule puts at time t (CfgWW::CONV)
      auto conversions_at = [&](int t) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              if (C::CONV.t[j][q][h] == t) convert_half(j, q, h);
      };
      auto mfma = [&](int i, int j, int q) {
        if (FIRST && q == 0) {
          mfma_32x32x16_bf16<true>(acc[i][j], wf[j].k[q], af[i].k[q]);
        } else {
          mfma_32x32x16_bf16<false>(acc[i][j], wf[j].k[q], af[i].k[q]);
        }
      };
      // The weights of this step were read from LDS during the previous step, which has
      // also converted the operands the schedule puts there; step 0 of a tile converts
      // those itself.
      if constexpr (FIRST) {
#pragma unroll
        for (int t = -C::S2; t < 0; ++t) conversions_at(t);
      }
      conversions_at(C::kConvTop);
      __builtin_amdgcn_sched_barrier(0);
      // first half: rows 0..H-1, MFMA step q of all their blocks before step q+1
      // (schedule: CfgWW::slot1 ...)
#pragma unroll
      for (int sl = 0; sl < C::S1; ++sl) {
        const int i = C::i_of_slot1(sl), q = C::q_of_slot1(sl), j = sl % TN;
        conversions_at(sl);
#pragma unroll
        for (int t = 0; t < C::T1; ++t) {
          if (C::slot1(t) != sl) continue;
          if (C::is_read1(t)) {
            const int r = C::read1_index(t);
            af[C::read1_row(r)].k[C::read1_step(r)] = read_a1(st, C::read1_row(r), C::read1_step(r));
          } else {
            dma_a(kd, a_prev, C::dma1_index(t));
          }
        }
        mfma(i, j, q);
        __builtin_amdgcn_sched_barrier(0);
      }
      // own LDS reads of this step done, own DMA of the next step landed (the steps
      // after it and the A panel issued above may still fly); then everyone's. In the
      // first D-1 steps of a later tile that DMA was waited for before the previous
      // epilogue's stores.
      if ((FIRST || D > 2) && kt <= D - 2 && tile != (int)blockIdx.x) {
        wait_and_barrier<63>();
      } else {
        wait_and_barrier<(D - 2) * C::ND + C::NDA>();
      }
      // second half: rows H..TM-1 in the same order; the next step's raw weights and A_0
      // are read, its first operands converted (in the last step of a tile: of no use,
      // step 0 of the next tile reads and converts its own) and the B panel D steps ahead
      // goes into the B stage of this step (schedule: CfgWW::slot_w ...)
#pragma unroll
      for (int sl = 0; sl < C::S2; ++sl) {
        const int q = sl / (C::R * TN), i = H + sl / TN % C::R, j = sl % TN;
#pragma unroll
        for (int qq = 0; qq < 4; ++qq)
          if (C::slot_a0(qq) == sl) af[0].k[qq] = read_a1(smem + a_next, 0, qq);
#pragma unroll
        for (int jj = 0; jj < TN; ++jj)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            if (C::slot_w(jj, t) == sl) wr[jj].t[t] = read_w1(smem + b_next, jj, t);
#pragma unroll
        for (int p = 0; p < C::NDB; ++p)
          if (C::slot_dma2(p) == sl) dma_b(kd, b_cur, p);
        conversions_at(sl - C::S2);
        if (sl == C::S2 - 1) {
          // the stages move on in front of the last MFMA, not behind it
          a_prev = a_cur;
          a_cur = a_next;
          a_next = a_next + C::A_BYTES == C::A_STAGES * C::A_BYTES ? 0 : a_next + C::A_BYTES;
          b_cur = b_next;
          b_next = b_next + C::B_BYTES == C::B_BASE + C::B_STAGES * C::B_BYTES
                       ? C::B_BASE
                       : b_next + C::B_BYTES;
        }
        mfma(i, j, q);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    step(0, std::true_type{}, std::true_type{});
    {
      const int events_from = KT - (D > 2 ? D : 2);  // first step that may have an event
      int kt = 1;
      for (; kt < events_from; ++kt) step(kt, std::false_type{}, std::false_type{});
      for (; kt < KT; ++kt) step(kt, std::false_type{}, std::true_type{});
    }
    // the last MFMAs (8 passes each) must have written their accumulators
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    // ---- epilogue: acc[i][j][r] is out[m][n] with
    //   m = m0 + wm*WM + 32i + (lane&31),  n = n0 + wn*WN + 32j + 16h + r
    const int nw = n0 + wn * C::WN + 16 * h;
    const int mw = m0 + wm * C::WM + r32;
    // epilogue operands of all column blocks (the fragment registers are free now):
    // staged in LDS two steps ago, read after the wait below
    v4f bs[TN][4];
    uint4 bi[TN][2];
    // every DMA issued so far (the next tile's first D steps) must have landed
    // before the stores go out: step 0 of the next tile then waits for nothing
    wait_vm<0>();
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int c = wn * C::WN + 16 * h + 32 * j;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        bs[j][q] = *reinterpret_cast<const v4f*>(smem + C::EPI_BS + (c + 4 * q) * 4);
      bi[j][0] = *reinterpret_cast<const uint4*>(smem + C::EPI_BI + c * 2);
      bi[j][1] = *reinterpret_cast<const uint4*>(smem + C::EPI_BI + c * 2 + 16);
    }
    // Accumulators are read with inline assembly, one block at a time (left to itself
    // the compiler copies all of them to VGPRs first and spills what else is live);
    // the GELU decision is taken once per tile, not once per element.
    // Stores: the memory pipeline merges the lanes of a store into one request only
    // when adjacent lanes write adjacent bytes; with lane = 32 h + r32 holding 32 bytes
    // of row r32 every lane is a request of its own, which costs four times the issue
    // time. So the packed words of a block are rearranged first: v_permlane16_swap
    // leaves lane r32 < 16 with the first 16 bytes of rows r32 and r32 + 16 and lane
    // r32 + 16 with their second 16 bytes, then ds_bpermute_b32 (the LDS crossbar, no
    // LDS memory) hands lane L the piece L & 3 of row L >> 2: two stores of 16 rows x
    // 64 contiguous bytes, lanes 4r .. 4r+3 on row r. They are issued while the next
    // block is computed, the last block's after the two copies of the epilogue join.
    const int bp_addr = 4 * (16 * (lane & 3) + (lane >> 2));
    // Buffer stores: the descriptor of a block covers the rows of it that exist (the
    // hardware drops lanes beyond), lanes whose columns do not exist get an offset
    // beyond any descriptor -- no bounds branches, no 64-bit address arithmetic per store.
    constexpr uint32_t kNoColumn = 0x80000000u;
    uint16_t* cur_out = g.out;
    int64_t cur_ldo = g.ldo;
    int cur_epilogue = g.epilogue;
    if constexpr (GROUPED) {
      cur_out = grp.out[cur];
      cur_ldo = grp.ldo[cur];
      cur_epilogue = grp.epilogue[cur];
    }
    const int cur_N = n_of(cur);
    uint8_t* const out_wave = reinterpret_cast<uint8_t*>(cur_out) +
                              ((int64_t)(m0 + wm * C::WM) * cur_ldo + (n0 + wn * C::WN)) * 2;
    const int rows_wave = m_of(cur_act) - (m0 + wm * C::WM);
    const uint32_t out_lane = ((uint32_t)(lane >> 2) * (uint32_t)cur_ldo + 8u * (lane & 3)) * 2;
    const uint32_t half_block = 16u * (uint32_t)cur_ldo * 2;
    uint32_t out_off[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      out_off[j] = n0 + wn * C::WN + 32 * j + 8 * (lane & 3) < cur_N ? out_lane + 64 * j : kNoColumn;
    uint32_t moved[8];
    auto store_moved = [&](int i, int j) {
      const int rows = __builtin_amdgcn_readfirstlane(min(max(rows_wave - 32 * i, 0), 32));
      const __amdgpu_buffer_rsrc_t block = __builtin_amdgcn_make_buffer_rsrc(
          out_wave + (int64_t)(32 * i) * cur_ldo * 2, 0, rows * cur_ldo * 2, 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b128(v4u{moved[0], moved[1], moved[2], moved[3]}, block,
                                             (int)out_off[j], 0, 2);
      __builtin_amdgcn_raw_buffer_store_b128(v4u{moved[4], moved[5], moved[6], moved[7]}, block,
                                             (int)(out_off[j] + half_block), 0, 2);
    };
    auto epilogue = [&](auto gelu_tag) {
      constexpr bool GELU = decltype(gelu_tag)::value;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const uint32_t bw[8] = {bi[j][0].x, bi[j][0].y, bi[j][0].z, bi[j][0].w,
                                bi[j][1].x, bi[j][1].y, bi[j][1].z, bi[j][1].w};
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          uint32_t pk[8];
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const float b0 = __uint_as_float(bw[r >> 1] << 16);
            const float b1 = __uint_as_float(bw[r >> 1] & 0xffff0000u);
            float a0, a1;
            asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(a0) : "a"(acc[i][j][r]));
            asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(a1) : "a"(acc[i][j][r + 1]));
            float v0 = __fmaf_rn(a0, bs[j][r >> 2][r & 3], b0);
            float v1 = __fmaf_rn(a1, bs[j][r >> 2][(r + 1) & 3], b1);
            if constexpr (GELU) {
              v0 = gelu_tanh(v0);
              v1 = gelu_tanh(v1);
            }
            pk[r >> 1] = pack_bf16x2(v0, v1);
          }
          // the previous block's words have had this block's arithmetic to arrive
          __builtin_amdgcn_sched_barrier(0);
          if (i > 0) {
            store_moved(i - 1, j);
          } else if (j > 0) {
            store_moved(TM - 1, j - 1);
          }
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const auto sw = __builtin_amdgcn_permlane16_swap(pk[k], pk[4 + k], false, false);
            moved[k] = (uint32_t)__builtin_amdgcn_ds_bpermute(bp_addr, (int)sw[0]);
            moved[4 + k] = (uint32_t)__builtin_amdgcn_ds_bpermute(bp_addr, (int)sw[1]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (cur_epilogue & CDIT_EPI_GELU_TANH) {
      epilogue(std::true_type{});
    } else {
      epilogue(std::false_type{});
    }
    store_moved(TM - 1, TN - 1);
    if (next_tile >= ntiles) break;
    m0 = nm0;
    n0 = nn0;
    cur = next_member;
    cur_act = next_act;
  }
  // the zero-record DMA of the last D steps must not outlive the workgroup
  wait_vm<0>();
}

template <class C, bool KTAIL = false>
int launch_wide(const GemmArgs& g, hipStream_t stream) {
  static bool lds_allowed[64];
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&gemm_w8a16_wide<C, false, KTAIL>),
                                 C::LDS_BYTES, lds_allowed))
    return rc;
  const int cus = cu_count();
  if (cus <= 0) {
    set_error("cannot query the CU count of the current device");
    return CDIT_EHIP;
  }
  const int tiles_m = (g.M + C::BM - 1) / C::BM, tiles_n = (g.N + C::BN - 1) / C::BN;
  const int ntiles = tiles_m * tiles_n;
  // one persistent workgroup per CU (its LDS and registers fill the CU)
  hipLaunchKernelGGL((gemm_w8a16_wide<C, false, KTAIL>), dim3(ntiles < cus ? ntiles : cus),
                     dim3(C::THREADS), C::LDS_BYTES, stream, g, tiles_m, tiles_n, NoGroup{});
  return 0;
}

// A GemmGroup as one launch: the launcher fills the tile tables of the group for this tile
// shape (grp is a copy).
template <class C>
int launch_wide_grouped(const GemmArgs& g, GemmGroup grp, hipStream_t stream) {
  static bool lds_allowed[64];
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&gemm_w8a16_wide<C, true>),
                                 C::LDS_BYTES, lds_allowed))
    return rc;
  const int cus = cu_count();
  if (cus <= 0) {
    set_error("cannot query the CU count of the current device");
    return CDIT_EHIP;
  }
  int ntiles = 0;
  for (int s = 0; s < grp.acts; ++s) {
    int cols = 0;
    for (int p = grp.first_member[s]; p < grp.first_member[s + 1]; ++p) {
      grp.col_begin[p] = cols;
      cols += (grp.N[p] + C::BN - 1) / C::BN;
    }
    grp.tiles_m[s] = (grp.M[s] + C::BM - 1) / C::BM;
    grp.tiles_n[s] = cols;
    grp.tile_begin[s] = ntiles;
    ntiles += grp.tiles_m[s] * cols;
  }
  for (int s = grp.acts; s <= kMaxActs; ++s) grp.tile_begin[s] = ntiles;
  for (int p = grp.count; p <= kMaxGroup; ++p) grp.col_begin[p] = 0x7fffffff;
  hipLaunchKernelGGL((gemm_w8a16_wide<C, true>), dim3(ntiles < cus ? ntiles : cus), dim3(C::THREADS),
                     C::LDS_BYTES, stream, g, 0, 0, grp);
  return 0;
}

// ---------------------------------------------------------------------------
// A few dozen rows (the prompt's projections: M = 17 to 128 or so) and few rows on many columns: a
// workgroup of two wavefronts per 32 x 32 tile. A 128 x 64 tile of the wide kernel gives such a
// problem to a few dozen CUs, whose prefetch cannot keep the weight stream in flight (one CU has
// some 60 GB/s from HBM); 32 x 32 tiles put it on all of them. A ring of D stages (A 32 rows x
// 128 B, B 32 rows x 64 B, the swizzles of the wide kernel) is filled D steps ahead by LDS-DMA of
// the one wavefront; the other reads the operands of a step one step ahead of their MFMAs. One
// barrier per step: in front of it step kt + 1 has landed, behind it the operands of step kt are in
// registers and its stage is free. MFMA, K order and epilogue arithmetic are those of the wide
// kernel, so the results are bit-identical to it (a member of a batch may run there).
// What bounds it: a chain of four dependent MFMAs (128 clocks) next to 16 conversions, and six DMA
// instructions per step, each on a wavefront of its own: about 250 clocks per step (500 with one
// wavefront issuing both in order). Two feeding wavefronts: 3 to 8 % faster with one tile per CU,
// 4 to 8 % slower with two. Conversions a step ahead of their MFMAs: the same or slower. D = 6: four
// workgroups fit the LDS of a CU (4 x 36 KiB), with 8 three, and a fourth is a second round. With up to two per CU 8
// is 1 to 5 % slower on matrices in the last-level cache; from HBM the same up to K = 4096 and 4 % faster beyond (geometric
// mean of 325 shapes); 4 is up to 27 % slower there.
// Another weight matrix per launch (M x K x N), us, one wavefront before -> now: 77 x 4096 x 3072
// 15.9 -> 11.2, 17 x 3072 x 3072 12.3 -> 8.5, 128 x 3072 x 3072 13.2 -> 9.5, 256 x 15360 x 1024 47.4
// -> 31, 100 x 1024 x 2048 6.3 -> 4.9; 128 x 64 tiles of the wide kernel -> now: 245 x 1664 x 2560 11.4 ->
// 8.1, 299 x 3328 x 2368 (740 tiles) 18.1 -> 15.1, 103 x 2816 x 6016 (752) 15.6 -> 10.9; beyond 768 tiles
// either way: 154 x 2560 x 5056 (790) 15.8 -> 13.7, 592 x 1664 x 1600 (950) 11.9 -> 14.9. Where it is taken:
// wavetile_better().
constexpr int kTileDepth = 6, kTileLds = kTileDepth * 32 * 3 * BKE;
template <bool GELU>
__global__ __launch_bounds__(128) void gemm_w8a16_wavetile(GemmArgs g, int tiles_m, int tiles_n) {
  constexpr int D = kTileDepth, A_BYTES = 32 * 2 * BKE, STAGE = kTileLds / D, NDMA = 6;
  static_assert(D >= 3 && (D - 1) * NDMA < 63 && D * STAGE <= 64 * 1024, "vmcnt has 6 bits; LDS without opt-in");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  // the row tiles of one column tile on one XCD (workgroups go to the 8 XCDs in turn): its
  // weights come from HBM once
  const int id = blockIdx.x;
  const int tn = id / 8 / tiles_m * 8 + id % 8, tm = id / 8 % tiles_m;
  if (tn >= tiles_n) return;
  const int lane = threadIdx.x & 63, m0 = tm * 32, n0 = tn * 32;
  const int h = lane >> 5, r32 = lane & 31;
  const int KT = (g.K + BKE - 1) / BKE;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 1) {
    // the feeding wavefront
    // DMA maps: an instruction fills 8 A rows (chunk (lane & 7) ^ swizzle, which differs between
    // even and odd instructions by 4) or 16 B rows
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(g.a)) + (int64_t)m0 * g.lda * 2, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(g.b) + (int64_t)n0 * g.ldb, 0, 0x7fffffff, 0x00020000);
    const int ca = (lane & 7) ^ (lane >> 4), cb = (lane & 3) ^ ((lane >> 4) & 3);
    uint32_t off[NDMA];
  #pragma unroll
    for (int p = 0; p < 4; ++p)
      off[p] = (uint32_t)min(8 * p + (lane >> 3), g.M - 1 - m0) * (uint32_t)(g.lda * 2) + (ca ^ (4 * (p & 1))) * 16;
  #pragma unroll
    for (int p = 0; p < 2; ++p)
      off[4 + p] = (uint32_t)min(16 * p + (lane >> 2), g.N - 1 - n0) * (uint32_t)g.ldb + cb * 16;
    // Elements beyond K (a partial last step, steps beyond the last) are fetched from beyond the
    // descriptor: zeros.
    auto dma = [&](int kt, int stage) {
      const int left = g.K - kt * BKE;
      const uint32_t a0 = ca * 8 < left ? 0u : 0x80000000u, a1 = (ca ^ 4) * 8 < left ? 0u : 0x80000000u;
      const uint32_t b0 = cb * 16 < left ? 0u : 0x80000000u;
      __attribute__((address_space(3))) uint8_t* st =
          (__attribute__((address_space(3))) uint8_t*)(smem) + stage;
  #pragma unroll
      for (int p = 0; p < 4; ++p)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(st + p * 1024), 16,
                                                 (int)(off[p] | (p & 1 ? a1 : a0)), kt * 2 * BKE, 0, 0);
  #pragma unroll
      for (int p = 0; p < 2; ++p)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(st + A_BYTES + p * 1024),
                                                 16, (int)(off[4 + p] | b0), kt * BKE, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < D; ++s) dma(s, s * STAGE);
    wait_and_barrier<(D - 1) * NDMA>();  // step 0 has landed
    int stage = 0;                       // of step kt
    for (int kt = 0; kt < KT; ++kt) {
      // step kt + 1 has landed; behind the barrier the operands of step kt are in registers
      wait_and_barrier<(D - 2) * NDMA>();
      dma(kt + D, stage);
      stage = stage + STAGE == D * STAGE ? 0 : stage + STAGE;
    }
    wait_vm<0>();  // no DMA outlives the workgroup
    return;
  }

  // scale and bias of the lane's 16 columns n0 + 16 h .. (N % 16 == 0: all in or all out)
  const int nw = n0 + 16 * h;
  const bool n_in = nw < g.N;
  v4f bs[4];
  uint4 bi[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
#pragma unroll
  for (int q = 0; q < 4; ++q)
    bs[q] = n_in ? reinterpret_cast<const v4f*>(g.b_scale + nw)[q] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
  if (n_in && g.bias) {
    bi[0] = reinterpret_cast<const uint4*>(g.bias + nw)[0];
    bi[1] = reinterpret_cast<const uint4*>(g.bias + nw)[1];
  }

  // operand read maps, as in the wide kernel
  const int wrow = 16 * ((r32 >> 2) & 1) + 4 * (r32 >> 3) + (r32 & 3);
  uint32_t rd_a[4], rd_b[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      rd_a[2 * t + e] = r32 * (2 * BKE) + (((4 * t + 2 * h + e) ^ ((r32 >> 1) & 7)) << 4);
    rd_b[t] = A_BYTES + wrow * BKE + (((2 * t + h) ^ ((wrow >> 2) & 3)) << 4);
  }
  struct Step {
    v8bf a[4];
    uint4 w[2];
  };
  // (__restrict__: see the wide kernel; without it every read would wait for the whole stream)
  auto read = [&](const uint8_t* __restrict__ st) -> Step {
    Step f;
#pragma unroll
    for (int q = 0; q < 4; ++q) f.a[q] = *reinterpret_cast<const v8bf*>(st + rd_a[q]);
#pragma unroll
    for (int t = 0; t < 2; ++t) f.w[t] = *reinterpret_cast<const uint4*>(st + rd_b[t]);
    return f;
  };

  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  wait_and_barrier<63>();
  Step even = read(smem), odd;
  int stage = STAGE;  // of step kt + 1
  // Step kt: its operands are in `f`; reads step kt + 1 into `nf`.
  auto step = [&](const Step& f, Step& nf) {
    wait_and_barrier<63>();
    nf = read(smem + stage);
    __builtin_amdgcn_sched_barrier(0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e4m3x8_to_bf16(f.w[0].x, f.w[0].y), f.a[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e4m3x8_to_bf16(f.w[0].z, f.w[0].w), f.a[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e4m3x8_to_bf16(f.w[1].x, f.w[1].y), f.a[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e4m3x8_to_bf16(f.w[1].z, f.w[1].w), f.a[3], acc, 0, 0, 0);
    stage = stage + STAGE == D * STAGE ? 0 : stage + STAGE;
  };
  for (int kt = 0; kt < KT; kt += 2) {
    step(even, odd);
    if (kt + 1 < KT) step(odd, even);
  }

  // acc[r] is out[m0 + r32][n0 + 16 h + r]
  const int m = m0 + r32;
  if (m >= g.M || !n_in) return;
  const uint32_t bw[8] = {bi[0].x, bi[0].y, bi[0].z, bi[0].w, bi[1].x, bi[1].y, bi[1].z, bi[1].w};
  uint32_t pk[8];
#pragma unroll
  for (int r = 0; r < 16; r += 2) {
    float v0 = __fmaf_rn(acc[r], bs[r >> 2][r & 3], __uint_as_float(bw[r >> 1] << 16));
    float v1 = __fmaf_rn(acc[r + 1], bs[r >> 2][(r + 1) & 3], __uint_as_float(bw[r >> 1] & 0xffff0000u));
    if constexpr (GELU) {
      v0 = gelu_tanh(v0);
      v1 = gelu_tanh(v1);
    }
    pk[r >> 1] = pack_bf16x2(v0, v1);
  }
  uint4* dst = reinterpret_cast<uint4*>(g.out + (int64_t)m * g.ldo + nw);
  dst[0] = uint4{pk[0], pk[1], pk[2], pk[3]};
  dst[1] = uint4{pk[4], pk[5], pk[6], pk[7]};
}

int launch_wavetile(const GemmArgs& g, hipStream_t stream) {
  const int tiles_m = (g.M + 31) / 32, tiles_n = (g.N + 31) / 32;
  const dim3 grid((tiles_n + 7) / 8 * 8 * tiles_m), block(128);
  if (g.epilogue & CDIT_EPI_GELU_TANH)
    hipLaunchKernelGGL(gemm_w8a16_wavetile<true>, grid, block, kTileLds, stream, g, tiles_m, tiles_n);
  else
    hipLaunchKernelGGL(gemm_w8a16_wavetile<false>, grid, block, kTileLds, stream, g, tiles_m, tiles_n);
  return 0;
}

// ---------------------------------------------------------------------------
// Problems that one round of tiles covers, as gemm_fp8_fed: bound by what one CU gets through its vector memory path (64 KB
// in flight: 52 to 60 GB/s from HBM, some 90 from the last-level cache), here (2 BM + BN) K bytes of the fullest CU. So tiles that
// are wider than they are high, and of as many shapes as it takes for every CU to get at most one. A wavefront multiplies all
// rows of the tile with its 16 columns, whose weights are then converted once per workgroup (8 conversions per 16
// columns and 64 elements next to 2 MFMAs per 16 x 16 block); two wavefronts only feed. A step is SUB times 64
// elements between two barriers: with 128 the small tiles, whose steps are short, take 4 % (48 x 64) to 20 % (32 x 32) less;
// the larger ones, with room for fewer stages then, 2 to 4 % more (64 x 96, 48 x 96).
// v_mfma_f32_16x16x32_bf16 adds its 32 products in the order of the lane groups that hold them, eight at a time, after
// the accumulator: a chain of them over the pieces in the order in which the wide kernel's 32x32x16 instructions take theirs
// (in each 32 elements the first, third, second and fourth eight) gives the same bits, which is what the swap of the piece's
// two low bits in the swizzle is for.
// us, another weight matrix per launch, the best of the other kernels -> this one, M x N x K: 77 x 3072 x 4096 14.0 -> 10.8 (16 x
// 64: 240 tiles; of the 288 of 32 x 32 some CUs get two), 200 x 2560 x 8192 31.1 -> 22.8 (48 x 64), 17 x 3072 x 3072 9.0 -> 7.4
// (32 x 32), 342 x 2752 x 12352 61.5 -> 46.6 (80 x 64).
template <int BM_, int BN_, int WAVES_, int SUB_, int DEPTH_>
struct CfgFedW {
  static constexpr int BM = BM_, BN = BN_, WAVES = WAVES_, SUB = SUB_, DEPTH = DEPTH_;
  static constexpr int GROUP_M = 8;  // (4: the same time)
  static constexpr int DMA_A = BM / 8, DMA_B = BN / 16;  // DMA instructions per 64 elements
  static constexpr int FEEDERS = 2, NDMA = (DMA_A + DMA_B) / FEEDERS, THREADS = 64 * (WAVES + FEEDERS);
  static constexpr int TM = BM / 16, TN = 1;  // fragments of 16 rows, and of 16 columns, per wavefront
  static constexpr int A_BYTES = BM * 2 * BKE, PART = A_BYTES + BN * BKE, STAGE = SUB * PART, LDS_BYTES = DEPTH * STAGE;
  static constexpr int NH = 0, ODD = 1;  // store_fed_tile
  static_assert(BM % 16 == 0 && BN == 16 * WAVES && (DMA_A + DMA_B) % FEEDERS == 0, "whole fragments, whole instructions");
  static_assert(DEPTH >= 3 && (DEPTH - 1) * NDMA * SUB <= 63 && LDS_BYTES <= 160 * 1024, "vmcnt has 6 bits; LDS");
  // first of the four columns (of the wavefront's) that lane group q holds
  __device__ static constexpr int col(int, int q) { return 4 * q; }
  // chunk c of B panel row r is stored at c ^ swizzle
  __device__ static int swz_b(int r) { return (r >> 2) & 3; }
};

template <class C>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2))) void
gemm_w8a16_fed(GemmArgs g, int tiles_m, int tiles_n) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  constexpr int D = C::DEPTH, TM = C::TM, SUB = C::SUB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KT = (g.K + SUB * BKE - 1) / (SUB * BKE);
  // workgroups go to the 8 XCDs in turn; each XCD gets consecutive tiles (any number of them), which share panels
  const int ntiles = tiles_m * tiles_n, xcd = blockIdx.x % 8;
  int tm, tn;
  tile_of_linear<C::GROUP_M>(xcd * (ntiles / 8) + min(xcd, ntiles % 8) + blockIdx.x / 8, tiles_m, tiles_n, &tm, &tn);
  const int m0 = tm * C::BM, n0 = tn * C::BN;

  if (wave >= C::WAVES) {
    // Feeding wavefront f: its instruction p is number f NDMA + p of a part of 64 elements: 8 A rows (lane l lands on row
    // l / 8, position l % 8) or, behind all of those, 16 B rows (row l / 4, position l % 4).
    const int f = wave - C::WAVES;
    const uint8_t* const a = static_cast<const uint8_t*>(g.a) + (int64_t)m0 * g.lda * 2;
    const uint8_t* const b = g.b + (int64_t)n0 * g.ldb;
    uint32_t off[C::NDMA];
    int first[C::NDMA];  // first element of the lane's piece
#pragma unroll
    for (int p = 0; p < C::NDMA; ++p) {
      const int q = f * C::NDMA + p;
      if (q < C::DMA_A) {
        const int row = 8 * q + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        const int piece = (c & 4) | ((c & 1) << 1) | ((c >> 1) & 1);
        off[p] = (uint32_t)min(row, g.M - 1 - m0) * (uint32_t)(g.lda * 2) + piece * 16;
        first[p] = piece * 8;
      } else {
        const int row = 16 * (q - C::DMA_A) + (lane >> 2), c = (lane & 3) ^ C::swz_b(row);
        off[p] = (uint32_t)min(row, g.N - 1 - n0) * (uint32_t)g.ldb + c * 16;
        first[p] = c * 16;
      }
    }
    // Elements beyond K (a partial last step, steps beyond the last) are fetched from beyond the descriptor: zeros.
    auto dma = [&](int kt, int stage) {
#pragma unroll
      for (int u = 0; u < SUB; ++u) {
        const int k = kt * SUB + u, left = g.K - k * BKE;
#pragma unroll
        for (int p = 0; p < C::NDMA; ++p) {
          const int q = f * C::NDMA + p;
          const bool is_a = q < C::DMA_A;
          const __amdgpu_buffer_rsrc_t src =
              __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(is_a ? a : b), 0, 0x7fffffff, 0x00020000);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              src, (__attribute__((address_space(3))) void*)(smem + stage + u * C::PART + q * 1024), 16,
              (int)(off[p] | (first[p] < left ? 0u : 0x80000000u)), k * (is_a ? 2 * BKE : BKE), 0, 0);
        }
      }
    };
#pragma unroll
    for (int s = 0; s < D; ++s) dma(s, s * C::STAGE);
    wait_and_barrier<(D - 1) * C::NDMA * SUB>();  // step 0 has landed
    int stage = 0;                                // of step kt
    for (int kt = 0; kt < KT; ++kt) {
      // step kt + 1 has landed; behind the barrier the operands of step kt are in registers
      wait_and_barrier<(D - 2) * C::NDMA * SUB>();
      dma(kt + D, stage);
      stage = stage + C::STAGE == D * C::STAGE ? 0 : stage + C::STAGE;
    }
    wait_vm<0>();  // no DMA outlives the workgroup
    return;
  }

  const int r16 = lane & 15, kg = lane >> 4, h = kg & 1, e = kg >> 1;
  const int nw = n0 + wave * 16;
  // scale and bias; what lies beyond N reads as zero, a null bias is an empty buffer
  auto vec = [](const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t bs_buf = vec(g.b_scale, g.N * 4), bi_buf = vec(g.bias, g.bias ? g.N * 2 : 0);
  const int n = nw + C::col(0, kg);
  const v4f bs[1] = {__builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(bs_buf, n * 4, 0, 0))};
  const uint2 bi[1] = {__builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(bi_buf, n * 2, 0, 0))};
  float as[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) as[i] = 1.0f;

  struct Step {
    v8bf a[2 * SUB][TM];
    uint2 w[2 * SUB];
  };
  const int a_swz = (r16 >> 1) & 7, brow = wave * 16 + r16;
  // operands of the 32 elements x of a step (__restrict__: see the wide kernel)
  auto read = [&](const uint8_t* __restrict__ stage_at, Step& f, int x) {
    const uint8_t* st = stage_at + (x >> 1) * C::PART;
    const int t = x & 1;
    f.w[x] = *reinterpret_cast<const uint2*>(st + C::A_BYTES + brow * BKE + (((2 * t + h) ^ C::swz_b(brow)) << 4) + 8 * e);
#pragma unroll
    for (int i = 0; i < TM; ++i)
      f.a[x][i] = *reinterpret_cast<const v8bf*>(st + (16 * i + r16) * (2 * BKE) + (((4 * t + kg) ^ a_swz) << 4));
  };
  v4f acc[TM][1];
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i][0] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  wait_and_barrier<63>();
  Step even, odd;
#pragma unroll
  for (int x = 0; x < 2 * SUB; ++x) read(smem, even, x);
  int stage = C::STAGE;  // of step kt + 1
  // Step kt: its operands are in `f`; reads step kt + 1 into `nf`, 32 elements in front of each 32 of the MFMAs, or, where
  // a step has few of those, all in front of the first.
  constexpr bool kReadsFirst = SUB * TM <= 4;
  auto step = [&](const Step& f, Step& nf) {
    wait_and_barrier<63>();
#pragma unroll
    for (int x = 0; x < 2 * SUB; ++x) {
      if (x == 0 || !kReadsFirst) {
#pragma unroll
        for (int y = x; y < (kReadsFirst ? 2 * SUB : x + 1); ++y) read(smem + stage, nf, y);
        __builtin_amdgcn_sched_barrier(0);
      }
      const v8bf b = e4m3x8_to_bf16(f.w[x].x, f.w[x].y);
      // operands swapped: result rows follow B (n), result columns follow A (m)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, f.a[x][i], acc[i][0], 0, 0, 0);
      if (!kReadsFirst) __builtin_amdgcn_sched_barrier(0);
    }
    stage = stage + C::STAGE == D * C::STAGE ? 0 : stage + C::STAGE;
  };
  for (int kt = 0; kt < KT; kt += 2) {
    step(even, odd);
    if (kt + 1 < KT) step(odd, even);
  }

  uint8_t* const out_wave = reinterpret_cast<uint8_t*>(g.out) + ((int64_t)m0 * g.ldo + nw) * 2;
  if (g.epilogue & CDIT_EPI_GELU_TANH) {
    store_fed_tile<C, CDIT_DT_BF16, true>(acc, as, bs, bi, out_wave, g.ldo, g.M - m0, g.N - nw, lane);
  } else {
    store_fed_tile<C, CDIT_DT_BF16, false>(acc, as, bs, bi, out_wave, g.ldo, g.M - m0, g.N - nw, lane);
  }
}

template <class C>
int launch_fed(const GemmArgs& g, hipStream_t stream) {
  static bool lds_allowed[64];
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&gemm_w8a16_fed<C>), C::LDS_BYTES, lds_allowed)) return rc;
  const int tiles_m = (g.M + C::BM - 1) / C::BM, tiles_n = (g.N + C::BN - 1) / C::BN;
  hipLaunchKernelGGL(gemm_w8a16_fed<C>, dim3(tiles_m * tiles_n), dim3(C::THREADS), C::LDS_BYTES, stream, g, tiles_m, tiles_n);
  return 0;
}

// ---------------------------------------------------------------------------
// Skinny kernel for M <= 16 where the whole-row kernel below is not taken: weight streaming. A
// workgroup of 4 waves owns 16 output channels, each wave a quarter of K. Per
// 128-element chunk a lane (weight row l&15, K group l>>4) loads 32 e4m3 bytes
// straight from HBM and the matching 32 bf16 activations (zero for rows >= M),
// converts the weights to bf16 and issues four v_mfma_f32_16x16x32_bf16; the four
// partial tiles are summed through LDS.
// KTAIL: K is not a multiple of 128; what lies beyond it is masked. The masks are kept out of the
// instance for whole chunks: each made the load a branch of its own, and the registers of the
// masked loads cost two of seven wavefronts per SIMD (16 rows, N = 18432, K = 3072: 26.5 us
// without, 32.4 with masks; K = 5120: 47.4 and 60.9).
template <bool KTAIL>
__global__ __launch_bounds__(256) void gemm_w8a16_skinny(GemmArgs g) {
  __shared__ float part[4][16][17];
  typedef float v4f_ __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int nrow = min(n0 + r, g.N - 1);
  const int KT = KTAIL ? (g.K + 127) / 128 : g.K / 128;
  const int per = (KT + 3) / 4;
  const int k_begin = wave * per, k_end = min(KT, k_begin + per);
  const uint8_t* __restrict__ wp = g.b + (int64_t)nrow * g.ldb + kg * 32;
  const uint16_t* __restrict__ ap =
      static_cast<const uint16_t*>(g.a) + (int64_t)min(r, g.M - 1) * g.lda + kg * 32;
  const bool a_valid = r < g.M;
  v4f_ acc = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = 3;  // chunks in flight
  for (int k0 = k_begin; k0 < k_end; k0 += U) {
    uint4 w[U][2];
    v8bf a[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kt = min(k0 + u, k_end - 1);
      const v8bf* aq = reinterpret_cast<const v8bf*>(ap + (int64_t)kt * 128);
      if constexpr (KTAIL) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {  // (16 elements beyond K are zeros on both sides)
          const bool in = kt * 128 + kg * 32 + e * 16 < g.K;
          w[u][e] = in ? *reinterpret_cast<const uint4*>(wp + kt * 128 + e * 16) : uint4{0u, 0u, 0u, 0u};
#pragma unroll
          for (int t = 2 * e; t < 2 * e + 2; ++t) a[u][t] = in ? aq[t] : v8bf{0, 0, 0, 0, 0, 0, 0, 0};
        }
      } else {
        const uint4* wq = reinterpret_cast<const uint4*>(wp + (int64_t)kt * 128);
        w[u][0] = wq[0];
        w[u][1] = wq[1];
#pragma unroll
        for (int t = 0; t < 4; ++t) a[u][t] = aq[t];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + u < k_end) {
        const uint32_t words[8] = {w[u][0].x, w[u][0].y, w[u][0].z, w[u][0].w,
                                   w[u][1].x, w[u][1].y, w[u][1].z, w[u][1].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          v8bf af = a[u][t];
          if (!a_valid) af = v8bf{0, 0, 0, 0, 0, 0, 0, 0};
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(e4m3x8_to_bf16(words[2 * t], words[2 * t + 1]), af,
                                                        acc, 0, 0, 0);
        }
      }
    }
  }
  // acc[e] = partial out[m = lane&15][n0 + 4*(lane>>4) + e]
#pragma unroll
  for (int e = 0; e < 4; ++e) part[wave][r][4 * kg + e] = acc[e];
  __syncthreads();
  if (wave == 0) {
    const int m = r, nl = 4 * kg;
    if (m < g.M && n0 + nl < g.N) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sum = (part[0][m][nl + e] + part[1][m][nl + e]) +
                          (part[2][m][nl + e] + part[3][m][nl + e]);
        const int n = n0 + nl + e;
        float t = sum * g.b_scale[n];
        if (g.bias) t += __uint_as_float((uint32_t)g.bias[n] << 16);
        if (g.epilogue & CDIT_EPI_GELU_TANH) t = gelu_tanh(t);
        v[e] = t;
      }
      uint2 pk;
      pk.x = pack_bf16x2(v[0], v[1]);
      pk.y = pack_bf16x2(v[2], v[3]);
      *reinterpret_cast<uint2*>(g.out + (int64_t)m * g.ldo + n0 + nl) = pk;
    }
  }
}

// One to four activation rows (the modulation Linears: one embedding per image, with guidance
// and a batch a few), K <= 4096 (whole_rows_better() below), with the access pattern of the w8a8 path's linear_fp8_row1: a
// load instruction of the wavefront reads 1 KiB of one weight row (lane l bytes 16 l ..
// 16 l + 15) where the 16-row arrangement above makes every lane a memory request of its own;
// the MFMA's 16 "rows" are 16 interleaved K subsets of that row, the activation is fetched at
// the same positions lane for lane (32 bytes of bf16 per 16 weight bytes), D[i][i] is the partial
// dot product over subset i and the diagonal sums to the whole one. A wavefront owns three whole
// weight rows, all of their loads in flight at once; each further activation row costs its
// MFMAs and a diagonal sum per weight row and no memory traffic to speak of.
// With a different weight matrix per launch, against the 16-row kernel below 5 rows: 2 rows
// 16.4 -> 14.2 us at N = 18432, K = 3072 (4.0 TB/s of weights), 8.2 -> 4.4 at 4096 x 1088;
// 4 rows 18.3 -> 17.6 and, at N = 9216, 12.3 -> 9.9. One row has a body of its own: through the
// one for several it took 1 to 4 % longer (4.39 -> 4.55 us at N = 960, K = 4096).
constexpr int kRow1Rows = 3, kRow1Waves = 4;
template <int CHK, int MA>
__global__ __launch_bounds__(64 * kRow1Waves, MA == 1 ? 1 : (MA == 2 ? 6 : 4) - (CHK == 4 ? MA / 2 : 0)) void
gemm_w8a16_rows(GemmArgs g) {
  constexpr int R = kRow1Rows;
  typedef float v4f_ __attribute__((ext_vector_type(4)));
  typedef unsigned int u4v __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = (blockIdx.x * kRow1Waves + wave) * R;
  const u4v zero4 = {0u, 0u, 0u, 0u};
  u4v w[R][CHK];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const uint8_t* __restrict__ wp = g.b + (int64_t)min(row0 + q, g.N - 1) * g.ldb + lane * 16;
#pragma unroll
    for (int c = 0; c < CHK; ++c) {
      if (c * 1024 + lane * 16 < g.K) {
        w[q][c] = __builtin_nontemporal_load(reinterpret_cast<const u4v*>(wp + c * 1024));
      } else {
        w[q][c] = zero4;
      }
    }
  }
  const v8bf zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // 1 KiB piece c of activation row m
  auto load_x = [&](v8bf (&x)[2], int m, int c) {
    const bool in = c * 1024 + lane * 16 < g.K;
    const v8bf* src = reinterpret_cast<const v8bf*>(static_cast<const uint16_t*>(g.a) + m * g.lda +
                                                    c * 1024 + lane * 16);
    x[0] = in ? src[0] : zero8;
    x[1] = in ? src[1] : zero8;
  };
  // lane l holds D[4 (l >> 4) + e][l & 15]: the diagonal entry of lanes 0-3, 20-23, 40-43, 60-63
  const int diag = (lane & 15) - 4 * (lane >> 4);
  float mine = 0.0f;  // lane q * MA + m keeps the dot product of weight row row0 + q, row m
  auto keep_diagonal = [&](const v4f_& acc, int q, int m) {
    float d = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) d = diag == e ? acc[e] : d;
    const float sum = wave_sum_f32(d);
    mine = lane == q * MA + m ? sum : mine;
  };
  if constexpr (MA == 1) {
    // one row: all of it is fetched right behind the weights, and a weight row's sum is under way
    // while the next one's MFMAs run
    v8bf xa[CHK][2];
#pragma unroll
    for (int c = 0; c < CHK; ++c) load_x(xa[c], 0, c);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      v4f_ acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < CHK; ++c) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(e4m3x8_to_bf16(w[q][c][2 * t], w[q][c][2 * t + 1]),
                                                        xa[c][t], acc, 0, 0, 0);
      }
      keep_diagonal(acc, q, 0);
    }
  } else {
    // (more rows: fetched inside the K loop; held across it they took the registers of the
    // wavefronts that keep the weight loads in flight)
    v4f_ acc[R][MA];
#pragma unroll
    for (int q = 0; q < R; ++q) {
#pragma unroll
      for (int m = 0; m < MA; ++m) acc[q][m] = v4f_{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int c = 0; c < CHK; ++c) {
      v8bf xa[MA][2];
#pragma unroll
      for (int m = 0; m < MA; ++m) load_x(xa[m], m, c);
#pragma unroll
      for (int q = 0; q < R; ++q) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const v8bf wf = e4m3x8_to_bf16(w[q][c][2 * t], w[q][c][2 * t + 1]);
#pragma unroll
          for (int m = 0; m < MA; ++m)
            acc[q][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xa[m][t], acc[q][m], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
#pragma unroll
      for (int m = 0; m < MA; ++m) keep_diagonal(acc[q][m], q, m);
    }
  }
  const int n = row0 + lane / MA, m = lane % MA;
  if (lane < R * MA && n < g.N) {
    float t = mine * g.b_scale[n];
    if (g.bias) t += __uint_as_float((uint32_t)g.bias[n] << 16);
    if (g.epilogue & CDIT_EPI_GELU_TANH) t = gelu_tanh(t);
    g.out[m * g.ldo + n] = (uint16_t)(pack_bf16x2(t, 0.0f) & 0xffffu);
  }
}

template <int CHK>
void launch_rows_chk(const GemmArgs& g, hipStream_t stream) {
  constexpr int rows_wg = kRow1Rows * kRow1Waves;
  const dim3 grid((g.N + rows_wg - 1) / rows_wg), block(64 * kRow1Waves);
  switch (g.M) {
    case 1: hipLaunchKernelGGL((gemm_w8a16_rows<CHK, 1>), grid, block, 0, stream, g); break;
    case 2: hipLaunchKernelGGL((gemm_w8a16_rows<CHK, 2>), grid, block, 0, stream, g); break;
    case 3: hipLaunchKernelGGL((gemm_w8a16_rows<CHK, 3>), grid, block, 0, stream, g); break;
    default: hipLaunchKernelGGL((gemm_w8a16_rows<CHK, 4>), grid, block, 0, stream, g); break;
  }
}

// Any shape: one output element per thread, scalar decode + FMA.
__global__ __launch_bounds__(256) void gemm_w8a16_generic(GemmArgs g) {
  const int n = blockIdx.x * 16 + (threadIdx.x & 15);
  const int m = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (m >= g.M || n >= g.N) return;
  const uint16_t* a = static_cast<const uint16_t*>(g.a) + (int64_t)m * g.lda;
  const uint8_t* b = g.b + (int64_t)n * g.ldb;
  float acc = 0.0f;
  for (int k = 0; k < g.K; ++k) {
    const float x = __uint_as_float((uint32_t)a[k] << 16);
    const float w = __builtin_amdgcn_cvt_f32_fp8((int)b[k], 0);
    acc = fmaf(x, w, acc);
  }
  float v = acc * g.b_scale[n];
  if (g.bias) v += __uint_as_float((uint32_t)g.bias[n] << 16);
  if (g.epilogue & CDIT_EPI_GELU_TANH) v = gelu_tanh(v);
  g.out[(int64_t)m * g.ldo + n] = (uint16_t)f32_to_bf16_bits(v);
}

template <class C>
int launch_tiled(const GemmArgs& g, hipStream_t stream) {
  static bool lds_allowed[64];
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&gemm_w8a16_tiled<C>), C::LDS_BYTES,
                                 lds_allowed))
    return rc;
  const int tiles_m = (g.M + C::BM - 1) / C::BM, tiles_n = (g.N + C::BN - 1) / C::BN;
  hipLaunchKernelGGL(gemm_w8a16_tiled<C>, dim3(tiles_m * tiles_n), dim3(C::THREADS), C::LDS_BYTES,
                     stream, g, tiles_m, tiles_n);
  return 0;
}

// What every kernel but the generic one asks of its operands; K is any multiple of 16 here.
bool aligned_ok(const GemmArgs& g) {
  return g.K >= 16 && g.K % 16 == 0 && g.N % 8 == 0 && g.lda % 8 == 0 && g.ldb % 16 == 0 &&
         g.ldo % 8 == 0 && reinterpret_cast<uintptr_t>(g.a) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(g.b) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(g.out) % 16 == 0 &&
         // the epilogues load scales as float4 and bias as 8-byte packs
         reinterpret_cast<uintptr_t>(g.b_scale) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(g.bias) % 16 == 0 &&
         (int64_t)1024 * g.lda < (int64_t)1 << 31 && (int64_t)512 * g.ldb < (int64_t)1 << 31 &&
         (int64_t)512 * g.ldo < (int64_t)1 << 29;  // 32-bit byte offsets within a block of rows
}

bool tiled_ok(const GemmArgs& g) { return g.K >= BKE && g.K % BKE == 0 && aligned_ok(g); }

}  // namespace

typedef CfgW<256, 256, 2, 2, true, 8> W0;   // 4 waves, 2 stages
typedef CfgW<128, 128, 2, 2, true, 8> W3;   // small tiles, two workgroups per CU
typedef CfgWW<256, 256, 4> W7;              // wide: 4 waves, 128x128 wave tiles
typedef CfgWW<256, 192, 4> W8;              // wide: 128x96 wave tiles
typedef CfgWW<192, 256, 4> W9;              // wide: 96x128 wave tiles
typedef CfgWW<128, 192, 4, 4> W10;          // wide: 64x96 wave tiles, DMA 4 steps ahead
typedef CfgWW<128, 128, 4, 5> W11;          // wide: 64x64 wave tiles, DMA 5 steps ahead
typedef CfgWW<128, 64, 4, 6> W12;           // wide: 64x32 wave tiles, DMA 6 steps ahead
//              BM  BN  waves sub depth
typedef CfgFedW<16, 64, 4, 2, 5> W21;
typedef CfgFedW<32, 32, 2, 2, 5> W22;
typedef CfgFedW<48, 32, 2, 2, 4> W23;
typedef CfgFedW<32, 64, 4, 2, 4> W24;
typedef CfgFedW<48, 64, 4, 2, 4> W25;
typedef CfgFedW<80, 64, 4, 1, 5> W26;
typedef CfgFedW<64, 96, 6, 1, 5> W27;
typedef CfgFedW<96, 96, 6, 1, 4> W28;
typedef CfgFedW<96, 128, 8, 1, 4> W29;

namespace {
struct TileChoice {
  int variant;
  int64_t ns;  // modelled time of the launch
};
// The wide kernel's tiles, larger ones first, fitted to 1190 times of single GEMMs and of batches
// (M 17 to 7000, K 640 to 15360, N 1024 to 12288; 6 % rms).
constexpr LaunchModel kLaunch = {5700, 600, 690};
constexpr TileTime kTiles[] = {{7, 256, 256, W7::DEPTH, 4400, 1271}, {8, 256, 192, W8::DEPTH, 2400, 1007},
                               {10, 128, 192, W10::DEPTH, 3000, 583}, {11, 128, 128, W11::DEPTH, 2000, 444},
                               {12, 128, 64, W12::DEPTH, 1100, 297}};

// Tile choice for a problem whose tile count for a bm x bn tile is tiles(bm, bn) (one GEMM,
// or a batch walked as one tile stream), with the modelled time of that choice.
template <class Tiles, class WideOk>
TileChoice choose_variant(Tiles tiles, WideOk wide_ok, int K) {
  const int64_t cus = cu_count() > 0 ? cu_count() : 256;
  auto ns = [&](const TileTime& c) {
    return launch_ns(kLaunch, c, tiles(c.bm, c.bn), cus, (K + BKE - 1) / BKE);
  };
  if (tiles(256, 256) * 256 >= 160 * cus && wide_ok(2)) {
    // Large problems: tile area times rounds over the CUs (one persistent workgroup each), a
    // last partial round of r tiles counting 0.4 + 0.6 r/CUs, as in the w8a8 entry point.
    auto cost = [&](int bm, int bn, int pen) {
      const int64_t t = tiles(bm, bn), full = t / cus, rem = t % cus;
      return (full * 10 * cus + (rem ? 4 * cus + 6 * rem : 0)) * bm * bn * pen;
    };
    // (256 x 192 against 256 x 256, measured: 0.98 at 4608 x 3072 x 12288, 0.955 at N = 15360,
    // 1.03 at 4096 x 3072 x 12288, 1.05 at N = 9216; a penalty of 2 % puts all four on the right side)
    const TileTime& c = cost(256, 192, 102) < cost(256, 256, 100) ? kTiles[1] : kTiles[0];
    return {c.variant, ns(c)};
  }
  // Smaller problems: the tile with the least modelled time, ties to the larger one, as in the
  // w8a8 entry point: within 0.2 % of the best tile over 360 problems with K from 640 to 15360
  // (geometric mean). 2084 x 3200 x 1024 (M x N x K): 18.8 us with 256 x 192, 24.1 with 128 x 128;
  // 634 x 10176 x 8192 the other way round, 115 with 128 x 128 and 120; 512 x 4480 x 2176 27.1
  // with 128 x 128 against 33 to 40. Tiles whose prefetch depth K cannot feed are left out; without any
  // wide tile (N not a multiple of 16, very short K) the 128x128 kernel runs.
  TileChoice best = {3, INT64_MAX / 1024};  // the 128x128 kernel takes what no wide tile can
  for (const auto& c : kTiles) {
    if (!wide_ok(c.depth)) continue;
    const int64_t t = ns(c);
    if (t < best.ns) best = {c.variant, t};
  }
  return best;
}
}  // namespace

namespace {
// Whether the whole-row kernel is the better one for up to four activation rows (K <= 4096). It
// works in pieces of 1 KiB of a weight row, and each activation row costs its share of a piece
// whether the piece is full or not: with a single piece that is mostly empty, or a second one
// that is, it loses to the 16-row kernel. Measured with a different weight matrix per launch (640
// MB of them) over K 256 to 4096, N 768 to 18432, time against the 16-row kernel for M = 2 / 3 / 4:
// K 3072, N 9216 0.75 / 0.80 / 0.85; K 1792, N 768 0.78 / 0.83 / 0.87; K 1024, N 4608 0.74 / 0.80 /
// 0.83; K 768, N 2304 0.88 / 0.92 / 0.94; K 512, N 1536 1.09 / 1.15 / 1.16; K 1152, N 18432 1.01 /
// 1.21 / 1.40, N 4608 0.92 / 1.00 / 1.03; K 1280, N 4608 0.85 / 0.92 / 0.97, N 768 1.01 / 1.08 / 1.12.
bool whole_rows_better(const GemmArgs& g) {
  // (the 16-row kernel masks its loads where K is not a multiple of 128)
  if (g.M == 1 || g.K >= 1600 || (g.K >= (g.K % 128 ? 640 : 768) && g.K <= 1024)) return true;
  if (g.K > 1024) return g.N >= 1536 && g.N <= 16384 && (g.M == 2 || (g.M == 3 && g.K >= 1280));
  return g.M == 2 && g.N >= 4608 && g.K >= 320;
}

// Whether 2 to 16 rows go to the kernel with a workgroup per 32 x 32 tile instead of the 16-row
// (or whole-row) kernel. The latter's time grows with the rows and the columns, the former's with
// neither until the tiles are more than the CUs: few columns stay where they are, many do not. us,
// another weight matrix per launch, 16-row / tiles: 16 x 18432 x 5120 (M x N x K) 48.4 / 30.6, 16 x 9216 x
// 1024 8.9 / 5.0, 8 x 18432 x 3072 19.5 / 16.4, 8 x 5120 x 4608 12.6 / 12.2, 5 x 9216 x 3072 11.8 / 10.7;
// 16 x 3072 x 3072 6.9 / 8.2, 8 x 4096 x 4608 8.6 / 12.3; whole-row / tiles: 4 x 18432 x 3072 17.6 /
// 15.9, 3 x 9216 x 3072 9.1 / 10.7, 2 x 18432 x 3072 14.0 / 16.5. Over 610 shapes (K 1024 to 5120,
// N 2048 to 18432) 0.8 % off the best of the three in the geometric mean (11 % without the tiles).
// K remainders, where the 16-row kernel masks its loads: from some 41,000 outputs on. 16-row / tiles,
// M x N x K: 16 x 18432 x 3136 40.6 / 17.0, 8 x 9216 x 5056 25.8 / 14.6, 4 x 9216 x 1360 7.8 / 7.9.
bool tiles_better_for_few(const GemmArgs& g) {
  if (g.K % 128) return (int64_t)g.M * g.N > 40960;
  if (g.M >= 7) return g.N > 4500;
  if (g.M == 6) return g.N > 7000;
  if (g.M >= 4) return g.N > 8000;  // (5 x 7952 x 2944 9.1 / 9.7, 5 x 7120 x 14208 28.1 / 32.2)
  if (g.M >= 3) return g.N > 10000;
  return g.M == 2 && g.K > 4096 && g.N > 8000;
}

// More than 16 rows on the workgroup-per-tile kernel, where one round of the tiles below is not in front of it
// (choose_one_round(), others_better()): up to three tiles per CU, unless some XCDs get many more columns than others
// (Tiles32::padded), more than four per CU of an XCD (1524 x 288 x 256, M x N x K, 768 padded, 7.1 us with the wide kernel and 4.0 with
// this one) or, from K = 1024 on, three; not more than two per CU on more than 20 MB of weights (158 x 4800 x 14400 59.2 / 72.1,
// 152 x 4768 x 6320 38.7 / 49.3).
bool wavetile_better(const GemmArgs& g) {
  if (g.N % 16) return false;
  const int64_t cus = cu_count() > 0 ? cu_count() : 256;
  const Tiles32 t = tiles32(g.M, g.N);
  if (t.tiles > 3 * cus || t.padded > 4 * cus) return false;
  if (g.K > 1024 && t.padded > 3 * cus) return false;
  return t.tiles <= 2 * cus || (int64_t)g.N * g.K <= 20000000;
}

// at least `depth` K steps to prefetch, and at least 3: the epilogue operands of a tile are
// staged in LDS two steps before its end, which must be behind the first barrier of the
// tile (before it, slower waves may still be reading the previous tile's)
struct WideOk {
  bool any_k;  // the instances for K remainders
  int K, N;
  bool operator()(int depth) const { return (any_k || K >= (depth > 3 ? depth : 3) * BKE) && N % 16 == 0; }
};
int choose_tile(const GemmArgs& g) {
  return choose_variant([&](int bm, int bn) { return (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn); },
                        WideOk{!tiled_ok(g), g.K, g.N}, g.K).variant;
}
}  // namespace

// Tiles for problems that one round of them covers, with their measured round times: the kernel above (21 to 29) and the
// wide kernel's. Fitted, with a start of 3 us, to the times of 300 problems with every tile (M 17 to 3000, K 1024 to 15360, N 1024
// to 12288, at most 128 tiles of 256 x 256, weights from HBM; 7 % rms): of those that one round covers it takes one that is
// 0.7 % off the best (geometric mean), 0.88 of the time that the choice among the other tiles gives. With K remainders
// from K = 320 on 0.86 (113 problems).
constexpr LaunchModel kOneLaunch = {2960, 852, 852};
constexpr TileTime kOneRound[] = {{8, 256, 192, W8::DEPTH, 3218, 912}, {10, 128, 192, W10::DEPTH, 3134, 560}, {11, 128, 128, W11::DEPTH, 2395, 424},
                                  {12, 128, 64, W12::DEPTH, 1467, 299},  {29, 96, 128, 0, 2087, 389},  {28, 96, 96, 0, 1366, 332},
                                  {27, 64, 96, 0, 953, 287},    {26, 80, 64, 0, 686, 252},    {25, 48, 64, 0, 1025, 178},
                                  {24, 32, 64, 0, 593, 163},    {23, 48, 32, 0, 362, 142},    {21, 16, 64, 0, 227, 125},
                                  {22, 32, 32, 0, 0, 105}};

// Whether what the other rules choose (a tile of the wide kernel, or 32 x 32 ones) is the better one where one round of
// `tile` is modelled as the shortest. us, theirs / `tile`, M x N x K.
// In place of up to two 32 x 32 tiles per CU of every XCD (Tiles32::padded; where some get three, those win next to never: 2489 x 256 x 1248
// 12.9 / 8.6, 1626 x 304 x 816 9.1 / 6.4):
// - 48 x 32 (23) for up to 48 rows to K = 1472 (41 x 5776 x 1104 6.8 / 7.2), 2448 with rows of weights that are no whole lines (42 x
//   7936 x 2128 10.2 / 10.7), and with K remainders for up to 44 rows (41 x 5776 x 9040 26.0 / 28.8). Also where the last tile's rows are
//   full and few CUs get a second 32 x 32: to 264 tiles (89 x 2768 x 12144, 261, 29.4 / 35.4; 96 x 2976 x 896, 279, 6.7 / 6.0), with long
//   K remainders to 288 (282 x 928 x 4272 12.6 / 14.9; 91 x 3008 x 10656, 282, of two rows of 48 x 32, 45.8 / 31.2).
// - 32 x 64 (24) to K = 1152 of up to 64 rows (20 x 8832 x 1088 6.9 / 7.2), of four 32-row tiles and their multiples on more than 1328
//   columns (103 x 3008 x 672 5.5 / 5.9), and beyond 730 rows; 200 x 2800 x 1104 11.4 / 10.5, 127 x 3072 x 4160 16.0 / 15.2.
// And of up to three per CU: 80 x 64 (26) for up to 128 rows and K = 1152 (98 x 5568 x 1136 8.3 / 9.1; 123 x 6112 x 1312 11.1 / 10.2).
// In place of one round of the wide kernel's tiles, whose rows beyond M are all the same row and cost next to nothing:
// - 64 x 96 (27) where the last tile of either has 41 to 64 rows, 128 x 64 the emptier one, from K = 2560 on: 178 x 8160 x 14896 91 / 105,
//   177 x 6144 x 13952 61 / 67; 248 x 5376 x 6016 36.6 / 33.3.
// - 80 x 64 (26) with its last tile full and up to 32 rows in 128 x 64's, from K = 4096 on, to 3.5 tiles of 32 x 32 per CU: 159 x 5312 x
//   14336 64 / 66.
// - 96 x 128 (29) where the last tile of 128 x 128 is the emptier one, K no multiple of 128 and not short: 1051 x 2336 x 8304 70 / 83; 1391 x
//   1888 x 5984 (111 of 128 rows) 60 / 51, 1331 x 2256 x 576 11.6 / 9.7.
// Drawn problems for which `tile` (23, 24, 26, 27, 29) differs from the other rules' one: what this takes is 0.49, 0.22, 0.10, 0.21 and
// 0.51 % off the better of both (geometric mean; `tile` always: 1.35, 1.10, 0.27, 1.01 and 1.51) and slower than theirs by more
// than 3 % for 76 of 1503, 42 of 1852, 17 of 2380, 9 of 1142 and 50 of 1400, 19 % the worst (`tile` always: 260, 293, 85, 152 and 243). Rules
// for 48 x 64 (25) and 96 x 96 (28) were measured to lose more than they give.
static bool others_better(const GemmArgs& g, int tile, int64_t cus) {
  auto rest = [&](int rows) { return (g.M - 1) % rows + 1; };  // rows of the last tile
  const Tiles32 t = tiles32(g.M, g.N);
  const bool two = t.padded <= 2 * cus;
  switch (tile) {
    case 23:
      if (!two) return false;
      if (g.M <= 48) {
        if (g.K > (g.K % 128 ? 2448 : 1472) && (g.K % BKE == 0 || g.M > 44)) return false;
      } else if (g.N <= 448 || rest(48) <= 34 || (t.tiles * 32 > 33 * cus && (g.K % BKE == 0 || g.K <= 2448 || g.M <= 96 || t.padded * 8 > 9 * cus))) {
        return false;
      }
      return wavetile_better(g);
    case 24:
      return two && g.K <= 1152 && (g.M <= 64 || g.M > 730 || ((g.M + 31) / 32 % 4 == 0 && g.N > 1328)) && wavetile_better(g);
    case 26:
      if (g.K > 4096) return rest(80) > 64 && rest(128) <= 32 && t.padded * 2 <= 7 * cus && choose_tile(g) == 12;
      return g.K <= 1152 && g.M <= 128 && wavetile_better(g);
    case 27: return rest(128) > 40 && rest(128) <= 64 && g.K > 2528 && choose_tile(g) == 12;
    case 29:
      return rest(128) <= 64 && rest(96) > rest(128) && g.K % 128 && g.K > (g.K % BKE ? 1024 : 832) && choose_tile(g) == 11;
    default: return false;
  }
}

// The tile of a problem that one round covers, -1 if there is none. Shorter K than 5 steps stays with the other rules (127 x
// 5584 x 192, M x N x K, 3.8 us and 5.2 with this one), than 10 where those take two or three 32 x 32 tiles per CU (53 x 6016 x
// 320 4.0 and 4.6; from there to K = 1024 0.96 of the time of those, from K = 1600 on 0.81).
static int choose_one_round(const GemmArgs& g) {
  if (g.N % 16 || g.K < 5 * BKE) return -1;
  const int64_t cus = cu_count() > 0 ? cu_count() : 256;
  if (g.K < 10 * BKE && tiles32(g.M, g.N).tiles > cus && wavetile_better(g)) return -1;
  int best = -1;
  int64_t time = INT64_MAX;
  for (const auto& c : kOneRound) {
    const int64_t tiles = (int64_t)((g.M + c.bm - 1) / c.bm) * ((g.N + c.bn - 1) / c.bn);
    if (tiles > cus || (c.variant < 21 && !WideOk{!tiled_ok(g), g.K, g.N}(c.depth))) continue;
    const int64_t t = launch_ns(kOneLaunch, c, tiles, cus, g.K / BKE);
    if (t < time) best = c.variant, time = t;
  }
  // One round of 256 x 192 tiles in place of two of 128 x 128: not where the weights' rows are whole lines of 128 bytes. us, two rounds / one, M x N x K: 616 x 12224 x 8064 119 / 132, 1152 x 6624 x
  // 11392 164 / 179 (36 such problems: 1.06 of the time, none faster); 630 x 12288 x 4800 89 / 82 (0.97 over 38 with K a multiple
  // of 64, 0.85 over 225 with K remainders).
  if (best < 21 && g.K % 128 == 0) return -1;
  return best >= 21 && others_better(g, best, cus) ? -1 : best;
}

// Up to 16 rows on tiles (tiles_better_for_few()): the kernel above in place of the 32 x 32 tiles, whose sums it gives bit for
// bit: 0.82 of their time where 32 x 32 tiles are one round, 0.96 with 16 x 64 (122 problems, none slower; 16 x 96 and
// 16 x 128: 1.13 and 1.49).
static int choose_few(const GemmArgs& g) {
  const int64_t cus = cu_count() > 0 ? cu_count() : 256;
  if (g.K < 5 * BKE) return 13;
  return (g.N + 31) / 32 <= cus ? 22 : (g.N + 63) / 64 <= cus ? 21 : 13;
}

int launch_gemm_w8a16_fed(const GemmArgs& g, int variant, hipStream_t stream) {
  switch (variant) {
    case 21: return launch_fed<W21>(g, stream);
    case 22: return launch_fed<W22>(g, stream);
    case 23: return launch_fed<W23>(g, stream);
    case 24: return launch_fed<W24>(g, stream);
    case 25: return launch_fed<W25>(g, stream);
    case 26: return launch_fed<W26>(g, stream);
    case 27: return launch_fed<W27>(g, stream);
    case 28: return launch_fed<W28>(g, stream);
    default: return launch_fed<W29>(g, stream);
  }
}

// The kernel for a problem: 100 for any shape and alignment, 51 whole rows (up to four), 50 up to 16 rows, 21 to 29 a tile of
// which one round covers it, 13 a workgroup per 32 x 32 tile, else a tile of the wide kernel (K remainders: of its
// instances for them) or of the tiled one.
int choose_gemm_w8a16(const GemmArgs& g) {
  if (!aligned_ok(g)) return 100;
  const bool few_on_tiles = g.M <= 16 && g.N % 16 == 0 && tiles_better_for_few(g);
  if (g.M <= 4 && g.K <= 4096 && whole_rows_better(g) && (g.K % 128 || !few_on_tiles)) return 51;
  if (g.M <= 16 && !few_on_tiles) return 50;
  if (few_on_tiles) return choose_few(g);
  // what is left of K remainders is for the wide kernel, which stores 16 columns per lane
  if (!tiled_ok(g) && g.N % 16 != 0) return 100;
  if (const int one = choose_one_round(g); one >= 0) return one;
  return wavetile_better(g) ? 13 : choose_tile(g);
}

int launch_gemm_w8a16(const GemmArgs& g, int variant, hipStream_t stream) {
  const bool k_tail = !tiled_ok(g);  // K not a whole number of steps
  if (variant < 0) variant = choose_gemm_w8a16(g);
  auto launch_generic = [&]() {
    dim3 grid((g.N + 15) / 16, (g.M + 15) / 16);
    hipLaunchKernelGGL(gemm_w8a16_generic, grid, dim3(256), 0, stream, g);
    return 0;
  };
  if (!aligned_ok(g) || variant == 100) return launch_generic();
  if (g.M <= 4 && g.K <= 4096 && variant == 51) {
    // (aligned_ok has checked the alignment of the operands and of lda and ldb)
    switch ((g.K + 1023) / 1024) {
      case 1: launch_rows_chk<1>(g, stream); break;
      case 2: launch_rows_chk<2>(g, stream); break;
      case 3: launch_rows_chk<3>(g, stream); break;
      default: launch_rows_chk<4>(g, stream); break;
    }
    return 0;
  }
  if (variant == 50) {
    if (g.M > 16) {
      set_error("cdit_w8a16_gemm: the skinny kernel takes M <= 16");
      return CDIT_EINVAL;
    }
    if (g.K % 128) {
      hipLaunchKernelGGL(gemm_w8a16_skinny<true>, dim3((g.N + 15) / 16), dim3(256), 0, stream, g);
    } else {
      hipLaunchKernelGGL(gemm_w8a16_skinny<false>, dim3((g.N + 15) / 16), dim3(256), 0, stream, g);
    }
    return 0;
  }
  if (k_tail && g.N % 16 != 0) return launch_generic();
  if (variant >= 21 && variant <= 29 && g.N % 16 == 0) return launch_gemm_w8a16_fed(g, variant, stream);
  if (variant == 13 && g.N % 16 == 0) return launch_wavetile(g, stream);
  const WideOk wide_ok{k_tail, g.K, g.N};
  if (k_tail && (variant < 7 || variant > 12)) variant = choose_tile(g);
  if (k_tail) {  // the KTAIL instances of the wide kernel take any K
    switch (variant) {
      case 7: return launch_wide<W7, true>(g, stream);
      case 8: return launch_wide<W8, true>(g, stream);
      case 9: return launch_wide<W9, true>(g, stream);
      case 10: return launch_wide<W10, true>(g, stream);
      case 11: return launch_wide<W11, true>(g, stream);
      default: return launch_wide<W12, true>(g, stream);
    }
  }
  switch (variant) {
    case 0: return launch_tiled<W0>(g, stream);
    case 3: return launch_tiled<W3>(g, stream);
    case 7: return wide_ok(W7::DEPTH) ? launch_wide<W7>(g, stream) : launch_tiled<W3>(g, stream);
    case 8: return wide_ok(W8::DEPTH) ? launch_wide<W8>(g, stream) : launch_tiled<W3>(g, stream);
    case 9: return wide_ok(W9::DEPTH) ? launch_wide<W9>(g, stream) : launch_tiled<W3>(g, stream);
    case 10: return wide_ok(W10::DEPTH) ? launch_wide<W10>(g, stream) : launch_tiled<W3>(g, stream);
    case 11: return wide_ok(W11::DEPTH) ? launch_wide<W11>(g, stream) : launch_tiled<W3>(g, stream);
    case 12: return wide_ok(W12::DEPTH) ? launch_wide<W12>(g, stream) : launch_tiled<W3>(g, stream);
    default:
      set_error("cdit_w8a16_gemm: unknown kernel variant %d", variant);
      return CDIT_EINVAL;
  }
}

// The batch as one launch (or, where the cost model says so, one launch per activation).
// Returns 0 when launched, -1 when the batch is not taken (the caller then runs the members
// one by one), a CDIT_E* code on error.
int launch_gemm_w8a16_grouped(const GemmArgs& common, const GemmGroup& grp, int variant,
                              hipStream_t stream) {
  if (grp.count < 2 || grp.count > kMaxGroup || grp.acts < 1 || grp.acts > kMaxActs ||
      common.out_dtype != CDIT_DT_BF16)
    return -1;
  bool n16 = true;
  for (int s = 0; s < grp.acts; ++s) {
    if (grp.M[s] <= 16 || grp.first_member[s + 1] <= grp.first_member[s]) return -1;
    for (int p = grp.first_member[s]; p < grp.first_member[s + 1]; ++p) {
      GemmArgs g = common;
      g.a = grp.a[s];
      g.M = grp.M[s];
      g.b = grp.b[p];
      g.b_scale = grp.b_scale[p];
      g.bias = grp.bias[p];
      g.out = grp.out[p];
      g.N = grp.N[p];
      g.ldo = grp.ldo[p];
      if (!tiled_ok(g) || g.N <= 0) return -1;
      n16 = n16 && g.N % 16 == 0;
    }
  }
  const WideOk wide_ok{false, common.K, n16 ? 16 : 1};
  auto tiles = [&](int bm, int bn) {
    int64_t t = 0;
    for (int s = 0; s < grp.acts; ++s) {
      int64_t cols = 0;
      for (int p = grp.first_member[s]; p < grp.first_member[s + 1]; ++p) cols += (grp.N[p] + bn - 1) / bn;
      t += (int64_t)((grp.M[s] + bm - 1) / bm) * cols;
    }
    return t;
  };
  if (variant < 0) {
    const TileChoice whole = choose_variant(tiles, wide_ok, common.K);
    variant = whole.variant;
    if (grp.acts > 1) {
      // one tile stream against one launch per activation, as in the w8a8 launcher: a small
      // activation can push a batch that filled whole rounds into one more, nearly empty one
      // (1104 + 100 rows, three members, K 2816: 63 us as one launch, 71 as two). As there, one round of
      // smaller tiles is not priced: over 150 joint-block stages of 17 to 512 text rows 0.4 % slower than the better
      // form, 8 more than 3 % (2254 + 106 rows, K 10240, N 2560 147 us as one launch, 131 as two)
      int64_t apart = 0;
      for (int s = 0; s < grp.acts; ++s) {
        auto tiles_s = [&](int bm, int bn) {
          int64_t cols = 0;
          for (int p = grp.first_member[s]; p < grp.first_member[s + 1]; ++p) cols += (grp.N[p] + bn - 1) / bn;
          return (int64_t)((grp.M[s] + bm - 1) / bm) * cols;
        };
        apart += choose_variant(tiles_s, wide_ok, common.K).ns;
      }
      if (apart * 100 < whole.ns * 98) {
        for (int s = 0; s < grp.acts; ++s) {
          GemmGroup one = {};
          one.acts = 1;
          one.count = grp.first_member[s + 1] - grp.first_member[s];
          one.a[0] = grp.a[s];
          one.M[0] = grp.M[s];
          one.first_member[0] = 0;
          one.first_member[1] = one.count;
          for (int p = 0; p < one.count; ++p) {
            const int src = grp.first_member[s] + p;
            one.b[p] = grp.b[src];
            one.b_scale[p] = grp.b_scale[src];
            one.bias[p] = grp.bias[src];
            one.out[p] = grp.out[src];
            one.N[p] = grp.N[src];
            one.ldo[p] = grp.ldo[src];
            one.epilogue[p] = grp.epilogue[src];
          }
          int rc = one.count >= 2 ? launch_gemm_w8a16_grouped(common, one, -1, stream) : -1;
          if (rc > 0) return rc;
          if (rc == 0) continue;
          for (int p = 0; p < one.count; ++p) {  // a single member, or a group that is not taken
            GemmArgs g = common;
            g.a = one.a[0];
            g.M = one.M[0];
            g.b = one.b[p];
            g.b_scale = one.b_scale[p];
            g.bias = one.bias[p];
            g.out = one.out[p];
            g.N = one.N[p];
            g.ldo = one.ldo[p];
            g.epilogue = one.epilogue[p];
            if ((rc = launch_gemm_w8a16(g, -1, stream))) return rc;
          }
        }
        return 0;
      }
    }
  }
  switch (variant) {
    case 7: return wide_ok(W7::DEPTH) ? launch_wide_grouped<W7>(common, grp, stream) : -1;
    case 8: return wide_ok(W8::DEPTH) ? launch_wide_grouped<W8>(common, grp, stream) : -1;
    case 9: return wide_ok(W9::DEPTH) ? launch_wide_grouped<W9>(common, grp, stream) : -1;
    case 10: return wide_ok(W10::DEPTH) ? launch_wide_grouped<W10>(common, grp, stream) : -1;
    case 11: return wide_ok(W11::DEPTH) ? launch_wide_grouped<W11>(common, grp, stream) : -1;
    case 12: return wide_ok(W12::DEPTH) ? launch_wide_grouped<W12>(common, grp, stream) : -1;
    default: return -1;  // the kernels without a tile stream have no grouped form
  }
}

}  // namespace cdit
