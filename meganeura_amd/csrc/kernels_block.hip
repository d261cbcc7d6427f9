// Blocked dequant-GEMM on the matrix cores for many rows: C[M,N] = A[M,K] x W (+ D), f32 or fp16 activations
// (prefill, and decode batches of more than some 32 rows on large weights).
//
// The arithmetic is that of the other tiled kernels (raw quants as the B operand of the matrix
// instructions, block scales on their results, block minima as a product of their own; Q8 with f32 activations
// multiplies signed bytes and has no such product), so the vector
// ALU owes 16 multiply-adds per 32 x 32 outputs and quant block whatever the tiling; with the matrix
// instructions (two of 32 cycles; four with f32 activations, which enter as fp16 pairs hi + lo) that is
// the bound: measured on one SIMD, v_mfma_f32_32x32x16_f16 occupies its pipe for 32 cycles and the vector
// issue port for about 8, a v_fma_f32 the port for 4, and two waves overlap the two almost fully.  The
// kernels this one takes over from ran far from it: a 32-row tile per wave unpacks the quants for
// every tile, stages activations through registers in every column group and keeps the matrix pipe
// 16 % busy.  What is different here:
//   * a wave owns 32 RT x 64 outputs (up to 128 x 64: 128 accumulator registers), so the 14 instructions that
//     unpack a column tile's quants serve RT row tiles, and the tiles' multiply-adds are woven between
//     the next tile's matrix instructions by hand;
//   * activations and quants travel from memory into LDS without touching registers (buffer loads with
//     the LDS bit), several substeps ahead, in rings; one barrier per substep.  What a lane reads
//     together is spread over the banks by an exclusive-or of its 16-byte unit with the row;
//   * everything the multiplication wants to know about the activations is worked out once per call by
//     a small launch in front (prepare_*): the blocks' means, and for f32 the fp16 pairs on a scale per
//     row.  One scale for the whole row, so that no accumulator is rescaled on the way: a slice of
//     256 elements that would be held in fewer bits than the tiled kernels hold it gets its own, and the
//     waves that meet such a row move their sums from scale to scale;
//   * K parts for different workgroups, where the tiles do not fill the chip, meet in the workspace and are added
//     in part order by a third launch.
// Measured (weights from memory; before -> now, us, Q4; machines differ by 4 %): fp16 2048 x 4096 x 14336 589 -> 263 (914
// TFLOP/s), f32 the same 1034 -> 444; f32 512 x 4096 x 14336 295 -> 115; f32 77 x 4096 x 14336 82 -> 38, 77 x 14336 x
// 4096 98 -> 40.  What remains on the large call: 448 workgroups on 256 CUs are 1.75 rounds, and a SIMD needs 1.3
// times its issue cycles (LDS and barrier waits).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <utility>

#include "kernels_operand.hip.h"

namespace mgn {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// f(0), f(1), .. f(N - 1) with compile-time indices
template <typename F, int... I>
__device__ __forceinline__ void static_for_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(f, std::make_integer_sequence<int, N>{});
}

constexpr int kCT = 2;  // column tiles of 32 columns per wave

constexpr int stage_blocks(int fmt) { return fmt == MGN_FMT_Q4 ? 4 : 2; }  // 64 bytes of quants per column

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// 64 x 16 bytes from memory straight into LDS: lane i's bytes land at lds + 16 i.  (In assembly, with the
// waits counted by hand: the compiler waits for every such load before any LDS read that might alias it.  Nor does
// it look in here for the five wait states that a load must keep from the vector unit's write of a scalar it
// reads, v_readfirstlane's and a spilled scalar's v_readlane among them: the move and the nop are these five.)
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t src, uint32_t lane_off, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(lane_off), "s"(src), "s"(__builtin_amdgcn_readfirstlane(off)) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// one dword of nibbles -> 8 fp16 in element order, each n * 2^-20
__device__ __forceinline__ half8 nibbles_in_order(uint32_t w) {
  const uint32_t ev = (w << 4) & 0xF0F0F0F0u, od = w & 0xF0F0F0F0u;
  return as_half8(__builtin_amdgcn_perm(od, ev, 0x0c040c00u), __builtin_amdgcn_perm(od, ev, 0x0c050c01u),
                  __builtin_amdgcn_perm(od, ev, 0x0c060c02u), __builtin_amdgcn_perm(od, ev, 0x0c070c03u));
}

// Q8 with f32 activations multiplies the bytes as they are; the other forms leave an additive part (Q4's minima, the
// bias of Q8's bytes) to a product of the blocks' means.  The bias of 128 is several times the bytes: it enters the
// running sum and leaves it again at every stage, and the sum's roundings are those of its size.  Four packed subtractions
// per operand keep it out, which the vector unit has room for with four matrix instructions per tile and block (not with
// fp16's two).  Error against f64 (2-norm, normal activations; the tiled kernels, biased here, signed) and time (biased,
// signed): 2048 x 14336 x 4096 9.4e-7, 1.03e-6, 2.8e-7, 560 -> 549 us; 77 x 4096 x 14336 7.1e-7, 7.2e-7, 1.1e-7,
// 43.8 -> 41.9 us.
constexpr bool has_additive(int fmt, bool f32a) { return fmt == MGN_FMT_Q4 || !f32a; }

// two dwords of int8 -> 8 fp16, the bytes' own values: 1024 + (q + 128) as bits, less 1152
__device__ __forceinline__ half8 signed_bytes_to_operand(uint32_t w0, uint32_t w1) {
  const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u, k1024 = 0x64646464u;
  const half8 v = as_half8(__builtin_amdgcn_perm(k1024, u0, 0x04010400u), __builtin_amdgcn_perm(k1024, u0, 0x04030402u),
                           __builtin_amdgcn_perm(k1024, u1, 0x04010400u), __builtin_amdgcn_perm(k1024, u1, 0x04030402u));
  return v - (half8)((_Float16)1152.0f);
}

// the j-th of NM equal shares of acc += dq * d
template <int NM, int j>
__device__ __forceinline__ void scale_part(floatx16& acc, const floatx16& d, float dq) {
  static_for<16 / NM>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = j * (16 / NM) + I;
    acc[i] = __fmaf_rn(dq, d[i], acc[i]);
  });
}

struct BlockArgs {
  const void* a;      // fp16 activations, or the prepared f32 ones
  const void* means;  // [stages][mpad]{hi x SB, lo x SB}
  const float* inv;   // [slices][mpad] inverse scales (f32 activations)
  const float* row_scale;  // [mpad] the inverse scale of a row's last slice; NaN for a row that holds a magnitude of 2^100 or more
  const uint32_t* mixed;  // [mpad] nonzero: the row's slices do not share one scale
  const void* meta;
  const void* quants;
  uint32_t a_pitch, a_bytes, quant_bytes, meta_bytes, means_bytes;
  uint32_t m, mpad, n, bpc, stages, rowgroups, colgroups, parts;
  uint32_t add_hi, add_lo;  // fp16 pairs: 2^lift and 2^(lift - 11)
  float unit;               // 2^-lift times the inverse operand scale
  float dscale;             // what a block scale is multiplied by: operand scale * 2^lift
  const float* dres;
  float* c;
  float* partial;  // [parts][m][n] when parts > 1
  uint32_t epilogue;
};

__device__ __forceinline__ float group_max32(float v) {
  v = fmaxf(v, dpp_move<kDppQuadXor1>(v));
  v = fmaxf(v, dpp_move<kDppQuadXor2>(v));
  v = fmaxf(v, dpp_move<kDppRowHalfMirror>(v));
  v = fmaxf(v, dpp_move<kDppRowMirror>(v));
  return fmaxf(v, __shfl_xor(v, 16, 64));
}

// Geometry of a workgroup: WM x WN waves side by side, each RT row tiles of 32 rows x 64 columns, and
// WK streams of them that take the stages (64 bytes of quants per column) in turn; substeps of SUBB
// blocks of activations, requested PD substeps ahead; stages requested SD stages ahead.
template <int FMT, bool F32A, int RT, int WM, int WN, int WK, int SUBB, int PD, int SD>
struct BlockShape {
  static constexpr int SB = stage_blocks(FMT);
  static constexpr int NSUB = SB / SUBB;
  static constexpr int WAVES = WM * WN * WK;
  static constexpr int ROWS = WM * RT * 32, COLS = WN * kCT * 32;
  static constexpr int PANELS = SUBB * (F32A ? 128 : 64) / 128;  // 128 bytes of activations per row each
  static constexpr int ARING = PD + 1, SRING = SD + 1;
  static constexpr uint32_t A_BYTES = WK * PANELS * ROWS * 128u, B_BYTES = WK * COLS * 64u, M_BYTES = WK * COLS * 16u;
  static constexpr uint32_t MEAN_STREAM = has_additive(FMT, F32A) ? (ROWS * SB * 4 + 1023) / 1024 * 1024 : 0, S_BYTES = WK * MEAN_STREAM;
  static constexpr uint32_t STAGE_BYTES = B_BYTES + M_BYTES + S_BYTES;
  static constexpr int NA = (int)(A_BYTES / 1024), NST = (int)(STAGE_BYTES / 1024);  // loads of 1 KiB
  static constexpr int NAW = (NA + WAVES - 1) / WAVES, NSTW = (NST + WAVES - 1) / WAVES;
  static constexpr size_t PIPE = (size_t)ARING * A_BYTES + (size_t)SRING * STAGE_BYTES;
  static constexpr size_t RED = WK > 1 ? (size_t)WAVES * RT * 4096 : 0, STRIP = (size_t)WAVES * 4096;
  static constexpr size_t LDS = PIPE > RED ? (PIPE > STRIP ? PIPE : STRIP) : (RED > STRIP ? RED : STRIP);
  // A wave's loads in issue order: in substep i the activations of substep i + PD, then, where it is a
  // stage's first, the stage SD ahead, dealt over the substep's tiles.  The substep's barrier stands in front of
  // tile TURN of its last block: by then a wave holds all operands of substep i that it has still to multiply, and
  // what it reads from there to the next barrier is substep i + 1's, and that one's stage.  So these must have
  // landed; the loads issued after the last of them may be in flight.  (With the barrier behind the last tile, the
  // next substep's first operands had to have landed a barrier earlier: at PD = 2 the loads of the very substep that
  // ends, and their whole latency was waited for.  us, weights from memory, both libraries in turn: Q4 fp16 2048 x 4096 x 14336
  // 291 -> 263, 512 x 4096 x 14336 85 -> 79, f32 2048 471 -> 444; Q8 f32 1024 x 4096 x 14336 260 -> 230.  Over 364 sizes, medians by
  // workgroup, 0.88 to 1.00 of the time at PD = 2 and 0.96 to 1.004 where PD is 3 or 4 already; single sizes up to 1.02: Q4 64 x 256
  // f32, K of 160 to 640, and 32 x 256 fp16, K of 320 to 416.)
  // f32 activations hold the operands of one row tile: the last ones have been read when its first column tile begins, and a
  // wave may turn there or a tile later.  With PD = 3 the next substep's operands have landed by then, and what the later turn
  // waits for is the next quants, read behind the barrier and unpacked at the end of the same tile: workgroups of two row tiles per
  // wave, medians of 8 to 22 sizes, barrier behind the last tile = 1, in front of it, a tile earlier: Q4 64 x 256 1.014, 1.004,
  // of two streams 1.004, 0.991, 128 x 256 1.001, 0.980; Q8 64 x 256 1.020, 0.998, 128 x 256 1.006, 0.981 (444 x 2176 x 8192 52.3, 54.4,
  // 52.6 us).  With one row tile the earlier turn is the whole substep's wait (Q4 32 x 256 0.988, 0.998; 64 x 128 0.977, 0.987).  At
  // PD = 2 both ways: 0.5 to 1 % faster with 96 to 256 rows, but Q8 96 x 256 of two streams 0.915, 0.932.
  // The barrier stays behind the last tile, with the next block's operands landed as well, where four waves with nothing to
  // spare (PD = 2) have a CU to themselves: one wave on each SIMD, and nobody works while it waits for what it may read only now.
  // That is Q8 with fp16 activations, us, behind, in front: 96 x 256 213 x 1472 x 20992 36.3, 38.1, 298 x 1376 x 13824 36.0, 37.6, 64 x 256
  // 444 x 1152 x 6656 25.7, 26.1; medians of 21 and 12 sizes 1, 1.010 and 1, 0.997.  (Q8 64 x 256 with f32 activations and PD = 3 is level.)
  static constexpr int TILES = RT * kCT, SLOTS = SUBB * TILES;
  static constexpr bool ALONE = WAVES == 4 && PD == 2 && 2 * LDS > 160 * 1024;
  static constexpr int TURN = ALONE ? TILES : F32A && (PD == 2 || RT == 1) ? TILES - 1 : TILES - 2;
  static constexpr int AHEAD = ALONE ? 2 : 1;  // at its barrier, substep i + AHEAD's operands must have landed
  static constexpr int issued(int i) { return NAW + ((i + 64 * NSUB) % NSUB == 0 ? NSTW : 0); }
  static constexpr int issued_before(int i, int slot) { return slot * issued(i) / SLOTS; }  // of them in front of tile `slot` of the substep
  static constexpr int since(int from, int to) {
    int n = 0;
    for (int i = from; i <= to; i++) n += issued(i);
    return n;
  }
  static constexpr int stage_of(int i) { return (i + 64 * NSUB) / NSUB - 64; }
  static constexpr int requested(int i) { return (stage_of(i) - SD) * NSUB; }  // the substep that asks for substep i's stage
  static constexpr int behind_a(int i) { return (i - PD + 64 * NSUB) % NSUB == 0 ? NSTW : 0; }  // loads behind substep i's activations in the substep that asks for them
  static constexpr int in_flight(int i) {
    const int here = issued_before(i, (SUBB - 1) * TILES + TURN), of = i + AHEAD;
    const int after_a = behind_a(of) + (of - PD < i ? since(of - PD + 1, i - 1) + here : 0);
    const int after_stage = since(requested(of) + 1, i - 1) + here;
    return after_a < after_stage ? after_a : after_stage;
  }
  // In front of the loop, in the same order, what the substeps before the first would have asked for: landed must be
  // the activations and the stage of the substeps that are read up to the first barrier.
  static constexpr int FIRST = -(PD > SD * NSUB ? PD : SD * NSUB);
  static constexpr int in_flight_first() {
    const int of = AHEAD - 1, after_a = behind_a(of) + since(of - PD + 1, -1), after_stage = since(requested(of) + 1, -1);
    return after_a < after_stage ? after_a : after_stage;
  }
  static_assert(PD >= 2 && requested(NSUB - 1 + AHEAD) < NSUB - 1, "what a substep waits for has been requested in whole");

  // The requests of three stages one by one, in the order and number in which the kernel issues them: whether at each of
  // its waits what may still be in flight holds none that must have landed.
  static constexpr bool waits_suffice() {
    int sent = 0, a_end[PD + 4 * NSUB] = {}, st_end[SD + 4] = {};  // requests up to and with the last of a substep's activations, of a stage
    for (int i = FIRST; i < 3 * NSUB; i++) {
      const bool first = (i + 64 * NSUB) % NSUB == 0 && stage_of(i) + SD >= 0;
      auto landed = [&](int in_flight, int sub) { return sent - in_flight >= a_end[sub] && sent - in_flight >= st_end[sub / NSUB]; };
      if (i == 0 && !landed(in_flight_first(), AHEAD - 1)) return false;
      const int all = i < 0 ? (i + PD >= 0 ? NAW : 0) + (first ? NSTW : 0) : issued_before(i, SLOTS);
      const int at_turn = i < 0 ? all : issued_before(i, (SUBB - 1) * TILES + TURN);
      const int before = sent;
      if (i + PD >= 0) a_end[i + PD] = before + NAW;
      if (first) st_end[stage_of(i) + SD] = before + all;
      sent = before + at_turn;
      if (i >= 0 && !landed(in_flight(i % NSUB), i + AHEAD)) return false;
      sent = before + all;
    }
    return true;
  }
};

template <int FMT, bool F32A, int RT, int WM, int WN, int WK, int SUBB, int PD, int SD>
__global__ __launch_bounds__(64 * WM * WN * WK, 2) void block_kernel(BlockArgs x) {
  using S = BlockShape<FMT, F32A, RT, WM, WN, WK, SUBB, PD, SD>;
  constexpr int SB = S::SB, NSUB = S::NSUB, ROWS = S::ROWS, COLS = S::COLS, PANELS = S::PANELS, ARING = S::ARING, SRING = S::SRING;
  constexpr int NAW = S::NAW, NSTW = S::NSTW;
  constexpr uint32_t A_BYTES = S::A_BYTES, B_BYTES = S::B_BYTES, M_BYTES = S::M_BYTES, STAGE_BYTES = S::STAGE_BYTES;
  constexpr uint32_t MEAN_STREAM = S::MEAN_STREAM;
  constexpr int QB = FMT == MGN_FMT_Q4 ? 16 : 32, MB = FMT == MGN_FMT_Q4 ? 4 : 2;
  constexpr int NM = F32A ? 4 : 2;             // matrix instructions per tile and block
  constexpr int TILES = S::TILES;
  static_assert(F32A || SUBB % 2 == 0, "fp16 activations: two blocks per 128 bytes");
  extern __shared__ uint4 lds4[];
  uint8_t* const lds = (uint8_t*)lds4;
  uint8_t* const lds_st = lds + ARING * A_BYTES;  // [SRING]{quants, block constants, means}
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t ks = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  const uint32_t c = lane & 31, h = lane >> 5;

  // The eight XCDs take workgroups in turn: each gets a contiguous run of all parts' tiles, row groups first, then column
  // groups, then parts.  (Before, an eighth of the tiles, rounded up, with all their parts: plans are made for full
  // rounds of the CUs, and that rounding was one more round on some XCDs for every sixth call that comes here.  us: f32 Q8 96 x 8544 x
  // 2606, 11 tiles in 17 parts, 45.4 -> 29.0, 508 x 3456 x 5248, 84 in 3, 85.6 -> 59.0, Q4 118 x 13056 x 1600 35.7 -> 28.8, fp16 641 x 9280 x
  // 4274 137 -> 95; 16 calls whose tiles divide by 8 0.97 to 1.017, median 0.997.  With as many workgroups launched as that takes, 192
  // for those 11 tiles where 272 had been, 36 ragged calls 0.98 to 1.02, median 0.996, 8 whose tiles divide by 8 0.97 to 1.01: those that returned at once cost nothing that shows.)
  const uint32_t tiles = x.rowgroups * x.colgroups;
  const uint32_t all = tiles * x.parts, per = (all + 7) / 8;
  const uint32_t at = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (at >= all) return;  // (a grid of 8 * per workgroups)
  const uint32_t part = at / tiles, tile = at - part * tiles;
  const uint32_t rg = tile % x.rowgroups, cg = tile / x.rowgroups;
  const uint32_t row0 = rg * ROWS, col0 = cg * COLS;

  // this part's stages, dealt to the WK streams in turn
  const uint32_t spp = (x.stages + x.parts - 1) / x.parts;
  const uint32_t st0 = part * spp, st1 = min(st0 + spp, x.stages);
  const uint32_t iters = (st1 - st0 + WK - 1) / WK;

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)x.a, 0, x.a_bytes, 0x00020000);
  // A wave's share of the loads.  Activations: load q brings 8 rows of one panel; in LDS a row's unit u
  // (16 bytes) lies at u ^ (row / 2 % 8), so that the operand reads of eight rows meet no bank twice.
  // Stage: 16 columns of quants (unit u of a column at u ^ (column / 4 % 4)), 64 columns of constants, or
  // 1 KiB of means, by load number.
  uint32_t a_off[NAW], st_off[NSTW];
#pragma unroll
  for (int j = 0; j < NAW; j++) {
    const uint32_t q = min(wave * NAW + j, (uint32_t)S::NA - 1) % (ROWS / 8);
    const uint32_t row = q * 8 + (lane >> 3);
    a_off[j] = min(row0 + row, x.m - 1) * x.a_pitch + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
  }
  // (what a stage load reads is settled here, per load, so that the loop issues it without a branch)
  constexpr uint32_t NBL = B_BYTES / 1024, NML = M_BYTES / 1024;
  __amdgpu_buffer_rsrc_t st_src[NSTW];
  uint32_t st_stream[NSTW], st_step[NSTW], st_base[NSTW];
#pragma unroll
  for (int j = 0; j < NSTW; j++) {
    const uint32_t q = min(wave * NSTW + j, (uint32_t)S::NST - 1);
    const void* base = x.quants;
    uint32_t bytes = x.quant_bytes;
    st_stream[j] = q / (COLS / 16), st_step[j] = 64, st_base[j] = 0;
    const uint32_t bcol = q % (COLS / 16) * 16 + (lane >> 2);
    st_off[j] = min(col0 + bcol, x.n - 1) * (x.bpc * QB) + (((lane & 3) ^ ((bcol >> 2) & 3)) << 4);
    if (MEAN_STREAM > 0 && q >= NBL + NML) {
      constexpr uint32_t KIB = MEAN_STREAM > 0 ? MEAN_STREAM / 1024 : 1;
      const uint32_t p = q - NBL - NML;
      base = x.means, bytes = x.means_bytes;
      st_stream[j] = p / KIB, st_step[j] = x.mpad * (SB * 4), st_base[j] = row0 * (SB * 4);
      st_off[j] = p % KIB * 1024u + lane * 16u;
    } else if (q >= NBL) {
      const uint32_t mcol = (q - NBL) % (COLS / 64) * 64 + lane;
      base = x.meta, bytes = x.meta_bytes;
      st_stream[j] = (q - NBL) / (COLS / 64), st_step[j] = SB * MB;
      st_off[j] = (min(col0 + mcol, x.n - 1) * (x.bpc * MB)) & ~3u;  // (Q8: the aligned words around two blocks' scales)
    }
    st_src[j] = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
  }
  const uint32_t lds_a0 = lds_address(lds), lds_s0 = lds_address(lds_st);
  // load j of this wave's share of the activations of (iteration it, substep u) into ring slot `slot`
  auto load_a = [&](int j, uint32_t it, uint32_t u, uint32_t slot) __attribute__((always_inline)) {
    const uint32_t q = min(wave * NAW + j, (uint32_t)S::NA - 1);
    const uint32_t stream = q / (PANELS * ROWS / 8), panel = q / (ROWS / 8) % PANELS;
    const uint32_t st = min(st0 + it * WK + stream, x.stages - 1);
    load_to_lds(ra, a_off[j], ((st * NSUB + u) * PANELS + panel) * 128u, lds_a0 + slot * A_BYTES + q * 1024u);
  };
  // load j of its share of an iteration's stage
  auto load_stage = [&](int j, uint32_t it, uint32_t slot) __attribute__((always_inline)) {
    const uint32_t q = min(wave * NSTW + j, (uint32_t)S::NST - 1);
    const uint32_t st = min(st0 + it * WK + st_stream[j], x.stages - 1);
    load_to_lds(st_src[j], st_off[j], st_base[j] + st * st_step[j], lds_s0 + slot * STAGE_BYTES + q * 1024u);
  };
  floatx16 acc[RT][kCT];
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int t = 0; t < kCT; t++) acc[r][t] = (floatx16)(0.0f);

  // lane addresses of the operand reads: unit q of a row or column is q ^ (its swizzle)
  const uint32_t a_rd = (ks * PANELS * ROWS + wm * (RT * 32) + c) * 128u + ((2 * h) ^ ((c >> 1) & 7)) * 16u;
  const uint32_t b_rd = (ks * COLS + wn * (kCT * 32) + c) * 64u + (FMT == MGN_FMT_Q4 ? ((c >> 2) & 3) * 16u + h * 8u : (h ^ ((c >> 2) & 3)) * 16u);
  const uint32_t m_rd = B_BYTES + (ks * COLS + wn * (kCT * 32) + c) * 16u;
  const uint32_t s_rd = B_BYTES + M_BYTES + ks * MEAN_STREAM + (wm * (RT * 32) + c) * (SB * 4u) + h * (SB * 2u);
  const uint32_t addp = h ? x.add_lo : x.add_hi;

  static_for<-S::FIRST>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = S::FIRST + I, a = i + PD;
    if constexpr (a >= 0) {
#pragma unroll
      for (int j = 0; j < NAW; j++) load_a(j, min((uint32_t)(a / NSUB), iters - 1), a % NSUB, a);
    }
    if constexpr ((i + 64 * NSUB) % NSUB == 0 && S::stage_of(i) + SD >= 0) {
#pragma unroll
      for (int j = 0; j < NSTW; j++) load_stage(j, min((uint32_t)(S::stage_of(i) + SD), iters - 1), S::stage_of(i) + SD);
    }
  });
  bool mixed = false;
  float row_scale[RT];  // of row c of each row tile
  if constexpr (F32A) {
    uint32_t any = 0;
#pragma unroll
    for (int r = 0; r < RT; r++) {
      any |= x.mixed[row0 + (wm * RT + r) * 32 + c];
      row_scale[r] = x.row_scale[row0 + (wm * RT + r) * 32 + c] * x.unit;
    }
    mixed = __builtin_amdgcn_ballot_w64(any != 0) != 0;
  }
  wait_loads<S::in_flight_first()>();
  lds_barrier();

  // What is in registers ahead of its use: the raw quants of the next block, the operands of its first
  // row tile, and (d[1], dqp) the products of the last tile, which are scaled under the next block's
  // first matrix instructions.
  uint32_t braw[kCT][FMT == MGN_FMT_Q4 ? 2 : 4], mcur[kCT][FMT == MGN_FMT_Q4 ? 4 : 1];
  half8 bop[kCT][2], aop[F32A ? 1 : 2][NM];
  floatx16 d[2];
  float dq[kCT], dqp = 0.0f;
  auto read_b = [&](int t, const uint8_t* pb, int sb) __attribute__((always_inline)) {
    if constexpr (FMT == MGN_FMT_Q4) {
      const uint2 q = *(const uint2*)(pb + (b_rd ^ (sb * 16u)) + t * 2048);
      braw[t][0] = q.x, braw[t][1] = q.y;
    } else {
      const uint4 q = *(const uint4*)(pb + (b_rd ^ (sb * 32u)) + t * 2048);
      braw[t][0] = q.x, braw[t][1] = q.y, braw[t][2] = q.z, braw[t][3] = q.w;
    }
  };
  auto unpack_b = [&](int t) __attribute__((always_inline)) {
    if constexpr (FMT == MGN_FMT_Q4) {
      bop[t][0] = nibbles_in_order(braw[t][0]);
      bop[t][1] = nibbles_in_order(braw[t][1]);
    } else if constexpr (F32A) {
      bop[t][0] = signed_bytes_to_operand(braw[t][0], braw[t][1]);
      bop[t][1] = signed_bytes_to_operand(braw[t][2], braw[t][3]);
    } else {
      bop[t][0] = bytes_to_operand(braw[t][0], braw[t][1]);
      bop[t][1] = bytes_to_operand(braw[t][2], braw[t][3]);
    }
  };
  // operand j of row tile r of block bl of a substep: fp16, k half j of block bl % 2 of panel bl / 2; f32,
  // k half j % 2 of the high (j < 2) or low halves, panel bl
  auto read_a = [&](int slot, int j, const uint8_t* pa, int bl, int r) __attribute__((always_inline)) {
    const uint32_t unit = (j & 1) * 16u + (F32A ? j >> 1 : bl & 1) * 64u, panel = F32A ? bl : bl >> 1;
    aop[slot][j] = __builtin_bit_cast(half8, *(const u32x4_t*)(pa + (a_rd ^ unit) + panel * (ROWS * 128u) + r * 4096));
  };
  d[1] = (floatx16)(0.0f);
  read_b(0, lds_st, 0);
  read_b(1, lds_st, 0);
#pragma unroll
  for (int j = 0; j < NM; j++) read_a(0, j, lds, 0, 0);
  unpack_b(0);

  uint32_t abuf = 0, sbuf = 0;  // ring slots in use
  for (uint32_t it = 0; it < iters; it++) {
    const uint32_t st = st0 + it * WK + ks;
    const uint32_t valid = st < st1 ? min((uint32_t)SB, x.bpc - st * SB) : 0u;  // blocks of this stage (uniform)
    // the block constants of the lane's own two columns
#pragma unroll
    for (int t = 0; t < kCT; t++) {
      const uint8_t* const pm = lds_st + sbuf * STAGE_BYTES + m_rd + t * 512;
      if constexpr (FMT == MGN_FMT_Q4) {
        const uint4 v = *(const uint4*)pm;
        mcur[t][0] = v.x, mcur[t][1] = v.y, mcur[t][2] = v.z, mcur[t][3] = v.w;
      } else {
        const uint2 v = *(const uint2*)pm;
        const uint32_t odd = (min(col0 + (wn * kCT + t) * 32 + c, x.n - 1) * x.bpc) & 1u;  // (a stage starts at an even block)
        mcur[t][0] = odd ? (v.x >> 16) | (v.y << 16) : v.x;
      }
    }
    if (valid < SB) {
#pragma unroll
      for (int t = 0; t < kCT; t++) {
        if constexpr (FMT == MGN_FMT_Q4) {
#pragma unroll
          for (int e = 0; e < 4; e++) mcur[t][e] = (uint32_t)e < valid ? mcur[t][e] : 0u;
        } else {
          mcur[t][0] = valid == 1 ? mcur[t][0] & 0xFFFFu : 0u;
        }
      }
    }
    if (!F32A && valid > 0 && valid < SB) {
      // What the loads brought in behind the row's last block is another row's, or nothing's.  (Each wave clears the
      // rows that it reads, so that its own order suffices; waves that share rows write the same zeros.  Block 0,
      // whose first operands are in registers by now, is always the row's own.  Cleared substep by substep, behind the
      // barriers inside the loop, the branch there costs the 128 x 64 tiles 250 spilled registers.  The wait and the barrier
      // cost a call 0.1 to 0.3 us, which shows where K is short: Q4 32 x 256, 326 x 352 x 7680 12.8 -> 13.0, 1240 x 416 x 3299 15.8 -> 16.0;
      // to leave in flight what need not have landed, at PD = 3, is level.)
      static_assert(F32A || NSUB <= 2, "one substep ahead has been requested");
      if constexpr (NSUB > 1) {
        wait_loads<0>();
        lds_barrier();
      }
      for (uint32_t i = lane; i < NSUB * PANELS * RT * 32 * 8; i += 64) {
        const uint32_t unit = i & 7, row = i / 8 % (RT * 32), panel = i / (RT * 32 * 8);  // panels of the stage
        const uint32_t buf = abuf + panel / PANELS >= ARING ? abuf + panel / PANELS - ARING : abuf + panel / PANELS;
        const uint32_t at = (ks * PANELS + panel % PANELS) * ROWS + wm * (RT * 32) + row;
        if (panel * 2 + unit / 4 >= valid) *(uint4*)(lds + buf * A_BYTES + at * 128u + ((unit ^ ((row >> 1) & 7)) << 4)) = make_uint4(0, 0, 0, 0);
      }
    }
    if (F32A && mixed && it > 0 && valid > 0) {
      // rows of very different magnitudes along K: the sums move on to the next slice's scale
      const uint32_t sl = st * SB / 8, pl = (st - WK) * SB / 8;
      if (sl != pl) {
        acc[RT - 1][kCT - 1] = __builtin_elementwise_fma(d[1], (floatx16)(dqp), acc[RT - 1][kCT - 1]);
        dqp = 0.0f;
#pragma unroll
        for (int r = 0; r < RT; r++) {
          floatx16 f;
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const uint32_t row = row0 + (wm * RT + r) * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
            const uint32_t now = __builtin_bit_cast(uint32_t, x.inv[(size_t)sl * x.mpad + row]);
            const uint32_t was = __builtin_bit_cast(uint32_t, x.inv[(size_t)pl * x.mpad + row]);
            f[i] = __builtin_bit_cast(float, 0x3F800000u + (was - now));
          }
#pragma unroll
          for (int t = 0; t < kCT; t++) acc[r][t] *= f;
        }
      }
    }
    // The additive part of the stage's blocks: means times m (Q4) or the scale (Q8).
    // Q4's come in front of the stage's last substep.  Q8's stand for a bias of 128 on the bytes, several times the products
    // themselves, which must be in the sum when they take it out: the subtraction leaves little and rounds nothing, where in front of the
    // products the matrix unit rounds sums of the bias's size.  (Error against f64, fp16 activations behind a silu, first behind
    // the stage's products, then in front: 77 x 4096 x 14336 6.9e-7, 8.2e-7, 200 x 2048 x 8192 6.1e-7, 7.1e-7; Q4, whose minima are of
    // the products' size, 4.0e-7, 3.6e-7 on 2048 x 4096 x 14336.)  They are read in front of the barrier that gives their buffer away.
    uint32_t means[RT][FMT == MGN_FMT_Q4 ? 2 : 1];
    auto read_means = [&]() __attribute__((always_inline)) {
      const uint8_t* const ps = lds_st + sbuf * STAGE_BYTES + s_rd;
#pragma unroll
      for (int r = 0; r < RT; r++) {
        if constexpr (FMT == MGN_FMT_Q4) {
          const uint2 v = *(const uint2*)(ps + r * (32 * SB * 4));
          means[r][0] = v.x, means[r][1] = v.y;
        } else {
          means[r][0] = *(const uint32_t*)(ps + r * (32 * SB * 4));
        }
      }
    };
    auto add_means = [&]() __attribute__((always_inline)) {
      half8 bm[kCT];
#pragma unroll
      for (int t = 0; t < kCT; t++) {
        uint32_t w0, w1 = 0;
        const half2_t mulp = __builtin_bit_cast(half2_t, addp);
        if constexpr (FMT == MGN_FMT_Q4) {
          w0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(mcur[t][1], mcur[t][0], 0x07060302u)) * mulp);
          w1 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(mcur[t][3], mcur[t][2], 0x07060302u)) * mulp);
        } else {
          w0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, mcur[t][0]) * mulp);
        }
        bm[t] = as_half8(w0, w1, 0u, 0u);
      }
      // (Q8: the last tile, whose products are still to be scaled, comes first)
      static_for<TILES>([&](auto TT) __attribute__((always_inline)) {
        constexpr int T = FMT == MGN_FMT_Q4 ? (int)TT : TILES - 1 - TT, r = T / kCT, t = T % kCT;
        const half8 am = as_half8(means[r][0], FMT == MGN_FMT_Q4 ? means[r][FMT == MGN_FMT_Q4] : 0u, 0u, 0u);
        acc[r][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, bm[t], acc[r][t], 0, 0, 0);
      });
    };
    constexpr bool means_first = FMT == MGN_FMT_Q4, means_last = FMT == MGN_FMT_Q8 && has_additive(FMT, F32A);
    static_for<NSUB>([&](auto U) __attribute__((always_inline)) {
      constexpr int u = U;
      constexpr bool last = u == NSUB - 1;
      constexpr int ahead = (u + PD) / NSUB, usub = (u + PD) % NSUB;  // the activations requested here: iterations ahead, substep
      const uint32_t anext = abuf + 1 == ARING ? 0 : abuf + 1, aload = abuf == 0 ? ARING - 1 : abuf - 1;
      const uint32_t snext = sbuf + 1 == SRING ? 0 : sbuf + 1, sload = sbuf == 0 ? SRING - 1 : sbuf - 1;
      const uint32_t ita = min(it + ahead, iters - 1), its = min(it + SD, iters - 1);
      // The loads go out a few at a time between the tiles: all waves' loads at once hold every wave
      // until the address unit has taken them.
      auto issue_load = [&](auto Qn) __attribute__((always_inline)) {
        constexpr int q = Qn;
        if constexpr (q >= NAW) load_stage(q - NAW, its, sload);
        else load_a(q, ita, usub, aload);
      };
      if constexpr (last && means_first) read_means(), add_means();
      __builtin_amdgcn_sched_barrier(0);
      static_for<SUBB>([&](auto BL) __attribute__((always_inline)) {
        constexpr int bl = BL, sb = u * SUBB + bl;
        constexpr bool ends_sub = bl == SUBB - 1, ends_stage = sb == SB - 1;
        const uint8_t* const pa = lds + abuf * A_BYTES;
        const uint8_t* const pan = ends_sub ? lds + anext * A_BYTES : pa;
        const uint8_t* const pbn = lds_st + (ends_stage ? snext : sbuf) * STAGE_BYTES;
#pragma unroll
        for (int t = 0; t < kCT; t++) {
          if constexpr (FMT == MGN_FMT_Q4) dq[t] = half_bits_to_float(mcur[t][sb] & 0xFFFFu) * x.dscale;
          else dq[t] = half_bits_to_float(sb ? mcur[t][0] >> 16 : mcur[t][0] & 0xFFFFu) * x.dscale;
        }
        // Tile T of the block: NM matrix instructions, and between them the scaling of tile T - 1
        static_for<TILES>([&](auto TT) __attribute__((always_inline)) {
          constexpr int T = TT, r = T / kCT, t = T % kCT, pr = T ? (T - 1) / kCT : RT - 1, pt = T ? (T - 1) % kCT : kCT - 1;
          constexpr int slot = F32A ? 0 : (sb * RT + r) & 1;
          constexpr int b_at = ends_sub && !S::ALONE && S::TURN > 1 ? S::TURN : 1;  // (a substep's first quants are read behind its barrier)
          if constexpr (ends_sub && T == S::TURN) {
            if constexpr (last && means_last) read_means();
            wait_loads<S::in_flight(u)>();
            lds_barrier();
          }
          static_for<NM>([&](auto J) __attribute__((always_inline)) {
            constexpr int j = J;
            d[T & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aop[slot][j], bop[t][j & 1], j == 0 ? (floatx16)(0.0f) : d[T & 1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (F32A ? t == kCT - 1 : t == 0) {
              // the next row tile's operands (f32: into the registers the instruction above was the last to read)
              constexpr int ns = F32A ? 0 : slot ^ 1;
              if constexpr (r + 1 < RT) read_a(ns, j, pa, bl, r + 1);
              else read_a(ns, j, pan, ends_sub ? 0 : bl + 1, 0);
            }
            if constexpr (j == 0 && T == 0) unpack_b(1);
            if constexpr (j == 0 && T == b_at) read_b(0, pbn, ends_stage ? 0 : sb + 1), read_b(1, pbn, ends_stage ? 0 : sb + 1);
            if constexpr (j == (TILES == 2 || b_at == TILES - 1 ? NM - 1 : 0) && T == TILES - 1) unpack_b(0);
            scale_part<NM, j>(acc[pr][pt], d[(T + 1) & 1], T ? dq[pt] : dqp);
            if constexpr (j == NM - 1) {
              constexpr int from = S::issued_before(u, bl * TILES + T), to = S::issued_before(u, bl * TILES + T + 1);
              static_for<to - from>([&](auto Qn) __attribute__((always_inline)) { issue_load(std::integral_constant<int, from + Qn>{}); });
            }
            __builtin_amdgcn_sched_barrier(0);
          });
        });
        dqp = dq[kCT - 1];
      });
      if constexpr (S::ALONE && last && means_last) read_means();
      if constexpr (last && means_last) add_means();
      if constexpr (S::ALONE) {
        wait_loads<S::in_flight(u)>();
        lds_barrier();
      }
      abuf = anext;
      if constexpr (last) sbuf = snext;
    });
  }
  acc[RT - 1][kCT - 1] = __builtin_elementwise_fma(d[1], (floatx16)(dqp), acc[RT - 1][kCT - 1]);
  wait_loads<0>();
  lds_barrier();

  // ---- true units ----
  if constexpr (F32A) {
    // the rows' scales from the lanes that hold them to the lanes that hold the rows' sums
    float* const sc = (float*)lds + wave * (RT * 32);
#pragma unroll
    for (int r = 0; r < RT; r++) sc[r * 32 + c] = row_scale[r];
    const uint32_t mine = st1 > st0 + ks ? (st1 - 1 - st0 - ks) / WK * WK + st0 + ks : 0u;  // the stream's last stage
#pragma unroll
    for (int r = 0; r < RT; r++) {
      floatx16 f;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        floatx4 v = *(const floatx4*)(sc + r * 32 + q * 8 + h * 4);
        if (mixed) {
          // the sums are on the scale of the stream's own last slice: from there to the row's last
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const uint32_t row = row0 + (wm * RT + r) * 32 + q * 8 + h * 4 + i;
            const uint32_t own = __builtin_bit_cast(uint32_t, x.inv[(size_t)(mine * SB / 8) * x.mpad + row]);
            const uint32_t end = __builtin_bit_cast(uint32_t, x.inv[(size_t)((x.bpc - 1) / 8) * x.mpad + row]);
            v[i] *= __builtin_bit_cast(float, 0x3F800000u + (own - end));
          }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) f[q * 4 + i] = v[i];
      }
#pragma unroll
      for (int t = 0; t < kCT; t++) acc[r][t] *= f;
    }
    if constexpr (WK > 1) lds_barrier();
  } else {
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int t = 0; t < kCT; t++) acc[r][t] *= x.unit;
  }
  if constexpr (WK > 1) {
    // The streams' sums meet in LDS: each stream keeps one of the two column tiles, hands the other one over and stores
    // what it kept, so that the exchange and the stores have all waves.  (Before, one stream's waves added up and stored
    // both tiles when the other's had ended, 3.4 of a workgroup's 28 us.  us, this step by itself: Q4 77 x 4096 x 14336 39.7 -> 38.8,
    // 77 x 14336 x 4096 41.4 -> 40.9; with the barrier in front of the last tile, on another machine, 38.9 -> 37.6, 42.1 -> 40.4, Q8 42.9 -> 39.5,
    // 43.9 -> 41.1; the 64-row shape level.)
    static_assert(WK == 2 && kCT == 2 && (WM * WN & (WM * WN - 1)) == 0, "a column tile per stream, and the other stream's wave a bit away");
    float* const red = (float*)lds4;
    const uint32_t other = wave ^ (WM * WN);
    if (ks != 0) {
#pragma unroll
      for (int r = 0; r < RT; r++) {
        const floatx16 kept = acc[r][1];
        acc[r][1] = acc[r][0], acc[r][0] = kept;
      }
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        *(floatx4*)(red + ((wave * RT + r) * 4 + i) * 256 + lane * 4) =
            floatx4{acc[r][1][4 * i], acc[r][1][4 * i + 1], acc[r][1][4 * i + 2], acc[r][1][4 * i + 3]};
    lds_barrier();
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const floatx4 v = *(const floatx4*)(red + ((other * RT + r) * 4 + i) * 256 + lane * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[r][0][4 * i + e] += v[e];
      }
  }
  // Stores through a buffer descriptor that ends with the last row: what lies past it is dropped.  (Stores like any other, also of
  // results far larger than the L2s: a row whose length is no multiple of 32 words shares its 128-byte lines between
  // workgroups, and only a cache that keeps them puts them together.  With the non-temporal hint, us, without -> with: fp16
  // activations 700 x 576 x 49151 Q4 88 -> 148, Q8 87 -> 146; 2048 x 1024 x 14337 Q4 89 -> 143, f32 137 -> 159.  In whole
  // lines it went both ways, 2048 x 4096 x 14336 Q4 277 -> 271 but 2048 x 576 x 49152 f32 321 -> 328, with a residual 391 -> 441; with a call
  // behind it that reads the result: 1250 x 1024 -> 14336 -> 1024 221 -> 225, 2048 the like 348 -> 350, 4096 728 -> 705.)
  const bool direct = x.parts == 1;
  const uint32_t bytes = x.m * x.n * 4u;
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((void*)(direct ? x.c : x.partial + (size_t)part * x.m * x.n), 0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc((void*)x.dres, 0, bytes, 0x00020000);
  const uint32_t ops = direct ? x.epilogue : 0u;
  const bool residual = direct && x.dres;
  // (unary operations run in a loop over the lane's own words, parked in LDS: unrolled over the
  // registers they would be most of the kernel)
  float* const strip = (float*)lds4 + wave * 1024 + lane;
  if (ops != 0) lds_barrier();
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int t = 0; t < kCT / WK; t++) {
      const uint32_t col = col0 + (wn * kCT + (WK > 1 ? ks : t)) * 32 + c;
      const uint32_t off = ((row0 + (wm * RT + r) * 32 + h * 4) * x.n + col) * 4u;
      if (col >= x.n) continue;
      if (residual) {
        float dv[16];
#pragma unroll
        for (int i = 0; i < 16; i++) dv[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(res, off + ((i >> 2) * 8 + (i & 3)) * x.n * 4u, 0, 0));
#pragma unroll
        for (int i = 0; i < 16; i++) acc[r][t][i] += dv[i];
      }
      if (ops != 0) {
#pragma unroll
        for (int i = 0; i < 16; i++) strip[i * 64] = acc[r][t][i];
#pragma nounroll
        for (int i = 0; i < 16; i++) strip[i * 64] = apply_epilogue(strip[i * 64], ops);
#pragma unroll
        for (int i = 0; i < 16; i++) acc[r][t][i] = strip[i * 64];
      }
#pragma unroll
      for (int i = 0; i < 16; i++)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, (float)acc[r][t][i]), out, off + ((i >> 2) * 8 + (i & 3)) * x.n * 4u, 0, 0);
    }
}

// ---- what the kernel needs to know about the activations, one workgroup per row ----
constexpr uint32_t kMaxSlices = 256;
constexpr int kTop = 14;  // a row's largest magnitude is brought into [2^14, 2^15)

__device__ __forceinline__ void store_mean(_Float16* means, int sb, uint32_t mpad, uint32_t row, uint32_t block, float mean) {
  _Float16* const p = means + ((size_t)(block / sb) * mpad + row) * (sb * 2) + block % sb;
  p[0] = (_Float16)mean;
  p[sb] = (_Float16)((mean - (float)p[0]) * 2048.0f);
}

// grid.x = mpad rows, 512 threads: half-wave w converts the row's slices w, w + 16, ..; HELD of them stay
// in registers between the search for the row's largest magnitude and the conversion, the rest of a
// longer row is read twice.
//
// Both halves of a pair are rounded to nearest (23 bits and no bias; cut, as the tiled kernels' pairs are, they
// carry 22 and all results come out 2^-24 to 2^-23 small), and a block's mean is that of its pairs.
template <int FMT, int HELD>
__global__ __launch_bounds__(512) void prepare_f32_kernel(const float* __restrict__ a, uint8_t* __restrict__ out, _Float16* __restrict__ means,
                                                          float* __restrict__ inv, float* __restrict__ row_scale, uint32_t* __restrict__ mixed,
                                                          uint32_t m, uint32_t k, uint32_t nslices, uint32_t mpad,
                                                          uint32_t* __restrict__ range_flag) {
  constexpr int SB = stage_blocks(FMT);
  __shared__ float smax[kMaxSlices];
  const uint32_t row = blockIdx.x, tid = threadIdx.x, l = tid & 31, hw = tid >> 5;
  const float* const src = a + (size_t)min(row, m - 1) * k;
  const bool live = row < m;
  floatx4 held[HELD][2];
  auto load = [&](uint32_t s, floatx4 (&v)[2]) __attribute__((always_inline)) {
    const uint32_t k0 = s * 256 + l * 8;
    const bool ok = live && k0 < k;
    const floatx4* const p = (const floatx4*)(src + (ok ? k0 : 0));
    v[0] = p[0], v[1] = p[1];
    if (!ok) v[0] = v[1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  auto largest = [&](const floatx4 (&v)[2], uint32_t s) __attribute__((always_inline)) {
    float am = fmaxf(fmaxf(fmaxf(fabsf(v[0].x), fabsf(v[0].y)), fmaxf(fabsf(v[0].z), fabsf(v[0].w))),
                     fmaxf(fmaxf(fabsf(v[1].x), fabsf(v[1].y)), fmaxf(fabsf(v[1].z), fabsf(v[1].w))));
    am = group_max32(am);
    if (l == 0) smax[s] = am;
  };
#pragma unroll
  for (int i = 0; i < HELD; i++) load(hw + 16 * i, held[i]);
#pragma unroll
  for (int i = 0; i < HELD; i++)
    if (hw + 16 * i < nslices) largest(held[i], hw + 16 * i);
  for (uint32_t s = hw + 16 * HELD; s < nslices; s += 16) {
    floatx4 v[2];
    load(s, v);
    largest(v, s);
  }
  __syncthreads();
  // (a NaN never wins fmaxf; an infinity does)
  float rmax = 0.0f, rmin = __builtin_inff();  // the largest, and the smallest of the slices that hold anything
  for (uint32_t s = l; s < nslices; s += 32) {
    const float v = smax[s];
    rmax = fmaxf(rmax, v);
    if (((__builtin_bit_cast(uint32_t, v) >> 23) & 255) > 27) rmin = fminf(rmin, v);  // above 2^-100
  }
  rmax = group_max32(rmax);
  rmin = -group_max32(-rmin);
  const int er = (int)(__builtin_bit_cast(uint32_t, rmax) >> 23) - 127;
  const bool bad = er >= 100;
  const bool scaled = er > -100 && !bad;  // (a flag of its own: a row whose largest is in [2^kTop, 2^(kTop + 1)) has a shift of 0 as well)
  const int shr = scaled ? kTop - er : 0;
  // One scale for the row, unless a slice's largest would come to lie more than a bit below where the tiled kernels
  // bring every slice's (2^7 with Q4, 2^11 with Q8; the low halves end at 2^-24, and what is rounded there is as close as
  // what is cut a bit further down): such slices get scales of their own, up to 2^60 times the row's (the sums of
  // the large slices move along and must stay finite).  Rows that have such slices cost: lognormal activations (sigma
  // 1.5), Q8 77 x 4096 x 14336 43.5 -> 46.8 us, Q4 level.
  constexpr int kLeast = FMT == MGN_FMT_Q4 ? 6 : 10;
  auto shift = [&](float smx) __attribute__((always_inline)) {
    const int es = (int)(__builtin_bit_cast(uint32_t, smx) >> 23) - 127;
    return scaled && es > -100 && es + shr < kLeast ? min(kTop - es, shr + 60) : shr;
  };
  const bool any_mixed = shift(rmin) != shr;
  auto convert = [&](const floatx4 (&v)[2], uint32_t s) __attribute__((always_inline)) {
    const int sh = any_mixed ? shift(smax[s]) : shr;
    const float scale = __builtin_bit_cast(float, (uint32_t)(127 + sh) << 23);
    if (l == 0) {
      const float back = __builtin_bit_cast(float, (uint32_t)(127 - sh) << 23);
      inv[(size_t)s * mpad + row] = back;
      if (s == nslices - 1) row_scale[row] = bad ? __builtin_nanf("") : back;
    }
    const floatx4 x0 = v[0] * scale, x1 = v[1] * scale;
    float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    half8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      hi[e] = (_Float16)x[e];
      lo[e] = (_Float16)(x[e] - (float)hi[e]);
      x[e] = (float)hi[e] + (float)lo[e];
    }
    float sum = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    if (live) {
      uint8_t* const dst = out + ((size_t)row * nslices * 8 + s * 8 + (l >> 2)) * 128 + (l & 3) * 16;
      *(half8*)dst = hi;
      *(half8*)(dst + 64) = lo;
    }
    sum += dpp_move<kDppQuadXor1>(sum);
    sum += dpp_move<kDppQuadXor2>(sum);
    if (has_additive(FMT, true) && (l & 3) == 0) store_mean(means, SB, mpad, row, s * 8 + (l >> 2), sum * 0.03125f);
  };
#pragma unroll
  for (int i = 0; i < HELD; i++)
    if (hw + 16 * i < nslices) convert(held[i], hw + 16 * i);
  for (uint32_t s = hw + 16 * HELD; s < nslices; s += 16) {
    floatx4 v[2];
    load(s, v);
    convert(v, s);
  }
  if (tid == 0) {
    mixed[row] = any_mixed ? 1u : 0u;
    if (range_flag && rmax >= 65504.0f) *range_flag = 1u;  // a promise (MGN_ACT_FP16_RANGE) that does not hold
  }
}

template <int FMT>
__global__ __launch_bounds__(256) void prepare_f16_kernel(const _Float16* __restrict__ a, _Float16* __restrict__ means, uint32_t m,
                                                          uint32_t k, uint32_t nslices, uint32_t mpad) {
  constexpr int SB = stage_blocks(FMT);
  const uint32_t row = blockIdx.x;
  for (uint32_t u = threadIdx.x; u < nslices * 32; u += 256) {
    const uint32_t k0 = u * 8;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row < m && k0 < k) v = *(const uint4*)(a + (size_t)row * k + k0);
    const half2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
    float s = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v.x), ones, 0.0f, false);
    s = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v.y), ones, s, false);
    s = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v.z), ones, s, false);
    s = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v.w), ones, s, false);
    s += dpp_move<kDppQuadXor1>(s);
    s += dpp_move<kDppQuadXor2>(s);
    if ((u & 3) == 0) store_mean(means, SB, mpad, row, u >> 2, s * 0.03125f);
  }
}

// C = f(sum over the parts, in part order, + D); V words per thread and step
template <int V>
__global__ __launch_bounds__(256) void add_parts_kernel(const float* __restrict__ partial, const float* __restrict__ dres, float* __restrict__ c,
                                                        uint64_t count, uint32_t parts, uint32_t epilogue) {
  typedef float vec __attribute__((ext_vector_type(V)));
  for (uint64_t i = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * V; i < count; i += (uint64_t)gridDim.x * 256 * V) {
    vec s = *(const vec*)(partial + i);
    uint32_t p = 1;
    for (; p + 4 <= parts; p += 4) {
      const vec a = *(const vec*)(partial + p * count + i), b = *(const vec*)(partial + (p + 1) * count + i);
      const vec e = *(const vec*)(partial + (p + 2) * count + i), f = *(const vec*)(partial + (p + 3) * count + i);
      s = s + a, s = s + b, s = s + e, s = s + f;
    }
    for (; p < parts; p++) s = s + *(const vec*)(partial + p * count + i);
    if (dres) s = s + *(const vec*)(dres + i);
    if (epilogue != 0) {
#pragma unroll
      for (int e = 0; e < V; e++) s[e] = apply_epilogue(s[e], epilogue);
    }
    *(vec*)(c + i) = s;
  }
}

// ---- plans ----
// The workgroup shapes that are built, by (format, activations): rows x columns per workgroup and what a
// stage costs on them, in us per 128 elements of K: one workgroup per CU on all 256 (t1), and each
// further round of 256 (tn; where two fit a CU, what the second costs beside the first).  Fitted before the barriers moved in front
// of the last tiles: the estimates made of them are now, median by workgroup over 364 sizes, 0.97 to 1.27 times what is measured
// (2048 x 4096 x 14336 Q4 fp16 337 against 263, f32 512 x 4096 x 14336 163 against 115, 77 x 4096 x 14336 48 against 38, 1500 x 1024 x 14336
// 110 against 106).  An estimate that is too high leaves a call to the kernel behind.
struct BlockConfig {
  void (*kernel)(BlockArgs);
  uint32_t rows, cols, threads, streams;
  size_t lds;
  double t1, tn;
};

template <int FMT, bool F32A, int RT, int WM, int WN, int SUBB, int PD, int SD, int WK = 1>
BlockConfig block_config(double t1, double tn) {
  // (fp16 activations are read where they are: a stream without a stage would multiply what lies behind K by zero)
  static_assert(WK == 1 || F32A, "streams may run out of stages only on prepared activations");
  using S = BlockShape<FMT, F32A, RT, WM, WN, WK, SUBB, PD, SD>;
  static_assert(S::LDS <= 160 * 1024, "fits a CU");
  static_assert(S::waits_suffice(), "a wave passes a barrier before its operands have landed");
  return {block_kernel<FMT, F32A, RT, WM, WN, WK, SUBB, PD, SD>, (uint32_t)S::ROWS, (uint32_t)S::COLS, 64u * S::WAVES, (uint32_t)WK, S::LDS, t1, tn};
}

constexpr int kBlockConfigs = 9;  // at most, per format and kind of activations
const BlockConfig* block_configs(int fmt, bool f32a) {
  static const BlockConfig q4_f16[kBlockConfigs] = {
      block_config<0, false, 4, 2, 4, 2, 2, 1>(5.7, 4.1), block_config<0, false, 3, 2, 4, 2, 2, 2>(4.65, 3.1),
      block_config<0, false, 2, 2, 4, 2, 2, 2>(3.6, 2.6), block_config<0, false, 3, 1, 4, 2, 2, 1>(2.9, 1.9),
      block_config<0, false, 2, 1, 4, 2, 2, 1>(2.3, 1.5), block_config<0, false, 1, 1, 4, 2, 3, 2>(1.33, 0.9),
      block_config<0, false, 1, 2, 2, 2, 2, 2>(1.45, 0.8)};
  static const BlockConfig q4_f32[kBlockConfigs] = {
      block_config<0, true, 4, 2, 4, 1, 2, 1>(7.6, 6.7), block_config<0, true, 3, 2, 4, 1, 2, 2>(6.3, 5.2),
      block_config<0, true, 2, 2, 4, 1, 3, 1>(4.7, 3.2), block_config<0, true, 3, 1, 4, 1, 2, 1>(4.4, 2.4),
      block_config<0, true, 2, 1, 4, 1, 3, 1>(2.95, 1.9), block_config<0, true, 1, 1, 4, 1, 4, 1>(2.0, 1.3),
      block_config<0, true, 1, 2, 2, 1, 3, 1>(1.65, 1.2), block_config<0, true, 3, 1, 4, 1, 2, 1, 2>(3.55, 3.3),
      block_config<0, true, 2, 1, 4, 1, 3, 1, 2>(2.45, 2.3)};
  static const BlockConfig q8_f16[kBlockConfigs] = {
      block_config<1, false, 3, 2, 4, 2, 2, 3>(5.3, 3.5), block_config<1, false, 2, 2, 4, 2, 2, 3>(4.35, 2.6), block_config<1, false, 3, 1, 4, 2, 2, 3>(3.3, 2.6),
      block_config<1, false, 2, 1, 4, 2, 2, 3>(2.65, 2.2), block_config<1, false, 1, 1, 4, 2, 3, 2>(1.95, 1.9),
      block_config<1, false, 1, 2, 2, 2, 2, 3>(1.6, 1.2)};
  static const BlockConfig q8_f32[kBlockConfigs] = {
      block_config<1, true, 4, 2, 4, 1, 2, 1>(8.4, 7.6), block_config<1, true, 3, 2, 4, 1, 2, 2>(6.9, 5.5),
      block_config<1, true, 2, 2, 4, 1, 3, 2>(5.4, 3.9), block_config<1, true, 3, 1, 4, 1, 2, 1>(5.25, 2.6),
      block_config<1, true, 2, 1, 4, 1, 3, 2>(3.6, 2.8), block_config<1, true, 1, 1, 4, 1, 4, 2>(2.4, 2.3),
      block_config<1, true, 1, 2, 2, 1, 3, 2>(2.45, 1.4), block_config<1, true, 3, 1, 4, 1, 2, 1, 2>(4.1, 3.9)};
  return fmt == MGN_FMT_Q4 ? (f32a ? q4_f32 : q4_f16) : (f32a ? q8_f32 : q8_f16);
}

// Two streams in one workgroup instead of two workgroups on a CU: the same waves and the same loads, but
// one set of sums leaves the CU, so a shape takes half the K parts and half the traffic of adding them up
// (f32, one stream -> two, us: Q4 128 x 4096 x 14336 59.0 -> 50.4, 77 x 4096 x 14336 43.5 -> 42.2, 160 x 14336 x
// 4096 75.1 -> 70.4; Q8 77 x 4096 x 14336 52.0 -> 47.0, 160 x 2048 x 8192 34.3 -> 32.7).  Not where a stream has
// fewer stages than this, the start of the rings and the meeting being most of it then (Q4 77 x 4096 x 4096, two
// stages each, 23.6 -> 25.7; Q8 26.1 -> 27.7), nor with 32 rows (level) or, Q8, 64 (64 x 4096 x 14336 37.2 -> 41.9).
constexpr uint32_t kStreamStages = 4;

struct BlockPlan {
  const BlockConfig* cfg;
  uint32_t rows_per_launch = 0, rowgroups, colgroups, parts, stages, nslices, mpad;
  size_t a_bytes, means_bytes, inv_bytes, partial_bytes;  // in the workspace, in this order (row scales and flags behind inv)
  double us = 0;
};
constexpr double kNoLimit = 1e30;

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// The best plan for m rows that is expected to take less than limit_us.  kNone: no shape of workgroup serves them; kSlow:
// none in that time.  A caller that weighs the kernel against another one pays for the search on calls that end up elsewhere
// too, so what cannot beat the limit, or the best plan so far, is left out by bounds from below: a shape by its
// rounds' share of the work, K parts by their traffic.  (Host time of a call with a runtime that does nothing, without
// this kernel, searched whole, with the bounds, us: 128 x 1024 x 3072 1.2, 1.7 (Q8 2.0), 1.35; 77 x 4096 x 14336, which it
// takes, 3.4, 7.0, 3.9 with one search for choice and launch.)
enum class Found { kNone, kSlow, kPlan };
Found plan_block_rows(const LaunchArgs& x, uint32_t m, double limit_us, BlockPlan* out) {
  const bool f32a = !x.a_is_f16;
  const uint64_t k = x.w.k, n = x.w.n;
  const uint32_t bpc = x.w.k / 32, sb = stage_blocks(x.w.fmt);
  const uint32_t stages = (bpc + sb - 1) / sb, nslices = (bpc + 7) / 8;
  if (m == 0 || bpc == 0 || nslices > kMaxSlices) return Found::kNone;
  if (n * bpc * 32 >= (1ull << 32)) return Found::kNone;  // a lane's weight offsets are 32-bit
  const BlockConfig* const cfgs = block_configs(x.w.fmt, f32a);
  const double outputs = (double)m * n * 4;
  const double mem = (double)bpc * n * (x.w.fmt == MGN_FMT_Q4 ? 20 : 34) / 5.0e6 + outputs / 4.0e6;
  // (f32: the workgroups that convert a row each are more than the chip holds at once beyond some 512 rows; without that term short
  // calls of 1024 to 2048 rows measured 2 to 3 us above their estimate)
  const double fixed = 3.5 + outputs / 8.0e6 + 2.2 + (double)m * k * (f32a ? 8 : 2) / 5.0e6 + (f32a && m > 512 ? (m - 512) * 2.2e-3 : 0.0);
  double best = limit_us;
  Found found = Found::kNone;
  for (int i = 0; i < kBlockConfigs; i++) {
    const BlockConfig& c = cfgs[i];
    if (!c.kernel) break;
    const uint32_t rowgroups = (m + c.rows - 1) / c.rows, mpad = rowgroups * c.rows;
    const uint64_t colgroups = (n + c.cols - 1) / c.cols;
    const uint64_t tiles = rowgroups * colgroups;
    if (tiles > (1u << 24) || (uint64_t)mpad * n * 4 >= (1ull << 32)) continue;
    const size_t a_bytes = f32a ? align256((size_t)m * nslices * 1024) : 0;
    const size_t a_read = f32a ? (size_t)m * nslices * 1024 : (size_t)m * k * 2;
    if (a_read >= (1ull << 32)) continue;
    const size_t means = has_additive(x.w.fmt, f32a) ? align256((size_t)nslices * 8 * mpad * 4 + 4096) : 0;
    const size_t inv = f32a ? align256((size_t)nslices * mpad * 4 + (size_t)mpad * 8) : 0;
    if (stages < c.streams * kStreamStages && c.streams > 1) continue;
    if (a_bytes + means + inv > x.block_ws_bytes) continue;
    if (found == Found::kNone) found = Found::kSlow;
    // (nk of a part times its rounds is never less than all of K times the tiles' share of a round, and no round costs less than tn)
    if (0.999 * ((double)stages * sb / 4.0 * c.tn * tiles / x.num_cus + fixed) >= best) continue;
    for (uint32_t parts = 1; parts <= stages && parts <= 32; parts++) {
      const double adding = parts > 1 ? 3.5 + (2.0 * parts + 1) * outputs / 5.0e6 : 0.0;
      if (0.999 * (std::max(mem, c.t1 * sb / 4.0) + fixed + adding) >= best) break;
      const uint32_t spp = (stages + parts - 1) / parts;
      if ((stages + spp - 1) / spp != parts) continue;  // same split, already seen
      if (spp < c.streams * kStreamStages && c.streams > 1) break;
      const size_t partial = parts > 1 ? (size_t)parts * m * n * 4 : 0;
      if (a_bytes + means + inv + partial > x.block_ws_bytes) break;
      const uint64_t wgs = tiles * parts;
      const double nk = (spp + c.streams - 1) / c.streams * c.streams * (double)sb / 4.0;
      const double rounds = std::ceil((double)wgs / x.num_cus);
      const double us = std::max(nk * (c.t1 + (rounds - 1) * c.tn) + (c.streams > 1 ? rounds : 0.0), mem) + fixed + adding;  // (rounds: the streams' meeting)
      if (us < best) {
        best = us;
        found = Found::kPlan;
        *out = BlockPlan{&c, m, rowgroups, (uint32_t)colgroups, parts, stages, nslices, mpad, a_bytes, means, inv, partial, us};
      }
    }
  }
  return found;
}

// As many rows per launch as the workspace has room for: all of them, or blocks of rows one after the other.
bool plan_block(const LaunchArgs& x, double limit_us, BlockPlan* out) {
  if (!x.block_ws || x.n_more != 0 || x.pro_kind != kProNone) return false;
  for (uint32_t rows = x.m;;) {
    const uint32_t launches = (x.m + rows - 1) / rows;
    const Found f = plan_block_rows(x, rows, limit_us / launches, out);
    out->us *= launches;
    if (f != Found::kNone) return f == Found::kPlan;
    if (rows <= 256) return false;
    rows = (rows / 2 + 255) / 256 * 256;
  }
}

uint32_t half_pair(float v) {
  const uint16_t b = f32_to_f16_bits(v);
  return b | ((uint32_t)b << 16);
}

template <int FMT>
int launch_block_rows(ihipStream_t* s, const LaunchArgs& x, const BlockPlan& p) {
  const bool f32a = !x.a_is_f16;
  char* const ws = (char*)x.block_ws;
  uint8_t* const prepared = (uint8_t*)ws;
  _Float16* const means = (_Float16*)(ws + p.a_bytes);
  float* const inv = (float*)(ws + p.a_bytes + p.means_bytes);
  float* const row_scale = inv + (size_t)p.nslices * p.mpad;
  uint32_t* const mixed = (uint32_t*)(row_scale + p.mpad);
  float* const partial = (float*)(ws + p.a_bytes + p.means_bytes + p.inv_bytes);
  if (f32a) {
    auto prep = p.nslices <= 16 ? prepare_f32_kernel<FMT, 1> : prepare_f32_kernel<FMT, 4>;
    hipLaunchKernelGGL(prep, dim3(p.mpad), dim3(512), 0, s, (const float*)x.a, prepared, means, inv, row_scale, mixed, x.m, x.w.k, p.nslices,
                       p.mpad, x.promised_range ? x.range_flag : nullptr);
  } else {
    hipLaunchKernelGGL(prepare_f16_kernel<FMT>, dim3(p.mpad), dim3(256), 0, s, (const _Float16*)x.a, means, x.m, x.w.k, p.nslices, p.mpad);
  }
  MGN_HIP_LAUNCH_CHECK();
  BlockArgs a{};
  a.a = f32a ? (const void*)prepared : x.a;
  a.means = means, a.inv = inv, a.row_scale = row_scale, a.mixed = mixed, a.meta = x.w.meta, a.quants = x.w.quants;
  const size_t nb = (size_t)(x.w.k / 32) * x.w.n;
  a.a_pitch = f32a ? p.nslices * 1024 : x.w.k * 2;
  a.a_bytes = x.m * a.a_pitch;
  // (256 zero blocks follow the weight's own, which a column's last stage may reach into)
  a.quant_bytes = (uint32_t)std::min<size_t>((nb + 256) * (FMT == MGN_FMT_Q4 ? 16 : 32), 0xFFFFFFFFu);
  a.meta_bytes = (uint32_t)((nb + 256) * (FMT == MGN_FMT_Q4 ? 4 : 2));
  a.means_bytes = (uint32_t)p.means_bytes;
  a.m = x.m, a.mpad = p.mpad, a.n = x.w.n, a.bpc = x.w.k / 32, a.stages = p.stages;
  a.rowgroups = p.rowgroups, a.colgroups = p.colgroups, a.parts = p.parts;
  // The sums run in units of 2^lift / 32 (Q4) or 2^lift / 4096 (Q8) of the result: the additive constants
  // enter times 2^lift (WeightView::additive_lift), their means as they are.  (Without an additive part: the result's own.)
  const int lift = (int)std::min<uint32_t>(x.w.additive_lift, 15u);
  const float sign = FMT == MGN_FMT_Q4 ? 1.0f : -1.0f;
  a.add_hi = half_pair(sign * std::ldexp(1.0f, lift)), a.add_lo = half_pair(sign * std::ldexp(1.0f, lift - 11));
  a.dscale = std::ldexp(1.0f, (FMT == MGN_FMT_Q4 ? 15 : 12) + lift);
  a.unit = std::ldexp(1.0f, (FMT == MGN_FMT_Q4 ? 5 : 12) - lift);
  if (!has_additive(FMT, f32a)) a.dscale = a.unit = 1.0f;
  a.dres = x.d, a.c = x.c, a.partial = partial, a.epilogue = x.epilogue;
  if (p.cfg->lds > 64 * 1024) {
    static std::atomic<uint64_t> big_lds_done[4][kBlockConfigs];
    const BlockConfig* const first = block_configs(FMT, f32a);
    if (int e = enable_big_lds(p.cfg->kernel, x.device, big_lds_done[FMT * 2 + f32a][p.cfg - first])) return e;
  }
  hipLaunchKernelGGL(p.cfg->kernel, dim3((p.rowgroups * p.colgroups * p.parts + 7) / 8 * 8), dim3(p.cfg->threads), p.cfg->lds, s, a);
  MGN_HIP_LAUNCH_CHECK();
  if (p.parts > 1) {
    const uint64_t count = (uint64_t)x.m * x.w.n;
    const bool wide = count % 4 == 0 && ((uintptr_t)x.c & 15) == 0 && ((uintptr_t)x.d & 15) == 0;
    const uint64_t steps = wide ? count / 4 : count;
    hipLaunchKernelGGL(wide ? add_parts_kernel<4> : add_parts_kernel<1>, dim3((unsigned)std::min<uint64_t>((steps + 255) / 256, 2048)), dim3(256), 0, s,
                       partial, x.d, x.c, count, p.parts, x.epilogue);
    MGN_HIP_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace

bool choose_block_mfma(const LaunchArgs& x, double limit_us, BlockChoice* out) {
  static_assert(sizeof(BlockPlan) <= sizeof out->plan && std::is_trivially_copyable_v<BlockPlan>, "a plan travels in a choice");
  BlockPlan p;
  if (!plan_block(x, limit_us > 0 ? limit_us : kNoLimit, &p)) return false;
  std::memcpy(out->plan, &p, sizeof p);
  return true;
}

int launch_matmul_block_mfma(ihipStream_t* s, const LaunchArgs& x, const BlockChoice& choice) {
  BlockPlan p;
  std::memcpy(&p, choice.plan, sizeof p);
  const uint32_t rows = p.rows_per_launch;
  for (uint32_t r0 = 0; r0 < x.m; r0 += rows) {
    LaunchArgs y = x;
    y.m = std::min(rows, x.m - r0);
    y.a = (const char*)x.a + (size_t)r0 * x.w.k * (x.a_is_f16 ? 2 : 4);
    y.c = x.c + (size_t)r0 * x.w.n;
    y.d = x.d ? x.d + (size_t)r0 * x.w.n : nullptr;
    if (y.m != rows && plan_block_rows(y, y.m, kNoLimit, &p) != Found::kPlan) return (int)hipErrorInvalidValue;
    const int e = x.w.fmt == MGN_FMT_Q4 ? launch_block_rows<MGN_FMT_Q4>(s, y, p) : launch_block_rows<MGN_FMT_Q8>(s, y, p);
    if (e) return e;
  }
  return 0;
}

bool describe_block_mfma(const LaunchArgs& x, mgn_block_plan* out) {
  BlockPlan p;
  if (!plan_block(x, kNoLimit, &p)) return false;
  out->rows = p.cfg->rows, out->cols = p.cfg->cols, out->threads = p.cfg->threads, out->lds_bytes = (uint32_t)p.cfg->lds;
  out->row_groups = p.rowgroups, out->col_groups = p.colgroups, out->k_parts = p.parts;
  out->launches = (x.m + p.rows_per_launch - 1) / p.rows_per_launch;
  out->workspace_bytes = p.a_bytes + p.means_bytes + p.inv_bytes + p.partial_bytes;
  out->us = (float)p.us;
  return true;
}

}  // namespace mgn
