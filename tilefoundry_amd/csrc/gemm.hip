// Dense bf16 GEMM for the prefill projections: C[M, N] = A[M, K] . B[N, K]^T
// (activations and weights both K-contiguous, f32 accumulate) on
// v_mfma_f32_32x32x16_bf16, with fused epilogues:
//
//   store         C = bf16(acc)
//   residual      C = bf16(R + bf16(acc))                      (o_proj + residual)
//   f32           C = acc, unrounded                           (prompt prefill; K may be
//                 split into ranges written as separate partial slices, which
//                 the consumers sum in split order)
//   qk_norm_rope  the qkv projection, laid out per token [q_0 | gate_0 | ... |
//                 q_{H-1} | gate_{H-1} | k_0 .. k_{G-1} | v_0 .. v_{G-1}], 256 per
//                 slice: q and k slices get the per-head RMSNorm with (1 + gamma)
//                 in f32 (from the bf16-landed projection) and rotate-half RoPE on
//                 their leading 64 dims (bf16 products and sum); gate and v slices
//                 are stored as the projection landed them.
//   swiglu        C[m, i] = bf16(bf16(silu(bf16 acc[m, 2i])) * bf16 acc[m, 2i + 1]),
//                 the gate and up rows of B interleaved (prompt prefill)
//   qk_rope       a decode model's q|k|v projection, heads of 128: q and k heads
//                 get the per-head RMSNorm and rotate-half RoPE of the decode step;
//                 queries to C, keys and values into their cache rows
//                 (prompt prefill)
//
// Block tiles (BM x BN x 64, two LDS stages) and wave layouts are template
// parameters; a launch picks (see launch()):
//   256 x 256, 8 waves of 128 x 64
//   128 x 128, 4 waves of  64 x 64  (two blocks per CU)
//   128 x 256, 8 waves of  64 x 64
// Two waves share each SIMD, so one wave's LDS reads and barrier waits sit under
// the other's MFMAs.
//
// Main loop: A and B k-slices stream global -> LDS with buffer_load_dwordx4 lds
// (16 bytes per lane, no registers). Rows of 8 16-byte chunks are stored at chunk
// ^ ((row >> 1) & 7), so the 32-row operand reads are conflict-free. A k-tile is
// four phases, one per quadrant of the wave's tile; every instruction beside the
// MFMAs has its slot after one of them (operand reads of the next phase first,
// then stage loads), and the two barriers of a k-tile stand where the operands of
// the phase after them are already in registers. What bounds it: at full grids
// the power limit -- on random data 1.16-1.34 PFLOP/s (8192 x 14336 x 5120, plain
// store 891 us, with the head-norm epilogue 901), on all-zero data 1.64 (734 us, 746)
// -- before that the LDS port, whose operand reads and stage writes take as many
// cycles as the MFMAs. One barrier and a full wait per k-tile, with the first
// reads behind it, took 1,040 us with the head norm where this took 960 (901 since
// the epilogue's sixteen lanes to a head row), and 64 us where this takes 50 (640 x
// 5120 x 6144 + residual with cached weights, 200 blocks of 128 x 128: one per CU, so
// nothing else hides the waits). Also measured, beside the 960: 4 waves of 128 x 128
// (a quarter less LDS traffic, but one wave per SIMD) 1,030 us; stage loads in a
// burst behind each barrier 986 us.
//
// Epilogue (bf16 outputs): the tile lands in bf16 into LDS (rows padded by 32
// bytes), then each wave takes whole rows -- 16 bytes per lane for the store, the
// residual and SwiGLU, 16 lanes per head row for the norm and RoPE -- so every
// global access is a run of whole lines. The f32 store goes straight from the
// accumulators.
//
// Blocks are ordered for the L2s: the dispatcher deals blocks to the 8 XCDs in
// turn, so block b is renumbered to give each XCD a contiguous run of tiles,
// and tiles are numbered in groups of 8 block-rows so that the blocks one XCD
// runs together share A and B k-slices (+17 % on the 8192-token qkv over
// groups of 4).
//
// Reference (jingchangshi/TileFoundry): examples/qwen3_8_27b_prefill-tilelang/kernels/gemm.py:104-356
// (gemm_kernel, "qk_norm_rope" epilogue :226-300, "residual" :193-198), model.py:271-303,326-333.
#include "abi_util.h"
#include "common.h"

using namespace tfa;

namespace {

constexpr int kBK = 64;
constexpr int kXcds = 8;
constexpr int kGroupM = 8;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

// Buffer descriptor of `bytes` from p on: raw (no stride), so a load at or past
// the end returns zero and reads nothing. bytes is wave-uniform.
TFA_DEV i32x4 buffer_of(const void* p, uint32_t bytes) {
  const uint64_t u = reinterpret_cast<uint64_t>(p);
  return i32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(u)),
               __builtin_amdgcn_readfirstlane(static_cast<int>(u >> 32) & 0xffff),
               __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00027000};
}

// 16 / 8 bytes at 8- / 4-byte alignment (the bf16 outputs and the residual need no
// more; the hardware's wide accesses want four bytes)
typedef uint32_t u32x4a8 __attribute__((ext_vector_type(4), aligned(8)));
typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));

TFA_DEV bf16x8 as_bf8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

enum { EPI_STORE = 0, EPI_RESID = 1, EPI_F32 = 2, EPI_QKNR = 3, EPI_SWIGLU = 4, EPI_QKROPE = 5 };

struct GemmArgs {
  const uint16_t* a;      // [M, lda]
  const uint16_t* b;      // [N, ldb]
  uint16_t* c;            // [M, ldc]
  float* cf;              // [M, ldc] (f32 store)
  int M, N, K, lda, ldb, ldc;
  const uint16_t* res;    // residual [M, ldr]
  int ldr;
  const uint16_t* gq;     // q / k head norm weights [256] (the norm scales by 1 + gamma)
  const uint16_t* gk;
  const uint16_t* cos_t;  // [M, 64] rows = positions
  const uint16_t* sin_t;
  int heads, kv_heads;
  float eps;
  int ksplit;             // f32 store: K split into ksplit ranges, range z -> cf + z * M * ldc
  // q|k|v projection of a decode model (head_dim 128): row m is position pos0 + m % seq of sequence m / seq
  uint16_t* kc;           // [batch, cap, kv_heads * 128]
  uint16_t* vc;
  int64_t cap;
  int seq, pos0;
};

TFA_DEV int swz(int row) { return (row >> 1) & 7; }

// Block b's tile (tm, tn) of an nm x nn grid: XCD-contiguous renumbering, then
// groups of GM tile rows walked column by column.
template <int GM>
TFA_DEV void tile_of(int b, int nm, int nn, int& tm, int& tn) {
  const int nb = nm * nn;
  const int per = nb / kXcds, rem = nb % kXcds;
  const int x = b % kXcds, i = b / kXcds;
  const int t = (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i;
  const int group = t / (GM * nn);
  const int first = group * GM;
  const int gsz = min(nm - first, GM);
  const int in = t % (GM * nn);
  tm = first + in % gsz;
  tn = in / gsz;
}

// BM x BN block tile of WM x WN waves, two LDS stages; GM tile rows per group.
template <int BM_, int BN_, int WM_, int WN_, int GM_ = kGroupM>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = 2, GM = GM_;
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kWTM = BM / WM, kWTN = BN / WN;    // wave tile
  static constexpr int kTI = kWTM / 32, kTJ = kWTN / 32;  // MFMA tiles per wave
  static constexpr int kRows = BM + BN;                   // LDS rows per stage: A rows, then B rows
  static constexpr int kStage = kRows * kBK;              // elements per stage
  static constexpr int kEpPitch = BN + 16;                // epilogue LDS row pitch (elements)
  static constexpr int kSmem = (S * kStage > BM * kEpPitch ? S * kStage : BM * kEpPitch);
  static_assert(kWTM % 64 == 0 && kWTN % 64 == 0, "wave tiles of whole quadrants of 32 x 32 MFMA tiles");
  static_assert(kSmem * 2 <= 160 * 1024, "LDS budget");
  static_assert(BN == 128 || BN == 256, "the epilogue's row pass covers 128 or 256 columns");
};

using C256 = Cfg<256, 256, 2, 4>;      // 8 waves of 128 x 64
using C128x256 = Cfg<128, 256, 2, 4>;  // 8 waves of 64 x 64
using C128 = Cfg<128, 128, 2, 2>;      // 4 waves of 64 x 64, two blocks per CU

constexpr int kWaitVm0 = waitcnt_vm(0);

template <class C, int EPI, bool WIDE>
__global__ __launch_bounds__(C::kThreads) void gemm_kernel(const GemmArgs a) {
  constexpr int BM = C::BM, BN = C::BN, TI = C::kTI, TJ = C::kTJ;
  __shared__ __attribute__((aligned(1024))) uint16_t smem[C::kSmem];

  const int lane = threadIdx.x & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n32 = lane & 31;
  const int kg = lane >> 5;
  const int wm = (wid / C::WN) * C::kWTM, wn = (wid % C::WN) * C::kWTN;
  const int nm = (a.M + BM - 1) / BM, nn = a.N / BN;
  int tm, tn;
  tile_of<C::GM>(blockIdx.x, nm, nn, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // f32 store with a split K: block row z of the grid takes k-tiles
  // [z nk / ksplit, (z + 1) nk / ksplit) and writes its own partial slice
  int nk = a.K / kBK;
  int kt0 = 0;
  if (EPI == EPI_F32 && a.ksplit > 1) {
    nk /= a.ksplit;
    kt0 = blockIdx.y * nk;
  }
  // Stage loads go out in two groups, each half of what every wave reads: group g
  // holds the g-th half of each wave's A rows and of its B rows. A load fills 8
  // stage rows; lane l lands at row + l/8, chunk slot l % 8, and so brings logical
  // chunk (l % 8) ^ swz(row). They are buffer loads: one descriptor per (group,
  // matrix) holds the wave's first row, the lane offsets are loop-invariant and a
  // k-tile is a scalar offset. Rows past M lie past the descriptor's end and come
  // as zeros (never stored); so does every row of a k-tile past the last one, whose
  // load is issued against an empty descriptor and moves nothing -- the k loop's
  // body and its wait counts are the same to the end. WIDE (row pitches whose 16
  // rows a 32-bit descriptor does not span): a 64-bit address per lane instead, with
  // rows past M reading row M - 1 and k-tiles past the last one the last again.
  constexpr int kHA = C::kWTM / 2, kHB = C::kWTN / 2;        // rows of one wave's half
  constexpr int kGA = BM / 16 / C::kWaves, kGB = BN / 16 / C::kWaves, kGD = kGA + kGB;   // loads per wave and group
  static_assert(kGA >= 1 && kGB >= 1 && kHA % (8 * kGA) == 0 && kHB % (8 * kGB) == 0 && kHA % 16 == 0 && kHB % 16 == 0,
                "a wave's loads of a group are consecutive rows of one half");
  static_assert(kGD * 2 * 8 * C::kWaves == C::kRows, "two groups fill a stage");
  i32x4 rsrc[2][2];                 // [group][A, B]
  uint32_t voff[kGD], dst[kGD];     // lane offsets (both groups); LDS byte offsets of group 0
  const char* wsrc[WIDE ? 2 : 1][WIDE ? kGD : 1];
  {
    const int ra = 8 * kGA * wid, rb = 8 * kGB * wid;
    const int rowa = ra / kHA * C::kWTM + ra % kHA, rowb = rb / kHB * C::kWTN + rb % kHB;   // stage rows of group 0
#pragma unroll
    for (int g = 0; g < 2 && !WIDE; ++g) {
      const int first = min(m0 + rowa + g * kHA, a.M - 1);
      rsrc[g][0] = buffer_of(a.a + static_cast<size_t>(first) * a.lda, 2u * a.lda * min(a.M - first, 8 * kGA));
      rsrc[g][1] = buffer_of(a.b + static_cast<size_t>(n0 + rowb + g * kHB) * a.ldb, 2u * a.ldb * (8 * kGB));
    }
    const int l3 = lane >> 3;
#pragma unroll
    for (int i = 0; i < kGD; ++i) {
      const bool isa = i < kGA;
      const int j = 8 * (isa ? i : i - kGA), row = (isa ? rowa : rowb) + j;
      const int chunk = 8 * ((lane & 7) ^ swz(row + l3));   // the same in both groups
      dst[i] = lds_offset(&smem[((isa ? 0 : BM) + row) * kBK]);
      if constexpr (WIDE) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const int r = row + g * (isa ? kHA : kHB) + l3;
          wsrc[g][i] = reinterpret_cast<const char*>(
              (isa ? a.a + static_cast<size_t>(min(m0 + r, a.M - 1)) * a.lda : a.b + static_cast<size_t>(n0 + r) * a.ldb) + chunk);
        }
      } else {
        voff[i] = 2u * ((j + l3) * (isa ? a.lda : a.ldb) + chunk);
      }
    }
  }
  // k-tile kt's scalar offset; past the last k-tile the descriptors are emptied
  auto at_tile = [&](int kt) __attribute__((always_inline)) {
    if constexpr (WIDE) return static_cast<uint32_t>((kt0 + min(kt, nk - 1)) * (kBK * 2));
    const int keep = kt < nk ? -1 : 0;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int x = 0; x < 2; ++x) rsrc[g][x][2] &= keep;
    return static_cast<uint32_t>((kt0 + kt) * (kBK * 2)) & static_cast<uint32_t>(keep);
  };
  // load i of group g into stage st
  auto dma1 = [&](int g, int i, uint32_t soff, int st) __attribute__((always_inline)) {
    const uint32_t half = (i < kGA ? kHA : kHB) * kBK * 2;
    const uint32_t to = dst[i] + g * half + st * C::kStage * 2;
    if constexpr (WIDE)
      lds_dma16(wsrc[g][i] + soff, to);
    else
      asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff[i]), "s"(rsrc[g][i < kGA ? 0 : 1]), "s"(soff),
                   "{m0}"(to) : "memory");
  };
  auto dma = [&](int g, uint32_t kt, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kGD; ++i) dma1(g, i, kt, st);
  };

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // K loop in four phases per k-tile, one per quadrant of the wave's tile (A half,
  // B half): (0,0) (0,1) (1,1) (1,0). The operands of a phase are read under the
  // MFMAs of the one before it, so group 0 of a stage is free again when phase 0
  // begins and group 1 when phase 3 does, and each is refilled there -- two tiles
  // on -- 1.25 to 1.75 k-tiles before it is read. Two barriers per k-tile:
  //   B0 (before phase 0)  group 1 of this tile landed; every wave has read group 0
  //   B3 (before phase 3)  group 0 of the next tile landed; every wave has read group 1
  constexpr int kKs = kBK / 16, HI = TI / 2, HJ = TJ / 2;
  const int sx = swz(n32);   // every operand row this lane reads is wm (or BM + wn) + 32 i + n32
  // LDS byte address of this lane's first chunk of its A and B rows. A k-step's
  // chunk is that address with bits 5..6 flipped (the row pitch is 128 bytes), so
  // one add-xor gives a read's address; the bases are kept opaque, or every
  // (k-step, stage) address would be held in a register of its own.
  typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
  uint32_t abase = lds_offset(&smem[(wm + n32) * kBK]) + 16 * (kg ^ sx);
  uint32_t bbase = lds_offset(&smem[(BM + wn + n32) * kBK]) + 16 * (kg ^ sx);
  uint4 av[2][kKs][HI], bv[2][kKs][HJ];
  auto lds16 = [&](uint32_t base, int ks, int bytes) __attribute__((always_inline)) {
    const u32x4 v = *reinterpret_cast<lds_u32x4*>((base ^ (32u * ks)) + static_cast<uint32_t>(bytes));
    return make_uint4(v.x, v.y, v.z, v.w);
  };
  auto rdA = [&](int st, int h, int idx) __attribute__((always_inline)) {
    const int ks = idx / HI, i = idx % HI;
    av[h][ks][i] = lds16(abase, ks, st * C::kStage * 2 + 32 * (h * HI + i) * kBK * 2);
  };
  auto rdB = [&](int st, int h, int slot, int idx) __attribute__((always_inline)) {
    const int ks = idx / HJ, j = idx % HJ;
    bv[slot][ks][j] = lds16(bbase, ks, st * C::kStage * 2 + 32 * (h * HJ + j) * kBK * 2);
  };
  constexpr int kPh = kKs * HI * HJ;   // MFMAs per phase
  // MFMA m of quadrant (ha, hb), B operands in slot
  auto mm = [&](int ha, int hb, int slot, int m) __attribute__((always_inline)) {
    const int ks = m / (HI * HJ), i = m % (HI * HJ) / HJ, j = m % HJ;
    acc[ha * HI + i][hb * HJ + j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        as_bf8(av[ha][ks][i]), as_bf8(bv[slot][ks][j]), acc[ha * HI + i][hb * HJ + j], 0, 0, 0);
  };
  constexpr int kRA = kKs * HI, kRB = kKs * HJ;   // operand reads of a half

  uint32_t soff = at_tile(0);
  dma(0, soff, 0);
  dma(1, soff, 0);
  soff = at_tile(1);
  dma(0, soff, 1);
  dma(1, soff, 1);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(3 * kGD));
  block_barrier();
#pragma unroll
  for (int r = 0; r < kRB; ++r) rdB(0, 0, 0, r);
#pragma unroll
  for (int r = 0; r < kRA; ++r) rdA(0, 0, r);
  // one phase: its MFMAs, with nr operand reads spread over the first half and nd
  // stage loads over the second, each pinned after its MFMA
  auto phase = [&](int ha, int hb, int slot, auto nrc, auto rd, auto ndc, auto ldd) __attribute__((always_inline)) {
    constexpr int nr = decltype(nrc)::value, nd = decltype(ndc)::value;
    constexpr int half = nd ? kPh / 2 : kPh * 3 / 4;
#pragma unroll
    for (int m = 0; m < kPh; ++m) {
      mm(ha, hb, slot, m);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = m * nr / half; r < (m + 1) * nr / half && r < nr; ++r) rd(r);
      if (nd && m >= half) {
#pragma unroll
        for (int d = (m - half) * nd / (kPh - half); d < (m + 1 - half) * nd / (kPh - half); ++d) ldd(d);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto none = [](int) {};
  using Z = std::integral_constant<int, 0>;
  // tile kt in stage ST, its B half 0 in slot ST
  auto tile = [&](int kt, auto stc) __attribute__((always_inline)) {
    constexpr int ST = decltype(stc)::value;
    using ND = std::integral_constant<int, kGD>;
    asm volatile("" : "+v"(abase), "+v"(bbase));
    const uint32_t soff = at_tile(kt + 2);
    // B0
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kGD) & kWaitLgkm0);
    block_barrier();
    __builtin_amdgcn_sched_barrier(0);
    phase(0, 0, ST, std::integral_constant<int, kRB>{}, [&](int r) __attribute__((always_inline)) { rdB(ST, 1, ST ^ 1, r); }, ND{},
          [&](int d) __attribute__((always_inline)) { dma1(0, d, soff, ST); });
    phase(0, 1, ST ^ 1, std::integral_constant<int, kRA>{}, [&](int r) __attribute__((always_inline)) { rdA(ST, 1, r); }, Z{}, none);
    phase(1, 1, ST ^ 1, Z{}, none, Z{}, none);
    // B3
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kGD) & kWaitLgkm0);
    block_barrier();
    __builtin_amdgcn_sched_barrier(0);
    phase(1, 0, ST, std::integral_constant<int, kRA + kRB>{},
          [&](int r) __attribute__((always_inline)) {
            if (r < kRB) rdB(ST ^ 1, 0, ST ^ 1, r);
            else rdA(ST ^ 1, 0, r - kRB);
          },
          ND{}, [&](int d) __attribute__((always_inline)) { dma1(1, d, soff, ST); });
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    tile(kt, S0{});
    tile(kt + 1, S1{});
  }
  if (kt < nk) tile(kt, S0{});
  __builtin_amdgcn_s_waitcnt(kWaitVm0);   // no load may still be writing this block's LDS

  // acc[i][j][4t + r]: tile row wm + 32 i + 8 t + 4 kg + r, column wn + 32 j + n32
  if (EPI == EPI_F32) {
    float* cf = a.cf + static_cast<size_t>(blockIdx.y) * a.M * a.ldc;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + wm + 32 * i + 8 * t + 4 * kg + r;
          if (row >= a.M) continue;
#pragma unroll
          for (int j = 0; j < TJ; ++j)
            cf[static_cast<size_t>(row) * a.ldc + n0 + wn + 32 * j + n32] = acc[i][j][4 * t + r];
        }
    return;
  }

  // bf16 tile into LDS (rows padded by 16 elements), then whole rows out
  block_barrier();   // every wave's last operand reads are consumed: the stages are free
  uint16_t* ep = smem;
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          ep[(wm + 32 * i + 8 * t + 4 * kg + r) * C::kEpPitch + wn + 32 * j + n32] =
              static_cast<uint16_t>(f2bf(acc[i][j][4 * t + r]));
  lds_barrier();

  // Every global input of the row passes -- the residual rows, or the rope rows --
  // is issued before the first pass, into the registers the accumulators held: one
  // memory round trip for the epilogue instead of one per pass. A pass is bound by
  // its vector instructions (a tile's passes take as long as 10-20 of its k-tiles),
  // so a row's sum and inverse root are shared by as many elements as the layout
  // allows: 16 lanes hold a head row, four rows to a wave.
  auto rows = [&](auto rppc, int sub, auto body) __attribute__((always_inline)) {
    constexpr int RPP = decltype(rppc)::value, kPasses = BM / (C::kWaves * RPP);
    static_assert(kPasses * C::kWaves * RPP == BM, "whole row passes per wave");
#pragma unroll
    for (int p = 0; p < kPasses; ++p) body(p, (p * C::kWaves + wid) * RPP + sub);
  };
  const int j16 = lane & 15, g16 = lane >> 4;
  if constexpr (EPI == EPI_STORE || EPI == EPI_RESID || EPI == EPI_SWIGLU) {
    constexpr int kLPR = BN / 8, RPP = kWave / kLPR;   // lanes per row, 8 elements each
    const int sub = lane / kLPR, cl = lane % kLPR * 8;
    using R = std::integral_constant<int, RPP>;
    u32x4a8 pre[EPI == EPI_RESID ? BM / (C::kWaves * RPP) : 1];
    if constexpr (EPI == EPI_RESID)
      rows(R{}, sub, [&](int p, int row) __attribute__((always_inline)) {
        const int grow = min(m0 + row, a.M - 1);
        pre[p] = *reinterpret_cast<const u32x4a8*>(a.res + static_cast<size_t>(grow) * a.ldr + n0 + cl);
      });
    rows(R{}, sub, [&](int p, int row) __attribute__((always_inline)) {
      const int grow = m0 + row;
      if (grow >= a.M) return;
      u32x4 v = *reinterpret_cast<const u32x4*>(ep + row * C::kEpPitch + cl);
      if constexpr (EPI == EPI_SWIGLU) {
        // columns 2 i, 2 i + 1 are gate and up of output i; the decode step's order and
        // its divided silu, so a prompt row lands as the same token decoded does:
        // bf16(bf16(silu(bf16 g)) * bf16 u)
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = lo_bf(v[i]);
          y[i] = round_bf(x / (1.0f + expf(-x))) * hi_bf(v[i]);
        }
        *reinterpret_cast<u32x2a4*>(a.c + static_cast<size_t>(grow) * a.ldc + (n0 + cl) / 2) =
            u32x2a4{pack_bf(y[0], y[1]), pack_bf(y[2], y[3])};
      } else {
        if constexpr (EPI == EPI_RESID) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = pack_bf(lo_bf(pre[p][i]) + lo_bf(v[i]), hi_bf(pre[p][i]) + hi_bf(v[i]));
        }
        *reinterpret_cast<u32x4a8*>(a.c + static_cast<size_t>(grow) * a.ldc + n0 + cl) = v;
      }
    });
  } else if constexpr (EPI == EPI_QKNR) {
    // a 256-column slice: lane j of a row's 16 holds columns 64 c + 4 j .. + 3, so the
    // 64 rotated columns are chunk 0 and partners (32 apart) are lanes j and j ^ 8
    using R = std::integral_constant<int, 4>;
    const int sl = n0 / 256;
    const bool norm = sl < 2 * a.heads ? (sl & 1) == 0 : sl < 2 * a.heads + a.kv_heads;   // not a gate or v slice
    const uint16_t* gamma = sl < 2 * a.heads ? a.gq : a.gk;
    float gm[4][4];
    uint2 pre_c[BM / (C::kWaves * 4)], pre_s[BM / (C::kWaves * 4)];
    if (norm) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint2 gv = *reinterpret_cast<const uint2*>(gamma + 64 * c + 4 * j16);
        gm[c][0] = 1.0f + lo_bf(gv.x); gm[c][1] = 1.0f + hi_bf(gv.x);
        gm[c][2] = 1.0f + lo_bf(gv.y); gm[c][3] = 1.0f + hi_bf(gv.y);
      }
      rows(R{}, g16, [&](int p, int row) __attribute__((always_inline)) {
        const size_t o = static_cast<size_t>(min(m0 + row, a.M - 1)) * 64 + 4 * j16;
        pre_c[p] = *reinterpret_cast<const uint2*>(a.cos_t + o);
        pre_s[p] = *reinterpret_cast<const uint2*>(a.sin_t + o);
      });
    }
    rows(R{}, g16, [&](int p, int row) __attribute__((always_inline)) {
      const int grow = m0 + row;
      uint2 v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = *reinterpret_cast<const uint2*>(ep + row * C::kEpPitch + 64 * c + 4 * j16);
      if (norm) {
        // x -> bf16(x * rsqrt(mean x^2 + eps) * (1 + gamma)) in f32; then rotate-half,
        // products and sum in bf16
        float x[4][4], ss = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          x[c][0] = lo_bf(v[c].x); x[c][1] = hi_bf(v[c].x); x[c][2] = lo_bf(v[c].y); x[c][3] = hi_bf(v[c].y);
#pragma unroll
          for (int i = 0; i < 4; ++i) ss = fmaf(x[c][i], x[c][i], ss);
        }
        const float inv = rsqrt_rn(row16_sum(ss) / 256.0f + a.eps);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) x[c][i] = x[c][i] * inv * gm[c][i];
#pragma unroll
        for (int c = 1; c < 4; ++c) v[c] = make_uint2(pack_bf(x[c][0], x[c][1]), pack_bf(x[c][2], x[c][3]));
        const float ct[4] = {lo_bf(pre_c[p].x), hi_bf(pre_c[p].x), lo_bf(pre_c[p].y), hi_bf(pre_c[p].y)};
        const float st[4] = {lo_bf(pre_s[p].x), hi_bf(pre_s[p].x), lo_bf(pre_s[p].y), hi_bf(pre_s[p].y)};
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float n = round_bf(x[0][i]);
          const float partner = xor_lane<8>(n, lane);   // rotate_half: the first half pairs with -x[d + 32]
          y[i] = round_bf(n * ct[i]) + round_bf((j16 < 8 ? -partner : partner) * st[i]);
        }
        v[0] = make_uint2(pack_bf(y[0], y[1]), pack_bf(y[2], y[3]));
      }
      if (grow >= a.M) return;
      uint16_t* dst = a.c + static_cast<size_t>(grow) * a.ldc + n0 + 4 * j16;
#pragma unroll
      for (int c = 0; c < 4; ++c) *reinterpret_cast<uint2*>(dst + 64 * c) = v[c];
    });
  } else {
    static_assert(EPI == EPI_QKROPE || EPI == EPI_F32, "every epilogue is handled");
    // heads of 128: lane j of a head row's 16 holds columns 4 j .. + 3 and 64 + 4 j ..,
    // so a pair (64 apart) is in one lane. The decode step's norm, x -> bf16(bf16(x r)
    // gamma), then rotate-half, each product in f32 and the sum landing; keys and
    // values go into their cache rows.
    constexpr int kHeads = BN / 128;   // heads in the tile's columns, one per 16 lanes
    using R = std::integral_constant<int, 4 / kHeads>;
    const int sub = g16 / kHeads, col = g16 % kHeads * 128 + 4 * j16;
    const int hh = n0 / 128 + g16 % kHeads;
    const bool norm = hh < a.heads + a.kv_heads;   // not a value head
    const uint16_t* gamma = hh < a.heads ? a.gq : a.gk;
    float gm[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint2 gv = *reinterpret_cast<const uint2*>(gamma + 64 * h + 4 * j16);
      gm[4 * h] = lo_bf(gv.x); gm[4 * h + 1] = hi_bf(gv.x); gm[4 * h + 2] = lo_bf(gv.y); gm[4 * h + 3] = hi_bf(gv.y);
    }
    uint2 pre_c[BM * kHeads / (C::kWaves * 4)][2], pre_s[BM * kHeads / (C::kWaves * 4)][2];
    rows(R{}, sub, [&](int p, int row) __attribute__((always_inline)) {
      const unsigned grow = min(m0 + row, a.M - 1);
      const size_t o = static_cast<size_t>(a.pos0 + grow % static_cast<unsigned>(a.seq)) * 128 + 4 * j16;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        pre_c[p][h] = *reinterpret_cast<const uint2*>(a.cos_t + o + 64 * h);
        pre_s[p][h] = *reinterpret_cast<const uint2*>(a.sin_t + o + 64 * h);
      }
    });
    rows(R{}, sub, [&](int p, int row) __attribute__((always_inline)) {
      const int grow = m0 + row;
      uint2 v[2];
      float x[8], ss = 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v[h] = *reinterpret_cast<const uint2*>(ep + row * C::kEpPitch + col + 64 * h);
        x[4 * h] = lo_bf(v[h].x); x[4 * h + 1] = hi_bf(v[h].x); x[4 * h + 2] = lo_bf(v[h].y); x[4 * h + 3] = hi_bf(v[h].y);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
      const float rs = rsqrt_rn(row16_sum(ss) / 128.0f + a.eps);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = round_bf(round_bf(x[i] * rs) * gm[i]);
      float y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint2 cv = pre_c[p][i / 4], sv = pre_s[p][i / 4];
        const uint32_t cw = (i & 2) ? cv.y : cv.x, sw = (i & 2) ? sv.y : sv.x;
        const float ct = (i & 1) ? hi_bf(cw) : lo_bf(cw), st = (i & 1) ? hi_bf(sw) : lo_bf(sw);
        y[i] = __fadd_rn(__fmul_rn(x[i], ct), __fmul_rn(i < 4 ? -x[i + 4] : x[i - 4], st));
      }
      if (norm) {
        v[0] = make_uint2(pack_bf(y[0], y[1]), pack_bf(y[2], y[3]));
        v[1] = make_uint2(pack_bf(y[4], y[5]), pack_bf(y[6], y[7]));
      }
      if (grow >= a.M) return;
      const unsigned b = static_cast<unsigned>(grow) / static_cast<unsigned>(a.seq);
      const int64_t crow = (b * a.cap + a.pos0 + (grow - b * a.seq)) * a.kv_heads;
      uint16_t* dst = hh < a.heads ? a.c + (static_cast<int64_t>(grow) * a.heads + hh) * 128
                      : norm       ? a.kc + (crow + hh - a.heads) * 128
                                   : a.vc + (crow + hh - a.heads - a.kv_heads) * 128;
      *reinterpret_cast<uint2*>(dst + 4 * j16) = v[0];
      *reinterpret_cast<uint2*>(dst + 64 + 4 * j16) = v[1];
    });
  }
}

template <class C, int EPI, bool WIDE = false>
int launch_cfg(const GemmArgs& g, hipStream_t st, const char* name) {
  const int nm = (g.M + C::BM - 1) / C::BM, nn = g.N / C::BN;
  const unsigned splits = EPI == EPI_F32 && g.ksplit > 1 ? (unsigned)g.ksplit : 1u;
  gemm_kernel<C, EPI, WIDE><<<dim3((unsigned)(nm * nn), splits), C::kThreads, 0, st>>>(g);
  return launched(name);
}

// The f32 store's choice, and the plan of its splits: a grid of 256 x 256 tiles that
// fills at least 80 % of its last round of one block per CU.
bool full_rounds_256(int64_t m, int64_t n, int cus) {
  const int64_t b256 = (m + 255) / 256 * (n / 256);
  const int64_t rounds = (b256 + cus - 1) / cus;
  return n % 256 == 0 && b256 * 5 >= rounds * cus * 4;
}

// K splits for the f32 store: a small grid (few token rows) of 128 x 128 tiles
// is split along K -- doubling while every block still gets a CU of its own, each
// range keeps at least 8 k-tiles (4 up to 64 rows, whose partials are small), and
// the count divides the k-tiles -- up to 8. Two blocks to a CU gain nothing in the
// product and double the partials. Measured with the consumer, over uncached
// weights, us, at 1 / 2 / 4 / 8 splits: 4096 x 2048 at 509 rows (128 blocks) 29.4 / 23.8 /
// 29.0 / 38.6, at 128 rows (32) 25.1 / 17.5 / 14.0 / 15.0, at 61 rows 23.0 / 15.9 / 12.5 /
// 11.5; 12288 x 2048 at 61 (96) 24.9 / 18.4 / 20.9 / 25.9; 2048 x 6144 at 509 (64) 63.3 /
// 38.9 / 27.7 / 33.4, at 999 (128) 65.6 / 42.2 / 45.4 / 57.9.
// The split count sets the order the consumers sum the partials in, and so the
// rounding of everything after the prompt prefill; it is therefore derived from
// the shape and MI355X's fixed 256 CUs, never from the device's reported count,
// so that a given prompt prefills to the same bits on any gfx950 part.
constexpr int kSplitPlanCus = 256;

int64_t splits_f32(int64_t m, int64_t n, int64_t k) {
  const int cus = kSplitPlanCus;
  if (full_rounds_256(m, n, cus) || n % 128 || k % kBK) return 1;
  const int64_t blocks = (m + 127) / 128 * (n / 128), nk = k / kBK;
  int64_t ks = 1;
  const int64_t least = m <= 64 ? 4 : 8;
  while (ks < kMaxSplitsK && blocks * ks * 2 <= cus && nk % (ks * 2) == 0 && nk / (ks * 2) >= least) ks *= 2;
  return ks;
}

// Whether a projection of the prompt prefill runs unsplit with its consumer in the
// epilogue (bf16 out) rather than as f32 split-K partials and a second launch. The
// fused form saves the partials' store and re-read (8 bytes a value and split),
// but with fewer 128 x 128 blocks than CUs it cannot draw the weights from HBM as
// fast as a split grid. Measured over weights not in any cache, split + consumer
// against fused, us: 12288 x 2048 (SwiGLU) 26.0 / 27.6 at 128 rows (96 blocks),
// 28.2 / 24.4 at 200 (192), 50.4 / 34.9 at 509, 493 / 356 at 8000; 4096 x 2048
// (norm, RoPE, cache rows) 29.0 / 28.5 at 509 (128), 33.2 / 28.4 at 700 (192), 214 /
// 146 at 8000; 2048 x 2048 (residual, norm) 25.7 / 26.9 at 999 (128), 31.8 / 27.9 at
// 1500 (192); 2048 x 6144 45.3 / 67.1 at 999, 66.8 / 67.3 at 1500, 71.1 / 67.0 at 2000
// (256). The line is three quarters of the CUs. Like the split plan it is a
// function of the shape alone.
bool fused_epilogue(int64_t m, int64_t n, int64_t k) {
  if (n % 128 || k % kBK) return false;
  return (m + 127) / 128 * (n / 128) * 4 >= kSplitPlanCus * 3;
}

// Tile choice of the bf16 stores: the least of three costs, in hundredths of a full
// round of 256 x 256 tiles (62 us at 12288 x 2048, 105 at 8192 x 4096, 155 at 5120 x
// 6144). Blocks run in rounds, one per CU (two of the 128 x 128 tile). A first round
// waits for weights out of HBM whatever it holds, so a part-filled round of large tiles
// costs most of a full one; later rounds overlap the one before and a nearly empty last
// one adds a third. Fitted to six shapes at 36 row counts each over uncached weights
// (with cached ones a round of 128 x 256 looks as cheap as 50 of 5120 x 6144's 75 us, and
// 101 is what it takes): the tile picked is within 5 % of the best at all of them.
// Examples, us, 256 x 256 / 128 x 256 / 128 x 128: 5120 x 6144 at 640
// rows 121 / 103 / 69, 896 121 / 102 / 94, 1152 117 / 101 / 114, 1664 130 / 159 / 153, 4608
// 277 / 270 / 305, 8192 452 / 511 / 541; 12288 x 2048 with SwiGLU at 509 51 / 36 / 40, 1500
// 106 / 95 / 85, 4000 186 / 207 / 205; 8192 x 4096 at 1280 88 / 111 / 99.
enum { TILE_256, TILE_128x256, TILE_128 };

int pick_tile(int64_t m, int64_t n, int64_t k, int cus) {
  if (n % 256) return TILE_128;
  const int64_t rows128 = (m + 127) / 128;
  const int64_t b256 = (m + 255) / 256 * (n / 256), bx = rows128 * (n / 256), b128 = rows128 * (n / 128);
  const int64_t l256 = b256 % cus, lx = bx % cus, l128 = b128 % (2 * cus);   // blocks of the last, part-filled round
  const int64_t c256 = b256 / cus * 100 + (l256 ? 71 + 21 * l256 / cus : 0);
  // (a lone round over a long K is a little dearer: 288 blocks of 128 x 128 take 94 us of 6144
  // where 144 take 102, 35.5 of 2048 where 144 take 33)
  const int64_t cx = bx <= cus ? (k > 4096 ? 66 : 65) : 65 + (bx / cus - 1) * 54 + (lx ? 30 + 18 * lx / cus : 0);
  auto two = [&](int one, int both, int more) -> int64_t {   // up to one block on each CU, or two on some
    return l128 == 0 ? 0 : l128 <= cus ? one : both + more * (l128 - cus) / cus;
  };
  const int64_t c128 = b128 < 2 * cus ? two(46, 64, 8) : 72 + (b128 / (2 * cus) - 1) * 57 + two(20, 50, 17);
  if (c256 <= cx && c256 <= c128) return TILE_256;
  return cx <= c128 ? TILE_128x256 : TILE_128;
}

// Row pitch (elements) from which a wave's 16 stage rows no longer fit a 32-bit
// descriptor: 16 rows * 2 bytes * 2^27 = 2^32, and the lane offsets wrap with it.
constexpr int kWidePitch = 1 << 27;

template <int EPI>
int launch(const GemmArgs& g, hipStream_t st, const char* name) {
  const int cus = device_cus();
  if constexpr (EPI != EPI_QKNR) {   // (its operands are contiguous, at most 2^24 wide)
    if (g.lda >= kWidePitch || g.ldb >= kWidePitch) return launch_cfg<C128, EPI, true>(g, st, name);
  }
  if constexpr (EPI == EPI_QKNR) {
    // Whole 256-column head slices: 256 or 128 rows, by rounds of one block per CU. A
    // 128-row round takes two thirds of a 256-row one (the weights' half of the
    // traffic is the same). Measured, 14336 x 5120 over uncached weights, us, 256 / 128
    // rows: 512 tokens 123 / 89 (one round each), 640 114 / 134 (one, two), 768 124 / 163,
    // 1152 218 / 181 (two, two), 1536 248 / 236 (two, three), 1792 252 / 281 (two, four).
    if (g.N % 256) return fail(TFA_ERR_SHAPE, "%s: the qkv width must be a multiple of 256", name);
    auto rounds = [&](int64_t rows) { return ((g.M + rows - 1) / rows * (g.N / 256) + cus - 1) / cus; };
    return rounds(128) * 66 < rounds(256) * 100 ? launch_cfg<C128x256, EPI>(g, st, name)
                                                : launch_cfg<C256, EPI>(g, st, name);
  } else if constexpr (EPI == EPI_F32) {
    return full_rounds_256(g.M, g.N, cus) && g.ksplit == 1 ? launch_cfg<C256, EPI>(g, st, name)
                                                            : launch_cfg<C128, EPI>(g, st, name);
  } else {
    switch (pick_tile(g.M, g.N, g.K, cus)) {
      case TILE_256: return launch_cfg<C256, EPI>(g, st, name);
      case TILE_128x256: return launch_cfg<C128x256, EPI>(g, st, name);
      default: return launch_cfg<C128, EPI>(g, st, name);
    }
  }
}

int check_gemm(const void* a, const void* b, const void* c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
               int64_t ldc, const char* fn) {
  if (!a || !b || !c) return fail(TFA_ERR_NULL, "%s: null pointer argument", fn);
  if (m < 1 || n < 128 || n % 128 || k < kBK || k % kBK || m > (1 << 24) || n > (1 << 24) || k > (1 << 24))
    return fail(TFA_ERR_SHAPE, "%s: m %lld must be positive, n %lld a multiple of 128, k %lld of 64", fn,
                (long long)m, (long long)n, (long long)k);
  if (lda < k || ldb < k || ldc < n || lda % 8 || ldb % 8 || ldc % 4)
    return fail(TFA_ERR_SHAPE, "%s: leading dimensions too small, or lda / ldb not multiples of 8, ldc of 4", fn);
  if (ldb > INT32_MAX || (m > 1 && (lda > INT32_MAX || ldc > INT32_MAX)))   // a single row has no pitch
    return fail(TFA_ERR_SHAPE, "%s: row pitches of 2^31 elements and more are not supported", fn);
  if (!aligned16(a) || !aligned16(b)) return fail(TFA_ERR_ALIGN, "%s: a / b not 16-byte aligned", fn);
  if ((reinterpret_cast<uintptr_t>(c) & 7u) != 0) return fail(TFA_ERR_ALIGN, "%s: c not 8-byte aligned", fn);
  return TFA_OK;
}

GemmArgs make(const void* a, const void* b, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc) {
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a);
  g.b = static_cast<const uint16_t*>(b);
  g.M = (int)m; g.N = (int)n; g.K = (int)k;
  g.lda = (int)(m == 1 ? k : lda);   // a single row has no pitch
  g.ldb = (int)ldb; g.ldc = (int)ldc;
  return g;
}

}  // namespace

extern "C" {

int tfa_gemm_nt(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                int64_t ldc, const void* residual, int64_t ldr, hipStream_t stream) {
  const int st = check_gemm(a, b, c, m, n, k, lda, ldb, ldc, "tfa_gemm_nt");
  if (st != TFA_OK) return st;
  GemmArgs g = make(a, b, m, n, k, lda, ldb, ldc);
  g.c = static_cast<uint16_t*>(c);
  if (residual) {
    TFA_REQUIRE(ldr >= n && ldr % 4 == 0 && (m == 1 || ldr <= INT32_MAX), TFA_ERR_SHAPE,
                "tfa_gemm_nt: ldr %lld < n %lld, not a multiple of 4 or past 2^31", (long long)ldr, (long long)n);
    TFA_REQUIRE((reinterpret_cast<uintptr_t>(residual) & 7u) == 0, TFA_ERR_ALIGN,
                "tfa_gemm_nt: residual not 8-byte aligned");
    g.res = static_cast<const uint16_t*>(residual);
    g.ldr = (int)ldr;
    return launch<EPI_RESID>(g, stream, "gemm_nt_residual");
  }
  return launch<EPI_STORE>(g, stream, "gemm_nt");
}

int tfa_gemm_nt_f32(const void* a, const void* b, float* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                    int64_t ldb, int64_t ldc, hipStream_t stream) {
  return tfa_gemm_nt_f32_split(a, b, c, m, n, k, lda, ldb, ldc, 1, stream);
}

int64_t tfa_gemm_f32_splits(int64_t m, int64_t n, int64_t k) { return splits_f32(m, n, k); }

int tfa_gemm_fused_epilogue(int64_t m, int64_t n, int64_t k) { return fused_epilogue(m, n, k) ? 1 : 0; }

int tfa_gemm_nt_f32_split(const void* a, const void* b, float* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                          int64_t ldb, int64_t ldc, int64_t ks, hipStream_t stream) {
  const int st = check_gemm(a, b, c, m, n, k, lda, ldb, ldc, "tfa_gemm_nt_f32");
  if (st != TFA_OK) return st;
  TFA_REQUIRE(ks >= 1 && ks <= kMaxSplitsK && (k / kBK) % ks == 0, TFA_ERR_SHAPE,
              "tfa_gemm_nt_f32: %lld splits must be in [1, %d] and divide the %lld k-tiles of 64", (long long)ks,
              kMaxSplitsK, (long long)(k / kBK));
  GemmArgs g = make(a, b, m, n, k, lda, ldb, ldc);
  g.cf = c;
  g.ksplit = (int)ks;
  return launch<EPI_F32>(g, stream, "gemm_nt_f32");
}

int tfa_gemm_nt_swiglu(const void* a, const void* b, void* act, int64_t m, int64_t n, int64_t k, int64_t lda,
                       int64_t ldb, int64_t ldact, hipStream_t stream) {
  const int st = check_gemm(a, b, act, m, n, k, lda, ldb, n, "tfa_gemm_nt_swiglu");
  if (st != TFA_OK) return st;
  TFA_REQUIRE(ldact >= n / 2 && ldact % 2 == 0 && (m == 1 || ldact <= INT32_MAX), TFA_ERR_SHAPE,
              "tfa_gemm_nt_swiglu: ldact %lld below n / 2 = %lld, odd or past 2^31", (long long)ldact, (long long)(n / 2));
  GemmArgs g = make(a, b, m, n, k, lda, ldb, ldact);
  g.c = static_cast<uint16_t*>(act);
  return launch<EPI_SWIGLU>(g, stream, "gemm_nt_swiglu");
}

int tfa_gemm_nt_qk_rope(const void* a, const void* w_qkv, int64_t batch, int64_t n, int64_t k, int64_t lda,
                        int64_t ldw, const void* gamma_q, const void* gamma_k, float eps_head, const void* cos_t,
                        const void* sin_t, int64_t rope_rows, int64_t pos0, void* k_cache, void* v_cache, int64_t cap,
                        void* q_out, int64_t hq, int64_t hkv, int64_t head_dim, hipStream_t stream) {
  if (!gamma_q || !gamma_k || !cos_t || !sin_t || !k_cache || !v_cache)
    return fail(TFA_ERR_NULL, "tfa_gemm_nt_qk_rope: null pointer argument");
  TFA_REQUIRE(head_dim == 128, TFA_ERR_SHAPE, "tfa_gemm_nt_qk_rope: head_dim %lld, only 128 supported",
              (long long)head_dim);
  TFA_REQUIRE(hq >= 1 && hkv >= 1 && hq <= 4096 && hkv <= 4096 && hq % hkv == 0, TFA_ERR_SHAPE,
              "tfa_gemm_nt_qk_rope: hq %lld not a multiple of hkv %lld, or out of range", (long long)hq, (long long)hkv);
  TFA_REQUIRE(batch >= 1 && n >= 1 && n <= (1 << 24) && batch <= (1 << 24) && pos0 >= 0 && pos0 <= (1 << 24) && cap >= 1,
              TFA_ERR_SHAPE, "tfa_gemm_nt_qk_rope: batch, rows (at most 2^24), cache or pos0 out of range");
  TFA_REQUIRE(pos0 + n <= cap, TFA_ERR_CAPACITY, "tfa_gemm_nt_qk_rope: positions %lld..%lld exceed the cache capacity %lld",
              (long long)pos0, (long long)(pos0 + n - 1), (long long)cap);
  TFA_REQUIRE(pos0 + n <= rope_rows, TFA_ERR_CAPACITY, "tfa_gemm_nt_qk_rope: positions up to %lld exceed the %lld rope rows",
              (long long)(pos0 + n - 1), (long long)rope_rows);
  const int64_t width = (hq + 2 * hkv) * 128;
  const int st = check_gemm(a, w_qkv, q_out, batch * n, width, k, lda, ldw, width, "tfa_gemm_nt_qk_rope");
  if (st != TFA_OK) return st;
  for (const void* p : {gamma_q, gamma_k, cos_t, sin_t, static_cast<const void*>(k_cache), static_cast<const void*>(v_cache)})
    TFA_REQUIRE((reinterpret_cast<uintptr_t>(p) & 7u) == 0, TFA_ERR_ALIGN,
                "tfa_gemm_nt_qk_rope: gammas, tables or caches not 8-byte aligned");
  GemmArgs g = make(a, w_qkv, batch * n, width, k, lda, ldw, hq * 128);
  g.c = static_cast<uint16_t*>(q_out);
  g.gq = static_cast<const uint16_t*>(gamma_q);
  g.gk = static_cast<const uint16_t*>(gamma_k);
  g.cos_t = static_cast<const uint16_t*>(cos_t);
  g.sin_t = static_cast<const uint16_t*>(sin_t);
  g.heads = (int)hq;
  g.kv_heads = (int)hkv;
  g.eps = eps_head;
  g.kc = static_cast<uint16_t*>(k_cache);
  g.vc = static_cast<uint16_t*>(v_cache);
  g.cap = cap;
  g.seq = (int)n;
  g.pos0 = (int)pos0;
  return launch<EPI_QKROPE>(g, stream, "gemm_nt_qk_rope");
}

int tfa_qkv_norm_rope(const void* hn, const void* w_qkv, void* out, int64_t n, int64_t hidden, int64_t heads,
                      int64_t kv_heads, int64_t head_dim, const void* gamma_q, const void* gamma_k, float eps,
                      const void* cos_t, const void* sin_t, int64_t rot, hipStream_t stream) {
  TFA_REQUIRE(head_dim == 256, TFA_ERR_SHAPE, "tfa_qkv_norm_rope: head_dim %lld, only 256 supported", (long long)head_dim);
  TFA_REQUIRE(rot == 64, TFA_ERR_SHAPE, "tfa_qkv_norm_rope: rot %lld, only 64 supported", (long long)rot);
  TFA_REQUIRE(heads >= 1 && kv_heads >= 1 && heads <= 4096 && kv_heads <= 4096, TFA_ERR_SHAPE,
              "tfa_qkv_norm_rope: head counts out of range");
  TFA_NONNULL(gamma_q);
  TFA_NONNULL(gamma_k);
  TFA_NONNULL(cos_t);
  TFA_NONNULL(sin_t);
  const int64_t width = (2 * heads + 2 * kv_heads) * head_dim;
  const int st = check_gemm(hn, w_qkv, out, n, width, hidden, hidden, hidden, width, "tfa_qkv_norm_rope");
  if (st != TFA_OK) return st;
  GemmArgs g = make(hn, w_qkv, n, width, hidden, hidden, hidden, width);
  g.c = static_cast<uint16_t*>(out);
  g.gq = static_cast<const uint16_t*>(gamma_q);
  g.gk = static_cast<const uint16_t*>(gamma_k);
  g.cos_t = static_cast<const uint16_t*>(cos_t);
  g.sin_t = static_cast<const uint16_t*>(sin_t);
  g.heads = (int)heads;
  g.kv_heads = (int)kv_heads;
  g.eps = eps;
  return launch<EPI_QKNR>(g, stream, "qkv_norm_rope");
}

}  // extern "C"
