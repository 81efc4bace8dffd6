// bf16 GEMM for the prefill projections on the gfx950 matrix cores:
//   Y[M, N] = X[M, K] W[N, K]^T            (fp32 accumulation, one bf16 rounding)
//   Y[M, N] = bf16(R[M, N] + bf16(X W^T))  with a residual R (same layout as Y;
//                                           R may be Y itself)
// Both operands are K-contiguous rows, the layout of activations [tokens,
// features] and of weights [out, in].
//
// Block tiles from 256 x 256 to 64 x 128 (pick_tile), K-steps of 64 or 128; 8
// waves (2 per SIMD) in two row groups of four, each wave RA x RB
// v_mfma_f32_32x32x16_bf16 accumulators (256 x 256: 4 x 2, 128 fp32 per lane).
// Operand layout of the 32x32x16 MFMA: lane 32h + i holds A[i][8h .. 8h+7] and
// B[8h .. 8h+7][i]; reg r of lane 32h + j holds C[8(r/4) + 4h + r%4][j].  With
// A = X rows and B[k][n] = W[n][k], both operands are 16-byte pieces of K-rows.
//
// Ping-pong schedule: the two waves of a SIMD belong to the two row groups
// (g = 0: waves 0-3, g = 1: waves 4-7) and run the same code, group 1 one
// block barrier behind, so in every interval between barriers one group
// reads a whole K-step's fragments from LDS (256 x 256: 24 ds_read_b128 into 96
// VGPRs) while the other issues that K-step's MFMAs from registers; the matrix
// pipe of each SIMD is fed by one wave at a time with nothing to wait for.
// (With both waves reading and multiplying in step, a double-buffered
// version ran at 0.7 of this.)
//
// The X and W tiles of a K-step land in LDS by DMA (buffer_load_dwordx4 ... lds:
// no staging registers; per-lane offsets computed once, the K offset and the
// row stride in a scalar register), in SX stages of X, filled by group 0, and SW
// stages of W, filled by group 1.  A stage is refilled one barrier after both
// groups have read it, and each group waits for its own DMA before the barrier
// that precedes the first read of that step.  A 256 x 256 step's 64 KiB take the
// CU's address unit ~1000 cycles, so the loads are issued between the fragment
// reads, one per three (all behind the reads, with W in two stages refilled
// while they could still be read: gate/up at 4096 tokens 683 -> 650 us, QKV
// 201 -> 192, o_proj 136 -> 126, down 331 -> 316; same run).
//
// What bounds it: LDS traffic (fragment reads + DMA writes) beside the MFMAs at the
// clock that this load leaves.  Counters at 4096 tokens, Qwen3-8B's gate/up, down,
// QKV, o_proj: 106, 104, 112 and 87 bytes per clock and CU of the LDS's 128, matrix
// cores busy 80, 79, 73 and 63% of the cycles, at 1.6-1.8 GHz.  256 x 256 needs 256
// KiB per step, as many cycles as its MFMAs.  Small tiles need more per flop but fill
// the chip at short prompts (740 tokens: 70-82 bytes per clock, a part-filled round);
// their K-steps of 128 halve the barriers and the scalar work per K (128 x 128 at K =
// 4096: 38 -> 29 us).
//
// Rows are stored with their 16-byte chunks XOR-swizzled (by (row >> 1) & 7, or
// row & 15 for 256-byte rows): gfx950's LDS is 64 banks (256 bytes) wide, and a
// 16-lane phase of a fragment read (16 consecutive rows) then covers all 16
// bank groups.  The DMA reads the global chunk that belongs at each fixed LDS
// slot; rows past M / N lie past the end of the tile's buffer resource and read
// zeros (never stored).  Fragment reads are asm: the compiler would otherwise
// wait for outstanding DMA (vmcnt 0) in front of every LDS read.
//
// Tiles are dealt to the XCDs in contiguous ranges (block b runs on XCD b % 8)
// and, within a range, in groups of 8 M-tiles (M fastest inside a group), so
// the blocks of one XCD share X and W panels in its L2.
#include "common.h"
#include "internal.h"
#include "prof.h"
#include "status.h"

namespace ez {

EZ_PROF_DEFINE(gemm)
namespace {

constexpr int kGWaves = 8;
constexpr int kGThreads = kGWaves * kWave;
constexpr int kGroupM = 8;  // M-tiles per tile group
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4v_t __attribute__((ext_vector_type(4)));

struct GemmArgs {
  const uint16_t* X; int64_t ldx;
  const uint16_t* W;
  uint16_t* Y; int64_t ldy;
  const uint16_t* R;
  int64_t M, N, K;
  int tm, tn;  // tiles along M and N
  int64_t IS;  // SwiGLU mode: rows [0, IS) of W are gate, [IS, 2 IS) up; Y is [M, IS]
};

// Fragment reads with immediate row-block offsets, up to three to an asm block
// so that a DMA can be issued between the blocks; frag_wait waits for a K-step's
// reads and, taking them as operands, keeps every use after the wait.
template <int O>
__device__ __forceinline__ void frag_issue(uint32_t a, u32x4v_t& r) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(r) : "v"(a), "i"(O));
}
template <int N>
__device__ __forceinline__ void frag_wait(u32x4v_t (&f)[N]) {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int k = 0; k < N; k += 4)
    asm volatile("" : "+v"(f[k]), "+v"(f[k + 1]), "+v"(f[k + 2]), "+v"(f[k + 3]));
  __builtin_amdgcn_sched_barrier(0);
}

// A wave multiplies RA x RB blocks of 32 x 32; the four waves of a row group
// sit GM x GN, the two groups above each other: tiles of 2 GM RA 32 rows and
// GN RB 32 columns.  Every shape accumulates an element over K in the same
// order, so all tile shapes give bit-identical results.
//
// SWIGLU: the tile's W rows are BN / 2 gate rows and the BN / 2 matching up rows,
// dealt so that a wave holds gate and up of the same features in the same lane
// and register; the epilogue writes silu(gate) * up: the prefill's SwiGLU
// without the [M, 2 IS] intermediate.  Rounding as the separate pass: gate and
// up rounded to bf16, the activation rounded, the product rounded.
template <bool SWIGLU, int RA, int RB, int GM, int GN, int BK, int SX, int SW, int WPE>
__global__ __launch_bounds__(kGThreads, WPE) void gemm_bf16_kernel(GemmArgs a) {
  static_assert(GM * GN == 4 && (!SWIGLU || RB == 2), "four waves per row group");
  constexpr int BM = 2 * GM * RA * 32, BN = GN * RB * 32;  // block tile
  constexpr int WC = SWIGLU ? 32 : 32 * RB;                // output columns per wave
  constexpr int CPR = BK / 8, RPL = 4 * kWave / CPR;       // 16-byte chunks per tile row; rows per DMA load of a group
  constexpr int NX = BM / RPL, NW = BN / RPL;              // DMA loads per thread of group 0 / 1 and K-step
  constexpr int kRowBytes = BK * 2, kSub = BK / 16;        // MFMA substeps per K-step
  constexpr int kXBytes = BM * kRowBytes, kWBytes = BN * kRowBytes;
  EZ_PROF_WAVE(kProfGemm);
  // SX stages of X tiles and SW of W tiles (256 x 256: two and three, 160 KiB); after
  // the K loop the same memory holds the block's C tile in bf16, wave by wave, for
  // row-contiguous stores.
  __shared__ __align__(16) uint16_t lds[(SX * BM + SW * BN) * BK];

  // tile of this block: XCD-contiguous ranges, groups of kGroupM M-tiles
  const int ntiles = a.tm * a.tn;
  int t = int(blockIdx.x);
  if (ntiles % 8 == 0) t = (t % 8) * (ntiles / 8) + t / 8;
  const int grp = t / (kGroupM * a.tn), gi = t % (kGroupM * a.tn);
  const int gm = a.tm - grp * kGroupM < kGroupM ? a.tm - grp * kGroupM : kGroupM;
  const int64_t m0 = int64_t(grp * kGroupM + gi % gm) * BM, n0 = int64_t(gi / gm) * (SWIGLU ? BN / 2 : BN);

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar LDS destinations
  const int g = wave >> 2, wg = wave & 3;         // row group, wave within the group
  const int wm = wg / GN, wn = wg % GN;           // the wave's place in the group
  const int wrow = g * (BM / 2) + wm * (RA * 32);  // first tile row of the wave
  const int h = lane >> 5, i = lane & 31;

  // DMA: load c of group wave wg fills LDS chunk p = (c * 4 + wg) * 64 + lane,
  // tile row p / CPR, slot p % CPR, which holds the row's logical chunk
  // slot ^ swz(row).  The per-lane offset does not depend on c (RPL c rows go in
  // the scalar offset).  SwiGLU: loads c >= NW / 2 come from the up rows.
  auto swz = [](int row) { return CPR == 8 ? (row >> 1) & 7 : row & 15; };
  const int dr = (wg * kWave + lane) / CPR, lc = (lane % CPR) ^ swz(dr);
  const int64_t mrows = a.M - m0 < BM ? a.M - m0 : BM, nrows = a.N - n0 < BN ? a.N - n0 : BN;
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.X + m0 * a.ldx), 0, int(((mrows - 1) * a.ldx + a.K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.W + n0 * a.K), 0, int((SWIGLU ? BN / 2 : nrows) * a.K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t ures = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.W + (SWIGLU ? a.IS + n0 : 0) * a.K), 0, int(BN / 2 * a.K * 2), 0x00020000);
  // The last steps' loads, of steps that do not exist, go to an empty buffer (no
  // traffic), so that the counts the waits rely on hold to the end.
  const __amdgpu_buffer_rsrc_t none = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.X), 0, 0, 0x00020000);
  const uint32_t voff = g ? uint32_t((dr * a.K + lc * 8) * 2) : uint32_t((dr * a.ldx + lc * 8) * 2);
  const uint32_t rstep = uint32_t((g ? a.K : a.ldx) * 2 * RPL);  // bytes of RPL rows
  const __amdgpu_buffer_rsrc_t res0 = g ? wres : xres, res1 = SWIGLU && g ? ures : res0;
  auto dma1 = [&](int c, const __amdgpu_buffer_rsrc_t& r0, const __amdgpu_buffer_rsrc_t& r1, uint32_t k0b, uint16_t* dst) {
    if (NX != NW && c >= (g ? NW : NX)) return;  // uniform
    const bool up = SWIGLU && c >= NW / 2;
    const uint32_t row = uint32_t(up && g ? c - NW / 2 : c) * rstep;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(up ? r1 : r0, (__attribute__((address_space(3))) void*)(dst + (c * 4 + wg) * kWave * 8),
                                             16, voff, k0b + row, 0, 0);
  };
  auto x_stage = [&](int st) { return &lds[st * BM * BK]; };
  auto w_stage = [&](int st) { return &lds[(SX * BM + st * BN) * BK]; };

  // Fragment addresses: substep s reads logical chunk 2s + h of A row wrow +
  // 32 ra + i and of B row 32 (RB wn + rb) + i (SwiGLU: rb BN / 2 + 32 wn + i);
  // the row blocks ra / rb are immediate offsets (32 rows keep the swizzle).
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint16_t*)(&lds[0])));
  uint32_t aaddr[kSub], baddr[kSub];
#pragma unroll
  for (int s = 0; s < kSub; ++s) {
    const uint32_t sw = uint32_t((2 * s + h) ^ swz(i)) << 4;
    aaddr[s] = lds0 + uint32_t(wrow + i) * kRowBytes + sw;
    baddr[s] = lds0 + uint32_t(SX * kXBytes) + uint32_t((SWIGLU ? 32 : 32 * RB) * wn + i) * kRowBytes + sw;
  }
  constexpr int kRA = 32 * kRowBytes, kRB = (SWIGLU ? BN / 2 : 32) * kRowBytes;

  f32x16_t acc[RA][RB];
#pragma unroll
  for (int ra = 0; ra < RA; ++ra)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[ra][rb][r] = 0.f;

  constexpr int FS = RA + RB;  // fragments per substep
  u32x4v_t fr[kSub * FS];     // one K-step: fr[FS s + ra] A pieces, fr[FS s + RA + rb] B pieces
  // One K-step's fragments from X stage `xs` and W stage `ws`, with the group's
  // DMA of a later step between the reads: the reads fill the LDS pipe and the
  // DMA the address unit, so neither waits for the other to be issued.
  constexpr int ND = NX > NW ? NX : NW, DPS = (ND + kSub - 1) / kSub;  // DMA loads, per substep
  auto read_step = [&](int xs, int ws, const __amdgpu_buffer_rsrc_t& r0, const __amdgpu_buffer_rsrc_t& r1, uint32_t k0b,
                       uint16_t* dst) {
    const uint32_t ao = uint32_t(xs * kXBytes), bo = uint32_t(ws * kWBytes);
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
      u32x4v_t* f = &fr[FS * s];
      const uint32_t aa = aaddr[s] + ao, ba = baddr[s] + bo;
      frag_issue<0>(aa, f[0]);
      if constexpr (RA > 1) frag_issue<kRA>(aa, f[1]);
      frag_issue<0>(ba, f[RA]);
      if (DPS * s < ND) dma1(DPS * s, r0, r1, k0b, dst);
      if constexpr (RA > 2) frag_issue<2 * kRA>(aa, f[2]);
      if constexpr (RA > 3) frag_issue<3 * kRA>(aa, f[3]);
      if constexpr (RB > 1) frag_issue<kRB>(ba, f[RA + 1]);
      if constexpr (RB > 2) frag_issue<2 * kRB>(ba, f[RA + 2]);
      if (DPS > 1 && DPS * s + 1 < ND) dma1(DPS * s + 1, r0, r1, k0b, dst);
    }
    frag_wait(fr);
  };
  // The last K-step of K % 64 != 0: the 16-byte pieces at or past K hold
  // the next row's elements (or zeros past the buffer); both operands'
  // pieces there are zeroed, so they add nothing.
  auto mask_tail = [&](int64_t k0) {
#pragma unroll
    for (int s = 0; s < kSub; ++s)
      if (k0 + (2 * s + h) * 8 >= a.K)
#pragma unroll
        for (int f = 0; f < FS; ++f) fr[FS * s + f] = u32x4v_t{0u, 0u, 0u, 0u};
  };
  auto mult_step = [&]() {
#pragma unroll
    for (int s = 0; s < kSub; ++s)
#pragma unroll
      for (int ra = 0; ra < RA; ++ra)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          acc[ra][rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fr[FS * s + ra]),
                                                                __builtin_bit_cast(bf16x8_t, fr[FS * s + RA + rb]),
                                                                acc[ra][rb], 0, 0, 0);
  };
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  const int64_t nk = (a.K + BK - 1) / BK;
  const bool ktail = a.K % BK != 0;
  // At step j group 0 loads X of step j + SX - 1 and group 1 W of step
  // j + SW - 1 while they read step j: the stage filled held step j - 1, which
  // both groups had read before the barrier that starts the interval.  The
  // steps before that are in flight before the loop.
  const int ahead = g ? SW - 1 : SX - 1;
  for (int p = 0; p < ahead; ++p) {
    const bool on = p < nk;
#pragma unroll
    for (int c = 0; c < ND; ++c) dma1(c, on ? res0 : none, on ? res1 : none, uint32_t(p * BK * 2), g ? w_stage(p) : x_stage(p));
  }
  if (g) wait_vm<(SW - 2) * NW>(); else wait_vm<(SX - 2) * NX>();  // step 0
  __syncthreads();
  if (g == 1) barrier();  // group 1 runs one interval behind
  int xs = 0, ws = 0;     // stages of step j
  auto step = [&](int64_t j, const __amdgpu_buffer_rsrc_t& r0, const __amdgpu_buffer_rsrc_t& r1, bool last) {
    const int xd = xs == 0 ? SX - 1 : xs - 1, wd = ws == 0 ? SW - 1 : ws - 1;  // the stages of step j - 1
    read_step(xs, ws, r0, r1, uint32_t((j + ahead) * BK * 2), g ? w_stage(wd) : x_stage(xd));
    if (last && ktail) mask_tail(j * BK);
    if (g == 1) {
      __builtin_amdgcn_sched_barrier(0);
      wait_vm<(SW - 2) * NW>();  // W of step j + 1 (the older loads)
    }
    barrier();
    mult_step();
    if (g == 0) {
      __builtin_amdgcn_sched_barrier(0);
      wait_vm<(SX - 2) * NX>();  // X of step j + 1
    }
    barrier();
    xs = xs == SX - 1 ? 0 : xs + 1;
    ws = ws == SW - 1 ? 0 : ws + 1;
  };
  int64_t j = 0;
  for (; j < nk - ahead; ++j) step(j, res0, res1, false);
  for (; j < nk; ++j) step(j, none, none, j + 1 == nk);
  if (g == 0) barrier();  // the same barrier count for both groups
  wait_vm<0>();           // the last (empty) loads

  // Epilogue.  Reg r of lane (h, i) in acc[ra][rb] is C[32 ra + 8(r/4) + 4h +
  // r%4][32 rb + i] of the wave's tile: rounded to bf16 into the wave's part of
  // the LDS (row-major, WC columns), then read back 16 bytes a lane for 16-byte
  // stores and residual loads.
  __syncthreads();  // every wave is done with the operand tiles
  uint16_t* ct = &lds[wave * RA * 32 * WC];
#pragma unroll
  for (int ra = 0; ra < RA; ++ra)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      uint16_t* c = &ct[(32 * ra + 8 * (r >> 2) + 4 * h + (r & 3)) * WC + i];
      if constexpr (SWIGLU) {
        c[0] = f2bf(round_bf(silu(round_bf(acc[ra][0][r]))) * round_bf(acc[ra][1][r]));
      } else {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) c[32 * rb] = f2bf(acc[ra][rb][r]);
      }
    }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's writes are in LDS before its reads
  const bool vec = a.ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(a.Y) & 15) == 0 &&
                   (!a.R || (reinterpret_cast<uintptr_t>(a.R) & 15) == 0);
  const int64_t nout = SWIGLU ? a.IS : a.N;
  constexpr int LPR = WC / 8;  // lanes per row
#pragma unroll 4
  for (int q = 0; q < RA * 32 * LPR / kWave; ++q) {
    const int idx = q * kWave + lane, rr = idx / LPR, lcb = (idx % LPR) * 8;
    const int64_t row = m0 + wrow + rr, col = n0 + WC * wn + lcb;
    if (row >= a.M || col >= nout) continue;
    const uint4 cv = *reinterpret_cast<const uint4*>(&ct[rr * WC + lcb]);
    uint16_t* y = a.Y + row * a.ldy + col;
    if (vec && col + 8 <= nout) {
      uint4 out = cv;
      if (a.R) {
        const uint4 rv = *reinterpret_cast<const uint4*>(a.R + row * a.ldy + col);
        const uint32_t* c32 = reinterpret_cast<const uint32_t*>(&cv);
        const uint32_t* r32 = reinterpret_cast<const uint32_t*>(&rv);
        uint32_t* o32 = reinterpret_cast<uint32_t*>(&out);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = __uint_as_float(r32[e] << 16) + __uint_as_float(c32[e] << 16);
          const float hi = __uint_as_float(r32[e] & 0xffff0000u) + __uint_as_float(c32[e] & 0xffff0000u);
          o32[e] = uint32_t(f2bf(lo)) | (uint32_t(f2bf(hi)) << 16);
        }
      }
      *reinterpret_cast<uint4*>(y) = out;
    } else {
      const uint16_t* c16 = reinterpret_cast<const uint16_t*>(&cv);
      for (int e = 0; e < 8 && col + e < nout; ++e)
        y[e] = a.R ? f2bf(bf2f(a.R[row * a.ldy + col + e]) + bf2f(c16[e])) : c16[e];
    }
  }
}

template <bool SWIGLU, int RA, int RB, int GM, int GN, int BK, int SX, int SW, int WPE>
void launch_tile(GemmArgs a, hipStream_t s) {
  constexpr int BM = 2 * GM * RA * 32, BN = GN * RB * 32;
  a.tm = int((a.M + BM - 1) / BM);
  a.tn = int((a.N + BN - 1) / BN);
  hipLaunchKernelGGL((gemm_bf16_kernel<SWIGLU, RA, RB, GM, GN, BK, SX, SW, WPE>), dim3(unsigned(a.tm * a.tn)), dim3(kGThreads), 0, s, a);
}

// Tile shapes.  One round (a block on every slot of the chip) of a K = 4096
// GEMM took, in us, with few blocks / with every slot taken (MI355X; the chip
// clocks lower under full load, and the time is proportional to K: K = 12288
// within 10%):
struct TileCost {
  int bm, bn, per_cu;  // tile, blocks per CU
  float lo, hi;
};
constexpr TileCost kTiles[] = {
    {256, 256, 1, 75.f, 112.f},  // 0
    {256, 192, 1, 57.f, 90.f},   // 1 (not SwiGLU)
    {256, 128, 1, 46.f, 68.f},   // 2
    {128, 128, 2, 38.f, 75.f},   // 3: two blocks per CU, K-steps of 64
    {128, 128, 1, 29.f, 44.f},   // 4: K-steps of 128
    {64, 128, 1, 23.f, 29.f},    // 5: K-steps of 128 (not SwiGLU)
    {192, 256, 1, 57.f, 90.f},   // 6
};

// The shape with the least estimated time: full rounds at `hi`, a part-filled
// last round between `lo` and `hi`.  Against 256-wide tiles for every GEMM of at
// least half a round and 256 x 128 below (the rule before), measured in us at
// Qwen3-8B's (QKV, o_proj, gate/up, down): 700 tokens 61 / 64 / 198 / 187 ->
// 50 / 35 / 152 / 100; 256 tokens 67 / 70 / 90 / 190 -> 25 / 24 / 80 / 80;
// 2048 tokens QKV 90 -> 84, o_proj 86 -> 68, down 247 -> 186; 3000 tokens QKV
// 167 -> 142, o_proj 95 -> 87, down 264 -> 246.
int pick_tile(int64_t M, int64_t N, bool swiglu, int64_t cus) {
  int best = 0;
  float least = 0.f;
  for (int t = 0; t < int(sizeof(kTiles) / sizeof(kTiles[0])); ++t) {
    if (swiglu && (t == 1 || t == 5)) continue;
    const TileCost& c = kTiles[t];
    const int64_t blocks = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn), slots = cus * c.per_cu;
    const float part = float(blocks % slots) / float(slots);
    const float cost = float(blocks / slots) * c.hi + (part > 0.f ? c.lo + (c.hi - c.lo) * part * part : 0.f);
    if (t == 0 || cost < least) {
      best = t;
      least = cost;
    }
  }
  return best;
}

template <bool SWIGLU>
void launch_gemm(const GemmArgs& a, hipStream_t s) {
  switch (pick_tile(a.M, a.N, SWIGLU, num_cus())) {
    case 0: return launch_tile<SWIGLU, 4, 2, 1, 4, 64, 2, 3, 2>(a, s);
    case 1: if constexpr (!SWIGLU) return launch_tile<SWIGLU, 2, 3, 2, 2, 64, 2, 4, 2>(a, s);
    case 2: return launch_tile<SWIGLU, 2, 2, 2, 2, 64, 3, 3, 2>(a, s);
    case 3: return launch_tile<SWIGLU, 1, 2, 2, 2, 64, 2, 3, 4>(a, s);
    case 4: return launch_tile<SWIGLU, 1, 2, 2, 2, 128, 2, 3, 2>(a, s);
    case 6: return launch_tile<SWIGLU, 3, 2, 1, 4, 64, 2, 3, 2>(a, s);
    default: if constexpr (!SWIGLU) return launch_tile<SWIGLU, 1, 1, 1, 4, 128, 3, 3, 2>(a, s);
  }
}

}  // namespace

bool gemm_mfma_supported(const uint16_t* X, int64_t ldx, const uint16_t* W, const uint16_t* Y, int64_t ldy,
                         const uint16_t* R, int64_t M, int64_t N, int64_t K) {
  (void)R;  // R shares Y's leading dimension
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  // 16-byte pieces of K-rows (K % 8 == 0; the last K-step may be partial);
  // the DMA addresses operands by 32-bit byte offsets from their base
  return X && W && Y && M >= 1 && N >= 1 && K >= 8 && K % 8 == 0 && ldx >= K && ldx % 8 == 0 && ldy >= N &&
         al16(X) && al16(W) && (M - 1) * ldx * 2 + K * 2 + 256 < (int64_t(1) << 31) &&
         (N - 1) * K * 2 + K * 2 + 256 < (int64_t(1) << 31);
}

int gemm_mfma(const uint16_t* X, int64_t ldx, const uint16_t* W, uint16_t* Y, int64_t ldy, const uint16_t* R,
              int64_t M, int64_t N, int64_t K, hipStream_t s) {
  EZ_REQUIRE(gemm_mfma_supported(X, ldx, W, Y, ldy, R, M, N, K), "gemm: shape or alignment not supported by the MFMA kernel");
  launch_gemm<false>(GemmArgs{X, ldx, W, Y, ldy, R, M, N, K, 0, 0, 0}, s);
  return launch_status("gemm (MFMA)");
}

bool gemm_swiglu_supported(const uint16_t* X, int64_t ldx, const uint16_t* W, const uint16_t* Y, int64_t ldy,
                           int64_t M, int64_t IS, int64_t K) {
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  return IS >= 1 && IS % 128 == 0 && ldy % 8 == 0 && al16(Y) && ldy >= IS &&
         gemm_mfma_supported(X, ldx, W, Y, 2 * IS, nullptr, M, 2 * IS, K);
}

int gemm_swiglu(const uint16_t* X, int64_t ldx, const uint16_t* W, uint16_t* Y, int64_t ldy, int64_t M, int64_t IS,
                int64_t K, hipStream_t s) {
  EZ_REQUIRE(gemm_swiglu_supported(X, ldx, W, Y, ldy, M, IS, K),
             "gemm_swiglu: shape or alignment not supported (IS %% 128, K %% 8, ldx >= K, 16-byte rows)");
  launch_gemm<true>(GemmArgs{X, ldx, W, Y, ldy, nullptr, M, 2 * IS, K, 0, 0, IS}, s);
  return launch_status("gemm_swiglu (MFMA)");
}

// Prefill GEMM entry: the MFMA kernel for 16-byte K-rows (K % 8 == 0,
// aligned operands); any other shape runs the linear-layer kernels of
// gemv.hip (the residual epilogue rounds as here: bf16(R + bf16(X W^T))).
int gemm_bf16(const uint16_t* X, int64_t ldx, const uint16_t* W, uint16_t* Y, int64_t ldy, const uint16_t* R,
              int64_t M, int64_t N, int64_t K, hipStream_t s) {
  EZ_REQUIRE(X && W && Y, "gemm: null pointer");
  EZ_REQUIRE(M >= 1 && N >= 1 && K >= 1 && ldx >= K && ldy >= N, "gemm: bad shape");
  if (gemm_mfma_supported(X, ldx, W, Y, ldy, R, M, N, K)) return gemm_mfma(X, ldx, W, Y, ldy, R, M, N, K, s);
  LinearArgs l{};
  l.X = X; l.ldx = ldx; l.W = W; l.Y = Y; l.ldy = ldy; l.M = M; l.N = N; l.K = K;
  l.res = R; l.ldr = ldy; l.epi = R ? kEpiResid : kEpiStore;
  return launch_linear(l, s);
}

}  // namespace ez

extern "C" size_t ezops_gemm_workspace_size(void) { return 0; }

extern "C" int ezops_gemm_tile(int64_t M, int64_t N, int swiglu, int64_t cus) {
  EZ_REQUIRE(M >= 1 && N >= 1 && cus >= 1, "gemm_tile: sizes must be >= 1");
  return ez::pick_tile(M, N, swiglu != 0, cus);
}

extern "C" int ezops_gemm_swiglu_bf16(const void* X, int64_t ldx, const void* Wgu, void* Y, int64_t ldy, int64_t M,
                                      int64_t IS, int64_t K, hipStream_t stream) {
  return ez::gemm_swiglu(static_cast<const uint16_t*>(X), ldx, static_cast<const uint16_t*>(Wgu),
                         static_cast<uint16_t*>(Y), ldy, M, IS, K, stream);
}

extern "C" int ezops_gemm_bf16(const void* X, int64_t ldx, const void* W, void* Y, int64_t ldy, const void* R,
                               int64_t M, int64_t N, int64_t K, void* ws, size_t ws_bytes, hipStream_t stream) {
  (void)ws;  // no workspace: kept for the ABI
  (void)ws_bytes;
  return ez::gemm_bf16(static_cast<const uint16_t*>(X), ldx, static_cast<const uint16_t*>(W),
                       static_cast<uint16_t*>(Y), ldy, static_cast<const uint16_t*>(R), M, N, K, stream);
}
