// Skinny linear layers for 5 to 64 batch rows (and more, 64 at a time):
// Y[M, N] = epi(X[M, K] . W[N, K]^T), every weight byte read once per 64 rows.
//
// The 16-row kernels of gemv.hip read W once per 16 batch rows (grid.y), so at
// 64 rows the projections took four times their weight traffic.  Here a block
// owns 16 weight rows (T = 2: 16 + 16, the gate and up rows of SwiGLU or two
// neighbouring tiles) against MT 16-row batch blocks: each weight fragment is
// read from LDS once and meets MT activation fragments.  (Matrices with too few
// 16-row tiles to fill the chip this way stay with the 16-row kernels: narrow() in
// gemv.hip.)
//
//   * 4 waves split K into 256-wide chunks; a chunk of a 16-row tile (8 KiB)
//     lands in LDS by DMA (buffer_load_dwordx4 ... lds) in 512-byte row pieces
//     at XOR-swizzled 16-byte slots (piece c of row r at slot c ^ r), through a
//     two-stage ring per wave, as in linear_mfma_kernel: no block barriers in
//     the K loop.
//   * X fragments (L2-resident activations, 1 KiB contiguous per fragment in
//     the packed layout) go straight to registers, half a chunk (4 k-steps x MT
//     fragments) at a time in two buffers, one half ahead of its MFMAs.
//   * The block walks tiles blockIdx.x, + gridDim.x, ... with one ring: the
//     next tile's first chunks are in flight during a tile's epilogue.
//   * Epilogue: the waves' partial tiles are summed through LDS, four
//     neighbouring outputs per thread (8-byte stores and residual loads).
//
// Bound: HBM (weights) up to 32 rows; at 64 the X fragments, MT / T times the
// weight bytes through each CU's L1.  Measured (MI355X, Qwen3-8B, kernel
// traces, this kernel against 16 rows per read of W): 64 rows: gate/up 45
// against 131.7 us, QKV 17-18 / 38.1, o_proj + down 48 / 116.  32 rows: gate/up
// 37.1, QKV 14.1 us (16 rows: 35.7, 15.6).  The X traffic costs about 1 us per
// 18 MB over the chip; requesting X a whole chunk ahead (two chunks in
// registers) changed nothing.  Up to 16 rows: VL-2B QKV + o_proj + down 24.4 ->
// 21.8 us, 0.6B 18.4 -> 16.7, the 0.6B LM head 110 -> 56 against the 16-row kernel
// (Qwen3-8B o_proj + down 29.9 / 29.6).
#include "common.h"
#include "internal.h"
#include "prof.h"
#include "status.h"

namespace ez {

EZ_PROF_DEFINE(linear_mt)
namespace {

constexpr int NW = 4;                  // waves per block, splitting K
constexpr int kKC = 256;               // K elements per chunk
constexpr int kSteps = kKC / 32;       // MFMA k-steps per chunk
constexpr int kHalf = kSteps / 2;      // k-steps per X buffer
constexpr int kSlices = 16 * kKC / 512;  // 1 KiB DMA slices per 16-row tile and chunk
constexpr int kTileChunk = 16 * kKC * 2;  // bytes of one 16-row tile's chunk
typedef unsigned int u32x4v_t __attribute__((ext_vector_type(4)));

// Four A fragments (k-steps) of one chunk half from a DMA-landed tile, with
// their wait.  asm: the compiler makes any LDS read behind an LDS DMA wait for
// every outstanding load, which would drain the ring; the caller has waited
// for this stage's DMA.
__device__ __forceinline__ void lds_read_a4(const uint32_t (&addr)[kHalf], u32x4v_t (&r)[kHalf]) {
  asm volatile(
      "ds_read_b128 %0, %4\n\t"
      "ds_read_b128 %1, %5\n\t"
      "ds_read_b128 %2, %6\n\t"
      "ds_read_b128 %3, %7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
      : "v"(addr[0]), "v"(addr[1]), "v"(addr[2]), "v"(addr[3]));
}
static_assert(kHalf == 4, "lds_read_a4 reads 4 fragments");

// Four neighbouring outputs n .. n + 3 of batch row m (v2: the up sums of SwiGLU).
template <bool SILU>
__device__ __forceinline__ void store4(const LinearArgs& a, bool vec, int64_t m, int64_t n, const f32x4_t& v,
                                       const f32x4_t& v2) {
  if (a.epi == kEpiStoreF32) {
    float* y = reinterpret_cast<float*>(a.Y) + m * a.ldy + n;
    for (int j = 0; j < 4; ++j)
      if (n + j < a.N) y[j] = v[j];
    return;
  }
  uint16_t* y = reinterpret_cast<uint16_t*>(a.Y) + (a.y_packed ? packed_index(m, n, a.ldy) : m * a.ldy + n);
  if (vec && n + 4 <= a.N) {
    uint32_t w[2];
    if constexpr (SILU) {
      float p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = round_bf(silu(round_bf(v[j]))) * round_bf(v2[j]);
      w[0] = pack_bf2(p[0], p[1]);
      w[1] = pack_bf2(p[2], p[3]);
    } else if (a.epi == kEpiResid) {
      const uint2 r = *reinterpret_cast<const uint2*>(a.res + m * a.ldr + n);
      w[0] = pack_bf2(bf_lo(r.x) + round_bf(v[0]), bf_hi(r.x) + round_bf(v[1]));
      w[1] = pack_bf2(bf_lo(r.y) + round_bf(v[2]), bf_hi(r.y) + round_bf(v[3]));
    } else {
      w[0] = pack_bf2(v[0], v[1]);
      w[1] = pack_bf2(v[2], v[3]);
    }
    *reinterpret_cast<uint2*>(y) = make_uint2(w[0], w[1]);
    return;
  }
  for (int j = 0; j < 4; ++j) {  // the packed layout keeps n .. n + 3 adjacent (n % 4 == 0)
    if (n + j >= a.N) break;
    float o = v[j];
    if constexpr (SILU) o = round_bf(silu(round_bf(v[j]))) * round_bf(v2[j]);
    else if (a.epi == kEpiResid) o = bf2f(a.res[m * a.ldr + n + j]) + round_bf(v[j]);
    y[j] = f2bf(o);
  }
}

// XP: X in the packed layout (K % 32 == 0).  Wave operands as in
// linear_mfma_kernel: lane 16 g + i of the A operand holds W[row + i][8 g ..],
// of B X[m + i][8 g ..], C[4 g + j][i] in register j.
template <int T, bool SILU, int MT, bool XP>
__global__ __launch_bounds__(NW * kWave) void linear_mt_kernel(LinearArgs a, bool vec) {
  static_assert(T == 1 || T == 2, "one or two 16-row tiles");
  static_assert(!SILU || T == 2, "SwiGLU: gate and up tile");
  EZ_PROF_WAVE(kProfLinearMfma);
  constexpr int XH = MT * kHalf;   // X loads per half chunk
  constexpr int DN = T * kSlices;  // DMA slices per chunk
  constexpr int TM = T * MT;
  constexpr int kRows = SILU ? 16 : 16 * T;  // output features per tile
  __shared__ __align__(16) unsigned char ring[NW][2][T][kTileChunk];
  __shared__ __align__(16) f32x4_t red[NW][TM][kWave];

  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int64_t m0 = int64_t(blockIdx.y) * 16 * MT;

  const int dr = lane >> 5, cs = lane & 31;
  __amdgpu_buffer_rsrc_t wres0, wres1;  // (an array of resources drops the kernel's host stub)
  uint32_t woff[kSlices];
  // Rows past N lie past the end of the tile's buffer and read zeros.
  auto tile_res = [&](const uint16_t* W, int64_t r0) {
    const int64_t rows = a.N - r0 < 16 ? (a.N - r0 > 0 ? a.N - r0 : 0) : 16;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W + (rows ? r0 : 0) * a.K), 0, int(rows * a.K * 2),
                                             0x00020000);
  };
  auto set_rows = [&](int64_t r0) {
    wres0 = tile_res(a.W, r0);
    wres1 = SILU ? tile_res(a.W2, r0) : (T == 2 ? tile_res(a.W, r0 + 16) : wres0);
  };
#pragma unroll
  for (int q = 0; q < kSlices; ++q) {
    const int row = 2 * q + dr;
    woff[q] = uint32_t((row * a.K + int64_t(cs ^ row) * 8) * 2);
  }

  const int nchunks = int((a.K + kKC - 1) / kKC);
  const int cb = nchunks * wave / NW, ce = nchunks * (wave + 1) / NW;
  const int64_t ksteps = a.K >> 5;

  // DMA of chunk c: pieces past K read the next row's weights (or zeros past
  // the buffer); they meet zeroed X below.
  const uint32_t ring0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)&ring[wave][0][0][0]));
  auto dma = [&](int c, int stage) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int q = 0; q < kSlices; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            t ? wres1 : wres0, (__attribute__((address_space(3))) void*)(&ring[wave][stage][t][q * 1024]), 16, woff[q],
            uint32_t(c) * (kKC * 2), 0, 2);
  };
  // X fragments of half h of chunk c by buffer loads: batch rows past M lie past
  // the end of the block's buffer and read zeros.
  const int64_t brows = a.M - m0 < 16 * MT ? a.M - m0 : 16 * MT;
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(XP ? a.X + (m0 >> 4) * ksteps * 512 : a.X + m0 * a.ldx), 0,
      XP ? int(((brows + 15) >> 4) * ksteps * 1024) : int(((brows - 1) * a.ldx + a.K) * 2), 0x00020000);
  // A step that does not exist still issues its loads, against an empty buffer
  // (no memory traffic), so that the loop has no branch around pending loads and
  // the counts below always hold.
  const __amdgpu_buffer_rsrc_t none = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.X), 0, 0, 0x00020000);
  uint32_t xoff[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xoff[mt] = XP ? uint32_t(mt * ksteps * 1024 + lane * 16) : uint32_t(((16 * mt + i) * a.ldx + 8 * g) * 2);
  auto xload = [&](const __amdgpu_buffer_rsrc_t& res, int c, int h, u32x4v_t (&x)[MT][kHalf]) {
#pragma unroll
    for (int s = 0; s < kHalf; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        x[mt][s] = __builtin_amdgcn_raw_buffer_load_b128(res, xoff[mt],
                                                         uint32_t(c * kSteps + h * kHalf + s) * (XP ? 1024u : 64u), 0);
  };

  f32x4_t acc[T][MT];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const bool ktail = a.K % kKC != 0;
  auto compute = [&](int c, int h, int stage, u32x4v_t (&x)[MT][kHalf]) {
    // the X registers count as redefined here: no use of them moves up to
    // their loads
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      asm volatile("" : "+v"(x[mt][0]), "+v"(x[mt][1]), "+v"(x[mt][2]), "+v"(x[mt][3]));
    u32x4v_t af[T][kHalf];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      uint32_t addr[kHalf];
#pragma unroll
      for (int s = 0; s < kHalf; ++s)
        addr[s] = ring0 + uint32_t((stage * T + t) * kTileChunk + (i >> 1) * 1024 + (i & 1) * 512 +
                                   (((4 * (h * kHalf + s) + g) ^ i) << 4));
      lds_read_a4(addr, af[t]);
    }
    if (ktail) {  // pieces past K: both operands zero
#pragma unroll
      for (int s = 0; s < kHalf; ++s)
        if (int64_t(c) * kKC + 32 * (h * kHalf + s) + 8 * g >= a.K) {
#pragma unroll
          for (int t = 0; t < T; ++t) af[t][s] = u32x4v_t{0u, 0u, 0u, 0u};
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) x[mt][s] = u32x4v_t{0u, 0u, 0u, 0u};
        }
    }
#pragma unroll
    for (int s = 0; s < kHalf; ++s)
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, af[t][s]),
                                                               __builtin_bit_cast(bf16x8_t, x[mt][s]), acc[t][mt], 0, 0, 0);
  };

  // The ring runs over (tile, chunk) pairs; `dt` / `dc` are the pair the next
  // DMA belongs to, X depends on the chunk alone.  Per step the loads are
  // issued in the order X half 0, X half 1, DMA (two steps ahead), so each
  // wait below leaves exactly the newer ones outstanding.
  const int64_t tiles = (a.N + kRows - 1) / kRows;
  u32x4v_t xa[MT][kHalf], xb[MT][kHalf];
  int64_t dt = blockIdx.x;
  int dc = cb, stage = 0;
  auto dma_next = [&](int st) {
    dma(dc, st);
    if (++dc == ce) {
      dc = cb;
      dt += gridDim.x;
      if (dt < tiles) set_rows(dt * kRows);
      else wres0 = wres1 = none;
    }
  };
  set_rows(dt * kRows);
  if (cb < ce) {  // (short K: a wave may have no chunk)
    dma_next(0);
    xload(xres, cb, 0, xa);
    xload(xres, cb, 1, xb);
    dma_next(1);
  }
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const bool last_tile = tile + gridDim.x >= tiles;
    for (int c = cb; c < ce; ++c) {
      const int cn = c + 1 < ce ? c + 1 : cb;
      const bool next = !last_tile || c + 1 < ce;
      const __amdgpu_buffer_rsrc_t xn = next ? xres : none;
      wait_vm<XH + DN>();
      compute(c, 0, stage, xa);
      xload(xn, cn, 0, xa);
      wait_vm<XH + DN>();
      compute(c, 1, stage, xb);
      xload(xn, cn, 1, xb);
      dma_next(stage);
      stage ^= 1;
    }
    // Sum of the waves' partial tiles.  LDS through asm (see lds_read_a4); the
    // leading s_nops cover the MFMA results, whose hazards the compiler does
    // not track into asm.
    const uint32_t red0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) f32x4_t*)&red[0][0][0])) + lane * 16;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        asm volatile("s_nop 15\n\ts_nop 3\n\tds_write_b128 %0, %1" ::"v"(red0 + uint32_t((wave * TM + t * MT + mt) * 1024)),
                     "v"(acc[t][mt])
                     : "memory");
        acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int u = wave; u < (SILU ? MT : TM); u += NW) {
      f32x4_t v = {0.f, 0.f, 0.f, 0.f}, v2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        f32x4_t p;
        asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(p) : "v"(red0 + uint32_t((w * TM + u) * 1024)));
        v += p;
        if constexpr (SILU) {
          f32x4_t p2;
          asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(p2)
                       : "v"(red0 + uint32_t((w * TM + MT + u) * 1024)));
          v2 += p2;
        }
      }
      const int t = SILU ? 0 : u / MT, mt = SILU ? u : u % MT;
      const int64_t m = m0 + 16 * mt + i, n = tile * kRows + 16 * t + 4 * g;
      if (m < a.M && n < a.N) store4<SILU>(a, vec, m, n, v, v2);
    }
    if (!last_tile) asm volatile("s_barrier" ::: "memory");  // red is rewritten by the next tile
  }
  wait_vm<0>();  // no DMA into this block's LDS outlives it
}

template <int T, bool SILU, int MT>
void launch_x(const LinearArgs& a, unsigned gx, bool vec, hipStream_t s) {
  const dim3 grid(gx, unsigned((a.M + 16 * MT - 1) / (16 * MT))), block(NW * kWave);
  if (a.x_packed) hipLaunchKernelGGL((linear_mt_kernel<T, SILU, MT, true>), grid, block, 0, s, a, vec);
  else hipLaunchKernelGGL((linear_mt_kernel<T, SILU, MT, false>), grid, block, 0, s, a, vec);
}

template <int MT>
void launch_m(const LinearArgs& a, bool vec, hipStream_t s) {
  const int64_t cus = num_cus(), tiles = (a.N + 15) / 16;
  auto grid = [&](int64_t t, int64_t slots) { return unsigned(t < slots ? t : slots); };
  if (a.epi == kEpiSilu) return launch_x<2, true, MT>(a, grid(tiles, cus), vec, s);
  // Two-tile blocks (each X fragment meets 32 weight rows) where most CUs still
  // have one: Qwen3-8B QKV (192 blocks) at 64 rows 22.1 -> 17-18 us, at 32 16.1 ->
  // 14.1; o_proj and down on half the CUs lose (together 49 -> 59 us).
  if (4 * tiles > 5 * cus) return launch_x<2, false, MT>(a, grid((a.N + 31) / 32, cus), vec, s);
  // Else 16-row tiles, 4 waves each (8 waves splitting K: VL-2B QKV + o_proj +
  // down at 40 rows 35.4 against 29.5 us, 0.6B at 64 rows 26.7 against 24.0).
  launch_x<1, false, MT>(a, grid(tiles, 2 * cus), vec, s);
}

}  // namespace

// M > 4, operands checked by launch_linear (16-byte rows, 32-bit extents).
// 65 to 96 rows go in two equal groups, not 64 and the rest: 0.6B gate/up 16.5 -> 15.2 us at
// 65 rows (13.9 with 16 rows per read of W), VL-2B o_proj 12.0 -> 10.0 (11.3), o_proj + FFN 0.6B
// 33.4 -> 31.2 (31.8), VL-2B 58 -> 52.
void launch_linear_mt(const LinearArgs& a, hipStream_t s) {
  const bool vec = a.ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(a.Y) & 7) == 0 &&
                   (a.epi != kEpiResid || (a.ldr % 4 == 0 && (reinterpret_cast<uintptr_t>(a.res) & 7) == 0));
  if (a.M <= 16) launch_m<1>(a, vec, s);
  else if (a.M <= 32) launch_m<2>(a, vec, s);
  else if (a.M <= 48 || (a.M > 64 && a.M <= 96)) launch_m<3>(a, vec, s);
  else launch_m<4>(a, vec, s);
}

}  // namespace ez
