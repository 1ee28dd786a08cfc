// Token-row linear layers with fused epilogues for gfx950 (bf16), the GEMM
// side of the C = 1024 half-blocks:
//
//   acc[m][f] = b[f] + sum_k x[m][k] W[f][k]      fp32 accumulation on MFMA
//
// followed by one of
//
//   store     y[m]    = bf16(acc)                              (nn.Linear)
//   gelu      y[m]    = GELU(bf16(acc))                        (fc1 + nn.GELU)
//   residual  y[m]    = bf16(r[m] + bf16(acc))                 (fc2 + shortcut)
//   scatter   y[t(m)] = bf16(r[t(m)] + bf16(acc))              (proj + window
//             reverse + inverse roll + shortcut: row m of window-order x goes
//             back to the grid token t(m) it was gathered from; frame-padding
//             rows are dropped)
//   gelu-keep h[m]    = bf16(acc), y[m] = GELU(h[m])           (fc1 + nn.GELU
//             of the training step, whose backward needs both)
//   gelu-bwd  y[m]    = bf16(acc * slope(h[m])), colsum += sum_m y[m]   (the
//             gradient of fc1's output: fc2's input-gradient product times the
//             GELU's derivative, and fc1's bias gradient)
//
// so that the activation, the residual add and the permutation back to the
// grid ride on the GEMM's output instead of making their own HBM passes.
//
// Shape: Y^T = W X^T on v_mfma_f32_16x16x32_bf16 (A = weight rows from the
// fragment-packed layout of terra_swin_pack_linear, B = token rows).  A
// workgroup (8 waves, one per CU) computes a 256-feature x 256-token tile;
// wave w owns features 128 (w >> 2) .. + 128 of tokens 64 (w & 3) .. + 64: 8 x
// 4 accumulator tiles.  Per 64-wide stage (two k-steps) the tile's weights (32
// packed 1 KB blocks) and token rows (256 whole 128-byte lines) stream
// straight into LDS by global->LDS loads, two 64 KB buffers, as one stream
// across a workgroup's tiles.
//
// What bounds it: the matrix cores, fed from LDS, at the clock the power limit
// leaves (1.5-1.9 GHz under this kernel).  A stage is four phases of 16 MFMAs
// per wave (one 64 x 32 quadrant each).  The order of MFMAs, fragment reads and
// loads is pinned (sched_barrier): a phase reads the fragments of the next one
// right after their registers' last use, so no LDS latency is exposed, and
// issues a quarter stage (16 KB) into LDS that the phase before last has read
// out, so eight quarter stages are in flight and the wait at a phase's end
// (vmcnt(10), with an LDS-only barrier) is for the one issued five phases
// earlier.  The order before left the reads to the compiler, which placed each
// next to its MFMA, and waited for a whole stage at once.  Rates (156672 rows,
// us; before -> after; hipBLASLt's plain product in brackets):
//   1024 -> 1024  380 -> 325-340 [350-370]     4096 -> 1024 1218 -> 980-1060 [980-1020]
//   1024 -> 4096 + GELU 1441 -> 1200-1270 [1030-1090 without GELU]
//   1024 -> 1024 + scatter + residual 440 -> 362
// A tile's stores (64 contiguous bytes per row and instruction, nontemporal:
// 192 -> 768 of 524288 rows 290 -> 226 us, the others within 1 %) are waited
// for only at the end of the next tile's first stage.
//
// Tiles are walked persistently and XCD-aware: workgroup b runs on XCD b % 8
// (the hardware's round-robin), XCD x takes token blocks x, x + 8, ... and
// its workgroups sweep all feature tiles of one token block before the next,
// so a token block is read from HBM once and re-read by its feature tiles
// from that XCD's L2, while the weight stream (2 MB for a 1024 x 1024 layer)
// stays L2-resident.
#include "common.h"
#include "attn_core.h"
#include "gelu.h"

#include <type_traits>

namespace terra {
namespace {

constexpr int kLinF = 256;                         // output features per tile
constexpr int kLinT = 256;                         // token rows per tile
constexpr int kLinKS = 64;                         // input features per stage (two k-steps)
constexpr int kLinStages = 2;
constexpr uint32_t kLinDrop = 0xffff0000u;         // byte offset outside every output descriptor (plus a row's column)
constexpr int kLinStores = 16;                    // output stores per wave and tile (16 bytes per lane)
constexpr int kLinThreads = 512;
constexpr int kLinWBytes = kLinF * kLinKS * 2;     // 16 feature tiles x 2 packed 1 KB blocks
constexpr int kLinXBytes = kLinT * kLinKS * 2;     // 256 rows x 128 bytes
constexpr int kLinStage = kLinWBytes + kLinXBytes;
constexpr int kLinMaxN = 4096;                     // output features (bias staged in LDS)
constexpr int kLinBiasOff = kLinStages * kLinStage;
constexpr int kLinGeluOff = kLinBiasOff + kLinMaxN * 4;
static_assert(kLinGeluOff + kGeluBytes <= 160 * 1024, "LDS");

// LDS of each epilogue past the stages: bias (or, gelu-bwd, the column sums),
// then the GELU or slope table.
enum { kEpiStore = 0, kEpiGelu = 1, kEpiResidual = 2, kEpiScatter = 3, kEpiGeluKeep = 4, kEpiGeluBwd = 5, kEpiScatterAny = 6 };

static_assert(kLinGeluOff + kSlopeTabBytes <= 160 * 1024, "LDS");

template <int kEpi>
constexpr int lin_lds_bytes() {
  return kLinGeluOff + (kEpi == kEpiGeluBwd ? kSlopeTabBytes : (kEpi == kEpiGelu || kEpi == kEpiGeluKeep) ? kGeluBytes : 0);
}


struct LinParams {
  const uint8_t* x;       // [M rows] x K bf16, row stride x_ld bytes
  const uint8_t* w;       // packed [N, K] bf16
  const float* bias;      // [N] or NULL
  const uint8_t* res;     // residual (kEpiResidual / kEpiScatter) or h (kEpiGeluBwd), row stride y_ld
  uint8_t* keep;          // kEpiGeluKeep: h, row stride y_ld
  float* colsum;          // kEpiGeluBwd: [N] or NULL
  uint8_t* y;             // output rows, row stride y_ld bytes
  int64_t x_ld, y_ld;
  int64_t y_bytes;        // kEpiScatter: bytes of y (and res)
  int32_t M, N, K;
  int32_t tiles_m, tiles_n;
  // kEpiScatter: window-order rows of 8x8 windows -> grid tokens
  int32_t H, W, Hp, Wp, shift_h, shift_w, pad_top, pad_left;
  FastDiv fd_nWe, fd_nWw;  // emitted windows per image, windows per frame row
  FastDiv fd_wn, fd_ws;    // kEpiScatterAny: tokens per window, window width
  int32_t ws;
};

// This lane's index in its wave, computed where it is used (a volatile asm
// is not hoisted out of the tile loop and held in a register across it).
__device__ __forceinline__ int lin_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// 16-byte slot of (row, chunk c < 8) in a stage's token rows: 128-byte rows,
// the chunk XOR-swizzled within aligned groups of 16 rows, so that the rows of
// a fragment read hit distinct banks whether the LDS serves 8 lanes from 128
// bytes of banks or 16 lanes from 256 bytes per cycle.
__device__ __forceinline__ int lin_swz(int row) { return (row ^ ((row >> 3) & 1)) & 7; }
__device__ __forceinline__ int lin_slot(int row, int c) { return row * 8 + (c ^ lin_swz(row)); }

// Rows of other windows go through kEpiScatterAny (window 32, 156672 x 1024: the
// block 2042 -> 1971 us against the library's product and the reverse kernel).
// Grid token of window-order row m (8x8 windows: window m / 64, token m % 64;
// kAny: windows of any size), or -1 for a frame-padding token: the position the
// partition read the row from (pad, then a cyclic shift by (shift_h, shift_w)).
template <bool kAny>
__device__ __forceinline__ int64_t lin_grid_row(const LinParams& p, int m) {
  uint32_t w = (uint32_t)m >> 6, s = (uint32_t)m & 63u;
  uint32_t sr = s >> 3, sc = s & 7u, ws = 8u;
  if constexpr (kAny) {
    ws = (uint32_t)p.ws;
    p.fd_wn.divmod((uint32_t)m, w, s);
    p.fd_ws.divmod(s, sr, sc);
  }
  uint32_t b, wl, wr, wc;
  p.fd_nWe.divmod(w, b, wl);
  p.fd_nWw.divmod(wl, wr, wc);
  int ph = (int)(wr * ws + sr) + p.shift_h;
  int pw = (int)(wc * ws + sc) + p.shift_w;
  if (ph >= p.Hp) ph -= p.Hp;
  if (pw >= p.Wp) pw -= p.Wp;
  const int sh = ph - p.pad_top, sw = pw - p.pad_left;
  if ((unsigned)sh >= (unsigned)p.H || (unsigned)sw >= (unsigned)p.W) return -1;
  return ((int64_t)b * p.H + sh) * p.W + sw;
}

// bf16(r + o) per element of four packed bf16 pairs' worth (fp32 add, one rounding).
__device__ __forceinline__ uint2 add_bf16x4(uint2 r, uint2 o) {
  const uint32_t rw[2] = {r.x, r.y}, ow[2] = {o.x, o.y};
  uint32_t out[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const float lo = __uint_as_float(rw[q] << 16) + __uint_as_float(ow[q] << 16);
    const float hi = __uint_as_float(rw[q] & 0xffff0000u) + __uint_as_float(ow[q] & 0xffff0000u);
    out[q] = pack_bf16x2(lo, hi);
  }
  return make_uint2(out[0], out[1]);
}

template <int kEpi, bool kFar>
__global__ __launch_bounds__(kLinThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void linear_kernel(const LinParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3, wm = wave >> 2;  // token quarter, feature half
  float* s_bias = reinterpret_cast<float*>(smem + kLinBiasOff);
  const uint16_t* s_gelu = reinterpret_cast<const uint16_t*>(smem + kLinGeluOff);
  // Bias (and the GELU table) in LDS: a global load at a tile's start would
  // complete only behind the loads already in flight for the next stages.
  for (int e = tid; e < p.N; e += kLinThreads) s_bias[e] = p.bias != nullptr ? p.bias[e] : 0.f;
  if constexpr (kEpi == kEpiGelu || kEpi == kEpiGeluKeep)
    gelu_table_fill(reinterpret_cast<uint16_t*>(smem + kLinGeluOff), tid, kLinThreads);
  if constexpr (kEpi == kEpiGeluBwd)  // s_bias holds the column sums
    slope_table_fill(reinterpret_cast<float*>(smem + kLinGeluOff), tid, kLinThreads);
  __syncthreads();
  const int xcd = (int)blockIdx.x & 7;
  const int nx = ((int)gridDim.x - xcd + 7) >> 3;  // workgroups with this blockIdx % 8
  const int ksteps = p.K / 32;
  const int nst = p.K / kLinKS;                     // stages per tile
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(smem));

  // Tile t of this workgroup: slot (blockIdx.x >> 3) + t nx of its XCD's list.
  auto tile_of = [&](int t, int& m0, int& f0) -> bool {
    const int s = ((int)blockIdx.x >> 3) + t * nx;
    const int tq = s / p.tiles_n;
    const int tb = tq * 8 + xcd;
    m0 = tb * kLinT;
    f0 = (s - tq * p.tiles_n) * kLinF;
    return tb < p.tiles_m;
  };
  int m0, f0;
  if (!tile_of(0, m0, f0)) return;  // uniform

  // One stream of units over all stages of all of this workgroup's tiles.
  // Unit 4 s + {0: B0, 1: A0, 2: B1, 3: A1} of stage s (LDS buffer s & 1) is
  // 16 KB, two 1 KB blocks per wave; phase P issues unit P + 8.  A half h:
  // features 128 wm + 64 h + .., i.e. packed row tiles rt = 8 wm + 4 h + ..;
  // this wave loads both k-steps of rt = 8 (wave >> 2) + 4 h + (wave & 3).
  // B half h: token rows 64 wn + 32 h + ..; this wave loads the 8-row blocks
  // 8 (wave >> 1) + 4 h + 2 (wave & 1) + {0, 1}.
  const uint8_t* xbase = nullptr;  // token row m0 of the issue tile (wave-uniform)
  const uint8_t* wbase = nullptr;  // first packed block of the issue tile's features (wave-uniform)
  uint32_t xoff[2][2];
  const uint32_t woff = (uint32_t)((tid & 63) ^ (4 * (wave & 1))) * 16u;
  int issue_tile = 0, issue_st = 0, issue_buf = 0;
  auto set_sources = [&](int t) -> bool {
    int im, jf;
    if (!tile_of(t, im, jf)) return false;
    const int lane = lin_lane();
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int row = 8 * (8 * (wave >> 1) + 4 * h + 2 * (wave & 1) + q) + (lane >> 3);
        const int c = (lane & 7) ^ lin_swz(row);
        const int r = im + row < p.M ? row : p.M - 1 - im;  // rows past the end: a valid row, never stored
        xoff[h][q] = (uint32_t)r * (uint32_t)p.x_ld + (uint32_t)c * 16u;
      }
    xbase = p.x + (int64_t)im * p.x_ld;
    wbase = p.w + (int64_t)(jf / 16) * ksteps * 1024;
    return true;
  };
  bool issue_valid = set_sources(0);
  auto issue_b = [&](int h, int q) {
    dma_to_lds16_at(xbase + issue_st * 128, xoff[h][q],
                    lds0 + issue_buf * kLinStage + kLinWBytes + (8 * (wave >> 1) + 4 * h + 2 * (wave & 1) + q) * 1024);
  };
  auto issue_a = [&](int h, int q) {
    const int rt = 8 * (wave >> 2) + 4 * h + (wave & 3);
    dma_to_lds16_at(wbase + ((int64_t)rt * ksteps + 2 * issue_st + q) * 1024, woff,
                    lds0 + issue_buf * kLinStage + rt * 2048 + q * 1024);
  };
  auto issue_advance = [&]() {  // after the stage's last unit
    issue_buf ^= 1;
    if (++issue_st == nst) {
      issue_st = 0;
      issue_valid = set_sources(++issue_tile);
    }
  };

  // Fragment addresses in buffer 0 (loop-invariant).  Row c16 of A tile i is
  // feature 32 (i >> 1) + 8 (c16 >> 2) + 4 (i & 1) + (c16 & 3) of the half, so
  // an accumulator lane g holds 8 consecutive features of a token in tiles
  // 2 q and 2 q + 1, and the four lanes g 64 contiguous bytes of the output
  // row.  Packed row tiles of odd index have their 64-byte row groups stored
  // pairwise swapped (woff), so a fragment's 16 rows hit distinct banks.
  uint32_t aaddr[2], baddr[2];
  {
    const int lane = tid & 63, g = lane >> 4, c16 = lane & 15;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      aaddr[i] = (8 * wm + (c16 >> 3)) * 2048 +
                 (16 * g + 8 * ((c16 >> 2) & 1) + 4 * (i ^ (c16 >> 3)) + (c16 & 3)) * 16;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) baddr[kk] = kLinWBytes + lin_slot(64 * wn + c16, 4 * kk + g) * 16;
  }
  auto frag_a = [&](uint32_t bo, int h, int kk, int i) {
    return *reinterpret_cast<const uint4*>(smem + bo + aaddr[i & 1] + h * 8192 + (i >> 1) * 4096 + kk * 1024);
  };
  auto frag_b = [&](uint32_t bo, int h, int kk, int j) {
    return *reinterpret_cast<const uint4*>(smem + bo + baddr[kk] + (32 * h + 16 * j) * 128);
  };

  f32x4 acc[8][4];
  auto mma = [&](int ah, int bh, int n, const uint4 (&a)[2][4], const uint4 (&b)[2][2]) {  // n-th of a quadrant's 16
    const int kk = n >> 3, j = (n >> 2) & 1, i = n & 3;
    f32x4& c = acc[4 * ah + i][2 * bh + j];
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[kk][i]),
                                                __builtin_bit_cast(bf16x8, b[kk][j]), c, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // End of phase P: units up to P + 3 have landed (all but the five newest, of
  // two loads each).  In a tile's first stage the previous tile's kLinStores
  // output stores (issued by every wave whatever its rows) lie between units
  // P + 4 and P + 8, so as many more may be open: the stores drain under the
  // MFMAs instead of being waited for.
  auto phase_end = [&](bool live, bool after_stores) {
    if (!live)
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    else if (after_stores)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(10 + (kEpi == kEpiGeluKeep ? 2 : 1) * kLinStores) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(10)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  uint4 a[2][4], bx[2][2], by[2][2];
  int buf = 0;
  // One stage: four phases of 16 MFMAs (a quadrant each), with the fragment
  // reads of the next phase and one unit's loads between them, in program
  // order.  A fragment is reloaded right after its last use: a[kk][i] after
  // MFMA 8 kk + 4 + i, b[kk][j] after MFMA 8 kk + 4 j + 3.  Fragments read in
  // one phase are waited for by the next phase's MFMAs, so a unit's place is
  // free from the phase after that on (B0's, read by MFMA 0 of the phase
  // before, from the next one on: lgkmcnt(4) leaves only the four newest A
  // reads open there).  On entry b0 holds B0; on exit b1 holds the next
  // stage's B0 and a its A0.
  auto stage = [&](uint4 (&b0)[2][2], uint4 (&b1)[2][2], bool after_stores) {
    const bool live = issue_valid;  // uniform
    const uint32_t cur = buf * kLinStage, nxt = cur ^ kLinStage;
#pragma unroll
    for (int n = 0; n < 16; ++n) {  // A0 B0; reads B1
      mma(0, 0, n, a, b0);
      if (n < 4) b1[n >> 1][n & 1] = frag_b(cur, 1, n >> 1, n & 1);
      if ((n == 6 || n == 10) && live) issue_b(0, n == 10);
      __builtin_amdgcn_sched_barrier(0);
    }
    phase_end(live, after_stores);
#pragma unroll
    for (int n = 0; n < 16; ++n) {  // A0 B1; reads A1
      mma(0, 1, n, a, b1);
      if (n & 4) a[n >> 3][n & 3] = frag_a(cur, 1, n >> 3, n & 3);
      if ((n == 1 || n == 9) && live) issue_a(0, n == 9);
      __builtin_amdgcn_sched_barrier(0);
    }
    phase_end(live, after_stores);
#pragma unroll
    for (int n = 0; n < 16; ++n) {  // A1 B1; reads the next stage's B0
      mma(1, 1, n, a, b1);
      if ((n & 3) == 3 && n < 15) b1[n >> 3][(n >> 2) & 1] = frag_b(nxt, 0, n >> 3, (n >> 2) & 1);
      if ((n == 5 || n == 9) && live) issue_b(1, n == 9);
      __builtin_amdgcn_sched_barrier(0);
    }
    phase_end(live, after_stores);
#pragma unroll
    for (int n = 0; n < 16; ++n) {  // A1 B0; reads the next stage's A0 (and the last of its B0)
      mma(1, 0, n, a, b0);
      if (n == 0) b1[1][1] = frag_b(nxt, 0, 1, 1);
      if (n & 4) a[n >> 3][n & 3] = frag_a(nxt, 0, n >> 3, n & 3);
      if ((n == 2 || n == 9) && live) issue_a(1, n == 9);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (live) issue_advance();
    asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
    phase_end(live, after_stores);
    buf ^= 1;
  };
  // Units 0 .. 7; unit 8 takes unit 0's place only once every wave has read it.
  auto issue_stage = [&]() {
    if (!issue_valid) return;  // uniform
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int q = 0; q < 2; ++q) issue_b(h, q);
#pragma unroll
      for (int q = 0; q < 2; ++q) issue_a(h, q);
    }
    issue_advance();
  };
  issue_stage();
  const bool second = issue_valid;
  issue_stage();
  phase_end(second, false);
#pragma unroll
  for (int n = 0; n < 8; ++n) a[n >> 2][n & 3] = frag_a(0, 0, n >> 2, n & 3);
#pragma unroll
  for (int n = 0; n < 4; ++n) bx[n >> 1][n & 1] = frag_b(0, 0, n >> 1, n & 1);
  lds_barrier();
  for (int t = 0;; ++t) {
    {
      const int g = lin_lane() >> 4;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const f32x4 bv = kEpi == kEpiGeluBwd ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4*>(s_bias + f0 + 128 * wm + 32 * (i >> 1) + 8 * g + 4 * (i & 1));
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = bv;
      }
    }
    for (int st = 0; st + 1 < nst; st += 2) {
      stage(bx, by, !kFar && st == 0 && t > 0);
      stage(by, bx, false);
    }
    if (nst & 1) {  // uniform
      stage(bx, by, !kFar && nst == 1 && t > 0);
#pragma unroll
      for (int n = 0; n < 4; ++n) bx[n >> 1][n & 1] = by[n >> 1][n & 1];
    }
    const int lane = lin_lane();
    const int g = lane >> 4, c16 = lane & 15;

    // Epilogue: lane (c16, g) of tiles (2 q + i, j), i < 2, holds the 8
    // features f0 + 128 wm + 32 q + 8 g .. of token row m0 + 64 wn + 16 j + c16:
    // 16 bytes at byte offset off[j] + 64 q of the output.  Through a
    // descriptor, rows past the end and frame padding take an offset outside
    // it: their loads give 0, their stores are dropped, and every wave issues
    // kLinStores stores.  Outputs of more bytes than a descriptor covers
    // (kFar) go through 64-bit addresses under a predicate.
    uint2 o[4][8];
    if constexpr (kEpi != kEpiGeluBwd) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          o[j][i] = make_uint2(pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3]));
      __builtin_amdgcn_sched_barrier(0);  // the fp32 accumulators end here
    }
    constexpr bool kScatter = kEpi == kEpiScatter || kEpi == kEpiScatterAny;
    constexpr bool kRes = kEpi == kEpiResidual || kScatter;
    const int64_t tile0 = kScatter ? 0 : (int64_t)m0 * p.y_ld;
    const int left = p.M - m0 < kLinT ? p.M - m0 : kLinT;
    const uint32_t span = kScatter ? (uint32_t)p.y_bytes : (uint32_t)((left - 1) * p.y_ld + p.N * 2);
    const __amdgpu_buffer_rsrc_t yr = buffer_rsrc(p.y + tile0, span);
    const __amdgpu_buffer_rsrc_t rr = buffer_rsrc(p.res + tile0, span);
    using Off = std::conditional_t<kFar, int64_t, uint32_t>;
    Off off[4];
    bool ok[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 64 * wn + 16 * j + c16;
      int64_t orow = row;
      ok[j] = row < left;
      if constexpr (kScatter) {
        orow = ok[j] ? lin_grid_row<kEpi == kEpiScatterAny>(p, m0 + row) : -1;
        ok[j] = orow >= 0;  // frame padding
      }
      const uint32_t col = (uint32_t)(f0 + 128 * wm + 8 * g) * 2u;
      if constexpr (kFar)
        off[j] = orow * p.y_ld + col;
      else
        off[j] = (ok[j] ? (uint32_t)(orow * p.y_ld) : kLinDrop) + col;
    }
    if constexpr (kRes) {
      // Every residual load before the first store (a later load would wait
      // for the stores ahead of it), in two batches for the registers' sake.
#pragma unroll
      for (int jb = 0; jb < 4; jb += 2) {
        u32x4 r[2][4];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if constexpr (kFar) {
              r[j][q] = u32x4{0, 0, 0, 0};
              if (ok[jb + j]) {
                const uint2* src = reinterpret_cast<const uint2*>(p.res + tile0 + off[jb + j] + 64 * q);
                r[j][q] = u32x4{src[0].x, src[0].y, src[1].x, src[1].y};
              }
            } else {
              r[j][q] = __builtin_amdgcn_raw_buffer_load_b128(rr, off[jb + j] + 64 * q, 0, 0);
            }
          }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            uint2(&v)[8] = o[jb + j];
            v[2 * q] = add_bf16x4(make_uint2(r[j][q][0], r[j][q][1]), v[2 * q]);
            v[2 * q + 1] = add_bf16x4(make_uint2(r[j][q][2], r[j][q][3]), v[2 * q + 1]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (kEpi == kEpiGeluBwd) {
      const uint8_t* s_slope = smem + kLinGeluOff;
      // Two of the four 32-feature groups q at a time: their h, their products
      // and column sums; every load before the first store.
#pragma unroll
      for (int qb = 0; qb < 4; qb += 2) {
        u32x4 h[2][4];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int j = 0; j < 4; ++j) h[q][j] = __builtin_amdgcn_raw_buffer_load_b128(rr, off[j] + 64 * (qb + q), 0, 0);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float sl[8];
            slope_chunk(h[q][j], s_slope, sl);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const f32x4& c = acc[2 * (qb + q) + (e >> 1)][j];
              const uint32_t v = pack_bf16x2(c[2 * (e & 1)] * sl[2 * e], c[2 * (e & 1) + 1] * sl[2 * e + 1]);
              uint2& d = o[j][2 * (qb + q) + (e >> 1)];
              if (e & 1)
                d.y = v;
              else
                d.x = v;
              // the values as written; rows past the end add nothing (their h is 0, but their products are not)
              if (ok[j]) {
                sum[2 * e] += __uint_as_float(v << 16);
                sum[2 * e + 1] += __uint_as_float(v & 0xffff0000u);
              }
            }
          }
          if (p.colsum != nullptr) {
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = row16_sum(sum[e]);
            if (c16 == 0) {
#pragma unroll
              for (int e = 0; e < 8; ++e) atomicAdd(&s_bias[f0 + 128 * wm + 32 * (qb + q) + 8 * g + e], sum[e]);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (kEpi == kEpiGeluKeep) {
        const __amdgpu_buffer_rsrc_t kr = buffer_rsrc(p.keep + tile0, span);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          __builtin_amdgcn_raw_buffer_store_b128(
              u32x4{o[j][2 * q].x, o[j][2 * q].y, o[j][2 * q + 1].x, o[j][2 * q + 1].y}, kr, off[j] + 64 * q, 0, kCacheNt);
      }
      if constexpr (kEpi == kEpiGelu || kEpi == kEpiGeluKeep) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t v[4] = {o[j][2 * q].x, o[j][2 * q].y, o[j][2 * q + 1].x, o[j][2 * q + 1].y};
          gelu_chunk(v, s_gelu);
          o[j][2 * q] = make_uint2(v[0], v[1]);
          o[j][2 * q + 1] = make_uint2(v[2], v[3]);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int d = 64 * q;
        const uint2 lo = o[j][2 * q], hi = o[j][2 * q + 1];
        if constexpr (kFar) {
          if (ok[j]) {
            uint2* dst = reinterpret_cast<uint2*>(p.y + tile0 + off[j] + d);
            dst[0] = lo;
            dst[1] = hi;
          }
        } else {
          __builtin_amdgcn_raw_buffer_store_b128(u32x4{lo.x, lo.y, hi.x, hi.y}, yr, off[j] + d, 0, kCacheNt);
        }
      }
    }
    if (!tile_of(t + 1, m0, f0)) break;  // uniform
  }
  if constexpr (kEpi == kEpiGeluBwd) {
    lds_barrier();  // every wave's column sums are in
    if (p.colsum != nullptr)
      for (int e = tid; e < p.N; e += kLinThreads)
        if (s_bias[e] != 0.f) unsafeAtomicAdd(p.colsum + e, s_bias[e]);
  }
}

template <int kEpi, bool kFar>
int launch_linear(const LinParams& p, hipStream_t s) {
  constexpr int lds = lin_lds_bytes<kEpi>();
  auto kern = linear_kernel<kEpi, kFar>;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return fail(TERRA_ERR_LAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(attr));
  constexpr int kMaxDevices = 64;
  static int cache[kMaxDevices] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(TERRA_ERR_LAUNCH, "cannot query the current device");
  if (cache[dev] == 0) {
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kLinThreads, lds) != hipSuccess)
      return fail(TERRA_ERR_LAUNCH, "cannot size the linear kernel grid for this device");
    const int resident = cus * (per_cu > 0 ? per_cu : 1);
    cache[dev] = resident >= 16 ? resident - resident % 8 : 8;  // whole XCD rounds
  }
  kern<<<cache[dev], kLinThreads, lds, s>>>(p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TERRA_ERR_LAUNCH, "linear kernel launch failed: %s", hipGetErrorString(e));
  return TERRA_OK;
}

// Outputs whose tiles (scatter: the whole grid) a buffer descriptor covers take
// the descriptor form: all but grids of 4 GiB and more, or row strides of 16
// MiB and more (the other epilogues' rows are contiguous, so never those).
template <int kEpi>
int dispatch_linear(const LinParams& p, hipStream_t s) {
  if constexpr (kEpi == kEpiStore || kEpi == kEpiGelu || kEpi == kEpiScatter || kEpi == kEpiScatterAny) {
    const int64_t bytes = kEpi == kEpiScatter || kEpi == kEpiScatterAny ? p.y_bytes : (int64_t)kLinT * p.y_ld;
    if (bytes >= (int64_t)kLinDrop) return launch_linear<kEpi, true>(p, s);
  }
  return launch_linear<kEpi, false>(p, s);
}

bool lin_overlap(const void* a, int64_t abytes, const void* b, int64_t bbytes) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return x < y + (uintptr_t)bbytes && y < x + (uintptr_t)abytes;
}

// Shared checks of both entry points; fills the GEMM fields of `p`.
int lin_validate(const void* x, const void* w, const float* bias, const void* y, int dtype, int64_t rows,
                 int in_features, int out_features, int64_t x_stride, int64_t y_stride, LinParams* p) {
  if (x == nullptr || w == nullptr || y == nullptr) return fail(TERRA_ERR_NULL, "x, weight and y must be non-NULL");
  if (dtype_size(dtype) == 0) return fail(TERRA_ERR_DTYPE, "unknown dtype %d", dtype);
  if (dtype != TERRA_DTYPE_BF16) return fail(TERRA_ERR_UNSUPPORTED, "the linear kernels are bf16 only");
  if (rows < 0 || rows >= (1ll << 31)) return fail(TERRA_ERR_SHAPE, "rows must be in [0, 2^31) (got %lld)",
                                                   (long long)rows);
  if (in_features <= 0 || in_features % kLinKS != 0 || out_features <= 0 || out_features % kLinF != 0 ||
      out_features > kLinMaxN)
    return fail(TERRA_ERR_SHAPE,
                "in_features must be a positive multiple of 64 and out_features a multiple of 256 up to %d (got %d, %d)",
                kLinMaxN, in_features, out_features);
  if (x_stride < in_features || y_stride < out_features || x_stride % 8 != 0 || y_stride % 4 != 0 ||
      x_stride * 2 * kLinT >= (1ll << 32))
    return fail(TERRA_ERR_SHAPE,
                "row strides must cover the rows (x_stride >= %d, a multiple of 8; y_stride >= %d, a multiple of 4)",
                in_features, out_features);
  if (((uintptr_t)x & 15u) != 0 || ((uintptr_t)w & 15u) != 0 || ((uintptr_t)bias & 15u) != 0 ||
      ((uintptr_t)y & 7u) != 0)
    return fail(TERRA_ERR_ALIGN, "x, weight and bias must be 16-byte aligned and y 8-byte aligned");
  if ((int64_t)out_features * in_features * 2 >= (1ll << 31))
    return fail(TERRA_ERR_SHAPE, "weight of %d x %d exceeds 2 GB", out_features, in_features);
  p->x = static_cast<const uint8_t*>(x);
  p->w = static_cast<const uint8_t*>(w);
  p->bias = bias;
  p->y = static_cast<uint8_t*>(const_cast<void*>(y));
  p->res = nullptr;
  p->x_ld = x_stride * 2;
  p->y_ld = y_stride * 2;
  p->M = (int32_t)rows;
  p->N = out_features;
  p->K = in_features;
  p->tiles_m = (int32_t)((rows + kLinT - 1) / kLinT);
  p->tiles_n = out_features / kLinF;
  return TERRA_OK;
}

}  // namespace
}  // namespace terra

using namespace terra;

extern "C" int terra_swin_linear(const void* x, void* y, int dtype, int64_t rows, int in_features,
                                 int out_features, int64_t x_stride, int64_t y_stride, const void* weight_packed,
                                 const float* bias, int epilogue, void* stream) {
  clear_error();
  LinParams p{};
  const int st =
      lin_validate(x, weight_packed, bias, y, dtype, rows, in_features, out_features, x_stride, y_stride, &p);
  if (st != TERRA_OK) return st;
  if (epilogue != TERRA_LINEAR_STORE && epilogue != TERRA_LINEAR_GELU)
    return fail(TERRA_ERR_SHAPE, "unknown epilogue %d", epilogue);
  const int64_t xb = (rows - 1) * p.x_ld + (int64_t)in_features * 2, yb = (rows - 1) * p.y_ld + (int64_t)out_features * 2;
  if (rows > 0 && lin_overlap(x, xb, y, yb)) return fail(TERRA_ERR_SHAPE, "y overlaps x");
  if (rows == 0) return TERRA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return epilogue == TERRA_LINEAR_GELU ? dispatch_linear<kEpiGelu>(p, s) : dispatch_linear<kEpiStore>(p, s);
}

// any_window: the entry takes windows of every size, else 8x8 ones.
static int linear_residual(const void* x, const void* residual, void* y, int dtype, int64_t rows, int in_features,
                           int out_features, const void* weight_packed, const float* bias,
                           const terra_swin_geom* geom, bool any_window, void* stream) {
  LinParams p{};
  const int st = lin_validate(x, weight_packed, bias, y, dtype, rows, in_features, out_features, in_features,
                              out_features, &p);
  if (st != TERRA_OK) return st;
  if (residual == nullptr) return fail(TERRA_ERR_NULL, "residual must be non-NULL");
  if (((uintptr_t)residual & 7u) != 0) return fail(TERRA_ERR_ALIGN, "residual must be 8-byte aligned");
  p.res = static_cast<const uint8_t*>(residual);
  int64_t out_rows = rows;  // rows of residual / y
  if (geom != nullptr) {
    GeomDims dims;
    const int gs = validate_geom(geom, &dims);
    if (gs != TERRA_OK) return gs;
    const terra_swin_geom& q = *geom;
    if (q.window != 8 && !any_window)
      return fail(TERRA_ERR_UNSUPPORTED, "the scatter epilogue needs 8x8 windows (got %d)", q.window);
    if (q.channels != out_features)
      return fail(TERRA_ERR_SHAPE, "geom channels (%d) must equal out_features (%d)", q.channels, out_features);
    // Every grid token must come from exactly one emitted window, so that the
    // scatter writes all of y: the whole frame emitted, no valid-window range.
    if (q.win_row_begin != 0 || dims.rows != dims.nWh || q.valid_end > 0)
      return fail(TERRA_ERR_UNSUPPORTED,
                  "the scatter epilogue needs every window of the frame emitted (no window-row or valid-window range)");
    const int64_t wn = (int64_t)q.window * q.window;
    if (rows != (int64_t)q.batch * dims.nWe * wn)
      return fail(TERRA_ERR_SHAPE, "rows (%lld) must be the window tokens of the frame (%lld)", (long long)rows,
                  (long long)((int64_t)q.batch * dims.nWe * wn));
    out_rows = (int64_t)q.batch * q.height * q.width;
    p.H = q.height; p.W = q.width; p.Hp = (int32_t)dims.Hp; p.Wp = (int32_t)dims.Wp;
    p.shift_h = q.shift_h; p.shift_w = q.shift_w; p.pad_top = q.pad_top; p.pad_left = q.pad_left;
    p.fd_nWe = FastDiv((uint32_t)dims.nWe);
    p.fd_nWw = FastDiv((uint32_t)dims.nWw);
    p.ws = q.window;
    p.fd_wn = FastDiv((uint32_t)wn);
    p.fd_ws = FastDiv((uint32_t)q.window);
  }
  const int64_t xb = rows * (int64_t)in_features * 2, yb = out_rows * (int64_t)out_features * 2;
  if (rows > 0 && lin_overlap(x, xb, y, yb)) return fail(TERRA_ERR_SHAPE, "y overlaps x");
  if (y != residual && lin_overlap(residual, yb, y, yb))
    return fail(TERRA_ERR_SHAPE, "y overlaps residual without being residual");
  if (rows == 0) return TERRA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  p.y_bytes = yb;
  if (geom == nullptr) return dispatch_linear<kEpiResidual>(p, s);
  // 8x8 windows split a row number by shifts, the others by two more divisions.
  return p.ws == 8 ? dispatch_linear<kEpiScatter>(p, s) : dispatch_linear<kEpiScatterAny>(p, s);
}

extern "C" int terra_swin_linear_residual(const void* x, const void* residual, void* y, int dtype, int64_t rows,
                                          int in_features, int out_features, const void* weight_packed,
                                          const float* bias, const terra_swin_geom* geom, void* stream) {
  clear_error();
  return linear_residual(x, residual, y, dtype, rows, in_features, out_features, weight_packed, bias, geom, false,
                         stream);
}

extern "C" int terra_swin_linear_scatter(const void* x, const void* residual, void* y, int dtype, int64_t rows,
                                         int in_features, int out_features, const void* weight_packed,
                                         const float* bias, const terra_swin_geom* geom, void* stream) {
  clear_error();
  if (geom == nullptr) return fail(TERRA_ERR_NULL, "geom must be non-NULL");
  return linear_residual(x, residual, y, dtype, rows, in_features, out_features, weight_packed, bias, geom, true,
                         stream);
}

extern "C" int terra_swin_linear_gelu_keep(const void* x, void* h, void* y, int dtype, int64_t rows, int in_features,
                                           int out_features, const void* weight_packed, const float* bias,
                                           void* stream) {
  clear_error();
  LinParams p{};
  const int st = lin_validate(x, weight_packed, bias, y, dtype, rows, in_features, out_features, in_features,
                              out_features, &p);
  if (st != TERRA_OK) return st;
  if (h == nullptr) return fail(TERRA_ERR_NULL, "h must be non-NULL");
  if (((uintptr_t)h & 7u) != 0) return fail(TERRA_ERR_ALIGN, "h must be 8-byte aligned");
  const int64_t xb = rows * (int64_t)in_features * 2, yb = rows * (int64_t)out_features * 2;
  if (rows > 0 && (lin_overlap(x, xb, y, yb) || lin_overlap(x, xb, h, yb) || lin_overlap(h, yb, y, yb)))
    return fail(TERRA_ERR_SHAPE, "x, h and y must not overlap");
  p.keep = static_cast<uint8_t*>(h);
  if (rows == 0) return TERRA_OK;
  return dispatch_linear<kEpiGeluKeep>(p, static_cast<hipStream_t>(stream));
}

extern "C" int terra_swin_linear_gelu_bwd(const void* dy, const void* h, void* dh, int dtype, int64_t rows,
                                          int in_features, int out_features, const void* weight_packed,
                                          float* column_sums, void* stream) {
  clear_error();
  LinParams p{};
  const int st = lin_validate(dy, weight_packed, nullptr, dh, dtype, rows, in_features, out_features, in_features,
                              out_features, &p);
  if (st != TERRA_OK) return st;
  if (h == nullptr) return fail(TERRA_ERR_NULL, "h must be non-NULL");
  if (((uintptr_t)h & 7u) != 0 || ((uintptr_t)column_sums & 3u) != 0)
    return fail(TERRA_ERR_ALIGN, "h must be 8-byte and column_sums 4-byte aligned");
  const int64_t xb = rows * (int64_t)in_features * 2, yb = rows * (int64_t)out_features * 2;
  if (rows > 0 && (lin_overlap(dy, xb, dh, yb) || lin_overlap(h, yb, dh, yb)))
    return fail(TERRA_ERR_SHAPE, "dh must not overlap dy or h");
  p.res = static_cast<const uint8_t*>(h);
  p.colsum = column_sums;
  if (rows == 0) return TERRA_OK;
  return dispatch_linear<kEpiGeluBwd>(p, static_cast<hipStream_t>(stream));
}
