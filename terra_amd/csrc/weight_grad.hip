// Weight gradients of the training step's linear layers for gfx950:
//
//   dW[o][i] = sum_t dY[t][o] X[t][i]      bf16 operands, fp32 sums and result
//
// (the autograd backward of an nn.Linear's weight over the token rows,
// models/attention.py:223-228, 281 and models/mlp.py:162-168).  The contraction
// runs over every token (10^5 - 10^6) and the result is small, so the tokens are
// cut into slices, each (output tile, slice) pair is one workgroup, and a second
// pass adds the slices in order.
//
// Both operands are stored with the contracted dimension (tokens) outermost.  A
// workgroup streams stages of 32 token rows of its two column ranges straight
// into LDS (global->LDS loads by buffer descriptor: rows past the end read 0),
// wg_bufs buffers (6 to 8), and reads MFMA fragments by transposed LDS reads
// (ds_read_b64_tr_b16: four tokens of one column per lane), so nothing is
// transposed through memory.  x is the A operand, so a lane's four accumulator
// rows are consecutive in dW; eight waves, 2 x 4, each WA / 2 x WB / 4 of the
// tile.
//
// Sums are taken in two levels: the matrix cores add kWgFold stages (1024
// tokens) to an accumulator, which is then added to a second one.  One chain
// over a slice rounds the growing sum at every stage.  Normwise errors against
// float64, 156672 x 4096 x 1024: 4 slices of one chain 1.3e-6, in two levels
// 2.5e-7, the library's product over 64 slices 3.1e-7; 524288 x 768 x 192: 5.2e-7,
// 2.1e-7, 4.0e-7.  Two accumulators per output leave room for tiles of 128 x 256
// where one had 256 x 256 (1137 us); the same error by one chain in each of 64
// slices costs 2 GB of partial results.
// Times, us, library / here: 156672 x 4096 x 1024 1562 / 1370 (1520 in 64
// slices), 156672 x 3072 x 1024 1183 / 1089, 524288 x 768 x 192 255 / 204,
// 524288 x 576 x 192 246 / 176, 32768 x 768 x 768 54 / 53, 2001 x 1024 x 1024 22 / 25.
//
// What bounds it: for narrow layers (C = 192) HBM, every operand row being read
// once (the output tiles of a slice share an XCD's L2); for wide ones (C =
// 1024) the matrix cores and the power limit, and 15 TB/s out of L2.  A stage's
// fragments are read while the one before is multiplied, each right after its
// registers' last use, in pinned order, and the loads run as many stages ahead
// as the LDS holds.  An XCD's workgroups take a square of a slice's tiles (the
// shorter side of their grid first), so that they share their rows (1024 x 4096:
// 1405 -> 1380 us).
#include "common.h"
#include "attn_core.h"

namespace terra {
namespace {

constexpr int kWgThreads = 512;
constexpr int kWgTok = 32;     // tokens per stage (one MFMA k-step)
constexpr int kWgFold = 32;    // stages per accumulator chain
constexpr int kWgCus = 256;    // one workgroup per CU
constexpr int kWgLong = 4096;  // per slice, from which a second round pays
constexpr int kWgMinTokens = 512;  // per slice: below this its fixed cost outweighs the split

struct WgParams {
  const uint8_t* a;   // x:  [rows] x na bf16
  const uint8_t* b;   // dy: [rows] x nb bf16
  float* out;         // [nb][na]; slice s at out + s * na * nb
  int64_t rows;
  int64_t slice_rows; // a multiple of kWgTok
  int32_t na, nb;
  int32_t tiles_a, tiles_b, tiles, slices;
  int32_t per_xcd;    // workgroups per XCD
};

// LDS buffers of a tile: as many stages as fit (6 for 128 x 256), at most 8.
constexpr int wg_bufs(int wa, int wb) {
  const int n = 160 * 1024 / (kWgTok * (wa + wb) * 2);
  return n < 8 ? n : 8;
}

// Chunk swizzle of token row r in a tile row of W columns: 32-byte pairs of
// 16-byte chunks move by 2 f(r) within 256-byte groups (row pitch a multiple
// of 256 bytes) or within 128-byte groups (pitch an odd multiple of 128, whose
// odd rows are already half a bank period off), so that the 16 tokens of a
// transposed read lie two to a bank.
template <int W>
__device__ __forceinline__ int wg_swz(int r) {
  return W % 128 == 0 ? 2 * (r & 7) : 2 * ((r >> 1) & 3);
}

template <int WA, int WB>
__global__ __launch_bounds__(kWgThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void weight_grad_kernel(const WgParams p) {
  constexpr int kPa = WA * 2, kPb = WB * 2;           // LDS row pitches
  constexpr int kStage = kWgTok * (kPa + kPb);
  constexpr int kBlkA = kWgTok * kPa / 1024, kBlkB = kWgTok * kPb / 1024;
  constexpr int kBlks = kBlkA + kBlkB;                // 1 KB loads per stage
  constexpr int kPer = (kBlks + 7) / 8;               // per wave, at most
  constexpr int kRem = kBlks % 8;                     // waves >= kRem (if any) make one less
  constexpr int NI = WA / 32, NJ = WB / 64;           // fragments per wave
  constexpr int kBufs = wg_bufs(WA, WB);
  static_assert(WA % 64 == 0 && WB % 64 == 0 && kBufs >= 4 && (kBufs - 3) * kPer < 64, "tile");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int id = ((int)blockIdx.x & 7) * p.per_xcd + ((int)blockIdx.x >> 3);
  if (id >= p.tiles * p.slices || ((int)blockIdx.x >> 3) >= p.per_xcd) return;  // uniform
  const int slice = id / p.tiles, tile = id - slice * p.tiles;
  const bool a_first = p.tiles_a <= p.tiles_b;
  const int side = a_first ? p.tiles_a : p.tiles_b;
  const int tq = tile / side, tr = tile - tq * side;
  const int ta = a_first ? tr : tq, tb = a_first ? tq : tr;
  const int wn = wave & 3, wm = wave >> 2;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(smem));

  // Loads of this wave: block q of the stage holds the A rows, then the B rows,
  // row-major.  The lane offsets are loop-invariant; the descriptors move.
  uint32_t voff[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int blk = wave + 8 * q;
    const bool isa = blk < kBlkA;
    const int byte = (isa ? blk : blk - kBlkA) * 1024 + lane * 16;
    const int pitch = isa ? kPa : kPb;
    const int r = byte / pitch, s = (byte - r * pitch) / 16;
    const int c = s ^ (isa ? wg_swz<WA>(r) : wg_swz<WB>(r));
    voff[q] = (uint32_t)r * (uint32_t)((isa ? p.na : p.nb) * 2) + (uint32_t)c * 16u;
  }
  const int64_t row0 = (int64_t)slice * p.slice_rows;
  const int64_t row1 = row0 + p.slice_rows < p.rows ? row0 + p.slice_rows : p.rows;
  const int stages = (int)((row1 - row0 + kWgTok - 1) / kWgTok);
  // Bytes of the tensors from a stage's first element on, at most 32 rows.
  const uint8_t* abase = p.a + row0 * p.na * 2 + (int64_t)ta * WA * 2;
  const uint8_t* bbase = p.b + row0 * p.nb * 2 + (int64_t)tb * WB * 2;
  int issue_stage = 0;
  uint32_t issue_off = 0;  // LDS buffer of issue_stage
  auto issue = [&](int q) {
    const int blk = wave + 8 * q;
    if (kRem != 0 && q == kPer - 1 && wave >= kRem) return;  // uniform
    const int64_t left = row1 - row0 - (int64_t)issue_stage * kWgTok;
    const int rows = left < kWgTok ? (int)left : kWgTok;
    const bool isa = blk < kBlkA;
    const int pitch = (isa ? p.na : p.nb) * 2;
    const int col = isa ? ta * WA * 2 : tb * WB * 2;
    const uint8_t* base = (isa ? abase : bbase) + (int64_t)issue_stage * kWgTok * pitch;
    dma_buffer_to_lds16(buffer_rsrc(base, (uint32_t)(rows * pitch - col)), voff[q],
                        lds0 + issue_off + blk * 1024);
  };
  auto next_buffer = [](uint32_t off) { return off + kStage == kBufs * kStage ? 0u : off + kStage; };
  auto issue_advance = [&]() {
    ++issue_stage;
    issue_off = next_buffer(issue_off);
  };

  // Fragment addresses in buffer 0: lane (c16, g) of a transposed read addresses
  // token 4 g + (c16 >> 2), columns c0 + 4 (c16 & 3) .., and receives column
  // c0 + c16 of tokens 4 g .. + 3; a second read 16 tokens on fills the k-step.
  uint32_t aaddr[NI], baddr[NJ];
  {
    const int g = lane >> 4, c16 = lane & 15;
    const int tok = 4 * g + (c16 >> 2);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int ch = (wm * (WA / 2) + 16 * i) / 8 + ((c16 & 3) >> 1);
      aaddr[i] = tok * kPa + (ch ^ wg_swz<WA>(tok)) * 16 + (c16 & 1) * 8;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int ch = (wn * (WB / 4) + 16 * j) / 8 + ((c16 & 3) >> 1);
      baddr[j] = kWgTok * kPa + tok * kPb + (ch ^ wg_swz<WB>(tok)) * 16 + (c16 & 1) * 8;
    }
  }
  auto frag = [&](uint32_t addr, int pitch) {
    const uint2 lo = lds_read_tr16(smem + addr), hi = lds_read_tr16(smem + addr + 16 * pitch);
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
  };
  // End of stage s: stage s + 2 has landed (s + 3 .. s + kBufs - 1 may be in
  // flight), and every wave has multiplied stage s, so its buffer may be filled
  // again.
  auto stage_end = [&](bool live) {
    if (!live) {
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    } else if (kRem == 0 || wave < kRem) {
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((kBufs - 3) * kPer) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((kBufs - 3) * (kPer - 1)) : "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x4 acc[NI][NJ], sum[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        sum[i][j] = sum[i][j] + acc[i][j];
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  for (int s = 0; s < kBufs - 1 && s < stages; ++s) {
#pragma unroll
    for (int q = 0; q < kPer; ++q) issue(q);
    issue_advance();
  }
  stage_end(stages >= kBufs - 1);  // stages 0 and 1
  uint4 a[NI], b[NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i) a[i] = frag(aaddr[i], kPa);
#pragma unroll
  for (int j = 0; j < NJ; ++j) b[j] = frag(baddr[j], kPb);
  uint32_t nxt = 0;
  for (int s = 0; s < stages; ++s) {
    nxt = next_buffer(nxt);  // past the last stage: unused
    const bool live = issue_stage < stages;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[i]),
                                                            __builtin_bit_cast(bf16x8, b[j]), acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (j == NJ - 1) a[i] = frag(nxt + aaddr[i], kPa);
        if (i == NI - 1) b[j] = frag(nxt + baddr[j], kPb);
        if (j == 0 && i < kPer && live) issue(i);
        __builtin_amdgcn_sched_barrier(0);
      }
    if (live) issue_advance();
    stage_end(live);
    if (s % kWgFold == kWgFold - 1) fold();  // uniform
  }
  fold();

  // Lane (c16, g) of (i, j): A indexes 16 i + 4 g + r of B index 16 j + c16.
  const int g = lane >> 4, c16 = lane & 15;
  float* out = p.out + (int64_t)slice * p.na * p.nb;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int ia = ta * WA + wm * (WA / 2) + 16 * i + 4 * g;
      const int ib = tb * WB + wn * (WB / 4) + 16 * j + c16;
      if (ia >= p.na || ib >= p.nb) continue;  // both multiples of 16
      *reinterpret_cast<f32x4*>(out + (int64_t)ib * p.na + ia) = sum[i][j];
    }
}

// out = the slices' sum: kG threads per 16-byte column group, each over
// consecutive slices in order, then their results pairwise.  Many slices of a
// small matrix need kG = 8 (128 slices of 128 x 128: 64 threads' worth of
// columns would read them in a chain; the call 20.6 -> 15.2 us).
template <int kG>
__global__ __launch_bounds__(256) void weight_grad_sum_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                              int64_t n4, int slices) {
  constexpr int kCols = 256 / kG;
  __shared__ f32x4 s_sum[256];
  const int c = (int)threadIdx.x % kCols, grp = (int)threadIdx.x / kCols;
  const int64_t i = (int64_t)blockIdx.x * kCols + c;
  const f32x4* src = reinterpret_cast<const f32x4*>(part) + (i < n4 ? i : n4 - 1);
  const int per = (slices + kG - 1) / kG;
  const int end = (grp + 1) * per < slices ? (grp + 1) * per : slices;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  int k = grp * per;
  for (; k + 8 <= end; k += 8) {
    f32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[(int64_t)(k + u) * n4];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < end; ++k) s += src[(int64_t)k * n4];
  if constexpr (kG > 1) {
    s_sum[threadIdx.x] = s;
    __syncthreads();
#pragma unroll
    for (int h = kG / 2; h > 0; h /= 2) {
      if (grp < h) s_sum[threadIdx.x] = s_sum[threadIdx.x] + s_sum[threadIdx.x + h * kCols];
      __syncthreads();
    }
    s = s_sum[threadIdx.x];
  }
  if (grp == 0 && i < n4) reinterpret_cast<f32x4*>(out)[i] = s;
}

// Tiles, x columns by dy columns: as large as two accumulators per output and
// the fragments fit (174 and 195 VGPRs for the first two).
struct WgTile {
  int wa, wb;
};
constexpr WgTile kWgTiles[] = {{128, 256}, {192, 192}, {192, 128}, {128, 192}, {128, 128}};

// The first tile that pads na x nb least.
WgTile wg_tile(int na, int nb) {
  WgTile best = kWgTiles[0];
  int64_t least = INT64_MAX;
  for (const WgTile& t : kWgTiles) {
    const int64_t area = (int64_t)((na + t.wa - 1) / t.wa * t.wa) * ((nb + t.wb - 1) / t.wb * t.wb);
    if (area < least) {
      best = t;
      least = area;
    }
  }
  return best;
}

struct WgPlan {
  int wa, wb, tiles_a, tiles_b, slices;
  int64_t slice_rows;
};

// Slices: as many (tile, slice) pairs as fill the CUs once, or, for slices of
// kWgLong tokens, up to four times where whole tiles would leave more than a
// tenth of them idle (96 tiles of 1024 x 3072: 192 pairs in one round, 480 in two:
// 156672 tokens 1200 -> 1089 us, but 4096 tokens 47 -> 53).
WgPlan wg_plan(int64_t rows, int na, int nb) {
  WgPlan q;
  const WgTile t = wg_tile(na, nb);
  q.wa = t.wa;
  q.wb = t.wb;
  q.tiles_a = (na + q.wa - 1) / q.wa;
  q.tiles_b = (nb + q.wb - 1) / q.wb;
  const int64_t tiles = (int64_t)q.tiles_a * q.tiles_b;
  int64_t s = 1, filled = 0;  // per mille of the CUs over the rounds
  for (int64_t rounds = 1; rounds <= 4 && filled < 900; ++rounds) {
    const int64_t n = kWgCus * rounds / tiles, f = n * tiles * 1000 / (kWgCus * rounds);
    if (n > 0 && f > filled && (rounds == 1 || rows >= n * kWgLong)) {
      s = n;
      filled = f;
    }
  }
  const int64_t most = (rows + kWgMinTokens - 1) / kWgMinTokens;
  if (s > most) s = most;
  q.slice_rows = ((rows + s - 1) / s + kWgTok - 1) / kWgTok * kWgTok;
  q.slices = (int)((rows + q.slice_rows - 1) / q.slice_rows);
  return q;
}

template <int WA, int WB>
int launch_weight_grad(const WgParams& p, hipStream_t s) {
  constexpr int lds = wg_bufs(WA, WB) * kWgTok * (WA + WB) * 2;
  auto kern = weight_grad_kernel<WA, WB>;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return fail(TERRA_ERR_LAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(attr));
  kern<<<8 * p.per_xcd, kWgThreads, lds, s>>>(p);
  return TERRA_OK;
}

int wg_check(int64_t rows, int out_features, int in_features) {
  if (rows < 0 || rows >= (1ll << 31)) return fail(TERRA_ERR_SHAPE, "rows must be in [0, 2^31)");
  if (out_features <= 0 || in_features <= 0 || out_features % 16 != 0 || in_features % 16 != 0 ||
      out_features > (1 << 20) || in_features > (1 << 20))
    return fail(TERRA_ERR_SHAPE, "out_features and in_features must be positive multiples of 16 up to 2^20 (got %d, %d)",
                out_features, in_features);
  return TERRA_OK;
}

}  // namespace
}  // namespace terra

using namespace terra;

extern "C" int terra_swin_weight_grad_slices(int64_t rows, int out_features, int in_features) {
  clear_error();
  if (const int st = wg_check(rows, out_features, in_features); st != TERRA_OK) return st;
  return rows == 0 ? 1 : wg_plan(rows, in_features, out_features).slices;
}

extern "C" int terra_swin_weight_grad(const void* dy, const void* x, float* dw, int dtype, int64_t rows,
                                      int out_features, int in_features, void* workspace, void* stream) {
  clear_error();
  if (dw == nullptr || (rows > 0 && (dy == nullptr || x == nullptr)))
    return fail(TERRA_ERR_NULL, "dy, x and dw must be non-NULL");
  if (dtype_size(dtype) == 0) return fail(TERRA_ERR_DTYPE, "unknown dtype %d", dtype);
  if (dtype != TERRA_DTYPE_BF16) return fail(TERRA_ERR_UNSUPPORTED, "the weight-gradient kernel is bf16 only");
  if (const int st = wg_check(rows, out_features, in_features); st != TERRA_OK) return st;
  for (const void* q : {dy, x, (const void*)dw, (const void*)workspace})
    if (((uintptr_t)q & 15u) != 0) return fail(TERRA_ERR_ALIGN, "dy, x, dw and workspace must be 16-byte aligned");
  if (rows == 0) return fail(TERRA_ERR_SHAPE, "rows must be positive (an empty sum is the caller's zero)");
  const int na = in_features, nb = out_features;
  const WgPlan q = wg_plan(rows, na, nb);
  if (q.slices > 1 && workspace == nullptr)
    return fail(TERRA_ERR_NULL, "a workspace of terra_swin_weight_grad_slices partial results is needed");
  WgParams p;
  memset(&p, 0, sizeof(p));
  p.a = static_cast<const uint8_t*>(x);
  p.b = static_cast<const uint8_t*>(dy);
  p.out = q.slices > 1 ? static_cast<float*>(workspace) : dw;
  p.rows = rows;
  p.slice_rows = q.slice_rows;
  p.na = na;
  p.nb = nb;
  p.tiles_a = q.tiles_a;
  p.tiles_b = q.tiles_b;
  p.tiles = q.tiles_a * q.tiles_b;
  p.slices = q.slices;
  p.per_xcd = (p.tiles * p.slices + 7) / 8;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int st;
  if (q.wb == 256)
    st = launch_weight_grad<128, 256>(p, s);
  else if (q.wb == 192)
    st = q.wa == 192 ? launch_weight_grad<192, 192>(p, s) : launch_weight_grad<128, 192>(p, s);
  else
    st = q.wa == 192 ? launch_weight_grad<192, 128>(p, s) : launch_weight_grad<128, 128>(p, s);
  if (st != TERRA_OK) return st;
  if (q.slices > 1) {
    const int64_t n4 = (int64_t)na * nb / 4;
    const float* part = static_cast<const float*>(workspace);
    if (q.slices >= 16)
      weight_grad_sum_kernel<8><<<(uint32_t)((n4 + 31) / 32), 256, 0, s>>>(part, dw, n4, q.slices);
    else
      weight_grad_sum_kernel<1><<<(uint32_t)((n4 + 255) / 256), 256, 0, s>>>(part, dw, n4, q.slices);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TERRA_ERR_LAUNCH, "terra_swin_weight_grad launch failed: %s", hipGetErrorString(e));
  return TERRA_OK;
}
