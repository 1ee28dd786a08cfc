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
// four buffers, and reads MFMA fragments by transposed LDS reads
// (ds_read_b64_tr_b16: four tokens of one column per lane), so nothing is
// transposed through memory.  x is the A operand, so a lane's four accumulator
// rows are consecutive in dW; eight waves, 2 x 4, each WA / 2 x WB / 4 of the
// tile.
//
// What bounds it: for narrow layers (C = 192) HBM, every operand row being read
// once (the output tiles of a slice share an XCD's L2); for wide ones (C =
// 1024) the matrix cores and the power limit.  A stage's fragments are read
// while the one before is multiplied, each right after its registers' last use,
// in pinned order, and the loads run as many stages ahead as the LDS holds.
#include "common.h"
#include "attn_core.h"

namespace terra {
namespace {

constexpr int kWgThreads = 512;
constexpr int kWgTok = 32;     // tokens per stage (one MFMA k-step)
constexpr int kWgCus = 256;    // one workgroup per CU
constexpr int kWgMinTokens = 512;  // per slice: below this its fixed cost outweighs the split

struct WgParams {
  const uint8_t* a;   // x:  [rows] x na bf16
  const uint8_t* b;   // dy: [rows] x nb bf16
  float* out;         // [nb][na]; slice s at out + s * na * nb
  int64_t rows;
  int64_t slice_rows; // a multiple of kWgTok
  int32_t na, nb;
  int32_t tiles_b, tiles, slices;
  int32_t per_xcd;    // workgroups per XCD
};

// LDS buffers of a tile: as many stages as fit (5 for 256 x 256), at most 8.
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
  const int ta = tile / p.tiles_b, tb = tile - ta * p.tiles_b;
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

  f32x4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
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
  }

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
      *reinterpret_cast<f32x4*>(out + (int64_t)ib * p.na + ia) = acc[i][j];
    }
}

// out = the slices' sum, in slice order.
__global__ __launch_bounds__(256) void weight_grad_sum_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                              int64_t n4, int slices) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const f32x4* src = reinterpret_cast<const f32x4*>(part) + i;
  f32x4 s = src[0];
  int k = 1;
  for (; k + 8 <= slices; k += 8) {
    f32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[(int64_t)(k + u) * n4];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < slices; ++k) s += src[(int64_t)k * n4];
  reinterpret_cast<f32x4*>(out)[i] = s;
}

// Tile width for n columns: the widest of 256, 192, 128 whose padding is least.
int wg_width(int n) {
  int best = 256, waste = (n + 255) / 256 * 256 - n;
  for (int w : {192, 128}) {
    const int u = (n + w - 1) / w * w - n;
    if (u < waste) {
      best = w;
      waste = u;
    }
  }
  return best;
}

struct WgPlan {
  int wa, wb, tiles_a, tiles_b, slices;
  int64_t slice_rows;
};

// Slices: as many as give each CU one (tile, slice) pair.
WgPlan wg_plan(int64_t rows, int na, int nb) {
  WgPlan q;
  q.wa = wg_width(na);
  q.wb = wg_width(nb);
  q.tiles_a = (na + q.wa - 1) / q.wa;
  q.tiles_b = (nb + q.wb - 1) / q.wb;
  const int tiles = q.tiles_a * q.tiles_b;
  int64_t s = kWgCus / tiles;
  const int64_t most = (rows + kWgMinTokens - 1) / kWgMinTokens;
  if (s > most) s = most;
  if (s < 1) s = 1;
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

template <int WA>
int dispatch_weight_grad(const WgParams& p, int wb, hipStream_t s) {
  return wb == 256 ? launch_weight_grad<WA, 256>(p, s)
                   : wb == 192 ? launch_weight_grad<WA, 192>(p, s) : launch_weight_grad<WA, 128>(p, s);
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
  p.tiles_b = q.tiles_b;
  p.tiles = q.tiles_a * q.tiles_b;
  p.slices = q.slices;
  p.per_xcd = (p.tiles * p.slices + 7) / 8;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int st = q.wa == 256 ? dispatch_weight_grad<256>(p, q.wb, s)
                             : q.wa == 192 ? dispatch_weight_grad<192>(p, q.wb, s) : dispatch_weight_grad<128>(p, q.wb, s);
  if (st != TERRA_OK) return st;
  if (q.slices > 1) {
    const int64_t n4 = (int64_t)na * nb / 4;
    weight_grad_sum_kernel<<<(uint32_t)((n4 + 255) / 256), 256, 0, s>>>(static_cast<const float*>(workspace), dw, n4,
                                                                       q.slices);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TERRA_ERR_LAUNCH, "terra_swin_weight_grad launch failed: %s", hipGetErrorString(e));
  return TERRA_OK;
}
