// Token-row linear layers with few input features for gfx950 (bf16): the
// narrow blocks' q|k|v, proj and fc1 in the training step and proj's input
// gradient,
//
//   acc[m][f] = b[f] + sum_k x[m][k] W[f][k]      K = 128 or 192, fp32 on MFMA
//
//   store      y[m] = bf16(acc)
//   gelu-keep  h[m] = bf16(acc), y[m] = GELU(h[m])
//
// What bounds it: HBM (a row of 192 inputs gives 768 outputs: 4 bytes written
// per byte read, 100 flop per byte).  The 256 x 256 tiles of the other linear
// kernel spend most of such a layer in their epilogue, where nothing else runs.  Here the weights stay in registers
// (a wave owns 32 output features, 2 x K / 32 fragments) and the token rows
// stream: 64-row tiles arrive in LDS by bounded buffer loads one tile ahead,
// every wave multiplies all of them and writes its own 64 bytes per row, and
// several workgroups per CU drift apart so that one's stores overlap another's
// MFMAs and loads.  One barrier per tile; a tile's stores are not waited for
// until the tile after next.  Stores carry nt and sc1: 64-byte halves of a line
// from two waves (gelu-keep 320 us, against 400-530 with nt alone, 440 with
// sc1, 430 plain).  524288 rows, us, before (other linear kernel or hipBLASLt)
// -> here: 192 -> 768 gelu-keep 499 -> 325 (1.8 GB at 5.6 TB/s), 192 -> 768
// 245 -> 205, 192 -> 576 300 -> 130, 192 -> 192 113 -> 60.
#include "common.h"
#include "attn_core.h"
#include "gelu.h"

namespace terra {
namespace {

constexpr int kShTok = 64;  // token rows per tile

enum { kShStore = 0, kShGeluKeep = 1 };

struct ShortParams {
  const uint8_t* x;       // [M] x K bf16
  const uint8_t* w;       // packed [N, K] bf16
  const float* bias;      // [N] or NULL
  uint8_t* y;             // [M] x N bf16
  uint8_t* keep;          // kShGeluKeep: [M] x N bf16
  int32_t M, N, tiles;
  int32_t blocks_n;       // N / (32 W)
  int32_t streams;        // token-tile streams: stream s takes tiles s, s + streams, ...
};

// LDS: two tiles of token rows, then the GELU table.
template <int KS>
constexpr int sh_tile_bytes() {
  return kShTok * KS * 64;
}
template <int KS, int kEpi>
constexpr int sh_lds_bytes() {
  return 2 * sh_tile_bytes<KS>() + (kEpi == kShGeluKeep ? kGeluBytes : 0);
}

// Chunk position of (row, 16-byte chunk) in a tile: 384-byte rows put odd rows
// half a bank period off and XOR pairs of rows within groups of 8 chunks;
// 256-byte rows XOR all 16.  The 16 rows of a fragment read hit distinct banks.
template <int KS>
__device__ __forceinline__ int sh_swz(int row) {
  return KS == 6 ? (row >> 1) & 7 : row & 15;
}

template <int KS, int W, int kEpi>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W / 2, W / 2)))
void linear_short_kernel(const ShortParams p) {
  constexpr int kThreads = 64 * W;
  constexpr int kChunks = KS * 4;                        // 16-byte chunks per row
  constexpr int kPitch = KS * 64;
  constexpr int kBlks = sh_tile_bytes<KS>() / 1024;      // 1 KB loads per tile
  constexpr int kPer = (kBlks + W - 1) / W, kRem = kBlks % W;
  constexpr int kStores = kEpi == kShGeluKeep ? 8 : 4;   // per wave and tile
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, g = lane >> 4, c16 = lane & 15;
  uint8_t* s_table = smem + 2 * sh_tile_bytes<KS>();
  if constexpr (kEpi == kShGeluKeep) gelu_table_fill(reinterpret_cast<uint16_t*>(s_table), tid, kThreads);

  // Workgroup b on XCD b % 8: the feature blocks of one stream of token tiles
  // are neighbours on one XCD, so the tiles are read from HBM once.
  const int q0 = (int)blockIdx.x >> 3;
  const int fb = q0 % p.blocks_n;
  const int stream = (q0 / p.blocks_n) * 8 + ((int)blockIdx.x & 7);
  if (stream >= p.streams) return;  // uniform
  const int f0 = (fb * W + wave) * 32;  // this wave's first feature

  // Weights: row c16 of A tile i is feature 8 (c16 >> 2) + 4 i + (c16 & 3) of
  // the wave's 32, so that an accumulator lane holds 8 consecutive features.
  uint4 wf[KS][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      wf[ks][i] = *reinterpret_cast<const uint4*>(
          p.w + ((int64_t)(f0 / 16 + (c16 >> 3)) * KS + ks) * 1024 +
          (8 * ((c16 >> 2) & 1) + 4 * i + (c16 & 3) + 16 * g) * 16);
  f32x4 bias[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    bias[i] = p.bias != nullptr ? *reinterpret_cast<const f32x4*>(p.bias + f0 + 8 * g + 4 * i) : f32x4{0.f, 0.f, 0.f, 0.f};

  uint32_t voff[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int slot = (wave + W * q) * 64 + lane;
    const int row = slot / kChunks, c = slot - row * kChunks;
    voff[q] = (uint32_t)(row * kPitch + (c ^ sh_swz<KS>(row)) * 16);
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(smem));
  auto fetch = [&](int t, int buf) {
    const int rows = p.M - t * kShTok < kShTok ? p.M - t * kShTok : kShTok;
    const __amdgpu_buffer_rsrc_t r = buffer_rsrc(p.x + (int64_t)t * kShTok * kPitch, (uint32_t)(rows * kPitch));
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      if (kRem != 0 && q == kPer - 1 && wave >= kRem) break;  // uniform
      dma_buffer_to_lds16(r, voff[q], lds0 + buf * sh_tile_bytes<KS>() + (wave + W * q) * 1024);
    }
  };
  const int out_pitch = p.N * 2;
  const uint32_t ooff = (uint32_t)(c16 * out_pitch + (f0 + 8 * g) * 2);  // + 16 tt rows
  auto rows_rsrc = [&](const uint8_t* base, int t) {
    const int rows = p.M - t * kShTok < kShTok ? p.M - t * kShTok : kShTok;
    return buffer_rsrc(base + (int64_t)t * kShTok * out_pitch, (uint32_t)(rows * out_pitch));
  };
  uint32_t xaddr[2];  // fragment of row 16 tt + c16, chunk 4 ks + g
#pragma unroll
  for (int q = 0; q < 2; ++q)
    xaddr[q] = KS == 6 ? (uint32_t)(c16 * kPitch + ((4 * q + g) ^ sh_swz<KS>(c16)) * 16) : 0u;
  auto frag = [&](int buf, int ks, int tt) {
    const uint8_t* b = smem + buf * sh_tile_bytes<KS>() + tt * 16 * kPitch;
    if constexpr (KS == 6)
      return *reinterpret_cast<const uint4*>(b + xaddr[ks & 1] + (ks >> 1) * 128);
    else
      return *reinterpret_cast<const uint4*>(b + c16 * kPitch + ((4 * ks + g) ^ c16) * 16);
  };

  int t = stream, buf = 0;
  if (t < p.tiles) fetch(t, 0);
  bool first = true;
  for (; t < p.tiles; t += p.streams, buf ^= 1) {  // uniform
    // The tile's rows have landed; only the previous tile's stores,
    // issued after them, may be open.
    if (first)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStores) : "memory");
    first = false;
    lds_barrier();  // every wave's loads are in; every wave has read the other buffer out
    const int next = t + p.streams;
    if (next < p.tiles) fetch(next, buf ^ 1);  // uniform
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) acc[i][tt] = bias[i];
    // A fragment is reloaded for the next k-step right after its last use.
    uint4 xf[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) xf[tt] = frag(buf, 0, tt);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[ks][i]),
                                                               __builtin_bit_cast(bf16x8, xf[tt]), acc[i][tt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (ks + 1 < KS) xf[tt] = frag(buf, ks + 1, tt);
        __builtin_amdgcn_sched_barrier(0);
      }
    // Lane (c16, g): features f0 + 8 g .. + 7 of token rows 16 tt + c16.  Rows
    // past the end fall outside the descriptors.
    const __amdgpu_buffer_rsrc_t yr = rows_rsrc(p.y, t);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x4& c = acc[e >> 1][tt];
        o[e] = pack_bf16x2(c[2 * (e & 1)], c[2 * (e & 1) + 1]);
      }
      const uint32_t off = ooff + 16 * tt * out_pitch;
      if constexpr (kEpi == kShGeluKeep) {
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{o[0], o[1], o[2], o[3]}, rows_rsrc(p.keep, t), off, 0, kCacheNt | kCacheSc1);
        gelu_chunk(o, reinterpret_cast<const uint16_t*>(s_table));
      }
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{o[0], o[1], o[2], o[3]}, yr, off, 0, kCacheNt | kCacheSc1);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int KS, int W, int kEpi>
int launch_short(ShortParams p, hipStream_t s) {
  constexpr int lds = sh_lds_bytes<KS, kEpi>();
  auto kern = linear_short_kernel<KS, W, kEpi>;
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
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 64 * W, lds) != hipSuccess)
      return fail(TERRA_ERR_LAUNCH, "cannot size the linear kernel grid for this device");
    cache[dev] = cus * (per_cu > 0 ? per_cu : 1);
  }
  p.tiles = (p.M + kShTok - 1) / kShTok;
  p.blocks_n = p.N / (32 * W);
  // Whole streams per XCD (a stream's feature blocks together), at most one per tile.
  const int per_xcd = cache[dev] / 8 / p.blocks_n;
  p.streams = 8 * (per_xcd > 0 ? per_xcd : 1);
  if (p.streams > p.tiles) p.streams = p.tiles;
  const int grid = (p.streams + 7) / 8 * 8 * p.blocks_n;
  kern<<<grid, 64 * W, lds, s>>>(p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TERRA_ERR_LAUNCH, "linear kernel launch failed: %s", hipGetErrorString(e));
  return TERRA_OK;
}

// Waves: a block of 192 features where they divide the outputs, else of 128
// (128 inputs: 512; 192 inputs: an MLP of 512 or 1024 hidden features, say).
template <int kEpi>
int dispatch_short(const ShortParams& p, int k, hipStream_t s) {
  if (k == 192) return p.N % 192 == 0 ? launch_short<6, 6, kEpi>(p, s) : launch_short<6, 4, kEpi>(p, s);
  return p.N % 192 == 0 ? launch_short<4, 6, kEpi>(p, s) : launch_short<4, 4, kEpi>(p, s);
}

bool sh_overlap(const void* a, int64_t abytes, const void* b, int64_t bbytes) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return x < y + (uintptr_t)bbytes && y < x + (uintptr_t)abytes;
}

}  // namespace
}  // namespace terra

using namespace terra;

extern "C" int terra_swin_linear_short(const void* x, void* y, void* keep, int dtype, int64_t rows,
                                       int in_features, int out_features, const void* weight_packed,
                                       const float* bias, int epilogue, void* stream) {
  clear_error();
  if (x == nullptr || weight_packed == nullptr || y == nullptr)
    return fail(TERRA_ERR_NULL, "x, weight and y must be non-NULL");
  if (dtype_size(dtype) == 0) return fail(TERRA_ERR_DTYPE, "unknown dtype %d", dtype);
  if (dtype != TERRA_DTYPE_BF16) return fail(TERRA_ERR_UNSUPPORTED, "the linear kernels are bf16 only");
  if (epilogue < TERRA_SHORT_STORE || epilogue > TERRA_SHORT_GELU_KEEP)
    return fail(TERRA_ERR_SHAPE, "unknown epilogue %d", epilogue);
  if ((epilogue == TERRA_SHORT_GELU_KEEP) != (keep != nullptr))
    return fail(TERRA_ERR_NULL, "keep belongs to the gelu-keep epilogue");
  if (rows < 0 || rows >= (1ll << 31) - kShTok) return fail(TERRA_ERR_SHAPE, "rows must be in [0, 2^31 - 64)");
  if ((in_features != 128 && in_features != 192) || out_features <= 0 ||
      (out_features % 192 != 0 && out_features % 128 != 0) || out_features > 4096)
    return fail(TERRA_ERR_SHAPE,
                "in_features must be 128 or 192 and out_features a multiple of 128 or 192 up to 4096 (got %d, %d)",
                in_features, out_features);
  for (const void* q : {x, (const void*)y, (const void*)keep, weight_packed, (const void*)bias})
    if (((uintptr_t)q & 15u) != 0) return fail(TERRA_ERR_ALIGN, "tensors must be 16-byte aligned");
  const int64_t xb = rows * (int64_t)in_features * 2, yb = rows * (int64_t)out_features * 2;
  if (rows > 0 && (sh_overlap(x, xb, y, yb) ||
                   (keep != nullptr && (sh_overlap(x, xb, keep, yb) || sh_overlap(keep, yb, y, yb)))))
    return fail(TERRA_ERR_SHAPE, "outputs must not overlap the inputs or each other");
  if (rows == 0) return TERRA_OK;
  ShortParams p;
  memset(&p, 0, sizeof(p));
  p.x = static_cast<const uint8_t*>(x);
  p.w = static_cast<const uint8_t*>(weight_packed);
  p.bias = bias;
  p.y = static_cast<uint8_t*>(y);
  p.keep = static_cast<uint8_t*>(keep);
  p.M = (int32_t)rows;
  p.N = out_features;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return epilogue == TERRA_SHORT_GELU_KEEP ? dispatch_short<kShGeluKeep>(p, in_features, s)
                                           : dispatch_short<kShStore>(p, in_features, s);
}
