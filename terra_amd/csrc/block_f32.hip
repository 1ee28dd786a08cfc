// Fused fp32 Swin attention half-block for gfx950: 7x7 windows, C = 96, 3 heads
// of dim 32 (the small fp32 configuration),
//
//   y = x + reverse(proj(attention(qkv(partition(LayerNorm(x))))))
//
// in one launch, everything in fp32 (models/transformer.py:142-300,
// models/attention.py:236-283).
//
// What bounds it: on small grids (56x56 tokens: 64 windows) the five launches of
// the staged path, 121 us per call of which 37 us ran on the GPU; on large ones
// the fp32 matrix cores (v_mfma_f32_16x16x4_f32, 32 cycles each; 3072 per window)
// and the barriers between phases.  One workgroup of 12 waves per window (a
// persistent loop over windows on large grids, with every weight fragment in
// registers): the window's q, k and V^T stay in LDS (103 KB), the probabilities in
// registers.
//
// MFMA operands: lane (c16, g) holds row (or column) c16 and k-slot g.  Both
// operands of a product take the channels as 16 s + 4 g + e for the e-th of four
// MFMAs, so a lane reads 16 bytes per operand and four MFMAs; the accumulators of
// S^T (keys 16 jt + 4 g + r of query c16) are then the B operand of P V as they are.
#include "attn_core.h"

namespace terra {
namespace {

constexpr int kFC = 96;            // channels
constexpr int kFHeads = 3;
constexpr int kFWs = 7;
constexpr int kFN = kFWs * kFWs;   // 49 tokens, padded to 64
constexpr int kFWaves = 12;        // 3 heads x 4 query tiles
constexpr int kFThreads = 64 * kFWaves;
constexpr int kFPitch = 100;       // floats per token row: 16 rows of 16-byte reads on distinct banks
constexpr int kFVPitch = 68;       // floats per V^T row (64 keys)
constexpr int kFTab = (2 * kFWs - 1) * (2 * kFWs - 1);  // 169

struct BlockF32Params {
  const float* x;
  float* y;                  // may equal x
  const float* gamma;        // [96] or NULL (1)
  const float* beta;         // [96] or NULL (0)
  const float* w_qkv;        // [288][96]
  const float* b_qkv;        // [288] or NULL
  const float* w_proj;       // [96][96]
  const float* b_proj;       // [96] or NULL
  const float* bias_table;   // [169][3] or NULL
  const uint64_t* land_bits; // [land_windows] or NULL
  float* keep_xn;            // kKeep: window tokens [B * nWe, 49, 96], q | k | v
  float* keep_qkv;           // [B * nWe, 49, 288] and attention output [B * nWe, 49,
  float* keep_o;             // 96] for the backward
  int32_t land_windows;
  int32_t layernorm, shift_mask;
  float eps, scale_l2e, mask_l2e;
  int32_t H, W, Hp, Wp, shift_h, shift_w, pad_top, pad_left;
  int32_t nWw, win_row_begin, win_rows, valid_begin, valid_end, nWe;
  int32_t units;             // batch * frame windows
  FastDiv fd_frame, fd_nWw;
};

struct BlockF32Lds {
  float xn[64 * kFPitch];    // LayerNorm rows, then O
  float q[64 * kFPitch];
  float k[64 * kFPitch];
  float vt[kFC * kFVPitch];  // V^T
  float tab[kFHeads * kFTab + 1];  // bias columns (x log2e), head-major
  int off[64];               // per token: bias-index term, region id, grid token (or -1)
  int rid[64];
  int gt[64];
};

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// Two products a b0, a b1 side by side (independent accumulators).
__device__ __forceinline__ void mfma4x2(const f32x4& a, const f32x4 (&b)[2], f32x4 (&c)[2]) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int j = 0; j < 2; ++j) c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[j][e], c[j], 0, 0, 0);
}

// acc += W x^T over 96 channels: one feature tile (fragments w) by two token
// tiles (rows at `row`, 16 rows apart), the next k-step's rows read under the
// current one's MFMAs.
__device__ __forceinline__ void rows_product(const f32x4 (&w)[6], const float* row, f32x4 (&acc)[2]) {
  f32x4 x[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) x[0][j] = ld4(row + 16 * j * kFPitch);
#pragma unroll
  for (int ks = 0; ks < 6; ++ks) {
    if (ks + 1 < 6)
#pragma unroll
      for (int j = 0; j < 2; ++j) x[(ks + 1) & 1][j] = ld4(row + 16 * j * kFPitch + 16 * (ks + 1));
    __builtin_amdgcn_sched_barrier(0);
    mfma4x2(w[ks], x[ks & 1], acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <bool kKeep>
__global__ __launch_bounds__(kFThreads) __attribute__((amdgpu_waves_per_eu(3, 3)))
void block_f32_kernel(const BlockF32Params p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  BlockF32Lds& s = *reinterpret_cast<BlockF32Lds*>(smem);
  const int tid0 = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  const int pft = wave % 6, ptp = wave / 6;  // proj unit: feature tile, token-tile pair
  for (int e = tid0; e < kFHeads * kFTab; e += kFThreads) {
    const int h = e / kFTab, i = e - h * kFTab;
    s.tab[e] = p.bias_table != nullptr ? p.bias_table[i * kFHeads + h] * kLog2e : 0.f;
  }

  for (int unit = (int)blockIdx.x; unit < p.units; unit += (int)gridDim.x) {  // uniform
    // Lane-derived addresses are recomputed per window, not held across the loop.
    int tid = tid0;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, g = lane >> 4, c16 = lane & 15;
    uint32_t b, rest, wr, wc;
    p.fd_frame.divmod((uint32_t)unit, b, rest);
    p.fd_nWw.divmod(rest, wr, wc);
    const int wl = ((int)wr - p.win_row_begin) * p.nWw + (int)wc;
    const bool computed = (unsigned)((int)wr - p.win_row_begin) < (unsigned)p.win_rows &&
                          (p.valid_end <= 0 || (wl >= p.valid_begin && wl < p.valid_end));
    // This wave's q|k|v units u = wave + 12 i (feature tile u % 18, token-tile
    // pair u / 18): weight fragments two units ahead, the first two requested
    // ahead of the rows.
    f32x4 wq[2][6], bq[2];
    auto load_unit = [&](int i) {
      const int ft = (wave + kFWaves * i) % 18;
#pragma unroll
      for (int ks = 0; ks < 6; ++ks) wq[i & 1][ks] = ld4(p.w_qkv + (16 * ft + c16) * kFC + 16 * ks + 4 * g);
      bq[i & 1] = p.b_qkv != nullptr ? ld4(p.b_qkv + 16 * ft + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    if (computed) {  // uniform
      load_unit(0);
      load_unit(1);
    }
    // ---- the window's rows: 8 lanes per token, 12 floats each -----------------
    const int t = tid >> 3, sub = tid & 7;
    int gtok = -1;
    if (t < kFN) {
      const int ti = t / kFWs, tj = t - ti * kFWs;
      int ph = (int)wr * kFWs + ti + p.shift_h, pw = (int)wc * kFWs + tj + p.shift_w;
      if (ph >= p.Hp) ph -= p.Hp;
      if (pw >= p.Wp) pw -= p.Wp;
      const int sh = ph - p.pad_top, sw = pw - p.pad_left;
      if ((unsigned)sh < (unsigned)p.H && (unsigned)sw < (unsigned)p.W) gtok = ((int)b * p.H + sh) * p.W + sw;
    }
    f32x4 v[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
      v[c] = gtok >= 0 ? ld4(p.x + (int64_t)gtok * kFC + 4 * (sub + 8 * c)) : f32x4{0.f, 0.f, 0.f, 0.f};
    if (!computed) {  // not emitted: x passes through
      if (gtok >= 0 && p.y != p.x)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          *reinterpret_cast<f32x4*>(p.y + (int64_t)gtok * kFC + 4 * (sub + 8 * c)) = v[c];
      continue;
    }
    const bool use_shift = p.shift_mask && (((int)wr + 2) * kFWs > p.Hp || ((int)wc + 2) * kFWs > p.Wp);
    const uint64_t land =
        p.land_bits != nullptr ? p.land_bits[((int64_t)b * p.nWe + wl) % p.land_windows] : 0ull;
    const int64_t row0 = ((int64_t)b * p.nWe + wl) * kFN;  // kKeep: the window's first token row
    if (t < 64) {  // waves 0 .. 7
      float sum = 0.f;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum += v[c][e];
      const float mean = group8_sum(sum) * (1.f / kFC);
      float sq = 0.f;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float d = v[c][e] - mean;
          sq += d * d;
        }
      const float rstd = rsqrtf(group8_sum(sq) * (1.f / kFC) + p.eps);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int c0 = 4 * (sub + 8 * c);
        f32x4 o = v[c];
        if (p.layernorm) {
          const f32x4 gm = p.gamma != nullptr ? ld4(p.gamma + c0) : f32x4{1.f, 1.f, 1.f, 1.f};
          const f32x4 bt = p.beta != nullptr ? ld4(p.beta + c0) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (v[c][e] - mean) * rstd * gm[e] + bt[e];
        }
        if (gtok < 0) o = f32x4{0.f, 0.f, 0.f, 0.f};  // frame padding and rows 49 .. 63
        if (kKeep && t < kFN) *reinterpret_cast<f32x4*>(p.keep_xn + (row0 + t) * kFC + c0) = o;
        *reinterpret_cast<f32x4*>(s.xn + t * kFPitch + c0) = o;
      }
      if (sub == 0) {
        const int tc = t < kFN ? t : kFN - 1;
        const int ti = tc / kFWs, tj = tc - ti * kFWs;
        s.off[t] = ti * (2 * kFWs - 1) + tj;
        s.rid[t] = use_shift ? 3 * region((int)wr * kFWs + ti, p.Hp, kFWs, p.shift_h) +
                                   region((int)wc * kFWs + tj, p.Wp, kFWs, p.shift_w)
                             : 0;
        s.gt[t] = gtok;
      }
    }
    __syncthreads();
    // ---- q | k | v ------------------------------------------------------------
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int u = wave + kFWaves * i, ft = u % 18, tp = u / 18;
      f32x4 acc[2] = {bq[i & 1], bq[i & 1]};
      rows_product(wq[i & 1], s.xn + (32 * tp + c16) * kFPitch + 4 * g, acc);
      if (i == 0) load_unit(2);
      const int part = ft / 6, f = (ft - 6 * part) * 16 + 4 * g;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int tok = 16 * (2 * tp + j) + c16;
        if (kKeep && tok < kFN)
          *reinterpret_cast<f32x4*>(p.keep_qkv + (row0 + tok) * (3 * kFC) + 16 * ft + 4 * g) = acc[j];
        if (part == 2) {  // uniform
#pragma unroll
          for (int r = 0; r < 4; ++r) s.vt[(f + r) * kFVPitch + tok] = acc[j][r];
        } else {
          *reinterpret_cast<f32x4*>((part == 0 ? s.q : s.k) + tok * kFPitch + f) = acc[j];
        }
      }
    }
    __syncthreads();
    // The proj unit's weights, requested ahead of the attention.
    f32x4 wp[6];
#pragma unroll
    for (int ks = 0; ks < 6; ++ks) wp[ks] = ld4(p.w_proj + (16 * pft + c16) * kFC + 16 * ks + 4 * g);
    const f32x4 bp = p.b_proj != nullptr ? ld4(p.b_proj + 16 * pft + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
    // ---- attention: head wave / 4, query tile wave % 4 -------------------------
    {
      const int h = wave >> 2, it = wave & 3;
      f32x4 st[4];
      f32x4 qf[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) qf[c] = ld4(s.q + (16 * it + c16) * kFPitch + 32 * h + 16 * c + 4 * g);
      {
        f32x4 kf[4][2];
#pragma unroll
        for (int jt = 0; jt < 4; ++jt)
#pragma unroll
          for (int c = 0; c < 2; ++c) kf[jt][c] = ld4(s.k + (16 * jt + c16) * kFPitch + 32 * h + 16 * c + 4 * g);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) st[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int jt = 0; jt < 4; ++jt)
              st[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[jt][c][e], qf[c][e], st[jt], 0, 0, 0);
      }
      const int i = 16 * it + c16;
      const float* tab = s.tab + h * kFTab + (kFWs - 1) * (2 * kFWs - 1) + kFWs - 1 + s.off[i];
      const int rid = s.rid[i];
      float mx = -INFINITY;
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {
        const int4 off = *reinterpret_cast<const int4*>(s.off + 16 * jt + 4 * g);
        const int o[4] = {off.x, off.y, off.z, off.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) st[jt][r] = __builtin_fmaf(st[jt][r], p.scale_l2e, tab[-o[r]]);
        if (use_shift || land != 0ull) {  // uniform
          const int4 rj = *reinterpret_cast<const int4*>(s.rid + 16 * jt + 4 * g);
          const int rr[4] = {rj.x, rj.y, rj.z, rj.w};
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool land_j = (land >> (16 * jt + 4 * g + r)) & 1ull;
            st[jt][r] += (rr[r] != rid ? p.mask_l2e : 0.f) + (land_j ? p.mask_l2e : 0.f);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (16 * jt + 4 * g + r >= kFN) st[jt][r] = -INFINITY;
          mx = max_nan(mx, st[jt][r]);
        }
      }
      mx = xor_max(mx);
      float sum = 0.f;
#pragma unroll
      for (int jt = 0; jt < 4; ++jt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          st[jt][r] = __builtin_amdgcn_exp2f(st[jt][r] - mx);
          sum += st[jt][r];
        }
      const float inv = __builtin_amdgcn_rcpf(xor_sum(sum));
      f32x4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {
        f32x4 vf[2];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) vf[ct] = ld4(s.vt + (32 * h + 16 * ct + c16) * kFVPitch + 16 * jt + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int ct = 0; ct < 2; ++ct)
            o[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[ct][e], st[jt][e], o[ct], 0, 0, 0);
      }
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const f32x4 v = o[ct] * inv;
        *reinterpret_cast<f32x4*>(s.xn + i * kFPitch + 32 * h + 16 * ct + 4 * g) = v;
        if (kKeep && i < kFN) *reinterpret_cast<f32x4*>(p.keep_o + (row0 + i) * kFC + 32 * h + 16 * ct + 4 * g) = v;
      }
    }
    __syncthreads();
    // ---- proj + residual ------------------------------------------------------
    {
      f32x4 acc[2] = {bp, bp};
      int gt[2];
      f32x4 xr[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        gt[j] = s.gt[16 * (2 * ptp + j) + c16];
        xr[j] = gt[j] >= 0 ? ld4(p.x + (int64_t)gt[j] * kFC + 16 * pft + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
      rows_product(wp, s.xn + (32 * ptp + c16) * kFPitch + 4 * g, acc);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (gt[j] >= 0) *reinterpret_cast<f32x4*>(p.y + (int64_t)gt[j] * kFC + 16 * pft + 4 * g) = xr[j] + acc[j];
    }
    __syncthreads();  // O and the token terms are read out before the next window
  }
}

template <bool kKeep>
int launch_block_f32(const BlockF32Params& p, hipStream_t s) {
  constexpr int lds = (int)sizeof(BlockF32Lds);
  static_assert(lds <= 160 * 1024, "LDS");
  auto kern = block_f32_kernel<kKeep>;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return fail(TERRA_ERR_LAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(attr));
  constexpr int kCus = 256;  // one workgroup per CU
  kern<<<p.units < kCus ? p.units : kCus, kFThreads, lds, s>>>(p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TERRA_ERR_LAUNCH, "fp32 block kernel launch failed: %s", hipGetErrorString(e));
  return TERRA_OK;
}

// keep: the training entry's three outputs, or NULL.
int block_f32(const float* x, float* y, float* const* keep, const terra_swin_block_desc* desc, const float* ln_gamma,
              const float* ln_beta, const float* qkv_weight, const float* qkv_bias, const float* proj_weight,
              const float* proj_bias, const float* bias_table, const uint64_t* land_bits, void* stream) {
  if (desc == nullptr) return fail(TERRA_ERR_NULL, "desc is NULL");
  if (x == nullptr || y == nullptr || qkv_weight == nullptr || proj_weight == nullptr)
    return fail(TERRA_ERR_NULL, "x, y, qkv_weight and proj_weight must be non-NULL");
  const terra_swin_block_desc& d = *desc;
  GeomDims dims;
  const int st = validate_geom(&d.geom, &dims);
  if (st != TERRA_OK) return st;
  const terra_swin_geom& q = d.geom;
  if (q.window != kFWs || d.heads != kFHeads || q.channels != kFC)
    return fail(TERRA_ERR_UNSUPPORTED, "the fp32 block kernel needs 7x7 windows, 96 channels and 3 heads (got %d, %d, %d)",
                q.window, q.channels, d.heads);
  if (d.packed_weights != 0) return fail(TERRA_ERR_UNSUPPORTED, "the fp32 block kernel takes plain row-major weights");
  if (d.layernorm != 0 && !(d.ln_eps >= 0.f)) return fail(TERRA_ERR_SHAPE, "ln_eps must be a non-negative number");
  if (land_bits != nullptr &&
      (d.land_windows <= 0 || ((int64_t)q.batch * dims.nWe) % d.land_windows != 0 || d.land_windows % dims.nWe != 0))
    return fail(TERRA_ERR_SHAPE,
                "land_windows (%d) must be a multiple of the emitted windows per image (%lld) dividing the batch's "
                "(%lld)", d.land_windows, (long long)dims.nWe, (long long)((int64_t)q.batch * dims.nWe));
  for (const void* ptr : {(const void*)x, (const void*)y, (const void*)qkv_weight, (const void*)proj_weight,
                          (const void*)ln_gamma, (const void*)ln_beta, (const void*)qkv_bias, (const void*)proj_bias})
    if (((uintptr_t)ptr & 15u) != 0) return fail(TERRA_ERR_ALIGN, "tensors must be 16-byte aligned");
  if (((uintptr_t)bias_table & 3u) != 0 || ((uintptr_t)land_bits & 7u) != 0)
    return fail(TERRA_ERR_ALIGN, "bias_table / land_bits misaligned");
  const int64_t tokens = (int64_t)q.batch * q.height * q.width;
  const int64_t frame_windows = dims.nWh * dims.nWw;
  const int64_t units = (int64_t)q.batch * frame_windows;
  if (units >= (1ll << 31) || tokens >= (1ll << 31) || (int64_t)q.batch * dims.nWe >= (1ll << 31))
    return fail(TERRA_ERR_SHAPE, "grid too large for one launch; split the batch");
  const uintptr_t xa = (uintptr_t)x, ya = (uintptr_t)y, bytes = (uintptr_t)(tokens * kFC * 4);
  if (x != y && xa < ya + bytes && ya < xa + bytes) return fail(TERRA_ERR_SHAPE, "y overlaps x without being x");
  BlockF32Params p;
  memset(&p, 0, sizeof(p));
  p.x = x;
  p.y = y;
  p.gamma = ln_gamma;
  p.beta = ln_beta;
  p.w_qkv = qkv_weight;
  p.b_qkv = qkv_bias;
  p.w_proj = proj_weight;
  p.b_proj = proj_bias;
  p.bias_table = bias_table;
  p.land_bits = land_bits;
  p.land_windows = land_bits != nullptr ? d.land_windows : 1;
  p.layernorm = d.layernorm != 0;
  p.shift_mask = d.shift_mask != 0;
  p.eps = d.ln_eps;
  p.scale_l2e = d.scale * kLog2e;
  p.mask_l2e = d.mask_value * kLog2e;
  p.H = q.height;
  p.W = q.width;
  p.Hp = (int32_t)dims.Hp;
  p.Wp = (int32_t)dims.Wp;
  p.shift_h = q.shift_h;
  p.shift_w = q.shift_w;
  p.pad_top = q.pad_top;
  p.pad_left = q.pad_left;
  p.nWw = (int32_t)dims.nWw;
  p.win_row_begin = q.win_row_begin;
  p.win_rows = (int32_t)dims.rows;
  p.valid_begin = q.valid_end > 0 ? q.valid_begin : 0;
  p.valid_end = q.valid_end > 0 ? q.valid_end : 0;
  p.nWe = (int32_t)dims.nWe;
  p.units = (int32_t)units;
  p.fd_frame = FastDiv((uint32_t)frame_windows);
  p.fd_nWw = FastDiv((uint32_t)dims.nWw);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (keep == nullptr) return launch_block_f32<false>(p, s);
  // A pad window's rows belong to the kept tensors but are not computed here.
  if (p.valid_end > 0) return fail(TERRA_ERR_UNSUPPORTED, "the training form needs every emitted window valid");
  for (int i = 0; i < 3; ++i) {
    if (keep[i] == nullptr) return fail(TERRA_ERR_NULL, "the kept tensors must be non-NULL");
    if (((uintptr_t)keep[i] & 15u) != 0) return fail(TERRA_ERR_ALIGN, "tensors must be 16-byte aligned");
  }
  p.keep_xn = keep[0];
  p.keep_qkv = keep[1];
  p.keep_o = keep[2];
  return launch_block_f32<true>(p, s);
}

}  // namespace
}  // namespace terra

using namespace terra;

extern "C" int terra_swin_block_f32_fwd(const float* x, float* y, const terra_swin_block_desc* desc,
                                        const float* ln_gamma, const float* ln_beta, const float* qkv_weight,
                                        const float* qkv_bias, const float* proj_weight, const float* proj_bias,
                                        const float* bias_table, const uint64_t* land_bits, void* stream) {
  clear_error();
  return block_f32(x, y, nullptr, desc, ln_gamma, ln_beta, qkv_weight, qkv_bias, proj_weight, proj_bias, bias_table,
                   land_bits, stream);
}

extern "C" int terra_swin_block_f32_train(const float* x, float* y, float* windows, float* qkv, float* o,
                                          const terra_swin_block_desc* desc, const float* ln_gamma,
                                          const float* ln_beta, const float* qkv_weight, const float* qkv_bias,
                                          const float* proj_weight, const float* proj_bias, const float* bias_table,
                                          const uint64_t* land_bits, void* stream) {
  clear_error();
  float* const keep[3] = {windows, qkv, o};
  return block_f32(x, y, keep, desc, ln_gamma, ln_beta, qkv_weight, qkv_bias, proj_weight, proj_bias, bias_table,
                   land_bits, stream);
}
