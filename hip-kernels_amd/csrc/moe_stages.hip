// moe_stages.hip -- single-stage kernels of the MoE block (gfx950).
//
// The fused decode path (moe_route.hip, moe_experts.hip) does not need these;
// they are the C-ABI replacements of the reference's individual launchers,
// with the same arithmetic as the fused kernels so every stage can be checked
// on its own:
//   dense MXFP4 GEMV   fused_mxfp4_gemv_forward   (fused_mxfp4_gemv.cu:452-464)
//   SwiGLU             swiglu_forward             (swiglu.cu:178-211)
//   combine            moe_combine_forward        (moe_combine.cu:175-204)
//   scatter            moe_scatter_tokens         (moe_permute.cu:241-259)
//   dequant            mxfp4_dequant_batched      (mxfp4_dequant.cu:353-375)
//   RMSNorm            rmsnorm_forward            (rmsnorm.cu:47-83), used by
//                      the layer's forward() entry.
#include "moe_device.h"
#include "moe_kernels.h"
#include "moe_stages.h"

namespace gxmoe {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Dense MXFP4 GEMV: grid (N/64 tiles, ceil(M / TC)), 64 parts threads.  Lane =
// row of the tile, wave = K-part; same canonical dot as the fused expert
// kernels: one ascending fmaf chain per (row, token) over the part, the part
// sums added in part order, + bias.
//
// Bound by the chains (a part is 480 dependent fmaf at K = 2880) and the
// issue of its loads.  A block of weights is one coalesced 16-byte load per
// lane, put in row order by four lane swaps (four dword loads per block, each
// over the same KiB, and a byte load per scale made a second work-group on a
// CU double its time).  The token values are the same for every lane, so they
// come through the scalar cache into scalar registers, a block of a row in one
// 64-byte load, and each fmaf takes one as its scalar operand (as LDS
// broadcasts, 16 bytes per four fmaf, they ran at the LDS rate).  The block
// loop is kept rolled: unrolled over the part it waits for instructions.  Rows
// that start between two dwords (kShift; x then points to element 1, so that
// every part of a scalar load's address is on four bytes) take the 30 elements
// of a block that whole dwords hold the same way and the two others from one
// load per lane ahead of the loop (element by element through vector loads,
// each of which waits for the weights in flight: N = 201088, M = 1: 605 us).
// Measured, N = 5760, K = 2880, M = 1 / 5 / 16 / 64: 20.5 / 48 / 70 / 115 us
// before, 8.1 / 13.1 / 21 / 62 now.
template <int TC, bool kShift>
__global__ __launch_bounds__(kTileRows * kMaxParts) void dense_gemv_kernel(
    const uint16_t* __restrict__ x, int M, const uint8_t* __restrict__ wn, const uint8_t* __restrict__ ws,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ y, TiledGeom g) {
  constexpr int kD = 4;  // weight blocks in flight (a dword of scale codes)
  __shared__ float s_part[kMaxParts][TC][kTileRows];
  const int tile = blockIdx.x;
  const int m0 = blockIdx.y * TC;
  const int mc = min(TC, M - m0);
  const int p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int K = g.K, bpp = g.bpp;
  const u32x4* src =
      reinterpret_cast<const u32x4*>(wn + (static_cast<size_t>(tile) * g.nb + static_cast<size_t>(p) * bpp) * 1024) + lane;
  const uint8_t* sc = ws + (static_cast<size_t>(tile) * g.parts + p) * kTileRows * g.spad +
                      static_cast<size_t>(lane) * g.spad;
  uint32_t codes[4];  // the part's scale codes, at most 16
  if ((reinterpret_cast<uintptr_t>(ws) & 3u) == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) codes[q] = reinterpret_cast<const uint32_t*>(sc)[min(q, (g.spad >> 2) - 1)];
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      codes[q] = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) codes[q] |= static_cast<uint32_t>(sc[min(4 * q + r, g.spad - 1)]) << (8 * r);
    }
  }
  u32x4 wv[kD];
#pragma unroll
  for (int u = 0; u < kD; ++u) wv[u] = src[static_cast<size_t>(min(u, bpp - 1)) * 64];
  const uint16_t* xr[TC];  // rows past M: the last row, their sums are not stored
#pragma unroll
  for (int m = 0; m < TC; ++m) xr[m] = x + static_cast<size_t>(m0 + min(m, mc - 1)) * K + p * bpp * 32;
  // kShift: lane 2 i holds each row's first element of block i, lane 2 i + 1
  // its last (the block's other 30 lie in whole dwords)
  float edge[kShift ? TC : 1];
  if constexpr (kShift) {
#pragma unroll
    for (int m = 0; m < TC; ++m) edge[m] = bf16_to_f32(xr[m][32 * min(lane >> 1, bpp - 1) + 31 * (lane & 1) - 1]);
  }
  auto edge_of = [&](int m, int l) -> float {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(edge[m]), l));
  };
  float acc[TC];
#pragma unroll
  for (int m = 0; m < TC; ++m) acc[m] = 0.0f;
#pragma clang loop unroll(disable)
  for (int i0 = 0; i0 < bpp; i0 += kD) {
#pragma unroll
    for (int u = 0; u < kD; ++u) {
      const int i = i0 + u;
      if (i < bpp) {
        float wf[32];
        const uint32_t code = (codes[0] >> (8 * (i & 3))) & 0xffu;
        const bool sp = (code - 1u) >= 254u;  // a scale code 0 or 255
        const float scale = e8m0_to_f32(code);
        const u32x4 wr = slot_to_row(wv[u]);
#pragma unroll
        for (int d = 0; d < 4; ++d) decode8_regular(wr[d], sp ? 1.0f : scale, wf + 8 * d);
        if (__ballot(sp) != 0ull) {
#pragma unroll
          for (int c = 0; c < 32; ++c) wf[c] = sp ? wf[c] * scale : wf[c];
        }
        wv[u] = src[static_cast<size_t>(min(i + kD, bpp - 1)) * 64];
        // the rows' chains side by side, a dword of two elements at a time
        constexpr int kDw = kShift ? 15 : 16;
        uint32_t xv[TC][kDw];
#pragma unroll
        for (int m = 0; m < TC; ++m)
#pragma unroll
          for (int c = 0; c < kDw; ++c) xv[m][c] = reinterpret_cast<const uint32_t*>(xr[m] + 32 * i)[c];
        if constexpr (kShift) {
#pragma unroll
          for (int m = 0; m < TC; ++m) acc[m] = __builtin_fmaf(edge_of(m, 2 * i), wf[0], acc[m]);
        }
#pragma unroll
        for (int c = 0; c < kDw; ++c) {
          constexpr int k0 = kShift ? 1 : 0;
#pragma unroll
          for (int m = 0; m < TC; ++m) acc[m] = __builtin_fmaf(__uint_as_float(xv[m][c] << 16), wf[2 * c + k0], acc[m]);
#pragma unroll
          for (int m = 0; m < TC; ++m)
            acc[m] = __builtin_fmaf(__uint_as_float(xv[m][c] & 0xffff0000u), wf[2 * c + 1 + k0], acc[m]);
        }
        if constexpr (kShift) {
#pragma unroll
          for (int m = 0; m < TC; ++m) acc[m] = __builtin_fmaf(edge_of(m, 2 * i + 1), wf[31], acc[m]);
        }
      }
    }
    codes[0] = codes[1];
    codes[1] = codes[2];
    codes[2] = codes[3];
  }
#pragma unroll
  for (int m = 0; m < TC; ++m) s_part[p][m][lane] = acc[m];
  __syncthreads();
  for (int q = threadIdx.x; q < mc * kTileRows; q += blockDim.x) {
    const int m = q >> 6, r = q & 63;
    float v = s_part[0][m][r];
    for (int pp = 1; pp < g.parts; ++pp) v = v + s_part[pp][m][r];
    const int n = tile * kTileRows + r;
    if (bias != nullptr) v = v + bf16_to_f32(bias[n]);
    y[static_cast<size_t>(m0 + m) * g.N + n] = f32_to_bf16(v);
  }
}

__global__ void swiglu_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int T, int I,
                              float alpha, float limit) {
  const size_t total = static_cast<size_t>(T) * I;
  for (size_t q = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; q < total;
       q += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t t = q / I, j = q % I;
    const float g = bf16_to_f32(in[t * 2 * I + 2 * j]);
    const float u = bf16_to_f32(in[t * 2 * I + 2 * j + 1]);
    out[q] = f32_to_bf16(gx_swiglu(g, u, alpha, limit));
  }
}

// One output per thread: rows or pointers that are not on 16 bytes.
__global__ void combine_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ y,
                               const int32_t* __restrict__ gather_map, const float* __restrict__ w,
                               const uint16_t* __restrict__ residual, int T, int H, int k) {
  const size_t total = static_cast<size_t>(T) * H;
  for (size_t q = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; q < total;
       q += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const int t = static_cast<int>(q / H), n = static_cast<int>(q % H);
    float acc = 0.0f;
    for (int s = 0; s < k; ++s) {
      const int gm = gather_map[t * k + s];
      if (gm < 0) continue;
      acc = __builtin_fmaf(w[t * k + s], bf16_to_f32(y[static_cast<size_t>(gm) * H + n]), acc);
    }
    if (residual != nullptr) acc = acc + bf16_to_f32(residual[q]);
    out[q] = f32_to_bf16(acc);
  }
}

__global__ void scatter_kernel(const uint16_t* __restrict__ x, const int32_t* __restrict__ gather_map,
                               uint16_t* __restrict__ permuted, int T, int H, int k) {
  const int S = T * k;
  const int chunks = H / 8;
  const size_t total = static_cast<size_t>(S) * chunks;
  for (size_t q = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; q < total;
       q += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const int s = static_cast<int>(q / chunks), c = static_cast<int>(q % chunks);
    const int gm = gather_map[s];
    if (gm < 0) continue;
    reinterpret_cast<uint4*>(permuted + static_cast<size_t>(gm) * H)[c] =
        reinterpret_cast<const uint4*>(x + static_cast<size_t>(s / k) * H)[c];
  }
}

__global__ void dequant_kernel(const uint8_t* __restrict__ wn, const uint8_t* __restrict__ ws, TiledGeom g,
                               uint16_t* __restrict__ out) {
  // one thread per (row, block): 32 outputs
  const size_t total = static_cast<size_t>(g.N) * g.nb;
  for (size_t q = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; q < total;
       q += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t row = q / g.nb, b = q % g.nb;
    const size_t tile = row / kTileRows, lane = row % kTileRows;
    const u32x4 blk = load_row_block(reinterpret_cast<const uint32_t*>(wn) + (tile * g.nb + b) * 256 +
                                     tiled_dword(static_cast<int>(lane), 0));
    const size_t p = b / g.bpp, i = b % g.bpp;
    const uint32_t code = ws[((tile * g.parts + p) * kTileRows + lane) * g.spad + i];
    uint16_t* o = out + row * g.K + b * 32;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      float wf[8];
      decode8(blk[d], code, wf);
#pragma unroll
      for (int c = 0; c < 8; ++c) o[d * 8 + c] = f32_to_bf16(wf[c]);
    }
  }
}

// RMSNorm: sum of squares with the gemv_bf16 tree (256 strided chains of
// 8-element chunks, xor butterfly, 4 waves in order), inv = 1/sqrt(mean+eps),
// out = bf16((x * inv) * w).
__global__ __launch_bounds__(256) void rmsnorm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                     uint16_t* __restrict__ out, int H, float eps) {
  __shared__ float s_w[4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, warp = tid >> 6;
  const uint16_t* xr = x + static_cast<size_t>(t) * H;
  float acc = 0.0f;
  const int KV = H >> 3;
  for (int kv = tid; kv < KV; kv += 256) {
    const uint4 v = reinterpret_cast<const uint4*>(xr)[kv];
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = __uint_as_float(d[i] << 16), b = __uint_as_float(d[i] & 0xffff0000u);
      acc = __builtin_fmaf(a, a, acc);
      acc = __builtin_fmaf(b, b, acc);
    }
  }
  for (int kk = KV * 8 + tid; kk < H; kk += 256) {
    const float a = bf16_to_f32(xr[kk]);
    acc = __builtin_fmaf(a, a, acc);
  }
  acc = wave_butterfly_sum(acc);
  if (lane == 0) s_w[warp] = acc;
  __syncthreads();
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) ss = ss + s_w[i];
  const float inv = 1.0f / __builtin_sqrtf(ss / static_cast<float>(H) + eps);
  for (int h = tid; h < H; h += 256)
    out[static_cast<size_t>(t) * H + h] = f32_to_bf16((bf16_to_f32(xr[h]) * inv) * bf16_to_f32(w[h]));
}

// Fused residual + RMSNorm (rmsnorm.cu:224-337): s = r + d in fp32 (kept
// per chunk: a thread's chunks are kv = tid, tid + 256), sum_out = bf16(s),
// the sum of squares of s with the same tree as rmsnorm_kernel, then
// normed = bf16((s * inv) * w).
__global__ __launch_bounds__(256) void residual_rmsnorm_kernel(const uint16_t* __restrict__ r,
                                                               const uint16_t* __restrict__ d,
                                                               const uint16_t* __restrict__ w,
                                                               uint16_t* __restrict__ normed,
                                                               uint16_t* __restrict__ sum_out, int H, float eps) {
  __shared__ float s_w[4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, warp = tid >> 6;
  const size_t row = static_cast<size_t>(t) * H;
  const int KV = H >> 3;
  auto sum8 = [&](int kv, float (&s8)[8]) __attribute__((always_inline)) {
    const uint4 a = reinterpret_cast<const uint4*>(r + row)[kv];
    const uint4 b = reinterpret_cast<const uint4*>(d + row)[kv];
    const uint32_t da[4] = {a.x, a.y, a.z, a.w}, db[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s8[2 * i] = __uint_as_float(da[i] << 16) + __uint_as_float(db[i] << 16);
      s8[2 * i + 1] = __uint_as_float(da[i] & 0xffff0000u) + __uint_as_float(db[i] & 0xffff0000u);
    }
  };
  float acc = 0.0f;
  for (int kv = tid; kv < KV; kv += 256) {
    float s8[8];
    sum8(kv, s8);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = __builtin_fmaf(s8[i], s8[i], acc);
    if (sum_out) {
      uint32_t o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = f32_to_bf16(s8[2 * i]) | (static_cast<uint32_t>(f32_to_bf16(s8[2 * i + 1])) << 16);
      reinterpret_cast<uint4*>(sum_out + row)[kv] = make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
  for (int kk = KV * 8 + tid; kk < H; kk += 256) {
    const float v = bf16_to_f32(r[row + kk]) + bf16_to_f32(d[row + kk]);
    acc = __builtin_fmaf(v, v, acc);
    if (sum_out) sum_out[row + kk] = f32_to_bf16(v);
  }
  acc = wave_butterfly_sum(acc);
  if (lane == 0) s_w[warp] = acc;
  __syncthreads();
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) ss = ss + s_w[i];
  const float inv = 1.0f / __builtin_sqrtf(ss / static_cast<float>(H) + eps);
  for (int h = tid; h < H; h += 256) {
    const float v = bf16_to_f32(r[row + h]) + bf16_to_f32(d[row + h]);
    normed[row + h] = f32_to_bf16((v * inv) * bf16_to_f32(w[h]));
  }
}

int grid_for(size_t total, int threads) {
  size_t b = (total + threads - 1) / threads;
  if (b > 4096) b = 4096;
  if (b < 1) b = 1;
  return static_cast<int>(b);
}

}  // namespace

hipError_t launch_dense_gemv(const uint16_t* x, int M, const uint8_t* wn, const uint8_t* ws, const uint16_t* bias,
                             uint16_t* y, int N, int K, hipStream_t s) {
  if (M <= 0) return hipSuccess;
  const TiledGeom g = tiled_geom(N, K);
  // Token rows per work-group, by the work-groups that one each would make
  // (N = 5760: 8 rows 15.6 / 17.6 / 15.0 us for 1 / 2 / 4 each, 11 rows 17.4 /
  // 19.6 / 24, 24 rows 34 / 27 / 30, 64 rows 73 / 59 / 62; N = 2880, K = 1536:
  // 16 rows 8.9 / 9.9 / 9.4, 32 rows 13.9 / 11.9 / 14.9, 64 rows 24 / 19 / 18).
  const int tiles = N / kTileRows;
  const long groups = static_cast<long>(tiles) * M;
  const int tc = groups <= 1024 ? 1 : groups <= 2560 ? 2 : 4;
  const bool shift = (reinterpret_cast<uintptr_t>(x) & 2u) != 0;  // x is only 2-byte aligned by contract
#define GX_GEMV(TC_, A_)                                                                                            \
  hipLaunchKernelGGL((dense_gemv_kernel<TC_, A_>), dim3(tiles, (M + TC_ - 1) / TC_), dim3(kTileRows* g.parts), 0, s, \
                     x + (A_ ? 1 : 0), M, wn, ws, bias, y, g)
#define GX_GEMV_L(TC_)             \
  do {                             \
    if (shift) GX_GEMV(TC_, true); \
    else GX_GEMV(TC_, false);      \
  } while (0)
  if (tc == 1) GX_GEMV_L(1);
  else if (tc == 2) GX_GEMV_L(2);
  else GX_GEMV_L(4);
#undef GX_GEMV_L
#undef GX_GEMV
  return hipGetLastError();
}

hipError_t launch_swiglu(const uint16_t* in, uint16_t* out, int T, int I, float alpha, float limit, hipStream_t s) {
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(swiglu_kernel, dim3(grid_for(static_cast<size_t>(T) * I, 256)), dim3(256), 0, s, in, out, T, I,
                     alpha, limit);
  return hipGetLastError();
}

hipError_t launch_combine(uint16_t* out, const uint16_t* y, const int32_t* gather_map, const float* w,
                          const uint16_t* residual, int T, int H, int k, hipStream_t s) {
  if (T <= 0) return hipSuccess;
  // The layer's kernel, 8 outputs per thread, where its 16-byte pieces and
  // 32-bit piece count fit (513 tokens of 2880, top-4: 12.2 us one output per
  // thread, 5.1 so; the same bits).
  const uintptr_t ptrs =
      reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(residual);
  if (H % 8 == 0 && (ptrs & 15u) == 0 && static_cast<size_t>(T) * (H / 8) < (1u << 30))
    return launch_combine8(out, y, gather_map, w, residual, T, H, k, KernelTimer{}, s);
  hipLaunchKernelGGL(combine_kernel, dim3(grid_for(static_cast<size_t>(T) * H, 256)), dim3(256), 0, s, out, y,
                     gather_map, w, residual, T, H, k);
  return hipGetLastError();
}

hipError_t launch_scatter(const uint16_t* x, const int32_t* gather_map, uint16_t* permuted, int T, int H, int k,
                          hipStream_t s) {
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(scatter_kernel, dim3(grid_for(static_cast<size_t>(T) * k * (H / 8), 256)), dim3(256), 0, s, x,
                     gather_map, permuted, T, H, k);
  return hipGetLastError();
}

hipError_t launch_dequant(const uint8_t* wn, const uint8_t* ws, int N, int K, uint16_t* out, hipStream_t s) {
  const TiledGeom g = tiled_geom(N, K);
  hipLaunchKernelGGL(dequant_kernel, dim3(grid_for(static_cast<size_t>(N) * g.nb, 256)), dim3(256), 0, s, wn, ws, g,
                     out);
  return hipGetLastError();
}

hipError_t launch_residual_rmsnorm(const uint16_t* r, const uint16_t* d, const uint16_t* w, uint16_t* normed,
                                   uint16_t* sum_out, int T, int H, float eps, hipStream_t s) {
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(residual_rmsnorm_kernel, dim3(T), dim3(256), 0, s, r, d, w, normed, sum_out, H, eps);
  return hipGetLastError();
}

hipError_t launch_rmsnorm(const uint16_t* x, const uint16_t* w, uint16_t* out, int T, int H, float eps,
                          hipStream_t s) {
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(T), dim3(256), 0, s, x, w, out, H, eps);
  return hipGetLastError();
}

}  // namespace gxmoe
