// ConvNeXt tail of the sparse decoder (reference SDecoder::convnext after its conv, src/sdec.cu:59-67):
//
//   y = x + W2 · silu(W1 · (LayerNorm(h) * gamma + beta) + b1) + b2        (per row; hidden width 4C)
//
// which the reference runs as layer_norm (f32 casts, src/ops.cu:30-75), linear (src/gemm.cu:24-63), act_ SILU,
// linear, add_ -- about ten passes over rows of C and 4C channels. C = 64 and 128 run in one kernel: each row is read
// once (h and x) and written once (y); the 4C-wide hidden activations never leave registers. C >= 256 run as
// LayerNorm + weight repack and two GEMMs (k_mlp_prep, k_gemm): fused, C = 256 was bound by its weight reads from LDS
// (one 1 KiB fragment per MFMA; a second block of rows per wavefront does not fit in registers), 58321 rows 162 us
// against 111 (15000: 86 / 39, 390000: 897 / 721).
//
// Work split. A workgroup of 4 wavefronts walks row tiles (persistent grid); each wavefront owns 32 rows.
// The hidden dimension is processed in chunks of 32:
//   GEMM1  H^T[32 hid x 32 rows] = W1[chunk rows, :] · Xn^T      (C/16 v_mfma_f32_32x32x16, K = channels)
//   H^T    += b1, SiLU, rounded to the operand type
//   GEMM2  Y^T[C x 32 rows]    += W2[:, chunk] · H^T            (2 MFMAs per 32 output channels)
// MFMA 32x32x16 layouts: lane l supplies A row l%32 and B column l%32 with K values (l/32)*8 .. +8; the result gives
// lane l column l%32 and rows (i/4)*8 + (l/32)*4 + i%4. So a lane's normalized row chunks (row l%32, channels
// t*16 + (l/32)*8 .. +8) are GEMM1's B operand as loaded, and GEMM1's result (column = row l%32, hidden rows
// (i/4)*8 + (l/32)*4 + i%4) is GEMM2's B operand without any transpose, provided W2's K order is permuted to match;
// the weight pack below stores W1 and W2 in exactly those operand orders, one 16-byte load per lane per MFMA.
// Weights live in LDS: all of them for C = 64 (64 KiB, loaded once per workgroup), else streamed per chunk through
// three chunk buffers shared by the 4 wavefronts (C = 128).
#include <algorithm>
#include <utility>

#include "lnact.h"
#include "spconv.h"

namespace {
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kOOR = 0xffff0000u;

template <bool F16>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}
template <bool F16>
__device__ __forceinline__ float lo(uint32_t v) {
  if constexpr (F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)v);
  else return __uint_as_float(v << 16);
}
template <bool F16>
__device__ __forceinline__ float hi(uint32_t v) {
  if constexpr (F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16));
  else return __uint_as_float(v & 0xffff0000u);
}
template <bool F16>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (F16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float silu(float v) { return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v)); }

constexpr int kMlpThreads = 256, kMlpRows = kMlpThreads / 64 * 32;  // rows of a workgroup's tile: 32 per wavefront

template <int C>
struct MlpShape {
  static constexpr int NCH = C / 8;                // hidden chunks of 32 (hidden width 4C)
  static constexpr int KS = C / 16;                // GEMM1 K steps per chunk
  static constexpr int YT = C / 32;                // 32-channel output tiles
  static constexpr int W1Q = KS * 64;              // 16-byte units of a chunk's W1 part
  static constexpr int CHUNK = W1Q + YT * 2 * 64;  // 16-byte units per chunk (W1 then W2)
  static constexpr bool RESIDENT = C == 64;        // all weights in LDS (NCH * CHUNK * 16 = 64 KiB)
  static constexpr int LDSQ = RESIDENT ? NCH * CHUNK : 3 * CHUNK;
};

// Weights into operand order: wp[chunk][W1: KS x 64 lanes | W2: YT x 2 x 64 lanes] 16-byte units.
//   W1 unit (t, lane): hidden chunk*32 + lane%32, channels t*16 + (lane/32)*8 .. +8             (w1 [4C, C])
//   W2 unit (tt, u, lane): output channel tt*32 + lane%32, hidden chunk*32 + u*16 + (lane/32)*4 + {0..3, 8..11}
//                                                                                             (w2 [C, 4C])
// and the parameters as f32 params [gamma C | beta C | b1 4C | b2 C] (null: 1, 0, 0, 0), in the same launch.
struct MlpParams {
  const void* p[4];
  int dt[4];
};
template <int C>
__global__ void __launch_bounds__(256) k_pack_mlp(const uint16_t* __restrict__ w1, const uint16_t* __restrict__ w2,
                                                  MlpParams mp, u32x4* __restrict__ wp, float* __restrict__ params) {
  using S = MlpShape<C>;
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= S::NCH * S::CHUNK) {
    q -= S::NCH * S::CHUNK;
    if (q >= 7 * C) return;
    const int k = q < C ? 0 : q < 2 * C ? 1 : q < 6 * C ? 2 : 3, i = q - (k == 0 ? 0 : k == 1 ? C : k == 2 ? 2 * C : 6 * C);
    const void* p = k == 0 ? mp.p[0] : k == 1 ? mp.p[1] : k == 2 ? mp.p[2] : mp.p[3];
    const int dt = k == 0 ? mp.dt[0] : k == 1 ? mp.dt[1] : k == 2 ? mp.dt[2] : mp.dt[3];
    float v = k == 0 ? 1.f : 0.f;
    if (p) {
      if (dt == F32) {
        v = ((const float*)p)[i];
      } else {
        const uint16_t u = ((const uint16_t*)p)[i];
        v = dt == BF16 ? __uint_as_float((uint32_t)u << 16) : (float)__builtin_bit_cast(_Float16, u);
      }
    }
    params[q] = v;
    return;
  }
  const int c = q / S::CHUNK, k = q % S::CHUNK, lane = k & 63;
  if (k < S::W1Q) {
    const int t = k >> 6;
    wp[q] = *(const u32x4*)&w1[(i64)(c * 32 + (lane & 31)) * C + t * 16 + (lane >> 5) * 8];
  } else {
    const int k2 = k - S::W1Q, u = (k2 >> 6) & 1, tt = k2 >> 7;
    const uint16_t* r = &w2[(i64)(tt * 32 + (lane & 31)) * (4 * C) + c * 32 + u * 16 + (lane >> 5) * 4];
    const u32x2 a = *(const u32x2*)r, b = *(const u32x2*)(r + 8);
    wp[q] = u32x4{a[0], a[1], b[0], b[1]};
  }
}

// params: f32 [gamma C | beta C | b1 4C | b2 C]
template <bool F16, int C>
__global__ void __launch_bounds__(kMlpThreads, 2) k_convnext_mlp(const uint16_t* h, const uint16_t* x, uint16_t* y,
                                                                 const u32x4* __restrict__ wp,
                                                                 const float* __restrict__ params, float eps, i64 n,
                                                                 i64 tiles, uint32_t h_bytes, uint32_t x_bytes,
                                                                 uint32_t y_bytes) {
  using S = MlpShape<C>;
  __shared__ u32x4 lw[S::LDSQ];
  __shared__ float lp[7 * C];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r32 = lane & 31, h8 = lane >> 5;
  const float* s_g = lp;
  const float* s_bt = lp + C;
  const float* s_b1 = lp + 2 * C;
  const float* s_b2 = lp + 6 * C;
  for (int i = tid; i < 7 * C; i += kMlpThreads) lp[i] = params[i];
  if constexpr (S::RESIDENT)
    for (int i = tid; i < S::LDSQ; i += kMlpThreads) lw[i] = wp[i];
  __syncthreads();
  const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(h), 0, (int)h_bytes,
                                                                      0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (int)x_bytes,
                                                                      0x00020000);
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y, 0, (int)y_bytes, 0x00020000);
  constexpr int SQ = (S::CHUNK + kMlpThreads - 1) / kMlpThreads;  // 16-byte units staged per thread and chunk

  for (i64 tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const i64 row = tile * kMlpRows + wave * 32 + r32;
    const bool ok = row < n;
    asm volatile("" ::: "memory");  // keeps the per-channel LDS parameter reads inside the loop (no 100-VGPR hoist)
    // rows of h (LayerNorm input) as GEMM1 B operands, and x (residual) in the output layout (at C = 128 only in the
    // epilogue: its registers in the loop would spill)
    u32x4 xn[S::KS];
    u32x2 xr[S::YT][4];
    auto load_x = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int tt = 0; tt < S::YT; tt++)
#pragma unroll
        for (int g = 0; g < 4; g++)
          xr[tt][g] = __builtin_amdgcn_raw_buffer_load_b64(
              rx, ok ? (uint32_t)((row * C + tt * 32 + g * 8 + h8 * 4) * 2) : kOOR, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < S::KS; t++)
      xn[t] = __builtin_amdgcn_raw_buffer_load_b128(rh, ok ? (uint32_t)((row * C + t * 16 + h8 * 8) * 2) : kOOR, 0,
                                                    0);
    if constexpr (C == 64) load_x();
    // LayerNorm: a row's C values sit in lanes r32 and r32 + 32; mean first, then the centred variance
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < S::KS; t++)
#pragma unroll
      for (int j = 0; j < 4; j++) s += lo<F16>(xn[t][j]) + hi<F16>(xn[t][j]);
    s += __shfl_xor(s, 32, 64);
    const float mean = s * (1.0f / C);
    float q = 0.f;
#pragma unroll
    for (int t = 0; t < S::KS; t++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float a = lo<F16>(xn[t][j]) - mean, b = hi<F16>(xn[t][j]) - mean;
        q += a * a + b * b;
      }
    q += __shfl_xor(q, 32, 64);
    const float rstd = rsqrtf(q * (1.0f / C) + eps);
#pragma unroll
    for (int t = 0; t < S::KS; t++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int ch = t * 16 + h8 * 8 + 2 * j;
        const float a = (lo<F16>(xn[t][j]) - mean) * rstd * s_g[ch] + s_bt[ch];
        const float b = (hi<F16>(xn[t][j]) - mean) * rstd * s_g[ch + 1] + s_bt[ch + 1];
        xn[t][j] = pack2<F16>(a, b);
      }

    f32x16 acc[S::YT];
#pragma unroll
    for (int tt = 0; tt < S::YT; tt++) acc[tt] = f32x16{};

    // Software pipeline over hidden chunks: GEMM1 of chunk c+1 is issued before the SiLU of chunk c, so the VALU
    // work overlaps MFMA execution. Streaming mode keeps three chunk buffers: in iteration c the wavefronts read
    // W1 of chunk c+1 and W2 of chunk c, and chunk c+2 is written into the buffer of chunk c-1.
    auto buf = [&](int c) -> const u32x4* { return S::RESIDENT ? lw + c * S::CHUNK : lw + (c % 3) * S::CHUNK; };
    auto gemm1 = [&](const u32x4* cw, f32x16& hacc) {
      hacc = f32x16{};
#pragma unroll
      for (int t = 0; t < S::KS; t++) {
        const u32x4 a = cw[t * 64 + lane];
        hacc = mfma32<F16>(a, xn[t], hacc);
      }
    };
    u32x4 stg[SQ];
    if constexpr (!S::RESIDENT) {  // chunks 0 and 1 into buffers 0 and 1, once every wavefront left the last tile
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 2 * SQ; k++)
        if ((k % SQ) * kMlpThreads + tid < S::CHUNK)
          lw[(k / SQ) * S::CHUNK + (k % SQ) * kMlpThreads + tid] = wp[(k / SQ) * S::CHUNK + (k % SQ) * kMlpThreads + tid];
      __syncthreads();
    }
    f32x16 hnext;
    gemm1(buf(0), hnext);
#pragma unroll 1
    for (int c = 0; c < S::NCH; c++) {
      if constexpr (!S::RESIDENT)
        if (c + 2 < S::NCH)
#pragma unroll
          for (int k = 0; k < SQ; k++)
            if (k * kMlpThreads + tid < S::CHUNK) stg[k] = wp[(c + 2) * S::CHUNK + k * kMlpThreads + tid];
      const f32x16 hacc = hnext;
      if (c + 1 < S::NCH) gemm1(buf(c + 1), hnext);
      u32x4 hb[2];
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int i = u * 8 + 2 * j;  // accumulators i, i+1: hidden rows (i/4)*8 + h8*4 + i%4 (+1)
          const int hid = c * 32 + (i >> 2) * 8 + h8 * 4 + (i & 3);
          hb[u][j] = pack2<F16>(silu(hacc[i] + s_b1[hid]), silu(hacc[i + 1] + s_b1[hid + 1]));
        }
      const u32x4* cw = buf(c);
#pragma unroll
      for (int tt = 0; tt < S::YT; tt++)
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const u32x4 a = cw[S::W1Q + (tt * 2 + u) * 64 + lane];
          acc[tt] = mfma32<F16>(a, hb[u], acc[tt]);
        }
      // buffer (c+2) % 3 held chunk c-1, last read in iteration c-1, which every wavefront finished before the
      // barrier that ended it; one barrier per chunk publishes the new contents
      if constexpr (!S::RESIDENT)
        if (c + 2 < S::NCH) {
#pragma unroll
          for (int k = 0; k < SQ; k++)
            if (k * kMlpThreads + tid < S::CHUNK) lw[((c + 2) % 3) * S::CHUNK + k * kMlpThreads + tid] = stg[k];
          __syncthreads();
        }
    }
    // y = x + acc + b2, 4 consecutive channels per (tile, group) as one 8-byte store; rows past n are dropped
    if constexpr (C != 64) load_x();
#pragma unroll
    for (int tt = 0; tt < S::YT; tt++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int co = tt * 32 + g * 8 + h8 * 4;
        const u32x2 xv = xr[tt][g];
        const float v0 = acc[tt][g * 4 + 0] + s_b2[co + 0] + lo<F16>(xv[0]);
        const float v1 = acc[tt][g * 4 + 1] + s_b2[co + 1] + hi<F16>(xv[0]);
        const float v2 = acc[tt][g * 4 + 2] + s_b2[co + 2] + lo<F16>(xv[1]);
        const float v3 = acc[tt][g * 4 + 3] + s_b2[co + 3] + hi<F16>(xv[1]);
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2<F16>(v0, v1), pack2<F16>(v2, v3)}, ry,
                                              ok ? (uint32_t)((row * C + co) * 2) : kOOR, 0, 0);
      }
  }
}

int device_cus() {
  static int n = [] {
    int dev = 0, v = 0;
    CK(hipGetDevice(&dev));
    CK(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev));
    return v;
  }();
  return n;
}

template <bool F16, int C>
void launch_mlp(const Tensor& h, const Tensor& x, const Tensor& w1, const Tensor& w2, const MlpParams& mp, float eps,
                Tensor& y) {
  using S = MlpShape<C>;
  const i64 n = h.size(0);
  Tensor wp = empty({(i64)S::NCH * S::CHUNK * 8}, h.dt), params = empty({7 * (i64)C}, F32);
  k_pack_mlp<C><<<cdiv(S::NCH * S::CHUNK + 7 * C, 256), 256, 0, stream()>>>(
      w1.ptr<uint16_t>(), w2.ptr<uint16_t>(), mp, (u32x4*)wp.p, params.ptr<float>());
  const i64 tiles = cdiv(n, kMlpRows);
  const i64 grid = std::min<i64>(tiles, (i64)device_cus() * 2);
  k_convnext_mlp<F16, C><<<(unsigned)grid, kMlpThreads, 0, stream()>>>(
      h.ptr<uint16_t>(), x.ptr<uint16_t>(), y.ptr<uint16_t>(), (const u32x4*)wp.p, params.ptr<float>(), eps, n, tiles,
      (uint32_t)h.bytes(), (uint32_t)x.bytes(), (uint32_t)y.bytes());
}

// Row-block GEMM of the tail's wide widths (their fused output tile does not fit in registers):
//   hid[m, n] = silu(A[m, :] . B[n, :] + bias[n])   or, with RES,   Y[m, n] = A[m, :] . B[n, :] + bias[n] + R[m, n]
// with one rounding to the operand type. A and B are in operand order: one 1 KiB block per (16 rows or columns, 32
// channels), lane l of v_mfma_f32_16x16x32 holding row l % 16, channels (l / 16) * 8 .. +8; the blocks of a 16-row
// group in channel order. hid is written in that order too (it is the next product's A, padded to whole 128-row
// tiles whose extra rows hold anything: a row of A reaches only its own output row); R and Y are [M,N] row-major.
//  * Operand order keeps the address path out of the loop: a load or LDS DMA is one contiguous 1 KiB, where 64-byte
//    pieces of 16 rows cost several times as much (the whole tail at C = 512, 25000 rows: 172 us with B read from its
//    rows, 143 with B repacked, 135 with A in operand order too; the former kernel, 128 x 128 tiles of both operands
//    staged through registers into LDS, 351).
//  * Tile BM rows x BN columns, 4 wavefronts (per K group) of BM rows x BN/4 columns each. A goes global -> LDS by DMA
//    (64-channel stages, a ring of DB + 2 slots); B goes straight into operand registers, DB stages ahead.
//  * Per stage: issue B(s + DB), then A(s + DB + 1); the counted wait before stage s leaves everything issued after
//    B(s) in flight, which also covers A(s). Stages past the end read through a zero-size resource (no memory
//    traffic), so the counts stay constant.
//  * KG = 2: two K groups of 4 wavefronts halve the K loop of a tile; each then owns half of the tile's rows and adds
//    the other group's sums through LDS (group 0 first), so nothing is split across workgroups.
//  * Epilogue through LDS, 16 rows at a time, as 16-byte pieces (row stride WN + 4 words: conflict-free both ways).
struct GemmArgs {
  const uint16_t *A, *B, *R;
  const void* bias;
  uint16_t* Y;
  int bias_dt, M, N, K, tiles_m, tiles_n, per, col_major;
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
template <int N>
__device__ __forceinline__ void wait_vm() {  // vmcnt(N) only
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void bare_barrier() {  // no fence: callers order LDS data with counted waits
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// 16 bytes per lane, global -> LDS: lane l's land at dst + l (dst uniform over the wavefront)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, u32x4* dst, uint32_t off, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, off, soff, 0, 0);
}
template <class F, int... I>
__device__ __forceinline__ void unroll_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unroll(F&& f) {
  unroll_impl(f, std::make_integer_sequence<int, N>{});
}
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <bool F16>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}
// 8 consecutive parameters p[i .. i + 8) of dtype dt (null: zeros); the buffer need only be element-aligned
__device__ __forceinline__ void load_param8(const void* p, int dt, int i, float (&o)[8]) {
  typedef float f32x8u __attribute__((ext_vector_type(8), aligned(4)));
  typedef uint16_t u16x8u __attribute__((ext_vector_type(8), aligned(2)));
#pragma unroll
  for (int q = 0; q < 8; q++) o[q] = 0.f;
  if (!p) return;
  if (dt == F32) {
    const f32x8u v = *(const f32x8u*)((const float*)p + i);
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = v[q];
  } else {
    const u16x8u v = *(const u16x8u*)((const uint16_t*)p + i);
    if (dt == BF16) {
#pragma unroll
      for (int q = 0; q < 8; q++) o[q] = __uint_as_float((uint32_t)v[q] << 16);
    } else {
#pragma unroll
      for (int q = 0; q < 8; q++) o[q] = (float)__builtin_bit_cast(_Float16, (uint16_t)v[q]);
    }
  }
}

// What the wide widths' products read, in one launch, both in k_gemm's operand order: workgroups below nln normalize
// their rows (LayerNorm + affine, rounded to the operand type; a row's C channels over up to 64 lanes, four 1 KiB loads
// per wavefront in flight and their reductions interleaved) and turn them through LDS, so that whole 1 KiB blocks are
// stored; the others repack the weights, four blocks per wavefront.
template <int C>
constexpr int kPrepRows = C >= 512 ? 16 : 16 * 512 / C;  // rows per workgroup
template <bool F16, int C>
__global__ void __launch_bounds__(256) k_mlp_prep(const uint16_t* __restrict__ h, i64 n, int nln, const void* gamma,
                                                  int gdt, const void* beta, int bdt, float eps,
                                                  u32x4* __restrict__ out, const u32x4* __restrict__ w1,
                                                  const u32x4* __restrict__ w2, u32x4* __restrict__ wp) {
  constexpr int LPR = C / 8 < 64 ? C / 8 : 64, CH = C / 8 / LPR, RP = 64 / LPR, P = 4;
  constexpr int WR = kPrepRows<C>;
  static_assert(WR == 4 * P * RP, "rows of four wavefronts");
  constexpr int RS = C / 8 + 1;  // row stride in 16-byte units: 16 rows' units of one column lie in distinct banks
  __shared__ u32x4 rows[WR * RS];
  const int tid = threadIdx.x, lane = tid & 63;
  if ((int)blockIdx.x >= nln) {
    constexpr int PER = 4 * C * C / 512;  // blocks per weight
    const int b0 = (((int)blockIdx.x - nln) * 4 + (tid >> 6)) * 4, first = b0 < PER;
    const int K = first ? C : 4 * C, b1 = first ? b0 : b0 - PER, cb = b1 / (K / 32), kb = b1 % (K / 32);
    const u32x4* src = (first ? w1 : w2) + (i64)(cb * 16 + (lane & 15)) * (K / 8) + kb * 4 + (lane >> 4);
    u32x4 q[4];
#pragma unroll
    for (int k = 0; k < 4; k++) q[k] = src[k * 4];  // K / 32 is a multiple of 4: one column group
#pragma unroll
    for (int k = 0; k < 4; k++) wp[(b0 + k) * 64 + lane] = q[k];
    return;
  }
  const int sub = lane % LPR, r0 = (tid >> 6) * (P * RP) + lane / LPR;  // this lane's row of pass p: r0 + p * RP
  const i64 row0 = (i64)blockIdx.x * WR;
  u32x4 q[P][CH];
#pragma unroll
  for (int p = 0; p < P; p++)
#pragma unroll
    for (int c = 0; c < CH; c++) q[p][c] = *(const u32x4*)&h[min(row0 + r0 + p * RP, n - 1) * C + (c * LPR + sub) * 8];
  float g8[CH][8], b8[CH][8];
#pragma unroll
  for (int c = 0; c < CH; c++) {
    load_param8(gamma, gdt, (c * LPR + sub) * 8, g8[c]);
    load_param8(beta, bdt, (c * LPR + sub) * 8, b8[c]);
  }
  float v[P][CH][8], mean[P], rstd[P];
#pragma unroll
  for (int p = 0; p < P; p++)
#pragma unroll
    for (int c = 0; c < CH; c++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v[p][c][2 * j] = lo<F16>(q[p][c][j]);
        v[p][c][2 * j + 1] = hi<F16>(q[p][c][j]);
      }
#pragma unroll
  for (int p = 0; p < P; p++) ln_stats<LPR, CH>(v[p], C, eps, mean[p], rstd[p]);
#pragma unroll
  for (int c = 0; c < CH; c++)
#pragma unroll
    for (int p = 0; p < P; p++) {
      float o[8];
      ln_out8(v[p][c], mean[p], rstd[p], gamma ? g8[c] : nullptr, beta ? b8[c] : nullptr, 0, o);
      rows[(r0 + p * RP) * RS + c * LPR + sub] =
          u32x4{pack2<F16>(o[0], o[1]), pack2<F16>(o[2], o[3]), pack2<F16>(o[4], o[5]), pack2<F16>(o[6], o[7])};
    }
  __syncthreads();
  constexpr int NB = WR / 16 * (C / 32);  // blocks of this workgroup's rows
#pragma unroll
  for (int k = 0; k < NB / 4; k++) {
    const int blk = k * 4 + (tid >> 6), rg = blk / (C / 32), kb = blk % (C / 32);
    out[((i64)blockIdx.x * NB + blk) * 64 + lane] = rows[(rg * 16 + (lane & 15)) * RS + kb * 4 + (lane >> 4)];
  }
}

template <bool F16, int BM, int BN, int KG, int DB, bool RES>
__global__ void __launch_bounds__(256 * KG, 2) k_gemm(GemmArgs g) {
  constexpr int WN = BN / 4, TM = BM / 16, TN = WN / 16, AL = BM / 32, NB = 2 * TN;
  constexpr int SLOTS = DB + 2, SETS = DB + 1, SQ = KG * BM * 8;  // 16-byte units per slot
  static_assert(SLOTS == 3 || SLOTS == 4, "ring of three or four named slots");
  __shared__ __attribute__((aligned(16))) u32x4 s0[SQ], s1[SQ], s2[SQ], s3[SLOTS == 4 ? SQ : 1];
  const int logical = (blockIdx.x % 8) * g.per + blockIdx.x / 8;  // each XCD walks one contiguous range of tiles
  if (logical >= g.tiles_m * g.tiles_n) return;
  const int tm = g.col_major ? logical % g.tiles_m : logical / g.tiles_n;
  const int tn = g.col_major ? logical / g.tiles_m : logical % g.tiles_n;
  const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave >> 2, wv = wave & 3;
  const int K = g.K, N = g.N, rows = min(BM, g.M - tm * BM), S = K / 64 / KG;
  const uint16_t* Ap = g.A + (i64)tm * BM * K + (i64)kg * S * 1024;  // a K group: 2 S blocks of 512 per row group
  const uint16_t* Bp = g.B + (i64)(tn * BN + wv * WN) * K + (i64)kg * S * 1024;
  const uint32_t a_bytes = (uint32_t)((TM - 1) * 16 * K + S * 1024) * 2u, b_bytes = (uint32_t)((TN - 1) * 16 * K + S * 1024) * 2u;
  auto slot = [&](auto I) __attribute__((always_inline)) -> u32x4* {
    constexpr int i = decltype(I)::value % SLOTS;
    return (i == 0 ? s0 : i == 1 ? s1 : i == 2 ? s2 : s3) + kg * (BM * 8);
  };
  // a slot holds the stage's 2 TM blocks: block d = 2 * (row group) + (32-channel half)
  auto dma_a = [&](u32x4* dst, int s) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = rsrc_of(Ap, s < S ? a_bytes : 0u);
#pragma unroll
    for (int k = 0; k < AL; k++) {
      const int d = wv * AL + k;
      dma16(r, &dst[d * 64], lane * 16, (d >> 1) * 32 * K + (d & 1) * 1024 + (s < S ? s * 2048 : 0));
    }
  };
  u32x4 rb[SETS][2][TN];
  auto load_b = [&](u32x4 (&d)[2][TN], int s) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = rsrc_of(Bp, s < S ? b_bytes : 0u);
#pragma unroll
    for (int t = 0; t < TN; t++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        d[j][t] = __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16 + j * 1024, (s < S ? s * 2048 : 0) + t * 32 * K, 0);
  };
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int t = 0; t < TN; t++) acc[i][t] = f32x4{};

  // prologue in the loop's issue order: A(0); then B(s), A(s + 1) for s < DB
  dma_a(slot(std::integral_constant<int, 0>{}), 0);
  unroll<DB>([&](auto I) __attribute__((always_inline)) {
    load_b(rb[I], I);
    dma_a(slot(std::integral_constant<int, I + 1>{}), I + 1);
  });
  constexpr int CH = TM < 4 ? TM : 4;  // operand fragments read ahead of their MFMAs
  auto stage = [&](auto I, int s) __attribute__((always_inline)) {
    constexpr int i0 = decltype(I)::value;
    wait_vm<AL + (DB - 1) * (NB + AL)>();
    bare_barrier();
    load_b(rb[(i0 + DB) % SETS], s + DB);
    dma_a(slot(std::integral_constant<int, i0 + DB + 1>{}), s + DB + 1);
    const u32x4* cur = slot(I);
    u32x4 fa[2][CH];
    auto read = [&](u32x4 (&f)[CH], int c) __attribute__((always_inline)) {  // chunk c: K step c / (TM/CH)
      const int j = c / (TM / CH), i = c % (TM / CH) * CH;
#pragma unroll
      for (int k = 0; k < CH; k++) f[k] = cur[((i + k) * 2 + j) * 64 + lane];
    };
    read(fa[0], 0);
#pragma unroll
    for (int c = 0; c < 2 * TM / CH; c++) {
      if (c + 1 < 2 * TM / CH) read(fa[(c + 1) & 1], c + 1);
      const int j = c / (TM / CH), i = c % (TM / CH) * CH;
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int k = 0; k < CH; k++)
#pragma unroll
        for (int t = 0; t < TN; t++) acc[i + k][t] = mfma16<F16>(fa[c & 1][k], rb[i0 % SETS][j][t], acc[i + k][t]);
      __builtin_amdgcn_s_setprio(0);
    }
  };
  constexpr int U = SLOTS * SETS;  // slots and register sets have fixed names in the unrolled loop
  for (int s = 0; s < S; s += U) {
    bool more = true;
    unroll<U>([&](auto I) __attribute__((always_inline)) {
      if (more && s + decltype(I)::value < S) stage(I, s + decltype(I)::value);
      else more = false;
    });
  }
  wait_vm<0>();
  __syncthreads();

  // each K group keeps TO = TM / KG of the 16-row groups, and gives the other its sums of the rest
  constexpr int TO = TM / KG;
  if constexpr (KG == 2) {
    constexpr int EC = TO * TN * 256 <= SQ ? TO : SQ / (TN * 256);  // row groups exchanged at a time
    static_assert(TO % EC == 0 && 4 * EC * TN * 64 <= SQ, "a group's exchange fits in a slot");
    f32x4* mine = (f32x4*)(kg == 0 ? s0 : s1) + wv * (EC * TN * 64);
    const f32x4* other = (const f32x4*)(kg == 0 ? s1 : s0) + wv * (EC * TN * 64);
#pragma unroll
    for (int i0 = 0; i0 < TO; i0 += EC) {
      if (i0) __syncthreads();
#pragma unroll
      for (int i = 0; i < EC; i++)
#pragma unroll
        for (int t = 0; t < TN; t++) mine[(i * TN + t) * 64 + lane] = kg == 0 ? acc[TO + i0 + i][t] : acc[i0 + i][t];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < EC; i++)
#pragma unroll
        for (int t = 0; t < TN; t++) {
          const f32x4 o = other[(i * TN + t) * 64 + lane];
          acc[i0 + i][t] = (kg == 0 ? acc[i0 + i][t] : acc[TO + i0 + i][t]) + o;
        }
    }
    __syncthreads();
  }
  const int rg = kg * TO * 16;  // first row of this wavefront's part of the tile
  // 16 rows x WN columns at a time through this wavefront's LDS area: lane l writes column l % 16 of 4 rows per
  // fragment and reads 8 consecutive columns of one row per piece
  constexpr int ES = WN + 4, NP = WN / 32, LPR = WN / 8;
  constexpr int APS = SQ * 16 / (16 * ES * 4);  // wavefronts' areas per slot
  static_assert(APS * SLOTS >= 4 * KG, "every wavefront has an area");
  const int as = (kg * 4 + wv) / APS;
  float* ew = (float*)(as == 0 ? s0 : as == 1 ? s1 : as == 2 ? s2 : s3) + (kg * 4 + wv) % APS * (16 * ES);
  // piece p of this lane: row prow(p) and column pcol(p) of the 16 x WN part; hid in operand order, Y by rows
  auto prow = [&](int p) __attribute__((always_inline)) { return RES ? p * (64 / LPR) + lane / LPR : r16; };
  auto pcol = [&](int p) __attribute__((always_inline)) { return RES ? lane % LPR * 8 : p * 32 + q4 * 8; };
  const int col0 = tn * BN + wv * WN;
  float b8[RES ? 1 : NP][8];
#pragma unroll
  for (int p = 0; p < (RES ? 1 : NP); p++) load_param8(g.bias, g.bias_dt, col0 + pcol(p), b8[p]);
  const i64 base = (i64)tm * BM * N;
  const uint32_t y_bytes = (uint32_t)((RES ? rows : BM) * N) * 2u;
  const __amdgpu_buffer_rsrc_t ry = rsrc_of(g.Y + base, y_bytes), rr = rsrc_of(RES ? g.R + base : nullptr, RES ? y_bytes : 0u);
  auto yoff = [&](int i, int p) __attribute__((always_inline)) {
    if (!RES) return (uint32_t)((rg + i * 16) * N * 2 + (col0 / 32 + p) * 1024 + lane * 16);
    const int r = rg + i * 16 + prow(p);
    return r < rows ? (uint32_t)(r * N + col0 + pcol(p)) * 2u : kOOR;
  };
  u32x4 res[2][NP];
  auto load_r = [&](u32x4 (&d)[NP], int i) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++) d[p] = __builtin_amdgcn_raw_buffer_load_b128(rr, yoff(i, p), 0, 0);
  };
  if constexpr (RES) load_r(res[0], 0);
#pragma unroll
  for (int i = 0; i < TO; i++) {
    if (RES && i + 1 < TO) load_r(res[(i + 1) & 1], i + 1);
#pragma unroll
    for (int t = 0; t < TN; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) ew[(q4 * 4 + q) * ES + t * 16 + r16] = acc[i][t][q];
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const float* e = &ew[prow(p) * ES + pcol(p)];
      float v[8];
      *(f32x4*)&v[0] = *(const f32x4*)e;
      *(f32x4*)&v[4] = *(const f32x4*)(e + 4);
#pragma unroll
      for (int q = 0; q < 8; q++) v[q] += b8[RES ? 0 : p][q];
      if constexpr (RES) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          v[2 * q] += lo<F16>(res[i & 1][p][q]);
          v[2 * q + 1] += hi<F16>(res[i & 1][p][q]);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = silu(v[q]);
      }
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{pack2<F16>(v[0], v[1]), pack2<F16>(v[2], v[3]), pack2<F16>(v[4], v[5]),
                                                   pack2<F16>(v[6], v[7])}, ry, yoff(i, p), 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  }
}

template <bool F16, int BM, int BN, int KG, int DB>
void launch_gemm(GemmArgs g) {
  g.tiles_m = cdiv(g.M, BM);
  g.tiles_n = g.N / BN;
  g.per = cdiv((i64)g.tiles_m * g.tiles_n, 8);
  // weights past half an XCD's L2: each XCD keeps to a range of columns; else to a range of rows
  g.col_major = (i64)g.N * g.K * 2 > (2 << 20);
  if (g.R) k_gemm<F16, BM, BN, KG, DB, true><<<g.per * 8, 256 * KG, 0, stream()>>>(g);
  else k_gemm<F16, BM, BN, KG, DB, false><<<g.per * 8, 256 * KG, 0, stream()>>>(g);
  CK(hipGetLastError());
}

// hid = silu(a . b^T + bias), or with r  y = a . b^T + bias + r, M rows; a, b and hid in operand order
template <bool F16>
void gemm_nt(const uint16_t* a, const uint16_t* b, const Tensor* bias, const uint16_t* r, i64 M, int N, int K,
             uint16_t* y) {
  GemmArgs g{};
  g.A = a;
  g.B = b;
  g.R = r;
  g.bias = bias ? bias->p : nullptr;
  g.bias_dt = bias ? bias->dt : F32;
  g.Y = y;
  REQ(M < (1ll << 31) - 128 && N % 128 == 0 && K % 128 == 0, "gemm M=%lld N=%d K=%d", (long long)M, N, K);
  g.M = (int)M;
  g.K = K;
  g.N = N;
  // 128 x 256 tiles (two workgroups per CU) move the fewest operand bytes per flop, but need a tile per CU and a long
  // K loop; 128 x 128 (three per CU) fill the chip sooner and overlap short K loops with epilogues; below 5/8 of a
  // tile per CU, 64 x 128 tiles with two K groups. us at 128 x 256 / 128 x 128 / 64 x 128, [M, N, K]:
  // [8192, 4096, 1024] 70 / 89 / 122, [25000, 512, 2048] 54 / 60 / 70, [25000, 2048, 512] 64 / 61 / 87,
  // [1803, 4096, 1024] 22 / 20 / 26, [3000, 1024, 4096] 57 / 37 / 41, [1803, 1024, 4096] 57 / 34 / 24.
  const i64 tm = cdiv(M, 128), cus = device_cus();
  if (K >= 1024 && N % 256 == 0 && tm * (N / 256) >= cus) launch_gemm<F16, 128, 256, 1, 1>(g);
  else if (tm * (N / 128) >= cus * 5 / 8) launch_gemm<F16, 128, 128, 1, 1>(g);
  else launch_gemm<F16, 64, 128, 2, 2>(g);
}

// The tail at C >= 256: LayerNorm + affine and the weight repack (one launch), then the two products with their
// epilogues (hidden rounded to the operand type, as in the fused kernel). The residual is read and y written by the
// same thread, so y may alias x, and a row of h is consumed before its y is written. Many rows go in equal parts
// whose hidden units stay below kHidBytes: they are then read back from the 256 MB cache, and the workspace is
// bounded.
constexpr i64 kHidBytes = 192ll << 20;
template <bool F16, int C>
void mlp_wide(const Tensor& h, const Tensor& x, const Tensor* gamma, const Tensor* beta, float eps, const Tensor& w1,
              const Tensor* b1, const Tensor& w2, const Tensor* b2, Tensor& y) {
  const i64 n = h.size(0), parts = (n * 4 * C * 2 + kHidBytes - 1) / kHidBytes;
  const i64 step = ((n + parts - 1) / parts + 127) / 128 * 128;  // a and hid hold whole 128-row tiles
  Tensor a = empty({step, C}, h.dt), hid = empty({step, 4 * (i64)C}, h.dt), wp = empty({8 * (i64)C * C}, h.dt);
  for (i64 r0 = 0; r0 < n; r0 += step) {
    const i64 m = std::min(step, n - r0);
    const int nln = cdiv(m, kPrepRows<C>), npack = r0 == 0 ? 8 * C * C / 512 / 16 : 0;
    k_mlp_prep<F16, C><<<nln + npack, 256, 0, stream()>>>(
        h.ptr<uint16_t>() + r0 * C, m, nln, gamma ? gamma->p : nullptr, gamma ? gamma->dt : F32,
        beta ? beta->p : nullptr, beta ? beta->dt : F32, eps, (u32x4*)a.p, (const u32x4*)w1.p, (const u32x4*)w2.p,
        (u32x4*)wp.p);
    CK(hipGetLastError());
    gemm_nt<F16>(a.ptr<uint16_t>(), wp.ptr<uint16_t>(), b1, nullptr, m, 4 * C, C, hid.ptr<uint16_t>());
    gemm_nt<F16>(hid.ptr<uint16_t>(), wp.ptr<uint16_t>() + 4 * (i64)C * C, b2, x.ptr<uint16_t>() + r0 * C, m, C, 4 * C,
                 y.ptr<uint16_t>() + r0 * C);
  }
}
}  // namespace

void convnext_mlp(const Tensor& h, const Tensor& x, const Tensor* gamma, const Tensor* beta, float eps, const Tensor& w1,
                  const Tensor* b1, const Tensor& w2, const Tensor* b2, Tensor& y) {
  REQ(h.dim() == 2 && (h.dt == BF16 || h.dt == F16), "h must be bf16/fp16 [N,C]");
  const i64 n = h.size(0);
  const int C = (int)h.size(1);
  REQ(C == 64 || C == 128 || C == 256 || C == 512 || C == 1024,
      "C=%d: the tail supports C = 64, 128 (fused) and 256, 512, 1024 (three passes)", C);
  REQ(x.dt == h.dt && x.dim() == 2 && x.size(0) == n && x.size(1) == C, "x must match h");
  REQ(y.dt == h.dt && y.dim() == 2 && y.size(0) == n && y.size(1) == C, "y must match h");
  REQ(w1.dt == h.dt && w1.dim() == 2 && w1.size(0) == 4 * C && w1.size(1) == C, "w1 must be [4C, C] of h's dtype");
  REQ(w2.dt == h.dt && w2.dim() == 2 && w2.size(0) == C && w2.size(1) == 4 * C, "w2 must be [C, 4C] of h's dtype");
  for (const Tensor* t : {gamma, beta, b2}) REQ(!t || t->numel() == C, "gamma/beta/b2 must have C elements");
  REQ(!b1 || b1->numel() == 4 * C, "b1 must have 4C elements");
  REQ((uint64_t)h.bytes() <= 0xfffe0000ull && (uint64_t)x.bytes() <= 0xfffe0000ull, "h/x larger than 4 GiB");
  REQ(((uintptr_t)h.p | (uintptr_t)x.p | (uintptr_t)y.p | (uintptr_t)w1.p | (uintptr_t)w2.p) % 16 == 0,
      "h, x, y, w1, w2 must be 16-byte aligned");
  if (n == 0) return;
  const bool f16 = h.dt == F16;
  auto wide = [&](auto Cc) {
    constexpr int W = decltype(Cc)::value;
    f16 ? mlp_wide<true, W>(h, x, gamma, beta, eps, w1, b1, w2, b2, y)
        : mlp_wide<false, W>(h, x, gamma, beta, eps, w1, b1, w2, b2, y);
  };
  if (C == 256) return wide(std::integral_constant<int, 256>{});
  if (C == 512) return wide(std::integral_constant<int, 512>{});
  if (C == 1024) return wide(std::integral_constant<int, 1024>{});
  MlpParams mp;
  const Tensor* ps[4] = {gamma, beta, b1, b2};
  for (int k = 0; k < 4; k++) {
    mp.p[k] = ps[k] ? ps[k]->p : nullptr;
    mp.dt[k] = ps[k] ? ps[k]->dt : F32;
  }
  // One 32-row block per wavefront and two wavefronts per SIMD: the SiLU (two quarter-rate operations per hidden unit) of
  // one runs beside the other's MFMAs. Two blocks per wavefront halve C = 128's weight reads from LDS, but take all
  // 512 registers and leave one wavefront per SIMD: 391007 rows 269 us against 197, 60000 rows 51 against 38.
  if (C == 64) f16 ? launch_mlp<true, 64>(h, x, w1, w2, mp, eps, y) : launch_mlp<false, 64>(h, x, w1, w2, mp, eps, y);
  else f16 ? launch_mlp<true, 128>(h, x, w1, w2, mp, eps, y) : launch_mlp<false, 128>(h, x, w1, w2, mp, eps, y);
  CK(hipGetLastError());
}
