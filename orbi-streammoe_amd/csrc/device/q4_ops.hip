// q4_ops.hip -- standalone gfx950 kernels behind the reference's single-op
// surface: affine q4 dequant (shaders/q4_dequant.comp), q4 GEMV
// (shaders/q4_gemv.comp), nibble unpack, SwiGLU (shaders/swiglu.comp),
// weighted accumulate (shaders/weighted_accumulate.comp) and RMSNorm
// (shaders/rmsnorm.comp). These serve arbitrary shapes and any group size;
// the routed-MoE hot path uses the fused kernels in moe_decode.hip.
#include "device_common.hpp"

namespace {

using namespace osmk;

// One thread per packed word; each writes its 8 dequantized columns. The
// value is rounded as the reference rounds it (src/cpu/reference_ops.cpp:57-59):
// scale*q first, then + bias, with no fused multiply-add.
template <int META>
__global__ void q4_dequant_kernel(const uint32_t* __restrict__ packed,
                                  const void* __restrict__ scales,
                                  const void* __restrict__ biases, uint32_t rows,
                                  uint32_t packed_cols, uint32_t group,
                                  float* __restrict__ out) {
#pragma clang fp contract(off)
  const size_t total = static_cast<size_t>(rows) * packed_cols;
  const uint32_t groups = packed_cols * 8u / group;
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t wi = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; wi < total;
       wi += stride) {
    const uint32_t r = static_cast<uint32_t>(wi / packed_cols);
    const uint32_t wc = static_cast<uint32_t>(wi - static_cast<size_t>(r) * packed_cols);
    const uint32_t w = packed[wi];
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t col = wc * 8u + j;
      const size_t gi = static_cast<size_t>(r) * groups + col / group;
      const float q = static_cast<float>((w >> (4 * j)) & 0xFu);
      const float prod = meta_at<META>(scales, gi) * q;
      v[j] = prod + meta_at<META>(biases, gi);
    }
    float4* o = reinterpret_cast<float4*>(out + wi * 8u);
    o[0] = make_float4(v[0], v[1], v[2], v[3]);
    o[1] = make_float4(v[4], v[5], v[6], v[7]);
  }
}

// One wavefront per output row, lanes striding over packed words. When a word
// lies inside one group the reference GEMV algebra applies
// (shaders/q4_gemv.comp:42-59): scale * sum(q*x) + bias * sum(x); otherwise
// each nibble is dequantized and multiplied.
template <int META>
__global__ void q4_gemv_kernel(const uint32_t* __restrict__ packed,
                               const void* __restrict__ scales,
                               const void* __restrict__ biases, uint32_t out_dim,
                               uint32_t packed_cols, uint32_t group,
                               const float* __restrict__ x, float* __restrict__ y) {
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t row = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (row >= out_dim) return;
  const uint32_t groups = packed_cols * 8u / group;
  const uint32_t* prow = packed + static_cast<size_t>(row) * packed_cols;
  const size_t gbase = static_cast<size_t>(row) * groups;
  float acc = 0.0f;
  if (group % 8u == 0u) {
    for (uint32_t w = lane; w < packed_cols; w += kWave) {
      const uint32_t col0 = w * 8u;
      const float* xc = x + col0;
      float xs = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) xs += xc[j];
      const size_t gi = gbase + col0 / group;
      acc += meta_at<META>(scales, gi) * nib_dot8(prow[w], xc) + meta_at<META>(biases, gi) * xs;
    }
  } else {
    for (uint32_t w = lane; w < packed_cols; w += kWave) {
      const uint32_t word = prow[w];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t col = w * 8u + j;
        const size_t gi = gbase + col / group;
        const float q = static_cast<float>((word >> (4 * j)) & 0xFu);
        acc += (meta_at<META>(scales, gi) * q + meta_at<META>(biases, gi)) * x[col];
      }
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) y[row] = acc;
}

// nib_dot8 of a word by the two in-place masks of nib_dot32, four products to
// a chain.
__device__ __forceinline__ float nib_dot8_masks(uint32_t w, const float* x) {
  const uint32_t t = w >> 8;
  const uint32_t p0 = w & 0x000F000Fu, p1 = w & 0x00F000F0u;
  const uint32_t p2 = t & 0x000F000Fu, p3 = t & 0x00F000F0u;
  float a = fmaf(f16_lo(p0), x[0], opaque_zero());
  float b = fmaf(f16_lo(p1), x[1], opaque_zero());
  a = fmaf(f16_lo(p2), x[2], a);
  b = fmaf(f16_lo(p3), x[3], b);
  a = fmaf(f16_hi(p0), x[4], a);
  b = fmaf(f16_hi(p1), x[5], b);
  a = fmaf(f16_hi(p2), x[6], a);
  b = fmaf(f16_hi(p3), x[7], b);
  return fmaf(b, kTwo20, a * kTwo24);
}

// The same GEMV for rows of whole 16-byte chunks (32 columns, each inside one
// group): LPR lanes share a row, a lane takes chunks c, c + LPR, ..., and a
// wavefront keeps RPW x (64 / LPR) rows in flight. x is staged in LDS, LPR
// chunks at a time and 36 floats apart so that the lanes' 16-byte reads
// spread over the banks, and read back once for all of a wavefront's rows.
// Bound by the latency of one round of loads up to a few MB of weights (a
// launch that does nothing takes 2.3 µs), then by the loads in flight. µs a
// launch, word-wise kernel above / this one, kernel trace: 640 x 2048 f32
// metadata 3.96 / 2.96, 4096 x 2048 f32 5.68 / 4.32, 1000 x 4992 bf16 8.28 /
// 5.44, 16384 x 2048 bf16 12.5 / 7.8, 16384 x 5120 f32 27.6 / 16.7 (3.1 TB/s).
// Loading the next chunks before multiplying these measured 7.0 and 16.3 at
// the two largest, and spilled at one row per wavefront.
template <int META, int LPR, int RPW>
__global__ __launch_bounds__(256) void q4_gemv_chunks_kernel(const uint32_t* __restrict__ packed,
                                                             const void* __restrict__ scales,
                                                             const void* __restrict__ biases, uint32_t out_dim,
                                                             uint32_t packed_cols, uint32_t group,
                                                             const float* __restrict__ x, float* __restrict__ y) {
  constexpr uint32_t kStep = kWave / LPR;  // rows side by side in a wavefront
  constexpr uint32_t kStride = 36;
  __shared__ __align__(16) float xs[LPR * kStride];
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t c0 = lane % LPR;
  const uint32_t r0 = (blockIdx.x * 4u + threadIdx.x / kWave) * (kStep * RPW) + lane / LPR;
  const uint32_t nch = packed_cols / 4u, groups = packed_cols * 8u / group;
  float acc[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) acc[i] = 0.0f;
  for (uint32_t cb = 0; cb < nch; cb += LPR) {
    // Lanes past the row's end and rows past the last read the last chunk or
    // row again; their values are not added, or not stored.
    const uint32_t cc = cb + c0 < nch ? cb + c0 : nch - 1u;
    const uint32_t g = cc * 32u / group;
    uint4 q[RPW];
    uint32_t sb[RPW], bb[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const uint32_t r = r0 + i * kStep < out_dim ? r0 + i * kStep : out_dim - 1u;
      q[i] = ldg16(packed + (static_cast<size_t>(r) * nch + cc) * 4u);
      const size_t gi = static_cast<size_t>(r) * groups + g;
      sb[i] = meta_bits<META>(scales, gi);
      bb[i] = meta_bits<META>(biases, gi);
    }
    if (cb > 0u) __syncthreads();  // the previous chunks are read
    const float4* x4 = reinterpret_cast<const float4*>(x) + cb * 8u;
    const uint32_t n4 = (nch - cb) * 8u;
    for (uint32_t f = threadIdx.x; f < LPR * 8u; f += 256u)
      *reinterpret_cast<float4*>(xs + (f / 8u) * kStride + (f % 8u) * 4u) =
          f < n4 ? x4[f] : make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    float xr[32];
    const float4* xl = reinterpret_cast<const float4*>(xs + c0 * kStride);
    float xsum[4];  // of each word's columns
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const float4 f = xl[v];
      xr[4 * v] = f.x; xr[4 * v + 1] = f.y; xr[4 * v + 2] = f.z; xr[4 * v + 3] = f.w;
      const float s4 = (f.x + f.y) + (f.z + f.w);
      xsum[v / 2] = v % 2 ? xsum[v / 2] + s4 : s4;
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      // Scale and bias per word, as the word-wise kernel adds them: their
      // products largely cancel, and summed over 32 columns first they leave
      // a larger error.
      const float sc = meta_widen<META>(sb[i]), bi = meta_widen<META>(bb[i]);
      const uint32_t w4[4] = {q[i].x, q[i].y, q[i].z, q[i].w};
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) v += sc * nib_dot8_masks(w4[k], xr + 8 * k) + bi * xsum[k];
      acc[i] += cb + c0 < nch ? v : 0.0f;
    }
  }
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    float v = acc[i];
    if constexpr (LPR == 64)
      v = wave_sum(v);
    else if constexpr (LPR == 32)
      v = group_sum(v, 32);
    else
      v = row_sum<LPR>(v);
    const uint32_t r = r0 + i * kStep;
    if (c0 == 0u && r < out_dim) y[r] = v;
  }
}

__global__ void unpack_kernel(const uint32_t* __restrict__ packed, size_t words,
                              uint8_t* __restrict__ out) {
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += stride) {
    // Byte j of the 8-byte output is nibble j of the word, low nibble first.
    const uint32_t w = packed[i];
    uint32_t b0 = 0, b1 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      b0 |= ((w >> (4 * j)) & 0xFu) << (8 * j);
      b1 |= ((w >> (4 * j + 16)) & 0xFu) << (8 * j);
    }
    reinterpret_cast<uint2*>(out)[i] = make_uint2(b0, b1);
  }
}

__global__ void swiglu_kernel(const float* __restrict__ g, const float* __restrict__ u,
                              float* __restrict__ out, size_t n) {
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = silu_mul(g[i], u[i]);
}

// acc[i] += weight * src[i], rounded as the reference's scalar loop rounds.
__global__ void weighted_accumulate_kernel(const float* __restrict__ src, float weight,
                                           float* __restrict__ acc, size_t n) {
#pragma clang fp contract(off)
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    acc[i] = acc[i] + weight * src[i];
}

// One workgroup per row: block-wide sum of squares, then
// v * (1/sqrt(mean + eps) * w) (reference_ops.cpp:112-127).
__global__ void rms_norm_kernel(const float* __restrict__ in, const float* __restrict__ w,
                                float* __restrict__ out, uint32_t dim, float eps) {
  __shared__ float partial[16];
  __shared__ float scale_s;
  const float* row = in + static_cast<size_t>(blockIdx.x) * dim;
  float* orow = out + static_cast<size_t>(blockIdx.x) * dim;
  float ss = 0.0f;
  for (uint32_t i = threadIdx.x; i < dim; i += blockDim.x) ss += row[i] * row[i];
  ss = wave_sum(ss);
  const uint32_t wave = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) partial[wave] = ss;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (uint32_t i = 0; i < blockDim.x / kWave; ++i) t += partial[i];
    scale_s = 1.0f / sqrtf(t / static_cast<float>(dim) + eps);
  }
  __syncthreads();
  const float scale = scale_s;
  for (uint32_t i = threadIdx.x; i < dim; i += blockDim.x)
    orow[i] = row[i] * (scale * (w ? w[i] : 1.0f));
}

unsigned grid_for(size_t n, unsigned block) {
  size_t g = (n + block - 1) / block;
  if (g == 0) g = 1;
  if (g > 65535u * 4u) g = 65535u * 4u;
  return static_cast<unsigned>(g);
}

// ---- affine q4 quantizer (src/conversion/single_expert_pilot.cpp:276-358) --
// Pass 1, one thread per (row, group): min, max, scale = range / 15 (1 when
// flat), bias = min, the group's error bound (scale * 0.5001 + 1e-6, or 1e-6
// when flat); flags bit 0 marks a non-finite weight. Pass 2, one
// thread per packed word: q = clamp(round-half-away((v - bias) / scale), 0,
// 15) per nibble (an overflowed range gives NaN, mapped to 0), the
// reconstruction error against the group bound (flags bit 1), and per-block
// error maximum and sum for the statistics. Every operation rounds on its
// own, as the reference's scalar loop does.
constexpr int kQuantThreads = 256;

__global__ void quant_groups_kernel(const float* __restrict__ v, size_t rows, size_t cols, size_t group,
                                    float* __restrict__ scales, float* __restrict__ biases,
                                    float* __restrict__ bounds, uint32_t* __restrict__ flags) {
#pragma clang fp contract(off)
  const size_t groups = cols / group;
  const size_t n = rows * groups;
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float* g = v + (i / groups) * cols + (i % groups) * group;
    float lo = INFINITY, hi = -INFINITY;
    bool finite = true;
    for (size_t j = 0; j < group; ++j) {
      const float x = g[j];
      finite = finite && isfinite(x);
      lo = fminf(lo, x);
      hi = fmaxf(hi, x);
    }
    if (!finite) atomicOr(flags, 1u);
    const float range = hi - lo;
    const float scale = range > 0.0f ? range / 15.0f : 1.0f;
    scales[i] = scale;
    biases[i] = lo;
    bounds[i] = range > 0.0f ? scale * 0.5001f + 1e-6f : 1e-6f;
  }
}

__global__ __launch_bounds__(kQuantThreads) void quant_pack_kernel(
    const float* __restrict__ v, size_t rows, size_t cols, size_t group,
    const float* __restrict__ scales, const float* __restrict__ biases,
    const float* __restrict__ bounds, uint32_t* __restrict__ packed,
    float* __restrict__ block_max, double* __restrict__ block_sum, uint32_t* __restrict__ flags) {
#pragma clang fp contract(off)
  __shared__ float smax[kQuantThreads];
  __shared__ double ssum[kQuantThreads];
  const size_t words_per_row = cols / 8u;
  const size_t groups = cols / group;
  const size_t n = rows * words_per_row;
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  float worst = 0.0f;
  double total = 0.0;
  bool over = false;
  for (size_t w = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; w < n; w += stride) {
    const size_t row = w / words_per_row;
    const size_t col0 = (w % words_per_row) * 8u;
    uint32_t word = 0u;
    for (uint32_t lane = 0; lane < 8u; ++lane) {
      const size_t col = col0 + lane;
      const size_t gi = row * groups + col / group;
      const float scale = scales[gi];
      const float bias = biases[gi];
      const float x = v[row * cols + col];
      const float t = (x - bias) / scale;
      const int r = isnan(t) ? 0 : static_cast<int>(fminf(fmaxf(roundf(t), -1.0f), 16.0f));
      const uint32_t q = static_cast<uint32_t>(r < 0 ? 0 : (r > 15 ? 15 : r));
      word |= q << (4u * lane);
      const float err = fabsf(scale * static_cast<float>(q) + bias - x);
      over = over || err > bounds[gi];
      worst = fmaxf(worst, err);
      total += static_cast<double>(err);
    }
    packed[w] = word;
  }
  if (over) atomicOr(flags, 2u);
  smax[threadIdx.x] = worst;
  ssum[threadIdx.x] = total;
  __syncthreads();
  for (int h = kQuantThreads / 2; h > 0; h >>= 1) {
    if (static_cast<int>(threadIdx.x) < h) {
      smax[threadIdx.x] = fmaxf(smax[threadIdx.x], smax[threadIdx.x + h]);
      ssum[threadIdx.x] += ssum[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    block_max[blockIdx.x] = smax[0];
    block_sum[blockIdx.x] = ssum[0];
  }
}

// Below this many packed words the word-wise kernel is as fast: its loads
// leave at once, without the barrier (µs, word-wise / chunks: 256 x 512 and
// 512 x 512 2.32 / 2.52, 2048 x 512 2.76 / 2.72; 640 x 2048 3.96 / 2.96).
constexpr uint64_t kGemvChunksMinWords = 1u << 17;

template <int META, int LPR, int RPW>
int launch_gemv_chunks(const osmd_q4_proj& p, const float* x, float* y, hipStream_t st) {
  constexpr uint32_t rows = 4u * (kWave / LPR) * RPW;  // per workgroup
  q4_gemv_chunks_kernel<META, LPR, RPW><<<(p.out_dim + rows - 1u) / rows, 256, 0, st>>>(
      p.packed, p.scales, p.biases, p.out_dim, p.packed_cols, p.group, x, y);
  return launch_status();
}

// Rows per wavefront: as many as leave 2,048 wavefronts, two to a SIMD.
template <int META, int LPR>
int launch_gemv_lanes(const osmd_q4_proj& p, const float* x, float* y, hipStream_t st) {
  const uint64_t waves = (static_cast<uint64_t>(p.out_dim) * LPR + kWave - 1u) / kWave;
  if (waves >= 4u * 2048u) return launch_gemv_chunks<META, LPR, 4>(p, x, y, st);
  if (waves >= 2u * 2048u) return launch_gemv_chunks<META, LPR, 2>(p, x, y, st);
  return launch_gemv_chunks<META, LPR, 1>(p, x, y, st);
}

template <int META>
int launch_gemv(const osmd_q4_proj& p, const float* x, float* y, hipStream_t st) {
  const uint64_t words = static_cast<uint64_t>(p.out_dim) * p.packed_cols;
  if (words >= kGemvChunksMinWords && p.packed_cols % 4u == 0u && p.group % 32u == 0u &&
      ((reinterpret_cast<uintptr_t>(p.packed) | reinterpret_cast<uintptr_t>(x)) & 15u) == 0u) {
    const uint32_t nch = p.packed_cols / 4u;
    if (nch <= 16u) return launch_gemv_lanes<META, 16>(p, x, y, st);
    if (nch <= 32u) return launch_gemv_lanes<META, 32>(p, x, y, st);
    return launch_gemv_lanes<META, 64>(p, x, y, st);
  }
  q4_gemv_kernel<META><<<(p.out_dim + 3u) / 4u, 256, 0, st>>>(p.packed, p.scales, p.biases, p.out_dim, p.packed_cols,
                                                             p.group, x, y);
  return launch_status();
}

}  // namespace

extern "C" {

int osmd_q4_dequant(const osmd_q4_proj* p, float* out, osmd_stream s) {
  const hipStream_t st = static_cast<hipStream_t>(s);
  const size_t words = static_cast<size_t>(p->out_dim) * p->packed_cols;
  const unsigned grid = grid_for(words, 256);
  switch (p->meta_dtype) {
    case OSM_META_F32:
      q4_dequant_kernel<OSM_META_F32><<<grid, 256, 0, st>>>(p->packed, p->scales, p->biases, p->out_dim, p->packed_cols, p->group, out);
      break;
    case OSM_META_F16:
      q4_dequant_kernel<OSM_META_F16><<<grid, 256, 0, st>>>(p->packed, p->scales, p->biases, p->out_dim, p->packed_cols, p->group, out);
      break;
    default:
      q4_dequant_kernel<OSM_META_BF16><<<grid, 256, 0, st>>>(p->packed, p->scales, p->biases, p->out_dim, p->packed_cols, p->group, out);
      break;
  }
  return launch_status();
}

int osmd_q4_gemv(const osmd_q4_proj* p, const float* x, float* y, osmd_stream s) {
  const hipStream_t st = static_cast<hipStream_t>(s);
  switch (p->meta_dtype) {
    case OSM_META_F32: return launch_gemv<OSM_META_F32>(*p, x, y, st);
    case OSM_META_F16: return launch_gemv<OSM_META_F16>(*p, x, y, st);
    default: return launch_gemv<OSM_META_BF16>(*p, x, y, st);
  }
}

int osmd_unpack_nibbles(const uint32_t* packed, size_t words, uint8_t* out, osmd_stream s) {
  unpack_kernel<<<grid_for(words, 256), 256, 0, static_cast<hipStream_t>(s)>>>(packed, words, out);
  return launch_status();
}

int osmd_swiglu(const float* gate, const float* up, float* out, size_t n, osmd_stream s) {
  swiglu_kernel<<<grid_for(n, 256), 256, 0, static_cast<hipStream_t>(s)>>>(gate, up, out, n);
  return launch_status();
}

int osmd_weighted_accumulate(const float* src, float weight, float* acc, size_t n, osmd_stream s) {
  weighted_accumulate_kernel<<<grid_for(n, 256), 256, 0, static_cast<hipStream_t>(s)>>>(src, weight, acc, n);
  return launch_status();
}

int osmd_rms_norm(const float* in, const float* weight, float* out, uint32_t rows, uint32_t dim,
                  float eps, osmd_stream s) {
  rms_norm_kernel<<<rows, 256, 0, static_cast<hipStream_t>(s)>>>(in, weight, out, dim, eps);
  return launch_status();
}

unsigned osmd_q4_quantize_blocks(size_t rows, size_t cols) {
  const size_t words = rows * (cols / 8u);
  size_t b = (words + kQuantThreads - 1) / kQuantThreads;
  if (b == 0) b = 1;
  if (b > 2048) b = 2048;
  return static_cast<unsigned>(b);
}

int osmd_q4_quantize(const float* values, size_t rows, size_t cols, size_t group, uint32_t* packed,
                     float* scales, float* biases, float* bounds, float* block_max, double* block_sum,
                     uint32_t* flags, osmd_stream s) {
  const hipStream_t st = static_cast<hipStream_t>(s);
  const size_t ngroups = rows * (cols / group);
  size_t gb = (ngroups + 255) / 256;
  if (gb > 4096) gb = 4096;
  quant_groups_kernel<<<static_cast<unsigned>(gb), 256, 0, st>>>(values, rows, cols, group, scales, biases,
                                                                 bounds, flags);
  quant_pack_kernel<<<osmd_q4_quantize_blocks(rows, cols), kQuantThreads, 0, st>>>(
      values, rows, cols, group, scales, biases, bounds, packed, block_max, block_sum, flags);
  return launch_status();
}

}  // extern "C"
