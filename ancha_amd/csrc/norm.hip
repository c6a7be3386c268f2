// Row L2 normalisation for CDNA4 (gfx950): out[r] = x[r] / max(||x[r]||_2, 1e-12) * scale.
// Replaces `unit_norm` (crates/ancha-models/src/roformer.rs:16-24) and `SourceNorm::forward`
// (:43-54, scale = sqrt(dim) * gamma) on the GPU path, where the reference runs them as
// separate Burn ops (roformer.rs:478,497,516-519).
//
// HBM-bound: one read and one write of the row. Rows of up to 1024 channels are held in registers
// between the sum of squares (fp32, per-lane partials then a reduction) and the scaled write; longer
// ones are read a second time (from L2). Each lane reads an element before it writes it, and reads
// and writes the same elements, so out may alias x.
#include <type_traits>

#include "buffer.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace ancha {
namespace {

constexpr int kRowsPerBlock = 4;

template <bool ALIGNED>
__global__ __launch_bounds__(256) void unit_norm_kernel(NormParams p) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= p.rows) return;
  const int dim = p.dim;
  const rsrc_t xr = make_rsrc(p.x + (long)row * p.ldx, (unsigned)dim * 4);
  const rsrc_t outr = make_rsrc(p.out + (long)row * dim, (unsigned)dim * 4);
  const rsrc_t sr = make_rsrc(p.scale ? p.scale : p.out, p.scale ? (unsigned)dim * 4 : 0u);
  float ss = 0.f;
  if constexpr (ALIGNED) {
    for (int c = 4 * lane; c < dim; c += 256) {
      const float4 v = bload4<true>(xr, c * 4);
      ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
  } else {
    for (int c = lane; c < dim; c += 64) {
      const float v = bload1(xr, c * 4);
      ss += v * v;
    }
  }
  for (int o = 1; o < 64; o <<= 1) ss += __shfl_xor(ss, o);
  const float inv = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
  if constexpr (ALIGNED) {
    for (int c = 4 * lane; c < dim; c += 256) {
      float4 v = scale4(bload4<true>(xr, c * 4), inv);
      if (p.scale) {
        const float4 s = bload4<true>(sr, c * 4);
        v = make_float4(v.x * s.x, v.y * s.y, v.z * s.z, v.w * s.w);
      }
      bstore4<true>(outr, c * 4, v);
    }
  } else {
    for (int c = lane; c < dim; c += 64) {
      float v = bload1(xr, c * 4) * inv;
      if (p.scale) v *= bload1(sr, c * 4);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), outr, c * 4, 0, 0);
    }
  }
}

// Rows in registers: half a wave per row (float4s, V per lane) for aligned rows, a wave per row
// (single floats, V per lane) otherwise; U rows of each in flight, the scale read once for them.
// 96 120 x 384 with scale: 62 -> 45 us kernel time (295 MB: 6.5 TB/s, a plain copy's rate); one wave
// per row had left half the lanes of its second float4 idle at dim 384 and read the row twice.
template <bool ALIGNED, int V, int U>
__global__ __launch_bounds__(256) void unit_norm_short_kernel(NormParams p) {
  constexpr int L = ALIGNED ? 32 : 64, E = ALIGNED ? 4 : 1;  // lanes per row, floats per access
  typedef typename std::conditional<ALIGNED, float4, float>::type vec;
  const int lane = threadIdx.x & (L - 1);
  const int unit = blockIdx.x * (256 / L) + threadIdx.x / L;
  const int wave_row = (blockIdx.x * (256 / L) + (threadIdx.x & ~63) / L) * U;
  if (wave_row >= p.rows) return;
  const int dim = p.dim;
  // The wave's rows: U units of 64 / L rows, so that each access covers neighbouring rows.
  const int nrows = min(64 / L * U, p.rows - wave_row);
  const rsrc_t xr = make_rsrc(p.x + (long)wave_row * p.ldx,
                              (unsigned)(((long)(nrows - 1) * p.ldx + dim) * 4));
  const rsrc_t outr = make_rsrc(p.out + (long)wave_row * dim, (unsigned)((long)nrows * dim * 4));
  const rsrc_t sr = make_rsrc(p.scale ? p.scale : p.out, p.scale ? (unsigned)dim * 4 : 0u);
  const int sub = unit & (64 / L - 1);
  vec v[U][V];
  float ss[U] = {};
#pragma unroll
  for (int u = 0; u < U; u++) {
    const unsigned row = (unsigned)(64 / L * u + sub);
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int c = E * (lane + L * i);
      // Past the row's end: past the descriptor's too, so it reads 0.
      const unsigned off = c < dim ? (row * (unsigned)p.ldx + c) * 4 : 0x7ffffff0u;
      if constexpr (ALIGNED)
        v[u][i] = bload4<true>(xr, off);
      else
        v[u][i] = bload1(xr, off);
    }
  }
  vec s[V];
  if (p.scale)
#pragma unroll
    for (int i = 0; i < V; i++) {
      if constexpr (ALIGNED)
        s[i] = bload4<true>(sr, 4 * E * (lane + L * i));
      else
        s[i] = bload1(sr, 4 * E * (lane + L * i));
    }
#pragma unroll
  for (int u = 0; u < U; u++) {
#pragma unroll
    for (int i = 0; i < V; i++) {
      if constexpr (ALIGNED)
        ss[u] += v[u][i].x * v[u][i].x + v[u][i].y * v[u][i].y + v[u][i].z * v[u][i].z +
                 v[u][i].w * v[u][i].w;
      else
        ss[u] += v[u][i] * v[u][i];
    }
#pragma unroll
    for (int o = 1; o < L; o <<= 1) ss[u] += __shfl_xor(ss[u], o);
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    const unsigned row = (unsigned)(64 / L * u + sub);
    const float inv = 1.0f / fmaxf(sqrtf(ss[u]), 1e-12f);
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int c = E * (lane + L * i);
      if (c >= dim) continue;
      const unsigned off = (row * (unsigned)dim + c) * 4;
      if constexpr (ALIGNED) {
        float4 y = scale4(v[u][i], inv);
        if (p.scale) y = make_float4(y.x * s[i].x, y.y * s[i].y, y.z * s[i].z, y.w * s[i].w);
        bstore4<true>(outr, off, y);
      } else {
        float y = v[u][i] * inv;
        if (p.scale) y *= s[i];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, y), outr, off, 0, 0);
      }
    }
  }
}

// One wave per row: sum of squares, optional scaled unit norm written back, second norm of that
// result, fp16 normalised copy. The fp16 row is the operand every block GEMM would round its
// input to, so the GEMM then runs on fp16 x without a norm of its own. Rows of up to 512
// channels stay in registers (two float4 per lane); longer rows are read again per pass.
__device__ __forceinline__ float wave_sum(float s) {
  for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
  return s;
}

__device__ __forceinline__ float sumsq(float4 v) {
  return v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
}

__device__ __forceinline__ float4 mul4(float4 v, float a, float4 s) {
  return make_float4(v.x * a * s.x, v.y * a * s.y, v.z * a * s.z, v.w * a * s.w);
}

__device__ __forceinline__ void store_h4(rsrc_t hr, unsigned chunk, float4 v, float inv) {
  const u32x2 pk = {pack_h2(v.x * inv, v.y * inv), pack_h2(v.z * inv, v.w * inv)};
  __builtin_amdgcn_raw_buffer_store_b64(pk, hr, chunk * 8, 0, 0);
}

template <bool SHORT>
__global__ __launch_bounds__(256) void norm_half_kernel(const float* x, int rows, int dim,
                                                        const float* scale, float* y,
                                                        _Float16* h) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const unsigned bytes = (unsigned)dim * 4;
  const rsrc_t xr = make_rsrc(x + (long)row * dim, bytes);
  const rsrc_t hr = make_rsrc(h + (long)row * dim, (unsigned)dim * 2);
  const rsrc_t sr = make_rsrc(scale ? scale : x, scale ? bytes : 0u);
  const rsrc_t yr = make_rsrc(y ? y + (long)row * dim : x, y ? bytes : 0u);
  const int chunks = dim / 4;  // float4 chunks; lanes past the end read 0 and store nothing
  if constexpr (SHORT) {
    float4 v[2];
    float ss = 0.f;
    for (int i = 0; i < 2; i++) {
      v[i] = bload4<true>(xr, (lane + 64 * i) * 16);
      ss += sumsq(v[i]);
    }
    ss = wave_sum(ss);
    if (scale) {
      const float inv = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
      ss = 0.f;
      for (int i = 0; i < 2; i++) {
        v[i] = mul4(v[i], inv, bload4<true>(sr, (lane + 64 * i) * 16));
        ss += sumsq(v[i]);
        if (y) bstore4<true>(yr, (lane + 64 * i) * 16, v[i]);
      }
      ss = wave_sum(ss);
    }
    const float inv = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
    for (int i = 0; i < 2; i++) store_h4(hr, lane + 64 * i, v[i], inv);
  } else {
    float ss = 0.f;
    for (int c = lane; c < chunks; c += 64) ss += sumsq(bload4<true>(xr, c * 16));
    ss = wave_sum(ss);
    float inv = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
    if (scale) {
      // y (or, without y, only its norm) first; the fp16 pass recomputes it from x (y does
      // not alias x here).
      const float inv1 = inv;
      ss = 0.f;
      for (int c = lane; c < chunks; c += 64) {
        const float4 v = mul4(bload4<true>(xr, c * 16), inv1, bload4<true>(sr, c * 16));
        ss += sumsq(v);
        if (y) bstore4<true>(yr, c * 16, v);
      }
      ss = wave_sum(ss);
      inv = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
      for (int c = lane; c < chunks; c += 64) {
        store_h4(hr, c, mul4(bload4<true>(xr, c * 16), inv1, bload4<true>(sr, c * 16)), inv);
      }
    } else {
      for (int c = lane; c < chunks; c += 64) store_h4(hr, c, bload4<true>(xr, c * 16), inv);
    }
  }
}

// fp16 copy of n floats, 8 per thread (n % 8 == 0), rounded to nearest even as the GEMMs
// round their fp32 operands.
__global__ __launch_bounds__(256) void cast_half_kernel(const float4* x, long n8, u32x4* h) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const float4 a = x[2 * i], b = x[2 * i + 1];
  h[i] = u32x4{pack_h2(a.x, a.y), pack_h2(a.z, a.w), pack_h2(b.x, b.y), pack_h2(b.z, b.w)};
}

}  // namespace

hipError_t launch_cast_half(const float* x, long n, _Float16* h, hipStream_t stream) {
  if (n < 0 || n % 8 || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(h) & 15))
    return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  const long n8 = n / 8;
  hipLaunchKernelGGL(cast_half_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, stream,
                     reinterpret_cast<const float4*>(x), n8, reinterpret_cast<u32x4*>(h));
  return hipGetLastError();
}

hipError_t launch_norm_half(const float* x, int rows, int dim, const float* scale, float* y,
                            _Float16* h, hipStream_t stream) {
  if (dim <= 0 || dim % 4 || (dim > 512 && scale && y == x)) return hipErrorInvalidValue;
  if (rows <= 0) return hipSuccess;
  const dim3 grid((rows + kRowsPerBlock - 1) / kRowsPerBlock), block(64 * kRowsPerBlock);
  if (dim <= 512)
    hipLaunchKernelGGL(norm_half_kernel<true>, grid, block, 0, stream, x, rows, dim, scale, y, h);
  else
    hipLaunchKernelGGL(norm_half_kernel<false>, grid, block, 0, stream, x, rows, dim, scale, y, h);
  return hipGetLastError();
}

template <bool ALIGNED, int V, int U>
static void launch_short(const NormParams& p, hipStream_t stream) {
  constexpr int kRows = 256 / (ALIGNED ? 32 : 64) * U;
  hipLaunchKernelGGL((unit_norm_short_kernel<ALIGNED, V, U>), dim3((p.rows + kRows - 1) / kRows),
                     dim3(256), 0, stream, p);
}

hipError_t launch_unit_norm(const NormParams& p, bool aligned, hipStream_t stream) {
  // Rows of one wave sit behind one 32-bit descriptor (four at most).
  if (p.dim <= 1024 && p.ldx < (1l << 26)) {
    if (aligned) {
      switch ((p.dim + 127) / 128) {
        case 1: launch_short<true, 1, 2>(p, stream); break;
        case 2: launch_short<true, 2, 2>(p, stream); break;
        case 3: launch_short<true, 3, 2>(p, stream); break;
        // One row per half wave from four vectors on, with two / with one / the reading kernel below, 96 120
        // rows: dim 512 69.9 / 67.4 / 72.8 us, 640 86.5 / 84.3 / 99.4, 768 103.6 / 101.2 / 114.6, 900
        // 126.8 / 124.6 / 156.4, 1024 144.1 / 133.5 / 161.2.
        case 4: launch_short<true, 4, 1>(p, stream); break;
        case 5:
        case 6: launch_short<true, 6, 1>(p, stream); break;
        default: launch_short<true, 8, 1>(p, stream);
      }
    } else {
      // A wave per row: from 385 channels on one or two rows in flight differ by at most 4 % either way
      // (96 120 x 512 66.7 us with one, 68.1 with two; 768 99.7, 102.5; 1000 137.1, 132.5); the reading
      // kernel below takes 150.9, 220.2 and 295.4.
      switch ((p.dim + 127) / 128) {
        case 1: launch_short<false, 2, 2>(p, stream); break;
        case 2: launch_short<false, 4, 2>(p, stream); break;
        case 3: launch_short<false, 6, 2>(p, stream); break;
        case 4: launch_short<false, 8, 2>(p, stream); break;
        case 5:
        case 6: launch_short<false, 12, 1>(p, stream); break;
        default: launch_short<false, 16, 1>(p, stream);
      }
    }
    return hipGetLastError();
  }
  const dim3 grid((p.rows + kRowsPerBlock - 1) / kRowsPerBlock), block(64 * kRowsPerBlock);
  if (aligned)
    hipLaunchKernelGGL(unit_norm_kernel<true>, grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL(unit_norm_kernel<false>, grid, block, 0, stream, p);
  return hipGetLastError();
}

}  // namespace ancha
