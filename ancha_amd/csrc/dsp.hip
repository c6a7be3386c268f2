// STFT / iSTFT and chunk bookkeeping of the separation runtime on the GPU (gfx950).
//
// The reference's Stft (crates/ancha-audio/src/dsp.rs:29-134) is PyTorch's center=true STFT:
// periodic Hann window, reflect padding, unnormalised FFT of n_fft = 2048 (the only size the
// model schema allows, config.rs:58-61). Both channels of a frame go through ONE complex FFT
// (channel 0 as the real part, channel 1 as the imaginary part) and are separated with the
// conjugate symmetry of real spectra; the inverse packs them the same way. A transform runs on
// 256 threads with 8 points each, in four self-sorting passes through LDS, in fp32 with
// twiddles from a table rounded from double.
//
// Layouts: audio / chunks [2][samples]; the model spectrum [frames][bins][channel][re, im]
// (runtime.rs:161-172, the band-split input); masks [rows = 2*bins][re, im][frames] per stem
// (network.rs Roformer::forward output); frames scratch [frames][n_fft][channel].
#include "common.hpp"
#include "kernels.hpp"

namespace ancha {
namespace {

constexpr int kN = 2048;             // FFT size
constexpr int kBins = kN / 2 + 1;
constexpr int kFftThreads = 256;     // threads per transform: 8 points each

__device__ __forceinline__ long reflect(long index, long length) {
  if (length <= 1) return 0;
  const long period = 2 * (length - 1);
  long i = index % period;
  if (i < 0) i += period;
  return i < length ? i : period - i;
}

// cos / sin of 2 pi m / 2048 for every m, formed in double at compile time: Taylor series on
// [0, pi / 4], the octants by symmetry. The transforms' twiddles and the window come from here.
struct Turn {
  float c, s;
};
struct Turns {
  Turn at[kN];
};
constexpr double taylor(double x, bool sine) {
  double term = sine ? x : 1.0, sum = term;
  for (int k = sine ? 2 : 1; k < 24; k += 2) {
    term *= -x * x / (k * (k + 1));
    sum += term;
  }
  return sum;
}
constexpr Turns make_turns() {
  Turns t{};
  constexpr double pi = 3.14159265358979323846;
  for (int m = 0; m <= kN / 8; m++) {
    const float c = (float)taylor(2 * pi * m / kN, false), s = (float)taylor(2 * pi * m / kN, true);
    // Angle a = 2 pi m / 2048 in the first octant and its seven images.
    t.at[m] = {c, s};
    t.at[kN / 4 - m] = {s, c};
    t.at[kN / 4 + m] = {-s, c};
    t.at[kN / 2 - m] = {-c, s};
    t.at[kN / 2 + m] = {-c, -s};
    t.at[3 * kN / 4 - m] = {-s, -c};
    t.at[3 * kN / 4 + m] = {s, -c};
    t.at[(kN - m) & (kN - 1)] = {c, m ? -s : s};
  }
  return t;
}
// The turns in the order the threads of a transform read them: a[r][k] = r k / 64 of a turn,
// b[r][k] = r k / 512, c[r][k] = r k / 2048 (neighbouring lanes read neighbouring k: four cache
// lines per load, where the turns themselves would be strided over up to 64), and the periodic
// Hann window (dsp.rs:31-33).
struct Tables {
  Turn a[8][8], b[8][64], c[4][512];
  float hann[kN];
};
constexpr Tables make_tables() {
  const Turns t = make_turns();
  Tables w{};
  for (int r = 0; r < 8; r++) {
    for (int k = 0; k < 8; k++) w.a[r][k] = t.at[r * k * (kN / 64)];
    for (int k = 0; k < 64; k++) w.b[r][k] = t.at[r * k * (kN / 512)];
  }
  for (int r = 0; r < 4; r++)
    for (int k = 0; k < 512; k++) w.c[r][k] = t.at[r * k];
  for (int i = 0; i < kN; i++) w.hann[i] = 0.5f - 0.5f * t.at[i].c;
  return w;
}
__device__ const Tables kTables = make_tables();
__device__ __forceinline__ float hann(int i) { return kTables.hann[i]; }

struct Cpx {
  float r, i;
};
__device__ __forceinline__ Cpx operator+(Cpx a, Cpx b) { return {a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ Cpx operator-(Cpx a, Cpx b) { return {a.r - b.r, a.i - b.i}; }

// x times the turn w (SIGN +1) or its conjugate (-1).
template <int SIGN>
__device__ __forceinline__ Cpx turn(Cpx x, Turn w) {
  const float s = SIGN > 0 ? w.s : -w.s;
  return {x.r * w.c - x.i * s, x.r * s + x.i * w.c};
}
// x times i (SIGN +1) or -i (-1).
template <int SIGN>
__device__ __forceinline__ Cpx quarter(Cpx x) {
  return SIGN > 0 ? Cpx{-x.i, x.r} : Cpx{x.i, -x.r};
}

template <int SIGN>
__device__ __forceinline__ void fft4(Cpx& x0, Cpx& x1, Cpx& x2, Cpx& x3) {
  const Cpx a = x0 + x2, b = x0 - x2, c = x1 + x3, d = quarter<SIGN>(x1 - x3);
  x0 = a + c;
  x1 = b + d;
  x2 = a - c;
  x3 = b - d;
}

template <int SIGN>
__device__ __forceinline__ void fft8(Cpx (&x)[8]) {
  constexpr float h = 0.70710678118654752f;
  Cpx a[4], b[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    a[i] = x[i] + x[i + 4];
    b[i] = x[i] - x[i + 4];
  }
  b[1] = SIGN > 0 ? Cpx{h * (b[1].r - b[1].i), h * (b[1].r + b[1].i)}
                  : Cpx{h * (b[1].r + b[1].i), h * (b[1].i - b[1].r)};
  b[2] = quarter<SIGN>(b[2]);
  b[3] = SIGN > 0 ? Cpx{-h * (b[3].r + b[3].i), h * (b[3].r - b[3].i)}
                  : Cpx{h * (b[3].i - b[3].r), -h * (b[3].r + b[3].i)};
  fft4<SIGN>(a[0], a[1], a[2], a[3]);
  fft4<SIGN>(b[0], b[1], b[2], b[3]);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    x[2 * i] = a[i];
    x[2 * i + 1] = b[i];
  }
}

// LDS place of point i of a transform: one pad per 8 points keeps the strided writes of the
// first two passes (8 points, then 64, apart per lane) on distinct banks of the 64.
__device__ __forceinline__ int place(int i) { return i + (i >> 3); }
// Points of LDS per transform; 8 more than the pads need, so that the same point of neighbouring
// transforms lies 16 banks apart.
constexpr int kPlaces = kN + kN / 8 + 8;

// Twiddles of the exchange passes of thread j: radix 8 after 8 and after 64 points, and the two
// radix-4 butterflies after 512.
struct Twiddles {
  Turn a[7], b[7], c[2][3];
};
__device__ __forceinline__ void load_twiddles(Twiddles& w, int j) {
#pragma unroll
  for (int r = 1; r < 8; r++) {
    w.a[r - 1] = kTables.a[r][j & 7];
    w.b[r - 1] = kTables.b[r][j & 63];
  }
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int r = 1; r < 4; r++) w.c[h][r - 1] = kTables.c[r][j + 256 * h];
}

// Unnormalised 2048-point transform (SIGN -1 forward, +1 inverse), 256 threads with 8 points
// each: self-sorting passes of radix 8, 8, 8, 4 with one exchange through z between passes.
// Thread j brings points x[r] = point j + 256 r and leaves with the result in the same order.
// The caller's z is free at entry (a barrier behind its last use). A transform is a chain of
// exchanges and barriers, so its twiddles are read ahead of it, beside the input.
template <int SIGN>
__device__ __forceinline__ void fft2048(Cpx (&x)[8], Cpx* z, int j, const Twiddles& tw) {
  fft8<SIGN>(x);
#pragma unroll
  for (int r = 0; r < 8; r++) z[place(8 * j + r)] = x[r];
  __syncthreads();
#pragma unroll
  for (int pass = 1; pass < 3; pass++) {
    const int ns = pass == 1 ? 8 : 64, k = j & (ns - 1);
    x[0] = z[place(j)];
#pragma unroll
    for (int r = 1; r < 8; r++)
      x[r] = turn<SIGN>(z[place(j + 256 * r)], pass == 1 ? tw.a[r - 1] : tw.b[r - 1]);
    fft8<SIGN>(x);
    __syncthreads();
    const int base = (j - k) * 8 + k;
#pragma unroll
    for (int r = 0; r < 8; r++) z[place(base + ns * r)] = x[r];
    __syncthreads();
  }
  // Two radix-4 butterflies per thread: points m + 512 r for m = j and j + 256.
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int m = j + 256 * h;
    Cpx y[4];
    y[0] = z[place(m)];
#pragma unroll
    for (int r = 1; r < 4; r++) y[r] = turn<SIGN>(z[place(m + 512 * r)], tw.c[h][r - 1]);
    fft4<SIGN>(y[0], y[1], y[2], y[3]);
#pragma unroll
    for (int r = 0; r < 4; r++) x[2 * r + h] = y[r];
  }
}

// Stft::forward for both channels of one frame (dsp.rs:46-84): spectrum packed
// [frame][bin][channel][re, im]. Neighbouring frames run on one XCD (they share samples and the
// output's partial lines). 3001 frames at hop 441: 71 -> 18 us (59.8 MB, 3.3 TB/s) against the
// eleven-stage radix-2 transform with a sincospif per butterfly; of that, reading the twiddles
// in lane order (the tables above) is 28 -> 18 us.
__global__ __launch_bounds__(kFftThreads) void stft_kernel(const float* chunk, long samples,
                                                           int hop, float* spectrum) {
  __shared__ Cpx z[kPlaces];
  const int t = xcd_remap(blockIdx.x, gridDim.x), j = threadIdx.x;
  const float* x0 = chunk;
  const float* x1 = chunk + samples;
  const long base = (long)t * hop - kN / 2;
  Cpx x[8];
  Twiddles tw;
  float win[8];
  if (base >= 0 && base + kN <= samples) {
#pragma unroll
    for (int r = 0; r < 8; r++) x[r] = {x0[base + j + 256 * r], x1[base + j + 256 * r]};
  } else {
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const long src = reflect(base + j + 256 * r, samples);
      x[r] = {x0[src], x1[src]};
    }
  }
#pragma unroll
  for (int r = 0; r < 8; r++) win[r] = hann(j + 256 * r);
  load_twiddles(tw, j);
#pragma unroll
  for (int r = 0; r < 8; r++) x[r] = {x[r].r * win[r], x[r].i * win[r]};
  fft2048<-1>(x, z, j, tw);
  __syncthreads();  // the last pass has read z
#pragma unroll
  for (int r = 0; r < 8; r++) z[place(j + 256 * r)] = x[r];
  __syncthreads();
  float* out = spectrum + (long)t * kBins * 4;
  for (int k = j; k < kBins; k += kFftThreads) {
    const Cpx u = z[place(k)], n = z[place((kN - k) & (kN - 1))];
    const float a = u.r, b = u.i, c = n.r, d = -n.i;  // Z[k], conj(Z[N-k])
    float4 v;
    v.x = 0.5f * (a + c);  // channel 0: (Z[k] + conj(Z[N-k])) / 2
    v.y = 0.5f * (b + d);
    v.z = 0.5f * (b - d);  // channel 1: (Z[k] - conj(Z[N-k])) / 2i
    v.w = -0.5f * (a - c);
    *reinterpret_cast<float4*>(out + k * 4) = v;
  }
}

// Masked spectrum of one stem -> windowed inverse frames (Stft::inverse, dsp.rs:100-125,
// with the complex mask multiply of runtime.rs:190-196 first): frames [frame][n][channel].
// The masks run along the frames, the spectrum along the bins: a workgroup takes kInvFrames
// neighbouring frames and its lanes run over 16 bins x 4 frames, so that a mask row is read as
// 16-byte pieces (one frame per workgroup read every 128-byte line 32 times, one float at a
// time) and the spectrum as 256-byte pieces; neighbouring groups of frames run on one XCD, whose
// L2 then serves a mask line's other readers. 801 frames: 44 -> 17 us (27.5 us without the XCD
// order and with the twiddles read inside the passes). More frames per workgroup would read fewer
// lines, but 801 frames in fours are already only 201 workgroups.
constexpr int kInvFrames = 4;
constexpr int kInvThreads = kInvFrames * kFftThreads;
// ALIGNED: the spectrum is 16-byte aligned (else its words are read one by one).
template <bool ALIGNED>
__global__ __launch_bounds__(kInvThreads) void istft_frames_kernel(const float* spectrum,
                                                                   const float* masks,
                                                                   int frames, int zero_dc,
                                                                   float* out) {
  __shared__ Cpx z[kInvFrames][kPlaces];
  const int t0 = xcd_remap(blockIdx.x, gridDim.x) * kInvFrames;
  const int fw = threadIdx.x / kFftThreads, j = threadIdx.x % kFftThreads;  // frame, thread of it
  Twiddles tw;
  float win[8];
  {
    const int f = threadIdx.x & (kInvFrames - 1), t = t0 + f;
    const bool live = t < frames;
    const float* m = masks + t;
    const float* s = spectrum + (long)t * kBins * 4;
    auto load = [&](int k, float4& a, float4& w) {
      if constexpr (ALIGNED)
        a = *reinterpret_cast<const float4*>(s + 4 * k);
      else
        a = make_float4(s[4 * k], s[4 * k + 1], s[4 * k + 2], s[4 * k + 3]);
      const float* row = m + (long)(4 * k) * frames;
      w = make_float4(row[0], row[frames], row[2 * (long)frames], row[3 * (long)frames]);
    };
    // Z = X0 + i X1 at k and, by conjugate symmetry of X0 and X1, at N - k.
    auto put = [&](int k, float4 a, float4 w) {
      float r0 = a.x * w.x - a.y * w.y, i0 = a.x * w.y + a.y * w.x;
      float r1 = a.z * w.z - a.w * w.w, i1 = a.z * w.w + a.w * w.z;
      if (k == 0 || k == kBins - 1) i0 = i1 = 0.0f;
      if (k == 0 && zero_dc) r0 = r1 = 0.0f;
      z[f][place(k)] = {r0 - i1, i0 + r1};
      if (k > 0 && k < kN / 2) z[f][place(kN - k)] = {r0 + i1, r1 - i0};
    };
    constexpr int kSteps = kN / 2 / (kInvThreads / kInvFrames);  // bins 0 .. 1023
    const int k0 = threadIdx.x / kInvFrames;
    float4 a[kSteps], w[kSteps];
    if (live) {
#pragma unroll
      for (int i = 0; i < kSteps; i++) load(k0 + i * (kInvThreads / kInvFrames), a[i], w[i]);
    }
    load_twiddles(tw, j);
#pragma unroll
    for (int r = 0; r < 8; r++) win[r] = hann(j + 256 * r) * (1.0f / kN);  // a power of two: exact
    if (live) {
#pragma unroll
      for (int i = 0; i < kSteps; i++) put(k0 + i * (kInvThreads / kInvFrames), a[i], w[i]);
      if (k0 == 0) {
        load(kN / 2, a[0], w[0]);
        put(kN / 2, a[0], w[0]);
      }
    }
  }
  __syncthreads();
  Cpx x[8];
#pragma unroll
  for (int r = 0; r < 8; r++) x[r] = z[fw][place(j + 256 * r)];
  __syncthreads();
  fft2048<1>(x, z[fw], j, tw);
  if (t0 + fw >= frames) return;
  float2* o = reinterpret_cast<float2*>(out) + (long)(t0 + fw) * kN;
#pragma unroll
  for (int r = 0; r < 8; r++)
    o[j + 256 * r] = make_float2(x[r].r * win[r], x[r].i * win[r]);
}

// Overlap-add of the inverse frames divided by the summed squared window (dsp.rs:118-132),
// samples [n/2, n/2 + length) of the chunk, then the fade-weighted accumulation of the chunk
// into the clip sums (ChunkPlan::weight + Accumulator::add, chunk.rs:27-73).
// sums [2][total], weights [total] (updated only when `count_weight`). FRESH: sums is written,
// not added to (one chunk covering all of it). I: the index type, 32-bit where every sample
// index of the chunk fits (a 64-bit division by hop is a long sequence of instructions).
template <typename I, bool FRESH>
__global__ void ola_accumulate_kernel(const float* frames_buf, int frames, int hop,
                                      long length, long start, long total, int first, int last,
                                      int count_weight, float* sums, float* weights,
                                      unsigned* flags) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= length) return;
  const long pos = start + i;
  const I j = (I)i + kN / 2, h = (I)hop;
  I t0 = j >= kN ? (j - kN) / h + 1 : 0;  // the first frame with t hop > j - n
  I t1 = j / h;
  if (t1 > (I)(frames - 1)) t1 = (I)(frames - 1);
  const float2* buf = reinterpret_cast<const float2*>(frames_buf);
  float a0 = 0.0f, a1 = 0.0f, den = 0.0f;
  for (I t = t0; t <= t1; t++) {
    const int o = (int)(j - t * h);
    const float w = hann(o);
    const float2 v = buf[(long)t * kN + o];
    a0 += v.x;
    a1 += v.y;
    den += w * w;
  }
  const float y0 = a0 / den, y1 = a1 / den;
  // Every sample of the chunk is checked, also those past the clip's end, which are not
  // accumulated (Stft::inverse and Accumulator::add check whole planes).
  if (flags) {
    if (!(den > 1e-11f)) raise_flag(flags, kFlagIstftUncovered);
    if (non_finite(y0) || non_finite(y1)) raise_flag(flags, kFlagChunk);
  }
  if (pos >= total) return;
  const long fade = length / 10 > 1 ? length / 10 : 1;
  float wt = 1.0f;
  if (!first && i < fade) wt = (float)(i + 1) / (float)fade;
  if (!last && i >= length - fade) wt = (float)(length - i) / (float)fade;
  if constexpr (FRESH) {
    sums[pos] = wt * y0;
    sums[total + pos] = wt * y1;
  } else {
    sums[pos] += wt * y0;
    sums[total + pos] += wt * y1;
  }
  if (count_weight) weights[pos] += wt;
}

// Chunk extraction of runtime.rs:118-136: reflect-bordered samples of the clip.
__global__ void chunk_gather_kernel(const float* audio, long n, long start, long border,
                                    long remaining, long samples, float* chunk,
                                    unsigned* flags) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= samples) return;
  float v0 = 0.0f, v1 = 0.0f;
  if (!(i >= remaining && remaining <= samples / 2)) {
    const long local = i < remaining ? i : reflect(i, remaining);
    const long src = reflect(start + local - border, n);
    v0 = audio[src];
    v1 = audio[n + src];
  }
  if (flags && (non_finite(v0) || non_finite(v1))) raise_flag(flags, kFlagInput);
  chunk[i] = v0;
  chunk[samples + i] = v1;
}

// Accumulator::finish + border crop (chunk.rs:75-88, runtime.rs:215-223); optionally the
// residual input - stem (runtime.rs:403-420).
__global__ void finish_kernel(const float* sums, const float* weights, long total, long border,
                              long n, const float* audio, float* out, float* residual,
                              unsigned* flags) {
  // One thread per accumulator sample: every weight is checked (Accumulator::finish), the
  // samples of the cropped clip [border, border + n) are written.
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const float w = weights[idx];
  if (flags && !(w > 0.0f)) raise_flag(flags, kFlagOlaUncovered);
  const long i = idx - border;
  if (i < 0 || i >= n) return;
  for (int c = 0; c < 2; c++) {
    const float y = sums[c * total + border + i] / w;
    out[c * n + i] = y;
    if (residual) residual[c * n + i] = audio[c * n + i] - y;
  }
}

__global__ void zero_kernel(float* p, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}

inline unsigned blocks_for(long n, int threads) { return (unsigned)((n + threads - 1) / threads); }

}  // namespace

hipError_t launch_stft(const float* chunk, long samples, int hop, float* spectrum,
                       hipStream_t stream) {
  const int frames = (int)(samples / hop + 1);
  hipLaunchKernelGGL(stft_kernel, dim3(frames), dim3(kFftThreads), 0, stream, chunk, samples, hop,
                     spectrum);
  return hipGetLastError();
}

hipError_t launch_istft_frames(const float* spectrum, const float* masks, int frames, int zero_dc,
                               float* frames_buf, hipStream_t stream) {
  const dim3 grid((frames + kInvFrames - 1) / kInvFrames), block(kInvThreads);
  if (reinterpret_cast<uintptr_t>(spectrum) & 15)
    hipLaunchKernelGGL(istft_frames_kernel<false>, grid, block, 0, stream, spectrum, masks, frames,
                       zero_dc, frames_buf);
  else
    hipLaunchKernelGGL(istft_frames_kernel<true>, grid, block, 0, stream, spectrum, masks, frames,
                       zero_dc, frames_buf);
  return hipGetLastError();
}

hipError_t launch_ola_accumulate(const float* frames_buf, int frames, int hop, long length,
                                 long start, long total, bool first, bool last, bool count_weight,
                                 bool fresh, float* sums, float* weights, unsigned* flags,
                                 hipStream_t stream) {
  const bool narrow = length < (1L << 31) - 2 * kN;
  const auto kernel = fresh ? (narrow ? ola_accumulate_kernel<unsigned, true>
                                      : ola_accumulate_kernel<long, true>)
                            : (narrow ? ola_accumulate_kernel<unsigned, false>
                                      : ola_accumulate_kernel<long, false>);
  hipLaunchKernelGGL(kernel, dim3(blocks_for(length, 256)), dim3(256), 0, stream, frames_buf,
                     frames, hop, length, start, total, (int)first, (int)last, (int)count_weight,
                     sums, weights, flags);
  return hipGetLastError();
}

hipError_t launch_chunk_gather(const float* audio, long n, long start, long border,
                               long remaining, long samples, float* chunk, unsigned* flags,
                               hipStream_t stream) {
  hipLaunchKernelGGL(chunk_gather_kernel, dim3(blocks_for(samples, 256)), dim3(256), 0, stream,
                     audio, n, start, border, remaining, samples, chunk, flags);
  return hipGetLastError();
}

hipError_t launch_finish(const float* sums, const float* weights, long total, long border, long n,
                         const float* audio, float* out, float* residual, unsigned* flags,
                         hipStream_t stream) {
  hipLaunchKernelGGL(finish_kernel, dim3(blocks_for(total, 256)), dim3(256), 0, stream, sums, weights,
                     total, border, n, audio, out, residual, flags);
  return hipGetLastError();
}

hipError_t launch_zero(float* p, long n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(zero_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, stream, p, n);
  return hipGetLastError();
}

}  // namespace ancha
