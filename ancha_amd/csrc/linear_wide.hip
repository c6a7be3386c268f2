// Projection GEMM with the weight laid out once per call: out = epilogue(x . w), the operation and
// the rounding points of linear.hip (fp32 operands in HBM, fp16 MFMA operands, fp32 accumulation;
// crates/ancha-models/src/fused/gemm.rs:46-211), for calls that bring scratch for the weight.
//
// linear.hip converts its fp32 weight tile again for every 128 rows, reads x again for every 128
// columns, and pays one memory latency per 64 k. Here a small first kernel (2-5 us) writes w as fp16
// in fragment-major order (one contiguous kilobyte per 32-column x 16-k MFMA operand), so a wave's
// weight operand is one coalesced load with no conversion and no LDS. Then, on D[column][row] =
// W^T . x^T of v_mfma_f32_32x32x16_f16:
//   resident (many columns, k <= 512): the row block's whole k in LDS, the 8 waves walk the columns;
//   stream   (otherwise): 32 - 128 rows x 128 - 512 columns in accumulators, x streamed through LDS.
// Both share one epilogue: a 32 x 32 tile goes through 4 KB of LDS of its wave, so that residual,
// rotary table and output are read and written as whole 128-byte row pieces.
//
// Measured, whole call, linear.hip -> here: 96 120 x 384 -> 1664 with norm, bias and rotary 517 ->
// 216 us (788 MB of operands: 3.6 TB/s); 18 060 x 1536 -> 384 with bias and residual 74 -> 47 us;
// 96 120 x 1536 -> 384 331 -> 216 us; 300 x 1536 -> 384 40 -> 14 us; 32 x 384 -> 1664 20 -> 8 us
// (the last two kernel time). What bounds the large ones is the epilogue's output and table traffic
// and, in the resident form, three rounds of loading, walking and draining a row block.
#include "buffer.hpp"
#include "common.hpp"
#include "gemm.hpp"
#include "kernels.hpp"

namespace ancha {
namespace {

constexpr int kFrag = 1024;   // bytes of one 32-column (or 32-row) x 16-k fp16 fragment
constexpr int kStage = 4096;  // epilogue staging of a wave: 32 rows x 32 fp32 columns

// ---- w fp32 [k][m] -> fp16 fragments: fragment (b, s) at (s * m / 32 + b) * 1 KB, lane l's eight
// halves = w[16 s + 8 (l / 32) + t][32 b + l % 32]. One wave per fragment.
__global__ __launch_bounds__(256) void weight_fragments_kernel(const float* w, int k, int m,
                                                               u32x4* frag) {
  const int lane = threadIdx.x & 63;
  const int steps = k / 16;
  const int f = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (f >= (m / 32) * steps) return;
  const int s = f / (m / 32), b = f - s * (m / 32);
  const rsrc_t wr = make_rsrc(w + (long)16 * s * m + 32 * b, (unsigned)(15 * m + 32) * 4);
  float v[8];
#pragma unroll
  for (int t = 0; t < 8; t++)
    v[t] = bload1(wr, (unsigned)((8 * (lane >> 5) + t) * m + (lane & 31)) * 4);
  frag[(long)f * 64 + lane] =
      u32x4{pack_h2(v[0], v[1]), pack_h2(v[2], v[3]), pack_h2(v[4], v[5]), pack_h2(v[6], v[7])};
}

__device__ __forceinline__ float sumsq4(float4 v) {
  return v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
}

// Operand rows in LDS: fragment (jb, s) = rows 32 jb .. + 31, k 16 s .. + 15, two 512-byte halves of
// eight k; row r of a half sits in 16-byte slot r ^ (its eight-k chunk % 8). Sixteen lanes that
// write one row's 64 k (read from HBM as 256 contiguous bytes) then fall on eight slots, not one.
__device__ __forceinline__ int slot_offset(int r, int kc) {
  return (kc >> 1) * kFrag + (kc & 1) * 512 + (((r & 31) ^ (kc & 7)) << 4);
}

__device__ __forceinline__ u32x2 pack4(float4 a) {
  return u32x2{pack_h2(a.x, a.y), pack_h2(a.z, a.w)};
}

// Descriptors of a row block's epilogue operands (absent ones are empty).
struct Rows {
  rsrc_t out, residual, bias, rope;
};

__device__ __forceinline__ Rows row_descriptors(const LinearParams& p, int row0, int nrows) {
  Rows d;
  const unsigned span = (unsigned)((long)nrows * p.m * 4);
  d.out = make_rsrc(p.out + (long)row0 * p.m, span);
  d.residual = make_rsrc(p.residual ? p.residual + (long)row0 * p.m : p.out, p.residual ? span : 0u);
  d.bias = make_rsrc(p.bias ? p.bias : p.out, p.bias ? (unsigned)p.m * 4 : 0u);
  d.rope = make_rsrc(p.rope ? p.rope : p.out, p.rope ? (unsigned)p.tokens * 1024 : 0u);
  return d;
}

// Epilogue of one 32 x 32 tile: rows r0 .. r0 + 31 of the row block, columns c0 .. c0 + 31. acc[4q +
// e] is row r0 + l % 32, column c0 + 8q + 4(l / 32) + e. The tile passes through `st` (row of 128
// bytes, 16-byte chunk c of row r at c ^ (r & 7): eight rows' writes and a row's reads cover all
// banks); then lane l has columns 4(l % 8) .. + 3 of rows 8i + l / 8. Rows past the block are
// dropped by the descriptors. Order: row norm, bias, GELU, rotary, residual (fused/gemm.rs:46-82).
template <int CP, int R>
__device__ __forceinline__ void epilogue_tile(const LinearParams& p, const Rows& d, const f32x16& acc,
                                              unsigned char* st, const float* inv, const int* tok,
                                              int r0, int c0, int lane) {
  const int half = lane >> 5, r = lane & 31;
  const int c = c0 + 4 * (lane & 7);
  const unsigned off = ((unsigned)(r0 + (lane >> 3)) * (unsigned)p.m + c) * 4;
  const unsigned row8 = (unsigned)p.m * 32;  // eight rows
#pragma unroll
  for (int q = 0; q < 4; q++)
    *reinterpret_cast<float4*>(st + r * 128 + (((2 * q + half) ^ (r & 7)) << 4)) =
        make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
  const bool rotary = p.rope && c0 < 2 * p.width;
  const unsigned table = ((c0 < p.width ? 0u : 2u) * p.tokens * 64 + (c & 63)) * 4;
  float4 b = {};
  if (p.bias) b = bload4<true>(d.bias, (unsigned)c * 4);
  // R rows of this lane at a time, their operands from memory all in flight together.
#pragma unroll
  for (int i0 = 0; i0 < 4; i0 += R) {
    float4 cs[R], sn[R], x[R], v[R];
    if (rotary)
#pragma unroll
      for (int i = 0; i < R; i++) {
        const unsigned o = table + (unsigned)tok[r0 + 8 * (i0 + i) + (lane >> 3)] * 256;
        cs[i] = bload4<true>(d.rope, o);
        sn[i] = bload4<true>(d.rope, o + (unsigned)p.tokens * 256);
      }
    if (p.residual)
#pragma unroll
      for (int i = 0; i < R; i++) x[i] = bload4<true>(d.residual, off + (i0 + i) * row8);
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int rr = 8 * (i0 + i) + (lane >> 3);
      v[i] = *reinterpret_cast<const float4*>(st + rr * 128 + (((lane & 7) ^ (rr & 7)) << 4));
      if (p.norm) v[i] = scale4(v[i], inv[r0 + rr]);
      v[i] = make_float4(v[i].x + b.x, v[i].y + b.y, v[i].z + b.z, v[i].w + b.w);
    }
    if (p.gelu)
#pragma unroll
      for (int i = 0; i < R; i++)
        v[i] = make_float4(gemm::gelu_erf(v[i].x), gemm::gelu_erf(v[i].y), gemm::gelu_erf(v[i].z),
                           gemm::gelu_erf(v[i].w));
    if (rotary)
#pragma unroll
      for (int i = 0; i < R; i++) v[i] = rotate4(v[i], cs[i], sn[i]);
    if (p.residual)
#pragma unroll
      for (int i = 0; i < R; i++)
        v[i] = make_float4(v[i].x + x[i].x, v[i].y + x[i].y, v[i].z + x[i].z, v[i].w + x[i].w);
#pragma unroll
    for (int i = 0; i < R; i++) bstore4<true, CP>(d.out, off + (i0 + i) * row8, v[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ---- resident: 96 rows of k = 16 SD in LDS as B fragments, the columns walked in pairs of 32-column
// blocks (pair p on wave p % 8), each weight fragment feeding three MFMAs and each operand fragment
// two. `splits` workgroups share a row block's pairs when there are fewer row blocks than CUs. One
// workgroup of 8 waves per CU; no barrier inside the walk. 96 rows: with 128 the epilogue's operands
// spill (96 120 x 384 -> 1664: 243-262 us against 235), 64 rows measured 251.
template <int SD>
__global__ __launch_bounds__(512, 1) void linear_resident_kernel(LinearParams p, int blocks,
                                                                 int splits) {
  constexpr int NR = 3, PD = 4;
  constexpr int kRows = 32 * NR, K = 16 * SD;
  __shared__ __attribute__((aligned(16))) unsigned char X[kRows * K * 2];
  __shared__ __attribute__((aligned(16))) unsigned char stage[8][kStage];
  __shared__ float inv[kRows];
  __shared__ int tok[kRows];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lane16 = (unsigned)lane * 16;
  const rsrc_t wr = make_rsrc(p.w, (unsigned)(p.m * K * 2));
  const int nb = p.m / 32, pairs = nb / 2;
  int bo[4];  // this lane's place in the fragments of step s % 4
#pragma unroll
  for (int i = 0; i < 4; i++) bo[i] = slot_offset(lane & 31, 2 * i + (lane >> 5)) - i * kFrag;

  for (int item = xcd_remap(blockIdx.x, gridDim.x); item < blocks * splits; item += gridDim.x) {
    const int blk = item / splits, part = item - blk * splits;
    const int p0 = pairs * part / splits, p1 = pairs * (part + 1) / splits;
    const int row0 = blk * kRows;
    const int nrows = min(kRows, p.n - row0);
    const rsrc_t xr = make_rsrc(p.x + (long)row0 * p.ldx,
                                (unsigned)(((long)(nrows - 1) * p.ldx + K) * 4));
    // Eight rows a step and wave: lane l reads k 4 (l % 16) .. + 3 of rows l / 16 and 4 + l / 16 in
    // each 64-k slice.
    for (int g = wave; g < NR * 4; g += 8) {
      const int r = 8 * g + (lane >> 4), k4 = lane & 15;
      float4 v[SD / 4][2];
#pragma unroll
      for (int t = 0; t < SD / 4; t++)
#pragma unroll
        for (int e = 0; e < 2; e++)
          v[t][e] = bload4<true>(xr, ((unsigned)(r + 4 * e) * (unsigned)p.ldx + 64 * t + 4 * k4) * 4);
      float ss[2] = {0.f, 0.f};
#pragma unroll
      for (int t = 0; t < SD / 4; t++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          ss[e] += sumsq4(v[t][e]);
          *reinterpret_cast<u32x2*>(X + ((r >> 5) * SD + 4 * t) * kFrag +
                                    slot_offset(r + 4 * e, k4 >> 1) + 8 * (k4 & 1)) = pack4(v[t][e]);
        }
      if (p.norm)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          ss[e] += __shfl_xor(ss[e], 1);
          ss[e] += __shfl_xor(ss[e], 2);
          ss[e] += __shfl_xor(ss[e], 4);
          ss[e] += __shfl_xor(ss[e], 8);
          if (k4 == 0) inv[r + 4 * e] = 1.0f / fmaxf(sqrtf(ss[e]), 1e-12f);
        }
    }
    if (p.rope && tid < kRows) tok[tid] = (row0 + tid) % p.tokens;
    __syncthreads();

    const Rows d = row_descriptors(p, row0, nrows);
    const int first = p0 + wave;
    u32x4 a[PD][2];
    if (first < p1) {
#pragma unroll
      for (int i = 0; i < PD; i++)
#pragma unroll
        for (int x = 0; x < 2; x++)
          a[i][x] = __builtin_amdgcn_raw_buffer_load_b128(
              wr, lane16, (unsigned)((i * nb + 2 * first + x) * kFrag), 0);
    }
    for (int pr = first; pr < p1; pr += 8) {
      // Opaque per pair: the compiler cannot hoist the operand reads out of the loop.
      int opaque = 0;
      asm volatile("" : "+s"(opaque));
      const unsigned char* B = X + opaque;
      f32x16 acc[2][NR];
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int j = 0; j < NR; j++) acc[x][j] = mfma32_zero();
      const unsigned here = (unsigned)(2 * pr * kFrag);
      // After the last pair its own first steps again: the ring stays in fixed registers.
      const unsigned next = pr + 8 < p1 ? here + (unsigned)(16 * kFrag) : here;
#pragma unroll
      for (int s = 0; s < SD; s++) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
          const u32x4 bf =
              *reinterpret_cast<const u32x4*>(B + (j * SD + s) * kFrag + bo[s % 4]);
#pragma unroll
          for (int x = 0; x < 2; x++) acc[x][j] = mfma32(a[s % PD][x], bf, acc[x][j]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 2; x++)
          a[s % PD][x] = __builtin_amdgcn_raw_buffer_load_b128(
              wr, lane16, s + PD < SD ? here + ((s + PD) * nb + x) * kFrag
                                      : next + ((s + PD - SD) * nb + x) * kFrag, 0);
      }
#pragma unroll
      for (int j = 0; j < NR; j++)
#pragma unroll
        for (int x = 0; x < 2; x++) {
          epilogue_tile<kStream, 2>(p, d, acc[x][j], stage[wave], inv, tok, 32 * j, 32 * (2 * pr + x),
                               lane);
        }
    }
    __syncthreads();  // the next item rewrites the rows
  }
}

// ---- stream: 32 RB rows x 128 NI columns per workgroup. Loads of a wave return in order, so a
// wave that streams x from HBM cannot also wait for its next weight fragment alone. Waves 0-3 (one
// per SIMD) therefore only run MFMAs, NI 32-column blocks of all rows each, on weight fragments
// four steps ahead in registers; waves 4-7 only load x, D tiles of 64 k ahead in registers, and
// write it as fp16 B fragments one tile ahead into a double-buffered LDS tile. One barrier per tile.
// Sixteen lanes read a row's 256 bytes: with lanes spread over rows (16 bytes of 8 rows side by
// side) the loaders' address processing paced every tile (18 060 x 1536 -> 384: 59 -> 47 us).
template <int NI, int RB, int D>
__global__ __launch_bounds__(512, 1) void linear_stream_kernel(LinearParams p, int groups) {
  constexpr int PD = 4;
  constexpr int kRows = 32 * RB;
  constexpr int kTile = kRows * 64 * 2;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2][kTile];
  __shared__ __attribute__((aligned(16))) unsigned char stage[4][kStage];
  __shared__ float inv[kRows];
  __shared__ int tok[kRows];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lane16 = (unsigned)lane * 16;
  const int item = xcd_remap(blockIdx.x, gridDim.x);
  const int blk = item / groups, grp = item - blk * groups;
  const int row0 = blk * kRows;
  const int nrows = min(kRows, p.n - row0);
  const int tiles = p.k / 64;

  if (wave >= 4) {
    // Rows 4 (wave % 4 + 4 i) + l / 16, k 4 (l % 16) .. + 3 of each tile.
    const rsrc_t xr = make_rsrc(p.x + (long)row0 * p.ldx,
                                (unsigned)(((long)(nrows - 1) * p.ldx + p.k) * 4));
    const int sr = 4 * (wave - 4) + (lane >> 4), k4 = lane & 15;
    float ss[2 * RB] = {};
    float4 v[D][2 * RB];
    auto load_x = [&](int t, float4 (&d)[2 * RB]) {
      // Past the last tile the last one again: no branch, so a tile's wait counts only the loads
      // before it.
      const int at = min(t, tiles - 1);
#pragma unroll
      for (int i = 0; i < 2 * RB; i++)
        d[i] = bload4<true, kStream>(
            xr, ((unsigned)(sr + 16 * i) * (unsigned)p.ldx + 64 * at + 4 * k4) * 4);
    };
    auto store_x = [&](int t, const float4 (&d)[2 * RB]) {
#pragma unroll
      for (int i = 0; i < 2 * RB; i++) {
        ss[i] += sumsq4(d[i]);
        *reinterpret_cast<u32x2*>(lds[t & 1] + (i >> 1) * 4 * kFrag +
                                  slot_offset(sr + 16 * i, k4 >> 1) + 8 * (k4 & 1)) = pack4(d[i]);
      }
    };
#pragma unroll
    for (int t = 0; t < D; t++) load_x(t, v[t]);
    // Interval t (before barrier t): tile t is written, while the MFMA waves read tile t - 1.
    for (int t0 = 0; t0 < tiles; t0 += D)
#pragma unroll
      for (int u = 0; u < D; u++) {
        store_x(t0 + u, v[u]);
        load_x(t0 + u + D, v[u]);
        __syncthreads();
      }
    if (p.norm)
#pragma unroll
      for (int i = 0; i < 2 * RB; i++) {
        ss[i] += __shfl_xor(ss[i], 1);
        ss[i] += __shfl_xor(ss[i], 2);
        ss[i] += __shfl_xor(ss[i], 4);
        ss[i] += __shfl_xor(ss[i], 8);
        if (k4 == 0) inv[sr + 16 * i] = 1.0f / fmaxf(sqrtf(ss[i]), 1e-12f);
      }
    const int e = tid - 256;
    if (p.rope && e < kRows) tok[e] = (row0 + e) % p.tokens;
    __syncthreads();
    return;
  }

  const int steps = 4 * tiles, nb = p.m / 32;
  const rsrc_t wr = make_rsrc(p.w, (unsigned)(p.m * p.k * 2));
  const int b0 = NI * (4 * grp + wave);  // this wave's first 32-column block
  u32x4 a[PD][NI];
  auto load_a = [&](int s, u32x4 (&dst)[NI]) {
    // Past the last step the last one again: the ring stays in fixed registers.
    const int at = min(s, steps - 1);
#pragma unroll
    for (int i = 0; i < NI; i++)
      dst[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, lane16,
                                                     (unsigned)((at * nb + b0 + i) * kFrag), 0);
  };
  int bo[4];  // this lane's place in the fragments of step s
#pragma unroll
  for (int i = 0; i < 4; i++) bo[i] = slot_offset(lane & 31, 2 * i + (lane >> 5)) - i * kFrag;
  f32x16 acc[NI][RB];
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int j = 0; j < RB; j++) acc[i][j] = mfma32_zero();
#pragma unroll
  for (int s = 0; s < PD; s++) load_a(s, a[s]);
  for (int t = 0; t < tiles; t++) {
    __syncthreads();  // tile t is in place
    const unsigned char* B = lds[t & 1];
    u32x4 b[2][RB];
    auto load_b = [&](int s) {
#pragma unroll
      for (int j = 0; j < RB; j++)
        b[s & 1][j] = *reinterpret_cast<const u32x4*>(B + (j * 4 + s) * kFrag + bo[s]);
    };
    load_b(0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      if (s < 3) load_b(s + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < RB; j++)
#pragma unroll
        for (int i = 0; i < NI; i++) acc[i][j] = mfma32(a[s % PD][i], b[s & 1][j], acc[i][j]);
      // After its last use, so that the fragment's registers are refilled in place (with a copy
      // taken before, the loop's back edge copies the ring and waits for every load in flight).
      __builtin_amdgcn_sched_barrier(0);
      load_a(4 * t + s + PD, a[s % PD]);
    }
  }
  __syncthreads();  // the row norms are in place
  const Rows d = row_descriptors(p, row0, nrows);
#pragma unroll
  for (int j = 0; j < RB; j++)
#pragma unroll
    for (int i = 0; i < NI; i++)
      epilogue_tile<0, 4>(p, d, acc[i][j], stage[wave], inv, tok, 32 * j, 32 * (b0 + i), lane);
}

template <int SD>
void launch_resident(const LinearParams& p, hipStream_t stream) {
  const int cus = device_cus(), blocks = (p.n + 95) / 96;
  // Fewer row blocks than CUs: the columns of each split over as many workgroups as fit.
  int splits = blocks < cus ? cus / blocks : 1;
  if (splits > p.m / 128) splits = p.m / 128;
  const int items = blocks * splits;
  hipLaunchKernelGGL((linear_resident_kernel<SD>), dim3(items < cus ? items : cus), dim3(512), 0,
                     stream, p, blocks, splits);
}

template <int NI, int RB>
void launch_stream(const LinearParams& p, hipStream_t stream) {
  const int blocks = (p.n + 32 * RB - 1) / (32 * RB), groups = p.m / (128 * NI);
  const dim3 grid(blocks * groups), block(512);
  if (p.k % 256 == 0)
    hipLaunchKernelGGL((linear_stream_kernel<NI, RB, 4>), grid, block, 0, stream, p, groups);
  else
    hipLaunchKernelGGL((linear_stream_kernel<NI, RB, 2>), grid, block, 0, stream, p, groups);
}

// The form a call takes (kGeneral: linear.hip).
enum class Form { kGeneral, kTile32x128, kTile64x128, kTile128x128, kTile96x384, kTile64x512, kResident };

Form choose(long n, long k, long m) {
  if (k % 128 || m % 128) return Form::kGeneral;
  const long cus = device_cus();
  const long small = (n + 63) / 64 * (m / 128);     // 64 x 128 tiles
  const long general = (n + 127) / 128 * (m / 128);  // 128 x 128 ones, linear.hip's too
  // Few rows on a very wide weight: laying it out costs more than it saves where linear.hip already
  // fills the chip (200 x 256 -> 16384 17.7 against 20.6 us, 500 x 512 -> 16384 29.7 against 34.5).
  if (m >= 8192 && k <= 512 && n <= 512 && 2 * general > cus) return Form::kGeneral;
  // Few tiles: the smallest ones, to use the chip at all (up to two 64 x 128 tiles per CU the stream
  // form is ahead also where the resident one applies: 300 x 384 -> 1664 6.0 against 12.5 us,
  // 1000 x 384 -> 1664 8.6 against 12.9). Then the resident form for wide outputs (x is read once), else the
  // widest stream tile that gives at least half the CUs a workgroup: 18 060 x 1536 -> 384 runs at 47
  // us in 96 x 384 tiles, 64 in 64 x 384 (a second round), 62 in 128 x 128.
  if (2 * small <= cus) return Form::kTile32x128;
  if (small <= 2 * cus) return Form::kTile64x128;
  if (m > 512 && (k == 128 || k == 256 || k == 384 || k == 512)) return Form::kResident;
  if (m % 384 == 0 && 2 * ((n + 95) / 96 * (m / 384)) >= cus) return Form::kTile96x384;
  if (m % 512 == 0 && 2 * ((n + 63) / 64 * (m / 512)) >= cus) return Form::kTile64x512;
  // What is left has 128 x 128 tiles either way, here one workgroup per CU against linear.hip's two. Here is
  // ahead with a long k and either enough tiles that the rounds' ends do not count (33 000 x 640 -> 1664
  // 225 -> 189 us), just more than one round of linear.hip's (40 000 x 1024 -> 256 83 -> 72), or an x of
  // 112 MiB and more, which linear.hip reads again for every column group (40 000 x 1536 -> 128
  // 82 -> 67). Elsewhere linear.hip: 65 000 x 256 -> 256 34 against 48, 24 576 x 1024 -> 256 37 against
  // 46, 10 500 x 640 -> 640 27 against 33, 20 000 x 640 -> 1664 103 against 121.
  const bool large = n * k * 4 >= (112l << 20) && (k >= 1536 || general > 2 * cus);
  if (k > 512 && (general >= 8 * cus || (general > 2 * cus && general <= 3 * cus) || large))
    return Form::kTile128x128;
  return Form::kGeneral;
}

}  // namespace

size_t linear_wide_workspace(size_t n, size_t k, size_t m) {
  // Past these sizes the call is refused.
  if (n == 0 || k == 0 || m == 0 || n > 0x7fffffff || m >= (size_t(1) << 22) ||
      k >= (size_t(1) << 30) / m)
    return 0;
  return choose((long)n, (long)k, (long)m) == Form::kGeneral ? 0 : k * m * 2;
}

hipError_t launch_linear_wide(const LinearParams& params, void* workspace, hipStream_t stream) {
  LinearParams p = params;
  const Form form = choose(p.n, p.k, p.m);
  if (form == Form::kGeneral) return hipErrorInvalidValue;  // linear_wide_workspace gave 0
  const int frags = (p.m / 32) * (p.k / 16);
  hipLaunchKernelGGL(weight_fragments_kernel, dim3((frags + 3) / 4), dim3(256), 0, stream, p.w, p.k,
                     p.m, static_cast<u32x4*>(workspace));
  p.w = static_cast<const float*>(workspace);  // fp16 fragments from here on
  switch (form) {
    case Form::kTile32x128: launch_stream<1, 1>(p, stream); break;
    case Form::kTile64x128: launch_stream<1, 2>(p, stream); break;
    case Form::kTile128x128: launch_stream<1, 4>(p, stream); break;
    case Form::kTile96x384: launch_stream<3, 3>(p, stream); break;
    case Form::kTile64x512: launch_stream<4, 2>(p, stream); break;
    case Form::kResident:
      switch (p.k) {
        case 128: launch_resident<8>(p, stream); break;
        case 256: launch_resident<16>(p, stream); break;
        case 384: launch_resident<24>(p, stream); break;
        default: launch_resident<32>(p, stream);
      }
      break;
    case Form::kGeneral: break;
  }
  return hipGetLastError();
}

}  // namespace ancha
