// NF4 double-quantised weights on gfx950: the HBM-rate dequant and the blockwise quantiser.
//
// Dequant (replaces solution/k_nf4.py:40-57).  Each wave converts one second-level block (2048
// packed dwords of 8 weights, 16384 weights), or a quarter of one where there are few, with nf4_dev.h's dq_wave_load / dq_wave_store: every
// load instruction of the wave reads 256 contiguous bytes and every store instruction writes the
// 64 lanes' 16-byte results, 1 KiB contiguous, straight from registers (no LDS staging, no
// barrier before the stores).  A workgroup's four waves fill the two LDS tables (NF4 values and
// the second-level codes) while their loads are in flight.  HBM traffic: 2.516 bytes per weight
// (0.5 packed + 1/64 code + 8/16384 scale/offset in, 2 out).
#include "nf4_dev.h"

using dk::kWaveDwords;
using dk::WaveLoadsOf;
using dk::dq_wave_load;
using dk::dq_wave_store;

namespace {

// W = 32 dwords per lane (256 weights) in 256-thread workgroups, 714 per Qwen2.5-1.5B layer: measured
// on MI355X over 28 layer buffers (graph-replayed, gaps included) 5.5-5.6 TB/s, against 4.8-5.0
// for the former one-quad-per-lane kernel with LDS-staged stores, 5.1-5.2 for 8 or 16 dwords per
// lane (16 with 512 threads), 4.8-5.1 for 8 or 16 with 1024 threads and 4.9 for 64; cached
// instead of non-temporal loads of the packed bytes cost 6-7 %.  With the conversion replaced by
// a plain copy of the packed words, 8 dwords per lane ran at the same 5.2 TB/s: more bytes in
// flight per wave, not less arithmetic, is what raised the rate (writes alone reach 6.9 TB/s)
constexpr int kDqThreads = 256;
// A weight that would not give every CU a workgroup of that form takes 8 dwords per lane, four times
// as many workgroups: its time is one wave's chain of loads and stores, not the rate.  Measured
// likewise on MI355X: [256, 1536] 6.8 -> 3.7 us, [1536, 1536] 7.5 -> 4.3 (16 dwords: 5.4),
// [4096, 1536] 8.8 -> 6.1, [8960, 1536] 9.8 -> 8.8; beyond the line [11008, 2048] 12.5 against
// 12.6 and [17920, 1536] 14.0 against 14.3.
constexpr int kDqFew = 8;
constexpr int64_t kDqFewMax = 256 * kDqThreads * kWaveDwords;   // dwords
static_assert(kDqThreads == 256, "one code2 entry per thread");

template <int W>
__global__ __launch_bounds__(kDqThreads) void nf4_dequant_kernel(
    const uint32_t* __restrict__ packed, const uint8_t* __restrict__ qabs,
    const float* __restrict__ scale2, const float* __restrict__ offset2,
    const float* __restrict__ code2, const float* __restrict__ nf4, u32x4* __restrict__ out,
    int64_t n_dwords) {
  __shared__ float lut[16];
  __shared__ float c2[256];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t d_wave = ((int64_t)blockIdx.x * kDqThreads + wave * 64) * W;
  const int64_t last = n_dwords - 1;
  // the tables' loads first (the LDS fill waits only for them), then the codes and the dwords
  const float c2v = code2[threadIdx.x];
  const float lutv = nf4[threadIdx.x & 15];
  WaveLoadsOf<W> L;
  dq_wave_load(packed, qabs, scale2, offset2, d_wave, last, lane, L);
  c2[threadIdx.x] = c2v;
  if (threadIdx.x < 16) lut[threadIdx.x] = lutv;
  __syncthreads();
  dq_wave_store<false>(L, c2, lut, out, d_wave, last, lane);
}

// ---------------------------------------------------------------------------------------------
// Quantiser.  Pass 1: four lanes per 64-weight block compute absmax = max|w|, the NF4 codes of
// w * fp32(1/absmax) (code = number of fp32 midpoints between consecutive NF4 values strictly
// below it; an all-zero block gives code 7) and the packed bytes, and add absmax to an exact
// integer sum in units of 2^-24.  Pass 2: one 256-thread block per second-level block
// subtracts offset = fp32(sum / n) and quantises each absmax against the 256-entry code table
// (nearest entry, ties to the lower index) after normalising by the block's max magnitude.
//
// Bound: memory (2 bytes read, 0.52 written per weight) once two other costs are out of the way.
// Comparing every weight with all 15 midpoints took 30 vector instructions; a weight now finds its
// 1/32-wide bucket of [-1, 1] and compares with the one midpoint that the bucket can hold, about 9
// instructions and one LDS read.  And every workgroup ends in an atomic on one word, about 20 ns
// apart: one workgroup per CU.  Measured on MI355X, a [8960, 1536] weight: 23.9 us before, 22.6
// with the buckets on 1024 workgroups, 15.0 on 256 of 1024 threads.

constexpr int kQThreads = 256;     // pass 2
constexpr int kQ1Threads = 1024;   // pass 1
constexpr int kQ1Groups = 256;     // its workgroups at most
constexpr int kBuckets = 64;           // of width 1/32 over [-1, 1]
constexpr float kBucketSlack = 1e-4f;  // far more than the rounding of x and of its bucket index

__global__ void zero_u64_kernel(uint64_t* p) { *p = 0; }

__global__ __launch_bounds__(kQ1Threads) void nf4_quant_pass1(
    const f16x8* __restrict__ w, const float* __restrict__ nf4, u32x2* __restrict__ packed,
    float* __restrict__ absmax_out, uint64_t* __restrict__ sum, int64_t n_qblocks) {
  __shared__ float mid[15];
  // per bucket: its midpoint (or +inf), and the number of midpoints below the bucket
  __shared__ f32x2 bucket[kBuckets];
  __shared__ int crowded;   // some bucket holds two midpoints: a table this search does not fit
  __shared__ uint64_t red[kQ1Threads / 64];
  const int tid = threadIdx.x;
  if (tid < 15) mid[tid] = __fmul_rn(__fadd_rn(nf4[tid], nf4[tid + 1]), 0.5f);
  if (tid == 0) crowded = 0;
  __syncthreads();
  if (tid < kBuckets) {
    // counted over the bucket widened by the slack on both sides, so that a weight whose index
    // was rounded into the neighbouring bucket finds the same code there
    const float lo = (float)tid * 0.03125f - 1.0f - kBucketSlack;
    const float hi = lo + 0.03125f + 2.0f * kBucketSlack;
    int below = 0, inside = 0;
    float m = INFINITY;
    for (int t = 0; t < 15; ++t) {
      const bool b = mid[t] < lo, in = !b && mid[t] <= hi;
      below += b;
      inside += in;
      if (in) m = mid[t];
      // midpoints outside the range, or a NaN: the plain count
      if (!(mid[t] > -0.99f && mid[t] < 0.99f)) inside = 2;
    }
    if (inside > 1) crowded = 1;
    bucket[tid] = f32x2{m, (float)below};
  }
  __syncthreads();
  const bool plain = crowded != 0;
  uint64_t units = 0;
  // every lane takes part in each turn (the block's maximum crosses lanes); blocks past the end
  // read the last one and store nothing
  constexpr int kPer = kQ1Threads / 4;
  for (int64_t q0 = (int64_t)blockIdx.x * kPer; q0 < n_qblocks; q0 += (int64_t)gridDim.x * kPer) {
    const int64_t q = q0 + (tid >> 2), qc = q < n_qblocks ? q : n_qblocks - 1;
    f16x8 v[2];   // 16 weights of the block: 16 (tid % 4) ..
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = w[qc * 8 + 2 * (tid & 3) + i];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf((float)v[i][e]));
    amax = fmaxf(amax, __shfl_xor(amax, 1));
    amax = fmaxf(amax, __shfl_xor(amax, 2));
    const float inv = amax != 0.0f ? __fdiv_rn(1.0f, amax) : 0.0f;
    u32x2 words;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t word = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = __fmul_rn((float)v[i][e], inv);
        uint32_t code = 0;
        if (!plain) {
          // (a NaN goes to bucket 0 and compares false: code 0, as no midpoint is below it)
          const float at = fminf(fmaxf(__fadd_rn(__fmul_rn(x, 32.0f), 32.0f), 0.0f), 63.0f);
          const f32x2 b = bucket[(int)at];
          code = (uint32_t)b[1] + (x > b[0] ? 1u : 0u);
        } else {
          for (int t = 0; t < 15; ++t) code += (x > mid[t]) ? 1u : 0u;
        }
        // element 2j -> high nibble of byte j
        word |= code << (8 * (e >> 1) + ((e & 1) ? 0 : 4));
      }
      words[i] = word;
    }
    if (q < n_qblocks) {
      packed[q * 4 + (tid & 3)] = words;
      if ((tid & 3) == 0) {
        absmax_out[q] = amax;
        units += (uint64_t)ldexpf(amax, 24);  // exact: amax is an fp16 magnitude, a multiple of 2^-24
      }
    }
  }
  // block sum of units, then one atomic per block (integer: order independent)
  for (int off = 32; off > 0; off >>= 1) units += __shfl_xor(units, off);
  if ((tid & 63) == 0) red[tid >> 6] = units;
  __syncthreads();
  if (tid == 0) {
    uint64_t s = 0;
    for (int i = 0; i < kQ1Threads / 64; ++i) s += red[i];
    atomicAdd((unsigned long long*)sum, (unsigned long long)s);
  }
}

__global__ __launch_bounds__(kQThreads) void nf4_quant_pass2(
    const float* __restrict__ absmax, const float* __restrict__ code2,
    const uint64_t* __restrict__ sum, uint8_t* __restrict__ qabs, float* __restrict__ scale2,
    float* __restrict__ offset2, int64_t n_qblocks) {
  __shared__ float table[256];
  __shared__ float red[kQThreads / 64];
  table[threadIdx.x] = code2[threadIdx.x];
  const float offset = (float)(((double)(*sum) / (double)n_qblocks) * 0x1p-24);
  const int64_t q = (int64_t)blockIdx.x * kQThreads + threadIdx.x;
  const float v = __fsub_rn(absmax[q], offset);
  float m = fabsf(v);
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  float a2 = red[0];
  for (int i = 1; i < kQThreads / 64; ++i) a2 = fmaxf(a2, red[i]);
  const float inv = a2 != 0.0f ? __fdiv_rn(1.0f, a2) : 0.0f;
  const float y = __fmul_rn(v, inv);
  // count = number of table entries <= y (the table is sorted ascending)
  int lo = 0, hi = 256;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (table[mid] <= y) lo = mid + 1; else hi = mid;
  }
  int i0 = lo - 1;
  if (i0 < 0) i0 = 0;
  const int i1 = i0 + 1 < 256 ? i0 + 1 : 255;
  const float d_hi = __fsub_rn(table[i1], y);
  const float d_lo = __fsub_rn(y, table[i0]);
  qabs[q] = (uint8_t)(d_hi < d_lo ? i1 : i0);
  if (threadIdx.x == 0) {
    scale2[blockIdx.x] = a2;
    offset2[blockIdx.x] = offset;
  }
}

}  // namespace

extern "C" int dk_nf4_dequant(const uint8_t* packed, const uint8_t* qabs, const float* scale2,
                              const float* offset2, const float* code2, const float* nf4,
                              void* out_f16, int64_t n_qblocks, hipStream_t stream) {
  if (n_qblocks < 0) return DK_ERR_INVALID;
  if (n_qblocks == 0) return 0;
  if (!packed || !qabs || !scale2 || !offset2 || !code2 || !nf4 || !out_f16) return DK_ERR_INVALID;
  if (!dk_aligned(packed, 16) || !dk_aligned(out_f16, 16)) return DK_ERR_ALIGN;
  const int64_t n_dwords = n_qblocks * 8;
  const bool few = n_dwords <= kDqFewMax;
  const int64_t per_wg = (int64_t)kDqThreads * (few ? kDqFew : kWaveDwords);
  const int64_t grid = (n_dwords + per_wg - 1) / per_wg;
  if (grid > 0x7fffffff) return DK_ERR_INVALID;
  hipLaunchKernelGGL(few ? nf4_dequant_kernel<kDqFew> : nf4_dequant_kernel<kWaveDwords>,
                     dim3((unsigned)grid), dim3(kDqThreads), 0, stream,
                     reinterpret_cast<const uint32_t*>(packed), qabs, scale2, offset2, code2, nf4,
                     reinterpret_cast<u32x4*>(out_f16), n_dwords);
  DK_CHECK_LAUNCH();
  return 0;
}

extern "C" int dk_nf4_quantize(const void* w_f16, int64_t numel, const float* code2,
                               const float* nf4, uint8_t* packed, uint8_t* qabs, float* scale2,
                               float* offset2, float* absmax_ws, uint64_t* sum_ws,
                               hipStream_t stream) {
  if (numel <= 0 || numel % DK_ELEMS_PER_SB) return DK_ERR_INVALID;
  if (!w_f16 || !code2 || !nf4 || !packed || !qabs || !scale2 || !offset2 || !absmax_ws || !sum_ws)
    return DK_ERR_INVALID;
  if (!dk_aligned(w_f16, 16) || !dk_aligned(packed, 16) || !dk_aligned(sum_ws, 8))
    return DK_ERR_ALIGN;
  const int64_t nq = numel / DK_QBLOCK;
  hipLaunchKernelGGL(zero_u64_kernel, dim3(1), dim3(1), 0, stream, sum_ws);
  DK_CHECK_LAUNCH();
  // one workgroup per CU: each ends in one atomic on the same word, about 20 ns apart
  const int64_t wgs = (nq + kQ1Threads / 4 - 1) / (kQ1Threads / 4);
  hipLaunchKernelGGL(nf4_quant_pass1, dim3((unsigned)(wgs < kQ1Groups ? wgs : kQ1Groups)),
                     dim3(kQ1Threads), 0, stream, reinterpret_cast<const f16x8*>(w_f16), nf4,
                     reinterpret_cast<u32x2*>(packed), absmax_ws, sum_ws, nq);
  DK_CHECK_LAUNCH();
  hipLaunchKernelGGL(nf4_quant_pass2, dim3((unsigned)(nq / DK_QBLOCK2)), dim3(kQThreads), 0, stream,
                     absmax_ws, code2, sum_ws, qabs, scale2, offset2, nq);
  DK_CHECK_LAUNCH();
  return 0;
}
