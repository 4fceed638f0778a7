#pragma once
// Shared device code of the attention kernels (attn_fwd.hip, attn.hip): the QKV layout, the
// block table, the LDS tile layout and DMA, the MFMA and transposing-read helpers.
//
// Variable-length causal GQA attention of the packed batch on gfx950: forward (online softmax) and
// backward (delta, dK/dV per query head, dQ).  Replaces solution/k_attn.py:40-245.
//
// Layout (the fused QKV buffer the QKV epilogue writes): row t of qkv [N, (NQ + 2 NKV) HD] fp16
// holds token t's query heads, then its key heads, then its value heads; query head h reads key /
// value head h / (NQ / NKV).  cu_seqlens [n_seq + 1] delimits the sequences; a block table of
// (sequence, first row) pairs names the workgroups, whose rows never straddle two sequences, so
// the mask is `key <= query` inside a sequence.  Scores are scaled by qk_scale = log2(e) / sqrt(HD)
// and the softmax runs in the exp2 domain; lse [NQ, N] holds m + log2(l) per (head, token).
//
// MFMA orientation: every product is v_mfma_f32_32x32x16_f16, arranged so that the index a
// softmax statistic belongs to sits on the lane.  Forward and dQ compute S^T = K Q^T (keys x
// queries: lane l % 32 is the query, the running max, sum and rescale are per lane) and O^T = V^T
// P^T, taking P^T straight from the score registers: the 32x32 result register v of lane l is row
// 8 (v / 4) + 4 (l / 32) + v % 4, so registers 8 t' .. 8 t' + 7 of a lane hold keys
// 16 t' + 8 (j / 4) + 4 (l / 32) + j % 4 (j = 0..7), and the other operand supplies the same keys
// in the same order, read as columns of the row-major LDS tile by ds_read_b64_tr_b16 (the k order
// of a product is free as long as both operands agree).  dK/dV compute S = Q K^T (the key on the
// lane) and use P and dS the same way.
#include "lds_dma.h"

namespace {

using dk::dma16s;
using dk::dma4;
using dk::lds_addr;
using dk::uniform64;
using dk::wait_vmem;

constexpr int kHD = 128;          // head size (Qwen2.5: 128)
constexpr int kAThreads = 256;    // 4 waves, 32 query rows (or keys) each
constexpr int kBM = 128;          // queries per forward / dQ workgroup, keys per dK/dV workgroup
constexpr int kBN = 64;           // keys per forward / dQ tile, queries per dK/dV tile
static_assert(kBM == 32 * (kAThreads / 64), "a wave owns 32 rows");

struct AttnArgs {
  const f16* qkv;
  const int32_t* cu;
  const int32_t* tab;
  int n_seq;
  int64_t n_tokens;
  int nq, nkv;
  float qk_scale, sm_scale;
};

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int v = 0; v < 16; ++v) z[v] = 0.0f;
  return z;
}

__device__ __forceinline__ f16x8 zero8() {
  f16x8 z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = (f16)0.0f;
  return z;
}

__device__ __forceinline__ f32x16 mfma(const f16x8& a, const f16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// K / V (or Q / dO) tiles in a ring of LDS stages filled by LDS DMA (global_load_lds_dwordx4:
// no registers, the next tiles' loads in flight while this one is computed on).  A tile is kBN
// rows of 256 bytes with no padding; the 16-byte chunks of row r are permuted by swz16(r), so
// that both reads of the tile are free of bank conflicts: the S^T operand (16 consecutive rows,
// one chunk each) and the transposing V reads (4 rows x 2 adjacent chunks per 16-lane group).
constexpr int kFwdStages = 4;                 // tiles t, t + 1 in use, t + 2, t + 3 in flight
constexpr int kTileHalves = kBN * kHD;        // one operand of one stage: 16 KB

__device__ __forceinline__ int swz16(int r) {
  return ((r & 3) << 1) | ((r >> 2) & 1) | (((r >> 3) & 1) << 3);
}
// offset (halves) of column c of row r in a swizzled tile
__device__ __forceinline__ int sw_off(int r, int c) {
  return r * kHD + ((((c >> 3) ^ swz16(r))) << 3) + (c & 7);
}

// The operand reads of a tile by LDS byte address.  The swizzle only flips chunk bits, so every
// operand of a tile is a lane's base address with a constant XORed into it (plus a constant row
// offset): K operand of sub-step s of rows 0..31 (+ 32 rows: 8192 bytes on) at kaddr ^ 32 s, and
// the transposed columns of head block hb at vaddr ^ 64 hb (rows + 8: ^ 64 (hb ^ 2), 2048 on).
typedef __attribute__((address_space(3))) const char lds_char;
__device__ __forceinline__ f16x8 lds_read8(unsigned addr, int off) {
  return *reinterpret_cast<__attribute__((address_space(3))) const f16x8*>((lds_char*)(size_t)addr + off);
}
__device__ __forceinline__ f16x4 lds_read_tr(unsigned addr, int off) {
  return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)((lds_char*)(size_t)addr + off)));
}
// this lane's base for lds_read8 (row c = lane % 32, columns 8 (lane / 32) .. + 7) and for
// lds_col8 (row 4 (lane / 32) + lane % 16 / 4, columns 16 (lane / 16 % 2) + 4 (lane % 4) .. + 3)
__device__ __forceinline__ unsigned row_base(int lane) {
  return (unsigned)(sw_off(lane & 31, 8 * (lane >> 5)) * 2);
}
__device__ __forceinline__ unsigned col_base(int lane) {
  return (unsigned)(sw_off(4 * (lane >> 5) + ((lane & 15) >> 2), 16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2);
}
// Column 32 hb + lane % 32 of rows p .. p + 3 and p + 8 .. p + 11 of a swizzled tile, p = 4 (lane / 32)
// (+ off / 256 rows): the 8 values of MFMA k index j = 0..7.  ds_read_b64_tr_b16: within a 16-lane
// group, lane 4a + b receives element b of the 4-half pieces addressed by lanes a, a + 4, a + 8,
// a + 12; with lane x of the group at row p + x / 4, columns 4 (x % 4) .. + 3 of the group's 16, lane
// x' receives column x' of the four rows.
__device__ __forceinline__ f16x8 lds_col8(unsigned caddr, int hb, int off) {
  const f16x4 lo = lds_read_tr(caddr ^ (unsigned)(64 * hb), off);
  const f16x4 hi = lds_read_tr(caddr ^ (unsigned)(64 * (hb ^ 2)), off + 2048);
  return f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}
// keeps the compiler from holding every XORed address in a register of its own across the loop
__device__ __forceinline__ unsigned fresh(unsigned a) {
  asm volatile("" : "+v"(a));
  return a;
}

// Two values rounded to fp16, computed where they stand: without the empty asm the compiler sinks
// the work down to its use, past the scheduling barriers that interleave it with MFMAs.
__device__ __forceinline__ f16x2 pinned(float lo, float hi) {
  f16x2 h = f16x2{(f16)lo, (f16)hi};
  asm volatile("" : "+v"(h));
  return h;
}
// elements i - 1, i (i odd) of 16-bit operands of 8
struct Frag8 {
  f16x2 h[4];
  __device__ __forceinline__ f16x8 get() const {
    return f16x8{h[0][0], h[0][1], h[1][0], h[1][1], h[2][0], h[2][1], h[3][0], h[3][1]};
  }
};

// 2^x on the hardware exponential (v_exp_f32); arguments here are <= 0 (scores minus their row
// maximum or log-sum-exp), results below the normal range flush to zero.
__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

// The sequence of a block-table entry; false when the entry names no sequence, a sequence that
// does not lie within the n_tokens rows, or a block start at or past the sequence's end (an empty
// sequence included).  A workgroup whose entry is refused returns before any load, so every row
// a kernel reads unconditionally (row start of the sequence) exists whatever the tables hold.
__device__ __forceinline__ bool block_of(const AttnArgs& a, int blk, int64_t* s0, int* seqlen,
                                         int* start) {
  const int seq = a.tab[2 * blk];
  *start = a.tab[2 * blk + 1];
  if (seq < 0 || seq >= a.n_seq || *start < 0) return false;
  *s0 = a.cu[seq];
  *seqlen = a.cu[seq + 1] - a.cu[seq];
  return *s0 >= 0 && *seqlen > 0 && *start < *seqlen && *s0 + *seqlen <= a.n_tokens;
}

// the launch arguments, with the checks every attention entry point shares
inline int attn_args(AttnArgs& a, const void* qkv, const int32_t* cu, int32_t n_seq,
                     const int32_t* tab, int32_t n_blocks, int64_t n_tokens, int32_t nq,
                     int32_t nkv, int32_t hd) {
  if (hd != kHD || nq < 1 || nkv < 1 || nq % nkv || nq > 65535 || n_seq < 0 || n_blocks < 0 ||
      n_tokens < 0)
    return DK_ERR_INVALID;
  if (n_blocks > 0 && (!qkv || !cu || !tab || n_seq < 1)) return DK_ERR_INVALID;
  if (!dk_aligned(qkv, 16) || !dk_aligned(cu, 4) || !dk_aligned(tab, 4)) return DK_ERR_ALIGN;
  const double log2e = 1.4426950408889634;
  a = AttnArgs{(const f16*)qkv, cu, tab, n_seq, n_tokens, nq, nkv,
               (float)(log2e / __builtin_sqrt((double)hd)), (float)(1.0 / __builtin_sqrt((double)hd))};
  return 0;
}

}  // namespace
