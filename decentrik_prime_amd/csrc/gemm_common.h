// Parameters shared by the fused GEMM kernels (w4gemm.hip: NF4 or fp16 weights, warp-specialised
// 128-row tiles; hgemm.hip: fp16 weights, 256 x 256 tiles fed by LDS-DMA loads).
#pragma once
#include "lora_dev.h"
#include "nf4_dev.h"

namespace dk {

enum { EPI_LINEAR = 0, EPI_SWIGLU_FWD = 1, EPI_SWIGLU_BWD = 2 };

// One LoRA term of the LINEAR epilogue.  Forward: adds s * fp32(fp16(z B^T)) to output columns
// [n_begin, n_end) (B holds the rows of those columns).  Backward: adds
// (mask ? fp32(fp16(dz A)) * keep_scale : 0) to every column.
struct LoraTerm {
  const f16* z;         // [M][rank]: z (forward) or dz (backward)
  const f16* r;         // forward: B [n_end - n_begin][rank]; backward: A [rank][N]
  const uint8_t* mask;  // backward keep-mask [M][N] or null (no dropout, no scale)
  int64_t n_begin, n_end;
  float scale;          // forward: s; backward: keep_scale
};

struct GemmParams {
  const f16* a;
  int64_t lda;
  int64_t M, N, K;
  const uint8_t* packed;
  const uint8_t* qabs;
  const float* scale2;
  const float* offset2;
  const float* code2;
  const float* nf4;
  const f16* w16;       // two-phase: the weight dequantised to fp16, stored order ([N][K] NT, [K][N] NN)
  int64_t inter;        // SwiGLU: gate/up width I
  const f16* bias;      // [N] or null
  LoraTerm lora[2];     // rank-r LoRA terms added in the LINEAR epilogue, in order
  int n_lora;
  int64_t rank;
  void* out;
  int64_t ldo;
  int out_mode;
  f16* gu;              // SWIGLU_FWD: optional [M][2I] output; SWIGLU_BWD: [M][2I] in/out
  int tiles_m, tiles_n;
  int m_fastest;        // tile order: row tiles fastest (1) or column tiles fastest (0)
  int xcd_gm;           // 256-tile kernel: the 128 x 128 quarters split into a block per XCD,
                        // xcd_gm blocks along M by 8 / xcd_gm along N (0: runs of quarters;
                        // below 0: a grid of 128-row tiles)
  int splits;           // split-K factor (1: none)
  float* part;          // split-K partial tiles [tiles][splits][BM * BN] fp32
  SideDequant side;     // dequant work carried by the launch's last side.wgs workgroups
  SideSums sums;        // LoRA column sums carried by the sums.wgs workgroups before those
  // LINEAR NT only: rotary embedding of output columns [0, rope_cols) (the q and k heads of a
  // fused QKV projection) in the epilogue, before the single fp16 rounding; null: none
  const int32_t* rope_pos;   // [M] token positions
  const float* rope_cos;     // [positions][rope_hd]
  const float* rope_sin;
  int rope_hd;               // head size: two 64-column wave blocks
  int64_t rope_cols;
};

constexpr int kBK = 64;   // K per step of both kernels

// Launch plan of w4gemm.hip's kernel: tile shape and split-K factor.  256 CUs.  A 128-row tile's workgroup needs
// 76.8 KB of LDS (60 KB at 64 columns) and at most 128 VGPRs, so two share a CU (512 slots).
// (256 x 128 tiles, one workgroup per CU, measured slower at these shapes and are not
// planned.)  Shapes with fewer tiles than slots split K (at least 8 steps per split) so that about
// 768 workgroups run: the fp32 partial tiles cost one extra pass over the output in the second
// launch, so short K (under 64 steps) prefers narrower tiles and splits only below 256 tiles.
struct Plan {
  int bm, bn, splits;
  int64_t tiles;
};

inline Plan plan_for(int64_t M, int64_t N, int64_t K, int epi) {
  const int64_t nk = K / kBK;
  const int64_t mt128 = (M + 127) / 128;
  Plan pl{128, 128, 1, mt128 * (N / 128)};
  if (N % 128 != 0) pl = {128, 64, 1, mt128 * (N / 64)};
  if (epi != EPI_LINEAR || pl.tiles >= 512) return pl;
  if (pl.bn == 128 && nk < 64) pl = {128, 64, 1, mt128 * (N / 64)};
  if ((pl.tiles < 256 && nk >= 16) || (pl.tiles < 512 && nk >= 64)) {
    int64_t s = (768 + pl.tiles - 1) / pl.tiles;
    if (s > nk / 8) s = nk / 8;
    if (s > 8) s = 8;
    if (s >= 2) pl.splits = (int)s;
  }
  return pl;
}

// Runs the GEMM of `p` (fp16 weight p.w16) on hgemm.hip's kernels when the shape suits them: output
// columns a multiple of 256, K a multiple of 64, and at least one 256 x 256 tile per CU or one of
// the smaller plans (128 x 128 tiles, 128 x 256 tiles, 256 x 256 tiles, the last two with or
// without split K, whose fp32 partials need hgemm_workspace bytes of `ws`) estimated faster than
// w4gemm.hip's kernel.  p.side's workgroups (if any) join the launch.  Returns kHgemmDeclined without launching
// anything otherwise, a HIP error code, or 0.
constexpr int kHgemmDeclined = -1000;
// W4: the weight read as packed NF4 (p.packed, p.qabs, p.scale2, p.offset2, p.code2, p.nf4; no
// p.w16) and dequantised by each workgroup into LDS, bit-identical to the fp16 form's results.
template <bool TRANS, int EPI, bool W4 = false>
int hgemm_launch(const GemmParams& p, void* ws, int64_t ws_bytes, hipStream_t stream);
// The NT GEMM of `p` for a few rows (skinny.hip), on packed NF4 weights or p.w16: up to 16 rows, or
// 32 for a LINEAR weight of at most 2048 x 1536.  Every 16 columns read all of A again, so large fp16
// weights with K >= N are left to the tiles from 13 rows on, which split K over all CUs (16 rows:
// 3584 x 18944 40.3 -> 35.2 us, 8192 x 8192 36.8 -> 33.7; at 12 rows 36.6 against 35.3, 33.7 against
// 33.9 and 4096 x 14336 29.9 against 31.7).
inline bool skinny_takes(const GemmParams& p, int epi) {
  if (p.M > 12 && p.w16 && epi == EPI_LINEAR && p.K >= p.N && p.N * p.K >= (int64_t)48 << 20) return false;
  return p.M <= 16 || (p.M <= 32 && epi == EPI_LINEAR && p.N * p.K <= (int64_t)2048 * 1536);
}
template <int EPI, bool F16>
int skinny_launch(const GemmParams& p, hipStream_t stream);
// Split-K partials the launch of that shape needs (0: no split; -1: the plan does not take the
// shape); nt: NT (W stored [N][K]).
int64_t hgemm_workspace(int64_t M, int64_t N, int64_t K, int epi, bool nt);
// Split-K partials that a LINEAR GEMM which has a workspace must find room for: 0 where its 128 x 128
// tiles fill half of the CUs and (NN) it has at most 3 row tiles of 256 or K below 4096, or with a 256 x 256
// tile per CU (such a call splits K for speed alone, if it does: it runs without where there is no
// scratch memory to be had); -1: w4gemm.hip's kernel decides.
int64_t hgemm_required(int64_t M, int64_t N, int64_t K, bool nt);

}  // namespace dk
