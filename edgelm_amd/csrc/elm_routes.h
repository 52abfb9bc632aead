// Which kernel a call takes, where that depends on sizes, types and alignment: the rules alone, in plain C++ (no HIP), so
// that they can be checked without a GPU. The launchers ask here; each rule's comment says what both sides measured.
#pragma once
#include <cstddef>
#include <cstdint>

namespace elmh {

// LDS a workgroup may allocate on gfx950 (160 KB per CU; kernels that use more than 64 KB raise their
// dynamic-LDS limit before the first launch on each device)
constexpr size_t kMaxLds = 160 * 1024;
// dynamic LDS the attention kernels may take (their static LDS is a few words; this leaves 1 KB for it)
constexpr size_t kMaxAttnLds = kMaxLds - 1024;

// ---------------------------------------------------------------- attention

constexpr int kAttnThreads = 256;
constexpr int kAttnVF = 20;                           // attention_kernel: float4 of values per thread per chunk
constexpr int kAttnChunkF4 = kAttnThreads * kAttnVF;  // 80 KB: 320 positions of head size 64
constexpr int attn_chunk_pos(int hd) { return (kAttnChunkF4 / (hd / 4)) & ~15; }
constexpr int kDecRows = 256;    // attention_decode64_kernel: rows per LDS buffer, one per thread
constexpr int kAttnQ = 4;        // attention_prefill_kernel, attention_prefill64_kernel: query tokens per workgroup
constexpr int kAttnPVPos = 96;   // attention_prefill_kernel: value rows per chunk (24 KB)
constexpr int kPfRows = 128;     // attention_prefill64_kernel: key and value rows per LDS chunk
constexpr int kStepWaves = 16;   // attention_step_kernel

// LDS of each kernel for n_cap score slots
inline size_t attention_decode_lds_bytes(int n_cap) {  // two row buffers, the scores, q and the step's key
  return ((size_t)2 * kDecRows * 64 + (size_t)((n_cap + 255) & ~255) + 128) * sizeof(float);
}
inline size_t attention_prefill_lds_bytes(int n_cap) {
  return ((size_t)kAttnQ * 64 + (size_t)kAttnQ * ((n_cap + 63) & ~63) + (size_t)kAttnPVPos * 64) * sizeof(float);
}
inline size_t attention_prefill64_lds_bytes(int n_cap) {
  return ((size_t)2 * kPfRows * 64 + (size_t)kAttnQ * ((n_cap + 255) & ~255) + (size_t)kAttnQ * 64) * sizeof(float);
}
inline size_t attention_lds_bytes(int hd, int n_max) {
  const size_t hdp = (size_t)((hd + 3) & ~3);
  return (2 * hdp + (size_t)((n_max + 63) & ~63) + (size_t)attn_chunk_pos(hd) * hd) * sizeof(float);
}
// attention_kernel with its score rows in global memory: LDS holds q, the fused key and a chunk
inline size_t attention_gs_lds_bytes(int hd) {
  return (2 * (size_t)((hd + 3) & ~3) + (size_t)attn_chunk_pos(hd) * hd) * sizeof(float);
}
// attention_rows_kernel for R rows per workgroup: the score row stride (a multiple of 4 that spreads the rows over the LDS
// banks) and the LDS it takes
inline int attention_rows_stride(int n_cap) { return ((n_cap + 63) & ~63) + 20; }
inline size_t attention_rows_lds_bytes(int R, int hd, int n_cap) {
  return ((size_t)R * attention_rows_stride(n_cap) + 256 + 4 * 1024 + (size_t)R * ((hd + 15) & ~15)) * sizeof(float);
}
inline size_t attention_step_lds_bytes(int hd, int n_cap) {
  return ((size_t)((n_cap + 15) & ~15) + 256 + kStepWaves * 1024 + 2 * (size_t)((hd + 15) & ~15)) * sizeof(float);
}

enum class AttnKernel {
  kStep,       // attention_step_kernel: a workgroup per (token, head)
  kRows4,      // attention_rows_kernel, 4 rows a workgroup
  kRows8,      //   and 8
  kPrefill64,  // attention_prefill64_kernel (the append inside)
  kPrefill,    // attention_prefill_kernel
  kDecode64,   // attention_decode64_kernel
  kWhole,      // attention_kernel, its score row in LDS
  kGlobal,     // attention_kernel, its score rows in global memory
};

struct AttnCall {
  int T;         // query tokens
  int n_cap;     // score slots: pos0 + T, or with the position in device memory the whole cache
  bool pos_dev;  // the position is in device memory (T == 1)
  int n_heads, n_kv, hd;
  bool quant;     // the output is asked for as the next GEMM's operand too (T > 1, head size 64)
  bool aligned;   // the key cache starts on 16 bytes
};

inline AttnKernel attention_route(const AttnCall& c) {
  const bool fuse = c.T == 1;
  const int grp = c.n_heads / c.n_kv;
  const int64_t pairs = (int64_t)c.T * c.n_heads;
  // The step and rows kernels copy key rows to LDS 16 bytes at a time; a key cache that starts elsewhere takes the kernels
  // that load them into registers (at head size 64 those that it took before: they copy rows too, except attention_kernel).
  //
  // A chunk of at most one (token, head) per CU: a 1024-thread workgroup each (32 heads of size 128 over 1000 cached
  // positions: 35 / 38 us for 2 / 8 tokens, against 51 us with rows of four in 256-thread workgroups; 16 tokens 55 against
  // 52). At head size 64 only where no GEMM operand is asked for, and past 128 positions, where attention_prefill64_kernel,
  // which has the append inside, starts a second chunk of rows: it takes 7.0 / 7.6 / 9.8 / 10.3 / 12.0 / 13.3 / 34.6 us for
  // 8 tokens of 9 heads over 96 / 128 / 144 / 192 / 256 / 288 / 1000 positions, the append and the step kernel 8.5 / 8.9 /
  // 9.1 / 9.8 / 10.8 / 11.2 / 21.9 (32 heads over 8 kv heads, 8 tokens: 7.1 / 7.7 / 9.7 / 10.4 / 12.2 / 13.4 / 35.6 and 8.2
  // / 8.6 / 9.0 / 9.5 / 10.4 / 11.2 / 23.2; 2 to 64 tokens alike). One token: always, but for the head-size-64 kernel's
  // caches (it takes the step's rows before it knows the position: 6.0 against 8.6 us at 200 positions, 15.4 against 19.9 at
  // 700).
  const bool step_fits = c.aligned && grp < 65536 && attention_step_lds_bytes(c.hd, c.n_cap) <= kMaxAttnLds;
  const bool step = step_fits && (fuse ? c.hd != 64 || attention_decode_lds_bytes(c.n_cap) > kMaxAttnLds
                                       : !c.pos_dev && pairs <= 256 && (c.hd != 64 || (!c.quant && c.n_cap > kPfRows)));
  if (step) return AttnKernel::kStep;
  // Longer chunks: attention_rows_kernel, at head size 64 from 4096 (token, head) pairs on (9 heads: 512 tokens 31 against
  // 48 us with attention_prefill64_kernel, 128 tokens 11 against 8.4; 32 heads, 64 tokens at 600 positions 34 against 32).
  // R = 8 rows a workgroup read the keys half as often as 4; 4 fill the chip at fewer rows and keep more workgroups per CU
  // where the score rows are long (32 heads of size 128 over 8 kv heads, 4 and 8 rows: 96 / 128 / 256 / 320 tokens at 256
  // positions 34 / 40 / 76 / 100 and 39 / 41 / 71 / 90 us; 256 at 600 / 1500 131 / 277 and 121 / 268, 384 at 600 / 1500 205
  // / 401 and 203 / 648, 512 at 1500 / 3000 545 / 1296 and 898 / 1605).
  auto groups = [&](int R) { return ((int64_t)c.T * grp + R - 1) / R; };
  const int R = c.n_kv * groups(8) >= 1024 && 3 * attention_rows_lds_bytes(8, c.hd, c.n_cap) <= kMaxLds ? 8 : 4;
  if (!fuse && !c.pos_dev && c.aligned && groups(R) < 65536 && (c.hd != 64 || pairs >= 4096) &&
      attention_rows_lds_bytes(R, c.hd, c.n_cap) <= kMaxAttnLds)
    return R == 8 ? AttnKernel::kRows8 : AttnKernel::kRows4;
  if (!fuse && c.hd == 64 && !c.pos_dev && attention_prefill64_lds_bytes(c.n_cap) <= kMaxAttnLds) return AttnKernel::kPrefill64;
  if (!fuse && c.hd == 64 && attention_prefill_lds_bytes(c.n_cap) <= kMaxAttnLds) return AttnKernel::kPrefill;
  if (fuse && c.hd == 64 && attention_decode_lds_bytes(c.n_cap) <= kMaxAttnLds) return AttnKernel::kDecode64;
  return attention_lds_bytes(c.hd, c.n_cap) <= kMaxAttnLds ? AttnKernel::kWhole : AttnKernel::kGlobal;
}

// Bytes of global score rows the call needs (0 unless it takes attention_kernel with its score rows in global memory)
inline size_t attention_global_score_bytes(const AttnCall& c) {
  if (attention_route(c) != AttnKernel::kGlobal) return 0;
  return (size_t)c.T * c.n_heads * (size_t)((c.n_cap + 63) & ~63) * sizeof(float);
}

// ---------------------------------------------------------------- int8 GEMM

constexpr int kLds16MaxBlocks = 48;  // gemm_lds16_kernel: rows of at most this many 32-blocks (K <= 1536)

// Whether gemm_split16_kernel (K split over a workgroup's waves) takes a GEMM of nb 32-blocks per row and T tokens that makes
// `wgs` of its workgroups (row tiles in eights, times groups of 16 tokens). swiglu: gate and up; token: one scale per token;
// ring: the ring kernel would take the call (gemm_wave16_kernel otherwise).
// Its time goes with its workgroups; gemm_wave16_kernel's hardly does until it fills the chip, so there is a count past
// which it is the faster one, higher the more a workgroup of the split has to gain. A workgroup walks K in whole rounds of
// 16 blocks, so workgroups are counted with nb rounded up to those. Times in us, the other kernel's first, then the split's
// (256 CUs):
//   q4, scale per block   4096 x 14336 at 16 / 64 / 128 / 256 tokens (256 / 1024 / 2048 / 4096 workgroups): 104 / 94 / 123 /
//                         145, 22 / 56 / 104 / 231; 8192 x 2048 at 64 / 65 tokens (2048 / 2560): 24 / 24, 23 / 26
//   q8, scale per block   4096 x 4096 at 96 / 112 / 128 tokens (1536 / 1792 / 2048): the split takes 0.82 / 0.93 / 1.02 of
//                         the other's time; 2048 x 2048 at 192 / 256 (1536 / 2048) 0.92 / 1.13
//   q4, scale per token   1536 x 1568 at 192 / 224 tokens (1152 / 1344 of 49 blocks): 15.8 / 15.9, 15.1 / 17.0; 2048 x 2048
//                         at 192 / 256 (1536 / 2048) 0.95 / 1.14; 4096 x 4096 at 112 (1792) 0.90; 4096 x 14336 at 128 (2048)
//                         0.90
//   q8, scale per token   (no rescale: sums of integers) 4096 x 4096 / 4096 x 14336 at 128 tokens (2048): 0.80 / 0.65
//   SwiGLU q4             14336 x 4096 at 16 / 17 to 32 tokens (896 / 1792): 0.9 / 1.05 (scale per block), 0.95 / 1.2 (per
//                         token); 1536 x 1568 at 128 / 160 (768 / 960 of 49 blocks): 0.94 / 1.08, 0.96 / 1.12
//   SwiGLU q8, per token  4096 x 4096 at 64 tokens (1024) 0.80, 1536 x 1568 at 192 (1152 of 49 blocks) 0.82, 14336 x 4096 at
//                         17 (1792) 0.99
//   SwiGLU q8, per block  (82 KB of LDS: one workgroup per CU) 14336 x 4096 at 16 (896): 31.7, 45.3; 11008 x 4096 at 16
//                         (688): 30.3, 35.1; 8192 x 4096 at 16 (512) 0.85; 2048 x 2048 at 64 / 65 (512 / 640) 0.96 / 1.26;
//                         1536 x 1568 at 48 (288 of 49 blocks): 15.1, 15.8
// More tokens over few rows fill the chip with the other's workgroups earlier (256 x 2048 q8 at 1536 tokens, 1536 workgroups
// 1.08, 256 x 4096 0.92; as SwiGLU q4 256 x 2048 / 4096 at 1024 tokens, 1024 workgroups 1.05 / 1.03). The ring kernel, which
// serves what makes 128 tiles of 128 rows x 64 tokens, is slower at few tokens: 16384 x 4096 at 16 tokens (1024 workgroups)
// 0.52 q4, 0.65 q8, SwiGLU 0.26 and 0.48; 32000 x 4096 at 16 (2000) 0.84 and 1.06, per token 0.76 and 1.00.
inline bool gemm_split16_route(bool q8, bool swiglu, bool token, bool ring, int nb, int T, int64_t wgs) {
  if (nb <= kLds16MaxBlocks) return false;
  const int64_t load = wgs * ((nb + 15) / 16 * 16) / nb;
  const bool many = T > (q8 && token ? 1024 : 768);
  if (swiglu) {
    if (q8 && !token && !ring) return load <= (nb < 64 || (many && nb < 128) ? 340 : 530);
    return load <= (many ? (nb < 128 ? 900 : 1100) : q8 && token ? 1536 : 1200);
  }
  if (many) return load <= (q8 && nb < 128 ? 1200 : 1600);
  if (q8) return load <= (!token ? 1840 : ring ? 1900 : 2100);
  return load <= (!token || ring || nb >= 256 ? 2100 : nb >= 96 ? 1840 : 1700);
}

// ---------------------------------------------------------------- f32-activation GEMM (more than one token)

// Rows x tokens of a workgroup: gemm_f32act_kernel, and the tiles of gemm_f32act_tile_kernel
enum class F32Gemm { k64x2, k16x8, k32x16, k64x16, k64x32 };

// N: the output rows of the n targets (SwiGLU: the gate's). Times in us at K = 4096 q4 unless said otherwise.
//
// Tiles: the largest that makes at least two workgroups per CU (one for 32 x 16), else 16 x 8: at 4096 rows and 256 / 128 /
// 64 / 32 / 16 tokens 64 x 32 tiles take 189 / 114 / 109 / 105 / 95, 64 x 16 220 / 115 / 71 / 68 / 67, 32 x 16 240 / 124 /
// 65 / 41 / 40, 16 x 8 343 / 179 / 95 / 50 / 29. A token tile that is mostly empty has waves that only stage: 64 x 32 needs
// more than 16 tokens (49152 x 576 at 2 / 8 / 16 tokens 35 / 36 / 38, with 64 x 16 26 / 26 / 32) and, with q8 weights, up to
// 64 tokens, more than half of its last tile (32768 x 1024 at 33 / 48: 124 / 129, 64 x 16 91 / 95; q4 96 / 101 and 88 / 92);
// up to 5 tokens, and 6 below K = 2048, there are 16 x 8 and 64 x 16 only (8192 x 2048 at 2 to 5: 15.4, 32 x 16 19.5; 24576
// x 576 at 5: 13.6 and 15.8; 14336 x 4096 at 6: 44 and 42). SwiGLU holds both selections, so at most 32 x 16 (3648 x 1088,
// 175 tokens, with its down projection: 148, 185 with 64 x 16), and 16 x 8 up to 384 of those: between 256 and 384 they run
// in two rounds of the CUs (1536 x 576 q8, 93 tokens, 288 of them, with its down projection: 35 against 42; 4096 rows at 17
// tokens, 256 half-empty ones: 56 against 60; with whole tiles in one round they would be the faster, 4096 rows at 32 tokens
// 86 against 73, 2048 x 2048 at 64 46 against 39).
//
// gemm_f32act_kernel (every weight dequantized for each pair of tokens, but all lanes at work): few tokens over many rows,
// and the shortest rows at a middling number of outputs, where the tiles' staging is not repaid. Its time first, then the
// tiles':
//   2 tokens   16384 x 576 / 1024 10.0 / 15.7 and 10.8 / 13.6; 24576 x 576 / 1024 / 2048 10.0 / 16.3 / 38.6 and 13.3 / 18.4
//              / 35; 32000 x 4096 72 and 82 (SwiGLU 93 and 124); 49152 x 576 12.5 and 26; 128256 x 2048 82 and 152; 14336 x
//              4096 65 and 40
//   3 or 4     24576 x 256 / 576 / 1024 6.6 / 10.8 / 21.2 and 8.8 / 13.3 / 20.5; 49152 x 576 18.9 and 25.5 (SwiGLU 34.7 and
//              37.1); 32000 x 4096 89 and 81; 128256 x 2048 142 and 150 to 160
//   5, 6       24576 x 256 8.2 and 8.8, x 576 15.8 and 13.6
//   8          49152 x 64 / 160 / 192 8.4 / 12.0 / 14.5 and 11.2 / 14.7 / 15.2
//   17         16384 x 192 11.2 and 12.2, 49152 x 192 as SwiGLU 56 and 62 (a second tile of one token)
//   9 to 33    with a quarter of the 16-token tiles empty, 49152 x 32 at 12 / 24 / 33 as SwiGLU q8 15.5 / 29 / 41 and 20 /
//              39 / 52; without (16, 32) 49152 x 64 30 and 22 at 16
//   K = 64     4096 x 33 tokens 5.1 and 6.0, 1536 x 93 5.0 and 5.8; 512 x 64 3.9 and 3.4, 4096 x 128 10.1 and 9.0
inline F32Gemm f32_gemm_route(bool q8, bool swiglu, int T, int K, const int* N, int n) {
  auto groups = [&](int rows) {
    int64_t g = 0;
    for (int i = 0; i < n; ++i) g += (N[i] + rows - 1) / rows;
    return g;
  };
  const int64_t rows = groups(1), outputs = rows * T;
  const bool many = rows > 24576;
  bool pair = false;
  if (rows <= 12288) pair = K <= 64 && outputs >= 40000 && outputs <= (swiglu ? 240000 : 400000);
  else if (T <= 2) pair = K <= 640 || many || (K < 2048 && rows > 20480);
  else if (T <= 4) pair = K <= (many || !swiglu ? 640 : 384) || rows > 98304;
  else if (T <= 6) pair = K <= (swiglu ? 128 : 256);
  else if (T <= 8) pair = K <= (swiglu ? 96 : 192);
  else if (T > 16 && T <= 20) pair = swiglu ? K <= (many ? 320 : 192) : !many && K <= 192;
  else if (T <= 40) pair = K <= 64 && 4 * T <= 48 * ((T + 15) / 16) && (swiglu || !many || T <= 12);
  if (pair && groups(64) <= 65535) return F32Gemm::k64x2;
  auto wgs = [&](int r, int t) { return groups(r) * ((T + t - 1) / t); };
  if (T <= (K < 2048 ? 6 : 5)) return !swiglu && wgs(64, 16) >= 512 ? F32Gemm::k64x16 : F32Gemm::k16x8;
  if (!swiglu && T > 16 && (!q8 || T > 64 || (T - 1) % 32 >= 16) && wgs(64, 32) >= 512) return F32Gemm::k64x32;
  if (!swiglu && wgs(64, 16) >= 512) return F32Gemm::k64x16;
  return wgs(32, 16) >= (swiglu ? 384 : 256) ? F32Gemm::k32x16 : F32Gemm::k16x8;
}

// Token tiles of one launch of gemm_f32act_tile_kernel over `groups` row groups: a dispatch counts a dimension's threads in
// 32 bits, and a workgroup has 512. 0: more row groups than one grid takes. (The token range of a launch costs nothing; a
// second grid dimension in the kernel took 0.3 us of 15.)
inline int f32_gemm_tiles_per_launch(int64_t groups) {
  constexpr int64_t kMost = int64_t(1) << 22;
  return groups < 1 ? 0 : (int)(kMost / groups);
}

// ---------------------------------------------------------------- f32-activation q4 GEMV (one token)

// gemv_f32act_q4_wide_kernel: nb groups per row spread over a workgroup's threads (256 up to 256 groups, which then hold
// several sets of rows; else nb rounded up to whole waves), 8 rows each
constexpr int kF32QRows = 8;
inline bool f32q4_wide_ok(int nb, int H) { return nb > 64 && nb <= 512 && H >= kF32QRows && H % kF32QRows == 0; }
inline int f32q4_wide_sets(int nb) { return nb <= 256 ? 256 / nb : 1; }
inline int f32q4_wide_threads(int nb) { return nb <= 256 ? 256 : (nb + 63) & ~63; }

// Whether it takes a call that gemv_f32act_q4_kernel can take too (rows: the outputs, SwiGLU's of one selection; norm:
// RMSNORM inside). It reads x and, with norm, takes the ordered sums once for 8 rows and more; against that stand threads
// without a group where nb does not fill them, and few workgroups where the rows are few. Times in us,
// gemv_f32act_q4_kernel's first:
//   norm          4096 x 2080 / 2400 / 4096 / 8192 11.3 / 12.3 / 20.3 / 57 and 8.8 / 9.4 / 11.4 / 20; 14336 x 2080 / 2400 /
//                 2720 / 4096 13.8 / 15.6 / 17.8 / 36 and 16.0 / 16.7 / 17.6 / 19; 32768 x 2080 27 and 22
//   norm, SwiGLU  256 x 2080 / 3072 / 3584 9.8 / 12.4 / 14.3 and 12.1 / 13.0 / 14.2; 1024 x 2080 12.7 and 12.2; 8192 x 2080
//                 15.6 and 17.2; 14336 x 2400 / 2720 / 2752 / 4096 24.9 / 27.3 / 27.0 / 53 and 27.3 / 28.4 / 25.9 / 30;
//                 65536 x 2080 / 2400 62 / 78 and 65 / 69
//   plain         4096 x 2080 / 3072 / 3584 / 4096 5.4 / 6.0 / 6.7 / 9.0 and 5.8 / 6.1 / 6.3 / 6.6; 576 / 1536 / 6144 / 8192
//                 x 4096 5.6 / 6.4 / 8.3 / 9.4 and 6.2 / 6.2 / 8.9 / 9.0; 2048 / 3072 / 8192 / 32768 x 4128 (half the
//                 threads) 7.5 / 7.3 / 10.2 / 31 and 5.9 / 7.7 / 12.3 / 41; 4096 / 6144 x 6144 (three quarters) 12.7 / 11.5
//                 and 8.6 / 12.8; 4096 / 14336 x 8192 19 / 38 and 9.4 / 27
//   SwiGLU        4096 x 2080 / 2720 / 3072 8.2 / 11.3 / 12.1 and 8.9 / 9.5 / 9.3; 14336 x 3072 / 4096 22.0 / 28.7 and 22.4
//                 / 23.9; 256 / 1024 x 4096 6.8 / 15.6 and 9.2 / 9.4; 8192 / 32768 x 4128 19.5 / 51 and 21.1 / 76
inline bool f32q4_wide_route(bool swiglu, bool norm, int nb, int64_t rows) {
  if (norm) {
    if (!swiglu) return nb >= 80 || rows <= 8192 || rows > 24576;
    return nb >= 112 || (nb >= 86 && rows >= 512) || (nb >= 75 && rows > 24576) || (rows >= 1024 && rows <= 6144);
  }
  const bool full = 100 * f32q4_wide_sets(nb) * nb >= 85 * f32q4_wide_threads(nb);  // 85% of the threads have a group
  if (nb >= 192) return full || rows <= 4096;
  if (swiglu) {
    if (nb >= 128) return rows >= 512 && (full || rows <= 4096);
    return nb >= 86 && rows >= (nb >= 112 ? 1024 : 2048) && rows <= (full ? 14336 : 4096);
  }
  if (nb < 128) return false;
  return full ? rows >= 1536 && (rows <= 4096 || rows >= 8192) : rows >= 512 && rows <= (nb >= 160 ? 4096 : 2048);
}

}  // namespace elmh
