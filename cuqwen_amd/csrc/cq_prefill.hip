// Batched prefill for gfx950: the prompt goes through the layers M tokens at
// a time instead of one decode step per token (the reference's prefill loop,
// src/main.cu:87-92, calls qwen_forward once per prompt token; batched
// prefill is its roadmap item, README.md:145).
//
// Per layer and chunk of M tokens:
//   RMSNorm         x -> half(x * w) and rsqrt(mean(x^2) + eps) per token
//                   (the decode GEMVs' fused RMSNorm, kernels.cu:689-751):
//                   with the embedding for layer 0, later in the epilogue of
//                   the residual GEMM that produces x
//   pf_gemm<QKV>    Q / K / V rows, bias, RoPE at each token's position, K / V
//                   into the cache (kernels.cu:402-474, :370-398, :326-347)
//   pf_attention    causal FlashDecoding over the cache (kernels.cu:105-288
//                   with a per-token key limit)
//   pf_gemm<RESID>  O-proj + residual (kernels.cu:640-687), + RMSNorm
//   pf_gemm<SWIGLU> (kernels.cu:523-585), pf_gemm<RESID> (down), + RMSNorm
// The GEMMs are M > 1, so they run on the matrix cores: each wave dequantizes
// its weight rows in registers (int4 / int8 to exact small-integer fp16,
// times the group's fp16 scale) as the A operand of v_mfma_f32_16x16x32_f16
// and takes 16-token slices of the activation tile, staged in LDS, as the B
// operand.
//
// Activation layout: the inputs of the GEMMs (normed x, attention output,
// SwiGLU output) are stored in the order in which the weights' unpack yields
// pairs (int4: each 8-group as [0,4,1,5,2,6,3,7] with the odd elements / 16;
// int8 / fp16: natural), so neither operand needs a shuffle in the main loop.
#include "cq_attention.h"
#include "cq_gemv.h"
#include "cq_prefill.h"

#include <algorithm>
#include <type_traits>

namespace cq {

constexpr int kPfWaves = 8;
constexpr int kPfThreads = kPfWaves * 64;
constexpr int kPfK = 128;         // K per main-loop step (one quantization group)
constexpr int kPfMaxSplit = 8;
constexpr size_t kPfKeptPart = 64u << 20;   // partials that keep_tile's split rule reckons with

// ------------------------------------------------------------- row norm
// RMSNorm of one token row by one block (dim a multiple of 8): A row =
// half(x * w) in the layout of the weights' format, inv = rsqrt(mean(x^2) +
// half(eps)).  Without w, A = x (in the layout) and no inv.  Thread t takes
// the 8-element groups t, t + blockDim.x, ... (the layout permutes within a
// group, so each group is one 16-byte load and one 16-byte store).
__device__ __forceinline__ void pf_norm_row(const _Float16* xr, const _Float16* w, float eps, int dim, _Float16* ar,
                                            float* inv_m, bool int4, float* red) {
  float ss = 0.f;
  for (int g = threadIdx.x; g < dim / 8; g += blockDim.x) {
    const h8_t xv = __builtin_bit_cast(h8_t, load_u4(xr + 8 * g));
    h8_t wv;
    if (w) wv = __builtin_bit_cast(h8_t, load_u4(w + 8 * g));
    h8_t o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = (float)xv[e];
      ss = fmaf(v, v, ss);
      // half(x * w) first (the decode GEMVs' staging), then the layout's scale
      const float y = w ? (float)(_Float16)(v * (float)wv[e]) : v;
      o[pf_pos(e, int4)] = pf_val(y, e, int4);
    }
    *reinterpret_cast<u4_t*>(ar + 8 * g) = __builtin_bit_cast(u4_t, o);
  }
  if (w) {
    ss = block_sum(ss, red);
    if (threadIdx.x == 0) *inv_m = rsqrtf(ss / (float)dim + (float)(_Float16)eps);
  }
}

// One block per token row.
__global__ __launch_bounds__(256) void pf_norm_rows(const _Float16* x, const _Float16* w, float eps, int dim,
                                                    _Float16* A, float* inv, bool int4) {
  __shared__ float red[16];
  const int m = blockIdx.x;
  pf_norm_row(x + (int64_t)m * dim, w, eps, dim, A + (int64_t)m * dim, inv + m, int4, red);
}

// Embedding rows of the chunk's tokens (kernels.cu:85-103), the first layer's
// input norm of them, and the RoPE sines and cosines of their positions,
// [M][half] each: every layer's QKV epilogue reads them (the angle is reduced
// in double: computed per pair they were a third of the unsplit epilogue).
struct PfEmbedArgs {
  const u4_t* embed;
  const int* tokens;
  _Float16* x;
  int dim;
  const double* inv_freq;
  int half, pos0;
  float* rope;
  const _Float16* norm_w;
  float eps;
  _Float16* norm_out;
  float* norm_inv;
  bool int4;
};
__global__ __launch_bounds__(256) void pf_embed(const PfEmbedArgs a) {
  __shared__ float red[16];
  const int m = blockIdx.x, vec_dim = a.dim / 8;
  const int64_t t = a.tokens[m];
  _Float16* xr = a.x + (int64_t)m * a.dim;
  for (int i = threadIdx.x; i < vec_dim; i += blockDim.x) *reinterpret_cast<u4_t*>(xr + 8 * i) = a.embed[t * vec_dim + i];
  if ((int)threadIdx.x < a.half) {
    float* sn = a.rope + (int64_t)m * a.half + threadIdx.x;
    rope_sincos(a.pos0 + m, a.inv_freq[threadIdx.x], sn, sn + (int64_t)gridDim.x * a.half);
  }
  // reads back the groups this thread has just written
  pf_norm_row(xr, a.norm_w, a.eps, a.dim, a.norm_out + (int64_t)m * a.dim, a.norm_inv + m, a.int4, red);
}

// ------------------------------------------------------------------ GEMM
template <int Q> struct PfW;   // 16-byte weight loads per lane per 128-wide step
template <> struct PfW<CQ_QUANT_INT4> { static constexpr int LOADS = 1; };
template <> struct PfW<CQ_QUANT_INT8> { static constexpr int LOADS = 2; };
template <> struct PfW<CQ_QUANT_FP16> { static constexpr int LOADS = 4; };

// The A operand (8 fp16 weights in the order [0,4,1,5,2,6,3,7] of true k
// j*32 + s*8 + e) for sub-step s from the lane's loaded bytes.
template <int Q>
__device__ __forceinline__ h8_t pf_unpack(const u4_t* w, int s, uint32_t m_lo, uint32_t m_hi, uint32_t magic) {
  u4_t o;
  if constexpr (Q == CQ_QUANT_INT4) {
    // word s: nibbles e0..e7 of true k j*32 + s*8 + e; after ^0x88888888 each
    // is n = q + 8.  (1024 + n) - 1032 = q for e0 e4 e2 e6; the odd nibbles
    // stay in place: (1024 + 16 n) - 1152 = 16 q against activations / 16.
    const uint32_t f = w[0][s] ^ kInt4Flip, f8 = f >> 8;
    const h2_t blo = {(_Float16)-1032.f, (_Float16)-1032.f}, bhi = {(_Float16)-1152.f, (_Float16)-1152.f};
    o.x = as_u32(as_h2(and_or(f, m_lo, 0x64006400u)) + blo);    // (e0, e4)
    o.y = as_u32(as_h2(and_or(f, m_hi, 0x64006400u)) + bhi);    // (16 e1, 16 e5)
    o.z = as_u32(as_h2(and_or(f8, m_lo, 0x64006400u)) + blo);   // (e2, e6)
    o.w = as_u32(as_h2(and_or(f8, m_hi, 0x64006400u)) + bhi);   // (16 e3, 16 e7)
  } else if constexpr (Q == CQ_QUANT_INT8) {
    // bytes 8s..8s+7 in natural order: (1152 + q) pairs, minus 1152
    const uint32_t f0 = w[s >> 1][(s & 1) * 2] ^ kInt8Flip, f1 = w[s >> 1][(s & 1) * 2 + 1] ^ kInt8Flip;
    const h2_t b = {(_Float16)-kInt8Bias, (_Float16)-kInt8Bias};
    o.x = as_u32(as_h2(int8_pair(f0, magic, 0)) + b);
    o.y = as_u32(as_h2(int8_pair(f0, magic, 1)) + b);
    o.z = as_u32(as_h2(int8_pair(f1, magic, 0)) + b);
    o.w = as_u32(as_h2(int8_pair(f1, magic, 1)) + b);
  } else {
    o = w[s];   // fp16, natural order
  }
  return __builtin_bit_cast(h8_t, o);
}

// Row r of the concatenated output (QKV: q rows, then k, then v) -> matrix.
__device__ __forceinline__ int pf_mat(const PfGemmArgs& a, int row, int* local) {
  if (row < a.rows[0]) { *local = row; return 0; }
  if (row < a.rows[0] + a.rows[1]) { *local = row - a.rows[0]; return 1; }
  *local = row - a.rows[0] - a.rows[1];
  return 2;
}

// Four consecutive rotated pairs (rows local + e, local + hd/2 + e of matrix
// mat, e < 4) of token m: q into the Q buffer, k / v into the fp16 cache at
// position pos0 + m.
__device__ __forceinline__ void pf_qkv_store4(const PfGemmArgs& a, int mat, int local, int m, h4_t h0, h4_t h1) {
  const int hd = a.head_dim, half = hd / 2;
  if (mat == 0) {
    *reinterpret_cast<h4_t*>(a.out + (int64_t)m * a.rows[0] + local) = h0;
    *reinterpret_cast<h4_t*>(a.out + (int64_t)m * a.rows[0] + local + half) = h1;
    return;
  }
  const int kvh = local / hd, i = local % hd, pos = a.pos0 + m;
  if (mat == 1) {   // four consecutive elements of a K row are contiguous in the tiled cache
    *reinterpret_cast<h4_t*>(a.kcache + kv_k_offset(kvh, pos, i, a.max_seq, hd)) = h0;
    *reinterpret_cast<h4_t*>(a.kcache + kv_k_offset(kvh, pos, i + half, a.max_seq, hd)) = h1;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a.vcache[kv_v_offset(kvh, pos, i + e, a.max_seq, hd)] = h0[e];
      a.vcache[kv_v_offset(kvh, pos, i + half + e, a.max_seq, hd)] = h1[e];
    }
  }
}
// RoPE of four consecutive pairs of token m (the table of pf_embed).
__device__ __forceinline__ void pf_rope4(const PfGemmArgs& a, int m, int i, float* y0, float* y1) {
  const int half = a.head_dim / 2;
  const float* p = a.rope + (int64_t)m * half + i;
  const f4_t sn = *reinterpret_cast<const f4_t*>(p), cs = *reinterpret_cast<const f4_t*>(p + (int64_t)a.M * half);
#pragma unroll
  for (int e = 0; e < 4; ++e) rope_apply(y0[e], y1[e], sn[e], cs[e]);
}

// One (token, kv head) row into the quantized cache: s = max|x| / code max
// (a zero row keeps s = 0 and q = 0), q = code of x / s (int8: rint clamped
// to +-127; E4M3: round to nearest even); element d from value(d).
template <typename F>
__device__ __forceinline__ void pf_kv8_store(const PfGemmArgs& a, int mat, int kvh, int pos, float amax, F value) {
  const int hd = a.head_dim;
  const bool f8 = a.kv_fmt == CQ_KV_FP8;
  const float sc = amax / (f8 ? kv_code_max<CQ_KV_FP8>() : kv_code_max<CQ_KV_INT8>());
  int8_t* c = mat == 1 ? a.kcache8 : a.vcache8;
  for (int d = 0; d < hd; ++d) {
    const float v = value(d) / sc;
    const int8_t q = sc == 0.f ? (int8_t)0 : (f8 ? kv_encode<CQ_KV_FP8>(v) : kv_encode<CQ_KV_INT8>(v));
    c[mat == 1 ? kv8_k_offset(kvh, pos, d, a.max_seq, hd) : kv8_v_offset(kvh, pos, d, a.max_seq, hd)] = q;
  }
  (mat == 1 ? a.kscale : a.vscale)[(int64_t)kvh * a.max_seq + pos] = sc;
}

template <int Q>
__device__ __forceinline__ void pf_load_w(const PfGemmArgs& a, const char* rowp, int ks, int j, u4_t* w) {
  constexpr int L = PfW<Q>::LOADS;
  // 64*L bytes of the row per step (panels: one panel row, panel stride N rows), L*16 per lane
  const int64_t kstep = a.panels ? (int64_t)a.N * (64 * L) : 64 * L;
  const char* p = rowp + (int64_t)ks * kstep + j * (L * 16);
#pragma unroll
  for (int i = 0; i < L; ++i) w[i] = load_u4(p + i * 16);
}

// Tile shape: RT 16-row slices per wave (SwiGLU: RT/2 gate and RT/2 up
// slices of the same output rows), 8 token slices of 16 per wave (the unpack
// of a weight fragment is shared by 8 matrix instructions); a block is 8
// waves over the same 128 tokens, two per SIMD.
template <int Q> struct PfTile { static constexpr int RT = 2; };
constexpr int kPfTT = 8;                         // token slices per wave
constexpr int kPfTok = 16 * kPfTT;               // tokens per block
template <int Q, int MODE> struct PfShape {
  static constexpr int NMAT = MODE == GM_SWIGLU ? 2 : 1;
  static constexpr int RT = PfTile<Q>::RT / NMAT;   // row slices per matrix
  static constexpr int WROWS = RT * 16;              // output rows per wave
  static constexpr int BN = kPfWaves * WROWS;        // output rows per block
};

// The block's (row block, token block) from its dispatch index, so that all
// token blocks of a row block run on one XCD and share its weight rows in
// that XCD's L2: dispatch goes round-robin over the 8 XCDs, so XCD x runs
// blocks x, x + 8, ...; those take a contiguous range of row-major tiles.
__device__ __forceinline__ void pf_block_tile(int n_tb, int* rb, int* tb) {
  const int id = blockIdx.x, n = gridDim.x;
  const int xcd = id & 7, k = id >> 3, base = n >> 3, rem = n & 7;
  const int L = xcd * base + min(xcd, rem) + k;
  *rb = L / n_tb;
  *tb = L % n_tb;
}

// 16-byte slot of K chunk c (0..15) in activation row t of a GEMM LDS stage,
// and, the map being an involution, the chunk held in slot c.  A 16-byte LDS
// read on gfx950 serves each 32-lane half of a wave in two passes of 16
// lanes split by the parity of lane bits 2..4 (lanes 0-3, 12-15, 20-27 and
// 4-11, 16-19, 28-31; measured with per-lane-pair probes and
// SQ_LDS_BANK_CONFLICT); a pass takes one cycle when its 16 lanes hit 16
// different 16-byte bank groups of the 256-byte bank row.  The B read has
// lane (r, j) = (lane % 16, lane / 16) at row r, chunk 4j + s4: XOR with
// f(r) = r ^ 8 * (bit 2 of r ^ bit 3 of r) gives every pass 16 different
// slots, where XOR with r alone puts two lanes of each pass on one slot.
__device__ __forceinline__ int pf_slot(int t, int c) {
  const int r = t & 15;
  return c ^ r ^ ((((r >> 2) ^ (r >> 3)) & 1) << 3);
}

// C^T tile of a wave: NMAT matrices (SwiGLU: gate and up) x RT row slices of
// 16 x 8 token slices of 16; lane holds rows 4*(lane/16)+v, token lane%16.
// The group scale multiplies the unpacked weights (half(q * s), one packed
// multiply per pair), so the matrix cores accumulate the whole K range
// directly into the tile.
template <int Q, int MODE, bool SPLIT>
__global__ __launch_bounds__(kPfThreads, 2) void pf_gemm_kernel(const PfGemmArgs a) {
  using SH = PfShape<Q, MODE>;
  constexpr int NMAT = SH::NMAT, RT = SH::RT, WROWS = SH::WROWS, BN = SH::BN, TT = kPfTT;
  constexpr int L = PfW<Q>::LOADS;
  constexpr int XS = kPfTok * kPfK;                         // halves of one activation stage
  constexpr int OT = MODE == GM_QKV ? kPfTok / 2 * (BN + 4) : 0;   // QKV epilogue tile (half the tokens x rows)
  constexpr int NS = 2;                                     // LDS stages
  // the epilogues reuse the stages: QKV tile, residual fp32 half tile
  constexpr int SM = std::max({NS * XS, OT, kPfTok / 2 * (BN + 4) * 2});
  __shared__ __align__(16) _Float16 smem[SM];
  _Float16* xs0 = smem;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int r = lane & 15, j = lane >> 4;
  const int n_tb = (a.M + kPfTok - 1) / kPfTok;
  int rb, tb;
  pf_block_tile(n_tb, &rb, &tb);
  const int m0 = tb * kPfTok;
  const int nb0 = rb * BN;                     // first output row of the block
  const int nw0 = nb0 + wave * WROWS;          // first output row of the wave
  const int K = a.K, nks = K / kPfK;
  // split-K: block z of gridDim.z sums K steps [kb, ke) into an fp32 partial
  const int kb = SPLIT ? (int)((int64_t)blockIdx.z * nks / gridDim.z) : 0;
  const int ke = SPLIT ? (int)((int64_t)(blockIdx.z + 1) * nks / gridDim.z) : nks;

  // weight row (A operand row r of each slice) and its scale row
  const int64_t sstep = a.panels ? a.N : 1;   // scale stride of one K step
  const char* rowp[NMAT][RT];
  const _Float16* srow[NMAT][RT];
#pragma unroll
  for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      int local, row = min(nw0 + rt * 16 + r, a.N - 1);
      const int mat = MODE == GM_SWIGLU ? mt : pf_mat(a, row, &local);
      if (MODE == GM_SWIGLU) local = row;
      // row-major: step ks is bytes [64*L*ks, 64*L*(ks+1)) of the row; panels: row
      // `local` of panel ks (wo_to_panels), scales [panel][N]
      const int64_t rbytes = a.panels ? 64 * L : Q == CQ_QUANT_INT4 ? K / 2 : Q == CQ_QUANT_INT8 ? K : 2 * K;
      rowp[mt][rt] = reinterpret_cast<const char*>(sel3(a.W, mat)) + (int64_t)local * rbytes;
      srow[mt][rt] = Q == CQ_QUANT_FP16 ? nullptr : sel3(a.S, mat) + (a.panels ? (int64_t)local : (int64_t)local * (K / kGroup));
    }

  // Activation tiles: global -> registers one step ahead, then 16-byte LDS
  // stores into one of two stages at the start of the step that reads them
  // (measured faster than global_load_lds straight into LDS).  A stage holds
  // 128 token rows of 256 bytes; 16-byte slot s of row t holds K chunk
  // pf_slot(t, s) (an involution), so the B-operand reads are free of bank
  // conflicts.  Piece q of a step (q = i * waves + wave) is rows
  // 4q .. 4q + 3: lane l holds row 4q + l / 16, slot l % 16.
  constexpr int XL = kPfTok / (4 * kPfWaves);
  u4_t xr[XL];
  auto x_load = [&](int ks) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int q = i * kPfWaves + wave, t = 4 * q + (lane >> 4), c = pf_slot(t, lane & 15);
      const int m = min(m0 + t, a.M - 1);
      xr[i] = load_u4(a.A + (int64_t)m * K + ks * kPfK + c * 8);
    }
  };
  auto x_store = [&](int stg) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int q = i * kPfWaves + wave;
      *reinterpret_cast<u4_t*>(xs0 + stg * XS + q * 512 + lane * 8) = xr[i];
    }
  };
  f4_t acc[NMAT][RT][TT];
#pragma unroll
  for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) acc[mt][rt][tt] = f4_t{0.f, 0.f, 0.f, 0.f};

  // Pipeline: at step k (after its barrier) the activations of step k+1
  // (into registers) and then the weights of step k+2 (into register set
  // k % 2) are requested; the K loop is unrolled by two so the weight
  // register sets keep compile-time indices.  At the start of step k a wave
  // waits until only the WL weight / scale loads of step k+1 are
  // outstanding, stores its piece of step k's activations into LDS stage
  // k % 2 (last read in step k-2, which every wave finished before step
  // k-1's barrier) and waits for the stores; the barrier then makes all
  // pieces visible.
  constexpr int WL = NMAT * RT * (L + (Q != CQ_QUANT_FP16 ? 1 : 0));
  static_assert(WL < 64, "vmcnt range");
  u4_t wv[2][NMAT][RT][L];
  _Float16 sv[2][NMAT][RT];
  auto load_w_step = [&](int ks, u4_t (&w)[NMAT][RT][L], _Float16 (&s)[NMAT][RT]) {
#pragma unroll
    for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        pf_load_w<Q>(a, rowp[mt][rt], ks, j, w[mt][rt]);
        if constexpr (Q != CQ_QUANT_FP16) s[mt][rt] = srow[mt][rt][(int64_t)ks * sstep];
      }
  };
  // Every load is issued unconditionally (step indices clamped to the last
  // step; the repeats past it are never used): with loads under branches the
  // compiler's wait-count tracking merges the paths conservatively and waits
  // for all loads, the next step's weight prefetch included, before the
  // activation stores of every step.
  load_w_step(kb, wv[0], sv[0]);
  x_load(kb);
  __builtin_amdgcn_sched_barrier(0);
  load_w_step(min(kb + 1, ke - 1), wv[1], sv[1]);

  const UnpackRegs uk = unpack_regs();
  auto step = [&](auto I, int ks) {
    constexpr int S = decltype(I)::value;   // weight register set of this step
    const int stg = (ks - kb) & 1;
    // simm16 of s_waitcnt on gfx9: vmcnt in bits [3:0] and [15:14], expcnt
    // [6:4], lgkmcnt [11:8]; the fields not waited on are left at their maxima
    __builtin_amdgcn_s_waitcnt(0x0F70 | (WL & 15) | ((WL >> 4) << 14));
    x_store(stg);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the LDS stores are done
    lds_barrier();
    const _Float16* xb0 = xs0 + stg * XS;
    h2_t s2[NMAT][RT];
    u4_t w[NMAT][RT][L];
#pragma unroll
    for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        s2[mt][rt] = h2_t{sv[S][mt][rt], sv[S][mt][rt]};
#pragma unroll
        for (int i = 0; i < L; ++i) w[mt][rt][i] = wv[S][mt][rt][i];
      }
    // activations first: the next step waits for them with the weights
    // requested here still in flight (the wait counts loads in issue order)
    x_load(min(ks + 1, ke - 1));
    __builtin_amdgcn_sched_barrier(0);
    load_w_step(min(ks + 2, ke - 1), wv[S], sv[S]);
    // B fragments of one sub-step
    auto read_b = [&](int s4, h8_t* xb) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)   // row tt*16 + r, K chunk 4j + s4 at slot pf_slot(r, 4j + s4)
        xb[tt] = *reinterpret_cast<const h8_t*>(&xb0[(tt * 16 + r) * kPfK + pf_slot(r, 4 * j + s4) * 8]);
    };
    // A fragments (dequantized weights) of sub-step s4
    auto unpack_a = [&](int s4, h8_t (&wa)[NMAT][RT]) {
#pragma unroll
      for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          h8_t u = pf_unpack<Q>(w[mt][rt], s4, uk.m_lo, uk.m_hi, uk.magic);
          if constexpr (Q != CQ_QUANT_FP16) {
            u4_t uu = __builtin_bit_cast(u4_t, u);
            uu.x = as_u32(as_h2(uu.x) * s2[mt][rt]);
            uu.y = as_u32(as_h2(uu.y) * s2[mt][rt]);
            uu.z = as_u32(as_h2(uu.z) * s2[mt][rt]);
            uu.w = as_u32(as_h2(uu.w) * s2[mt][rt]);
            u = __builtin_bit_cast(h8_t, uu);
          }
          wa[mt][rt] = u;
        }
    };
    constexpr int NMF = NMAT * RT * TT;   // matrix instructions per sub-step
    auto mfma_all = [&](const h8_t (&wa)[NMAT][RT], const h8_t* xb) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            acc[mt][rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[mt][rt], xb[tt], acc[mt][rt][tt], 0, 0, 0);
    };
    if constexpr (Q != CQ_QUANT_FP16) {
      // Software pipeline over the four sub-steps: the B fragments (LDS) and
      // A fragments (unpack) of sub-step s4 + 1 are produced while the
      // matrix instructions of s4 run; the scheduling groups interleave them
      // (the LDS reads first, then one matrix instruction and two vector
      // instructions at a time) so the unpack co-executes with the matrix
      // cores instead of alternating with them.  (The fp16 weight registers
      // leave no room for the second fragment set.)
      h8_t xb[2][TT];
      h8_t wa[2][NMAT][RT];
      read_b(0, xb[0]);
      unpack_a(0, wa[0]);
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        __builtin_amdgcn_sched_barrier(0);
        if (s4 < 3) {
          read_b(s4 + 1, xb[(s4 + 1) & 1]);
          unpack_a(s4 + 1, wa[(s4 + 1) & 1]);
        }
        mfma_all(wa[s4 & 1], xb[s4 & 1]);
        if (s4 < 3) {
          __builtin_amdgcn_sched_group_barrier(0x100, TT, 0);   // LDS reads
#pragma unroll
          for (int i = 0; i < NMF; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one matrix instruction
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two vector instructions
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        h8_t xb[TT];
        h8_t wa[NMAT][RT];
        read_b(s4, xb);
        unpack_a(s4, wa);
        mfma_all(wa, xb);
      }
    }
  };
  int ks = kb;
  for (; ks + 1 < ke; ks += 2) {
    step(std::integral_constant<int, 0>{}, ks);
    step(std::integral_constant<int, 1>{}, ks + 1);
  }
  if (ks < ke) step(std::integral_constant<int, 0>{}, ks);
  __syncthreads();   // every wave's last LDS reads are done before the QKV epilogue reuses the buffers

  if constexpr (SPLIT) {
    // fp32 partial [z][mat][M][N]; the split epilogue sums and finishes
#pragma unroll
    for (int mt = 0; mt < NMAT; ++mt)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
          const int n = nw0 + rt * 16 + 4 * j, m = m0 + tt * 16 + r;
          if (m < a.M && n + 3 < a.N) {
            *reinterpret_cast<f4_t*>(&a.part[(((int64_t)blockIdx.z * NMAT + mt) * a.M + m) * a.N + n]) = acc[mt][rt][tt];
          } else if (m < a.M) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
              if (n + v < a.N) a.part[(((int64_t)blockIdx.z * NMAT + mt) * a.M + m) * a.N + n + v] = acc[mt][rt][tt][v];
          }
        }
    return;
  }

  // ---- epilogues: lane holds rows nw0 + rt*16 + 4j + v, token m0 + tt*16 + r.
  // The residual and SwiGLU outputs go through LDS (the activation buffers,
  // free after the loop's last barrier) so that every token row is read and
  // written in 16-byte pieces rather than 2 bytes per lane.
  if constexpr (MODE == GM_RESID) {
    // fp32 sums, 64 tokens per pass: x = half(x + y), residual stays fp16 (kernels.cu:621)
    constexpr int LDF = BN + 4;   // padded fp32 row
    constexpr int HT = kPfTok / 2;
    static_assert(HT * LDF * 2 <= SM, "residual staging fits");
    float* ft = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h) __syncthreads();
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int tt = h * TT / 2; tt < (h + 1) * TT / 2; ++tt)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            ft[(tt * 16 + r - h * HT) * LDF + wave * WROWS + rt * 16 + 4 * j + v] = acc[0][rt][tt][v];
      __syncthreads();
      for (int idx = threadIdx.x; idx < HT * (BN / 4); idx += kPfThreads) {
        const int ml = idx / (BN / 4), c = idx % (BN / 4);
        const int m = m0 + h * HT + ml, n = nb0 + 4 * c;
        if (m >= a.M || n >= a.N) continue;
        _Float16* p = a.out + (int64_t)m * a.N + n;
        h4_t x = *reinterpret_cast<const h4_t*>(p);
        const f4_t y = *reinterpret_cast<const f4_t*>(&ft[ml * LDF + 4 * c]);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (_Float16)((float)x[e] + y[e]);
        *reinterpret_cast<h4_t*>(p) = x;
      }
    }
  } else if constexpr (MODE == GM_SWIGLU) {
    constexpr int LD = BN + 8;   // padded fp16 row
    static_assert(kPfTok * LD <= SM, "swiglu staging fits");
    _Float16* ot = smem;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int nl = wave * WROWS + rt * 16 + 4 * j + v, ml = tt * 16 + r;
          const int m = min(m0 + ml, a.M - 1);
          const float s = a.inv[m];
          const float g = acc[0][rt][tt][v] * s, u = acc[1][rt][tt][v] * s;
          const float sig = 1.f / (1.f + expf(-g));   // kernels.cu:566
          // nb0 is a multiple of 8, so the layout's permutation stays inside the tile
          ot[ml * LD + pf_pos(nl, Q == CQ_QUANT_INT4)] = pf_val((float)(_Float16)((g * sig) * u), nl, Q == CQ_QUANT_INT4);
        }
    __syncthreads();
    for (int idx = threadIdx.x; idx < kPfTok * (BN / 8); idx += kPfThreads) {
      const int ml = idx / (BN / 8), c = idx % (BN / 8);
      const int m = m0 + ml, n = nb0 + 8 * c;
      if (m < a.M && n < a.N)
        *reinterpret_cast<u4_t*>(a.out + (int64_t)m * a.N + n) = *reinterpret_cast<const u4_t*>(&ot[ml * LD + 8 * c]);
    }
  } else {
    // QKV: norm scale, bias, fp16 into LDS (over the activation buffers, all
    // reads of which finished at the loop's last barrier), 64 tokens per
    // pass, token-major rows; then pairs (i, i + hd/2) of each head rotate
    // (q, k) and go to Q or the KV cache, four pairs per thread, consecutive
    // threads taking consecutive pairs of one token (so Q's stores are contiguous)
    constexpr int HT = kPfTok / 2;
    constexpr int LDQ = BN + 4;   // 8-byte rows for the four-pair reads
    static_assert(HT * LDQ <= SM, "QKV staging fits");
    _Float16* ot = smem;
    const int hd = a.head_dim, half = hd / 2;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h) __syncthreads();
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int tt = h * TT / 2; tt < (h + 1) * TT / 2; ++tt)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int nl = wave * WROWS + rt * 16 + 4 * j + v, ml = tt * 16 + r;
            const int n = nb0 + nl, m = min(m0 + ml, a.M - 1);
            int local;
            const int mat = pf_mat(a, min(n, a.N - 1), &local);
            const _Float16* b = a.bias[mat];
            const float y = acc[0][rt][tt][v] * a.inv[m] + (b ? (float)b[local] : 0.f);
            ot[(ml - h * HT) * LDQ + nl] = (_Float16)y;   // q/k/v are fp16 before RoPE (kernels.cu:470)
          }
      __syncthreads();
      for (int idx = threadIdx.x; idx < (BN / 8) * HT; idx += kPfThreads) {
        const int pi = 4 * (idx % (BN / 8)), ml = idx / (BN / 8);   // pairs pi .. pi + 3 of the block's BN/2
        const int nl0 = (pi / half) * hd + pi % half, nl1 = nl0 + half;
        const int n0 = nb0 + nl0, m = m0 + h * HT + ml;
        if (n0 >= a.N || m >= a.M) continue;
        int local;
        const int mat = pf_mat(a, n0, &local);
        if (mat == 2) continue;   // not rotated: stored as they stand below
        h4_t h0 = *reinterpret_cast<const h4_t*>(&ot[ml * LDQ + nl0]), h1 = *reinterpret_cast<const h4_t*>(&ot[ml * LDQ + nl1]);
        float y0[4], y1[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y0[e] = (float)h0[e];
          y1[e] = (float)h1[e];
        }
        pf_rope4(a, m, local % hd, y0, y1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          h0[e] = (_Float16)y0[e];
          h1[e] = (_Float16)y1[e];
        }
        if (a.kcache8 && mat > 0) {
          // quantized cache: rotated values back into the tile, quantized per head below
          *reinterpret_cast<h4_t*>(&ot[ml * LDQ + nl0]) = h0;
          *reinterpret_cast<h4_t*>(&ot[ml * LDQ + nl1]) = h1;
        } else {
          pf_qkv_store4(a, mat, local, m, h0, h1);
        }
      }
      if (!a.kcache8) {
        // V: the tiled cache keeps the four positions of an aligned group of
        // four side by side, so a thread takes one dim of such a group (8
        // bytes; one position at a time, 2 bytes to a line each, the two
        // blocks of V rows took 20 us longer than the rest of the launch)
        const int v0 = max(a.rows[0] + a.rows[1] - nb0, 0), nv = min(BN, a.N - nb0) - v0;
        const int p0 = a.pos0 + m0 + h * HT, cnt = min(HT, a.M - m0 - h * HT);
        const int g0 = p0 >> 2, ng = nv > 0 && cnt > 0 ? ((p0 + cnt - 1) >> 2) - g0 + 1 : 0;
        for (int idx = threadIdx.x; idx < ng * nv; idx += kPfThreads) {
          const int nl = v0 + idx % nv, pos = 4 * (g0 + idx / nv), ml = pos - p0;
          const int local = nb0 + nl - a.rows[0] - a.rows[1];
          _Float16* dst = a.vcache + kv_v_offset(local / hd, pos, local % hd, a.max_seq, hd);
          h4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = ot[min(max(ml + e, 0), HT - 1) * LDQ + nl];
          if (ml >= 0 && ml + 3 < cnt) {
            *reinterpret_cast<h4_t*>(dst) = v;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (ml + e >= 0 && ml + e < cnt) dst[e] = v[e];
          }
        }
      } else {
        __syncthreads();
        const int heads = BN / hd;
        for (int idx = threadIdx.x; idx < heads * HT; idx += kPfThreads) {
          const int hb = idx / HT, ml = idx % HT;
          const int n0 = nb0 + hb * hd, m = m0 + h * HT + ml;
          if (n0 >= a.N || m >= a.M) continue;
          int local;
          const int mat = pf_mat(a, n0, &local);
          if (mat == 0) continue;
          float amax = 0.f;
          for (int d = 0; d < hd; ++d) amax = fmaxf(amax, fabsf((float)ot[ml * LDQ + hb * hd + d]));
          pf_kv8_store(a, mat, local / hd, a.pos0 + m, amax, [&](int d) { return (float)ot[ml * LDQ + hb * hd + d]; });
        }
      }
    }
  }
}

// --------------------------------------------------- few tokens: weight stream
// The GEMM of a short prompt (or of a small matrix).  A block is TT slices of
// 16 tokens by 128 weight rows: 4 row groups of 32 rows times 2 K groups (each
// takes one half of the block's K steps [kb, ke)), whose sums meet in LDS.  A
// ninth wave streams the activations straight into LDS, NST - 1 stages ahead:
// loads complete in issue order per wave, so a wave that requested both would
// wait for weights of later steps whenever it needs activations.
// What bounds it: each wave's step (unpack, LDS reads, matrix instructions,
// a barrier) and the weight bytes about equally, not overlapped as they should
// be: D steps of weights are requested ahead, but the step's branches make the
// compiler wait for all of them at the first of every four steps.  7B int4
// gate/up at 27 tokens 34.6 us = 2.0 TB/s; with the weight loads alone 20, with
// everything but them 21-25.  The 128-token tile it replaces there does the work of 128
// tokens: 69 us as it was split, 54 unsplit; down 43 -> 22, QKV 18 -> 13, O
// 16 -> 11 (with their epilogues).  0.5B int4 at 27 tokens: gate/up 37 -> 7.
// Measured on the way: four scales per load instead of one 28 -> 22 us (8
// tokens), K halves in one block instead of a second partial 43 -> 35.
// FORM PS_ROWS / PS_PANELS: rows of the concatenated matrices (q | k | v, gate
// | up), row-major or in 128-column panels; the fp32 sums are a partial that
// the split epilogue finishes.  PS_SWIGLU: 16 gate and the same 16 up rows per
// wave over the whole K, finished here.
enum { PS_ROWS, PS_PANELS, PS_SWIGLU };
constexpr int kPsRG = 4, kPsKG = 2;
constexpr int kPsWaves = kPsRG * kPsKG, kPsThreads = (kPsWaves + 1) * kWave;
constexpr int kPsRows = kPsRG * 32;
constexpr int kPsUnroll = 4;   // steps per loop iteration: scales are fetched four groups at a time
template <int Q, int TT> struct PsShape {
  static constexpr int D = Q == CQ_QUANT_INT4 ? 4 : 2;   // weight steps requested ahead
  static constexpr int NST = TT == 4 ? 3 : 4;            // stages
  static constexpr int XT = 16 * TT * kPfK;              // halves of one step's activations
  static constexpr int XS = kPsKG * XT;                  // a stage: one step of each K group
  static constexpr int OCC = TT == 4 ? 3 : 5;            // waves per SIMD (5: two blocks on a CU)
};
struct __attribute__((packed, aligned(2))) PsScales { uint64_t v; };   // four consecutive fp16 scales of a row

template <int Q, int FORM, int TT>
__global__ __launch_bounds__(kPsThreads, (PsShape<Q, TT>::OCC)) void pf_stream_kernel(const PfGemmArgs a) {
  using SH = PsShape<Q, TT>;
  constexpr int RT = 2, L = PfW<Q>::LOADS, D = SH::D, NST = SH::NST, XT = SH::XT, XS = SH::XS, U = kPsUnroll;
  static_assert(U % D == 0, "register sets keep fixed indices");
  __shared__ __align__(16) _Float16 xs[NST * XS];
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane & 15, j = lane >> 4;
  int rb, tb;
  pf_block_tile((a.M + 16 * TT - 1) / (16 * TT), &rb, &tb);
  const int m0 = tb * 16 * TT;
  const int K = a.K, nks = K / kPfK;
  const int kb = (int)((int64_t)blockIdx.z * nks / gridDim.z), ke = (int)((int64_t)(blockIdx.z + 1) * nks / gridDim.z);
  const int n_st = (ke - kb + 1) / 2;   // K group 0 takes [kb, kb + n_st), K group 1 the rest

  if (wave == kPsWaves) {
    // 1 KB pieces of 4 token rows of one step, swizzled like the large tile's
    // (pf_slot); steps past the range repeat the last
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)xs;
    const char* row[4 * TT];
#pragma unroll
    for (int q = 0; q < 4 * TT; ++q) {
      const int t = 4 * q + (lane >> 4);
      row[q] = reinterpret_cast<const char*>(a.A + (int64_t)min(m0 + t, a.M - 1) * K + pf_slot(t, lane & 15) * 8);
    }
    auto request = [&](int st) {
#pragma unroll
      for (int kg = 0; kg < kPsKG; ++kg)
#pragma unroll
        for (int q = 0; q < 4 * TT; ++q)
          lds_load_1k(lds0 + ((st % NST) * XS + kg * XT + q * 512) * 2, row[q] + min(kb + kg * n_st + st, ke - 1) * (kPfK * 2));
    };
#pragma unroll
    for (int st = 0; st < NST - 1; ++st) request(st);
    for (int st = 0; st < n_st; ++st) {
      wait_vm<(NST - 2) * kPsKG * 4 * TT>();   // stage st is there
      lds_barrier();
      request(st + NST - 1);   // into the slot of stage st - 1, read before this barrier
    }
    wait_vm<0>();   // nothing may land once the stages are reused
    __syncthreads();
    __syncthreads();
    if constexpr (FORM == PS_SWIGLU) __syncthreads();
    return;
  }

  const int rg = wave % kPsRG, kg = wave / kPsRG;
  const int k0 = kb + kg * n_st, n_k = min(n_st, ke - k0);   // the wave's steps
  const int nt = FORM == PS_SWIGLU ? a.N : a.rows[0] + a.rows[1] + a.rows[2];
  const int nw0 = FORM == PS_SWIGLU ? rb * (kPsRows / 2) + rg * 16 : rb * kPsRows + rg * 32;   // first row of the wave
  const char* rowp[RT];
  const _Float16* srow[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int local, mat;
    if constexpr (FORM == PS_SWIGLU) {
      mat = rt;
      local = min(nw0 + r, nt - 1);
    } else {
      mat = pf_mat(a, min(nw0 + rt * 16 + r, nt - 1), &local);
    }
    const int64_t rbytes = FORM == PS_PANELS ? 64 * L : Q == CQ_QUANT_INT4 ? K / 2 : Q == CQ_QUANT_INT8 ? K : 2 * K;
    rowp[rt] = reinterpret_cast<const char*>(sel3(a.W, mat)) + (int64_t)local * rbytes;
    srow[rt] = Q == CQ_QUANT_FP16 ? nullptr : sel3(a.S, mat) + (FORM == PS_PANELS ? (int64_t)local : (int64_t)local * nks);
  }
  u4_t wv[D][RT][L];
  auto w_load = [&](int i, int set) {   // the wave's step i (past the range: the block's last)
    const int k = max(min(k0 + i, ke - 1), 0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const char* p = rowp[rt] + (int64_t)k * (FORM == PS_PANELS ? (int64_t)a.N * (64 * L) : 64 * L) + j * (L * 16);
#pragma unroll
      for (int l = 0; l < L; ++l) wv[set][rt][l] = load_u4(p + l * 16);
    }
  };
  // scales of steps i .. i + 3, 16 bits each; a row-major row holds at least
  // four (host), its last four are fetched where fewer follow
  uint64_t sv[2][RT];
  auto s_load = [&](int i, int set) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if constexpr (FORM == PS_PANELS) {
        uint64_t v = 0;
#pragma unroll
        for (int e = 0; e < U; ++e)
          v |= (uint64_t)__builtin_bit_cast(uint16_t, srow[rt][(int64_t)min(k0 + i + e, ke - 1) * a.N]) << (16 * e);
        sv[set][rt] = v;
      } else {
        const int k = k0 + i, k4 = max(min(k, nks - 4), 0);
        sv[set][rt] = reinterpret_cast<const PsScales*>(srow[rt] + k4)->v >> (16 * min(k - k4, 3));
      }
    }
  };
  f4_t acc[RT][TT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[rt][tt] = f4_t{0.f, 0.f, 0.f, 0.f};
  const UnpackRegs uk = unpack_regs();
  if constexpr (Q != CQ_QUANT_FP16) s_load(0, 0);
#pragma unroll
  for (int d = 0; d < D; ++d) w_load(d, d);
  for (int i0 = 0; i0 < n_st; i0 += U) {
    if constexpr (Q != CQ_QUANT_FP16) s_load(i0 + U, 1);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u;
      if (u && i >= n_st) break;
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the stage before this one has been read
      lds_barrier();
      if (i < n_k) {
        const _Float16* xb0 = xs + (i % NST) * XS + kg * XT;
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          h8_t xb[TT];
#pragma unroll
          for (int tt = 0; tt < TT; ++tt)
            xb[tt] = *reinterpret_cast<const h8_t*>(&xb0[(tt * 16 + r) * kPfK + pf_slot(r, 4 * j + s4) * 8]);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            h8_t w = pf_unpack<Q>(wv[u % D][rt], s4, uk.m_lo, uk.m_hi, uk.magic);
            if constexpr (Q != CQ_QUANT_FP16) {
              const _Float16 sc = __builtin_bit_cast(_Float16, (uint16_t)(sv[0][rt] >> (16 * u)));
              const h2_t s2 = {sc, sc};
              u4_t uu = __builtin_bit_cast(u4_t, w);
              uu.x = as_u32(as_h2(uu.x) * s2);
              uu.y = as_u32(as_h2(uu.y) * s2);
              uu.z = as_u32(as_h2(uu.z) * s2);
              uu.w = as_u32(as_h2(uu.w) * s2);
              w = __builtin_bit_cast(h8_t, uu);
            }
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
              acc[rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, xb[tt], acc[rt][tt], 0, 0, 0);
          }
        }
      }
      w_load(i + D, u % D);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) sv[0][rt] = sv[1][rt];
  }
  // K group 1's sums into group 0's, over the stages
  __syncthreads();
  f4_t* red = reinterpret_cast<f4_t*>(xs) + rg * kWave * RT * TT + lane;
  static_assert(kPsRG * kWave * 2 * TT * 16 <= NST * XS * 2, "sums fit");
  if (kg == 1) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) red[(rt * TT + tt) * kWave] = acc[rt][tt];
  }
  __syncthreads();
  if (kg == 0) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) acc[rt][tt] += red[(rt * TT + tt) * kWave];
  }
  if constexpr (FORM == PS_SWIGLU) {
    // [token][64 rows] through LDS behind the sums, out in 8-element groups
    constexpr int OS = kPsRows / 2 + 8;
    static_assert(kPsRG * kWave * 2 * TT * 16 + 16 * TT * OS * 2 <= NST * XS * 2, "output tile fits");
    _Float16* ot = xs + kPsRG * kWave * RT * TT * 8;
    if (kg == 0) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const float s = a.inv[min(m0 + tt * 16 + r, a.M - 1)];
        h4_t o;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float g = acc[0][tt][v] * s, u = acc[1][tt][v] * s;
          o[v] = (_Float16)((g * (1.f / (1.f + expf(-g)))) * u);
        }
        *reinterpret_cast<h4_t*>(ot + (tt * 16 + r) * OS + rg * 16 + 4 * j) = o;
      }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < 16 * TT * (kPsRows / 16); idx += kPsWaves * kWave) {
      const int ml = idx / (kPsRows / 16), c = idx % (kPsRows / 16);
      const int m = m0 + ml, n = rb * (kPsRows / 2) + 8 * c;
      if (m < a.M && n < a.N)
        *reinterpret_cast<h8_t*>(a.out + (int64_t)m * a.N + n) =
            pf_group(*reinterpret_cast<const h8_t*>(ot + ml * OS + 8 * c), Q == CQ_QUANT_INT4);
    }
  } else if (kg == 0) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int n = nw0 + rt * 16 + 4 * j;   // four rows of one matrix (their counts are multiples of 16)
      if (n >= nt) continue;
      int local;
      const int mat = pf_mat(a, n, &local);
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const int m = m0 + tt * 16 + r;
        if (m >= a.M) continue;
        float* p = a.mode == GM_SWIGLU ? a.part + (((int64_t)blockIdx.z * 2 + mat) * a.M + m) * a.N + local
                                       : a.part + ((int64_t)blockIdx.z * a.M + m) * a.N + n;
        *reinterpret_cast<f4_t*>(p) = acc[rt][tt];
      }
    }
  }
}

// half(a * b) with the product rounded once (v_fma_mixlo_f16), whatever the
// code around it: two conversions that the compiler packs into one
// instruction round the product to 32 bits first, and a prompt's E4M3 codes
// hang on that last bit.
__device__ __forceinline__ _Float16 mul_to_half(float a, float b) {
  _Float16 r = (_Float16)(a * b);
  asm("" : "+v"(r));
  return r;
}

// Split-K epilogue of the SwiGLU GEMM: sums the S partials of each output
// and applies the fused epilogue's arithmetic, one 8-element group (the
// layout's unit) per thread.
__global__ __launch_bounds__(256) void pf_split_swiglu(const PfGemmArgs a, int S) {
  const int64_t MN = (int64_t)a.M * a.N;
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;   // N is a multiple of 8
  if (i >= MN) return;
  const float inv = a.inv[i / a.N];
  float v[2][8] = {};
#pragma unroll 4
  for (int z = 0; z < S; ++z)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const f4_t* p = reinterpret_cast<const f4_t*>(a.part + ((int64_t)z * 2 + mt) * MN + i);
      const f4_t p0 = p[0], p1 = p[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[mt][e] += p0[e];
        v[mt][4 + e] += p1[e];
      }
    }
  h8_t o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float g = v[0][e] * inv, u = v[1][e] * inv;
    const float sig = 1.f / (1.f + expf(-g));
    o[e] = mul_to_half(g * sig, u);
  }
  *reinterpret_cast<h8_t*>(a.out + i) = pf_group(o, a.quant == CQ_QUANT_INT4);
}

// Split-K epilogue of a residual GEMM, one block per token row (N a
// multiple of 8): x = half(x + sum of the S partials), then, when asked, the
// RMSNorm of the new row (the next GEMM's input) in the same pass.
constexpr int kPfResidThreads = 512;   // one 8-element group per thread up to 4096-wide rows
__global__ __launch_bounds__(kPfResidThreads) void pf_split_resid(const PfGemmArgs a, int S) {
  __shared__ float red[16];
  const int m = blockIdx.x;
  const int64_t MN = (int64_t)a.M * a.N;
  _Float16* xr = a.out + (int64_t)m * a.N;
  for (int g = threadIdx.x; g < a.N / 8; g += blockDim.x) {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < S; ++z) {
      const f4_t* pz = reinterpret_cast<const f4_t*>(a.part + z * MN + (int64_t)m * a.N + 8 * g);
      const f4_t p0 = pz[0], p1 = pz[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += p0[e];
        v[4 + e] += p1[e];
      }
    }
    h8_t x = __builtin_bit_cast(h8_t, load_u4(xr + 8 * g));
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (_Float16)((float)x[e] + v[e]);   // residual stays fp16 (kernels.cu:621)
    *reinterpret_cast<u4_t*>(xr + 8 * g) = __builtin_bit_cast(u4_t, x);
  }
  // the norm reads back the groups this thread has just written
  if (a.norm_w)
    pf_norm_row(xr, a.norm_w, a.norm_eps, a.N, a.norm_out + (int64_t)m * a.N, a.norm_inv + m,
                a.quant == CQ_QUANT_INT4, red);
}

// Split-K epilogue of the QKV GEMM, blockIdx.x = token: sums the partials,
// applies the norm scale and bias (q / k / v are fp16 before RoPE,
// kernels.cu:470), rotates q and k with the token's sines and cosines and
// stores q, and k / v into the cache; block y
// takes pairs [1024 y, 1024 y + 1024), four per thread.  A quantized cache takes each (k or v,
// kv head) row through one wave of the blocks past the pairs.
constexpr int kPfQkvThreads = 256;
template <int HD>
__global__ __launch_bounds__(kPfQkvThreads) void pf_split_qkv(const PfGemmArgs a, int S) {
  constexpr int HALF = HD / 2;
  const int m = blockIdx.x, pos = a.pos0 + m;
  const int64_t MN = (int64_t)a.M * a.N;
  const float inv = a.inv[m];
  const float* prow = a.part + (int64_t)m * a.N;
  // fp16 value of row n (bias added, before RoPE)
  auto raw = [&](int n) {
    float v = 0.f;
#pragma unroll 4
    for (int z = 0; z < S; ++z) v += prow[z * MN + n];
    int local;
    const int mat = pf_mat(a, n, &local);
    const _Float16* b = a.bias[mat];
    return (float)(_Float16)(v * inv + (b ? (float)b[local] : 0.f));
  };
  const int np_store = (a.kcache8 ? a.rows[0] : a.N) / 2;   // quantized cache: k / v rows go per head below
  const int pair_blocks = (np_store / 4 + kPfQkvThreads - 1) / kPfQkvThreads;
  if ((int)blockIdx.y < pair_blocks) {
    // four consecutive pairs (i .. i+3, i + HALF .. i + HALF + 3) per thread
    const int p = 4 * (blockIdx.y * kPfQkvThreads + threadIdx.x);
    if (p >= np_store) return;
    const int i = p % HALF, n0 = (p / HALF) * HD + i;
    int local;
    const int mat = pf_mat(a, n0, &local);
    f4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < S; ++z) {
      s0 += *reinterpret_cast<const f4_t*>(prow + z * MN + n0);
      s1 += *reinterpret_cast<const f4_t*>(prow + z * MN + n0 + HALF);
    }
    const _Float16* b = a.bias[mat];
    float y0[4], y1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y0[e] = (float)(_Float16)(s0[e] * inv + (b ? (float)b[local + e] : 0.f));
      y1[e] = (float)(_Float16)(s1[e] * inv + (b ? (float)b[local + HALF + e] : 0.f));
    }
    if (mat < 2) pf_rope4(a, m, i, y0, y1);
    h4_t h0, h1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h0[e] = (_Float16)y0[e];
      h1[e] = (_Float16)y1[e];
    }
    pf_qkv_store4(a, mat, local, m, h0, h1);
  } else {
    constexpr int E = HD / kWave;   // consecutive elements per lane
    const int lane = threadIdx.x & (kWave - 1), n_kv = a.rows[1] / HD;
    const int r = (blockIdx.y - pair_blocks) * (kPfQkvThreads / kWave) + threadIdx.x / kWave;
    if (r < 2 * n_kv) {
      const int mat = 1 + r / n_kv, kvh = r % n_kv;
      const int nb = a.rows[0] + (mat == 2 ? a.rows[1] : 0) + kvh * HD;
      float x[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int d = lane * E + e, i = d % HALF;
        float y0 = raw(nb + i), y1 = raw(nb + i + HALF);
        if (mat == 1) {
          const float* p = a.rope + (int64_t)m * HALF + i;
          rope_apply(y0, y1, p[0], p[(int64_t)a.M * HALF]);
        }
        x[e] = (float)(_Float16)(d < HALF ? y0 : y1);
      }
      int8_t q[E];
      const float sc = a.kv_fmt == CQ_KV_FP8 ? quant_row8_wave<HD, CQ_KV_FP8>(x, q) : quant_row8_wave<HD, CQ_KV_INT8>(x, q);
      int8_t* c = mat == 1 ? a.kcache8 : a.vcache8;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int d = lane * E + e;
        c[mat == 1 ? kv8_k_offset(kvh, pos, d, a.max_seq, HD) : kv8_v_offset(kvh, pos, d, a.max_seq, HD)] = q[e];
      }
      if (lane == 0) (mat == 1 ? a.kscale : a.vscale)[(int64_t)kvh * a.max_seq + pos] = sc;
    }
  }
}

// The last token's rows for the decode kernels that finish it: its attention
// output back to natural order (the int4 layout stores each 8-group as
// [0,4,1,5,2,6,3,7] with the odd elements / 16; the scale is a power of two,
// so the round trip is exact for odd elements of magnitude at least 2^-10 --
// smaller ones lost low bits to the subnormal range on the way in), and its
// residual.
__global__ __launch_bounds__(256) void pf_last_row(const _Float16* src, _Float16* dst, int n, bool int4,
                                                   const _Float16* x, _Float16* x_out, int dim) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] = (_Float16)((float)src[pf_pos(k, int4)] * ((int4 && (k & 1)) ? 16.0f : 1.0f));
  if (k < dim) x_out[k] = x[k];
}

// ------------------------------------------------------------------ host
int launch_pf_last_row(const __half* src, __half* dst, int n, int quant, const __half* x, __half* x_out, int dim,
                       hipStream_t stream) {
  hipLaunchKernelGGL(pf_last_row, dim3((std::max(n, dim) + 255) / 256), dim3(256), 0, stream, (const _Float16*)src,
                     (_Float16*)dst, n, quant == CQ_QUANT_INT4, (const _Float16*)x, (_Float16*)x_out, dim);
  CQ_HIP(hipGetLastError());
  return CQ_OK;
}

int launch_pf_embed(const __half* embed, const int* tokens, int M, int dim, __half* x, const double* inv_freq,
                    int head_dim, int pos0, float* rope, const __half* norm_w, float eps, __half* norm_out,
                    float* norm_inv, int quant, hipStream_t stream) {
  if (M <= 0 || dim <= 0 || dim % 8) return fail(CQ_EINVAL, "prefill norm: rows must be a multiple of 8 wide");
  PfEmbedArgs a{reinterpret_cast<const u4_t*>(embed), tokens, (_Float16*)x, dim, inv_freq, head_dim / 2, pos0, rope,
                (const _Float16*)norm_w, eps, (_Float16*)norm_out, norm_inv, quant == CQ_QUANT_INT4};
  hipLaunchKernelGGL(pf_embed, dim3(M), dim3(256), 0, stream, a);
  CQ_HIP(hipGetLastError());
  return CQ_OK;
}

// Sums S fp32 partials and finishes the GEMM.
template <int MODE>
static int launch_pf_split(const PfGemmArgs& a, int S, hipStream_t stream) {
  if constexpr (MODE == GM_QKV) {
    const int np_store = (a.kcache8 ? a.rows[0] : a.N) / 2, waves = kPfQkvThreads / kWave;
    const int ny = (np_store / 4 + kPfQkvThreads - 1) / kPfQkvThreads +
                   (a.kcache8 ? (2 * (a.rows[1] / a.head_dim) + waves - 1) / waves : 0);
    if (a.head_dim == 128) hipLaunchKernelGGL((pf_split_qkv<128>), dim3(a.M, ny), dim3(kPfQkvThreads), 0, stream, a, S);
    else hipLaunchKernelGGL((pf_split_qkv<64>), dim3(a.M, ny), dim3(kPfQkvThreads), 0, stream, a, S);
  } else if constexpr (MODE == GM_RESID) {
    hipLaunchKernelGGL(pf_split_resid, dim3(a.M), dim3(kPfResidThreads), 0, stream, a, S);
  } else {
    const int64_t groups = (int64_t)a.M * a.N / 8;
    hipLaunchKernelGGL(pf_split_swiglu, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, stream, a, S);
  }
  CQ_HIP(hipGetLastError());
  return CQ_OK;
}

// The weight stream with TT token slices, K split S ways (0: PS_SWIGLU).
template <int Q, int MODE, int TT>
static int launch_pf_stream(const PfGemmArgs& a, int S, hipStream_t stream) {
  const int n_tb = (a.M + 16 * TT - 1) / (16 * TT);
  if (MODE == GM_SWIGLU && S == 0) {
    const int gx = ((a.N + kPsRows / 2 - 1) / (kPsRows / 2)) * n_tb;
    hipLaunchKernelGGL((pf_stream_kernel<Q, PS_SWIGLU, TT>), dim3(gx), dim3(kPsThreads), 0, stream, a);
    CQ_HIP(hipGetLastError());
    return CQ_OK;
  }
  const int gx = ((a.rows[0] + a.rows[1] + a.rows[2] + kPsRows - 1) / kPsRows) * n_tb;
  if (MODE == GM_RESID && a.panels)
    hipLaunchKernelGGL((pf_stream_kernel<Q, PS_PANELS, TT>), dim3(gx, 1, S), dim3(kPsThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((pf_stream_kernel<Q, PS_ROWS, TT>), dim3(gx, 1, S), dim3(kPsThreads), 0, stream, a);
  CQ_HIP(hipGetLastError());
  return launch_pf_split<MODE>(a, S, stream);
}

// The 128-token tile, split S ways over K (1: its fused epilogue).
template <int Q, int MODE>
static int launch_pf_tile(const PfGemmArgs& a, int S, hipStream_t stream) {
  const int bn = PfShape<Q, MODE>::BN;
  const int gx = ((a.N + bn - 1) / bn) * ((a.M + kPfTok - 1) / kPfTok);   // row blocks x token blocks
  if (S > 1) {
    hipLaunchKernelGGL((pf_gemm_kernel<Q, MODE, true>), dim3(gx, 1, S), dim3(kPfThreads), 0, stream, a);
    CQ_HIP(hipGetLastError());
    return launch_pf_split<MODE>(a, S, stream);
  }
  hipLaunchKernelGGL((pf_gemm_kernel<Q, MODE, false>), dim3(gx), dim3(kPfThreads), 0, stream, a);
  CQ_HIP(hipGetLastError());
  if (MODE == GM_RESID && a.norm_w) {
    hipLaunchKernelGGL(pf_norm_rows, dim3(a.M), dim3(256), 0, stream, (const _Float16*)a.out, a.norm_w, a.norm_eps,
                       a.N, a.norm_out, a.norm_inv, Q == CQ_QUANT_INT4);
    CQ_HIP(hipGetLastError());
  }
  return CQ_OK;
}

// How a GEMM runs: the weight stream with tt token slices (split ways over K,
// 0: PS_SWIGLU), or, tt = 0, the 128-token tile (split ways, 1: unsplit).
struct PfPlan { int tt, split; };

// The tile's split for more than 512 tokens.  Model: one block fits a CU (its
// LDS), so B blocks take ceil(B / CUs) rounds and S splits ceil(S B / CUs)
// rounds of 1/S the work; a full-K block runs at ~4.2 TFLOP/s per CU
// (measured: int4 gate/up, 56 us per round of 256 blocks at K = 3584); the
// split epilogue reads the S fp32 partials at ~2.8 TB/s after a launch of ~2
// us (measured: QKV's 3 x 18.9 MB in 20.4 us, the residual's 2 x 14.7 MB in
// 10.7 us).  Within the workspace.
template <int Q, int MODE>
static int pf_tile_split(const PfGemmArgs& a) {
  const int bn = PfShape<Q, MODE>::BN;
  const int gx = ((a.N + bn - 1) / bn) * ((a.M + kPfTok - 1) / kPfTok);   // row blocks x token blocks
  const int nks = a.K / kPfK, nmat = MODE == GM_SWIGLU ? 2 : 1;
  int S = 1;
  if (a.part) {
    auto rounds = [&](int s) { return (double)(((int64_t)gx * s + kNumCUs - 1) / kNumCUs); };
    const double t1 = (double)bn * nmat * kPfTok * a.K * 2 / 4.2e6;     // us, one round of full-K blocks
    const double part_us = (double)nmat * a.M * a.N * sizeof(float) / 2.8e6;   // us per split of partials
    // QKV's unsplit epilogue (RoPE through an LDS tile, cache stores) costs
    // about what a split epilogue's pass does (measured: 7B at 1024 tokens 75
    // us unsplit, 72 split 3 ways; at 1536 72 and 100, at 2048 136 and 125
    // split 2 ways)
    double best = rounds(1) * t1 + (MODE == GM_QKV ? part_us + 2.0 : 0.0);
    for (int s = 2; s <= std::min(kPfMaxSplit, nks); ++s) {
      if ((size_t)s * nmat * a.M * a.N * sizeof(float) > (a.keep_tile ? std::min(a.part_bytes, kPfKeptPart) : a.part_bytes)) break;
      const double t = rounds(s) / s * t1 + s * part_us + 2.0;
      if (t < best) { best = t; S = s; }
    }
  }
  return S;
}

// Microseconds of either form, fitted to 54,000 measured points: the five
// presets' four GEMMs, three precisions, 36 token counts from 2 to 1024, every
// token tile and split, 2 us added for a launch of the epilogue's own; rms error
// 6 %.  What is picked by it costs 0.7 % over the best measured form on average;
// nine of 2104 shapes are over 2 % behind the tile by the split rule above alone
// (one by 7.5 %, the rest under 4.2), no layer's four GEMMs together over 0.8.
// Tile: rounds of one block per CU, each with its K steps, and the split
// epilogue with the partials written and read, or the fused one.
// Stream: the K steps of a wave on the fullest CU, the blocks after the first
// there, and the fused SwiGLU of each or the split epilogue.
// Both: the weights' bytes once.  (Without that term, and with no cost of its
// own for the fused SwiGLU, the stream was up to 25 % too cheap and was picked
// for gate/up where the tile is faster: 14B int8 at 288 tokens 192 against 161
// us, 7B int8 at 256 141 against 122.)
template <int Q> constexpr double pf_by(double int4, double int8, double fp16) {
  return Q == CQ_QUANT_INT4 ? int4 : Q == CQ_QUANT_INT8 ? int8 : fp16;
}
template <int Q, int MODE>
static double pf_tile_us(const PfGemmArgs& a, int S) {
  constexpr double kRound = pf_by<Q>(0.1, 0.46, 0.48), kStep = pf_by<Q>(1.6, 1.84, 2.57);
  constexpr double kSplit = pf_by<Q>(11.4, 11.4, 12.3), kPerMb = pf_by<Q>(0.39, 0.39, 0.365);
  const int bn = PfShape<Q, MODE>::BN, nmat = MODE == GM_SWIGLU ? 2 : 1, nks = a.K / kPfK;
  const int64_t blocks = (int64_t)((a.N + bn - 1) / bn) * ((a.M + kPfTok - 1) / kPfTok) * S;
  const double rounds = (double)((blocks + kNumCUs - 1) / kNumCUs), mb = (double)S * nmat * a.M * a.N * sizeof(float) / 1e6;
  const double weight_mb = (double)nmat * a.N * a.K * pf_by<Q>(0.5, 1, 2) / 1e6;
  const double fused = MODE == GM_QKV      ? pf_by<Q>(19.6, 19.7, 19.9)
                       : MODE == GM_SWIGLU ? pf_by<Q>(6.9, 5.7, 4.8) * rounds
                                           : pf_by<Q>(13.3, 12.7, 14.2);
  return pf_by<Q>(0.051, 0.055, 0.057) * weight_mb + rounds * (kRound + (nks + S - 1) / S * kStep) +
         (S > 1 ? kSplit + kPerMb * mb : fused);
}
template <int Q>
static double pf_stream_us(const PfGemmArgs& a, int tt, int S) {
  constexpr double kStep[3] = {pf_by<Q>(0.584, 1.12, 1.87), pf_by<Q>(0.784, 1.13, 2.14), pf_by<Q>(1.066, 1.37, 2.39)};
  constexpr double kBlock[3] = {pf_by<Q>(2.25, 2.2, 3.8), pf_by<Q>(2.38, 2.6, 3.7), pf_by<Q>(3.3, 3.3, 4.2)};
  constexpr double kSwiglu[3] = {pf_by<Q>(0.26, 0.11, 0.2), pf_by<Q>(0.95, 0.96, 0.85), pf_by<Q>(1.26, 1.95, 1.18)};
  const int rows = a.rows[0] + a.rows[1] + a.rows[2], s = std::max(S, 1), nks = a.K / kPfK;
  const int64_t blocks = (int64_t)((rows + kPsRows - 1) / kPsRows) * ((a.M + 16 * tt - 1) / (16 * tt)) * s;
  const double per_cu = (double)((blocks + kNumCUs - 1) / kNumCUs), steps = ((nks + s - 1) / s + 1) / 2;
  const double weight_mb = (double)rows * a.K * pf_by<Q>(0.5, 1, 2) / 1e6, mb = (double)S * a.M * rows * sizeof(float) / 1e6;
  return pf_by<Q>(3.73, 3.88, 4.47) + pf_by<Q>(0.077, 0.066, 0.061) * weight_mb + steps * kStep[tt / 2] * per_cu +
         kBlock[tt / 2] * (per_cu - 1) +
         (S ? pf_by<Q>(7.0, 7.5, 8.4) + pf_by<Q>(0.334, 0.38, 0.357) * mb : kSwiglu[tt / 2] * per_cu);
}

template <int Q, int MODE>
static PfPlan pf_plan(const PfGemmArgs& a) {
  const int nks = a.K / kPfK, nmat = MODE == GM_SWIGLU ? 2 : 1;
  if (a.want_tokens) {
    const int most = (int)std::min<size_t>(nks, a.part_bytes / ((size_t)nmat * a.M * a.N * sizeof(float)));
    if (a.want_tokens == kPfTok) return PfPlan{0, std::max(std::min({a.want_split, kPfMaxSplit, most}), 1)};
    const int s = std::min(a.want_split, most);
    return PfPlan{a.want_tokens / 16, MODE == GM_SWIGLU && s <= 1 ? 0 : s};
  }
  PfPlan best{0, pf_tile_split<Q, MODE>(a)};
  // above 1024 tokens the tile is the faster form at every preset's shapes;
  // the stream fetches four scales of a row at a time
  if (a.keep_tile || !a.part || a.M > 1024 || nks < 4) return best;
  auto fits = [&](int s) { return (size_t)s * nmat * a.M * a.N * sizeof(float) <= a.part_bytes; };
  // up to 512 tokens the fitted split is as good as the rule's or better (above,
  // not always: 3B int4 QKV at 1024 33 against 31 us)
  if (a.M <= 512) {
    for (int s = 1; s <= std::min(kPfMaxSplit, nks) && (s == 1 || fits(s)); ++s)
      if (s == 1 || pf_tile_us<Q, MODE>(a, s) < pf_tile_us<Q, MODE>(a, best.split)) best.split = s;
  }
  // above 512 tokens partials make the stream err by more: it has to win by that
  // (0.5B fp16 down at 704 32 against 29 us without)
  double t = (a.M <= 512 || MODE == GM_SWIGLU ? 1.0 : 0.95) * pf_tile_us<Q, MODE>(a, best.split);
  for (int tt = 1; tt <= 4; tt *= 2)
    for (int s = MODE == GM_SWIGLU ? 0 : 1; s <= std::min(32, nks) && fits(s); ++s)
      if (const double u = pf_stream_us<Q>(a, tt, s); u < t) {
        t = u;
        best = PfPlan{tt, s};
      }
  return best;
}

template <int Q, int MODE>
static int launch_pf_gemm_m(const PfGemmArgs& a, hipStream_t stream) {
  const PfPlan p = pf_plan<Q, MODE>(a);
  if (p.tt == 1) return launch_pf_stream<Q, MODE, 1>(a, p.split, stream);
  if (p.tt == 2) return launch_pf_stream<Q, MODE, 2>(a, p.split, stream);
  if (p.tt == 4) return launch_pf_stream<Q, MODE, 4>(a, p.split, stream);
  return launch_pf_tile<Q, MODE>(a, p.split, stream);
}

template <int Q>
static int launch_pf_gemm_q(const PfGemmArgs& a, hipStream_t stream) {
  if (a.mode == GM_QKV) return launch_pf_gemm_m<Q, GM_QKV>(a, stream);
  if (a.mode == GM_SWIGLU) return launch_pf_gemm_m<Q, GM_SWIGLU>(a, stream);
  return launch_pf_gemm_m<Q, GM_RESID>(a, stream);
}

int launch_pf_gemm(const PfGemmArgs& a, hipStream_t stream) {
  if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.K % kPfK) return fail(CQ_EINVAL, "prefill gemm: K must be a multiple of 128");
  if (!a.A || !a.W[0] || !a.out) return fail(CQ_EINVAL, "prefill gemm: null operand");
  if (a.quant != CQ_QUANT_FP16 && !a.S[0]) return fail(CQ_EINVAL, "prefill gemm: quantized weights need scales");
  if (a.mode == GM_SWIGLU && (!a.W[1] || !a.inv || a.N % 8))
    return fail(CQ_EINVAL, "prefill gemm: swiglu needs gate, up, the norm and rows a multiple of 8");
  if (a.mode == GM_RESID && (a.N % 8 || (a.norm_w && (!a.norm_out || !a.norm_inv))))
    return fail(CQ_EINVAL, "prefill gemm: residual rows must be a multiple of 8 wide; the norm needs its outputs");
  if (a.panels && a.mode != GM_RESID) return fail(CQ_EINVAL, "prefill gemm: paneled weights are a residual-mode option");
  if (a.mode == GM_QKV) {
    if (!a.inv || !a.W[1] || !a.W[2] || !a.rope) return fail(CQ_EINVAL, "prefill gemm: qkv operands");
    if (a.kcache8 ? (!a.vcache8 || !a.kscale || !a.vscale) : (!a.kcache || !a.vcache))
      return fail(CQ_EINVAL, "prefill gemm: qkv cache pointers");
    if (PfShape<CQ_QUANT_FP16, GM_QKV>::BN % a.head_dim || a.rows[0] % a.head_dim || a.rows[1] % a.head_dim || a.rows[0] + a.rows[1] + a.rows[2] != a.N)
      return fail(CQ_EINVAL, "prefill gemm: qkv rows must be whole heads");
  }
  if (a.want_tokens) {
    if (a.want_tokens != 16 && a.want_tokens != 32 && a.want_tokens != 64 && a.want_tokens != kPfTok)
      return fail(CQ_EINVAL, "prefill gemm: no form with that many tokens");
    if (a.want_tokens != kPfTok && a.K / kPfK < 4) return fail(CQ_EINVAL, "prefill gemm: the weight stream needs K of 512");
    if (a.want_split < 1 || !a.part) return fail(CQ_EINVAL, "prefill gemm: a wanted form needs a split and the workspace");
    if (a.want_tokens != kPfTok && a.mode != GM_SWIGLU && (size_t)a.M * a.N * sizeof(float) > a.part_bytes)
      return fail(CQ_ERANGE, "prefill gemm: the weight stream's partials do not fit");
  }
  switch (a.quant) {
    case CQ_QUANT_FP16: return launch_pf_gemm_q<CQ_QUANT_FP16>(a, stream);
    case CQ_QUANT_INT8: return launch_pf_gemm_q<CQ_QUANT_INT8>(a, stream);
    default: return launch_pf_gemm_q<CQ_QUANT_INT4>(a, stream);
  }
}

}  // namespace cq
