// Causal attention of the batched prefill (kernels.cu:105-288 with a
// per-token key limit), over the fp16 or the int8 tiled cache (E4M3: the
// kernel at the end).
//
// The query rows of a kv head are its group's heads of every token, token
// major: row r is head r % g of token r / g.  A block takes 32 * RG
// consecutive rows of one kv head, a wave 32 of them (two 16-column slices
// of S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_16x16x32_f16), so every
// K / V operand a wave reads from LDS feeds two matrix instructions and no
// wave idles whatever the group size.  The 8 waves are RG row groups times
// KH = 8 / RG key groups: key group k takes TPW of every KH * TPW
// consecutive 32-key tiles, and the key groups merge in LDS at the end.
// Where rows and key groups leave CUs idle the key range is also cut over S
// blocks, whose fp32 partials a second launch merges (pa_plan).
//
// What bounds it: at long contexts matrix units that wait (7B heads, 2048
// tokens after 30720, fp16 cache, KH = 2: 1.03-1.11 ms a layer, 840-910
// TFLOP/s, the units busy 40 % of the active cycles; with the exponentials, the
// LDS reads, the staging and the barriers all taken out the same loop took
// 0.90-0.95) and power (on a cache of zeros 0.87 against 1.08 ms, the clock at
// 2.08 of 2.4 GHz on random values); at short ones the chain of launch, first
// loads, a few steps and the epilogue (7 us).  Why this shape: one head per
// wave and 16 rows per wave made each K / V fragment feed one instruction and
// left LDS and the softmax arithmetic in front (1.86 ms); 32 rows per wave
// 1.31, the score and value products overlapped with the softmax of the
// neighbouring step 1.19, requests straight into LDS 1.03.  7B heads: 1024
// tokens 36 -> 26 us; 27 tokens after 1500, whose 8 blocks once walked the whole
// context, 45 -> 16 us.  The scores stay in 32 bits up to the exponent (the
// decode step rounds them to fp16).
#include "cq_attention.h"
#include "cq_prefill.h"

#include <algorithm>
#include <cmath>

namespace cq {

namespace {

constexpr int kPaWaves = 8;
constexpr int kPaThreads = kPaWaves * kWave;
constexpr int kPaCols = 2;   // 16-row slices per wave
constexpr float kLog2e = 1.4426950408889634f;

template <int HD, int KV8, int KH, int TPW>
struct PaShape {
  static constexpr int RG = kPaWaves / KH, ROWS = RG * 16 * kPaCols;
  static constexpr int TPS = KH * TPW;                  // tiles per step
  static constexpr int TILE = kTileKeys * HD;           // halves of K (or V) per tile
  static constexpr int STAGE = 2 * TPS * TILE;          // halves: K tiles, then V tiles
  // LDS slots: three (requests two steps ahead) where they fit 96 KB, that is
  // with KH = 1 and, at head size 64, 2; else two (one step ahead)
  static constexpr int NS = KV8 == 0 && 3 * STAGE * 2 <= 96 * 1024 ? 3 : 2;
  static constexpr int DT = HD / 16;
  static constexpr int STATE = kPaCols * (2 + 4 * DT);  // floats of one lane's softmax state (whole f4_t)
  static constexpr int OS = HD + 8;                     // padded output row
  static constexpr int SM = std::max({NS * STAGE, (KH - 1) * RG * kWave * STATE * 2, ROWS * OS});
};

// Largest of v over the four lanes that share a column (lane % 16).
__device__ __forceinline__ float col_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  v = fmaxf(__builtin_bit_cast(float, a[0]), __builtin_bit_cast(float, a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  return fmaxf(__builtin_bit_cast(float, b[0]), __builtin_bit_cast(float, b[1]));
}

// One v_max3_f32, and not written as asm: the operands are matrix results, and
// the compiler adds the wait states that these ask for (and that a register
// that a product has yet to write asks of its next writer) only in front of
// instructions of its own.
__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

template <int HD, int KV8, int KH, int TPW>   // KV8: 0 fp16 cache, CQ_KV_INT8 int8 codes
__global__ __launch_bounds__(kPaThreads, 2) void pf_attention_kernel(const PfAttnArgs a) {
  using SH = PaShape<HD, KV8, KH, TPW>;
  constexpr int KK = HD / 32, DT = SH::DT, CG = kPaCols, ST = 2 * TPW;   // ST 16-key slices per wave and step
  constexpr int RG = SH::RG, TPS = SH::TPS, TILE = SH::TILE;
  __shared__ __align__(16) _Float16 smem[SH::SM];
  __shared__ __align__(16) float scl[KV8 ? 2 : 1][KV8 ? 2 : 1][KV8 ? TPS * kTileKeys : 1];   // [stage][K / V][key]
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int h = lane & 15, j = lane >> 4;
  const int rg = wave % RG, kg = wave / RG;
  // the longest rows first; the kv head is the fastest index, so each XCD
  // (dispatch goes round-robin over 8) keeps to a few kv heads' keys
  const int g = a.n_heads / a.n_kv, R = a.M * g;
  const int kvh = blockIdx.x % a.n_kv, z = (blockIdx.x / a.n_kv) % a.splits;
  const int rb = a.n_rb - 1 - blockIdx.x / (a.n_kv * a.splits);
  const int r0 = rb * SH::ROWS, rw = r0 + rg * 16 * CG;   // first row of the block, of the wave
  const int t_max = a.pos0 + min(r0 + SH::ROWS - 1, R - 1) / g + 1;   // keys visible to the block
  const int n_tiles = (t_max + kTileKeys - 1) / kTileKeys;
  const int tb = (int)((int64_t)n_tiles * z / a.splits), te = (int)((int64_t)n_tiles * (z + 1) / a.splits);
  const int lim_lo = min(a.pos0 + min(rw, R - 1) / g + 1, te * kTileKeys);   // fewest keys a row of the wave sees

  // K and V of TPS consecutive tiles are one contiguous run of the cache
  // each.  Group i = (K of step i + 1, V of step i) is requested NS - 1 steps
  // ahead.  Tiles past the range repeat its last one (masked below); an empty
  // range (a row block with fewer tiles than ranges) takes no step and leaves
  // m = -inf.
  constexpr int NS = SH::NS;
  const int n_steps = (te - tb + TPS - 1) / TPS;
  const char* base_kv[2] = {KV8 ? (const char*)a.kcache8 + (int64_t)kvh * a.max_seq * HD : (const char*)(a.kcache + (int64_t)kvh * a.max_seq * HD),
                            KV8 ? (const char*)a.vcache8 + (int64_t)kvh * a.max_seq * HD : (const char*)(a.vcache + (int64_t)kvh * a.max_seq * HD)};
  const float c2 = kLog2e / sqrtf((float)HD);   // score -> log2 units
  auto tile_at = [&](int ti) { return max(min(ti, te - 1), 0); };
  // fp16 cache: straight into LDS, 1 KB per wave instruction, no registers
  constexpr int TB = TILE * 2 / 1024, PW = TPS * TB / kPaWaves;   // KB of a tile's K (or V); instructions per wave and step
  static_assert(KV8 || PW * kPaWaves == TPS * TB, "whole pieces per wave");
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t lane16 = lane * 16;
  auto dma = [&](int step, int part) {
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int p = i * kPaWaves + wave;
      const char* src = base_kv[part] + (int64_t)tile_at(tb + step * TPS + p / TB) * (TILE * 2) + p % TB * 1024;
      lds_load_1k(lds0 + ((step % NS) * SH::STAGE + part * TPS * TILE) * 2 + p * 1024, lane16, src);
    }
  };
  // keys past the end may hold anything: keep them out of P*V (each wave
  // clears them in the pieces of V that it requested, once they are there)
  auto clear_tail = [&](int step) {
    if ((tb + (step + 1) * TPS) * kTileKeys <= t_max) return;
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int p = i * kPaWaves + wave, k0 = tile_at(tb + step * TPS + p / TB) * kTileKeys + 4 * j;
      h8_t* q = reinterpret_cast<h8_t*>(smem + (step % NS) * SH::STAGE + TPS * TILE + p * 512 + lane * 8);
      h8_t v = *q;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k0 + (e < 4 ? e : 12 + e) >= t_max) v[e] = (_Float16)0.f;
      *q = v;
    }
  };
  // quantized cache: 16-byte pieces through registers, converted to fp16 on
  // the way into LDS, so the codes are expanded once per block
  constexpr int TP = TILE / 16, QL = KV8 ? (TPS * TP + kPaThreads - 1) / kPaThreads : 1;   // pieces of a tile; per thread
  constexpr bool FULL = QL * kPaThreads == TPS * TP;   // else (one piece) the last threads have none
  static_assert(!KV8 || FULL || QL == 1, "whole pieces per thread");
  const uint32_t magic = vgpr_const(0x64646464u);
  struct Pieces { u4_t w[QL]; float s; };
  const float* base_s[2] = {KV8 ? a.kscale + (int64_t)kvh * a.max_seq : nullptr, KV8 ? a.vscale + (int64_t)kvh * a.max_seq : nullptr};
  auto load = [&](Pieces& r, int step, int part) {
    const int base = tb + step * TPS;
#pragma unroll
    for (int i = 0; i < QL; ++i) {
      const int c = FULL ? i * kPaThreads + threadIdx.x : min((int)threadIdx.x, TPS * TP - 1);
      r.w[i] = load_u4(base_kv[part] + ((int64_t)tile_at(base + c / TP) * TP + c % TP) * 16);
    }
    const int c = threadIdx.x, key = tile_at(base + c / kTileKeys) * kTileKeys + c % kTileKeys;
    if (c < TPS * kTileKeys) r.s = key < t_max ? base_s[part][key] : 0.f;
  };
  auto store = [&](const Pieces& r, int step, int part) {
    const int slot = step % NS;
    _Float16* dst = smem + slot * SH::STAGE + part * TPS * TILE;
#pragma unroll
    for (int i = 0; i < QL; ++i) {
      const int c = i * kPaThreads + threadIdx.x, q = c % TP;
      if (!FULL && c >= TPS * TP) break;
      // 16 bytes: the operand pieces of two instructions
      _Float16* d = dst + (c / TP) * TILE + ((q / 64) * 128 + q % 64) * 8;
      *reinterpret_cast<h8_t*>(d) = codes_to_h8<KV8>(u2_t{r.w[i].x, r.w[i].y}, magic);
      *reinterpret_cast<h8_t*>(d + 512) = codes_to_h8<KV8>(u2_t{r.w[i].z, r.w[i].w}, magic);
    }
    const int c = threadIdx.x;
    if (c < TPS * kTileKeys) scl[slot][part][c] = part ? r.s : r.s * c2;
  };
  Pieces pk, pv8;
  auto request = [&](int g) {
    if constexpr (KV8 != 0) {
      load(pk, g + 1, 0);
      load(pv8, g, 1);
    } else {
      dma(g + 1, 0);
      dma(g, 1);
    }
  };
  // group g in LDS for every wave (its readers' slots free since the last barrier)
  auto arrive = [&](int g) {
    if constexpr (KV8 != 0) {
      store(pk, g + 1, 0);
      store(pv8, g, 1);
    } else {
      wait_vm<(NS - 2) * 2 * PW>();
      clear_tail(g);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    lds_barrier();
  };

  h8_t qb[CG][KK];
  int lim[CG];   // keys visible to the lane's rows within this block's range
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    const int r = min(rw + cg * 16 + h, R - 1), t = r / g;
    lim[cg] = min(a.pos0 + t + 1, te * kTileKeys);
    const _Float16* q = a.q + ((int64_t)t * a.n_heads + kvh * g + (r - t * g)) * HD;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qb[cg][kk] = __builtin_bit_cast(h8_t, load_u4(q + kk * 32 + j * 8));
  }
  float m[CG], l[CG];   // running maximum (fp16 cache: of the raw products; else log2 units), lane's sum
  f4_t o[DT][CG];
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    m[cg] = -INFINITY;
    l[cg] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt][cg] = f4_t{0.f, 0.f, 0.f, 0.f};
  }
  constexpr bool RAW = KV8 == 0;   // scores stay raw and the scale rides on the exponent's fma
  typedef f4_t S_t[ST][CG];
  auto qk = [&](S_t& s, int step) {   // S^T of the wave's tiles
    const _Float16* kt = smem + (step % NS) * SH::STAGE + kg * TPW * TILE;
#pragma unroll
    for (int st = 0; st < ST; ++st) {
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) s[st][cg] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const h8_t ka = *reinterpret_cast<const h8_t*>(kt + st * 16 * HD + (kk * 64 + lane) * 8);
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) s[st][cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[cg][kk], s[st][cg], 0, 0, 0);
      }
    }
  };
  auto scale_mask = [&](S_t& s, int step) {
    const int t0 = tb + step * TPS + kg * TPW;   // the wave's first tile
    if constexpr (KV8 != 0) {
#pragma unroll
      for (int st = 0; st < ST; ++st) {
        const f4_t ks = *reinterpret_cast<const f4_t*>(&scl[step % NS][0][kg * TPW * kTileKeys + st * 16 + 4 * j]);
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) s[st][cg] *= ks;
      }
    }
    if ((t0 + TPW) * kTileKeys > lim_lo) {
#pragma unroll
      for (int st = 0; st < ST; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = t0 * kTileKeys + st * 16 + 4 * j + i;
#pragma unroll
          for (int cg = 0; cg < CG; ++cg) s[st][cg][i] = key >= lim[cg] ? -INFINITY : s[st][cg][i];
        }
    }
  };
  float mn[CG];
  auto row_max = [&](const S_t& s) {   // the running maximum with s
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
      float mx = m[cg];
#pragma unroll
      for (int st = 0; st < ST; ++st) mx = max3(max3(mx, s[st][cg][0], s[st][cg][1]), s[st][cg][2], s[st][cg][3]);
      mn[cg] = col_max(mx);
    }
  };
  auto rescale = [&]() {   // rare once a row has seen some keys
    bool grow = false;
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) grow |= mn[cg] > m[cg];
    if (__any(grow)) {
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) {
        const float d = m[cg] - mn[cg];
        const float alpha = mn[cg] == m[cg] ? 1.f : __builtin_amdgcn_exp2f(RAW ? d * c2 : d);
        m[cg] = mn[cg];
        l[cg] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt][cg] *= alpha;
      }
    }
  };
  h8_t pb[TPW][CG];
  auto probs = [&](const S_t& s, int step) {   // P^T and the row sums
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
      // a row without a valid key yet keeps m = -inf: its masked scores give exp2(-inf) = 0
      const float mm = m[cg] == -INFINITY ? 0.f : RAW ? m[cg] * c2 : m[cg];
#pragma unroll
      for (int st = 0; st < ST; ++st) {
        f4_t vs;
        if constexpr (KV8 != 0) vs = *reinterpret_cast<const f4_t*>(&scl[step % NS][1][kg * TPW * kTileKeys + st * 16 + 4 * j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(RAW ? fmaf(s[st][cg][i], c2, -mm) : s[st][cg][i] - mm);
          l[cg] += p;
          pb[st / 2][cg][(st & 1) * 4 + i] = (_Float16)(RAW ? p : p * vs[i]);
        }
      }
    }
  };
  auto pv = [&](int step) {
    const _Float16* vt = smem + (step % NS) * SH::STAGE + (TPS + kg * TPW) * TILE;
#pragma unroll
    for (int tw = 0; tw < TPW; ++tw)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const h8_t va = *reinterpret_cast<const h8_t*>(vt + tw * TILE + (dt * 64 + lane) * 8);
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) o[dt][cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[tw][cg], o[dt][cg], 0, 0, 0);
      }
  };

  // Software pipeline: step n forms P(n) from S(n) while the matrix cores
  // take S(n + 1), then takes P(n) V(n) while the maximum of S(n + 1) is
  // formed; it reads group n (K(n + 1), V(n)) from LDS.
  S_t sa, sb;
  if constexpr (KV8 != 0) {
    load(pk, 0, 0);
    store(pk, 0, 0);
    request(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);
  } else {
    dma(0, 0);
#pragma unroll
    for (int g = 0; g < NS - 1; ++g) request(g);
    wait_vm<(NS - 1) * 2 * PW>();
  }
  lds_barrier();
  if (n_steps > 0) {
    qk(sa, 0);
    scale_mask(sa, 0);
    row_max(sa);
    rescale();
  }
  arrive(0);
  auto step = [&](S_t& cur, S_t& nxt, int n) {
    request(n + NS - 1);
    __builtin_amdgcn_sched_barrier(0);
    qk(nxt, n + 1);
    probs(cur, n);
    // P(n) is formed here, among the matrix instructions of S(n + 1), not
    // moved down to its use
#pragma unroll
    for (int tw = 0; tw < TPW; ++tw)
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) asm volatile("" : "+v"(pb[tw][cg]));
    __builtin_amdgcn_sched_barrier(0);
    scale_mask(nxt, n + 1);
    pv(n);
    row_max(nxt);
    rescale();
    arrive(n + 1);
  };
  int n = 0;
  for (; n + 2 < n_steps; n += 2) {
    step(sa, sb, n);
    step(sb, sa, n + 1);
  }
  if (n + 1 < n_steps) {
    step(sa, sb, n);
    probs(sb, n + 1);
    pv(n + 1);
  } else if (n < n_steps) {
    probs(sa, n);
    pv(n);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the requests past the range land before the slots are reused
  __syncthreads();
#pragma unroll
  for (int cg = 0; cg < CG; ++cg) {
    if (RAW) m[cg] *= c2;   // log2 units from here on
    l[cg] += __shfl_xor(l[cg], 16, kWave);
    l[cg] += __shfl_xor(l[cg], 32, kWave);
  }
  if constexpr (KH > 1) {
    // the other key groups' states into group 0's (over the stages, which the
    // last step's barrier has freed)
    f4_t* mg = reinterpret_cast<f4_t*>(smem);
    if (kg > 0) {
      f4_t* w = mg + ((kg - 1) * RG + rg) * kWave * (SH::STATE / 4) + lane;
      *w = f4_t{m[0], l[0], m[1], l[1]};
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) *(w += kWave) = o[dt][cg];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int k = 1; k < KH; ++k) {
        const f4_t* w = mg + ((k - 1) * RG + rg) * kWave * (SH::STATE / 4) + lane;
        const f4_t ml = *w;
        float f0[CG], f1[CG];
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
          const float m1 = ml[2 * cg], M = fmaxf(m[cg], m1);
          f0[cg] = m[cg] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[cg] - M);
          f1[cg] = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - M);
          m[cg] = M;
          l[cg] = l[cg] * f0[cg] + ml[2 * cg + 1] * f1[cg];
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int cg = 0; cg < CG; ++cg) {
            const f4_t p = *(w += kWave);
            o[dt][cg] = o[dt][cg] * f0[cg] + p * f1[cg];
          }
      }
    }
    __syncthreads();
  }
  if (a.splits > 1) {
    // fp32 partials of this key range: O [z][row][HD], then (m, l) [z][row]
    if (kg == 0) {
      const int64_t rows = (int64_t)a.n_kv * R, slot = (int64_t)z * rows + (int64_t)kvh * R;
      float* ml = a.part + (int64_t)a.splits * rows * HD;
#pragma unroll
      for (int cg = 0; cg < CG; ++cg) {
        const int r = rw + cg * 16 + h;
        if (r >= R) continue;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f4_t*>(a.part + (slot + r) * HD + dt * 16 + 4 * j) = o[dt][cg];
        if (j == 0) {
          ml[(slot + r) * 2] = m[cg];
          ml[(slot + r) * 2 + 1] = l[cg];
        }
      }
    }
    return;
  }
  // normalised rows through LDS (padded by 16 bytes so that the 16 rows of a
  // slice fall on different banks), written in 16-byte pieces
  if (kg == 0) {
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
      const float inv = 1.0f / (l[cg] + 1e-9f);
      _Float16* ot = smem + (rg * 16 * CG + cg * 16 + h) * SH::OS + 4 * j;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        h4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (_Float16)(o[dt][cg][i] * inv);
        *reinterpret_cast<h4_t*>(ot + dt * 16) = v;
      }
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < SH::ROWS * (HD / 8); idx += kPaThreads) {
    const int rl = idx / (HD / 8), p8 = idx % (HD / 8), r = r0 + rl;
    if (r >= R) break;
    const int t = r / g;
    *reinterpret_cast<h8_t*>(a.out + ((int64_t)t * a.n_heads + kvh * g + (r - t * g)) * HD + 8 * p8) =
        pf_group(*reinterpret_cast<const h8_t*>(smem + rl * SH::OS + 8 * p8), a.int4_layout);
  }
}

// Merge of the key ranges' partials, one thread per (row, 8 dims).
constexpr int kPaMergeThreads = 256;
template <int HD>
__global__ __launch_bounds__(kPaMergeThreads) void pf_attention_merge(const PfAttnArgs a) {
  const int g = a.n_heads / a.n_kv, R = a.M * g;
  const int64_t rows = (int64_t)a.n_kv * R;
  const int64_t idx = (int64_t)blockIdx.x * kPaMergeThreads + threadIdx.x;
  const int64_t row = idx / (HD / 8);
  const int p8 = (int)(idx % (HD / 8));
  if (row >= rows) return;
  const float* ml = a.part + (int64_t)a.splits * rows * HD;
  float M = -INFINITY;
#pragma unroll 8
  for (int z = 0; z < a.splits; ++z) M = fmaxf(M, ml[(z * rows + row) * 2]);
  float L = 0.f, v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int z = 0; z < a.splits; ++z) {
    const float mz = ml[(z * rows + row) * 2], lz = ml[(z * rows + row) * 2 + 1];
    const f4_t* p = reinterpret_cast<const f4_t*>(a.part + (z * rows + row) * HD + 8 * p8);
    const f4_t p0 = p[0], p1 = p[1];
    const float f = mz == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mz - M);
    L += lz * f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = fmaf(p0[e], f, v[e]);
      v[4 + e] = fmaf(p1[e], f, v[4 + e]);
    }
  }
  const float inv = 1.0f / (L + 1e-9f);
  h8_t o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (_Float16)(v[e] * inv);
  const int kvh = (int)(row / R), r = (int)(row % R), t = r / g;
  *reinterpret_cast<h8_t*>(a.out + ((int64_t)t * a.n_heads + kvh * g + (r - t * g)) * HD + 8 * p8) = pf_group(o, a.int4_layout);
}

// E4M3 cache: block = (16 consecutive tokens, one query head), the 16 tokens
// being the columns of S^T = K Q^T; 8 waves take every 8th 32-key tile up to
// the last token's position and merge in LDS.  A code of this cache is a
// coarse number (a step is up to 1/8 of the value), so one different rounding
// anywhere in the layers before turns some of a prompt's codes into their
// neighbours.  Prompts over this cache therefore keep this kernel (and the
// GEMMs' 128-token tile, PfGemmArgs::keep_tile) and with them the codes that
// they have always had, although the kernel above is the faster one (84 ->
// 47 us with int8 codes at 777 tokens after 3000, 12 / 2 heads).  (Bit for
// bit where the QKV tile is split over K; passes of more than about 1000
// tokens run it unsplit, and its rotation is contracted differently since
// the sines come from a table: 3 in a million of a layer's K codes.)
template <int HD>
__global__ __launch_bounds__(kAttnThreads) void pf_attention_e4m3_kernel(const PfAttnArgs a) {
  constexpr int KK = HD / 32, DT = HD / 16;
  const int t0 = blockIdx.x * 16, hq = blockIdx.y;
  const int g = a.n_heads / a.n_kv, kvh = hq / g;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int h = lane & 15, j = lane >> 4;   // h: token column
  const int tcol = min(t0 + h, a.M - 1);
  const int t_lane = a.pos0 + tcol + 1;                       // keys visible to this column
  const int t_max = a.pos0 + min(t0 + 16, a.M);               // keys visible to the block
  const int n_tiles = (t_max + kTileKeys - 1) / kTileKeys;
  const float scale = 1.0f / sqrtf((float)HD);
  h8_t qb[KK];
  const _Float16* q = a.q + (int64_t)tcol * a.n_heads * HD + hq * HD;
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) qb[kk] = __builtin_bit_cast(h8_t, load_u4(q + kk * 32 + j * 8));
  float m = -INFINITY, l = 0.f;
  f4_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f4_t{0.f, 0.f, 0.f, 0.f};
  int ti = wave;
  const int8_t* kb8 = a.kcache8 + (int64_t)kvh * a.max_seq * HD;
  const int8_t* vb8 = a.vcache8 + (int64_t)kvh * a.max_seq * HD;
  const float* ksc = a.kscale + (int64_t)kvh * a.max_seq;
  const float* vsc = a.vscale + (int64_t)kvh * a.max_seq;
  const uint32_t magic = vgpr_const(0x64646464u);
  KVTile8<HD> A, B;
  if (ti < n_tiles) load_tile8<HD>(A, kb8, vb8, ksc, vsc, ti, lane);
  for (; ti < n_tiles; ti += 2 * kAttnWaves) {
    const int t1 = ti + kAttnWaves;
    if (t1 < n_tiles) load_tile8<HD>(B, kb8, vb8, ksc, vsc, t1, lane);
    attend_tile8<HD, CQ_KV_FP8>(A, qb, ti, t_lane, scale, j, m, l, o, magic);
    if (t1 >= n_tiles) break;
    if (t1 + kAttnWaves < n_tiles) load_tile8<HD>(A, kb8, vb8, ksc, vsc, t1 + kAttnWaves, lane);
    attend_tile8<HD, CQ_KV_FP8>(B, qb, t1, t_lane, scale, j, m, l, o, magic);
  }
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);

  __shared__ float wm[kAttnWaves][16], wl[kAttnWaves][16];
  __shared__ float wo[kAttnWaves][16][HD + 1];
  if (j == 0) { wm[wave][h] = m; wl[wave][h] = l; }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) wo[wave][h][dt * 16 + 4 * j + i] = o[dt][i];
  __syncthreads();
  const int qd = a.n_heads * HD;
  for (int idx = threadIdx.x; idx < 16 * HD; idx += kAttnThreads) {
    const int c = idx / HD, d = idx % HD;
    if (t0 + c >= a.M) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) M = fmaxf(M, wm[w][c]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      const float f = wm[w][c] == -INFINITY ? 0.f : __expf(wm[w][c] - M);
      L += wl[w][c] * f;
      O += wo[w][c][d] * f;
    }
    const int k = hq * HD + d;
    a.out[(int64_t)(t0 + c) * qd + pf_pos(k, a.int4_layout)] =
        pf_val((float)(_Float16)(O * (1.0f / (L + 1e-9f))), k, a.int4_layout);
  }
}

// Rows per block (through the key groups KH) and key ranges S.  Model, in
// microseconds, fitted to 14 shapes x 3 KH x up to 10 S (within 20 % of the
// measured times, picks within 10 % of the best): one block fits a CU; a key
// group takes c per 32-key tile, a block 7 besides (4 of them hidden behind
// its predecessor in later rounds); a round lasts as long as its longest
// block, the blocks being dispatched longest first; merging the key groups in
// LDS takes 0.7 (KH = 2) or 1.4; the ranges' fp32 partials
// are written and read at 5 TB/s, and merging S of them takes 4 + 0.3 S.
struct PaPlan { int kh, splits; };
PaPlan pa_plan(const PfAttnArgs& a) {
  const int R = a.M * (a.n_heads / a.n_kv);
  const double tiles_hi = (a.pos0 + a.M + kTileKeys - 1) / kTileKeys, tiles_lo = (double)(a.pos0 + 1) / kTileKeys;
  const size_t row_bytes = (size_t)a.n_kv * R * (a.head_dim + 2) * sizeof(float);   // partials of one range
  if (a.want_rows) {
    const int most = (int)std::min<size_t>((size_t)tiles_hi, a.part_bytes / row_bytes);
    return PaPlan{kPaWaves * 16 * kPaCols / a.want_rows, std::max(std::min(a.want_splits, most), 1)};
  }
  PaPlan best{1, 1};
  double best_t = 1e30;
  for (int kh = 1; kh <= 4; kh *= 2) {
    const int rows = kPaWaves / kh * 16 * kPaCols, n_rb = (R + rows - 1) / rows;
    const double c = (a.head_dim == 64 ? 0.68 : kh == 4 ? 1.4 : 1.05) * (a.kcache8 ? 1.15 : 1.0);
    for (int s = 1; s <= 64 && s <= tiles_hi; ++s) {
      if (s > 1 && (!a.part || s * row_bytes > a.part_bytes)) break;
      const int64_t blocks = (int64_t)n_rb * a.n_kv * s;
      const double hi = std::ceil(tiles_hi / (kh * s)), lo = std::max(1.0, tiles_lo / (kh * s));
      double t = 4.0 + 0.7 * (kh / 2) + (s > 1 ? 4.0 + 0.3 * s + 2.0 * s * row_bytes / 5e6 : 0.0);
      for (int64_t first = 0; first < blocks && t < best_t; first += kNumCUs) t += (hi - (hi - lo) * first / blocks) * c + 3.0;
      if (t < best_t) { best_t = t; best = PaPlan{kh, s}; }
    }
  }
  return best;
}

template <int HD, int KV8, int KH, int TPW>
int pa_launch(PfAttnArgs a, int splits, hipStream_t stream) {
  const int g = a.n_heads / a.n_kv;
  a.n_rb = (a.M * g + PaShape<HD, KV8, KH, TPW>::ROWS - 1) / PaShape<HD, KV8, KH, TPW>::ROWS;
  a.splits = splits;
  hipLaunchKernelGGL((pf_attention_kernel<HD, KV8, KH, TPW>), dim3(a.n_rb * a.n_kv * splits), dim3(kPaThreads), 0, stream, a);
  CQ_HIP(hipGetLastError());
  if (splits > 1) {
    const int64_t n = (int64_t)a.M * a.n_heads * (HD / 8);
    hipLaunchKernelGGL((pf_attention_merge<HD>), dim3((unsigned)((n + kPaMergeThreads - 1) / kPaMergeThreads)),
                       dim3(kPaMergeThreads), 0, stream, a);
    CQ_HIP(hipGetLastError());
  }
  return CQ_OK;
}

template <int HD, int KV8>
int pa_dispatch(const PfAttnArgs& a, hipStream_t stream) {
  const PaPlan p = pa_plan(a);
  if (p.kh == 1) return pa_launch<HD, KV8, 1, 2>(a, p.splits, stream);
  if (p.kh == 2) return pa_launch<HD, KV8, 2, HD == 128 && KV8 ? 1 : 2>(a, p.splits, stream);
  return pa_launch<HD, KV8, 4, HD == 64 ? 2 : 1>(a, p.splits, stream);
}

template <int HD>
int pa_format(const PfAttnArgs& a, hipStream_t stream) {
  if (!a.kcache8) return pa_dispatch<HD, 0>(a, stream);
  if (a.kv_fmt != CQ_KV_FP8) return pa_dispatch<HD, CQ_KV_INT8>(a, stream);
  hipLaunchKernelGGL((pf_attention_e4m3_kernel<HD>), dim3((a.M + 15) / 16, a.n_heads), dim3(kAttnThreads), 0, stream, a);
  CQ_HIP(hipGetLastError());
  return CQ_OK;
}

}  // namespace

int launch_pf_attention(const PfAttnArgs& a, hipStream_t stream) {
  if (a.head_dim != 64 && a.head_dim != 128) return fail(CQ_EINVAL, "prefill attention: head_dim must be 64 or 128");
  if (a.M <= 0 || a.pos0 < 0 || a.pos0 + a.M > a.max_seq) return fail(CQ_ERANGE, "prefill attention: positions");
  if (a.kcache8 && (!a.vcache8 || !a.kscale || !a.vscale)) return fail(CQ_EINVAL, "prefill attention: quantized cache pointers");
  if (a.want_rows) {
    if (a.want_rows != 64 && a.want_rows != 128 && a.want_rows != 256)
      return fail(CQ_EINVAL, "prefill attention: no form with that many rows");
    if (a.want_splits < 1 || (a.want_splits > 1 && !a.part)) return fail(CQ_EINVAL, "prefill attention: key ranges");
  }
  return a.head_dim == 128 ? pa_format<128>(a, stream) : pa_format<64>(a, stream);
}

}  // namespace cq
