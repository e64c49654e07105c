// Backbone prefill on MI355X (gfx950): the S prompt tokens through every layer at once, the
// projections and both attention products on bf16 MFMA with f32 accumulation, K and V written
// straight into the decode kernels' cache layout [layers, 8, max_seq, 128] bf16.
//
// What it replaces: the reference prefills with the qwen_tts PyTorch talker forward in bf16
// (generator.py:209-225: transformers Qwen3DecoderLayer op order, TF/qwen3/modeling_qwen3.py
// :50-64, :140-208, :211-324) and then copies that DynamicCache into the megakernel cache
// (generator.py:245-257, megakernel_backbone.py:285-294); the first group-0 token comes from
// the last position's hidden through the codec head (generator.py:113-117). Every value is
// rounded where that bf16 forward rounds it:
//   xn  = w x / sqrt(mean(x^2) + eps)                                  RMSNorm (:59-64), as bf16(x w) into
//         the next product and 1 / sqrt(..) on its f32 sums (one rounding of xn; transformers has two);
//         the q/k norms and the final norm round as transformers does
//   q,k,v = bf16(W xn); q,k per head through RMSNorm, then
//   rope = bf16(bf16(q * cos) + bf16(rotate_half(q) * sin))            bf16 cos/sin tables
//   s   = scale * (q . k) in f32; att = bf16((sum_j bf16(e^(s_j - m)) v_j) / sum_j e^(s_j - m))
//         with the running max m: the scores and softmax as flash-style attention kernels
//         (torch's sdpa on bf16) keep and round them, normalised after the P V product (eager
//         torch rounds s = bf16(bf16(q . k) * scale) and p = bf16(e / l) before it; :185-208)
//   h1  = bf16(h + bf16(W_o att)); a = bf16(bf16(silu(bf16(W_g xn))) * bf16(W_u xn))
//   h   = bf16(h1 + bf16(W_d a)); hidden = RMSNorm_final(h[S-1]); logits = bf16(W_head hidden)
// The f32 sums run in MFMA order rather than the CPU's, so an f32 result can land on the other
// side of a bf16 rounding boundary now and then; parity is a tolerance, not bit equality.
//
// Kernels (the host loop over layers is in qtts_backbone_prefill below), five launches a layer:
//   embed_kernel       the embeddings into the residual stream, layer 0's norm inputs
//   tile_gemm_kernel   the four projections, K unsplit, with the norms, RoPE, K/V write, residual and SwiGLU
//                      in their epilogues
//   attn_kernel        causal GQA, 4 waves per (32-query block, query head) splitting the key blocks: S^T = K
//                      Q^T on MFMA (each lane then holds one query's scores, so the row max and sum stay in
//                      the lane and its partner half-wave), one pass with a running max, O^T += V^T P^T on
//                      MFMA with V^T read from the row-major V block through LDS transpose reads; further
//                      workgroups read the weights of the launches that follow
//   attn_pair_kernel   the same for long prompts: 8 waves per (32-query block, KV head), the two query heads
//                      sharing each staged K and V block
//   final_head_kernel  the last token's final norm and codec head
//   select_kernel      suppress mask + EOS suppression + the decode kernels' selection
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include "qwentts_amd.h"
#include "qtts_common.h"
#include "qtts_select.h"

namespace qtts {
namespace pf {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float EPS = 1e-6f;                 // Qwen3RMSNorm eps (config rms_norm_eps)
constexpr int QROW = 136;                    // LDS row of the query block: 128 dims + 16-byte pad

__device__ __forceinline__ bf16x8 as_bf8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// bf16 rounding (round to nearest even) with gfx950's conversion instruction
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float rbh(float x) { return (float)(__bf16)x; }
__device__ __forceinline__ bf16_t f2bh(float x) { return __builtin_bit_cast(bf16_t, (__bf16)x); }
__device__ __forceinline__ uint32_t pack_bh(float lo, float hi) {
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

#define QTTS_PF_INLINE __attribute__((always_inline))
typedef __attribute__((address_space(1))) void gvoid_t;
typedef __attribute__((address_space(3))) void lvoid_t;

__device__ __forceinline__ const bf16_t* tbl(const TTSLayerWeights* lw, int field) {
  return reinterpret_cast<const bf16_t*>(ld_const(reinterpret_cast<const void* const*>(lw) + field));
}

// x sigmoid(x) in f32 from the hardware exp2 and reciprocal (about 2 ulp of f32 from x / (1 + e^-x),
// far below the bf16 rounding that follows; large |x| gives x or -0 as the exact form does)
__device__ __forceinline__ float silu_f(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}

// The last token's final norm (hidden, bf16 values as f32) and, with a codec head, its logits: every wave
// norms the row for itself (2 KB) and takes RPW rows of the head. One launch; as a norm, a split-K matrix
// product and its reduction it took three, 14 us together.
constexpr int RPW = 4;
__global__ void __launch_bounds__(256) final_head_kernel(const bf16_t* x, const bf16_t* gain, const bf16_t* head, int vocab,
                                                         float* out_hidden, bf16_t* logits) {
  const int lane = threadIdx.x & 63, w = blockIdx.x * 4 + (threadIdx.x >> 6);
  u32x4 v[2], gw[2], hw[RPW][2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    v[k] = ldw(x + 8 * (lane + 64 * k));
    gw[k] = ldw(gain + 8 * (lane + 64 * k));
  }
  if (head != nullptr) {
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
      for (int k = 0; k < 2; ++k) hw[r][k] = ldw(head + (size_t)min(RPW * w + r, vocab - 1) * HID + 8 * (lane + 64 * k));
  }
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += bflo(v[k][e]) * bflo(v[k][e]) + bfhi(v[k][e]) * bfhi(v[k][e]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
  const float rs = 1.0f / sqrtf(ss / (float)HID + EPS);
  float y[16];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[8 * k + 2 * e] = rbh(bflo(gw[k][e]) * rbh(bflo(v[k][e]) * rs));
      y[8 * k + 2 * e + 1] = rbh(bfhi(gw[k][e]) * rbh(bfhi(v[k][e]) * rs));
    }
  if (w == 0 && out_hidden != nullptr) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) out_hidden[8 * (lane + 64 * k) + e] = y[8 * k + e];
  }
  if (head == nullptr) return;
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) s += bflo(hw[r][k][e]) * y[8 * k + 2 * e] + bfhi(hw[r][k][e]) * y[8 * k + 2 * e + 1];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0 && RPW * w + r < vocab) logits[RPW * w + r] = f2bh(s);
  }
}

// Causal GQA attention of S queries (positions p0 .. p0 + S - 1) over cache positions
// 0 .. p0 + S - 1, one workgroup of AW waves per (32-query block, query head); wave w takes the
// 32-key blocks kb = w, w + AW, ... in one pass with a running (online) softmax:
//   * S^T = K Q^T on MFMA 32x32x16 (A = the K block staged in the wave's LDS rows, B = Q^T from
//     the block's queries in LDS): lane (half hf, column c) holds query 32 qb + c's scores for
//     keys 8 (r >> 2) + 4 hf + (r & 3), r < 16, so a query's row max and sum stay in the lane and
//     its partner half-wave. The scores stay in f32 and the scale goes into the exponent:
//     e^(s - m) = 2^((q . k - m') scale log2 e) for the unscaled running max m'.
//   * The running max m moves to m' = max(m, block max); O^T and the sum l scale by e^(m - m')
//     (skipped when no query of the wave moved); p = e^(s - m') rounded to bf16 is the B operand
//     of O^T += V^T P^T, reusing the score registers in place (k-index 8 hf + j of step kk2 is key
//     16 kk2 + 8 (j >> 2) + 4 hf + (j & 3)); l sums the f32 e^(s - m').
//   * V^T comes from the V block staged row-major (16-byte writes) through the LDS transpose read
//     ds_read_b64_tr_b16: in each 16-lane group, with M[l][j] = the 4 bf16 at lane l's address,
//     lane i receives M[4 j + (i >> 2)][i & 3], j < 4. Lane i of group g (hf = g >> 1) passes
//     row 16 kk2 + 4 hf (+ 8) + (i >> 2), columns 32 mb + 16 (g & 1) + 4 (i & 3): it receives
//     dims 32 mb + 16 (g & 1) + i, keys 16 kk2 + 4 hf (+ 8) + 0..3, the A operand of O^T.
// The softmax normalisation comes last (att = bf16(O / l)), as in flash-style kernels; the waves'
// (m, l, O^T) merge through LDS in wave order. Grid: 16 x (query blocks) workgroups, KV head =
// linear id mod 8 (one head per XCD's L2), the longest query blocks first.
constexpr int AW = 4;
constexpr int VROW = 160;     // LDS row of a staged V block (bf16): 320 B puts the 4 rows one
                              // transpose read touches 16 banks apart
constexpr int WST = 32 * VROW;                      // a wave's staging region (K block, then V)
constexpr int ATT_Q = 32 * QROW;                    // the query block
constexpr int ATT_SMEM = std::max((ATT_Q + AW * WST) * 2, AW * HDIM * 32 * 4 + AW * 2 * 32 * 4);
static_assert(32 * QROW <= WST, "a wave's LDS region holds its staged K block");

typedef short v4s __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 lds_tr16(const bf16_t* p) {
  const v4s r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) v4s*)((__attribute__((address_space(3))) void*)p));
  return __builtin_bit_cast(u32x2, r);
}

// The weights that follow the attention are read while it runs: attn_kernel leaves most of the memory system
// idle, and the projections after it would wait for each line to come from HBM. A workgroup reads one 16 KB
// piece (64 bytes a thread) of the layer's O, gate, up and down weights and of the next layer's q, k and v,
// into the memory-side cache. Us a layer over 28 layers without and with: 13 tokens 37.9 : 34.3, 64 40.1 : 35.9,
// 128 40.0 : 36.8, 200 42.9 : 41.4, 333 56.3 : 53.7, 512 60.1 : 55.8, 700 76.0 : 70.9 (without the next layer's
// 0.4 to 0.9 more; 192 workgroups that share the pieces 1 to 3 more). Done by the projections themselves for
// their own operands it was slower.
constexpr int PIECE = 16384;
constexpr int kPiecesSq = HID * NQH * HDIM * 2 / PIECE, kPiecesKv = kPiecesSq / 2, kPiecesMlp = INTER * HID * 2 / PIECE;
constexpr int kPiecesLayer = kPiecesSq + 3 * kPiecesMlp, kPiecesNext = kPiecesSq + 2 * kPiecesKv;
static_assert(64 * AW * 64 == PIECE, "64 bytes a thread");
__device__ __forceinline__ void weight_piece_ahead(const TTSLayerWeights* lw, int u) {
  int field = 6;                                        // O
  if (u >= kPiecesLayer) {
    u -= kPiecesLayer;
    ++lw;
    field = u < kPiecesSq ? 1 : (u < kPiecesSq + kPiecesKv ? 2 : 3);
    u -= field == 1 ? 0 : (field == 2 ? kPiecesSq : kPiecesSq + kPiecesKv);
  } else if (u >= kPiecesSq) {
    u -= kPiecesSq;
    field = 8 + u / kPiecesMlp;
    u %= kPiecesMlp;
  }
  const bf16_t* p = tbl(lw, field) + (size_t)u * (PIECE / 2);
  u32x4 v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = ldw(p + (threadIdx.x + 64 * AW * r) * 8);
#pragma unroll
  for (int r = 0; r < 4; ++r) asm volatile("" ::"v"(v[r]));   // (keeps the loads)
}

__global__ void __launch_bounds__(64 * AW, 2) attn_kernel(const bf16_t* qrows, const bf16_t* kc, const bf16_t* vc,
                                                       int layer, int max_seq, int p0, int S, bf16_t* att,
                                                       float scale, const TTSLayerWeights* layers) {
  if ((int)blockIdx.x >= (S + 31) / 32 * NQH) {   // workgroups past the queries'
    weight_piece_ahead(layers + layer, (int)blockIdx.x - (S + 31) / 32 * NQH);
    return;
  }
  __shared__ __attribute__((aligned(16))) char smem[ATT_SMEM];
  bf16_t* sq = reinterpret_cast<bf16_t*>(smem);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, hf = lane >> 5, c = lane & 31;
  // XCD-aware order: workgroups go to the XCDs round-robin by linear id, so id & 7 picks the KV
  // head and each XCD's L2 holds one head's K and V; within it, the longest query blocks first
  const int nqb = (S + 31) / 32, id = blockIdx.x;
  const int kvh = id & 7, rest = id >> 3;
  const int hq = 2 * kvh + (rest & 1), qb = nqb - 1 - (rest >> 1);
  const int i = 32 * qb + c;
  const bool qok = i < S;
  const int qpos = p0 + i;
  const int last = p0 + min(S, 32 * qb + 32) - 1;   // last key any query of the block sees
  const int nkb = last / 32 + 1;
  bf16_t* st = sq + ATT_Q + w * WST;   // the wave's K block, then its V block

  // the block's 32 query rows (512 16-byte chunks) go to LDS once
#pragma unroll
  for (int j = 0; j < 512 / (64 * AW); ++j) {
    const int ch = threadIdx.x + 64 * AW * j, qrow = ch >> 4, qcol = 8 * (ch & 15);
    const int qi = 32 * qb + qrow;
    const u32x4 v = ldw(qrows + (size_t)(qi < S ? qi : 0) * (NQH * HDIM) + hq * HDIM + qcol);   // clamped row
    *reinterpret_cast<u32x4*>(&sq[qrow * QROW + qcol]) = qi < S ? v : u32x4{0u, 0u, 0u, 0u};
  }
  __syncthreads();
  const size_t hbase = ((size_t)layer * NKVH + kvh) * max_seq * HDIM;
  const bf16_t* kb_ = kc + hbase;
  const bf16_t* vb_ = vc + hbase;

  // K and V blocks (32 keys x 128 dims each) in 8 coalesced 1 KB rounds, issued a block ahead:
  // round r, lane j loads key 32 kb + 4 r + (j >> 4), dims 8 (j & 15) .. + 7. Loads are
  // unconditional from a clamped row (row 0 past `last`) and staged as loaded: a load or a store
  // under a branch makes the compiler wait for every outstanding load, the prefetch included. Keys
  // past `last` are past every query of the block, so their scores are masked to -inf and their
  // weights are exactly 0 against the finite K and V of row 0.
  auto load = [&](const bf16_t* base, int kb, u32x4 (&rr)[8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int key = 32 * kb + 4 * r + (lane >> 4);
      rr[r] = ldw(base + (size_t)(key <= last ? key : 0) * HDIM + 8 * (lane & 15));
    }
  };
  auto stage = [&](const u32x4 (&rr)[8], int pitch) {
#pragma unroll
    for (int r = 0; r < 8; ++r) *reinterpret_cast<u32x4*>(&st[(4 * r + (lane >> 4)) * pitch + 8 * (lane & 15)]) = rr[r];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  };
  auto scores = [&](int kb, float (&sc)[16]) {
    // two independent 4-step MFMA chains (even and odd 16-dim steps), added at the end; Q^T
    // (query c, dims 16 kk + 8 hf ..) and K (key c, the same dims) from LDS, both with row pitch
    // QROW; the offset is opaque so the reads stay in the loop instead of being hoisted
    f32x16 acc, acc2;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = acc2[r] = 0.0f;
    int qo = c * QROW + 8 * hf;
    asm volatile("" : "+v"(qo));
    const bf16_t* qp = &sq[qo];
    const bf16_t* kp = &st[qo];
#pragma unroll
    for (int kk = 0; kk < 8; kk += 2) {
      const u32x4 q0 = *reinterpret_cast<const u32x4*>(qp + 16 * kk);
      const u32x4 q1 = *reinterpret_cast<const u32x4*>(qp + 16 * kk + 16);
      const u32x4 k0 = *reinterpret_cast<const u32x4*>(kp + 16 * kk);
      const u32x4 k1 = *reinterpret_cast<const u32x4*>(kp + 16 * kk + 16);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(k0), as_bf8(q0), acc, 0, 0, 0);
      acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(k1), as_bf8(q1), acc2, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += acc2[r];
    // blocks that every query of the block sees whole (the wave-uniform common case) skip the mask
    if (32 * kb + 31 <= p0 + 32 * qb && 32 * qb + 31 < S) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[r] = acc[r];
    } else {
      const int lim = qok ? qpos : -1;   // last key this lane's query sees (none past the prompt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * kb + 8 * (r >> 2) + 4 * hf + (r & 3);
        sc[r] = kr <= lim ? acc[r] : -INFINITY;
      }
    }
  };
  // e^(scale (s - m)) as 2^(s scale log2 e - m scale log2 e): one fma into the hardware exp2
  const float SL = scale * 1.4426950408889634f;
  auto ex = [SL](float s, float nm) { return __builtin_amdgcn_exp2f(fmaf(s, SL, nm)); };

  float m = -INFINITY, l = 0.0f;
  f32x16 o[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[mb][r] = 0.0f;
  // transpose-read addresses of this lane (see above), relative to the staged V block
  const int gi = lane & 15, g = lane >> 4;
  const int tr_off = (4 * (g >> 1) + (gi >> 2)) * VROW + 16 * (g & 1) + 4 * (gi & 3);
  u32x4 kr[8], vr[8];
  // K before V here as in the loop: with the same load order on both edges into the loop, the
  // wait before each staging counts only the block it stages (the other block's prefetch stays in
  // flight); with V scheduled first here, the compiler waited for every load at the loop top
  load(kb_, w, kr);
  __builtin_amdgcn_sched_barrier(0);
  load(vb_, w, vr);
  for (int kb = w; kb < nkb; kb += AW) {
    stage(kr, QROW);
    load(kb_, kb + AW, kr);
    float sc[16];
    scores(kb, sc);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // K reads before the V staging
    stage(vr, VROW);
    load(vb_, kb + AW, vr);
    // running max; a fully masked row so far keeps m = -inf and adds nothing
    float bm = sc[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) bm = fmaxf(bm, sc[r]);
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
    const float mn = fmaxf(m, bm);
    const float nm = mn == -INFINITY ? 0.0f : -mn * SL;
    if (__builtin_amdgcn_ballot_w64(mn != m) != 0ull) {
      const float al = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * SL);
      l *= al;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[mb][r] *= al;
    }
    m = mn;
    float e[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      e[r] = ex(sc[r], nm);
      l += e[r];
    }
#pragma unroll
    for (int kk2 = 0; kk2 < 2; ++kk2) {
      u32x4 pb;
#pragma unroll
      for (int j = 0; j < 4; ++j) pb[j] = pack_bh(e[8 * kk2 + 2 * j], e[8 * kk2 + 2 * j + 1]);
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const bf16_t* vp = &st[16 * kk2 * VROW + 32 * mb + tr_off];
        const u32x2 lo = lds_tr16(vp);
        const u32x2 hi = lds_tr16(vp + 8 * VROW);
        const u32x4 av = {lo[0], lo[1], hi[0], hi[1]};
        o[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(av), as_bf8(pb), o[mb], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // V reads before the next K staging
  }
  l += __shfl_xor(l, 32, 64);

  // merge the waves: M = max m_w, L = sum l_w e^(m_w - M), O = sum O_w e^(m_w - M) (wave order), wave w
  // finishing dims 32 w .. 32 w + 31 (one wave that merged and stored all of them took up to 1 us longer)
  float* ob = reinterpret_cast<float*>(smem);   // [wave][dim block][register quad][lane][4]
  float* sml = ob + AW * HDIM * 32;             // [AW][2][32]
  __syncthreads();   // every wave's staging region is dead
  if (hf == 0) {
    sml[(w * 2) * 32 + c] = m;
    sml[(w * 2 + 1) * 32 + c] = l;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int v = 0; v < AW; ++v) M = fmaxf(M, sml[(v * 2) * 32 + c]);
  float L = 0.0f;
#pragma unroll
  for (int v = 0; v < AW; ++v) {
    const float mv = sml[(v * 2) * 32 + c];
    L += mv == -INFINITY ? 0.0f : sml[(v * 2 + 1) * 32 + c] * __builtin_amdgcn_exp2f((mv - M) * SL);
  }
  const float sw = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - M) * SL);
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = o[mb][4 * r + e] * sw;
      *reinterpret_cast<f32x4*>(ob + ((w * 4 + mb) * 4 + r) * 256 + lane * 4) = x;
    }
  __syncthreads();
  if (!qok) return;
  const float rl = L > 0.0f ? 1.0f / L : 0.0f;
  // O^T layout: column = query c, register r of block mb = dim 32 mb + 8 (r >> 2) + 4 hf + (r & 3)
  static_assert(AW == 4, "a dim block per wave");
  bf16_t* orow = att + (size_t)i * (NQH * HDIM) + hq * HDIM + 32 * w + 4 * hf;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    f32x4 x = *reinterpret_cast<const f32x4*>(ob + (w * 4 + r) * 256 + lane * 4);
#pragma unroll
    for (int v = 1; v < AW; ++v) x += *reinterpret_cast<const f32x4*>(ob + ((v * 4 + w) * 4 + r) * 256 + lane * 4);
    u32x2 pk;
    pk[0] = pack_bh(x[0] * rl, x[1] * rl);
    pk[1] = pack_bh(x[2] * rl, x[3] * rl);
    *reinterpret_cast<u32x2*>(orow + 8 * r) = pk;
  }
}

// Wait until at most N of this wave's vector-memory instructions and none of its LDS reads are in flight (the
// compiler does not track LDS writes made by DMA).
template <int N>
__device__ __forceinline__ void wait_vm_lds() {
  static_assert(N >= 0 && N <= 63, "vmcnt field");
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

// The same attention for long prompts, one workgroup of 8 waves per (32-query block, KV head): wave (hd, ks)
// takes query head 2 kvh + hd and the 32-key blocks kb = ks, ks + 4, ... in one pass with a running (online)
// softmax. The two heads of a KV head share each staged K and V block, and the queries stay in registers, so
// that a wave's 32 x 32 block costs 24 KB of LDS traffic (40 KB in attn_kernel): 44.8 -> 34.6 us at 2048 tokens
// (kernel trace).
// What bounds it now is the chain of a step (1.6 us: wait and barrier 0.4, copies issued 0.3, scores, softmax and
// P V 0.3 each) at two waves a SIMD: taking the next block's scores under this one's softmax, or staging through
// registers two steps ahead, changed nothing.
//   * K and V blocks (32 keys x 128 dims) come by DMA into the pair's two buffers, one step ahead; chunk c
//     (16 bytes) of row r sits at position c ^ (r & 7).
//   * The layouts of S^T, P and O^T are attn_kernel's; O^T and l are rescaled only when some query's block
//     max passes the running one by more than 2^8.
// The key splits of a head merge through LDS in split order, wave ks finishing dims 32 ks .. 32 ks + 31.
// Workgroups: KV head = linear id mod 8 (one head per XCD's L2), the longest query blocks first.
constexpr int AKS = 4;                              // key splits
constexpr int ABLK = 32 * HDIM * 2;                 // bytes of a K or V block
constexpr int ATTP_SMEM = AKS * 2 * 2 * ABLK + 2 * AKS * 2 * 32 * 4;   // (K, V) x 2 buffers per split; (m, l) of the merge

// The 8 transpose reads of a 16-key step: the low and high 4 keys of 4 dim blocks at LDS addresses a[0..3],
// OFF bytes further. In assembly, with their wait: before the builtin the compiler waits for every DMA in
// flight, the next block's among them (it takes any of them for the read's source).
template <int OFF>
__device__ __forceinline__ void lds_tr16x8(const uint32_t (&a)[4], u32x2 (&lo)[4], u32x2 (&hi)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%c12\n\tds_read_b64_tr_b16 %4, %8 offset:%c13\n\t"
      "ds_read_b64_tr_b16 %1, %9 offset:%c12\n\tds_read_b64_tr_b16 %5, %9 offset:%c13\n\t"
      "ds_read_b64_tr_b16 %2, %10 offset:%c12\n\tds_read_b64_tr_b16 %6, %10 offset:%c13\n\t"
      "ds_read_b64_tr_b16 %3, %11 offset:%c12\n\tds_read_b64_tr_b16 %7, %11 offset:%c13\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(lo[1]), "=&v"(lo[2]), "=&v"(lo[3]), "=&v"(hi[0]), "=&v"(hi[1]), "=&v"(hi[2]), "=&v"(hi[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "i"(OFF), "i"(OFF + 8 * HDIM * 2)
      : "memory");
}

__global__ void __launch_bounds__(128 * AKS, 2) attn_pair_kernel(const bf16_t* qrows, const bf16_t* kc, const bf16_t* vc,
                                                            int layer, int max_seq, int p0, int S, bf16_t* att, float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[ATTP_SMEM];   // (one LDS object, as in tile_gemm_kernel)
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int hd = w & 1, ks = w >> 1, hf = lane >> 5, c = lane & 31;
  const int nqb = (S + 31) / 32, id = blockIdx.x;
  const int kvh = id & 7, qb = nqb - 1 - (id >> 3);
  const int hq = 2 * kvh + hd;
  const int i = 32 * qb + c;
  const bool qok = i < S;
  const int last = p0 + min(S, 32 * qb + 32) - 1;   // last key any query of the block sees
  const int nkb = last / 32 + 1, nst = (nkb + AKS - 1) / AKS;
  const size_t hbase = ((size_t)layer * NKVH + kvh) * max_seq * HDIM;

  // wave (hd, ks) copies rows 16 hd .. 16 hd + 15 of the split's K block and of its V block, 4 rows an
  // instruction, through buffer descriptors that end after row `last`: rows past it come as zeros (their
  // scores are masked), and a step moves one scalar offset, no vector address
  char* const buf = smem + ks * 4 * ABLK;
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(kc + hbase), (short)0,
                                                                       (last + 1) * HDIM * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(vc + hbase), (short)0,
                                                                       (last + 1) * HDIM * 2, 0x00020000);
  const int drow = 16 * hd + (lane >> 4);
  int doff[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) doff[r] = (drow + 4 * r) * HDIM * 2 + ((lane & 15) ^ ((drow + 4 * r) & 7)) * 16;
  auto issue = [&](int b, int kb) QTTS_PF_INLINE {
    const int so = min(kb, nkb - 1) * ABLK;   // inside the descriptor: only the rows of a block can pass its end
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      char* dst = buf + b * 2 * ABLK + (16 * hd + 4 * r) * HDIM * 2;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (lvoid_t*)dst, 16, doff[r], so, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (lvoid_t*)(dst + ABLK), 16, doff[r], so, 0, 0);
    }
  };
  // e^(scale (s - m)) as 2^(s scale log2 e - m scale log2 e): one fma into the hardware exp2
  const float SL = scale * 1.4426950408889634f;
  auto ex = [SL](float s, float nm) QTTS_PF_INLINE { return __builtin_amdgcn_exp2f(fmaf(s, SL, nm)); };

  float m = -INFINITY, l = 0.0f;
  f32x16 o[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[mb][r] = 0.0f;
  // LDS offsets of this lane: K row c (chunk 2 kk + hf), and the transpose reads of V (row vr, chunk
  // 4 mb + vch, 8 bytes at vin; rows 8 and 16 further have the same swizzle)
  const int gi = lane & 15, gg = lane >> 4;
  const int vrow = 4 * (gg >> 1) + (gi >> 2), vch = 2 * (gg & 1) + ((gi & 3) >> 1), vin = 8 * (gi & 1);
  uint32_t vaddr[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
    vaddr[mb] = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)buf + ABLK + vrow * HDIM * 2 +
                ((4 * mb + vch) ^ (vrow & 7)) * 16 + vin;

  // the two heads' 32 query rows come by DMA too, into the split-0 buffer that the second step fills (read
  // in operand order from memory, 16 rows an instruction, they kept the address unit busy for 1.9 us), head
  // h's into block h; then every wave takes its own, the B operand: query c, dims 16 kk + 8 hf ..
  char* const qbuf = smem + 2 * ABLK;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int row = 8 * ks + 4 * r + (lane >> 4);
    const bf16_t* src = qrows + (size_t)min(32 * qb + row, S - 1) * (NQH * HDIM) + hq * HDIM + ((lane & 15) ^ (row & 7)) * 8;
    __builtin_amdgcn_global_load_lds((gvoid_t*)src, (lvoid_t*)(qbuf + hd * ABLK + (8 * ks + 4 * r) * HDIM * 2), 16, 0, 0);
  }
  issue(0, ks);
  wait_vm_lds<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  u32x4 q[8];
#pragma unroll
  for (int kk = 0; kk < 8; ++kk)
    q[kk] = *reinterpret_cast<const u32x4*>(qbuf + hd * ABLK + c * HDIM * 2 + ((2 * kk + hf) ^ (c & 7)) * 16);
#pragma unroll 1
  for (int t = 0; t < nst; ++t) {
    const int kb = ks + AKS * t, b = t & 1;
    wait_vm_lds<0>();                 // this wave's copies have landed, its reads of the other buffer are done
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");    // no LDS access moves across
    issue(b ^ 1, kb + AKS);           // (past the end: the last block again, which nothing reads)
    if (kb >= nkb) continue;
    const char* K = buf + b * 2 * ABLK;
    u32x4 kf[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
      kf[kk] = *reinterpret_cast<const u32x4*>(K + c * HDIM * 2 + ((2 * kk + hf) ^ (c & 7)) * 16);
    f32x16 acc, acc2;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = acc2[r] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 8; kk += 2) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(kf[kk]), as_bf8(q[kk]), acc, 0, 0, 0);
      acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(kf[kk + 1]), as_bf8(q[kk + 1]), acc2, 0, 0, 0);
    }
    float sc[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = acc[r] + acc2[r];
    // blocks that every query of the block sees whole (the wave-uniform common case) skip the mask
    if (!(32 * kb + 31 <= p0 + 32 * qb && 32 * qb + 31 < S)) {
      const int lim = qok ? p0 + i : -1;   // last key this lane's query sees (none past the prompt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * kb + 8 * (r >> 2) + 4 * hf + (r & 3) > lim) sc[r] = -INFINITY;
    }
    // running max; a fully masked row so far keeps m = -inf and adds nothing. It moves only when some
    // query's block max passes it by more than a factor 2^8 of the weights (p <= 256 keeps its relative
    // rounding, and the sums are f32), so that most steps do not rescale O^T
    // (v_max3 by name: fmaxf first quiets each operand)
    float bm = sc[0];
    auto max3 = [](float x, float y, float z) QTTS_PF_INLINE {
      float r;
      asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
      return r;
    };
    {
      const float x0 = max3(sc[0], sc[1], sc[2]), x1 = max3(sc[3], sc[4], sc[5]), x2 = max3(sc[6], sc[7], sc[8]);
      const float x3 = max3(sc[9], sc[10], sc[11]), x4 = max3(sc[12], sc[13], sc[14]);
      bm = max3(max3(x0, x1, sc[15]), x2, max3(x3, x4, x4));
    }
    bm = fmaxf(bm, __uint_as_float(xlane<5>(__float_as_uint(bm))));
    if (__builtin_amdgcn_ballot_w64(bm > m + 8.0f / SL) != 0ull) {
      const float mn = fmaxf(m, bm);
      const float al = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * SL);
      l *= al;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[mb][r] *= al;
      m = mn;
    }
    const float nm = m == -INFINITY ? 0.0f : -m * SL;
    float e[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) e[r] = ex(sc[r], nm);
    l += (((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]))) +
         (((e[8] + e[9]) + (e[10] + e[11])) + ((e[12] + e[13]) + (e[14] + e[15])));
    uint32_t va[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) va[mb] = vaddr[mb] + b * 2 * ABLK;
    auto pv = [&](auto kk_) QTTS_PF_INLINE {
      constexpr int kk2 = decltype(kk_)::value;
      u32x4 pb;
#pragma unroll
      for (int j = 0; j < 4; ++j) pb[j] = pack_bh(e[8 * kk2 + 2 * j], e[8 * kk2 + 2 * j + 1]);
      u32x2 lo[4], hi[4];
      lds_tr16x8<16 * kk2 * HDIM * 2>(va, lo, hi);
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const u32x4 av = {lo[mb][0], lo[mb][1], hi[mb][0], hi[mb][1]};
        o[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(av), as_bf8(pb), o[mb], 0, 0, 0);
      }
    };
    pv(std::integral_constant<int, 0>{});
    pv(std::integral_constant<int, 1>{});
  }
  l += __uint_as_float(xlane<5>(__float_as_uint(l)));

  // merge the splits: M = max m_s, L = sum l_s e^(m_s - M), O = sum O_s e^(m_s - M) (split order)
  float* sml = reinterpret_cast<float*>(smem + AKS * 4 * ABLK) + hd * AKS * 2 * 32;   // [split][2][32]
  if (hf == 0) {
    sml[(ks * 2) * 32 + c] = m;
    sml[(ks * 2 + 1) * 32 + c] = l;
  }
  wait_vm_lds<0>();
  __syncthreads();   // every buffer is dead
  float M = -INFINITY;
#pragma unroll
  for (int v = 0; v < AKS; ++v) M = fmaxf(M, sml[(v * 2) * 32 + c]);
  float L = 0.0f;
#pragma unroll
  for (int v = 0; v < AKS; ++v) {
    const float mv = sml[(v * 2) * 32 + c];
    L += mv == -INFINITY ? 0.0f : sml[(v * 2 + 1) * 32 + c] * __builtin_amdgcn_exp2f((mv - M) * SL);
  }
  const float sw = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - M) * SL);
  // [head][split][dim block][register quad][lane][4]: every wave leaves its sums of all 128 dims
  float* ob = reinterpret_cast<float*>(smem) + hd * AKS * 64 * 64;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = o[mb][4 * r + e] * sw;
      *reinterpret_cast<f32x4*>(ob + ((ks * 4 + mb) * 4 + r) * 256 + lane * 4) = x;
    }
  __syncthreads();
  if (!qok) return;
  const float rl = L > 0.0f ? 1.0f / L : 0.0f;
  // O^T layout: column = query c, register r of block mb = dim 32 mb + 8 (r >> 2) + 4 hf + (r & 3)
  bf16_t* orow = att + (size_t)i * (NQH * HDIM) + hq * HDIM + 32 * ks + 4 * hf;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    f32x4 x = *reinterpret_cast<const f32x4*>(ob + (ks * 4 + r) * 256 + lane * 4);
#pragma unroll
    for (int v = 1; v < AKS; ++v) x += *reinterpret_cast<const f32x4*>(ob + ((v * 4 + ks) * 4 + r) * 256 + lane * 4);
    u32x2 pk;
    pk[0] = pack_bh(x[0] * rl, x[1] * rl);
    pk[1] = pack_bh(x[2] * rl, x[3] * rl);
    *reinterpret_cast<u32x2*>(orow + 8 * r) = pk;
  }
}

// Layer projection C = A W^T of a TM x TN tile (tokens x weight rows), the whole K range in one
// workgroup, with everything that follows it up to the next matrix product in its epilogue, so that a
// layer is five launches at every prompt length (QKV, attention, O, gate/up, down):
//   QKV   rstd, q/k RMSNorm, interleaved mRoPE, K/V cache write (a tile is one head, TN = 128)
//   GU    rstd, SwiGLU (gate and up rows interleaved by 16)
//   O, D  residual add, x * gain of the next norm, and the sum of squares that this norm needs
// RMSNorm is applied around the product: xn = x gain rstd, and rstd is one number per token, so the
// producer writes bf16(x * gain) with the tile's part of sum(x^2), and the consumer scales its f32 sums by
// rstd (one bf16 rounding where transformers' form, bf16(gain * bf16(x rstd)), has two). What this removes:
// split-K partials (f32, written and read back), their reductions and the norms, three launches of 4 to
// 8 us a layer, each with a launch gap and a memory round trip.
//
// Operands are copied global -> LDS by DMA (global_load_lds_dwordx4: each wave instruction writes 64 x 16
// bytes at a wave-uniform LDS address) through NS stages of BK, NS - 1 of them in flight, one barrier a
// stage. LDS tile: row r of a stage holds its BK / 8 chunks of 16 bytes with chunk c at position
// c ^ (r & 7): a DMA instruction reads whole 128- or 256-byte row segments (adjacent lanes on one row: the
// address unit takes 4 times as long for the MFMA operand order, rows first), and the MFMA operand reads (16
// rows at one chunk) are conflict-free. Weights are the MFMA's A operand, so a lane ends with 4 consecutive
// columns of one token: lane l, register e of block (nb, mb) = weight row 16 nb + 4 (l >> 4) + e, token
// 16 mb + (l & 15). Rows past M read row M - 1; their sums are never stored.
enum Mode { P_QKV, P_O, P_GU, P_DOWN };
constexpr int kdim(int mode) { return mode == P_O ? NQH * HDIM : (mode == P_DOWN ? INTER : HID); }
constexpr int ndim(int mode) { return mode == P_QKV ? 4096 : (mode == P_GU ? 2 * INTER : HID); }
constexpr int QW = NQH * HDIM;               // a token's rotated queries
constexpr int SQP = 32;                      // sum-of-squares parts per token (one per column tile)

struct TileArgs {
  const bf16_t* A;                 // [M, K] activations
  const TTSLayerWeights* layers;   // device table
  int layer;
  int M;
  int xm, xn;                      // the XCDs as a grid over the tiles: xm x xn = 8
  const float* ssq;                // QKV, GU: [M][SQP] parts of each token's sum(x^2), nsq of them valid
  int nsq;
  bf16_t* out;                     // QKV: q [M, QW]; GU: [M, INTER]
  bf16_t* h;                       // O, down: residual stream, updated in place
  bf16_t* xg;                      // ... bf16(h * gain), gain = field nfield of layer nlayer (nlayer < 0: none)
  float* ssq_out;
  int nlayer, nfield;
  const bf16_t* cos_t;             // QKV: tables, (t, h, w) rows [3][M] or nullptr (row = p0 + token), cache
  const bf16_t* sin_t;
  const int* pos3;
  int p0;
  bf16_t* kc;
  bf16_t* vc;
  int max_seq;
};

// weight row of column n of tile tn (GU: 16 gate rows, then the 16 up rows of the same outputs; FINE, for
// waves of an odd number of 16-column blocks: 2 gate rows, then the 2 up rows)
template <int MODE, int TN, bool FINE>
__device__ __forceinline__ const bf16_t* tile_weight_row(const TTSLayerWeights* lw, int tn, int n) {
  constexpr int K = kdim(MODE);
  const int c = tn * TN + n;
  if constexpr (MODE == P_QKV) {
    return c < 2048 ? tbl(lw, 1) + (size_t)c * K
                    : (c < 3072 ? tbl(lw, 2) + (size_t)(c - 2048) * K : tbl(lw, 3) + (size_t)(c - 3072) * K);
  } else if constexpr (MODE == P_O) {
    return tbl(lw, 6) + (size_t)c * K;
  } else if constexpr (MODE == P_GU) {
    const int row = (TN / 2) * tn + (FINE ? 2 * (n >> 2) + (n & 1) : 16 * (n >> 5) + (n & 15));
    return ((n >> (FINE ? 1 : 4)) & 1 ? tbl(lw, 9) : tbl(lw, 8)) + (size_t)row * K;
  } else {
    return tbl(lw, 10) + (size_t)c * K;
  }
}

// q/k RMSNorm and interleaved mRoPE of a tile's head: TM token rows (bf16 rows of pitch tr in LDS, the first
// one token m0), 8 threads of 8 channel pairs (d, d + 64) a row, to rows of stride ld at dst. The table rows
// of the next row go out before this one's arithmetic.
template <int TM, int NT>
__device__ __forceinline__ void head_finish(const TileArgs& g, const bf16_t* T, int tr, int m0, int t, const bf16_t* gn,
                                            bf16_t* dst, int ld) {
  constexpr int RP = NT / 8, NP = (TM + RP - 1) / RP;   // rows a pass, passes
  const int d0 = 8 * (t & 7);
  const u32x4 g0 = ldw(gn + d0), g1 = ldw(gn + d0 + 64);
  auto unpack8 = [](const u32x4& v, float (&f)[8]) QTTS_PF_INLINE {
#pragma unroll
    for (int e = 0; e < 4; ++e) { f[2 * e] = bflo(v[e]); f[2 * e + 1] = bfhi(v[e]); }
  };
  struct Cs { u32x4 c0, c1, s0, s1; };
  auto load = [&](int row) QTTS_PF_INLINE {
    const int m = min(m0 + min(row, TM - 1), g.M - 1);
    Cs r;
    if (g.pos3 == nullptr) {
      const size_t ro = (size_t)(g.p0 + m) * HDIM + d0;
      r = {ldw(g.cos_t + ro), ldw(g.cos_t + ro + 64), ldw(g.sin_t + ro), ldw(g.sin_t + ro + 64)};
    } else {
      // table rows of the three sections (t, h, w); channel d < 60 takes h when d % 3 == 1 and w when
      // d % 3 == 2, every other channel t (the same row for d and d + 64); clamped into the table
      Cs v[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const size_t ro = (size_t)min(max(g.pos3[j * g.M + m], 0), g.max_seq - 1) * HDIM + d0;
        v[j] = {ldw(g.cos_t + ro), ldw(g.cos_t + ro + 64), ldw(g.sin_t + ro), ldw(g.sin_t + ro + 64)};
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        auto sec = [&](int k) QTTS_PF_INLINE { const int d = d0 + k; return d < 60 ? d % 3 : 0; };
        const int a = sec(2 * e), b = sec(2 * e + 1);
        auto pick = [&](uint32_t x, uint32_t y, uint32_t z) QTTS_PF_INLINE {
          const uint32_t lo = a == 0 ? x : (a == 1 ? y : z), hi = b == 0 ? x : (b == 1 ? y : z);
          return (lo & 0xffffu) | (hi & 0xffff0000u);
        };
        r.c0[e] = pick(v[0].c0[e], v[1].c0[e], v[2].c0[e]);
        r.c1[e] = pick(v[0].c1[e], v[1].c1[e], v[2].c1[e]);
        r.s0[e] = pick(v[0].s0[e], v[1].s0[e], v[2].s0[e]);
        r.s1[e] = pick(v[0].s1[e], v[1].s1[e], v[2].s1[e]);
      }
    }
    return r;
  };
  Cs cs[2];
  cs[0] = load(t >> 3);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int row = (t >> 3) + RP * p;
    if (p + 1 < NP) cs[(p + 1) & 1] = load(row + RP);
    if (TM < RP && row >= TM) break;
    const u32x4 xa = *reinterpret_cast<const u32x4*>(T + row * tr + d0);
    const u32x4 xb = *reinterpret_cast<const u32x4*>(T + row * tr + d0 + 64);
    float x0[8], x1[8], c0[8], c1[8], s0[8], s1[8], ga[8], gb[8];
    unpack8(xa, x0); unpack8(xb, x1);
    const Cs& c = cs[p & 1];
    unpack8(c.c0, c0); unpack8(c.c1, c1); unpack8(c.s0, s0); unpack8(c.s1, s1); unpack8(g0, ga); unpack8(g1, gb);
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) ss += x0[k] * x0[k] + x1[k] * x1[k];
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) ss += __shfl_xor(ss, o, 64);
    const float rs = 1.0f / sqrtf(ss / (float)HDIM + EPS);
    float r0[8], r1[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float y0 = rbh(ga[k] * rbh(x0[k] * rs)), y1 = rbh(gb[k] * rbh(x1[k] * rs));
      r0[k] = rbh(y0 * c0[k]) + rbh(-y1 * s0[k]);
      r1[k] = rbh(y1 * c1[k]) + rbh(y0 * s1[k]);
    }
    u32x4 o0, o1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o0[e] = pack_bh(r0[2 * e], r0[2 * e + 1]);
      o1[e] = pack_bh(r1[2 * e], r1[2 * e + 1]);
    }
    if (m0 + row < g.M) {
      *reinterpret_cast<u32x4*>(dst + (size_t)row * ld + d0) = o0;
      *reinterpret_cast<u32x4*>(dst + (size_t)row * ld + d0 + 64) = o1;
    }
  }
}

template <int MODE, int TM, int TN, int NWM, int NWN, int NWK, int NS, int BK>
__global__ void __launch_bounds__(64 * NWM * NWN * NWK, 2) tile_gemm_kernel(const TileArgs g) {
  constexpr int K = kdim(MODE), NW = NWM * NWN * NWK, NT = 64 * NW, NK = K / BK;
  constexpr int KK = BK / 32 / NWK;                         // a wave's MFMA steps per stage
  constexpr int CPR = BK / 8, RPI = 64 / CPR;               // 16-byte chunks per row, rows per DMA instruction
  constexpr int NIW = (TM + TN) / RPI / NW;                 // DMA instructions per wave and stage
  constexpr int STAGE = (TM + TN) * BK * 2;
  constexpr int MB = TM / NWM / 16, NB = TN / NWN / 16;     // a wave's 16 x 16 blocks
  constexpr bool NORMED = MODE == P_QKV || MODE == P_GU;
  constexpr int TR = HDIM + 8;                              // QKV: bf16 row of the staged head tile
  static_assert((TM + TN) % (RPI * NW) == 0 && TM % RPI == 0 && K % BK == 0 && NK >= NS - 1, "stages");
  static_assert(KK >= 2 && KK % 2 == 0 && NWK * NWM * NWN == NW, "operand double buffer");
  static_assert(NWK == 1 || (NWK - 1) * TM * TN * 4 <= NS * STAGE, "K parts of the sums");
  static_assert(MODE != P_QKV || (TN == HDIM && TM * TR * 2 <= NS * STAGE), "QKV: one head per tile");
  constexpr bool FINE = MODE == P_GU && (TN / NWN) % 32 != 0;   // gate/up interleave (tile_weight_row)
  static_assert(ndim(MODE) % TN == 0 && (MODE == P_QKV || MODE == P_GU || ndim(MODE) / TN <= SQP), "column tiles");
  // one LDS object: with several, the compiler tracks which of them a DMA may write and waits for every
  // DMA in flight before each LDS read
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE + (NORMED ? 1 : NWN) * TM * 4];
  float* rstd = reinterpret_cast<float*>(lds + NS * STAGE);   // NORMED
  float* sred = rstd;                                         // O, down: the waves' sums of squares
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = w % NWM, wn = w / NWM % NWN, wk = w / (NWM * NWN);
  // XCD-aware tile order: workgroups reach the XCDs round-robin by linear id; XCD x takes the sub-grid
  // (x % xm, x / xm) of the tiles, row tiles first
  const int tm_n = (g.M + TM - 1) / TM, x = blockIdx.x & 7, r0 = blockIdx.x >> 3;
  const int mx = tm_n / g.xm, nx = ndim(MODE) / TN / g.xn;
  const int tm = (x % g.xm) * mx + r0 % mx, tn = (x / g.xm) * nx + r0 / mx;
  const int m0 = tm * TM, n0 = tn * TN;
  const TTSLayerWeights* lw = g.layers + g.layer;

  // loads that the epilogue needs go out ahead of the DMA: the row's sum-of-squares parts, or the residual
  // and the next norm's gain
  const int lm = 16 * MB * wm + (lane & 15), ln = 16 * NB * wn + 4 * (lane >> 4);   // this lane's first token, column
  float sq[NORMED ? (TM + NT - 1) / NT : 1];
  u32x2 hr[NORMED ? 1 : MB][NORMED ? 1 : NB], gw[NORMED ? 1 : NB];
  if constexpr (NORMED) {
#pragma unroll
    for (int i = 0; i < (TM + NT - 1) / NT; ++i) {
      const int m = min(m0 + t + NT * i, g.M - 1);
      float s = 0.0f;
      const u32x4* p = reinterpret_cast<const u32x4*>(g.ssq + (size_t)m * SQP);
#pragma unroll
      for (int q = 0; q < SQP / 4; ++q) {
        const u32x4 v = p[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) s += 4 * q + e < g.nsq ? __uint_as_float(v[e]) : 0.0f;
      }
      sq[i] = s;
    }
  } else {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        hr[mb][nb] = *reinterpret_cast<const u32x2*>(g.h + (size_t)min(m0 + lm + 16 * mb, g.M - 1) * HID + n0 + ln + 16 * nb);
    const bf16_t* gp = tbl(g.layers + max(g.nlayer, 0), g.nfield);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) gw[nb] = *reinterpret_cast<const u32x2*>(gp + n0 + ln + 16 * nb);
  }

  // this lane's source of DMA instruction i: stage row RPI (NIW w + i) + lane / CPR (token rows, then
  // weight rows), the chunk that belongs at position lane % CPR
  const bf16_t* src[NIW];
#pragma unroll
  for (int i = 0; i < NIW; ++i) {
    const int r = RPI * (NIW * w + i) + lane / CPR, c = (lane % CPR) ^ (r & 7);
    const bf16_t* p = r < TM ? g.A + (size_t)min(m0 + r, g.M - 1) * K : tile_weight_row<MODE, TN, FINE>(lw, tn, r - TM);
    src[i] = p + 8 * c;
  }
  auto issue = [&](int s, int kt) QTTS_PF_INLINE {   // stage s <- K step kt (clamped: past the end the last one again)
    const int k = BK * min(kt, NK - 1);
    char* base = lds + s * STAGE + 1024 * NIW * w;
#pragma unroll
    for (int i = 0; i < NIW; ++i)
      __builtin_amdgcn_global_load_lds((gvoid_t*)(src[i] + k), (lvoid_t*)(base + 1024 * i), 16, 0, 0);
  };
  f32x4 acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // MFMA operands of step i of stage s: (stage row r, chunk c) at byte r BK 2 + 16 (c ^ (r & 7)); r & 7 is
  // the lane's alone (block rows are multiples of 16)
  bf16x8 av[2][MB], bv[2][NB];
  auto read = [&](int s, int i, bf16x8 (&x)[MB], bf16x8 (&y)[NB]) QTTS_PF_INLINE {
    const int co = ((4 * (i * NWK + wk) + (lane >> 4)) ^ (lane & 7)) * 16;
    const char* a = lds + s * STAGE + (16 * MB * wm + (lane & 15)) * BK * 2 + co;
    const char* b = lds + s * STAGE + (TM + 16 * NB * wn + (lane & 15)) * BK * 2 + co;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) y[nb] = as_bf8(*reinterpret_cast<const u32x4*>(b + nb * 16 * BK * 2));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) x[mb] = as_bf8(*reinterpret_cast<const u32x4*>(a + mb * 16 * BK * 2));
  };
  auto mfma = [&](const bf16x8 (&x)[MB], const bf16x8 (&y)[NB]) QTTS_PF_INLINE {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        acc[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y[nb], x[mb], acc[nb][mb], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s, s);
  if constexpr (NORMED) {
#pragma unroll
    for (int i = 0; i < (TM + NT - 1) / NT; ++i)
      if (t + NT * i < TM) rstd[t + NT * i] = 1.0f / sqrtf(sq[i] / (float)HID + EPS);
  }
  // The operands of each step are read one step ahead, those of a stage's first step before the last MFMAs
  // of the stage before it, so that the LDS reads run under the MFMAs.
  // Next stage kt: this wave's DMA has landed and its reads of the stage before are done; then every
  // wave's, and the buffer of the stage before is free for stage kt + NS - 1.
  auto next = [&](int kt, int free_buf) QTTS_PF_INLINE {
    wait_vm_lds<(NS - 2) * NIW>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");   // no LDS access moves across
    issue(free_buf, kt + NS - 1);
  };
  next(0, NS - 1);
  read(0, 0, av[0], bv[0]);
  int st = 0;
#pragma unroll 1
  for (int kt = 0; kt < NK; ++kt) {
    const int sn = st + 1 == NS ? 0 : st + 1;
#pragma unroll
    for (int i = 0; i < KK; ++i) {
      if (i + 1 < KK) {
        read(st, i + 1, av[(i + 1) & 1], bv[(i + 1) & 1]);
      } else {
        next(kt + 1, st);            // (past the last stage: clamped copies that nothing uses)
        read(sn, 0, av[0], bv[0]);
      }
      mfma(av[i & 1], bv[i & 1]);
    }
    st = sn;
  }
  wait_vm_lds<0>();                  // no DMA may still target LDS when it is used again or given back
  __syncthreads();
  if constexpr (NWK > 1) {
    // the waves of a tile part add their K parts, in K order
    float* part = reinterpret_cast<float*>(lds);
    constexpr int PW = NWM * NWN * NB * MB * 4 * 64;   // floats of one K part
    const int at = (wm + NWM * wn) * NB * MB * 4 * 64 + lane * 4;
    if (wk > 0) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          *reinterpret_cast<f32x4*>(part + (wk - 1) * PW + at + (nb * MB + mb) * 256) = acc[nb][mb];
    }
    __syncthreads();
    if (wk == 0) {
#pragma unroll
      for (int j = 0; j < NWK - 1; ++j)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) acc[nb][mb] += *reinterpret_cast<const f32x4*>(part + j * PW + at + (nb * MB + mb) * 256);
    }
    if constexpr (MODE == P_QKV) __syncthreads();     // the parts have been read: their LDS takes the head tile
  }

  if constexpr (MODE == P_QKV) {
    bf16_t* T = reinterpret_cast<bf16_t*>(lds);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if (wk > 0) break;
      const float rs = rstd[lm + 16 * mb];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const f32x4 v = acc[nb][mb];
        u32x2 o;
        o[0] = pack_bh(v[0] * rs, v[1] * rs);
        o[1] = pack_bh(v[2] * rs, v[3] * rs);
        *reinterpret_cast<u32x2*>(T + (lm + 16 * mb) * TR + ln + 16 * nb) = o;
      }
    }
    __syncthreads();
    const int head = tn;   // q heads 0..15, k heads 16..23, v heads 24..31
    if (head >= NQH + NKVH) {
      bf16_t* vbase = g.vc + ((size_t)g.layer * NKVH + (head - NQH - NKVH)) * g.max_seq * HDIM;
      for (int q = t; q < TM * 16; q += NT) {
        const int row = q >> 4, ch = 8 * (q & 15), m = m0 + row;
        if (m < g.M)
          *reinterpret_cast<u32x4*>(vbase + (size_t)(g.p0 + m) * HDIM + ch) = *reinterpret_cast<const u32x4*>(T + row * TR + ch);
      }
      return;
    }
    const bool isq = head < NQH;
    const bf16_t* gn = tbl(lw, isq ? 4 : 5);
    head_finish<TM, NT>(g, T, TR, m0, t, gn,
                        isq ? g.out + (size_t)m0 * QW + head * HDIM
                            : g.kc + (((size_t)g.layer * NKVH + (head - NQH)) * g.max_seq + g.p0 + m0) * HDIM,
                        isq ? QW : HDIM);
  } else if constexpr (MODE == P_GU) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = m0 + lm + 16 * mb;
      const float rs = rstd[lm + 16 * mb];
      if (m >= g.M || wk > 0) continue;
      bf16_t* o = g.out + (size_t)m * INTER + n0 / 2 + 8 * NB * wn + 4 * (lane >> 4);
      if constexpr (FINE) {
        // (gate, gate, up, up) of outputs 8 nb + 2 (l >> 4) + {0, 1}
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const f32x4 v = acc[nb][mb];
          const float a0 = rbh(silu_f(rbh(v[0] * rs))) * rbh(v[2] * rs), a1 = rbh(silu_f(rbh(v[1] * rs))) * rbh(v[3] * rs);
          *reinterpret_cast<uint32_t*>(o - 2 * (lane >> 4) + 8 * nb) = pack_bh(a0, a1);
        }
        continue;
      }
#pragma unroll
      for (int p = 0; p < NB / 2; ++p) {
        const f32x4 gs = acc[2 * p][mb], us = acc[2 * p + 1][mb];
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = rbh(silu_f(rbh(gs[e] * rs))) * rbh(us[e] * rs);
        u32x2 v;
        v[0] = pack_bh(a[0], a[1]);
        v[1] = pack_bh(a[2], a[3]);
        *reinterpret_cast<u32x2*>(o + 16 * p) = v;
      }
    }
  } else {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if (wk > 0) break;
      const int m = m0 + lm + 16 * mb;
      float ss = 0.0f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const f32x4 v = acc[nb][mb];
        const u32x2 r = hr[mb][nb];
        const float a0 = rbh(bflo(r[0]) + rbh(v[0])), a1 = rbh(bfhi(r[0]) + rbh(v[1]));
        const float a2 = rbh(bflo(r[1]) + rbh(v[2])), a3 = rbh(bfhi(r[1]) + rbh(v[3]));
        ss += (a0 * a0 + a1 * a1) + (a2 * a2 + a3 * a3);
        if (m < g.M) {
          const size_t at = (size_t)m * HID + n0 + ln + 16 * nb;
          u32x2 o;
          o[0] = pack_bh(a0, a1);
          o[1] = pack_bh(a2, a3);
          *reinterpret_cast<u32x2*>(g.h + at) = o;
          if (g.nlayer >= 0) {
            u32x2 y;
            y[0] = pack_bh(a0 * bflo(gw[nb][0]), a1 * bfhi(gw[nb][0]));
            y[1] = pack_bh(a2 * bflo(gw[nb][1]), a3 * bfhi(gw[nb][1]));
            *reinterpret_cast<u32x2*>(g.xg + at) = y;
          }
        }
      }
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      if (lane < 16) sred[wn * TM + lm + 16 * mb] = ss;
    }
    __syncthreads();
    for (int q = t; q < TM; q += NT) {
      float s = sred[q];
#pragma unroll
      for (int j = 1; j < NWN; ++j) s += sred[j * TM + q];
      if (m0 + q < g.M) g.ssq_out[(size_t)(m0 + q) * SQP + tn] = s;
    }
  }
}

// The prompt embeddings into the residual stream, with bf16(x * gain) and sum(x^2) of layer 0's input
// norm; one wave per token.
__global__ void __launch_bounds__(256) embed_kernel(const bf16_t* x, const TTSLayerWeights* layers, bf16_t* h, bf16_t* xg,
                                                    float* ssq, int M) {
  const int lane = threadIdx.x & 63, m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  const bf16_t* w = tbl(layers, 0);
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int e0 = 8 * (lane + 64 * k);
    const u32x4 v = ldw(x + (size_t)m * HID + e0), gw = ldw(w + e0);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = bflo(v[e]), b = bfhi(v[e]);
      ss += a * a + b * b;
      o[e] = pack_bh(a * bflo(gw[e]), b * bfhi(gw[e]));
    }
    *reinterpret_cast<u32x4*>(h + (size_t)m * HID + e0) = v;
    *reinterpret_cast<u32x4*>(xg + (size_t)m * HID + e0) = o;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
  if (lane == 0) ssq[(size_t)m * SQP] = ss;
}

// First group-0 token from bf16 logits: ids [n-1024, n) except EOS suppressed when mask_tail
// (generator.py:71-75, :116), EOS suppressed when suppress_eos (min_new_tokens, :117-119), then
// the decode kernels' selection (greedy argmax, or temperature / top-k / top-p / Gumbel-max).
__global__ void __launch_bounds__(64) select_kernel(const bf16_t* logits, int n, int mask_tail, int eos_id,
                                                    int suppress_eos, SelParams sp, float* out_logits,
                                                    int* out_token) {
  __shared__ SelScratch sc;
  const int lane = threadIdx.x;
  // every logit load is issued before the first is used (a rolled loop waited for each in turn);
  // loads past n are clamped to n - 1 and dropped
  bf16_t lv[SEL_NJ];
#pragma unroll
  for (int j = 0; j < SEL_NJ; ++j) lv[j] = *gmem(logits + min(lane + 64 * j, n - 1));
  uint32_t w[SEL_NJ], best = 0u;
#pragma unroll
  for (int j = 0; j < SEL_NJ; ++j) {
    const int i = lane + 64 * j;
    float v = bf2f(lv[j]);
    if (out_logits && i < n) out_logits[i] = v;
    if ((mask_tail && i >= n - 1024 && i != eos_id) || (suppress_eos && i == eos_id)) v = -INFINITY;
    w[j] = i < n ? (bfkey(v) << 16) | (uint32_t)i : 0u;
    best = max(best, i < n ? greedy_word(v, i) : 0u);
  }
  const int tok = sp.do_sample ? wave_sample(w, n, sp, &sc) : greedy_id(best, n);
  if (lane == 0) *out_token = tok;
}

// ---- host ----------------------------------------------------------------------------------

// One launch of a projection: tile TM x TN (NWM x NWN waves), NS stages of BK.
template <int MODE, int TM, int TN, int NWM, int NWN, int NWK, int NS, int BK>
void launch_tile(TileArgs& g, hipStream_t st) {
  const int tm = (g.M + TM - 1) / TM, tn = ndim(MODE) / TN;
  // the XCD grid xm x xn that re-reads least: every XCD column reads the activations, every XCD row the weights
  g.xm = 1;
  double best = 1e30;
  for (int xm = 1; xm <= 8; xm *= 2) {
    if (tm % xm != 0 || tn % (8 / xm) != 0) continue;
    const double cost = (double)g.M * (8 / xm) + (double)ndim(MODE) * xm;
    if (cost < best) { best = cost; g.xm = xm; }
  }
  g.xn = 8 / g.xm;
  static_assert(ndim(MODE) / TN % 8 == 0, "column tiles over the XCDs");
  hipLaunchKernelGGL((tile_gemm_kernel<MODE, TM, TN, NWM, NWN, NWK, NS, BK>), dim3(tm * tn), dim3(64 * NWM * NWN * NWK), 0, st, g);
}

// Tiles by prompt length M. A projection's time is its workgroups' K loop (operand bytes per CU through
// LDS) plus about 4 us of launch, first loads and epilogue, so the tile grows with M as slowly as one round of at
// most 256 workgroups, one a CU, allows: it doubles at 256, 512 and 1024 tokens, where a grid is whole, and just
// past them 144 to 192 workgroups run; up to 32 tokens QKV, O and down have 32, gate/up 96 or 192. Measured over
// prompts of 13 to 2048 tokens, without reads ahead (us a layer, against the best alternative):
//   QKV (a head's 128 columns)  32 tokens up to 256, 64 to 512, 128 to 1024, then 256; a step too small
//                               or too large costs 2 to 10 us
//   GU    16 x 64 up to 32 tokens (at 13: 1.2 us less than 32 x 96), 32 x 96 to 128, 64 x 96 to 256 (32 x 96:
//         +1.8 to 2.1), 64 x 192 to 512 (64 x 96: +1.4 to 2.1), 128 x 192 to 1024, then 256 x 192 (at 1500:
//         3.9 less)
//   O, D  16 x 32 up to 128, 32 x 32 to 256 (+2 to 3 either way), 32 x 64 to 512, 64 x 64 to 1024, then
//         128 x 64; two or four waves share a block's K range where one wave's chain of MFMAs and LDS reads
//         is what a stage waits for (0.7 to 2 us less each)
// Past 2048 tokens those tiles no longer fit the CUs at once, and the last 32 of 288 workgroups take as long as
// the first 256. Tiles of four waves and at most 80 KB of LDS, two workgroups a CU, leave less of a last round
// (us, large tile : these):
//   QKV   128 x 128 to 4096: 2049 tokens 44.3 : 41.7, 2560 49.5 : 43.9, 3073 54.8 : 53.4, 4096 60.1 : 58.3
//         (6000 81.2 : 86.1)
//   GU    128 x 128 to 2688 (two rounds of 512): 2049 46.4 : 41.3, 2560 55.0 : 46.3 (3072 56.5 : 58.9)
//   O, D  128 x 64, no K shares: O 2049 33.2 : 24.6, 3072 36.8 : 32.0, 6000 74.6 : 65.3; down 43.6 : 35.4,
//         49.6 : 43.8, 100.4 : 92.1
void project_qkv(TileArgs& g, hipStream_t st) {
  if (g.M <= 256) launch_tile<P_QKV, 32, 128, 1, 4, 1, 6, 64>(g, st);
  else if (g.M <= 512) launch_tile<P_QKV, 64, 128, 2, 2, 1, 5, 64>(g, st);
  else if (g.M <= 1024) launch_tile<P_QKV, 128, 128, 4, 2, 1, 4, 64>(g, st);
  else if (g.M > 2048 && g.M <= 4096) launch_tile<P_QKV, 128, 128, 2, 2, 1, 2, 64>(g, st);
  else launch_tile<P_QKV, 256, 128, 4, 2, 1, 3, 64>(g, st);
}
void project_gate_up(TileArgs& g, hipStream_t st) {
  if (g.M <= 32) launch_tile<P_GU, 16, 64, 1, 4, 1, 4, 128>(g, st);
  else if (g.M <= 128) launch_tile<P_GU, 32, 96, 2, 2, 1, 4, 64>(g, st);
  else if (g.M <= 256) launch_tile<P_GU, 64, 96, 2, 2, 1, 3, 64>(g, st);
  else if (g.M <= 512) launch_tile<P_GU, 64, 192, 2, 2, 1, 4, 64>(g, st);
  else if (g.M <= 1024) launch_tile<P_GU, 128, 192, 4, 2, 1, 3, 64>(g, st);
  else if (g.M > 2048 && g.M <= 2688) launch_tile<P_GU, 128, 128, 2, 2, 1, 2, 64>(g, st);
  else launch_tile<P_GU, 256, 192, 4, 2, 1, 2, 64>(g, st);
}
// O or down: also leaves in g.nsq how many sum-of-squares parts it wrote per token
template <int MODE>
void project_residual(TileArgs& g, hipStream_t st) {
  g.nsq = g.M <= 256 ? HID / 32 : HID / 64;
  if (g.M <= 128) launch_tile<MODE, 16, 32, 1, 2, 4, 5, 256>(g, st);
  else if (g.M <= 256) launch_tile<MODE, 32, 32, 2, 2, 2, 6, 128>(g, st);
  else if (g.M <= 512) launch_tile<MODE, 32, 64, 2, 2, 2, 5, 128>(g, st);
  else if (g.M <= 1024) launch_tile<MODE, 64, 64, 2, 2, 2, 4, 128>(g, st);
  else if (g.M <= 2048) launch_tile<MODE, 128, 64, 2, 2, 2, 3, 128>(g, st);
  else launch_tile<MODE, 128, 64, 2, 2, 1, 3, 64>(g, st);
}


size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct Layout {
  size_t h, xg, ssq, q, att, act, logits, total;
};

Layout layout(int S, int vocab) {
  Layout L;
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o = align256(o + bytes); return at; };
  L.h = take((size_t)S * HID * 2);
  L.xg = take((size_t)S * HID * 2);
  L.ssq = take((size_t)S * SQP * 4);
  L.q = take((size_t)S * QW * 2);
  L.att = take((size_t)S * QW * 2);
  L.act = take((size_t)S * INTER * 2);
  L.logits = take((size_t)(vocab > 0 ? vocab : MAXV) * 2);
  L.total = o;
  return L;
}

}  // namespace pf
}  // namespace qtts

using namespace qtts;
using namespace qtts::pf;

extern "C" {

size_t qtts_prefill_workspace_bytes(int n_tokens, int vocab) {
  if (n_tokens < 1 || vocab < 0 || vocab > MAXV) return 0;
  return layout(n_tokens, vocab).total;
}

hipError_t qtts_backbone_prefill(void* workspace, size_t workspace_bytes, const TTSLayerWeights* layer_weights,
                                 int num_layers, const void* final_norm_weight, const void* cos_table,
                                 const void* sin_table, void* k_cache, void* v_cache, int max_seq_len, int position,
                                 int n_tokens, const int* pos3, const void* input_embeddings, float* out_hidden,
                                 const void* codec_head, int vocab, float* out_logits, int* out_token, int mask_tail,
                                 int eos_id, int suppress_eos, const QttsSampling* sampling, int frame_step,
                                 hipStream_t stream) {
  const int S = n_tokens;
  if (workspace == nullptr || layer_weights == nullptr || final_norm_weight == nullptr || cos_table == nullptr ||
      sin_table == nullptr || k_cache == nullptr || v_cache == nullptr || input_embeddings == nullptr)
    return hipErrorInvalidValue;
  if (num_layers < 1 || S < 1 || position < 0 || max_seq_len < 1 || position + S > max_seq_len)
    return hipErrorInvalidValue;
  if (codec_head != nullptr && (vocab < 128 || vocab > MAXV || vocab % 128 != 0 || out_token == nullptr))
    return hipErrorInvalidValue;
  if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0 || (reinterpret_cast<uintptr_t>(input_embeddings) & 15u) != 0)
    return hipErrorInvalidValue;
  const Layout L = layout(S, codec_head ? vocab : 0);
  if (workspace_bytes < L.total) return hipErrorInvalidValue;
  char* ws = static_cast<char*>(workspace);
  bf16_t* h = reinterpret_cast<bf16_t*>(ws + L.h);
  bf16_t* xg = reinterpret_cast<bf16_t*>(ws + L.xg);
  float* ssq = reinterpret_cast<float*>(ws + L.ssq);
  bf16_t* q = reinterpret_cast<bf16_t*>(ws + L.q);
  bf16_t* att = reinterpret_cast<bf16_t*>(ws + L.att);
  bf16_t* act = reinterpret_cast<bf16_t*>(ws + L.act);
  auto* kc = static_cast<bf16_t*>(k_cache);
  auto* vc = static_cast<bf16_t*>(v_cache);
  const auto* cs = static_cast<const bf16_t*>(cos_table);
  const auto* sn = static_cast<const bf16_t*>(sin_table);
  const float scale = 1.0f / sqrtf((float)HDIM);
  const unsigned embed_grid = (unsigned)((S + 3) / 4);
  hipLaunchKernelGGL(embed_kernel, dim3(embed_grid), dim3(256), 0, stream, static_cast<const bf16_t*>(input_embeddings),
                     layer_weights, h, xg, ssq, S);
  TileArgs g{};
  g.layers = layer_weights;
  g.M = S;
  g.ssq = ssq;
  g.ssq_out = ssq;
  g.h = h;
  g.xg = xg;
  g.cos_t = cs;
  g.sin_t = sn;
  g.pos3 = pos3;
  g.p0 = position;
  g.kc = kc;
  g.vc = vc;
  g.max_seq = max_seq_len;
  g.nsq = 1;   // the embeddings' sums of squares are whole
  for (int l = 0; l < num_layers; ++l) {
    g.layer = l;
    g.A = xg; g.out = q;
    project_qkv(g, stream);
    // the two-head kernel for prompts that fill the chip with half the workgroups; below, the per-head kernel
    // and its reads ahead (us a layer, per head against two heads: 640 tokens 69.2 : 75.2, 768 72.0 : 76.9,
    // 1000 79.4 : 81.6, 1280 111.1 : 116.2, 1500 117.0 : 118.4, 2048 141.5 : 137.4, 3000 248.2 : 246.4; with a
    // prefix before the prompt 768 after 1500 90.3 : 95.3, 1000 after 2000 106.8 : 106.4, 1500 after 1500
    // 151.2 : 150.4, 2048 after 1500 181.3 : 170.1)
    if ((S + 31) / 32 * NKVH >= 448)
      hipLaunchKernelGGL(attn_pair_kernel, dim3((S + 31) / 32 * NKVH), dim3(128 * AKS), 0, stream, q, kc, vc, l, max_seq_len,
                         position, S, att, scale);
    else
      hipLaunchKernelGGL(attn_kernel, dim3((S + 31) / 32 * NQH + kPiecesLayer + (l + 1 < num_layers ? kPiecesNext : 0)),
                         dim3(64 * AW), 0, stream, q, kc, vc, l, max_seq_len, position, S, att, scale, layer_weights);
    g.A = att; g.nlayer = l; g.nfield = 7;
    project_residual<P_O>(g, stream);
    g.A = xg; g.out = act;
    project_gate_up(g, stream);
    g.A = act; g.nlayer = l + 1 < num_layers ? l + 1 : -1; g.nfield = 0;
    project_residual<P_DOWN>(g, stream);
  }
  // the last token's final norm -> hidden, and its logits
  bf16_t* lg = reinterpret_cast<bf16_t*>(ws + L.logits);
  const int head_grid = codec_head != nullptr ? (vocab + 4 * RPW - 1) / (4 * RPW) : 1;
  hipLaunchKernelGGL(final_head_kernel, dim3(head_grid), dim3(256), 0, stream, h + (size_t)(S - 1) * HID,
                     static_cast<const bf16_t*>(final_norm_weight), static_cast<const bf16_t*>(codec_head), vocab, out_hidden,
                     lg);
  if (codec_head != nullptr) {
    SelParams sp{};
    sp.do_sample = sampling ? sampling->do_sample : 0;
    sp.temperature = sampling ? sampling->temperature : 1.0f;
    sp.top_k = sampling ? sampling->top_k : 0;
    sp.top_p = sampling ? sampling->top_p : 1.0f;
    sp.seed = sampling ? sampling->seed : 0ull;
    sp.frame_step = frame_step;
    sp.group = 0;
    hipLaunchKernelGGL(select_kernel, dim3(1), dim3(64), 0, stream, lg, vocab, mask_tail, eos_id, suppress_eos, sp,
                       out_logits, out_token);
  }
  return hipGetLastError();
}

}  // extern "C"
