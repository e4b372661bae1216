// Flash attention (fp16 in/out, fp32 softmax and accumulation, head_dim 64,
// no mask) for VGGT's frame and global attention on gfx950.
//
// Sequences: B sequences of L tokens each (frame attention: B = frames,
// L = 1374; global attention: B = 1, L = frames * 1374).  q/k/v/out are
// token-major with arbitrary token strides and head stride 64, so q, k and v
// can be read straight out of the fused qkv projection output.
//
// Workgroup: 4 waves of QB 32-query blocks each (128 QB queries of one
// (sequence, head); QB = 2 or 1, see attention_fwd_kernel).
// Per 64-key tile a wave computes S^T = K Q^T for its query blocks
// (QB x 2 x 4 v_mfma_f32_32x32x16_f16, every K fragment read from LDS feeding
// all its blocks), the online softmax in registers, and O^T += V^T P^T (as
// many MFMAs again, each V^T fragment likewise shared).
// The softmax is trimmed to what the MFMAs cannot hide: key masking only on
// the last (partial) tile; Q pre-scaled by scale * log2(e) and the score
// accumulators started at -m (the running reference), so P = 2^S takes one
// exp2 per score and nothing else; row sums by v_dot2 on
// the fp16 pairs that the PV product uses, so that P's rounding cancels in the
// quotient (fp32 adds of the unrounded P raised the error against 64 bits by
// 2-4 % at sharp scores: 300 tokens, q scaled 4 times, 4.82e-4 -> 5.01e-4; same
// box, they took 7.17 ms against 7.13 at 43968 tokens, 94.3 us against 96.2 at
// 4122, 47.8 against 49.1 at 2748; v_fma_mix_f32 adds of the fp16 values were
// 1-3 % slower than the unrounded ones from 4122 tokens on);
// and a lazy rescale -- the reference moves only when a tile exceeds it by
// 2^8, so most tiles skip the O *= alpha pass, and the tile maximum itself is
// only computed when a lane's tile sum says some P may have exceeded 2^8.
// Layouts:
//  * S^T layout: lane (h = lane/32, q = lane%32) holds, for key block kb,
//    keys 32kb + 8*(r/4) + 4h + r%4 (r = 0..15) of query q.  A query's 64
//    scores are split between lanes q and q+32: one cross-lane exchange per
//    max / sum.
//  * P^T is the PV B operand without any shuffle: k-step s = 2kb + p takes
//    registers 8p..8p+7 of block kb, i.e. keys 32kb + 16p + {0..3, 8..11} + 4h.
//  * K and V tiles arrive by LDS DMA in their natural [key][dim] layout
//    (128-byte rows; 16-byte chunk c of row r at c ^ fk(r) for K and
//    c ^ fv(r) for V), one DMA tile ahead.  At QB = 2 a DMA tile holds 128
//    keys, consumed as two 64-key compute tiles, so the workgroup meets at
//    one barrier per 128 keys (1-2 % faster than one per 64, bit-identical);
//    at QB = 1 it copies 64-key tiles.
//  * V^T (the PV A operand) comes out of LDS through ds_read_b64_tr_b16: two
//    transposed 8-byte reads give each lane its dim's 8 keys in k-slot order,
//    with no register staging or transposed stores.
#include "common.h"

namespace qv {

constexpr int ATT_BK = 64;                 // keys per compute tile

constexpr float RESCALE_SLACK = 8.0f;  // log2 units: P <= 256 between rescales
constexpr float P_SUM_LIMIT = 256.0f;  // 2^RESCALE_SLACK: a lane's tile sum above it may hide a P above it

__device__ __forceinline__ int fk(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// V rows swizzle: 16-byte chunk c of key row r sits at c ^ fv(r).  The
// transposed reads below touch 4 consecutive rows per 16-lane group; fv moves
// rows r and r + 2 to opposite halves of the 128-byte row, so each 32-lane
// half of a read covers all 64 banks once.
__device__ __forceinline__ int fv(int r) { return 4 * ((r >> 1) & 1); }

typedef short v4i16 __attribute__((ext_vector_type(4)));
// ds_read_b64_tr_b16: within each 16-lane group, lane j = 4a + b receives
// element b of the 8-byte segments addressed by lanes a, a + 4, a + 8, a + 12.
__device__ __forceinline__ uint2 lds_read_tr16(const uint8_t* p) {
  const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) v4i16*)(__attribute__((address_space(3))) uint8_t*)p);
  return __builtin_bit_cast(uint2, r);
}

// max / sum of x over lanes l and l ^ 32.  v_permlane32_swap exchanges the
// upper half of its first operand with the lower half of its second; with
// both holding x, lane l ends with {x[l & 31], x[(l & 31) + 32]} in the pair.
// Written as inline asm: the compiler's model of the builtin folds the two
// results into one when both operands carry the same value.  The s_nop
// covers the VALU-write -> permlane-read hazard.
__device__ __forceinline__ void half_pair(float x, float& a, float& b) {
  a = x;
  b = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float half_max(float x) {
  float a, b;
  half_pair(x, a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float half_sum(float x) {
  float a, b;
  half_pair(x, a, b);
  return a + b;
}

// Two forms, bit-identical (a query's keys come in the same order, and the
// lazy rescale of a query depends on its own scores alone):
//  * wide (QB = 2): 64 queries a wave, 256 VGPRs, two 64 KB workgroups a CU.
//    Every LDS fragment feeds two MFMAs; bound by VALU issue and by what of it
//    two free-running waves overlap with MFMAs: 43968 tokens 7.1-7.7 ms
//    (1.03-1.11 PFLOP/s, boxes differ), 8 x 1374 77 us.
//  * fine (QB = 1): 32 queries a wave, 157 VGPRs, three 32 KB workgroups a CU.
//    Twice the LDS reads per MFMA (6-9 % slower on launches of many rounds),
//    but twice as many workgroups, which fill the CUs of a small launch.  Bound
//    by the chain QK -> exp2 -> PV of the one or two waves a SIMD then holds.
//    Against the wide form and 2-wave workgroups of it (what small launches
//    ran before), same box: 1 x 1374 32 / 29.7 -> 19.8 us, 2 x 1374 33 / 44 ->
//    28, 4 x 1374 52 / 47 -> 42, 6 x 1374 72 -> 65, 1 x 2748 57 / 78 -> 49,
//    1 x 4122 127 / 117 -> 98, 1 x 5496 172 / 156 -> 140, 1 x 8244 364 -> 325.
template <int WAVES, int SUB, int QB>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(QB == 2 ? 2 : 3, QB == 2 ? 2 : 3))) void attention_fwd_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    uint16_t* __restrict__ out, int L, int H, long q_ts, long kv_ts, long v_ts, long o_ts, float scale_log2) {
  constexpr int ATT_WAVES = WAVES;               // waves per workgroup
  constexpr int ATT_QW = 32 * QB;                // queries per wave
  constexpr int ATT_BQ = ATT_WAVES * ATT_QW;     // queries per workgroup
  constexpr int ATT_SUB = SUB;                   // compute tiles per DMA tile (one barrier per DMA tile)
  constexpr int ATT_BKD = ATT_BK * ATT_SUB;      // keys per DMA tile
  constexpr int ATT_DMA = ATT_BKD / 8 / ATT_WAVES;  // 1 KB (8-key) DMA rows per wave per DMA tile, K and V each
  static_assert(ATT_DMA * 8 * ATT_WAVES == ATT_BKD, "DMA rows split evenly over the waves");
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds[2][ATT_BKD * 128];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds[2][ATT_BKD * 128];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, l32 = lane & 31;
  const int qtiles = (L + ATT_BQ - 1) / ATT_BQ;
  // consecutive q-tiles of one (sequence, head) share an XCD (and its L2),
  // which then streams that head's K / V once for all of them
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int qt = lid % qtiles;
  const int head = (lid / qtiles) % H;
  const int seq = lid / (qtiles * H);
  const long tok0 = (long)seq * L;
  const bool live = qt * ATT_BQ + wave * ATT_QW < L;   // wave-uniform

  // ---- Q^T fragments (B operand of S^T = K Q^T): per query block, 4 k-steps of 16 dims
  uint4 qf[QB][4];
  int qi[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    qi[qb] = qt * ATT_BQ + wave * ATT_QW + 32 * qb + l32;     // query index in the sequence
    const int qc = qi[qb] < L ? qi[qb] : L - 1;
    const uint16_t* qp = q + (tok0 + qc) * q_ts + (long)head * 64;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // pre-scaled by scale * log2(e) (one fp16 rounding), so the MFMA yields
      // scores in log2 units and the softmax needs no per-score multiply
      const uint4 raw = *reinterpret_cast<const uint4*>(qp + 16 * s + 8 * h);
      const uint32_t rw[4] = {raw.x, raw.y, raw.z, raw.w};
      uint32_t sw[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f16x2 hv = __builtin_bit_cast(f16x2, rw[e]);
        const f16x2 sv = {(_Float16)((float)hv[0] * scale_log2), (_Float16)((float)hv[1] * scale_log2)};
        sw[e] = __builtin_bit_cast(uint32_t, sv);
      }
      qf[qb][s] = make_uint4(sw[0], sw[1], sw[2], sw[3]);
    }
  }

  // ---- K tile DMA: 16 x 1 KB per DMA tile, 4 per wave; lane L lands at key
  // r0 + L/8, physical chunk L%8, so it fetches logical chunk (L%8) ^ fk(row).
  const auto rsK = make_rsrc(k + tok0 * kv_ts + (long)head * 64, (uint64_t)L * kv_ts * 2);
  uint32_t k_voff[ATT_DMA];
#pragma unroll
  for (int w2 = 0; w2 < ATT_DMA; ++w2) {
    const int row = 8 * (ATT_DMA * wave + w2) + (lane >> 3);
    const int c = (lane & 7) ^ fk(row);
    k_voff[w2] = (uint32_t)((lane >> 3) * kv_ts * 2 + c * 16);
  }
  const uint32_t klds0 = lds_addr(k_lds);
  auto issue_k = [&](int tile, int buf) {
#pragma unroll
    for (int w2 = 0; w2 < ATT_DMA; ++w2) {
      const int r0 = 8 * (ATT_DMA * wave + w2);
      lds_dma16(rsK, k_voff[w2], (uint32_t)((tile * ATT_BKD + r0) * kv_ts * 2),
                klds0 + buf * (ATT_BKD * 128) + r0 * 128);
    }
  };
  // ---- V tile DMA, natural [key][dim] layout with the fv swizzle
  const auto rsV = make_rsrc(v + tok0 * v_ts + (long)head * 64, (uint64_t)L * v_ts * 2);
  uint32_t v_voff[ATT_DMA];
#pragma unroll
  for (int w2 = 0; w2 < ATT_DMA; ++w2) {
    const int row = 8 * (ATT_DMA * wave + w2) + (lane >> 3);
    const int c = (lane & 7) ^ fv(row);
    v_voff[w2] = (uint32_t)((lane >> 3) * v_ts * 2 + c * 16);
  }
  const uint32_t vlds0 = lds_addr(v_lds);
  auto issue_v = [&](int tile, int buf) {
#pragma unroll
    for (int w2 = 0; w2 < ATT_DMA; ++w2) {
      const int r0 = 8 * (ATT_DMA * wave + w2);
      lds_dma16(rsV, v_voff[w2], (uint32_t)((tile * ATT_BKD + r0) * v_ts * 2),
                vlds0 + buf * (ATT_BKD * 128) + r0 * 128);
    }
  };
  // Transposed V^T fragments: for k-step st (keys 16 st + {0..3, 8..11} + 4h
  // in k-slot order) and dim block db, lane (group G = lane / 16, i = lane % 16)
  // addresses key 16 st + 8 r + 4h + i / 4, dims 32 db + 16 (G & 1) + 4 (i & 3)
  // for reads r = 0, 1; the transpose hands lane l32 its dim's 8 keys.
  const int tr_key = 4 * h + ((lane & 15) >> 2);
  const int tr_dim = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int ntiles = (L + ATT_BKD - 1) / ATT_BKD;   // DMA tiles
  f32x16 o[QB][2];   // [query block][dim block]
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[qb][db][r] = 0.f;
  // m_use: the running reference maximum in log2 units.  It is only raised
  // when a tile's maximum exceeds it by more than RESCALE_SLACK, so P values
  // stay <= 2^RESCALE_SLACK and most tiles skip the O rescale.
  float m_use[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
  // base: the reference the score accumulators start from (S' = S - base,
  // the MFMA's C input), equal to m_use after the first tile, so P = 2^S'
  // needs one exp2 per score and nothing else
  float base[2] = {0.f, 0.f};

  // one 64-key compute tile: keys key0.., K / V rows at kb_lds / vb
  auto ctile = [&](int key0, const uint8_t* kb_lds, const uint8_t* vb, bool mask) __attribute__((always_inline)) {
    f32x16 sc[QB][2];   // [query block][key block]
    uint4 kf[2][4], vfr[2][4], pf[QB][4];
    float t = 0.f;
    auto qk1 = [&](int qb, int kb, int st) __attribute__((always_inline)) {
      sc[qb][kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, kf[kb][st]),
                                                          __builtin_bit_cast(f16x8, qf[qb][st]),
                                                          st == 0 ? f32x16{} - base[qb] : sc[qb][kb], 0, 0, 0);
    };
    auto pv1 = [&](int qb, int db, int st) __attribute__((always_inline)) {
      o[qb][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, vfr[db][st]),
                                                         __builtin_bit_cast(f16x8, pf[qb][st]), o[qb][db], 0, 0, 0);
    };
    auto read_v = [&](int db, int st) __attribute__((always_inline)) {
      const int dim = 32 * db + tr_dim;
      uint2 vv[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int key = 16 * st + 8 * r + tr_key;
        vv[r] = lds_read_tr16(vb + key * 128 + (((dim >> 3) ^ fv(key)) * 16) + ((dim >> 2) & 1) * 8);
      }
      vfr[db][st] = make_uint4(vv[0].x, vv[0].y, vv[1].x, vv[1].y);
    };
    auto mask_keys = [&](int qb) __attribute__((always_inline)) {
      const int kh = key0 + 4 * h;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kh + 32 * kb + 8 * (r >> 2) + (r & 3) >= L) sc[qb][kb][r] = -INFINITY;
    };
    // word w (0..15) of a query block's packed P: its scores 2 w, 2 w + 1
    auto p_word = [&](int qb, int w, bool shift, float off) __attribute__((always_inline)) {
      const float s0 = sc[qb][w >> 3][2 * (w & 7)], s1 = sc[qb][w >> 3][2 * (w & 7) + 1];
      const float p0 = __builtin_amdgcn_exp2f(shift ? s0 + off : s0);
      const float p1 = __builtin_amdgcn_exp2f(shift ? s1 + off : s1);
      const f16x2 ph = {(_Float16)p0, (_Float16)p1};
      return __builtin_bit_cast(uint32_t, ph);
    };
    auto add_p = [&](uint32_t w) __attribute__((always_inline)) {
      t = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w), (f16x2){(_Float16)1.0f, (_Float16)1.0f}, t, false);
    };
    auto set_p = [&](int qb, const uint32_t (&pw)[16]) __attribute__((always_inline)) {
#pragma unroll
      for (int st = 0; st < 4; ++st) pf[qb][st] = make_uint4(pw[4 * st], pw[4 * st + 1], pw[4 * st + 2], pw[4 * st + 3]);
    };
    // P = 2^S' = 2^(S - m_use) of a query block in fp16 against the current
    // reference, with the tile's partial row sum t (of the fp16 values).  The
    // tile maximum is only needed when some P could exceed 2^RESCALE_SLACK,
    // and every such P makes t exceed it too (P >= 0), so the maximum is
    // computed only for waves where some lane's t does, and on the first tile
    // (no reference yet).
    // QB = 2: slot(i) comes before each of 8 fenced groups of four exp2, so
    // that block 1's QK MFMAs run beside block 0's exp2 and block 0's PV MFMAs
    // beside block 1's (left to the compiler the MFMAs clustered: 10992 tokens
    // 488 -> 481 us, 8 x 1374 75.2 -> 73.0, 43968 7.12 -> 7.07 ms, the same
    // bits; at QB = 1 fencing cost 5 % at 1 x 1374 and is left out).  A
    // group's sums come one group later, at QB = 1 after all groups (in the
    // group itself 1 x 4122 took 2 % more, 1 x 2748 3 %).
    auto softmax = [&](int qb, auto&& slot) __attribute__((always_inline)) {
      if (mask) mask_keys(qb);
      uint32_t pw[16];
      t = 0.f;
      if constexpr (QB == 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        slot(i);
        if (QB == 2 && i > 0) {
          add_p(pw[2 * i - 2]);
          add_p(pw[2 * i - 1]);
        }
        pw[2 * i] = p_word(qb, 2 * i, false, 0.f);
        pw[2 * i + 1] = p_word(qb, 2 * i + 1, false, 0.f);
        if constexpr (QB == 2) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int w = QB == 2 ? 14 : 0; w < 16; ++w) add_p(pw[w]);
      if (__builtin_amdgcn_ballot_w64(!(t <= P_SUM_LIMIT) || m_use[qb] == -INFINITY)) {
        // ---- tile maximum of this query (both lane halves hold 32 keys each)
        float mx = sc[qb][0][0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[qb][0][r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[qb][1][r]);
        mx = half_max(mx) + base[qb];
        const bool need = mx > m_use[qb] + RESCALE_SLACK;
        if (__builtin_amdgcn_ballot_w64(need)) {
          const float m_new = need ? mx : m_use[qb];
          const float alpha = __builtin_amdgcn_exp2f(m_use[qb] - m_new);  // 0 on the first tile, 1 if !need
          m_use[qb] = m_new;
          l_run[qb] *= alpha;
#pragma unroll
          for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[qb][db][r] *= alpha;
          t = 0.f;
          const float off = base[qb] - m_new;
#pragma unroll
          for (int w = 0; w < 16; ++w) pw[w] = p_word(qb, w, true, off);
#pragma unroll
          for (int w = 0; w < 16; ++w) add_p(pw[w]);
        }
        base[qb] = m_use[qb];
      }
      l_run[qb] += t;
      set_p(qb, pw);
    };
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int row = 32 * kb + l32;
        kf[kb][st] = *reinterpret_cast<const uint4*>(kb_lds + row * 128 + (((2 * st + h) ^ fk(row)) * 16));
      }
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) qk1(0, kb, st);
    if constexpr (QB == 2) {
      softmax(0, [&](int i) __attribute__((always_inline)) {
        qk1(1, i & 1, i >> 1);
        if (i >= 4) {   // V^T fragments, as the K fragments' registers fall free
          read_v(0, i - 4);
          read_v(1, i - 4);
        }
      });
      softmax(1, [&](int i) __attribute__((always_inline)) { pv1(0, i & 1, i >> 1); });
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int db = 0; db < 2; ++db) pv1(1, db, st);
    } else {
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        read_v(0, st);
        read_v(1, st);
      }
      softmax(0, [](int) __attribute__((always_inline)) {});
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int db = 0; db < 2; ++db) pv1(0, db, st);
    }
  };
  auto tile = [&](int j, bool last) {
    const int buf = j & 1;
    const bool more = j + 1 < ntiles;
    if (more) {
      issue_k(j + 1, buf ^ 1);
      issue_v(j + 1, buf ^ 1);
    }
    // a wave whose queries all lie past the sequence end (the last query
    // tile of a frame) only issues its share of the DMA and keeps the barriers
    if (live) {
#pragma unroll
      for (int u = 0; u < ATT_SUB; ++u) {
        const int key0 = j * ATT_BKD + u * ATT_BK;
        if (!last) {
          ctile(key0, k_lds[buf] + u * ATT_BK * 128, v_lds[buf] + u * ATT_BK * 128, false);
        } else if (key0 < L) {
          ctile(key0, k_lds[buf] + u * ATT_BK * 128, v_lds[buf] + u * ATT_BK * 128, key0 + ATT_BK > L);
        }
      }
    }
    if (more) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): next K and V tiles landed
    lds_barrier();
  };

  issue_k(0, 0);
  issue_v(0, 0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  lds_barrier();
  const int nfull = L / ATT_BKD;       // DMA tiles with every key valid
  for (int j = 0; j < nfull; ++j) tile(j, false);
  if (nfull < ntiles) tile(nfull, true);

  // ---- normalise and store: lane (h, q) holds dims 32db + 8*(r/4) + 4h + r%4
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float l_tot = half_sum(l_run[qb]);
    const float inv = 1.0f / l_tot;
    if (qi[qb] < L) {
      uint16_t* op = out + (tok0 + qi[qb]) * o_ts + (long)head * 64;
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          uint2 w;
          w.x = pack2<false>(o[qb][db][4 * g] * inv, o[qb][db][4 * g + 1] * inv);
          w.y = pack2<false>(o[qb][db][4 * g + 2] * inv, o[qb][db][4 * g + 3] * inv);
          *reinterpret_cast<uint2*>(op + 32 * db + 8 * g + 4 * h) = w;
        }
    }
  }
}

// Which form a launch of BH (sequence, head) pairs runs, from its estimated
// time in hundredths of a full wide round (512 workgroups of 256 queries, two
// a CU).  Wide: whole rounds, then a last one that costs 45 up to one
// workgroup a CU (64 where it is the only one) and 100 above.  Fine: 82 per
// 768 workgroups (three a CU) + 13.  Both fitted to the times above and to
// launches on either side of the line: wide keeps 1 x 6870 (217 against 227
// us), 1 x 10992 (500 / 527), 8 x 1374 (74 / 77), 16 x 1374 (146 / 146);
// fine takes 6 x 1374 (72 / 65) and 1 x 8244 (362 / 322).
static bool attention_fine(long BH, long L) {
  const long wide = BH * ((L + 255) / 256), fine = BH * ((L + 127) / 128);
  const long rem = wide % 512;
  const long wide_cost = wide / 512 * 100 + (rem == 0 ? 0 : rem > 256 ? 100 : wide < 512 ? 64 : 45);
  return fine * 82 / 768 + 13 < wide_cost;
}

}  // namespace qv

extern "C" int qv_attention_fwd(const void* q, const void* k, const void* v, void* out, int64_t B, int64_t L,
                                int64_t H, int64_t head_dim, int64_t q_token_stride, int64_t k_token_stride,
                                int64_t v_token_stride, int64_t out_token_stride, float scale, void* stream) {
  QV_CHECK_ARG(head_dim == 64, "only head_dim 64 is supported (got %lld)", (long long)head_dim);
  QV_CHECK_ARG(B >= 0 && L >= 0 && H > 0, "bad shape B=%lld L=%lld H=%lld", (long long)B, (long long)L, (long long)H);
  if (B == 0 || L == 0) return QV_OK;
  QV_CHECK_ARG(q && k && v && out, "null pointer argument");
  QV_CHECK_ARG(q_token_stride % 8 == 0 && k_token_stride % 8 == 0 && v_token_stride % 8 == 0 &&
                   out_token_stride % 4 == 0 && q_token_stride >= H * 64 && k_token_stride >= H * 64 &&
                   v_token_stride >= H * 64 && out_token_stride >= H * 64,
               "token strides must cover the heads and keep 16-byte alignment");
  QV_CHECK_ARG(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0 &&
                   ((uintptr_t)out % 8) == 0,
               "q, k, v must be 16-byte and out 8-byte aligned");
  QV_CHECK_ARG((uint64_t)L * k_token_stride * 2 < (1ull << 32) && (uint64_t)L * v_token_stride * 2 < (1ull << 32),
               "sequence too long for 32-bit offsets");
  const bool fine = qv::attention_fine(B * H, L);
  const long nwg = B * H * (fine ? (L + 127) / 128 : (L + 255) / 256);
  QV_CHECK_ARG(nwg <= INT32_MAX, "grid too large");
  const float scale_log2 = scale * 1.4426950408889634f;
#define QV_ATT_ARGS                                                                                       \
  (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)out, (int)L, (int)H, (long)q_token_stride, \
      (long)k_token_stride, (long)v_token_stride, (long)out_token_stride, scale_log2
  if (fine)
    hipLaunchKernelGGL((qv::attention_fwd_kernel<4, 1, 1>), dim3((unsigned)nwg), dim3(256), 0, (hipStream_t)stream,
                       QV_ATT_ARGS);
  else
    hipLaunchKernelGGL((qv::attention_fwd_kernel<4, 2, 2>), dim3((unsigned)nwg), dim3(256), 0, (hipStream_t)stream,
                       QV_ATT_ARGS);
#undef QV_ATT_ARGS
  return qv::check_launch("attention_fwd");
}
