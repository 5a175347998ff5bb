// Decode at other head dims and in float32 on the matrix cores: head_dim_v in
// {64, 128, 256, 512} with rope_dim in {16, 32, 64} and 16-byte aligned rows,
// the dims a model with a smaller (or wider-RoPE) latent than 512 + 64 has
// and the float32 check of one. Other accepted dims keep the forms of
// mla_decode_generic.hip, which calls in here.
//
// Both kernels walk the split-KV partition of decode_common.h (uniform
// pieces, or one balanced range per worker), stream the cache through an
// LDS ring with LDS-DMA copies, and write a float32 partial row and its
// base-2 log-sum-exp per (slot, head) (the reference's formats,
// src/triton_mla/kernel.py:126-138), or the output itself where one worker
// covers the sequence; mla_dims_combine_kernel merges (kernel.py:159-181).
//
// mla_dims_kernel (bf16 / fp16). A cache row is read once per 128 heads. The
// S^T = K . Q^T, softmax and O^T += V^T . P^T of 32 heads x 32 tokens belong
// to one wave (the register-to-register scheme of mla_partial_own_kernel:
// the score tile's layout is the value product's operand layout), and up to
// 256 value dims leave room for two waves per SIMD: a workgroup is 4 waves
// along the heads x 2 along the tokens, so one wave's softmax and waits run
// under the other's MFMAs without a hand-made schedule, and the two token
// waves' results merge in LDS, not in memory (half the float32 partials).
// 32 sequences of 8,192 tokens, 128 heads, 256 + 32 in bf16: 64 us for both
// kernels (414 us with mla_generic_mfma_kernel, which re-read and transposed
// the rows through registers); the step loop runs at 1.1 PFLOP/s, where a
// large bf16 matmul reaches 1.2 on this card; start-up 6, merge 5 and the
// combine 9 us are most of the rest. A wave priority for one of the two waves
// and longer read-ahead changed nothing.
//
// mla_dims_f32_kernel (float32). v_mfma_f32_16x16x4_f32 (float32 products
// and sums). A workgroup takes 16 (or 32) heads; its 4 waves split the dims
// of one 16-token slice: each contracts a quarter of the score dims, the
// partial scores meet in LDS, every wave runs the (small) softmax and owns a
// quarter of the value dims. One b128 read feeds four MFMAs. 16 sequences of
// 5,003 to 8,192 tokens, 16 heads, 512 + 64: 77 us for both kernels (257 us
// with the vector-ALU form); a slice takes 2.1 us, of which the card's copy
// rate (5.1 TB/s) needs 1.85. With the softmax and the copies beside the score
// MFMAs of the next slice: 2.13 us a slice, 2.4 with them after the value
// MFMAs.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "cdna.h"
#include "decode_common.h"
#include "dims.h"
#include "triton_mla.h"

namespace tmla {
namespace dims {

constexpr int kSub = 32;  // tokens of a sub-tile (16-bit kernel)
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void pin_v16(f32x16& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin_a16(f32x16& x) { asm volatile("" : "+a"(x)); }
template <int N>
__device__ __forceinline__ void lgkm() {
  static_assert(N >= 0 && N <= 15, "lgkmcnt range");
  asm volatile("s_waitcnt lgkmcnt(%0)" : : "i"(N));
}
__device__ __forceinline__ void tie8(i16x8& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void tie4(i16x4& x) { asm volatile("" : "+v"(x)); }
template <class T>
__device__ __forceinline__ void tie_v(T& x) {
  asm volatile("" : "+v"(x));
}
__device__ __forceinline__ void ds_write_f4(char LDS_AS* p, const f32x4& v) {
  asm volatile("ds_write_b128 %0, %1" : : "v"(p), "v"(v));
}
// F (1, 2 or 4) consecutive floats of LDS as the compiler-opaque reads above
template <int F>
struct VecF {
  typedef f32x4 T;
};
template <>
struct VecF<2> {
  typedef f32x2 T;
};
template <>
struct VecF<1> {
  typedef float T;
};
template <int F, int OFF>
__device__ __forceinline__ typename VecF<F>::T ds_read_f(const char LDS_AS* p) {
  typename VecF<F>::T r;
  if constexpr (F == 4)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(p), "i"(OFF));
  else if constexpr (F == 2)
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(p), "i"(OFF));
  else
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(r) : "v"(p), "i"(OFF));
  return r;
}
template <int F>
__device__ __forceinline__ float elem(const typename VecF<F>::T& v, int i) {
  if constexpr (F == 1)
    return v;
  else
    return v[i];
}

// S^T MFMAs: volatile asm with the accumulator in VGPRs (the softmax reads
// it; the value accumulators live in AGPRs). s_fence before VALU reads it.
template <int DT>
__device__ __forceinline__ f32x16 s_first(const i16x8& a, const i16x8& b) {
  f32x16 d;
  if constexpr (DT == TMLA_BF16)
    asm volatile(TMLA_MFMA_GAP "v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  else
    asm volatile(TMLA_MFMA_GAP "v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  return d;
}
template <int DT>
__device__ __forceinline__ void s_acc(f32x16& d, const i16x8& a, const i16x8& b) {
  if constexpr (DT == TMLA_BF16)
    asm volatile(TMLA_MFMA_GAP "v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  else
    asm volatile(TMLA_MFMA_GAP "v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void s_fence(f32x16& d) {
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+v"(d));
}

template <int DT>
__device__ __forceinline__ float pack2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  if constexpr (DT == TMLA_BF16)
    return __builtin_bit_cast(float, __builtin_convertvector((f32x2){a, b}, bf16x2));
  else
    return __builtin_bit_cast(float, __builtin_convertvector((f32x2){a, b}, f16x2));
}

// Byte offset of token t's row (t below the capacity) given its raw table
// entry (paged: clamped into the cache; dense: unused).
__device__ __forceinline__ int64_t row_off(const PartialArgs& a, bool paged, int b, int t, int raw) {
  if (!paged) return (int64_t)b * a.kv_s0 + (int64_t)t * a.kv_s1;
  const int in_page = a.page_shift >= 0 ? (t & (a.page_size - 1)) : (t % a.page_size);
  return (int64_t)min(max(raw, 0), a.max_page) * a.kv_s0 + (int64_t)in_page * a.kv_s1;
}

// Rows of `tok` from the finished (m, l, O) of one segment: where they go
struct RowTarget {
  float* part;   // partial row of head 0 of the slot, or
  float* plse;
  char* out;     // the output row of head 0 (direct)
  int64_t out_sh;
  float* lse;    // may be NULL
  bool direct;
};

__device__ __forceinline__ RowTarget row_target(const DimsArgs& a, const SegmentSlot& ss, int b, int dv, int es) {
  RowTarget t;
  t.direct = ss.direct;
  t.part = a.part + (int64_t)ss.slot * a.num_heads * dv;
  t.plse = a.part_lse + (int64_t)ss.slot * a.num_heads;
  t.out = a.out + (int64_t)b * a.out_sb * es;
  t.out_sh = a.out_sh;
  t.lse = a.lse == nullptr ? nullptr : a.lse + (int64_t)b * a.num_heads;
  return t;
}

// ---------------------------------------------------------------------------
// 16-bit kernel
// ---------------------------------------------------------------------------
// LDS: kRing slots of TW sub-tiles; a sub-tile is the V part in the blocks of
// 8 rows x 128 bytes and the piece swizzle of the 512 + 64 kernels (row
// group, column block), then the rope rows (DR * 2 bytes each, pieces
// XOR-swizzled by row so that 16 rows' reads of one piece spread over all
// banks). Then the Q^T operands that do not stay in registers, one KiB per
// (chunk, head wave). The token waves' results meet in the whole of it.
template <int DV, int DR>
struct Cfg {
  static constexpr int HW = 4;                  // waves along the heads, 32 each
  static constexpr int TW = DV >= 512 ? 1 : 2;  // waves along the tokens
  static constexpr int NW = HW * TW;
  static constexpr int NVB = DV / 64;           // 128-byte column blocks of the V part
  static constexpr int NKL = DV / 16, NKC = (DV + DR) / 16;  // k-chunks: latent, all
  static constexpr int NDB = DV / 32;
  // k-chunks whose Q^T operand stays in VGPRs. At 256 dims two waves per SIMD
  // leave 128 VGPRs beside the 128 accumulators: half of the latent chunks
  // (11 of 16 where the LDS has no room for more).
  static constexpr int NQR = DV == 256 ? (DR == 64 ? 11 : 8) : NKL;
  static constexpr int SUBV = 4 * NVB * 1024, SUBR = kSub * DR * 2, SUB = SUBV + SUBR;
  static constexpr int RING = 3;
  static constexpr int OFF_Q = RING * TW * SUB;
  static constexpr int OFF_ML = OFF_Q + (NKC - NQR) * HW * 1024;  // (m, l) of every wave's heads
  static constexpr int PDIM = DV >= 256 ? 128 : 64;              // value dims per merge pass
  static constexpr int OPITCH = PDIM * 4 + 16;
  static constexpr int MERGE = TW * HW * 32 * OPITCH;
  static constexpr int SMEM = (OFF_ML > MERGE ? OFF_ML : MERGE) + TW * HW * 32 * 8;
  static constexpr int LOADS = NVB + 1;  // copies per wave and step (one row group)
  static constexpr int PD = 2;  // operand reads ahead, in MFMA steps (3 and 4: the same time; 512 dims 6% slower)
  // LDS reads of step t of a sub-tile: one K operand (and a Q^T one), or two
  // V^T halves
  static constexpr int reads(int t) { return t < NKC ? (t < NQR ? 1 : 2) : (t < NKC + 2 * NDB ? 2 : 0); }
};

template <int DT, int DV, int DR>
__device__ __forceinline__ void dims_body(const DimsArgs& a, bool paged) {
  using C = Cfg<DV, DR>;
  constexpr int NKC = C::NKC, NDB = C::NDB, NT = NKC + 2 * NDB, PD = C::PD;
  static_assert(C::SMEM <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
  char LDS_AS* const lds = (char LDS_AS*)(void LDS_AS*)smem;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hw = wave / C::TW, tw = wave % C::TW;  // token waves of one head block on neighbouring SIMDs
  const int lane = tid & 63, hi = lane >> 5;
  const int head_base = blockIdx.y * 32 * C::HW + hw * 32;
  const bool busy = head_base < a.num_heads;  // the others only copy
  const CappedLens len_of{a.seqlens, a.len_cap};

  WorkRange wr;
  const int worker = worker_index(a);
  if (!work_range(a, len_of, worker, wr) || wr.tile_lo >= wr.tile_hi) return;
  const float cabs = fabsf(a.qk_scale_log2);
  const bool negate = a.qk_scale_log2 < 0.0f;

  // Operand read offsets inside a sub-tile; the pieces differ from one base
  // by XORs, since the swizzle is one:
  // K operand: token lane%32, piece 2 (kc%4) + hi of column block kc/4
  int k_base;
  {
    const int rg = (lane & 31) >> 3, r = lane & 7;
    k_base = rg * C::NVB * 1024 + (r * 8 + (hi ^ piece_swizzle(r, rg))) * 16;
  }
  // V^T operand of dim block db, k-step c, half e2 (ds_read_b64_tr_b16): as
  // in mla_partial_own_kernel
  int v_base;
  {
    const int g = lane >> 4, L = lane & 15, r = 4 * (g >> 1) + (L >> 2);
    v_base = (r * 8 + ((2 * (g & 1) + ((L & 3) >> 1)) ^ piece_swizzle(r, 0))) * 16 + 8 * (L & 1);
  }
  // rope K operand: piece 2c + hi of row lane%32, swizzled by row
  constexpr int NP = DR / 8;  // 16-byte pieces of a rope row
  const int r_base = C::SUBV + (lane & 31) * DR * 2 + ((hi ^ ((lane & 31) / (16 / NP))) & (NP - 1)) * 16;

  int b = wr.b_first, t_start = wr.tile_lo, remaining = wr.tile_hi - wr.tile_lo, seg_off = wr.off_first;
  while (remaining > 0) {
    const int n_b = len_of(b);
    const int nt_b = tiles_of(n_b);
    if (nt_b == 0) {
      ++b;
      continue;
    }
    const int t_end = min(nt_b, t_start + remaining);
    const SegmentSlot ss = segment_slot(a, wr, worker, b, t_start, nt_b, seg_off);
    const int tok0 = t_start * kTileTokens, end = min(t_end * kTileTokens, n_b);
    const int steps = (end - tok0 + kSub * C::TW - 1) / (kSub * C::TW);
    const int32_t* bt_row = paged ? a.bt + (int64_t)b * a.bt_sb : nullptr;

    // Copies: this wave's row group hw of sub-tile tw. Row lane/8 of the V
    // blocks (lane%8 = swizzled piece), row lane / NP of the rope rows; rows
    // past the piece read its last row again. (Lane offsets are recomputed
    // where used: kept across the loop they would not fit the registers.)
    auto v_row = [&]() __attribute__((always_inline)) { return 8 * hw + (lane_id_fresh() >> 3); };
    auto r_row = [&]() __attribute__((always_inline)) { return 8 * hw + ((lane_id_fresh() / NP) & 7); };
    auto tok_of = [&](int st, int row) __attribute__((always_inline)) {
      return token_or_last(tok0, ((uint32_t)st * C::TW + tw) * kSub + row, end);
    };
    auto raw_page = [&](int t) __attribute__((always_inline)) { return paged ? bt_row[page_slot_of(a, t)] : 0; };
    // Table entries of step st: the sub-tile's one page where a page holds
    // whole sub-tiles (a.uni), else this lane's two rows'
    struct Pages {
      int v, r;
    };
    auto pages_of = [&](int st) __attribute__((always_inline)) {
      Pages pg{0, 0};
      if (a.uni) {
        pg.v = raw_page(tok_of(st, 0));
      } else if (paged) {
        pg.v = raw_page(tok_of(st, v_row()));
        pg.r = raw_page(tok_of(st, r_row()));
      }
      return pg;
    };
    auto issue = [&](int st, const Pages& pg) __attribute__((always_inline)) {
      char LDS_AS* dst = lds + ((unsigned)st % C::RING * C::TW + tw) * C::SUB;
      const int ln = lane_id_fresh();
      const int rr = 8 * hw + ((ln / NP) & 7);
      const int v_piece = ((ln & 7) ^ piece_swizzle(ln >> 3, hw)) * 16;
      const int r_piece = DV * 2 + ((ln % NP) ^ ((rr / (16 / NP)) & (NP - 1))) * 16;
      const uint32_t ahead = ((uint32_t)st * C::TW + tw) * kSub;
      const char *src, *rsrc;
      if (a.uni && tokens_before(tok0, ahead, kSub, end)) {
        // one scalar base and 32-bit lane offsets
        const int t0 = tok0 + ahead;
        const char* row0 = a.kv + row_off(a, paged, b, t0, __builtin_amdgcn_readfirstlane(pg.v));
        src = row0 + (uint32_t)((8 * hw + (ln >> 3)) * (uint32_t)a.kv_s1 + v_piece);
        rsrc = row0 + (uint32_t)(rr * (uint32_t)a.kv_s1 + r_piece);
      } else {
        // (a.uni: rows past the piece clamp to its last, in the same page)
        src = a.kv + row_off(a, paged, b, tok_of(st, 8 * hw + (ln >> 3)), pg.v) + v_piece;
        rsrc = a.kv + row_off(a, paged, b, tok_of(st, rr), a.uni ? pg.v : pg.r) + r_piece;
      }
      static_for<C::NVB>([&](auto CB) __attribute__((always_inline)) {
        constexpr int cb = decltype(CB)::value;
        lds_copy16<cb * 128>(src, dst + (hw * C::NVB + cb) * 1024);
      });
      if (ln < 8 * NP) lds_copy16<0>(rsrc, dst + C::SUBV + hw * 8 * DR * 2);
    };

    f32x16 acc[NDB];
#pragma unroll
    for (int d = 0; d < NDB; ++d) acc[d] = (f32x16)0.0f;
    float m_run = kNoMax, l_run = 0.0f;

    // Start-up: the copies of step 0, Q, the copies of step 1, so that the
    // first rows and Q arrive in one round trip and only step 1's copies are
    // behind Q in the order that vmcnt counts.
    Pages pg = pages_of(0), pg1 = pages_of(1);
    issue(0, pg);
    asm volatile("" ::: "memory");
    // Q^T operands: lane (head lane%32, half hi) holds dims 16c + 8hi ..+7;
    // heads past num_heads run on head 0's row and are not stored
    i16x8 qop[C::NQR];
    {
      const int head = head_base + (lane & 31);
      const short* qrow = reinterpret_cast<const short*>(a.q) + (int64_t)b * a.q_sb +
                          (int64_t)(head < a.num_heads ? head : 0) * a.q_sh + 8 * hi;
      const i16x8 sgn = negate ? (i16x8)(short)0x8000 : (i16x8)(short)0;
#pragma unroll
      for (int c = 0; c < C::NQR; ++c) qop[c] = *reinterpret_cast<const i16x8*>(qrow + 16 * c) ^ sgn;
      if (tw == 0) {
#pragma unroll
        for (int c = C::NQR; c < NKC; ++c)
          *reinterpret_cast<i16x8 LDS_AS*>(lds + C::OFF_Q + ((c - C::NQR) * C::HW + hw) * 1024 + lane * 16) =
              *reinterpret_cast<const i16x8*>(qrow + 16 * c) ^ sgn;
      }
    }
    asm volatile("" ::: "memory");
    pg = pages_of(2);
    issue(1, pg1);
#pragma unroll
    for (int c = 0; c < C::NQR; ++c) tie8(qop[c]);

    for (int st = 0; st < steps; ++st) {
      // own copies of step st have landed (those of step st + 1 may fly);
      // then everyone's have, and everyone is done with step st - 1
      wait_vmcnt<C::LOADS>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      lds_barrier();
      {
        const Pages pn = pages_of(st + 3);
        asm volatile("" ::: "memory");
        issue(st + 2, pg);
        pg = pn;
      }
      const int base = tok0 + (st * C::TW + tw) * kSub;
      if (!busy || base >= end) continue;
      const char LDS_AS* sub = lds + ((st % C::RING) * C::TW + tw) * C::SUB;
      const int kb0 = (int)(size_t)(sub - lds) + k_base, vb0 = (int)(size_t)(sub - lds) + v_base;
      const int rb0 = (int)(size_t)(sub - lds) + r_base;
      const char LDS_AS* qp = lds + C::OFF_Q + hw * 1024 + lane * 16;

      i16x8 kb[PD + 1], qb[PD + 1];
      i16x4 vl[PD + 1], vh[PD + 1];
      f32x16 s;
      f32x4 pk[2];
      auto fetch = [&](auto T) __attribute__((always_inline)) {
        constexpr int t = decltype(T)::value, r = t % (PD + 1);
        if constexpr (t < NKC) {
          if constexpr (t < C::NKL)
            kb[r] = ds_read_b128<(t >> 2) * 1024>(lds + (kb0 ^ ((t & 3) << 5)));
          else
            kb[r] = ds_read_b128<0>(lds + (rb0 ^ ((t - C::NKL) << 5)));
          if constexpr (t >= C::NQR) qb[r] = ds_read_b128<(t - C::NQR) * C::HW * 1024>(qp);
        } else if constexpr (t < NT) {
          constexpr int g = t - NKC, c = g / NDB, db = g % NDB;
          constexpr int off = c * 2 * C::NVB * 1024 + (db >> 1) * 1024;
          vl[r] = ds_read_tr<off>(lds + (vb0 ^ ((db & 1) << 6)));
          vh[r] = ds_read_tr<off + C::NVB * 1024>(lds + (vb0 ^ ((db & 1) << 6) ^ 32));
        }
      };
      static_for<PD>([&](auto T) __attribute__((always_inline)) { fetch(T); });
      static_for<NT>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value, r = j % (PD + 1);
        if constexpr (j + PD < NT) fetch(std::integral_constant<int, j + PD>{});
        constexpr int after = [] {
          int n = 0;
          for (int t = j + 1; t <= (j + PD < NT - 1 ? j + PD : NT - 1); ++t) n += C::reads(t);
          return n;
        }();
        lgkm<after>();
        if constexpr (j < NKC) {
          tie8(kb[r]);
          if constexpr (j < C::NQR) {
            if constexpr (j == 0)
              s = s_first<DT>(kb[r], qop[j]);
            else
              s_acc<DT>(s, kb[r], qop[j]);
          } else {
            tie8(qb[r]);
            s_acc<DT>(s, kb[r], qb[r]);
          }
        } else {
          tie4(vl[r]);
          tie4(vh[r]);
          constexpr int g = j - NKC, c = g / NDB, db = g % NDB;
          const i16x4 lo = vl[r], h4 = vh[r];
          const i16x8 vop = {lo[0], lo[1], lo[2], lo[3], h4[0], h4[1], h4[2], h4[3]};
          acc[db] = Elt<DT>::mfma(vop, __builtin_bit_cast(i16x8, pk[c]), acc[db]);
          pin_a16(acc[db]);
        }
        if constexpr (j == NKC - 1) {
          // online softmax, base 2, with the lazy rescale: lane holds head
          // lane%32, tokens 8 (r / 4) + 4 hi + r % 4 in register r. (A
          // reference that follows every new max leaves that token's
          // probability exact: error against float64 1.728e-3 instead of
          // 1.752e-3 at 32 sequences, 256 + 32 in bf16, 1.76e-3 instead of
          // 1.81e-3 at 512 + 32; it takes 68.7 us instead of 61 and 61.5
          // instead of 50.7. v_exp_f32 and exp2f give the same error.)
          s_fence(s);
          if (base + kSub > end) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (base + 4 * hi + 8 * (i >> 2) + (i & 3) >= end) s[i] = -INFINITY;
          }
          float mx = s[0];
#pragma unroll
          for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
          mx *= cabs;
          if (__builtin_amdgcn_ballot_w64(mx > m_run + kRescaleLog2) != 0) {
            float x = mx, y = mx;
            swap_rows32(x, y);
            const float m_new = fmaxf(m_run, fmaxf(x, y));
            if (m_run != kNoMax) {
              const float f = fast_exp2(m_run - m_new);
              l_run *= f;
#pragma unroll
              for (int d = 0; d < NDB; ++d) {
                f32x16 t = acc[d];
                pin_v16(t);
                t *= f;
                acc[d] = t;
                pin_a16(acc[d]);
              }
            }
            m_run = m_new;
          }
#pragma unroll
          for (int i = 0; i < 16; i += 2) {
            const float p0 = fast_exp2(fmaf(s[i], cabs, -m_run)), p1 = fast_exp2(fmaf(s[i + 1], cabs, -m_run));
            l_run += p0 + p1;
            pk[i / 8][(i / 2) % 4] = pack2<DT>(p0, p1);
          }
        }
      });
    }
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
    wait_vmcnt<0>();
    lds_barrier();  // every wave is done with the ring

    // ---- merge of the token waves and the rows out -----------------------
    // The token waves of a head block exchange (m, l); each scales its
    // accumulators by its share (lane = head) and puts them into LDS rows,
    // PDIM dims at a time, where a row's parts only have to be added.
    {
      const int lane = lane_id_fresh(), hi = lane >> 5;  // (not kept live across the loop)
      float la = l_run, lb = l_run;
      swap_rows32(la, lb);
      float l = la + lb, m = m_run, f = 1.0f;
      if constexpr (C::TW == 2) {
        char LDS_AS* ml = lds + C::SMEM - C::TW * C::HW * 32 * 8 + (hw * 32 + (lane & 31)) * 8;
        if (hi == 0) *reinterpret_cast<f32x2 LDS_AS*>(ml + tw * C::HW * 32 * 8) = f32x2{m, l};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        lds_barrier();
        const f32x2 other = *reinterpret_cast<const f32x2 LDS_AS*>(ml + (1 - tw) * C::HW * 32 * 8);
        m = fmaxf(m_run, other[0]);
        f = fast_exp2(m_run - m);
        const float fo = fast_exp2(other[0] - m);
        l = tw == 0 ? l * f + other[1] * fo : other[1] * fo + l * f;
      }
      const bool has = l > 0.0f;
      f *= has ? 1.0f / l : 0.0f;
      const RowTarget tgt = row_target(a, ss, b, DV, 2);
      const int rows = min(32, a.num_heads - head_base);
      if (tw == 0 && lane < rows && hi == 0) {
        if (!tgt.direct)
          tgt.plse[head_base + lane] = has ? m + fast_log2(l) : -INFINITY;
        else if (tgt.lse)
          tgt.lse[head_base + lane] = has ? (m + fast_log2(l)) * kLn2 : -INFINITY;
      }
      constexpr int RPW = 32 / C::TW;  // rows (heads) a wave stores
#pragma unroll
      for (int p = 0; p < DV / C::PDIM; ++p) {
        if (busy) {
#pragma unroll
          for (int d = 0; d < C::PDIM / 32; ++d) {
            f32x16 t = acc[p * (C::PDIM / 32) + d];
            pin_v16(t);
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
              *reinterpret_cast<f32x4 LDS_AS*>(lds + ((tw * C::HW + hw) * 32 + (lane & 31)) * C::OPITCH +
                                               (32 * d + 8 * q4 + 4 * hi) * 4) =
                  f32x4{t[4 * q4] * f, t[4 * q4 + 1] * f, t[4 * q4 + 2] * f, t[4 * q4 + 3] * f};
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        lds_barrier();
        // four rows per store, 16 bytes per lane (PDIM = 64: 16 lanes a row;
        // 128: 32 lanes a row, two rows)
        constexpr int LPR = C::PDIM / 4, RPS = 64 / LPR;  // lanes per row, rows per store
        const int dim = p * C::PDIM + (lane % LPR) * 4;
#pragma unroll 2
        for (int i = 0; i < RPW; i += RPS) {
          const int h = tw * RPW + i + lane / LPR, off = h * C::OPITCH + (lane % LPR) * 16;
          f32x4 o = *reinterpret_cast<const f32x4 LDS_AS*>(lds + hw * 32 * C::OPITCH + off);
          if constexpr (C::TW == 2) o += *reinterpret_cast<const f32x4 LDS_AS*>(lds + (C::HW + hw) * 32 * C::OPITCH + off);
          if (h < rows) {
            if (tgt.direct) {
              f32x2 r = {pack2<DT>(o[0], o[1]), pack2<DT>(o[2], o[3])};
              *reinterpret_cast<f32x2*>(reinterpret_cast<short*>(tgt.out) + (int64_t)(head_base + h) * tgt.out_sh + dim) = r;
            } else {
              *reinterpret_cast<f32x4*>(tgt.part + (int64_t)(head_base + h) * DV + dim) = o;
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        lds_barrier();  // rows read: the next pass (or segment) overwrites them
      }
    }
    remaining -= t_end - t_start + wr.seg_cost;
    seg_off += nt_b + wr.seg_cost;
    ++b;
    t_start = 0;
  }
}

// (two waves per SIMD up to 256 value dims: 256 registers each; one at 512)
template <int DT, int DV, int DR>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
void mla_dims_kernel(DimsArgs a) {
  dims_body<DT, DV, DR>(a, a.bt != nullptr);
}
template <int DT, int DV, int DR>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void mla_dims512_kernel(DimsArgs a) {
  dims_body<DT, DV, DR>(a, a.bt != nullptr);
}

// ---------------------------------------------------------------------------
// float32 kernel
// ---------------------------------------------------------------------------
// A slice is 16 rows: the latent part row by row (256-byte groups of 16
// pieces, piece p of row r at position p ^ r inside its group: 16 rows' reads
// of one piece and one row's reads of 16 pieces both touch every bank once),
// then the rope rows (DR / 4 pieces, swizzled by row likewise). Wave w copies
// rows 4w .. 4w + 3.
template <int DV, int DR, int HG>
struct CfgF {
  static constexpr int NCL = DV / 64;   // latent k-chunks (16 dims) of a wave
  static constexpr int NRC = DR / 16;   // rope k-chunks; wave w takes chunk w
  static constexpr int VW = DV / 64;    // value dims per lane and token
  static constexpr int SLOTV = 16 * DV * 4, SLOTR = 16 * DR * 4, SLOT = SLOTV + SLOTR;
  static constexpr int XBYTES = HG * 4 * 1024;  // partial scores of the four waves
  // ring depth: four slices at 512 dims (one workgroup per CU; three where 32
  // heads leave no room), three below (two workgroups per CU)
  static constexpr int RING = DV == 512 && HG == 1 ? 4 : 3;
  static constexpr int OFF_X = RING * SLOT;
  static constexpr int SMEM = OFF_X + 2 * XBYTES;
  static constexpr int LOADS = NCL + 1;
};

template <int DV, int DR, int HG>
__global__ __launch_bounds__(256) void mla_dims_f32_kernel(DimsArgs a) {
  using C = CfgF<DV, DR, HG>;
  static_assert(C::SMEM <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
  char LDS_AS* const lds = (char LDS_AS*)(void LDS_AS*)smem;
  const bool paged = a.bt != nullptr;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, g = lane >> 4, n = lane & 15;
  const int head0 = blockIdx.y * 16 * HG;
  const CappedLens len_of{a.seqlens, a.len_cap};
  WorkRange wr;
  const int worker = worker_index(a);
  if (!work_range(a, len_of, worker, wr) || wr.tile_lo >= wr.tile_hi) return;
  const bool has_rope = wave < C::NRC;

  // K operand: row n, piece 4 (4j + wave) + g of the latent part (chunk 4j +
  // wave: 256-byte group j), and of the rope part (chunk `wave`)
  const int k_off = n * DV * 4 + (((4 * wave + g) ^ n) & 15) * 16;
  constexpr int NPR = DR / 4;
  const int k_rope = C::SLOTV + n * DR * 4 + (((4 * (has_rope ? wave : 0) + g) ^ (n / (16 / NPR))) & (NPR - 1)) * 16;
  // V operand: row 4g + s, this lane's VW dims of the wave's DV / 4: value
  // dims wave * DV / 4 + 64 D + F n + j (F = min(VW, 4) per read)
  constexpr int F = C::VW < 4 ? C::VW : 4;
  int v_off[4];
  {
    const int fl = wave * (DV / 4) + F * n;  // first float
    const int p = fl >> 2;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      v_off[s] = (4 * g + s) * DV * 4 + ((p & ~15) | ((p ^ (4 * g + s)) & 15)) * 16 + (fl & 3) * 4;
  }
  // copies of the wave's four rows: this lane's offsets from the slice's
  // first row where it lies in one page
  constexpr int PPR = DV / 4;  // latent pieces per row
  uint32_t c_off[C::NCL + 1];
#pragma unroll
  for (int j = 0; j < C::NCL; ++j) {
    const int P = 64 * j + lane, pos = P % PPR, row = 4 * wave + P / PPR;
    c_off[j] = (uint32_t)row * (uint32_t)a.kv_s1 + ((pos & ~15) | ((pos ^ row) & 15)) * 16;
  }
  {
    const int row = 4 * wave + ((lane / NPR) & 3);
    c_off[C::NCL] = (uint32_t)row * (uint32_t)a.kv_s1 + DV * 4 +
                    (((lane % NPR) ^ (row / (16 / NPR))) & (NPR - 1)) * 16;
  }

  int b = wr.b_first, t_start = wr.tile_lo, remaining = wr.tile_hi - wr.tile_lo, seg_off = wr.off_first;
  while (remaining > 0) {
    const int n_b = len_of(b);
    const int nt_b = tiles_of(n_b);
    if (nt_b == 0) {
      ++b;
      continue;
    }
    const int t_end = min(nt_b, t_start + remaining);
    const SegmentSlot ss = segment_slot(a, wr, worker, b, t_start, nt_b, seg_off);
    const int tok0 = t_start * kTileTokens, end = min(t_end * kTileTokens, n_b);
    const int slices = (end - tok0 + 15) / 16;
    const int32_t* bt_row = paged ? a.bt + (int64_t)b * a.bt_sb : nullptr;

    // (RING slices of 16 tokens past the end: within what kMaxGenericLen leaves)
    static_assert((C::RING + 2) * 16 <= INT32_MAX - kMaxGenericLen, "look-ahead");
    auto tok_of = [&](int sl, int row) __attribute__((always_inline)) { return min(tok0 + sl * 16 + row, end - 1); };
    // raw table entry of the slice's one page (a.uni: pages of whole slices),
    // else of row 4 * wave + lane % 4 of slice sl
    auto raw_page = [&](int sl) __attribute__((always_inline)) {
      int pg = 0;
      if (a.uni) {
        if (paged) pg = bt_row[page_slot_of(a, tok_of(sl, 0))];
      } else {
        if (paged) pg = bt_row[page_slot_of(a, tok_of(sl, 4 * wave + (lane & 3)))];
      }
      return pg;
    };
    // Copy j (of LOADS) of slice sl into its ring slot: from the slice's first
    // row (row0) where it is whole and in one page, else row by row (rows past
    // the piece read its last row again).
    auto row0_of = [&](int sl, int pg) __attribute__((always_inline)) -> const char* {
      const int t0 = tok0 + sl * 16;
      return a.uni && t0 + 16 <= end ? a.kv + row_off(a, paged, b, t0, __builtin_amdgcn_readfirstlane(pg)) : nullptr;
    };
    auto copy_one = [&](int sl, int pg, const char* row0, auto J) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value;
      constexpr bool rope = j == C::NCL;
      char LDS_AS* dst = lds + (sl % C::RING) * C::SLOT +
                         (rope ? C::SLOTV + wave * 4 * DR * 4 : wave * 4 * DV * 4 + j * 1024);
      const char* src;
      if (row0 != nullptr) {
        src = row0 + c_off[j];
      } else {
        const int rr = rope ? (lane / NPR) & 3 : (64 * j + lane) / PPR, row = 4 * wave + rr;
        const int raw = a.uni ? pg : __shfl(pg, rr);
        src = a.kv + row_off(a, paged, b, tok_of(sl, row), raw) + (int)(c_off[j] - (uint32_t)row * (uint32_t)a.kv_s1);
      }
      if (!rope || lane < 4 * NPR) lds_copy16<0>(src, dst);
    };
    auto issue = [&](int sl, int pg) __attribute__((always_inline)) {
      const char* row0 = row0_of(sl, pg);
      static_for<C::LOADS>([&](auto J) __attribute__((always_inline)) { copy_one(sl, pg, row0, J); });
    };

    f32x4 acc[HG][C::VW];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg)
#pragma unroll
      for (int d = 0; d < C::VW; ++d) acc[hg][d] = (f32x4)0.0f;
    float m_run[HG], l_run[HG];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
      m_run[hg] = kNoMax;
      l_run[hg] = 0.0f;
    }

    // start-up: the copies of slice 0, Q, the copies of the next slices
    int pg = raw_page(0), pn0 = raw_page(1);
    issue(0, pg);
    asm volatile("" ::: "memory");
    // Q^T operands: lane (head n, group g) holds dims 16c + 4g ..+3 of its
    // chunks, times scale * log2 e as the scores are base-2 exponents
    f32x4 qop[HG][C::NCL + 1];
#pragma unroll
    for (int hg = 0; hg < HG; ++hg) {
      const int head = head0 + 16 * hg + n;
      const float* qrow = reinterpret_cast<const float*>(a.q) + (int64_t)b * a.q_sb +
                          (int64_t)(head < a.num_heads ? head : 0) * a.q_sh + 4 * g;
#pragma unroll
      for (int j = 0; j < C::NCL; ++j)
        qop[hg][j] = *reinterpret_cast<const f32x4*>(qrow + 16 * (4 * j + wave)) * a.qk_scale_log2;
      qop[hg][C::NCL] = *reinterpret_cast<const f32x4*>(qrow + DV + 16 * (has_rope ? wave : 0)) * a.qk_scale_log2;
    }

    asm volatile("" ::: "memory");
    pg = pn0;
#pragma unroll 1
    for (int i = 1; i < C::RING - 1; ++i) {
      const int pn = raw_page(i + 1);
      asm volatile("" ::: "memory");
      issue(i, pg);
      pg = pn;
    }
#pragma unroll
    for (int hg = 0; hg < HG; ++hg)
#pragma unroll
      for (int j = 0; j <= C::NCL; ++j) tie_v(qop[hg][j]);
    wait_vmcnt<(C::RING - 2) * C::LOADS>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    lds_barrier();  // slice 0 is there

    // Partial scores of a slice over this wave's dims: the operand reads, then
    // NCL + 1 chunks of four MFMAs per head group in two accumulation chains;
    // hook(j) runs after chunk j.
    f32x4 kop[C::NCL + 1];
    auto k_reads = [&](int sl) __attribute__((always_inline)) {
      const char LDS_AS* p = lds + (sl % C::RING) * C::SLOT;
      static_for<C::NCL>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        kop[j] = __builtin_bit_cast(f32x4, ds_read_b128<j * 256>(p + k_off));
      });
      kop[C::NCL] = __builtin_bit_cast(f32x4, ds_read_b128<0>(p + k_rope));
    };
    auto k_mfma = [&](f32x4 (&s)[HG], auto&& hook) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i <= C::NCL; ++i) tie_v(kop[i]);
      f32x4 s1[HG];
#pragma unroll
      for (int hg = 0; hg < HG; ++hg) s[hg] = s1[hg] = (f32x4)0.0f;
      static_for<C::NCL + 1>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        if (j < C::NCL || has_rope) {
#pragma unroll
          for (int hg = 0; hg < HG; ++hg) {
            s[hg] = __builtin_amdgcn_mfma_f32_16x16x4f32(kop[j][0], qop[hg][j][0], s[hg], 0, 0, 0);
            s1[hg] = __builtin_amdgcn_mfma_f32_16x16x4f32(kop[j][1], qop[hg][j][1], s1[hg], 0, 0, 0);
            s[hg] = __builtin_amdgcn_mfma_f32_16x16x4f32(kop[j][2], qop[hg][j][2], s[hg], 0, 0, 0);
            s1[hg] = __builtin_amdgcn_mfma_f32_16x16x4f32(kop[j][3], qop[hg][j][3], s1[hg], 0, 0, 0);
          }
        }
        hook(J);
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int hg = 0; hg < HG; ++hg) s[hg] += s1[hg];
    };
    f32x4 s[HG];
    k_reads(0);
    lgkm<0>();
    k_mfma(s, [](auto) {});

    // Turn sl: the partial scores of slice sl meet; the score MFMAs of slice
    // sl + 1 run beside the softmax of slice sl and the copies of slice sl +
    // RING - 1, then the value MFMAs of slice sl. (The last turn's scores, of
    // rows past the piece, are not used.)
    for (int sl = 0; sl < slices; ++sl) {
      char LDS_AS* x = lds + C::OFF_X + (sl & 1) * C::XBYTES;
#pragma unroll
      for (int hg = 0; hg < HG; ++hg) ds_write_f4(x + (hg * 4 + wave) * 1024 + lane * 16, s[hg]);
      wait_vmcnt<(C::RING - 3) * C::LOADS>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      // every wave's scores of slice sl and copies of slice sl + 1 are there,
      // and every wave is done with slice sl - 1
      lds_barrier();
      const int pn = raw_page(sl + C::RING);
      const char* const row0 = row0_of(sl + C::RING - 1, pg);
      f32x4 sp[HG][4];
      static_for<HG * 4>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        sp[i / 4][i % 4] = __builtin_bit_cast(f32x4, ds_read_b128<i * 1024>(x + lane * 16));
      });
      k_reads(sl + 1);
      lgkm<C::NCL + 1>();
      f32x4 sc[HG];
      float mx[HG];
#pragma unroll
      for (int hg = 0; hg < HG; ++hg) {
#pragma unroll
        for (int w = 0; w < 4; ++w) tie_v(sp[hg][w]);
        sc[hg] = (sp[hg][0] + sp[hg][1]) + (sp[hg][2] + sp[hg][3]);
        const int t0 = tok0 + sl * 16 + 4 * g;
        if (tok0 + sl * 16 + 16 > end) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (t0 + r >= end) sc[hg][r] = -INFINITY;
        }
        mx[hg] = fmaxf(fmaxf(sc[hg][0], sc[hg][1]), fmaxf(sc[hg][2], sc[hg][3]));
      }
      const char LDS_AS* vp = lds + (sl % C::RING) * C::SLOT;
      constexpr int NV = C::VW > 4 ? C::VW / 4 : 1;  // reads per token
      typename VecF<F>::T vop[4][NV];
      static_for<4>([&](auto S) __attribute__((always_inline)) {
        constexpr int si = decltype(S)::value;
        static_for<NV>([&](auto D) __attribute__((always_inline)) {
          constexpr int d = decltype(D)::value;
          vop[si][d] = ds_read_f<F, d * 256>(vp + v_off[si]);
        });
      });
      lgkm<4 * NV>();
      k_mfma(s, [&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        constexpr int M = C::NCL > 2 ? 1 : 0;  // the reference max after chunk M, exponentials from chunk M + 1 on
        if constexpr (j == M) {
#pragma unroll
          for (int hg = 0; hg < HG; ++hg) {
            if (__builtin_amdgcn_ballot_w64(mx[hg] > m_run[hg] + kRescaleLog2) != 0) {
              float p = mx[hg], q = mx[hg];
              swap_rows16(p, q);
              p = fmaxf(p, q);
              q = p;
              swap_rows32(p, q);
              const float m_new = fmaxf(m_run[hg], fmaxf(p, q));
              if (m_run[hg] != kNoMax) {
                const float f = exp2f(m_run[hg] - m_new);
                l_run[hg] *= f;
#pragma unroll
                for (int d = 0; d < C::VW; ++d) acc[hg][d] *= f;
              }
              m_run[hg] = m_new;
            }
          }
        }
        constexpr int E0 = M + 1, SPAN = C::NCL - M;  // chunks E0 .. NCL take the four tokens' exponentials
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if constexpr (j >= E0) {
            if ((r < SPAN ? r : SPAN - 1) + E0 == j) {
#pragma unroll
              for (int hg = 0; hg < HG; ++hg) {
                sc[hg][r] = exp2f(sc[hg][r] - m_run[hg]);
                l_run[hg] += sc[hg][r];
              }
            }
          }
        copy_one(sl + C::RING - 1, pg, row0, J);
      });
      pg = pn;
      lgkm<0>();
#pragma unroll
      for (int si = 0; si < 4; ++si)
#pragma unroll
        for (int d = 0; d < NV; ++d) tie_v(vop[si][d]);
      // tokens 4g + si are k-step si of both operands
#pragma unroll
      for (int si = 0; si < 4; ++si)
#pragma unroll
        for (int d = 0; d < C::VW; ++d)
#pragma unroll
          for (int hg = 0; hg < HG; ++hg)
            acc[hg][d] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(elem<F>(vop[si][d / 4], d % 4), sc[hg][si], acc[hg][d], 0, 0, 0);
    }
    wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    lds_barrier();  // the next segment refills the ring

    // ---- rows out: lane (g, head n) holds dims 64 D + F (4g + r) + j -------
    {
      const RowTarget tgt = row_target(a, ss, b, DV, 4);
#pragma unroll
      for (int hg = 0; hg < HG; ++hg) {
        const int head = head0 + 16 * hg + n;
        float p = l_run[hg], q = l_run[hg];
        swap_rows16(p, q);
        p += q;
        q = p;
        swap_rows32(p, q);
        const float l = p + q;
        const bool has = l > 0.0f;
        const float inv = has ? 1.0f / l : 0.0f;
        if (head < a.num_heads) {
          float* dst = (tgt.direct ? reinterpret_cast<float*>(tgt.out) + (int64_t)head * tgt.out_sh
                                   : tgt.part + (int64_t)head * DV) +
                       wave * (DV / 4) + F * 4 * g;
          constexpr int NQ = C::VW > 4 ? C::VW / 4 : 1;
#pragma unroll
          for (int d = 0; d < NQ; ++d)
#pragma unroll
            for (int i = 0; i < F; ++i) {  // dims 4i .. 4i + 3 of the lane's 4F
              f32x4 v;
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = acc[hg][4 * d + (4 * i + e) % F][(4 * i + e) / F] * inv;
              *reinterpret_cast<f32x4*>(dst + 64 * d + 4 * i) = v;
            }
          if (wave == 0 && g == 0) {
            if (tgt.direct) {
              if (tgt.lse) tgt.lse[head] = has ? (m_run[hg] + log2f(l)) * kLn2 : -INFINITY;
            } else {
              tgt.plse[head] = has ? m_run[hg] + log2f(l) : -INFINITY;
            }
          }
        }
      }
    }
    remaining -= t_end - t_start + wr.seg_cost;
    seg_off += nt_b + wr.seg_cost;
    ++b;
    t_start = 0;
  }
}

// ---------------------------------------------------------------------------
// Merge of the float32 partials: a wave per (sequence, head), up to eight
// slots' rows in flight, summed in slot order.
// ---------------------------------------------------------------------------
template <int DT, int DV>
__global__ __launch_bounds__(256) void mla_dims_combine_kernel(DimsArgs a) {
  constexpr int E = DV / 64;  // dims per lane
  constexpr int NB = 8;
  constexpr int VE = E < 4 ? E : 4, NV = E / VE;
  typedef typename VecF<VE>::T vec;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = blockIdx.x, head = blockIdx.y * 4 + wave;
  int slot0, count;
  sequence_slots(CappedLens{a.seqlens, a.len_cap}, a.batch, a.num_splits, a.num_workers, b, slot0, count);
  if (count == 1 || head >= a.num_heads) return;
  const float* ml = a.part_lse + (int64_t)slot0 * a.num_heads + head;
  const float* mo = a.part + ((int64_t)slot0 * a.num_heads + head) * DV + lane * VE;
  const int64_t step = (int64_t)a.num_heads * DV;
  float m = -INFINITY;
  for (int s = lane; s < count; s += 64) m = fmaxf(m, ml[(int64_t)s * a.num_heads]);
  for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
  if (m == -INFINITY) m = 0.0f;
  float acc[E], wsum = 0.0f;
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = 0.0f;
  for (int s0 = 0; s0 < count; s0 += NB) {
    float w[NB];
    vec v[NB][NV];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int s = min(s0 + j, count - 1);
      w[j] = ml[(int64_t)s * a.num_heads];
#pragma unroll
      for (int k = 0; k < NV; ++k) v[j][k] = *reinterpret_cast<const vec*>(mo + s * step + 64 * VE * k);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const bool ok = s0 + j < count;  // (slots past the last repeat it, not counted)
      const float f = exp2f(w[j] - m);
      wsum += ok ? f : 0.0f;
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] = ok ? fmaf(f, elem<VE>(v[j][e / VE], e % VE), acc[e]) : acc[e];
    }
  }
  const float inv = wsum > 0.0f ? 1.0f / wsum : 1.0f;
  const int64_t row = (int64_t)b * a.out_sb + (int64_t)head * a.out_sh;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    typedef typename std::conditional<DT == TMLA_FP32, float, short>::type elt;
    struct alignas(sizeof(elt) * VE) Row {
      elt e[VE];
    } o;
#pragma unroll
    for (int e = 0; e < VE; ++e) {
      if constexpr (DT == TMLA_FP32)
        o.e[e] = acc[k * VE + e] * inv;
      else
        o.e[e] = Elt<DT>::from_float(acc[k * VE + e] * inv);
    }
    *reinterpret_cast<Row*>(reinterpret_cast<elt*>(a.out) + row + 64 * VE * k + lane * VE) = o;
  }
  if (lane == 0 && a.lse)
    a.lse[(int64_t)b * a.num_heads + head] = wsum > 0.0f ? (m + log2f(wsum)) * kLn2 : -INFINITY;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <int DT, int DV, int DR>
void launch16(const DimsArgs& a, dim3 grid, hipStream_t st) {
  if constexpr (DV == 512)
    hipLaunchKernelGGL((mla_dims512_kernel<DT, DV, DR>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((mla_dims_kernel<DT, DV, DR>), grid, dim3(512), 0, st, a);
}
template <int DV, int DR>
void launch32(const DimsArgs& a, dim3 grid, int hg, hipStream_t st) {
  if (hg == 1)
    hipLaunchKernelGGL((mla_dims_f32_kernel<DV, DR, 1>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((mla_dims_f32_kernel<DV, DR, 2>), grid, dim3(256), 0, st, a);
}
template <int DV, int DR>
void launch_dr(const DimsArgs& a, int dtype, dim3 grid, int hg, hipStream_t st) {
  if (dtype == TMLA_FP32)
    launch32<DV, DR>(a, grid, hg, st);
  else if (dtype == TMLA_BF16)
    launch16<TMLA_BF16, DV, DR>(a, grid, st);
  else
    launch16<TMLA_FP16, DV, DR>(a, grid, st);
}
template <int DV>
void launch_dv(const DimsArgs& a, int dtype, int dr, dim3 grid, int hg, hipStream_t st) {
  switch (dr) {
    case 16: return launch_dr<DV, 16>(a, dtype, grid, hg, st);
    case 32: return launch_dr<DV, 32>(a, dtype, grid, hg, st);
    default: return launch_dr<DV, 64>(a, dtype, grid, hg, st);
  }
}
template <int DV>
void launch_combine(const DimsArgs& a, int dtype, hipStream_t st) {
  const dim3 grid(a.batch, (a.num_heads + 3) / 4);
  if (dtype == TMLA_FP32)
    hipLaunchKernelGGL((mla_dims_combine_kernel<TMLA_FP32, DV>), grid, dim3(256), 0, st, a);
  else if (dtype == TMLA_BF16)
    hipLaunchKernelGGL((mla_dims_combine_kernel<TMLA_BF16, DV>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((mla_dims_combine_kernel<TMLA_FP16, DV>), grid, dim3(256), 0, st, a);
}

hipError_t launch(const DimsArgs& a, int dv, int dr, int dtype, int64_t capacity_tokens, hipStream_t st) {
  const int heads_per_wg = dims_heads_per_workgroup(dtype, a.num_heads);
  const dim3 grid(worker_grid(a.batch, a.num_splits, a.num_workers, capacity_tokens),
                  (a.num_heads + heads_per_wg - 1) / heads_per_wg);
  const int hg = heads_per_wg / 16;  // (float32)
  switch (dv) {
    case 64: launch_dv<64>(a, dtype, dr, grid, hg, st); break;
    case 128: launch_dv<128>(a, dtype, dr, grid, hg, st); break;
    case 256: launch_dv<256>(a, dtype, dr, grid, hg, st); break;
    default: launch_dv<512>(a, dtype, dr, grid, hg, st); break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  switch (dv) {
    case 64: launch_combine<64>(a, dtype, st); break;
    case 128: launch_combine<128>(a, dtype, st); break;
    case 256: launch_combine<256>(a, dtype, st); break;
    default: launch_combine<512>(a, dtype, st); break;
  }
  return hipGetLastError();
}

}  // namespace dims
}  // namespace tmla
