// flash_attn.hip — unmasked multi-head attention over contiguous [B, H, T, 64] fp16 / bf16
// tensors: out = softmax(scale * q k^T) v per (batch, head).  This is the audio tower's
// self-attention (Qwen3-ASR-0.6B: 14 heads of 64 dims, T ~ 1500 frames), the operation of
// flash_attn_bhwd (megaqwen/triton_flash_attn.py:27-171, kernel body :63-129).
//
// Organisation (gfx950, v_mfma_f32_32x32x16_{bf16,f16}, fp32 accumulation):
//   * a workgroup is 32 or 64 queries of one (batch * head), XCD-major (see the item mapping in
//     the kernel); its 4 waves split the key tiles (32 keys each) into contiguous ranges and merge
//     their (max, sum, O) partials through LDS at the end;
//   * S^T = K Q^T: rows are keys, so each lane holds the scores of ONE query (lanes l and l+32
//     split its 32 keys), and the softmax max / sum need one lane swap;
//   * K tile row r carries key fa_key_perm(r) (bits 2 and 3 of r swapped).  That makes score
//     accumulator element j of lane l the key 16 (j / 8) + 8 (l / 32) + j % 8, which is the
//     B-operand layout of two 16-key MFMA steps: O^T += V^T P^T takes P^T from registers;
//   * each wave copies its K and V tiles from the [T, 64] tensors to LDS (4 KB of contiguous
//     memory each) and takes its operands from there, V^T by transposing LDS reads.  Operand
//     loads straight from the rows would touch 16-32 cache lines each; an operand-order copy of K
//     and V made by a kernel in front cost 4.7 us and a launch of a 27 us call;
//   * the scores are exact fp32 dot products of the 16-bit inputs (up to accumulation order),
//     the softmax is fp32, and P enters the MFMA as a hi + lo pair of the input type (two
//     MFMAs), ~16 bits more than one rounding of P; the output is o / l rounded to nearest-even
//     in the input type (triton_flash_attn.py:126-127).
// What bounds it: a (32 queries, 32 keys) unit is 12 MFMAs (384 matrix cycles) and ~105 VALU
// instructions, 16 of them exponentials, which a SIMD issues in ~480 cycles; a loop of just that
// mix, interleaved, runs 550-600 cycles per unit.  The matrix products of one unit are therefore
// interleaved with the weights of another.  Neither shape below reaches that loop:
//   14 heads, T = 1500, bf16 (25.4 -> 20.8 us per call): one round of 658 workgroups, ~30 units per
//     SIMD; 19% MFMA-busy, the waves wait on memory for 28% of their cycles (a tile is copied half a
//     unit before the wait for it) and issue in 35%;
//   4 x 14 heads, T = 3000, fp16 (271 -> 226 us): 43% MFMA-busy, ~910 cycles per unit at 1.9 GHz, a
//     seventh of them because 2632 workgroups are 5.14 rounds run as 6.
// Keys >= T (the last tile) get score -inf and zero V^T entries; queries >= T read row T-1 and
// store nothing.  All accesses stay inside the tensors.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mq_device.h"
#include "mq_flash.h"

#define FA_D 64           // head dim
#define FA_KT 32          // keys per tile
#define FA_WAVES 4        // waves per workgroup (split of the key tiles)
// N groups of one MFMA followed by V VALU instructions
#define FA_INTERLEAVE(N, V)                              \
  _Pragma("unroll") for (int z = 0; z < (N); ++z) {      \
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     \
    __builtin_amdgcn_sched_group_barrier(0x2, (V), 0);   \
  }
#define FA_RESCALE 8.0f   // exponent headroom of the lazily raised softmax reference point

typedef float fa_f32x16 __attribute__((ext_vector_type(16)));
typedef float fa_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 fa_bf16x2 __attribute__((ext_vector_type(2)));

template <bool F16> struct FaType;
template <> struct FaType<false> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  typedef __bf16 scalar;
  static __device__ __forceinline__ fa_f32x16 mfma(v8 a, v8 b, fa_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct FaType<true> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 scalar;
  static __device__ __forceinline__ fa_f32x16 mfma(v8 a, v8 b, fa_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

MQ_DEV int fa_key_perm(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

template <bool F16> MQ_DEV uint32_t fa_pack2(float a, float b) {
  if constexpr (F16) {
    const _Float16 ha = (_Float16)a, hb = (_Float16)b;
    return (uint32_t)__builtin_bit_cast(uint16_t, ha) |
           ((uint32_t)__builtin_bit_cast(uint16_t, hb) << 16);
  } else {
    return (uint32_t)f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16);
  }
}

// Largest (HI) or smallest of two raw scores
template <bool HI> MQ_DEV float fa_extreme(float a, float b) {
  if constexpr (HI) return __builtin_elementwise_maximum(a, b);
  else return __builtin_elementwise_minimum(a, b);
}

// Two weights as packed 16-bit hi parts (truncated, so that lo is never negative) and lo parts (the
// exact remainder p - hi, rounded once).  An infinite v gives an infinite output where lo is not 0;
// where the weight is exact in 16 bits (T = 1, say) lo is 0 and the output NaN.
// The remainder is one instruction per weight: a two-element dot product of the packed
// hi pair with (-1, 0) or (0, -1) plus p, or a mixed-precision fma for fp16.
template <bool F16> MQ_DEV void fa_split2(float p0, float p1, uint32_t& hi, uint32_t& lo) {
  if constexpr (F16) {
    const auto h = __builtin_amdgcn_cvt_pkrtz(p0, p1);
    const auto r = __builtin_amdgcn_cvt_pkrtz(fmaf((float)h[0], -1.0f, p0), fmaf((float)h[1], -1.0f, p1));
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, r);
  } else {
    const uint32_t hw =
        __builtin_amdgcn_perm(__float_as_uint(p1), __float_as_uint(p0), 0x07060302u);
    const fa_bf16x2 h = __builtin_bit_cast(fa_bf16x2, hw);
    // (-1, 0) and (0, -1) in scalar registers the compiler cannot see through: as a constant it
    // encodes (-1, 0) as the inline operand -1.0, which the hardware reads as the pair (0, -1)
    uint32_t c0 = 0x0000bf80u, c1 = 0xbf800000u;
    asm("" : "+s"(c0), "+s"(c1));
    const fa_f32x2 r = {
        __builtin_amdgcn_fdot2_f32_bf16(h, __builtin_bit_cast(fa_bf16x2, c0), p0, false),
        __builtin_amdgcn_fdot2_f32_bf16(h, __builtin_bit_cast(fa_bf16x2, c1), p1, false)};
    hi = hw;
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, fa_bf16x2));
  }
}

// Chunk of 8 values (16 bytes) c of row r in a 32-row LDS tile of 64 16-bit values per row: the
// chunks of a row are permuted so that the operand reads of 8 (K) or 4 (V) consecutive rows at one
// dim offset fall into different banks.
MQ_DEV int fa_k_slot(int r, int c) { return 8 * r + (c ^ (r & 7)); }
MQ_DEV int fa_v_slot(int r, int c) { return 8 * r + (c ^ ((r & 2) << 1) ^ ((r & 1) << 1)); }

typedef short fa_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) fa_s16x4* fa_lds_s16x4;

// One workgroup: 32 QN queries of one (batch * head); its 4 waves split the key tiles.
// CPOS: the scale is >= 0 (the softmax max is taken over the raw scores; otherwise their min),
// a compile-time choice so that a tile carries neither the other extreme nor selects between them
template <bool F16, bool CPOS, int QN>
__global__ void __launch_bounds__(64 * FA_WAVES, QN == 1 ? 3 : 2)
fa_bhwd_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
               const uint16_t* __restrict__ v, uint16_t* __restrict__ out, int T,
               float scale_log2, int nqb, int items, int per_xcd) {
  typedef FaType<F16> Ty;
  typedef typename Ty::v8 v8;
  // LDS: each wave's K and V tile (no other wave reads them) during the key loop; the waves'
  // partials (o: 32 per lane, m, l, per 32-query block) afterwards.
  union FaLds {
    struct {
      uint4 k[FA_WAVES][256], v[FA_WAVES][256];
    } loop;
    float red[FA_WAVES][QN][34][64];
  };
  __shared__ __attribute__((aligned(16))) FaLds lds;

  // Work item = (batch * head, query block), head-major.  Workgroups are dealt to the 8 XCDs
  // round robin (linear id % 8), so XCD x is given the contiguous items [x * per_xcd, ..): the
  // workgroups resident on one XCD share one or two heads' K and V, which its L2 then holds,
  // instead of every XCD streaming every head's K and V from HBM once per query block.
  const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (item >= items) return;                       // grid padding (uniform per workgroup)
  const int bh = item / nqb, qb = item - bh * nqb;
  // the wave index in a scalar register: the tile loop, its addresses and branches are scalar
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 31, hh = lane >> 5;
  const size_t base = (size_t)bh * T * FA_D;
  const int q0 = qb * 32 * QN;
  const int ntiles = (T + FA_KT - 1) / FA_KT;
  const int t0 = ntiles * wave / FA_WAVES, t1 = ntiles * (wave + 1) / FA_WAVES;

  // Q^T operands: query q0 + 32 i + lane % 32 (rows >= T read row T - 1, never stored), dims
  // 16 s + 8 (lane / 32) .. + 8
  uint4 qf[QN][4];
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    const uint16_t* src = q + base + (size_t)min(q0 + 32 * i + fr, T - 1) * FA_D + 8 * hh;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[i][s] = ld16(src + 16 * s);
  }

  uint4* kl = lds.loop.k[wave];
  uint4* vl = lds.loop.v[wave];
  // A tile's K or V rows are 4 KB of contiguous memory.  They go straight to LDS, 16 bytes per
  // lane: lane i lands at chunk i of each 1 KB, so it fetches the chunk that belongs there (the
  // chunk permutation of a row is its own inverse).  Buffer loads with the size of the tile's
  // existing rows: rows >= T are written as 0 without an access.
  const int r8 = lane >> 3, c8 = lane & 7;
  const int koff = 16 * fa_k_slot(r8, c8), voff = 16 * fa_v_slot(r8, c8);
  auto dma = [&](int t, const uint16_t* src, uint4* dst, int off) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(src + base + (size_t)t * (FA_KT * FA_D)), (short)0,
        min(T - t * FA_KT, FA_KT) * FA_D * 2, 0x00020000);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r, (__attribute__((address_space(3))) void*)(dst + 64 * c), 16, off + 1024 * c, 0, 0, 0);
  };
  auto lds_reads_done = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  // K operand: tile row fr holds key fa_key_perm(fr), dims 16 s + 8 hh .. + 8
  uint4 kr[4];
  auto read_k = [&]() {
#pragma unroll
    for (int s = 0; s < 4; ++s) kr[s] = kl[fa_k_slot(fa_key_perm(fr), 2 * s + hh)];
  };
  // V^T operand (nt, s): dim 32 nt + fr, keys 16 s + 8 hh + e, e = 0..7, by two transposing reads
  // of 4 keys: in each group of 16 lanes, lane x addresses dims 4 (x % 4) .. + 4 (of the group's
  // 16) of key x / 4 and receives dim x of the group's 4 keys
  uint2 vr[2][2][2];
  auto read_v = [&]() {
    const int key = 8 * hh + ((lane >> 2) & 3), dim = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int row = 16 * s + 4 * h + key, d = 32 * nt + dim;
          const uint16_t* a = reinterpret_cast<const uint16_t*>(vl + fa_v_slot(row, d >> 3)) + (d & 7);
          vr[nt][s][h] = __builtin_bit_cast(
              uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4)a));
        }
  };

  fa_f32x16 o[QN][2];
  // m: the reference point of the exponentials (log2 units), raised only when a score exceeds
  // it by more than FA_RESCALE (every weight is <= 2^FA_RESCALE, and o, l are rescaled rarely
  // instead of at every new maximum); l: the sum of the weights
  float m[QN], l[QN];
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int j = 0; j < 16; ++j) o[i][nt][j] = 0.f;
  }
  // S^T of query block i and the tile whose K operand is in kr
  auto scores = [&](const uint4 (&qq)[4]) {
    fa_f32x16 acc;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = Ty::mfma(__builtin_bit_cast(v8, kr[s]), __builtin_bit_cast(v8, qq[s]), acc);
    return acc;
  };
  // Scaled extreme of a query's 32 scores.  max_j (s_j * c) is max_j(s_j) * c for c >= 0 and
  // min_j(s_j) * c for c < 0 (rounding is monotonic), so the extreme is taken over the raw
  // scores.  maximum / minimum (which return NaN for a NaN score) are one v_maximum3_f32 per two
  // scores; fmaxf costs a canonicalising v_max_f32 per operand on top.  A NaN score makes its
  // weight, the row sum and the output NaN either way.
  auto extreme = [&](const fa_f32x16& sv) {
    float mr = fa_extreme<CPOS>(sv[0], sv[1]);
#pragma unroll
    for (int j = 2; j < 16; j += 2) mr = fa_extreme<CPOS>(fa_extreme<CPOS>(mr, sv[j]), sv[j + 1]);
    const float2 pr = swap32(mr);
    return fa_extreme<CPOS>(pr.x, pr.y) * scale_log2;
  };
  // P of the last finished unit, as hi + lo 16-bit parts in B-operand order
  uint32_t ph[8], pl[8];
  auto pv = [&](fa_f32x16 (&oo)[2]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const v8 bh_ = __builtin_bit_cast(v8, make_uint4(ph[4 * s], ph[4 * s + 1], ph[4 * s + 2], ph[4 * s + 3]));
      const v8 bl_ = __builtin_bit_cast(v8, make_uint4(pl[4 * s], pl[4 * s + 1], pl[4 * s + 2], pl[4 * s + 3]));
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const v8 vb = __builtin_bit_cast(v8, make_uint4(vr[nt][s][0].x, vr[nt][s][0].y,
                                                        vr[nt][s][1].x, vr[nt][s][1].y));
        oo[nt] = Ty::mfma(vb, bh_, oo[nt]);
        oo[nt] = Ty::mfma(vb, bl_, oo[nt]);
      }
    }
  };

  // The loop runs over units (key tile, query block).  While the VALU computes unit u's weights,
  // the matrix cores run unit u + 1's scores and unit u - 1's O^T update, which are independent
  // of it; sv is unit u's scores and mt their scaled extreme.
  fa_f32x16 sv;
  float mt;
  auto rescale = [&](float& mi, float& li, fa_f32x16 (&oo)[2]) {
    if (__builtin_amdgcn_ballot_w64(mt > mi + FA_RESCALE) != 0) {
      const float m_new = mt > mi + FA_RESCALE ? mt : mi;
      // (an unraised lane keeps its sums as they are: m may still be -inf there)
      const float alpha = mt > mi + FA_RESCALE ? __builtin_amdgcn_exp2f(mi - m_new) : 1.0f;
      mi = m_new;
      li *= alpha;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int j = 0; j < 16; ++j) oo[nt][j] *= alpha;
    }
  };
  // weights of words [W0, W1) of a unit: p = 2^(s c - m), summed into ls and split
  auto weights = [&](const fa_f32x16& x, float mi, float (&ls)[2], uint32_t (&h)[8],
                     uint32_t (&lo)[8], auto w0_tag, auto w1_tag) {
#pragma unroll
    for (int w = decltype(w0_tag)::value; w < decltype(w1_tag)::value; ++w) {
      const float p0 = __builtin_amdgcn_exp2f(fmaf(x[2 * w], scale_log2, -mi));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(x[2 * w + 1], scale_log2, -mi));
      ls[0] += p0;
      ls[1] += p1;
      fa_split2<F16>(p0, p1, h[w], lo[w]);
      asm volatile("" : "+v"(h[w]), "+v"(lo[w]));
    }
    asm volatile("" : "+v"(ls[0]), "+v"(ls[1]));
  };
  if constexpr (QN == 1) {
    float alpha = 1.0f;
    bool pend = false;               // the last unit raised m: o is still to be scaled by alpha
    if (t0 < t1) {
      dma(t0, k, kl, koff);
      read_k();
      lds_reads_done();
      dma(min(t0 + 1, t1 - 1), k, kl, koff);
      // the first unit's O^T update (of no unit before it) multiplies zeros
#pragma unroll
      for (int c = 0; c < 4; ++c) vl[lane + 64 * c] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int w = 0; w < 8; ++w) ph[w] = pl[w] = 0u;
      sv = scores(qf[0]);
      mt = extreme(sv);
      auto unit = [&](int t, auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        if (LAST && t == ntiles - 1 && T % FA_KT != 0) {
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (t * FA_KT + 16 * (j >> 3) + 8 * hh + (j & 7) >= T) sv[j] = CPOS ? -INFINITY : INFINITY;
          mt = extreme(sv);
        }
        // o lags one unit behind m and l: the O^T update of unit t - 1 runs below
        if (pend) {
#pragma unroll
          for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int j = 0; j < 16; ++j) o[0][nt][j] *= alpha;
        }
        asm volatile("" : "+v"(o[0][0]), "+v"(o[0][1]));
        pend = __builtin_amdgcn_ballot_w64(mt > m[0] + FA_RESCALE) != 0;
        if (pend) {
          const float m_new = mt > m[0] + FA_RESCALE ? mt : m[0];
          alpha = mt > m[0] + FA_RESCALE ? __builtin_amdgcn_exp2f(m[0] - m_new) : 1.0f;
          m[0] = m_new;
          l[0] *= alpha;
        }
        float ls[2] = {0.f, 0.f};
        uint32_t nh[8], nl[8];
        fa_f32x16 snext;
        if (!LAST) read_k();
        read_v();
        __builtin_amdgcn_sched_barrier(0);
        if (!LAST) snext = scores(qf[0]);
        weights(sv, m[0], ls, nh, nl, std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
        FA_INTERLEAVE(4, 8)
        __builtin_amdgcn_sched_barrier(0);
        // both LDS tiles are in registers: their buffers take the next tiles
        lds_reads_done();
        if (!LAST) dma(min(t + 2, t1 - 1), k, kl, koff);
        dma(t, v, vl, voff);
        pv(o[0]);
        weights(sv, m[0], ls, nh, nl, std::integral_constant<int, 3>{}, std::integral_constant<int, 8>{});
        FA_INTERLEAVE(8, 6)
        __builtin_amdgcn_sched_barrier(0);
        l[0] += ls[0] + ls[1];
        asm volatile("" : "+v"(o[0][0]), "+v"(o[0][1]));
#pragma unroll
        for (int w = 0; w < 8; ++w) {
          ph[w] = nh[w];
          pl[w] = nl[w];
        }
        if (!LAST) {
          sv = snext;
          mt = extreme(sv);
        }
      };
      int t = t0;
      for (; t + 1 < t1; ++t) unit(t, std::false_type{});
      unit(t, std::true_type{});
      if (pend) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int j = 0; j < 16; ++j) o[0][nt][j] *= alpha;
      }
      read_v();
      pv(o[0]);
    }
  } else if (t0 < t1) {
    dma(t0, k, kl, koff);
    dma(t0, v, vl, voff);
    read_k();
    lds_reads_done();
    dma(min(t0 + 1, t1 - 1), k, kl, koff);
#pragma unroll
    for (int w = 0; w < 8; ++w) ph[w] = pl[w] = 0u;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int s = 0; s < 2; ++s) vr[nt][s][0] = vr[nt][s][1] = make_uint2(0u, 0u);
    sv = scores(qf[0]);
    mt = extreme(sv);
    // One unit: query block I of tile t.  LAST: the wave's last tile, the only one that may hold
    // keys >= T (their scores become -inf) and after which no tile follows.
    auto unit = [&](int t, auto itag, auto last_tag) {
      constexpr int I = decltype(itag)::value;
      constexpr bool LAST = decltype(last_tag)::value;
      if (LAST && t == ntiles - 1 && T % FA_KT != 0) {
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (t * FA_KT + 16 * (j >> 3) + 8 * hh + (j & 7) >= T) sv[j] = CPOS ? -INFINITY : INFINITY;
        mt = extreme(sv);
      }
      rescale(m[I], l[I], o[I]);
#pragma unroll
      for (int z = 0; z < QN; ++z) asm volatile("" : "+v"(o[z][0]), "+v"(o[z][1]));
      // Scheduled by hand: the scores of the next unit with the first weights, then the O^T update
      // with the rest, then the next unit's extreme, by when its scores are complete.
      float ls[2] = {0.f, 0.f};
      uint32_t nh[8], nl[8];
      fa_f32x16 snext;
      __builtin_amdgcn_sched_barrier(0);
      if (!LAST || I < QN - 1) snext = scores(qf[(I + 1) % QN]);
      weights(sv, m[I], ls, nh, nl, std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
      FA_INTERLEAVE(4, 8)
      __builtin_amdgcn_sched_barrier(0);
      if (!LAST && I == QN - 2) read_k();
      pv(o[(I + QN - 1) % QN]);
      weights(sv, m[I], ls, nh, nl, std::integral_constant<int, 3>{}, std::integral_constant<int, 8>{});
      FA_INTERLEAVE(8, 6)
      __builtin_amdgcn_sched_barrier(0);
      if (I == 0) {
        read_v();
        if (!LAST) {
          lds_reads_done();
          dma(min(t + 2, t1 - 1), k, kl, koff);
          dma(t + 1, v, vl, voff);
        }
      }
      l[I] += ls[0] + ls[1];
#pragma unroll
      for (int z = 0; z < QN; ++z) asm volatile("" : "+v"(o[z][0]), "+v"(o[z][1]));
#pragma unroll
      for (int w = 0; w < 8; ++w) {
        ph[w] = nh[w];
        pl[w] = nl[w];
      }
      if (!LAST || I < QN - 1) {
        sv = snext;
        mt = extreme(sv);
      }
    };
    auto tile_units = [&](int t, auto last_tag) {
      unit(t, std::integral_constant<int, 0>{}, last_tag);
      unit(t, std::integral_constant<int, 1>{}, last_tag);
    };
    int t = t0;
    for (; t + 1 < t1; ++t) tile_units(t, std::false_type{});
    tile_units(t, std::true_type{});
    pv(o[QN - 1]);
  }

  // Merge of the key ranges: every wave leaves its partials (o, m, l) in LDS and merges a quarter
  // of the dims (8 of the 32 accumulator elements) of every query, in wave order.  A wave
  // without tiles has m = -inf and adds 0; at least one wave has a tile, so the common max is
  // finite.
  __syncthreads();                                 // every wave is done with its tiles
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    float* r = &lds.red[wave][i][0][lane];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int j = 0; j < 16; ++j) r[(16 * nt + j) * 64] = o[i][nt][j];
    r[32 * 64] = m[i];
    r[33 * 64] = l[i];
  }
  __syncthreads();
  static_assert(FA_WAVES == 4, "a wave merges 8 of the 32 accumulator elements");
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    float a[FA_WAVES], mx = -INFINITY, lt = 0.f;
#pragma unroll
    for (int w = 0; w < FA_WAVES; ++w) {
      a[w] = lds.red[w][i][32][lane];
      mx = fmaxf(mx, a[w]);
    }
#pragma unroll
    for (int w = 0; w < FA_WAVES; ++w) {
      a[w] = __builtin_amdgcn_exp2f(a[w] - mx);
      lt = fmaf(lds.red[w][i][33][lane], a[w], lt);
    }
    const float inv = 1.0f / sum_xor32(lt);        // lanes l, l+32 summed different keys
    float r8v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      r8v[j] = 0.f;
#pragma unroll
      for (int w = 0; w < FA_WAVES; ++w)
        r8v[j] = fmaf(lds.red[w][i][8 * wave + j][lane], a[w], r8v[j]);
    }
    const int qi = q0 + 32 * i + fr;
    if (qi < T) {
      // O^T accumulator element j of tile nt: dim 32 nt + 8 (j / 4) + 4 hh + j % 4
      uint16_t* dst = out + base + (size_t)qi * FA_D + 16 * wave + 4 * hh;
#pragma unroll
      for (int jg = 0; jg < 2; ++jg) {
        uint2 w;
        w.x = fa_pack2<F16>(r8v[4 * jg] * inv, r8v[4 * jg + 1] * inv);
        w.y = fa_pack2<F16>(r8v[4 * jg + 2] * inv, r8v[4 * jg + 3] * inv);
        *reinterpret_cast<uint2*>(dst + 8 * jg) = w;
      }
    }
  }
}

size_t mq_flash_attn_workspace(int bh, int T) {
  return (size_t)2 * bh * ((T + FA_KT - 1) / FA_KT) * FA_KT * FA_D * 2;
}

template <int QN>
static bool fa_launch(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* out,
                      int bh, int T, bool f16, float scale_log2, hipStream_t stream) {
  const int nqb = (int)(((long long)T + 32 * QN - 1) / (32 * QN));
  const long long items = (long long)nqb * bh, per = (items + 7) / 8;
  if (8 * per > 0x7fffffffLL) return false;
  const dim3 grid((unsigned)(8 * per)), block(64 * FA_WAVES);
  const bool cpos = scale_log2 >= 0.f;
  if (f16 && cpos)
    hipLaunchKernelGGL((fa_bhwd_kernel<true, true, QN>), grid, block, 0, stream, q, k, v, out, T,
                       scale_log2, nqb, (int)items, (int)per);
  else if (f16)
    hipLaunchKernelGGL((fa_bhwd_kernel<true, false, QN>), grid, block, 0, stream, q, k, v, out, T,
                       scale_log2, nqb, (int)items, (int)per);
  else if (cpos)
    hipLaunchKernelGGL((fa_bhwd_kernel<false, true, QN>), grid, block, 0, stream, q, k, v, out, T,
                       scale_log2, nqb, (int)items, (int)per);
  else
    hipLaunchKernelGGL((fa_bhwd_kernel<false, false, QN>), grid, block, 0, stream, q, k, v, out, T,
                       scale_log2, nqb, (int)items, (int)per);
  return true;
}

int mq_launch_flash_attn_bhwd(const void* q, const void* k, const void* v, void* out, int bh,
                              int T, bool f16, float scale_log2, hipStream_t stream) {
  // scale 0: every weight 1.  The smallest denormal gives that for every finite score and keeps
  // the masked keys' -inf * scale at -inf (-inf * 0 would be NaN).
  if (scale_log2 == 0.f) scale_log2 = 1.401298464e-45f;
  const uint16_t* qq = static_cast<const uint16_t*>(q);
  const uint16_t* kk = static_cast<const uint16_t*>(k);
  const uint16_t* vv = static_cast<const uint16_t*>(v);
  uint16_t* oo = static_cast<uint16_t*>(out);
  // 64 queries per wave move half the operand bytes per query, but come in units twice as large.
  // So by rounds of resident workgroups on 256 CUs (3 of 32 queries per CU, 2 of 64): 64 queries when
  // that takes fewer rounds, or as many, more than one, with the last round of the 32-query grid
  // more than 65% full: above two thirds it puts a third workgroup on CUs.  Measured per call, 32
  // against 64 queries (us), with the fill of the last 32-query round: 14 heads T 2592 (48%) 52.9 /
  // 55.2, T 2848 (62%) 59.2 / 60.2, T 2912 (66%) 60.8 / 61.2, T 2976 (70%) 69.2 / 62.9; 28 heads T 1440
  // (64%) 33.8 / 35.0, T 1480 (71%) 39.5 / 36.4; 56 heads T 704 (60%) 20.4 / 21.7, T 736 (68%) 23.5 /
  // 22.0, T 1153 (70% of a third round) 47.1 / 46.2; fewer rounds: 42 heads T 1500 53.2 / 46.7.
  const long long i1 = (long long)bh * ((T + 31) / 32), i2 = (long long)bh * ((T + 63) / 64);
  const long long r1 = (i1 + 767) / 768, r2 = (i2 + 511) / 512;
  const bool wide = r2 < r1 || (r2 == r1 && r1 > 1 && 20 * i1 > 768 * (20 * r1 - 7));
  const bool ok = wide ? fa_launch<2>(qq, kk, vv, oo, bh, T, f16, scale_log2, stream)
                       : fa_launch<1>(qq, kk, vv, oo, bh, T, f16, scale_log2, stream);
  if (!ok) return -1;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
