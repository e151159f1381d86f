// Flash attention forward with an additive mask, bf16 inputs, fp32
// accumulation, gfx950 MFMA.  (Mask-free calls go to the software-pipelined
// kernel in sdpa_flash_bf16_pipe.hip.)
//
// Workgroup = 4 wavefronts = 128 query rows of one (batch, head); each
// wavefront owns 32 query rows.  K/V stream through LDS in 64-key tiles, two
// stages: while tile t is computed, tile t+1 is copied global -> LDS by the
// asynchronous LDS-DMA loads (buffer_load_dwordx4 ... lds: no registers, no
// VALU), and one vmcnt wait + barrier per tile publishes it.
//
// Both products use v_mfma_f32_32x32x16_bf16 and are arranged so that the
// online softmax needs almost no cross-lane traffic:
//   S^T = K Q^T   A = K tile rows (from LDS), B = Q rows (registers).  The
//                 32x32 accumulator gives lane l query (l % 32) and 16 keys,
//                 so a query's row max / sum is 16 in-lane values plus one
//                 exchange with lane l ^ 32.
//   O^T = V^T P^T A = V^T fragments read from the row-major V tile with the
//                 transposing LDS read (ds_read_b64_tr_b16: 16 lanes x 4
//                 keys per read), B = P taken straight from the S^T
//                 accumulator: the contraction index (key) is permuted
//                 identically in A and B, so the accumulator registers are
//                 already the B operand.
// Each lane also owns one query of O^T, so the online-softmax rescale is a
// per-lane scalar multiply, and it is lazy (see kSlack).
//
// Tiles are row-major with 16-byte chunks XOR-swizzled per row, so the K
// operand reads (8 lanes on 8 rows) and the transposing V reads (4 rows x 32
// bytes per 16 lanes) are bank-conflict free; the DMA writes 1 KiB runs.
//
// Causal tiles past a wavefront's last query are skipped; the blockIdx ->
// (head, q-block) map keeps the q-blocks of one head on one XCD (blocks are
// dealt to the 8 XCDs round-robin) and issues each XCD's blocks longest
// first, which balances the causal triangle across the CUs.
#include <type_traits>

#include "sdpa_elem.h"
#include "sdpa_mask.h"
#include "sdpa_tiles.h"

namespace mfx {
namespace {

constexpr int kBM = 128;  // query rows per workgroup
constexpr int kBN = 64;        // keys per tile
constexpr int kMT = kBN / 32;  // 32-key score blocks per tile
constexpr int kKS = kBN / 16;  // 16-key PV steps per tile
constexpr int kNT = 256;  // threads per workgroup

using tiles::kSlack;
using tiles::lds_s16x4_t;
using tiles::s16x4;
using tiles::tile_swz;
using tiles::wait_dma;
using tiles::fence;
template <int D>
using TileLoader = tiles::TileLoader<D, kBN, kNT / 64>;

// D: LDS row width (64, 128 or 256), DV <= D: the head size.  MT: the mask's
// type (mask_code) read in runs; kAnyMask: any type and key stride, read
// element by element; 0: no mask (D = 256 only).
// D = 256: one workgroup per CU (four 32 KB tiles; O, Q and S of a wavefront
// take ~300 registers).
template <int D, int DV, int MT, int E>
__global__ __launch_bounds__(kNT, D > 128 ? 1 : 2) void flash_bf16_kernel(SdpaParams p) {
  __shared__ __attribute__((aligned(16))) bf16 k0[kBN * D];
  __shared__ __attribute__((aligned(16))) bf16 v0[kBN * D];
  __shared__ __attribute__((aligned(16))) bf16 k1[kBN * D];
  __shared__ __attribute__((aligned(16))) bf16 v1[kBN * D];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int half = lane >> 5;
  const int l32 = lane & 31;

  const int nmb = (p.Tq + kBM - 1) / kBM;
  const int BH = p.B * p.Hq;
  const int id = blockIdx.x;
  int bh, mblk;
  if ((BH & 7) == 0) {
    // Blocks are dealt to the 8 XCDs round-robin; within an XCD the issue
    // order is longest causal q-block first across all of its heads (LPT
    // list scheduling), so the short blocks fill the tail.
    const int xcd = id & 7, slot = id >> 3, bpx = BH >> 3;
    bh = (slot % bpx) * 8 + xcd;
    mblk = nmb - 1 - slot / bpx;
  } else {
    bh = id % BH;
    mblk = nmb - 1 - id / BH;
  }
  const int b = bh / p.Hq, h = bh % p.Hq, hk = h / p.group;
  const bf16* qp = static_cast<const bf16*>(p.q) + b * p.qs[0] + h * p.qs[1];
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.ks[0] + hk * p.ks[1];
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.vs[0] + hk * p.vs[1];
  bf16* op = static_cast<bf16*>(p.out) + b * p.os[0] + h * p.os[1];
  const int64_t qs2 = p.qs[2], ks2 = p.ks[2], vs2 = p.vs[2], os2 = p.os[2];
  const int Tq = p.Tq, Tk = p.Tk;

  const int q0 = mblk * kBM + wave * 32;
  const int qi = q0 + l32;

  // Only the causal form is compiled (the other spills at D = 256): key j is
  // visible to query i when j <= i + co, co = 0 for a causal call and 2^30
  // (every key) otherwise.
  const int co = !p.causal ? (1 << 30) : 0;
  const int kv_end = min(Tk, min(Tq + co, (mblk + 1) * kBM + co));
  const int ntiles = (kv_end + kBN - 1) / kBN;
  const TileLoader<D> kload(kp, ks2, Tk, DV, wave, lane), vload(vp, vs2, Tk, DV, wave, lane);
  auto issue = [&](int t, bf16* kl, bf16* vl) {
    kload.load(t, kl, wave);
    vload.load(t, vl, wave);
  };
  if (ntiles > 0) issue(0, k0, v0);
  constexpr bool MASK = MT != 0;
  // D <= 128: the tile's mask values, loaded a tile ahead.  (D = 256 has no
  // registers for that and loads each run where it is used.)
  constexpr bool RUNS = MASK && MT != kAnyMask;
  constexpr bool AHEAD = RUNS && D <= 128;
  constexpr bool FENCE = D > 128;
  // Head sizes 32 and 96: the per-row kernel, which these calls took before,
  // keeps probabilities in fp32, so here they enter PV as three 16-bit terms,
  // which hold all 24 bits of each (f16: to 2^-25 of the row's largest): the
  // output's error is its own rounding, as the per-row kernel's is (1.66e-3 in
  // 2-norm with a bf16 bias at 2048 keys; with one term 2.3e-3), and where V
  // cancels in the sum it is fp32's.  [4,16,2048,D] takes 157 (D = 32) and 237 us
  // (D = 96), against 10.2 and 17.0 ms there (with two terms 140 and 218).
  constexpr bool SPLIT = DV != D;
  using Run = MaskRun<RUNS ? MT : 1>;
  Run mk[AHEAD ? kKS : 1];
  const int64_t moff = MASK ? b * p.ms[0] + h * p.ms[1] + (int64_t)min(qi, Tq - 1) * p.ms[2] : 0;
  const auto* mrow = static_cast<const typename Run::Elem*>(p.mask) + moff;
  const bool odd = RUNS && mask_runs_odd<RUNS ? MT : 1>(p);
  auto mask_load = [&](int kb) __attribute__((always_inline)) {
    if (kb + kBN <= Tk) {
      const auto* at = mrow + (kb + half * 8);
#pragma unroll
      for (int g = 0; g < kKS; ++g) mk[AHEAD ? g : 0].load(at + g * 16, odd);
    } else {
#pragma unroll
      for (int g = 0; g < kKS; ++g) mk[AHEAD ? g : 0].load(mrow, kb + g * 16 + half * 8, Tk, odd);
    }
  };
  if constexpr (AHEAD) mask_load(0);

  // Rows past Tq load a valid row and are zeroed, so no load is predicated.
  bf16x8 qf[DV / 16];
  {
    const bf16* qrow = qp + (int64_t)min(qi, Tq - 1) * qs2 + half * 8;
#pragma unroll
    for (int kk = 0; kk < DV / 16; ++kk) {
      u32x4 raw = *reinterpret_cast<const u32x4*>(qrow + kk * 16);
      if (qi >= Tq) raw = u32x4{0u, 0u, 0u, 0u};
      qf[kk] = __builtin_bit_cast(bf16x8, raw);
    }
  }

  f32x16 o[DV / 32];
#pragma unroll
  for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  // Running exp2 base (log2 units, shared by lanes l and l^32) and the
  // lane's partial row sum.
  float b_run = -INFINITY, l_run = 0.f;
  const float sl2 = p.scale_log2;  // > 0 (checked on the host)

  // Per-lane LDS byte offsets of the operand reads.  Row r of a 32-key score
  // block is key r with bits 2 and 3 swapped, so that a lane's scores of a
  // 16-key step belong to eight consecutive keys, half*8 + (0..7): a run of
  // the mask's row.  The swizzle xors chunk bits below the row's, so chunk
  // c + 2j (K) and c + 4j (V) of a row are the first one's offset xor 32j, 64j.
  const int k_row = (l32 & ~12) | (l32 & 4) << 1 | (l32 & 8) >> 1;
  const uint32_t k_off = k_row * D * 2 + (half ^ tile_swz<D>(k_row)) * 16;
  const int tj = lane & 15, tg = (lane >> 4) & 1;
  const int v_row = 8 * half + (tj >> 2);  // + ks*16 + 4*r
  const int v_chunk = tg * 2 + ((tj & 3) >> 1);
  const uint32_t v_off = v_row * D * 2 + (v_chunk ^ tile_swz<D>(v_row)) * 16 + (tj & 1) * 8;
  const uint32_t v_off4 = (v_row + 4) * D * 2 + (v_chunk ^ tile_swz<D>(v_row + 4)) * 16 + (tj & 1) * 8;

  // One 64-key tile for this wave's 32 queries.  EDGE tiles (ragged end,
  // causal diagonal) mask per element; interior tiles do no mask work.
  auto compute = [&](const bf16* kl, const bf16* vl, int kb, auto edge_tag) {
    constexpr bool EDGE = decltype(edge_tag)::value;
    // Opaque: otherwise every chunk's offset into each of the four arrays is
    // hoisted out of the loop into a register of its own, and D = 128 spills.
    uint32_t ka = k_off, va = v_off, va4 = v_off4;
    asm volatile("" : "+v"(ka), "+v"(va), "+v"(va4));
    const char* kb8 = reinterpret_cast<const char*>(kl);
    const char* vb8 = reinterpret_cast<const char*>(vl);
    const bool more = kb + kBN < kv_end;
    // Nothing visible: a band or block mask's tiles outside it.
    bool off = false;
    if constexpr (AHEAD) {
      const bool ragged = EDGE && kb + kBN > Tk;
      if (odd || ragged) place_runs(mk, mrow, kb + half * 8, Tk, odd, ragged);
      off = runs_all_off(mk);
    }
    // kAnyMask: the tile's values, all in flight at once under the products,
    // in steps of 16 keys up to the row's end.  Loaded where each was used,
    // behind a branch on the type and waited for alone, past the row's end
    // too, they took 9.8 us a call on [1,8,300,64] with 7 keys (bf16 mask) and
    // 65 on [1,16,1024,64] GQA with strided keys (f32); 6.0 and 38 here.
    float any[MT == kAnyMask ? kMT * 16 : 1] = {};
    if constexpr (MT == kAnyMask) {
      auto rd = [&](auto mt_tag) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < kKS; ++g)
          if (!EDGE || g == 0 || kb + g * 16 < Tk)
#pragma unroll
            for (int i = 0; i < 8; ++i)
              any[g * 8 + i] = load_mask_t<decltype(mt_tag)::value>(
                  p.mask, moff + min(kb + g * 16 + half * 8 + i, Tk - 1) * p.ms[3]);
      };
      if (p.mask_dtype == MFX_F32) rd(std::integral_constant<int, 1>{});
      else if (p.mask_dtype == MFX_BF16) rd(std::integral_constant<int, 2>{});
      else rd(std::integral_constant<int, 3>{});
    }
    f32x16 s[kMT];
    float mx = -INFINITY;
    if (!off) {
    // Where registers are short, the phases of a tile (S, softmax, PV) and
    // the tiles stay apart, so no tile's fragments are live across another's.
    if constexpr (FENCE) fence();
    // The two waves of a SIMD alternate between MFMA blocks and softmax
    // work; raising a wave's priority for its MFMA blocks lets the arbiter
    // keep the matrix core fed while the other wave's vector work fills in.
    __builtin_amdgcn_s_setprio(3);
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[mt][i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < DV / 16; ++kk) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(kb8 + mt * 32 * D * 2 + (ka ^ kk * 32));
        s[mt] = mfma16<E>(a, qf[kk], s[mt]);
        // ... and at most four operand reads run ahead of their MFMAs.
        if constexpr (FENCE)
          if ((kk & 3) == 3) fence();
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if constexpr (FENCE) fence();
    // MASK: scores move to the log2 domain here (scale and mask folded);
    // otherwise they stay raw and the scale is folded into the exp2 FMA.
    // Score i of block mt is slot i & 7 of step mt*2 + (i >> 3).
    //
    // mask_log2's clamp keeps -inf; here -inf takes part as the clamp value
    // (one instruction fewer per clause), whose exp2 is 0 all the same beside
    // any row base above -1e37, and is put back where no key of a row has
    // come near that yet.  (f16 masks have no value below the clamp.)
    // EDGE: the last key of the tile the query sees, counted from the lane's
    // first (opaque, or its 32 comparands are hoisted out of the loop).
    int lim = min(qi + co, Tk - 1) - kb - half * 8;
    if constexpr (EDGE) asm volatile("" : "+v"(lim));
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float x = s[mt][i];
        const int g = mt * 2 + (i >> 3), key = kb + g * 16 + half * 8 + (i & 7);
        if constexpr (MT == kAnyMask) {
          x = x * sl2 + mask_log2(any[g * 8 + (i & 7)]);
        } else if constexpr (MASK) {
          Run& run = mk[AHEAD ? g : 0];
          if constexpr (!AHEAD)
            if ((i & 7) == 0) {
              fence();
              run.load(mrow, key, Tk, odd);
              place_runs(mk, mrow, key, Tk, odd, EDGE && kb + kBN > Tk);
            }
          float m = run.get(i & 7);
          if constexpr (AHEAD) {
            if constexpr (MT != 3) m = __builtin_elementwise_maximum(m, kMaskMin);
            x = fmaf(m, kLog2e, x * sl2);
          } else {
            x = x * sl2 + mask_log2(m);
          }
        }
        if constexpr (EDGE) {
          if (g * 16 + (i & 7) > lim) x = -INFINITY;
        }
        s[mt][i] = x;
        mx = fmaxf(mx, x);
        if constexpr (FENCE && AHEAD)
          if ((i & 3) == 3) fence();
      }
    if constexpr (AHEAD && MT != 3) {
      if (__ballot(fmaxf(mx, b_run) < -1e37f)) {
        mx = -INFINITY;
#pragma unroll
        for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            if (mk[AHEAD ? mt * 2 + (i >> 3) : 0].get(i & 7) == -INFINITY) s[mt][i] = -INFINITY;
            mx = fmaxf(mx, s[mt][i]);
          }
      }
    }
    }
    // The next tile's mask, on its way under this tile's exps and PV.
    if constexpr (AHEAD) {
      if (more) mask_load(kb + kBN);
      if (off) return;
    }
    // Lanes l and l^32 hold the two halves of one query's keys.
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const float m_l2 = MASK ? mx : mx * sl2;
    const bool need = m_l2 > b_run + kSlack;
    if (__ballot(need)) {
      const float nb = need ? m_l2 : b_run;
      const float alpha = need ? __builtin_amdgcn_exp2f(b_run - nb) : 1.f;
      b_run = nb;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    const float nbase = b_run == -INFINITY ? 0.f : -b_run;
    auto pexp = [&](int mt, int i) {
      return MASK ? __builtin_amdgcn_exp2f(s[mt][i] + nbase) : __builtin_amdgcn_exp2f(fmaf(s[mt][i], sl2, nbase));
    };
    // P rounded to the element type and the row sum of exactly the rounded
    // values the PV product consumes, two per instruction.  (SPLIT: P stays in
    // s until its step of the product.)
    bf16x8 pb[SPLIT ? 1 : kKS];
    float l0 = 0.f, l1 = 0.f;
    if constexpr (SPLIT) {
#pragma unroll
      for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[mt][i] = pexp(mt, i);
          (i & 1 ? l1 : l0) += s[mt][i];
        }
    } else if constexpr (E == 0) {
#pragma unroll
      for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) pb[mt * 2 + (i >> 3)][i & 7] = f32_elem<E>(pexp(mt, i));
#pragma unroll
      for (int j = 0; j < kKS; ++j) {
        const bf16x8 w = pb[j];
        l0 = dot2_at<E>(w, 0, l0);
        l1 = dot2_at<E>(w, 2, l1);
        l0 = dot2_at<E>(w, 4, l0);
        l1 = dot2_at<E>(w, 6, l1);
      }
    } else {
      // f16: pairs packed into dwords first.  (Element inserts into the
      // 16-bit vector followed by per-element dot2 operands compile to
      // wrong row sums for f16: pairs built from one value twice.)
      u32x4 pw[kKS];
#pragma unroll
      for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          const uint32_t w = pack2<E>(pexp(mt, i), pexp(mt, i + 1));
          pw[mt * 2 + (i >> 3)][(i & 7) >> 1] = w;
          if ((i & 2) == 0) l0 = dot2<E>(w, l0);
          else l1 = dot2<E>(w, l1);
        }
#pragma unroll
      for (int j = 0; j < kKS; ++j) pb[j] = __builtin_bit_cast(bf16x8, pw[j]);
    }
    l_run += l0 + l1;
    if constexpr (FENCE) fence();
    __builtin_amdgcn_s_setprio(3);
    // k-slots 0-3: keys ks*16 + 8*half + e; slots 4-7: the same + 4.
    auto v_frag = [&](int ks, int dt) __attribute__((always_inline)) {
      const char* v_rows = vb8 + ks * 16 * D * 2;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(v_rows + (va ^ dt * 64)));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(v_rows + (va4 ^ dt * 64)));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    if constexpr (SPLIT) {
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        bf16x8 term[3];
        float rest[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) rest[j] = s[ks >> 1][(ks & 1) * 8 + j];
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          u32x4 w;
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            w[j >> 1] = pack2<E>(rest[j], rest[j + 1]);
            rest[j] -= E == 0 ? __uint_as_float(w[j >> 1] << 16) : f16_lo(w[j >> 1]);
            rest[j + 1] -= E == 0 ? __uint_as_float(w[j >> 1] & 0xFFFF0000u) : f16_hi(w[j >> 1]);
          }
          term[n] = __builtin_bit_cast(bf16x8, w);
        }
#pragma unroll
        for (int dt = 0; dt < DV / 32; ++dt) {
          const bf16x8 a = v_frag(ks, dt);
#pragma unroll
          for (int n = 0; n < 3; ++n) o[dt] = mfma16<E>(a, term[n], o[dt]);
        }
      }
    } else {
#pragma unroll
      for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
        for (int ks = 0; ks < kKS; ++ks) {
          o[dt] = mfma16<E>(v_frag(ks, dt), pb[ks], o[dt]);
          if constexpr (FENCE)
            if ((ks & 1) == 1) fence();
        }
    }
    if constexpr (FENCE) fence();
  };

  auto step = [&](int t, const bf16* kl, const bf16* vl) __attribute__((always_inline)) {
    const int kb = t * kBN;
    if (q0 >= Tq || kb > q0 + 31 + co) return;  // nothing of this tile is visible
    const bool edge = (kb + kBN > Tk) || (kb + kBN - 1 > q0 + co);
    if (edge)
      compute(kl, vl, kb, std::true_type{});
    else
      compute(kl, vl, kb, std::false_type{});
  };

  wait_dma();
  __syncthreads();
  // Two stages with distinct LDS arrays (so the compiler's LDS-DMA tracking
  // sees that the loads in flight never alias the tile being read).
  // The restrict-qualified parameters give every access of one iteration
  // scoped no-alias metadata, so the waitcnt pass does not make the tile's
  // reads wait for the next tile's LDS-DMA writes.
  auto iter = [&](int t, const bf16* __restrict__ kc, const bf16* __restrict__ vc, bf16* __restrict__ kn,
                  bf16* __restrict__ vn) {
    if (t + 1 < ntiles) issue(t + 1, kn, vn);
    step(t, kc, vc);
  };
  for (int t = 0; t < ntiles; t += 2) {
    iter(t, k0, v0, k1, v1);
    wait_dma();
    __syncthreads();
    if (t + 1 >= ntiles) break;
    iter(t + 1, k1, v1, k0, v0);
    wait_dma();
    __syncthreads();
  }

  const float lt = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = 1.0f / lt;
  if (p.lse && half == 0 && qi < Tq) p.lse[(int64_t)bh * Tq + qi] = b_run + __log2f(lt);
  if constexpr (D <= 128 && DV == D) {
    // Every iteration ended at a barrier after its reads and with no load in
    // flight: the tile arrays take the output rows on their way out (k0
    // holds wavefronts 0 and 1, v0 wavefronts 2 and 3), stored as whole
    // rows streamed past the L2.  (The first row comes from an opaque copy,
    // so no address is hoisted into the loop.)  At D = 256, one workgroup per
    // CU, nothing would cover the LDS round trip: 8-byte pieces there.
    int r0 = q0;
    asm volatile("" : "+v"(r0));
    store_rows_lds<D, E>((wave < 2 ? k0 : v0) + (wave & 1) * 32 * D, op + (int64_t)r0 * os2, os2,
                         min(max(Tq - r0, 0), 32), o, l32, half, lane, inv);
  } else if (qi < Tq) {
    bf16* orow = op + qi * os2;
#pragma unroll
    for (int dt = 0; dt < DV / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u16x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = store_e<E>(o[dt][g * 4 + e] * inv);
        *reinterpret_cast<u16x4*>(orow + dt * 32 + g * 8 + half * 4) = w;
      }
  }
}

template <int D, int DV, int MT, int E>
int launch_t(const SdpaParams& p, hipStream_t s) {
  const int nmb = (p.Tq + kBM - 1) / kBM;
  const int64_t blocks = (int64_t)nmb * p.B * p.Hq;
  hipLaunchKernelGGL((flash_bf16_kernel<D, DV, MT, E>), dim3((unsigned)blocks), dim3(kNT), 0, s, p);
  return launch_status("flash_bf16_kernel");
}

template <int D, int DV, int E>
int launch_m(const SdpaParams& p, hipStream_t s) {
  switch (mask_run_code(p)) {
    case 1: return launch_t<D, DV, 1, E>(p, s);
    case 2: return launch_t<D, DV, 2, E>(p, s);
    case 3: return launch_t<D, DV, 3, E>(p, s);
    default: return launch_t<D, DV, kAnyMask, E>(p, s);
  }
}

// Head size 256 comes here in every mask form (the pipelined kernel stops at
// 128).
template <int E>
int launch_d(const SdpaParams& p, hipStream_t s) {
  switch (p.D) {
    case 32: return launch_m<64, 32, E>(p, s);
    case 64: return launch_m<64, 64, E>(p, s);
    case 96: return launch_m<128, 96, E>(p, s);
    case 128: return launch_m<128, 128, E>(p, s);
    default: return p.mask ? launch_m<256, 256, E>(p, s) : launch_t<256, 256, 0, E>(p, s);
  }
}

bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15) == 0; }

}  // namespace

bool flash_bf16_supports(const SdpaParams& p) {
  if (p.dtype != MFX_BF16 && p.dtype != MFX_F16) return false;
  if (!(p.scale_log2 > 0.f)) return false;  // the exp2 FMA folds a positive scale
  // K/V rows are read through one buffer resource per head ending at its
  // last row's last feature, range-checked on 31-bit lane offsets: row
  // strides of at least D (rows past Tk then start at or past the extent and
  // read as zeros; a smaller stride, such as 0 for a broadcast view, would
  // leave rows past Tk inside it).
  if (p.ks[2] < p.D || p.vs[2] < p.Dv) return false;
  if ((int64_t)p.Tk * p.ks[2] * 2 >= (1LL << 31) || (int64_t)p.Tk * p.vs[2] * 2 >= (1LL << 31)) return false;
  if (p.D != p.Dv || (p.D != 32 && p.D != 64 && p.D != 96 && p.D != 128 && p.D != 256)) return false;
  if (!aligned16(p.q) || !aligned16(p.k) || !aligned16(p.v) || !aligned16(p.out)) return false;
  for (int i = 0; i < 3; ++i)
    if (p.qs[i] % 8 || p.ks[i] % 8 || p.vs[i] % 8 || p.os[i] % 8) return false;  // 16-byte rows
  return true;
}

int launch_flash_bf16(const SdpaParams& p, hipStream_t s) {
  // Without an additive mask, or with one that does not vary along query
  // rows, the software-pipelined kernel runs (sdpa_flash_bf16_pipe.hip);
  // this file's kernel serves masks with a query-row stride, and head size
  // 256 in every form.  (With one query row the pipelined kernel's mask row
  // is that row.)
  if (p.D != 256 && (!p.mask || p.ms[2] == 0 || p.Tq == 1)) return launch_flash_bf16_pipe(p, s);
  return p.dtype == MFX_F16 ? launch_d<1>(p, s) : launch_d<0>(p, s);
}

}  // namespace mfx
