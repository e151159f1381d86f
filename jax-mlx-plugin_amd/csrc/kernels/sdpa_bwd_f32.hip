// SDPA backward in fp32 on the matrix cores (v_mfma_f32_32x32x2_f32: fp32
// products and accumulation), head size 32, 64, 96 or 128 (D == Dv).
//
// Two kernels, each owning its outputs (deterministic, no atomics), with the
// forward kernel's operand layouts (sdpa_flash_f32.hip): a product's k-slots
// are permuted alike in A and B, so row operands are 16-byte LDS reads,
// column operands conflict-light 4-byte reads, and P / dS feed the next
// product straight from the accumulators.
//
// dq: a wavefront owns 32 queries (Q and dO rows in registers, as B) and
//   walks 32-key K / V tiles: S^T = K Q^T, dP^T = V dO^T (lane = query, so
//   lse and delta are per-lane scalars), dQ^T += K^T dS^T.  It runs first and
//   also writes each row's delta = rowsum(dO * O) for the other kernel.
// dkdv: a wavefront owns 32 keys (K and V rows in registers, as B) and walks
//   32-query Q / dO tiles of every query head of the group: S = Q K^T,
//   dP = dO V^T (lane = key), dV^T += dO^T P, dK^T += Q^T dS.
//
// What bounds them: the fp32 matrix rate (one 32x32x2 product takes ~65
// cycles; a tile is 3 D/2 or 4 D/2 of them per wavefront beside ~16 exps and
// D/2 + D/2 LDS reads).  Work that fits neither is small, so plain LDS
// double buffering (global -> registers -> LDS, one barrier per tile) is
// enough.  A workgroup is NW = 4 wavefronts sharing the tiles, or a single
// one where 4-wavefront workgroups would leave CUs without work
// (bwd_f32_waves).
//
// Measured on [32,256,8,64] BTNH without a mask: dQ 69 us (93 TFLOP/s) and
// dK / dV 89 us (97), against 1177 and 7445 us for the one-wavefront-per-row
// kernels (sdpa_bwd.hip) that ran these calls before, the matrix cores 60-63%
// busy; the whole recomputing call 181 against 8712 us.  Every call that meets
// bwd_f32_supports comes here: also where a wavefront walks all its tiles alone
// the per-row kernels, whose wavefronts walk as many rows one by one, take
// longer (from residuals at D = 64, this file against theirs in us: one tile
// [1,1,32] 14 and 30; 8 heads over 1 kv head, 4096 queries, 64 keys 4957 and
// 14767; 64 over 1, 512 queries, one key 4939 and 14648; one query, 8192 keys
// 914 and 1575; 64 heads of one query and one key 14 and 17; at D = 32 to 128
// over 96 such shapes 0.03 to 0.87 of their time).
#include "sdpa_f32.h"

namespace mfx {
namespace {

constexpr int kTile = 32;  // rows per LDS tile

// Rows of D floats padded by 16 bytes: lanes on consecutive rows then cover
// all banks with 16-byte reads.
template <int D>
constexpr int kRow = D + 4;

// One pair of [kTile][D] tiles (K and V, or Q and dO) on its way global ->
// registers -> LDS, shared by NW wavefronts.  Rows past the end read as
// zeros (row strides are at least D: checked on the host).
template <int D, int NW>
struct PairLoader {
  static constexpr int DCH = D / 4;                    // 16-byte chunks per row
  static constexpr int CH = kTile * DCH / (64 * NW);   // chunks per thread
  static_assert(kTile * DCH % (64 * NW) == 0, "a tile is whole chunks per thread");
  int off_a[CH], off_b[CH];
  f32x4 ra[CH], rb[CH];
  __device__ __forceinline__ PairLoader(int tid, int64_t sa, int64_t sb) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = tid + i * 64 * NW, row = c / DCH, col = c % DCH;
      off_a[i] = (int)((row * sa + col * 4) * 4);
      off_b[i] = (int)((row * sb + col * 4) * 4);
    }
  }
  // `rows` valid rows (at most kTile are read) at a and b.
  __device__ __forceinline__ void load(const float* a, int64_t sa, const float* b, int64_t sb, int rows) {
    rows = min(rows, kTile);
    const auto fa = f32_rsrc(a, rows_extent<D>(rows, sa));
    const auto fb = f32_rsrc(b, rows_extent<D>(rows, sb));
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      ra[i] = ld4(fa, off_a[i]);
      rb[i] = ld4(fb, off_b[i]);
    }
  }
  __device__ __forceinline__ void store(float* a, float* b, int tid) const {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = tid + i * 64 * NW, row = c / DCH, col = c % DCH;
      *reinterpret_cast<f32x4*>(a + row * kRow<D> + col * 4) = ra[i];
      *reinterpret_cast<f32x4*>(b + row * kRow<D> + col * 4) = rb[i];
    }
  }
};

// acc = A B over the D features: A = tile rows (lane row l32), B = the
// wavefront's own rows in registers (r[c*4 + e] = feature c*8 + half*4 + e).
template <int D>
__device__ __forceinline__ f32x16 row_product(const float* tile, const float (&r)[D / 2], int l32, int half) {
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(tile + l32 * kRow<D> + c * 8 + half * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], r[c * 4 + e], acc, 0, 0, 0);
  }
  return acc;
}

// out[dt] += A B over the tile's 32 rows: A = tile columns (feature dt*32 +
// l32), B = w (accumulator layout: w[i] belongs to row (i>>2)*8 + half*4 + (i&3)).
template <int D>
__device__ __forceinline__ void col_product(const float* tile, const f32x16& w, f32x16 (&out)[D / 32], int l32,
                                            int half) {
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float a = tile[((i >> 2) * 8 + half * 4 + (i & 3)) * kRow<D> + dt * 32 + l32];
      out[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, w[i], out[dt], 0, 0, 0);
    }
}

// Whether a lane's sums hold a NaN or an infinity.
template <int D>
__device__ __forceinline__ bool nonfinite(const f32x16 (&acc)[D / 32]) {
  float t[4] = {};  // zeros or NaN
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) t[i & 3] = fmaf(acc[dt][i], 0.f, t[i & 3]);
  const float any = (t[0] + t[1]) + (t[2] + t[3]);
  return __ballot(any != any) != 0;
}

// The lane's half of row `row` as a B operand, zero when !valid.
template <int D>
__device__ __forceinline__ void load_row(const float* row, bool valid, int half, float (&r)[D / 2]) {
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    f32x4 t = *reinterpret_cast<const f32x4*>(row + c * 8 + half * 4);
    if (!valid) t = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) r[c * 4 + e] = t[e];
  }
}

// Stores a transposed accumulator set (lane = row, features dt*32 + g*8 +
// half*4 + e), times mul.
template <int D>
__device__ __forceinline__ void store_row(float* row, const f32x16 (&acc)[D / 32], int half, float mul) {
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = acc[dt][g * 4 + e] * mul;
      *reinterpret_cast<f32x4*>(row + dt * 32 + g * 8 + half * 4) = w;
    }
}

// Bit r: row r of 32 (n of them there) holds a NaN or an infinity; with ALL,
// nothing but NaN.
template <int D, bool ALL>
__device__ __forceinline__ uint32_t odd_rows(const float* rows, int64_t stride, int n, int l32, int half) {
  if (n <= 0) return 0;
  const float* row = rows + min(l32, n - 1) * stride + half * 4;
  bool any = false, all = true;
#pragma unroll 2
  for (int c = 0; c < D / 8; ++c) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(row + c * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float z = a[e] * 0.f;  // NaN unless finite
      any |= z != z;
      all &= a[e] != a[e];
    }
  }
  const uint64_t b = __ballot(l32 < n && (ALL ? all : any));
  return ALL ? (uint32_t)b & (uint32_t)(b >> 32) : (uint32_t)b | (uint32_t)(b >> 32);
}

// A matrix product multiplies the rows that causality hides too, by zero,
// which is NaN where such a row is not finite; but hidden rows must not take
// part at all.  They lie in the tile on a wavefront's diagonal.  So where a
// causal call's sums are not all finite, the rows among the wavefront's 32 that
// hide such a row, and are not NaN throughout by what they see, are computed
// again by these, one at a time from what the row sees: a lane per row of the
// other axis for the scores, then per feature for the sums.  (Asking the sums
// costs D / 2 instructions, D in dkdv, once a wavefront: [16,8,20,64] goes from
// 14.9 to 15.2 us, [1,1,2048,64] stays at 538, and K of NaN throughout costs
// [1,8,2048,64] GQA 2% of its 2.85 ms.)
//
// Features f*64 + lane of a row.
template <int D>
constexpr int kFeat = (D + 63) / 64;

template <int D>
__device__ __forceinline__ float row_dot(const float* a, const float* b) {
  float s = 0.f;
#pragma unroll 4
  for (int d = 0; d < D; ++d) s = fmaf(a[d], b[d], s);
  return s;
}

template <int D, int MT>
__device__ __forceinline__ float row_score(const SdpaBwdParams& p, const float* q, const float* k, int64_t moff) {
  float s = row_dot<D>(q, k) * p.scale_log2;
  if constexpr (MT != 0) s += mask_log2(load_mask_t<MT>(p.mask, moff));
  return s;
}

template <int D>
__device__ __forceinline__ void add_row(const float* row, float w, int lane, float (&acc)[kFeat<D>]) {
#pragma unroll
  for (int f = 0; f < kFeat<D>; ++f)
    if (f * 64 + lane < D) acc[f] = fmaf(w, row[f * 64 + lane], acc[f]);
}

template <int D>
__device__ __forceinline__ void put_row(float* row, float mul, int lane, const float (&acc)[kFeat<D>]) {
#pragma unroll
  for (int f = 0; f < kFeat<D>; ++f)
    if (f * 64 + lane < D) row[f * 64 + lane] = acc[f] * mul;
}

// dQ of query i, which sees keys 0 .. i.
template <int D, int MT>
__device__ __forceinline__ void dq_row(const SdpaBwdParams& p, int b, int h, int i, float lse, float delta, int lane) {
  const int hk = h / p.group;
  const float* q = static_cast<const float*>(p.q) + b * p.qs[0] + h * p.qs[1] + (int64_t)i * p.qs[2];
  const float* g = static_cast<const float*>(p.dout) + b * p.dos[0] + h * p.dos[1] + (int64_t)i * p.dos[2];
  const float* k = static_cast<const float*>(p.k) + b * p.ks[0] + hk * p.ks[1];
  const float* v = static_cast<const float*>(p.v) + b * p.vs[0] + hk * p.vs[1];
  const int64_t mrow = MT ? b * p.ms[0] + h * p.ms[1] + (int64_t)i * p.ms[2] : 0;
  float acc[kFeat<D>] = {};
  const int end = min(p.Tk, i + 1);
  for (int kb = 0; kb < end; kb += 64) {
    const int j = min(kb + lane, end - 1);
    const float x = row_score<D, MT>(p, q, k + (int64_t)j * p.ks[2], mrow + (MT ? j * p.ms[3] : 0));
    const float ds = __builtin_amdgcn_exp2f(x - lse) * (row_dot<D>(g, v + (int64_t)j * p.vs[2]) - delta);
    const int n = min(64, end - kb);
    for (int jj = 0; jj < n; ++jj) add_row<D>(k + (int64_t)(kb + jj) * p.ks[2], __shfl(ds, jj, 64), lane, acc);
  }
  put_row<D>(static_cast<float*>(p.dq) + b * p.dqs[0] + h * p.dqs[1] + (int64_t)i * p.dqs[2], p.scale, lane, acc);
}

// dK and dV of key j, which queries j .. Tq - 1 of every head of the group see.
template <int D, int MT>
__device__ __forceinline__ void dkdv_row(const SdpaBwdParams& p, int b, int hk, int j, int lane) {
  const float* k = static_cast<const float*>(p.k) + b * p.ks[0] + hk * p.ks[1] + (int64_t)j * p.ks[2];
  const float* v = static_cast<const float*>(p.v) + b * p.vs[0] + hk * p.vs[1] + (int64_t)j * p.vs[2];
  float dk[kFeat<D>] = {}, dv[kFeat<D>] = {};
  for (int h = hk * p.group; h < (hk + 1) * p.group; ++h) {
    const float* q = static_cast<const float*>(p.q) + b * p.qs[0] + h * p.qs[1];
    const float* g = static_cast<const float*>(p.dout) + b * p.dos[0] + h * p.dos[1];
    const int64_t mcol = MT ? b * p.ms[0] + h * p.ms[1] + j * p.ms[3] : 0, rows = ((int64_t)b * p.Hq + h) * p.Tq;
    for (int qb = j; qb < p.Tq; qb += 64) {
      const int i = min(qb + lane, p.Tq - 1);
      const float x = row_score<D, MT>(p, q + (int64_t)i * p.qs[2], k, mcol + (MT ? i * p.ms[2] : 0));
      const float pr = __builtin_amdgcn_exp2f(x - p.lse[rows + i]);
      const float ds = pr * (row_dot<D>(g + (int64_t)i * p.dos[2], v) - p.delta[rows + i]);
      const int n = min(64, p.Tq - qb);
      for (int ii = 0; ii < n; ++ii) {
        add_row<D>(q + (int64_t)(qb + ii) * p.qs[2], __shfl(ds, ii, 64), lane, dk);
        add_row<D>(g + (int64_t)(qb + ii) * p.dos[2], __shfl(pr, ii, 64), lane, dv);
      }
    }
  }
  put_row<D>(static_cast<float*>(p.dk) + b * p.dks[0] + hk * p.dks[1] + (int64_t)j * p.dks[2], p.scale, lane, dk);
  put_row<D>(static_cast<float*>(p.dv) + b * p.dvs[0] + hk * p.dvs[1] + (int64_t)j * p.dvs[2], 1.f, lane, dv);
}

// (head, block) of a workgroup: a head's blocks on one XCD (workgroups are
// dealt to the 8 XCDs round-robin) when the heads divide by 8.
__device__ __forceinline__ void map_block(int id, int heads, int blocks, int& head, int& block) {
  if ((heads & 7) == 0) {
    const int slot = id >> 3;
    head = (slot / blocks) * 8 + (id & 7);
    block = slot % blocks;
  } else {
    head = id % heads;
    block = id / heads;
  }
}

// Two wavefronts per SIMD (256 registers) up to D = 64; D = 96 and 128 hold
// 2 D/2 operand and D/2 or D accumulator registers and take one.
template <int D, int NW, int MT>
__global__ __launch_bounds__(64 * NW, D <= 64 ? 2 : 1) void bwd_f32_dq_kernel(SdpaBwdParams p) {
  __shared__ __attribute__((aligned(16))) float k_lds[2][kTile * kRow<D>];
  __shared__ __attribute__((aligned(16))) float v_lds[2][kTile * kRow<D>];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  const int nb = (p.Tq + 32 * NW - 1) / (32 * NW);
  int bh, blk;
  map_block(blockIdx.x, p.B * p.Hq, nb, bh, blk);
  blk = nb - 1 - blk;  // longest causal blocks first
  const int b = bh / p.Hq, h = bh % p.Hq, hk = h / p.group;
  const int Tq = p.Tq, Tk = p.Tk;
  const bool causal = p.causal;  // (uniform: not worth a second kernel)
  const int64_t ks2 = p.ks[2], vs2 = p.vs[2];
  const float* kp = static_cast<const float*>(p.k) + b * p.ks[0] + hk * p.ks[1];
  const float* vp = static_cast<const float*>(p.v) + b * p.vs[0] + hk * p.vs[1];
  const int q0 = (blk * NW + wave) * 32, qi = q0 + l32;
  const int qc = min(qi, Tq - 1);
  const bool qv = qi < Tq;

  int kv_end = Tk;
  if (causal) kv_end = min(Tk, min(Tq, (blk + 1) * 32 * NW));
  const int ntiles = (kv_end + kTile - 1) / kTile;
  PairLoader<D, NW> ld(tid, ks2, vs2);
  auto fetch = [&](int t) {
    ld.load(kp + (int64_t)t * kTile * ks2, ks2, vp + (int64_t)t * kTile * vs2, vs2, Tk - t * kTile);
  };
  fetch(0);

  float qf[D / 2], gf[D / 2];
  load_row<D>(static_cast<const float*>(p.q) + b * p.qs[0] + h * p.qs[1] + (int64_t)qc * p.qs[2], qv, half, qf);
  load_row<D>(static_cast<const float*>(p.dout) + b * p.dos[0] + h * p.dos[1] + (int64_t)qc * p.dos[2], qv, half, gf);
  const int64_t row = (int64_t)bh * Tq + qc;
  const float lse = p.lse[row];
  float delta = 0.f;
  {
    // The same half-row layout: one exchange completes the sum.
    float of[D / 2];
    load_row<D>(static_cast<const float*>(p.o) + b * p.os[0] + h * p.os[1] + (int64_t)qc * p.os[2], qv, half, of);
#pragma unroll
    for (int j = 0; j < D / 2; ++j) delta += of[j] * gf[j];
    delta += __shfl_xor(delta, 32, 64);
    if (half == 0 && qv) p.delta[row] = delta;
  }
  const int64_t mrow = MT ? b * p.ms[0] + h * p.ms[1] + (int64_t)qc * p.ms[2] : 0;
  const float sl2 = p.scale_log2;
  f32x16 dq[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[dt][i] = 0.f;

  ld.store(k_lds[0], v_lds[0], tid);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    const int kb = t * kTile;
    const float* kt = k_lds[t & 1];
    const float* vt = v_lds[t & 1];
    if (t + 1 < ntiles) fetch(t + 1);
    if (q0 < Tq && (!causal || kb <= q0 + 31)) {
      // The mask values are all in flight under the two products.
      float m[16];
      if constexpr (MT != 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          m[i] = load_mask_t<MT>(p.mask, mrow + min(kb + (i >> 2) * 8 + half * 4 + (i & 3), Tk - 1) * p.ms[3]);
      }
      f32x16 s = row_product<D>(kt, qf, l32, half);
      const f32x16 dp = row_product<D>(vt, gf, l32, half);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = kb + (i >> 2) * 8 + half * 4 + (i & 3);
        float x = s[i] * sl2;
        if constexpr (MT != 0) x += mask_log2(m[i]);
        const float w = __builtin_amdgcn_exp2f(x - lse) * (dp[i] - delta);
        s[i] = key >= Tk || (causal && key > qi) ? 0.f : w;
      }
      col_product<D>(kt, s, dq, l32, half);
    }
    if (t + 1 < ntiles) ld.store(k_lds[(t + 1) & 1], v_lds[(t + 1) & 1], tid);
    __syncthreads();
  }
  uint32_t again = 0;  // rows for dq_row
  if (causal && __builtin_expect(nonfinite<D>(dq), false)) {
    const uint32_t odd = odd_rows<D, false>(kp + (int64_t)q0 * ks2, ks2, min(32, Tk - q0), l32, half);
    // A NaN lse or delta makes the whole row NaN.
    const bool nan = lse != lse || delta != delta;
    again = (uint32_t)__ballot(qv && !nan && (odd >> l32 >> 1) != 0);
  }
  if (qv && !(again >> l32 & 1))
    store_row<D>(static_cast<float*>(p.dq) + b * p.dqs[0] + h * p.dqs[1] + (int64_t)qi * p.dqs[2], dq, half, p.scale);
  for (; again; again &= again - 1) {
    const int r = __builtin_ctz(again);
    dq_row<D, MT>(p, b, h, q0 + r, __shfl(lse, r, 64), __shfl(delta, r, 64), lane);
  }
}

template <int D, int NW, int MT>
__global__ __launch_bounds__(64 * NW, D <= 64 ? 2 : 1) void bwd_f32_dkdv_kernel(SdpaBwdParams p) {
  __shared__ __attribute__((aligned(16))) float q_lds[2][kTile * kRow<D>];
  __shared__ __attribute__((aligned(16))) float g_lds[2][kTile * kRow<D>];
  __shared__ __attribute__((aligned(16))) float r_lds[2][2 * kTile];  // lse, then delta, of the tile's rows
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  const int nb = (p.Tk + 32 * NW - 1) / (32 * NW);
  int bhk, blk;
  map_block(blockIdx.x, p.B * p.Hkv, nb, bhk, blk);
  const int b = bhk / p.Hkv, hk = bhk % p.Hkv;
  const int Tq = p.Tq, Tk = p.Tk, G = p.group;
  const bool causal = p.causal;
  const int64_t qs2 = p.qs[2], gs2 = p.dos[2];
  const int k0 = (blk * NW + wave) * 32, key = k0 + l32;
  const int kc = min(key, Tk - 1);

  // Query tiles of every head of the group; causal: from the block's first
  // key's tile (none when the block lies past the last query).
  const int tile0 = causal ? blk * NW : 0;
  const int ntq = max((Tq + kTile - 1) / kTile - tile0, 0);
  const int n = ntq * G;
  PairLoader<D, NW> ld(tid, qs2, gs2);
  float rr = 0.f;  // this thread's element of r_lds
  auto fetch = [&](int it) {
    const int h = hk * G + it / ntq, i0 = (tile0 + it % ntq) * kTile;
    ld.load(static_cast<const float*>(p.q) + b * p.qs[0] + h * p.qs[1] + (int64_t)i0 * qs2, qs2,
            static_cast<const float*>(p.dout) + b * p.dos[0] + h * p.dos[1] + (int64_t)i0 * gs2, gs2, Tq - i0);
    if (tid < 2 * kTile) {
      const int i = min(i0 + (tid & (kTile - 1)), Tq - 1);
      rr = (tid < kTile ? p.lse : p.delta)[((int64_t)b * p.Hq + h) * Tq + i];
    }
  };
  auto store = [&](int buf) {
    ld.store(q_lds[buf], g_lds[buf], tid);
    if (tid < 2 * kTile) r_lds[buf][tid] = rr;
  };

  float kf[D / 2], vf[D / 2];
  load_row<D>(static_cast<const float*>(p.k) + b * p.ks[0] + hk * p.ks[1] + (int64_t)kc * p.ks[2], key < Tk, half, kf);
  load_row<D>(static_cast<const float*>(p.v) + b * p.vs[0] + hk * p.vs[1] + (int64_t)kc * p.vs[2], key < Tk, half, vf);
  const float sl2 = p.scale_log2;
  f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[dt][i] = dv[dt][i] = 0.f;

  if (n > 0) {
    fetch(0);
    store(0);
  }
  __syncthreads();
  for (int it = 0; it < n; ++it) {
    const int h = hk * G + it / ntq, i0 = (tile0 + it % ntq) * kTile;
    const float* qt = q_lds[it & 1];
    const float* gt = g_lds[it & 1];
    if (it + 1 < n) fetch(it + 1);
    if (k0 < Tk && (!causal || i0 + kTile > k0)) {
      float m[16];
      if constexpr (MT != 0) {
        const int64_t mb = b * p.ms[0] + h * p.ms[1] + kc * p.ms[3];
#pragma unroll
        for (int i = 0; i < 16; ++i)
          m[i] = load_mask_t<MT>(p.mask, mb + min(i0 + (i >> 2) * 8 + half * 4 + (i & 3), Tq - 1) * p.ms[2]);
      }
      f32x16 s = row_product<D>(qt, kf, l32, half);
      f32x16 dp = row_product<D>(gt, vf, l32, half);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 lse = *reinterpret_cast<const f32x4*>(&r_lds[it & 1][g * 8 + half * 4]);
        const f32x4 delta = *reinterpret_cast<const f32x4*>(&r_lds[it & 1][kTile + g * 8 + half * 4]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = g * 4 + e, q = i0 + g * 8 + half * 4 + e;
          float x = s[i] * sl2;
          if constexpr (MT != 0) x += mask_log2(m[i]);
          const float pr = __builtin_amdgcn_exp2f(x - lse[e]);
          const float ds = pr * (dp[i] - delta[e]);
          const bool off = q >= Tq || (causal && key > q);
          s[i] = off ? 0.f : pr;
          dp[i] = off ? 0.f : ds;
        }
      }
      col_product<D>(gt, s, dv, l32, half);
      col_product<D>(qt, dp, dk, l32, half);
    }
    if (it + 1 < n) store((it + 1) & 1);
    __syncthreads();
  }
  uint32_t again = 0;  // rows for dkdv_row
  if (causal && __builtin_expect(nonfinite<D>(dk) || nonfinite<D>(dv), false)) {
    uint32_t odd = 0, blank = 0;       // of the diagonal's query rows, in any head: not finite, dO all NaN
    int nan_lse = -1, nan_delta = -1;  // the last such query
    for (int h = hk * G; h < (hk + 1) * G; ++h) {
      const float* q = static_cast<const float*>(p.q) + b * p.qs[0] + h * p.qs[1] + (int64_t)k0 * qs2;
      const float* g = static_cast<const float*>(p.dout) + b * p.dos[0] + h * p.dos[1] + (int64_t)k0 * gs2;
      const int m = min(32, Tq - k0);
      odd |= odd_rows<D, false>(q, qs2, m, l32, half) | odd_rows<D, false>(g, gs2, m, l32, half);
      blank |= odd_rows<D, true>(g, gs2, m, l32, half);
      const int64_t rows = ((int64_t)b * p.Hq + h) * Tq;
      for (int i = k0 + lane; i < Tq; i += 64) {
        if (p.lse[rows + i] != p.lse[rows + i]) nan_lse = max(nan_lse, i);
        if (p.delta[rows + i] != p.delta[rows + i]) nan_delta = max(nan_delta, i);
      }
    }
#pragma unroll
    for (int o = 32; o; o >>= 1) {
      nan_lse = max(nan_lse, __shfl_xor(nan_lse, o, 64));
      nan_delta = max(nan_delta, __shfl_xor(nan_delta, o, 64));
    }
    // A query with a NaN lse makes dK and dV of all it sees NaN, a NaN delta
    // dK; the key's own query dV where its dO is.
    const bool nan = key <= nan_lse || (key <= nan_delta && (blank >> l32 & 1));
    again = (uint32_t)__ballot(key < Tk && !nan && (odd & ((1u << l32) - 1)) != 0);
  }
  if (key < Tk && !(again >> l32 & 1)) {
    store_row<D>(static_cast<float*>(p.dk) + b * p.dks[0] + hk * p.dks[1] + (int64_t)key * p.dks[2], dk, half, p.scale);
    store_row<D>(static_cast<float*>(p.dv) + b * p.dvs[0] + hk * p.dvs[1] + (int64_t)key * p.dvs[2], dv, half, 1.f);
  }
  for (; again; again &= again - 1) dkdv_row<D, MT>(p, b, hk, k0 + __builtin_ctz(again), lane);
}

// Wavefronts per workgroup of a kernel whose wavefronts own 32 of T rows in
// each of `heads` heads: four share a tile's loads once that still gives
// every CU its two workgroups (256 registers, 35 KB of LDS at D = 64);
// below, one-wavefront workgroups reach up to four times the CUs.
int bwd_f32_waves(int64_t heads, int T) {
  return heads * ((T + 127) / 128) >= 2LL * device_cu_count() ? 4 : 1;
}

template <int D, int MT>
int launch_t(const SdpaBwdParams& p, hipStream_t s) {
  const int64_t hq = (int64_t)p.B * p.Hq, hk = (int64_t)p.B * p.Hkv;
  if (bwd_f32_waves(hq, p.Tq) == 4)
    hipLaunchKernelGGL((bwd_f32_dq_kernel<D, 4, MT>), dim3((unsigned)(hq * ((p.Tq + 127) / 128))), dim3(256),
                       0, s, p);
  else
    hipLaunchKernelGGL((bwd_f32_dq_kernel<D, 1, MT>), dim3((unsigned)(hq * ((p.Tq + 31) / 32))), dim3(64), 0,
                       s, p);
  const int rc = launch_status("bwd_f32_dq_kernel");
  if (rc != MFX_OK) return rc;
  if (bwd_f32_waves(hk, p.Tk) == 4)
    hipLaunchKernelGGL((bwd_f32_dkdv_kernel<D, 4, MT>), dim3((unsigned)(hk * ((p.Tk + 127) / 128))), dim3(256),
                       0, s, p);
  else
    hipLaunchKernelGGL((bwd_f32_dkdv_kernel<D, 1, MT>), dim3((unsigned)(hk * ((p.Tk + 31) / 32))), dim3(64), 0,
                       s, p);
  return launch_status("bwd_f32_dkdv_kernel");
}

template <int D>
int launch_d(const SdpaBwdParams& p, hipStream_t s) {
  if (!p.mask) return launch_t<D, 0>(p, s);
  switch (mask_code(p.mask_dtype)) {
    case 1: return launch_t<D, 1>(p, s);
    case 2: return launch_t<D, 2>(p, s);
    default: return launch_t<D, 3>(p, s);
  }
}

}  // namespace

// f32 tensors whose rows are whole 16-byte chunks and do not overlap (rows
// past the end must read as zeros: the products multiply them by exact
// zeros), with a tile of rows inside a 32-bit byte range.
bool bwd_f32_supports(const SdpaBwdParams& p) {
  if (p.dtype != MFX_F32 || p.D != p.Dv || p.D % 32 != 0 || p.D > 128) return false;
  const void* ptrs[8] = {p.q, p.k, p.v, p.o, p.dout, p.dq, p.dk, p.dv};
  for (const void* ptr : ptrs)
    if ((uintptr_t)ptr & 15) return false;  // (p.o null: recomputed into the 256-byte aligned workspace)
  for (int i = 0; i < 3; ++i)
    if (p.qs[i] % 4 || p.ks[i] % 4 || p.vs[i] % 4 || p.os[i] % 4 || p.dos[i] % 4 || p.dqs[i] % 4 || p.dks[i] % 4 ||
        p.dvs[i] % 4)
      return false;
  for (int64_t st : {p.qs[2], p.ks[2], p.vs[2], p.dos[2]})
    if (st < p.D || st >= (int64_t(1) << 23)) return false;
  return true;
}

int launch_bwd_f32(const SdpaBwdParams& p, hipStream_t s) {
  switch (p.D) {
    case 32: return launch_d<32>(p, s);
    case 64: return launch_d<64>(p, s);
    case 96: return launch_d<96>(p, s);
    default: return launch_d<128>(p, s);
  }
}

}  // namespace mfx
