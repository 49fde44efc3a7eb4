// Fused attention forward for grids too small to fill the chip: the waves of
// a workgroup share one 32-row query block and split its keys.
//
// fwd_kernel gives each 32 query rows to one wave, which walks every key
// tile of its rows: with few (batch, head, 128-row) blocks most CUs are idle
// and the call takes as long as one wave's serial walk.  Here wave w of KW
// walks the 32-key tiles w, w + KW, ... of one 32-row block with a running
// max, row sum and O of its own, and the KW results meet in LDS once at the
// end (O = sum 2^(m_w - M) O_w / sum 2^(m_w - M) l_w).  The waves share no
// tile, so the walk has no barrier: each wave loads whole K and V rows into
// registers (with RoPE it rotates K there, so that the call needs no
// key-rotation launch) and passes them through LDS tiles of its own, the
// next tile's rows on their way while a tile is computed.  (K rows read
// straight into the MFMA operand layout are 32-byte pieces of 32 rows per
// load and were fetched several times over: 10 rows against 4096 keys, 32
// heads of 128 dims, 41 us.  V loaded into LDS directly: the compiler waits
// for every load in flight, the next tile's included, before it reads the
// tile.)
//
// Scores, softmax (log2 units, lazy running max), rounding of P, row sums of
// the rounded P and RoPE rounding are those of fwd_kernel.  Mask kind and
// ALiBi are uniform runtime switches: the time is latency, not issue.
#pragma once

#include "fwd_kernel.hpp"

namespace af {

struct FwdKeysParams {
  FwdParams f;      // n_mblocks = 32-row blocks of one head
  int32_t mask, alibi;
};

template <int D, int KW>
struct KeysLds {
  static constexpr int TILE = 32 * D;           // a wave's K tile, then its V tile (16-bit elements)
  static constexpr int OP = D + 4;              // row pitch of a wave's O (floats)
  static constexpr int WAVE_BYTES = 32 * OP * 4 > 4 * TILE ? 32 * OP * 4 : 4 * TILE;
};

// Whether the kernel rotates K itself, tile by tile in registers.  At head
// dim 128 a tile's rotation takes longer than its attention (300 rows, 32
// heads: 16.3 us against 9.4 without RoPE), so there K comes rotated by
// rope_rows_kernel and the kernel rotates its queries only.
constexpr bool keys_rotates_k(int D) { return D <= 64; }

// Waves per 32-row query block, or 0 where fwd_kernel is the better one.  The
// line lies where the key-split waves no longer all fit the chip at once (3
// waves per SIMD at D = 64, 5 at 32, 2 at 128): past it they queue, and
// fwd_kernel, which reads a K/V tile once for 128 query rows, has less work.
// Without a causal mask every block walks all its keys and the line comes
// earlier.  RoPE does not enter, so that fused RoPE keeps giving the bits of
// the plain forward on rotated inputs.  Measured (us, fwd_kernel / 4 waves /
// 8 waves; 32-row blocks in brackets), D = 64:
//   causal  12 heads x 512 [192]      10.4 /  6.6 /  6.7
//           24 x 1000 [768]           16.7 / 12.0 / 15.8
//           96 x 256 [768]             7.9 /  7.1 / 10.9
//           128 x 256 [1024]           8.1 /  8.9 / 13.6
//   dense   24 x 100, 1500 keys [96]  20.9 / 12.2 / 10.2
//           16 x 1024 [512]           15.8 / 12.8 / 15.3
//           24 x 1024 [768]           15.8 / 16.9 / 21.7
//   RoPE    12 x 512 [192]            15.1 /  8.4 /  7.6
//           24 x 1000 [768]           21.8 / 16.1 / 19.2
// D = 128: causal 32 x 300 [320] 10.7 / 9.1 / 10.4, 96 x 160 [480] 9.2 / 8.1
// / 11.2, 128 x 160 [640] 9.4 / 10.7 / 14.8, 256 x 64 [512] 6.4 / 7.3 / 10.1;
// dense 32 x 200, 4096 keys [224] 78.7 / 40.3 / 33.0, 32 x 600 [608] 17.6 /
// 20.5 / 25.7; RoPE 32 x 200 [224] 14.0 / 10.1 / 9.6, 32 x 440 [448] 18.4 /
// 14.0 / 16.0.
// D = 32: causal 32 x 1024 [1024] 13.9 / 9.8 / 12.4, 64 x 1024 [2048] 14.4 /
// 15.8 / 22.1.
inline int fwd_key_waves(int D, int mask, int64_t blocks32) {
  int64_t most = 0, most8 = 160;
  switch (D) {
    case 32: most = mask == MASK_CAUSAL ? 1024 : 640; break;
    case 64: most = mask == MASK_CAUSAL ? 768 : 512; break;
    case 128: most = 448; most8 = 256; break;
  }
  return blocks32 > most ? 0 : blocks32 <= most8 ? 8 : 4;
}

template <class E, int D, bool ROPE, int KW>
__global__ void __launch_bounds__(KW * 64) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 3 : 2)))
    fwd_keys_kernel(const FwdKeysParams P) {
  constexpr int KS = D / 16, DB = D / 32;
  constexpr int BN = 32;
  using L = KeysLds<D, KW>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[KW * L::WAVE_BYTES];
  __shared__ float red[KW][2][32];
  __shared__ __attribute__((aligned(16))) uint16_t qlds[ROPE ? 32 * D : 8];   // q~, rotated once

  const FwdParams& p = P.f;
  const int mask = P.mask;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c = lane & 31;
  const int BH = p.B * p.Hq;
  const int bh = xcd_head(blockIdx.x % BH, BH), mbi = blockIdx.x / BH;
  // causal-type masks: the longest walks first
  const int mb = (mask == MASK_CAUSAL || mask == MASK_CSW) ? p.n_mblocks - 1 - mbi : mbi;
  const int b = bh / p.Hq, hq = bh - b * p.Hq, hk = hq / p.G;
  const int q0 = 32 * mb, qrow = q0 + c;

  const uint16_t* qbase = p.q + b * p.qs[0] + hq * p.qs[1];
  const int64_t kstr = p.ks[2], vstr = p.vs[2];
  const auto krs = make_rsrc(p.k + b * p.ks[0] + hk * p.ks[1], span_bytes<D>(p.Nkv, kstr));
  const float c2 = p.scale * kLog2e;
  const float slope2 = P.alibi ? p.slopes[hq] * kLog2e : 0.f;

  // ---- key tiles of this query block (32 keys; the range starts at a
  // multiple of 64 so that the visit counters see whole 64-key stages)
  int n_lo = 0, n_hi = p.Nkv;
  if (mask == MASK_SW || mask == MASK_CSW) n_lo = max(q0 - p.window + 1, 0) & ~63;
  if (mask == MASK_CAUSAL || mask == MASK_CSW) n_hi = min(q0 + 32, p.Nkv);
  if (mask == MASK_SW) n_hi = min(q0 + 31 + p.window, p.Nkv);
  const int ntiles = n_hi > n_lo ? (n_hi - n_lo + BN - 1) / BN : 0;

  // ---- loads ---------------------------------------------------------------
  uint16_t* const vlds = reinterpret_cast<uint16_t*>(lds + w * L::WAVE_BYTES);
  uint16_t* const klds = vlds + L::TILE;
  const auto vrs = make_rsrc(p.v + b * p.vs[0] + hk * p.vs[1], span_bytes<D>(p.Nkv, vstr));
  // A wave's load covers 64 16-byte chunks: of V 512 / D whole rows, of K
  // one chunk j and its rotate-half partner j + D/16 in two loads of 1024 / D
  // rows.  Rows past the end read as zeros.
  constexpr int VL = BN * D / 512, KP = VL / 2, RPV = 512 / D, TPR = D / 16, RPK = 64 / TPR;
  u32x4 vr[VL], kl[KP], kh[KP];
  const int vrow = lane / (D / 8), vch = lane % (D / 8), krow = lane / TPR, kj = lane % TPR;
  const uint32_t vlane = dma_off(vrow, vstr, 8 * vch), klane = dma_off(krow, kstr, 8 * kj);
  auto load_tile = [&](int t) {
    const int n0 = n_lo + BN * t;
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const uint32_t off = klane + (uint32_t)(n0 + RPK * i) * (uint32_t)kstr * 2u;
      kl[i] = buf_ld16(krs, off);
      kh[i] = buf_ld16(krs, off + D);
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) vr[i] = buf_ld16(vrs, vlane + (uint32_t)(n0 + RPV * i) * (uint32_t)vstr * 2u);
  };

  int t = w;
  if (t < ntiles) load_tile(t);
  // Q fragment (B operand).  With RoPE the workgroup rotates the 32 rows
  // once, through LDS (rotated by every wave for itself they took up to half
  // of a short walk).
  u32x4 qf[KS];
  if constexpr (ROPE) {
    for (int idx = tid; idx < 32 * TPR; idx += 64 * KW) {
      const int r = idx / TPR, j = idx % TPR, n = q0 + r, dl = 8 * j, dh = dl + D / 2;
      u32x4 lo = u32x4{0, 0, 0, 0}, hi = u32x4{0, 0, 0, 0};
      if (n < p.Nq) {
        const uint16_t* qr = qbase + n * p.qs[2];
        const uint16_t* cr = p.cos + n * p.rs[0];
        const uint16_t* sr = p.sin + n * p.rs[0];
        lo = ld16(qr + dl);
        hi = ld16(qr + dh);
        rope_pair<E>(lo, hi, ld16(cr + dl), ld16(sr + dl), ld16(cr + dh), ld16(sr + dh));
      }
      st16(qlds + lds_at<D>(r, dl), lo);
      st16(qlds + lds_at<D>(r, dh), hi);
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = ld16(qlds + lds_at<D>(c, 16 * ks + 8 * h));
  } else {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = qrow < p.Nq ? ld16(qbase + qrow * p.qs[2] + 16 * ks + 8 * h) : u32x4{0, 0, 0, 0};
  }
  int voff[DB][2];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    voff[db][0] = tr_at<D>(lane, 0, db);
    voff[db][1] = tr_at<D>(lane, 1, db);
  }

  constexpr float kTau = 8.f;
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x16{};
  float m_run = -1.0e30f, lsum = 0.f;

  for (; t < ntiles; t += KW) {
    const int n0 = n_lo + BN * t;
    // ---- K(t), V(t) into LDS, then the next tile on its way
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      if constexpr (ROPE && keys_rotates_k(D)) {
        // the table rows are read here and not with the K rows, a tile
        // ahead: held over a whole tile they cost head dim 128 its second
        // wave per SIMD
        const int64_t r = min(n0 + RPK * i + krow, p.Nkv - 1) * p.rs[0] + 8 * kj;
        rope_pair<E>(kl[i], kh[i], ld16(p.cos + r), ld16(p.sin + r), ld16(p.cos + r + D / 2), ld16(p.sin + r + D / 2));
      }
      st16(klds + lds_at<D>(RPK * i + krow, 8 * kj), kl[i]);
      st16(klds + lds_at<D>(RPK * i + krow, 8 * kj + D / 2), kh[i]);
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) st16(vlds + lds_at<D>(RPV * i + vrow, 8 * vch), vr[i]);
    if (t + KW < ntiles) load_tile(t + KW);
    wave_lds_fence();
    // ---- S^T = K Q^T
    f32x16 s = f32x16{};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = E::mfma32(ld16(klds + lds_at<D>(kperm(c), 16 * ks + 8 * h)), qf[ks], s);
    // ---- bias and mask
    if (p.coverage != nullptr && (n0 & 63) == 0 && lane == 0) {
      const int64_t ci = ((int64_t)bh * p.cov_nq + mb) * p.cov_nk + (n0 >> 6);
      atomicAdd(p.coverage + ci, 1u);
    }
    const int base = n0 + 8 * h;              // register r holds key base + 16 (r/8) + r%8
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = s[r] * c2;
    if (P.alibi) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        x[r] = __builtin_fmaf(-slope2, (float)abs(qrow - (base + 16 * (r >> 3) + (r & 7))), x[r]);
    }
    bool need_mask = n0 + BN > p.Nkv;
    if (mask == MASK_CAUSAL || mask == MASK_CSW) need_mask = need_mask || n0 + BN - 1 > q0;
    if (mask == MASK_SW) need_mask = need_mask || n0 + BN - 1 - q0 >= p.window;
    if (mask == MASK_SW || mask == MASK_CSW) need_mask = need_mask || q0 + 31 - n0 >= p.window;
    if (need_mask) {
      int hi = p.Nkv - 1 - base, lo = -base;
      if (mask == MASK_CAUSAL || mask == MASK_CSW) hi = min(hi, qrow - base);
      if (mask == MASK_SW) hi = min(hi, qrow + p.window - 1 - base);
      if (mask == MASK_SW || mask == MASK_CSW) lo = qrow - p.window + 1 - base;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 16 * (r >> 3) + (r & 7);
        x[r] = (kr <= hi && kr >= lo) ? x[r] : -INFINITY;
      }
    }
    // ---- online softmax; the max moves only past the slack kTau
    float mz = x[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mz = fmaxf(mz, x[r]);
    const float mx = max_xor32(mz);
    const bool grow = mx > m_run + kTau;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float m_new = grow ? mx : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
      lsum *= alpha;
      m_run = m_new;
    }
    u32x4 pf[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = __builtin_amdgcn_exp2f(x[r] - m_run);
#pragma unroll
    for (int i = 0; i < 8; ++i) pf[i >> 2][i & 3] = E::pack(x[2 * i], x[2 * i + 1]);
    float ts[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) E::dot_first(pf[0][i], ts[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) E::dot_pair(pf[1][i], ts[i]);
    E::sums_ready(ts[0], ts[1], ts[2], ts[3]);
    lsum += (ts[0] + ts[1]) + (ts[2] + ts[3]);
    // ---- O^T += V^T P^T
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const u32x2 lo = lds_read_tr16(vlds + 16 * j * D + voff[db][0]);
        const u32x2 hi = lds_read_tr16(vlds + 16 * j * D + voff[db][1]);
        o[db] = E::mfma32(u32x4{lo[0], lo[1], hi[0], hi[1]}, pf[j], o[db]);
      }
    wave_lds_fence();
  }

  // ---- merge ---------------------------------------------------------------
  const float lt = lsum + xor32(lsum);
  float* const ow = reinterpret_cast<float*>(lds + w * L::WAVE_BYTES) + c * L::OP;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(ow + 32 * db + 8 * g + 4 * h) =
          f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
  if (h == 0) {
    red[w][0][c] = m_run;
    red[w][1][c] = lt;
  }
  __syncthreads();
  for (int idx = tid; idx < 32 * (D / 8); idx += 64 * KW) {
    const int r = idx / (D / 8), d0 = 8 * (idx % (D / 8));
    const int n = q0 + r;
    if (n >= p.Nq) break;                       // rows ascend with idx
    float M = red[0][0][r];
#pragma unroll
    for (int i = 1; i < KW; ++i) M = fmaxf(M, red[i][0][r]);
    float acc[8], l = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll
    for (int i = 0; i < KW; ++i) {
      const float f = __builtin_amdgcn_exp2f(red[i][0][r] - M);
      l = __builtin_fmaf(f, red[i][1][r], l);
      const float* src = reinterpret_cast<const float*>(lds + i * L::WAVE_BYTES) + r * L::OP + d0;
      const f32x4 a = *reinterpret_cast<const f32x4*>(src), z = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[e] = __builtin_fmaf(f, a[e], acc[e]);
        acc[4 + e] = __builtin_fmaf(f, z[e], acc[4 + e]);
      }
    }
    const float inv = (l == 0.f) ? 1.f : 1.f / l;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= inv;
    st16(p.o + b * p.os[0] + hq * p.os[1] + (int64_t)n * p.os[2] + d0, pack8<E>(acc));
    if (p.lse != nullptr && d0 == 0) {
      float Lv = -INFINITY;
      if (l > 0.f) Lv = (M + __log2f(l)) * kLn2;
      p.lse[b * p.ls[0] + hq * p.ls[1] + (int64_t)n * p.ls[2]] = Lv;
    }
  }
}

}  // namespace af
