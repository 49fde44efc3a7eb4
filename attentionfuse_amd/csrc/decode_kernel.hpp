// Flash-decoding for gfx950 (piece (b)): one query row per head, the KV
// cache split over workgroups, then a log-sum-exp combine.
//
// Semantics follow the reference decode kernels
// (reference: attnfuse/compiler/codegen_decode.py:46-211): per split, an
// online softmax over its keys gives (m, l, acc); the combine kernel merges
// m* = max m_s, l* = sum e^(m_s - m*) l_s, O = sum e^(m_s - m*) acc_s / l*.
// ALiBi uses the query position N_kv - 1: bias = -slope_h |(N_kv-1) - j|
// (codegen_decode.py:142-145).  Unlike the reference, split boundaries are
// exact: every key is counted once whatever N_kv is.
//
// Work decomposition:
//  * one workgroup = (split, batch, kv head, chunk of up to 16 query heads
//    of that kv head's GQA group): the group shares every K/V byte read, so
//    the cache is streamed once per (batch, kv head) whatever the group size;
//  * the four waves interleave 32-key steps inside the split; each wave
//    keeps its own (m, l, O^T) and the waves merge through LDS at the end;
//  * S^T = K Q^T on the 16x16x32 MFMA with K read straight from HBM into the
//    A operand (16-byte loads, no LDS); O^T += V^T P^T on the same MFMA with
//    V rows passed through a per-wave LDS tile, read transposed; P^T feeds
//    the MFMA from registers;
//  * a cache that is not split (one workgroup per key/value head fills the
//    chip, or the cache is short) is finished by its workgroup: no partials
//    and no combine launch.
//
// Bound by HBM for large caches (bf16, B = 8, 8 key/value heads of 128 dims,
// 32768 keys: 1.07 GB in 181 us, 5.9 TB/s, where a read-only probe peaks at
// 6.2) and by latency for small ones.  V rows written whole to LDS and read
// back by transposing reads, vector partials, and a combine that reads all
// splits' (m, l) at once took one sequence's step (8 key/value heads) from
// 12.2 to 7.6 us at 1024 keys, 16.4 to 9.2 at 4096, 48.4 to 30.4 at 32768, and
// 16 x 12 heads of 64 dims x 3001 keys from 39.3 to 31.8 (before, V was
// written transposed word by word and the (m, l) pairs were read one after the
// other).
#pragma once

#include "af_common.hpp"

namespace af {

struct DecodeParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  const float* slopes;
  float* ws_acc;   // (S, B, Hq, D) fp32: unnormalised accumulator
  float* ws_ml;    // (S, B, Hq, 2) fp32: m (log2 units), l
  int64_t qs[4], ks[4], vs[4], os[4];
  int32_t B, Hq, Hkv, Nkv, G, nqc, nsplit, split_len;
  float scale;
};

// 16x16x32 MFMA layouts (lane l, group g = l / 16):
//   A (16 x 32): row l%16, k-slots 8g..8g+7     B (32 x 16): column l%16
//   C (16 x 16, 4 fp32): register r holds row 4g + r, column l%16.
// Two 16-key score blocks give lane (g, q) keys {4g + r} and {16 + 4g + r};
// those eight values are the B operand of the P*V MFMA over 32 keys when the
// V^T A operand uses the same key slots: slot e < 4 -> key 4g + e,
// slot e >= 4 -> key 16 + 4g + (e - 4).

// LDS chunk (16 bytes) of chunk k of row r of a wave's V tile.  A transposing
// read takes 8 rows of one 32-byte chunk pair per 32 lanes: XORing the pair
// with the row spreads them over all 64 banks (rows of 64 and 128 bytes share
// a bank row four and two at a time).
template <int D>
__device__ __forceinline__ int dec_v_chunk(int r, int k) {
  const int f = D >= 128 ? r & 7 : D == 64 ? (r >> 1) & 3 : (r >> 2) & 1;
  return k ^ (2 * f);
}

template <class E, int D, int BIAS>
__global__ void __launch_bounds__(256) decode_split_kernel(const DecodeParams p) {
  constexpr int KSD = D / 32;      // 32-deep k-steps of K Q^T
  constexpr int DB = D / 16;       // 16-row blocks of O^T
  constexpr int VT_ELEMS = 32 * D; // a wave's V tile
  constexpr int RPV = 512 / D;     // V rows per wave load
  constexpr int VL = 32 / RPV;     // loads per V tile
  // the waves' V tiles; after the walk their (m, l) and O
  constexpr int LDS_BYTES = 4 * VT_ELEMS * 2 > (128 + 64 * D) * 4 ? 4 * VT_ELEMS * 2 : (128 + 64 * D) * 4;
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_BYTES];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int split = blockIdx.x;
  int rest = blockIdx.y;
  const int qc = rest % p.nqc; rest /= p.nqc;
  const int hk = rest % p.Hkv;
  const int b = rest / p.Hkv;
  const int hq0 = hk * p.G + 16 * qc;
  const int nq = min(16, p.G - 16 * qc);   // real query heads in this chunk
  const int hq = hq0 + c;                  // this lane's query column
  const bool qreal = c < nq;

  const int64_t kstr = p.ks[2], vstr = p.vs[2];
  const int vrow = lane / (D / 8), vch = lane % (D / 8);
  const uint16_t* __restrict__ kbase = p.k + b * p.ks[0] + hk * p.ks[1] + c * kstr + 8 * g;
  const uint16_t* __restrict__ vbase = p.v + b * p.vs[0] + hk * p.vs[1] + vrow * vstr + 8 * vch;

  // Q^T as B operand: lane (g, q = c) holds Q[q][32 ks + 8 g .. +7].
  u32x4 qf[KSD];
  {
    const uint16_t* qrow = p.q + b * p.qs[0] + (int64_t)(qreal ? hq : hq0) * p.qs[1];
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks)
      qf[ks] = qreal ? ld16(qrow + 32 * ks + 8 * g) : u32x4{0, 0, 0, 0};
  }
  const float c2 = p.scale * kLog2e;
  float slope2 = 0.f;
  if constexpr (BIAS == 1) slope2 = qreal ? p.slopes[hq] * kLog2e : 0.f;

  const int s_lo = split * p.split_len;
  const int s_hi = min(s_lo + p.split_len, p.Nkv);
  const int nsteps = s_hi > s_lo ? (s_hi - s_lo + 31) / 32 : 0;

  f32x4 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x4{};
  float m_run = -INFINITY, l_run = 0.f;
  uint16_t* vt = reinterpret_cast<uint16_t*>(lds) + w * VT_ELEMS;
  // LDS element offsets of this lane's V chunk of load i (16-byte writes) and
  // of its transposing reads: within a 16-lane group, result lane L element i
  // is element L % 4 of the 8 bytes that lane L / 4 + 4 i addresses, so lane
  // a + 4 i addresses key row 4 g + i (+ 16 for the second read), dims 4 a.
  auto v_at = [&](int row, int col) -> int { return row * D + 8 * dec_v_chunk<D>(row, col >> 3) + (col & 7); };
  const int trow = 4 * g + (c >> 2), tcol = 4 * (c & 3);

  // One 32-key step of this wave: K rows (A operand of S^T, keys k0 + 16 kb
  // + c) and V rows straight from HBM into registers; only a split's last
  // step has rows past its end (zeros).
  struct StepRegs {
    u32x4 ka[2][KSD];
    u32x4 va[VL];
  };
  auto load_step = [&](int st, StepRegs& r) {
    const int k0 = s_lo + 32 * st;
    const uint16_t* kp = kbase + k0 * kstr;
    const uint16_t* vp = vbase + k0 * vstr;
    if (k0 + 32 <= s_hi) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks) r.ka[kb][ks] = ld16(kp + 16 * kb * kstr + 32 * ks);
#pragma unroll
      for (int i = 0; i < VL; ++i) r.va[i] = ld16(vp + RPV * i * vstr);
    } else {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int ks = 0; ks < KSD; ++ks)
          r.ka[kb][ks] = k0 + 16 * kb + c < s_hi ? ld16(kp + 16 * kb * kstr + 32 * ks) : u32x4{0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < VL; ++i)
        r.va[i] = k0 + RPV * i + vrow < s_hi ? ld16(vp + RPV * i * vstr) : u32x4{0, 0, 0, 0};
    }
  };
  auto compute_step = [&](int st, const StepRegs& r) {
    const int k0 = s_lo + 32 * st;
    // S^T blocks.
    f32x4 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s[kb] = f32x4{};
#pragma unroll
      for (int ks = 0; ks < KSD; ++ks) s[kb] = E::mfma16(r.ka[kb][ks], qf[ks], s[kb]);
    }
    // V rows into this wave's LDS tile.
#pragma unroll
    for (int i = 0; i < VL; ++i) st16(vt + v_at(RPV * i + vrow, 8 * vch), r.va[i]);
    // Online softmax on this lane's eight keys of query c.
    float x[8];
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int key = k0 + 16 * kb + 4 * g + rr;
        float v = s[kb][rr] * c2;
        if constexpr (BIAS == 1) v -= slope2 * (float)abs((p.Nkv - 1) - key);
        v = key < s_hi ? v : -INFINITY;
        x[4 * kb + rr] = v;
        mx = fmaxf(mx, v);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    float ls = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = __builtin_amdgcn_exp2f(x[i] - m_use);
      ls += x[i];
    }
    l_run = l_run * alpha + ls;
    m_run = m_new;
    u32x4 pb;
#pragma unroll
    for (int i = 0; i < 4; ++i) pb[i] = E::pack(x[2 * i], x[2 * i + 1]);

    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const u32x2 lo = lds_read_tr16(vt + v_at(trow, 16 * db + tcol));
      const u32x2 hi = lds_read_tr16(vt + v_at(trow + 16, 16 * db + tcol));
      const u32x4 va4 = {lo[0], lo[1], hi[0], hi[1]};
      o[db] = o[db] * alpha;
      o[db] = E::mfma16(va4, pb, o[db]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // The loads of step st + 4 are issued before step st is computed, so each
  // wave keeps two steps (16 KB at D = 128) of K/V in flight.
  StepRegs ra, rb;
  if (w < nsteps) load_step(w, ra);
  for (int st = w; st < nsteps; st += 8) {
    if (st + 4 < nsteps) load_step(st + 4, rb);
    compute_step(st, ra);
    if (st + 4 >= nsteps) break;
    if (st + 8 < nsteps) load_step(st + 8, ra);
    compute_step(st + 4, rb);
  }

  // ---- merge the four waves through LDS ------------------------------------
  // Per wave: l summed over the four lane groups; m is already uniform.
  float lw = l_run + __shfl_xor(l_run, 16, 64);
  lw += __shfl_xor(lw, 32, 64);
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
  float* red_m = red;              // [4][16]
  float* red_l = red + 64;         // [4][16]
  float* red_o = red + 128;        // [4][16][D]  (q-major)
  if (qreal) {
    if (g == 0) {
      red_m[w * 16 + c] = m_run;
      red_l[w * 16 + c] = lw;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db)
      *reinterpret_cast<f32x4*>(red_o + (w * 16 + c) * D + 16 * db + 4 * g) = o[db];
  }
  __syncthreads();
  // 256 threads merge the nq x D outputs, four dims each.
  for (int idx = tid; idx < nq * (D / 4); idx += 256) {
    const int qq = idx / (D / 4), d = 4 * (idx % (D / 4));
    float mstar = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) mstar = fmaxf(mstar, red_m[ww * 16 + qq]);
    const float mu = (mstar == -INFINITY) ? 0.f : mstar;
    f32x4 acc = f32x4{};
    float lsum = 0.f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      const float f = __builtin_amdgcn_exp2f(red_m[ww * 16 + qq] - mu);
      const f32x4 ov = *reinterpret_cast<const f32x4*>(red_o + (ww * 16 + qq) * D + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += f * ov[e];
      lsum += f * red_l[ww * 16 + qq];
    }
    if (p.nsplit == 1) {
      const float inv = (lsum == 0.f) ? 1.f : 1.f / lsum;
      uint16_t* orow = p.o + b * p.os[0] + (hq0 + qq) * p.os[1] + d;
#pragma unroll
      for (int e = 0; e < 4; ++e) orow[e] = E::one(acc[e] * inv);   // o has no alignment promise
    } else {
      const int64_t row = ((int64_t)split * p.B + b) * p.Hq + hq0 + qq;
      *reinterpret_cast<f32x4*>(p.ws_acc + row * D + d) = acc;
      if (d == 0) *reinterpret_cast<f32x2*>(p.ws_ml + 2 * row) = f32x2{mstar, lsum};
    }
  }
}

// Combine: one 256-thread workgroup per (batch, query head).  Each wave takes
// the maximum of all splits' m on its own, one per lane; thread t then turns
// the (m, l) pair of split t into a weight 2^(m_t - m*) in LDS, and a thread
// sums four output dims over every NG-th split (its loads are independent),
// the NG sums meeting in LDS.  Read one after the other by every thread, the
// pairs of 64 splits took most of the kernel.
template <class E, int D, bool F32OUT = false>
__global__ void __launch_bounds__(256) decode_combine_kernel(const DecodeParams p) {
  constexpr int TPR = D / 4;                  // threads per partial row
  constexpr int NG = 256 / TPR;
  __shared__ __attribute__((aligned(16))) float red_acc[NG][D];
  __shared__ float wt[256];
  __shared__ float red_l[4];
  const int t = threadIdx.x, lane = t & 63;
  const int d = 4 * (t % TPR), grp = t / TPR;
  const int row = blockIdx.x;                 // b * Hq + hq
  const int b = row / p.Hq, hq = row - b * p.Hq;
  const int S = p.nsplit;
  const int64_t plane = (int64_t)p.B * p.Hq;
  float mstar = -INFINITY;
  for (int s = lane; s < S; s += 64) mstar = fmaxf(mstar, p.ws_ml[2 * (s * plane + row)]);
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) mstar = fmaxf(mstar, __shfl_xor(mstar, off, 64));
  const float mu = (mstar == -INFINITY) ? 0.f : mstar;
  float lsum = 0.f;
  f32x4 acc = f32x4{};
  for (int c0 = 0; c0 < S; c0 += 256) {       // one pass but for explicit split counts
    if (c0 > 0) __syncthreads();
    if (c0 + t < S) {
      const f32x2 ml = *reinterpret_cast<const f32x2*>(p.ws_ml + 2 * ((c0 + t) * plane + row));
      const float f = __builtin_amdgcn_exp2f(ml[0] - mu);
      wt[t] = f;
      lsum += f * ml[1];
    }
    __syncthreads();
    const int n = min(256, S - c0);
#pragma unroll 4
    for (int s = grp; s < n; s += NG) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(p.ws_acc + ((c0 + s) * plane + row) * D + d);
      const float f = wt[s];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += f * x[e];
    }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) lsum += __shfl_xor(lsum, off, 64);
  if (lane == 0) red_l[t >> 6] = lsum;
  *reinterpret_cast<f32x4*>(&red_acc[grp][d]) = acc;
  __syncthreads();
  if (t < D) {
    const float l = (red_l[0] + red_l[1]) + (red_l[2] + red_l[3]);
    float a = 0.f;
#pragma unroll
    for (int g2 = 0; g2 < NG; ++g2) a += red_acc[g2][t];
    a *= (l == 0.f) ? 1.f : 1.f / l;
    if constexpr (F32OUT)
      reinterpret_cast<float*>(p.o)[b * p.os[0] + hq * p.os[1] + t] = a;
    else
      p.o[b * p.os[0] + hq * p.os[1] + t] = E::one(a);
  }
}

// ---------------------------------------------------------------------------
// fp32 split kernel.  Decode reads every K/V byte once and does 4 FLOP per
// 4 bytes read, so fp32 FMAs on the VALU keep up with HBM and no fp32 MFMA
// is needed.  Lane (k, c) = (lane / 8, lane % 8) holds dims [c D/8, (c+1)
// D/8) of key slot k: a wave covers 8 keys per step, the dot products are
// finished with three xor shuffles inside each group of 8 lanes, and the
// running max of a query head is wave-uniform after three more.  A
// workgroup serves up to kF32DecHeads(D) query heads of one key/value head,
// so each K/V row is read once for all of them; each wave keeps the K/V rows
// of its next step in flight while it computes the current one.  The
// partials (m in log2 units, l, acc) use the 16-bit kernel's workspace
// layout, so the combine kernel is the same.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int f32_decode_heads(int D) { return 64 / (D / 8) < 16 ? 64 / (D / 8) : 16; }
template <int D>
constexpr int kF32DecHeads() { return f32_decode_heads(D); }

// GQ: query heads per workgroup, kF32DecHeads(D), or 1 where every key/value
// head has one query head (the other slots would repeat it: 4 x 12 heads of 64
// dims, 4096 keys, 54.6 -> 22.2 us).
template <int D, int BIAS, int GQ>
__global__ void __launch_bounds__(256) decode_split_f32_kernel(const DecodeParams p) {
  constexpr int CH = D / 8;                 // dims per lane
  __shared__ float red[4][GQ][2 + D];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int kk = lane >> 3, c = lane & 7;
  const int split = blockIdx.x;
  int rest = blockIdx.y;
  const int qc = rest % p.nqc;
  rest /= p.nqc;
  const int hk = rest % p.Hkv;
  const int b = rest / p.Hkv;
  const int hq0 = hk * p.G + GQ * qc;
  const int nq = min(GQ, p.G - GQ * qc);    // real query heads in this chunk

  const float* kbase = reinterpret_cast<const float*>(p.k) + b * p.ks[0] + hk * p.ks[1] + CH * c;
  const float* vbase = reinterpret_cast<const float*>(p.v) + b * p.vs[0] + hk * p.vs[1] + CH * c;
  // this lane's dims of every query head of the chunk, pre-scaled to log2
  // units (the scale multiplies the fp32 dot product; no rounding involved)
  const float c2 = p.scale * kLog2e;
  float q[GQ][CH];
#pragma unroll
  for (int g = 0; g < GQ; ++g) {
    const float* qr = reinterpret_cast<const float*>(p.q) + b * p.qs[0] + (int64_t)(hq0 + min(g, nq - 1)) * p.qs[1] +
                      CH * c;
#pragma unroll
    for (int e = 0; e < CH; e += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(qr + e);
#pragma unroll
      for (int j = 0; j < 4; ++j) q[g][e + j] = v[j];
    }
  }
  float slope2[GQ];
#pragma unroll
  for (int g = 0; g < GQ; ++g) slope2[g] = BIAS == 1 ? p.slopes[hq0 + min(g, nq - 1)] * kLog2e : 0.f;

  const int s_lo = split * p.split_len;
  const int s_hi = min(s_lo + p.split_len, p.Nkv);
  const int nsteps = s_hi > s_lo ? (s_hi - s_lo + 7) / 8 : 0;

  float m[GQ], l[GQ], acc[GQ][CH];
#pragma unroll
  for (int g = 0; g < GQ; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < CH; ++e) acc[g][e] = 0.f;
  }

  // rows of key slot kk of step st (clamped to the last key: every load is
  // in bounds, and scores of keys >= s_hi are masked)
  auto load = [&](int st, float (&kr)[CH], float (&vr)[CH]) {
    const int key = min(s_lo + 8 * st + kk, s_hi - 1);
#pragma unroll
    for (int e = 0; e < CH; e += 4) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(kbase + (int64_t)key * p.ks[2] + e);
      const f32x4 v = *reinterpret_cast<const f32x4*>(vbase + (int64_t)key * p.vs[2] + e);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kr[e + j] = a[j];
        vr[e + j] = v[j];
      }
    }
  };
  auto compute = [&](int st, const float (&kr)[CH], const float (&vr)[CH]) {
    const int key = s_lo + 8 * st + kk;
    const bool ok = key < s_hi;
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < CH; ++e) d = __builtin_fmaf(q[g][e], kr[e], d);
      d += __shfl_xor(d, 1, 64);
      d += __shfl_xor(d, 2, 64);
      d += __shfl_xor(d, 4, 64);
      float x = d * c2;
      if constexpr (BIAS == 1) x -= slope2[g] * (float)abs((p.Nkv - 1) - key);
      x = ok ? x : -INFINITY;
      float mx = fmaxf(x, __shfl_xor(x, 8, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m[g], mx);   // wave-uniform
      if (m_new > m[g]) {
        const float alpha = __builtin_amdgcn_exp2f(m[g] - m_new);   // 0 while m = -inf
        l[g] *= alpha;
#pragma unroll
        for (int e = 0; e < CH; ++e) acc[g][e] *= alpha;
        m[g] = m_new;
      }
      const float pr = (m[g] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(x - m[g]);
      l[g] += pr;
#pragma unroll
      for (int e = 0; e < CH; ++e) acc[g][e] = __builtin_fmaf(pr, vr[e], acc[g][e]);
    }
  };
  float ka[CH], va[CH], kb2[CH], vb[CH];
  if (w < nsteps) load(w, ka, va);
  for (int st = w; st < nsteps; st += 8) {
    if (st + 4 < nsteps) load(st + 4, kb2, vb);
    compute(st, ka, va);
    if (st + 4 >= nsteps) break;
    if (st + 8 < nsteps) load(st + 8, ka, va);
    compute(st + 4, kb2, vb);
  }

  // ---- per wave: sums over the 8 key slots, then the 4 waves through LDS --
#pragma unroll
  for (int g = 0; g < GQ; ++g) {
    l[g] += __shfl_xor(l[g], 8, 64);
    l[g] += __shfl_xor(l[g], 16, 64);
    l[g] += __shfl_xor(l[g], 32, 64);
#pragma unroll
    for (int e = 0; e < CH; ++e) {
      float a = acc[g][e];
      a += __shfl_xor(a, 8, 64);
      a += __shfl_xor(a, 16, 64);
      a += __shfl_xor(a, 32, 64);
      acc[g][e] = a;
    }
  }
  if (kk == 0) {
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
      if (c == 0) {
        red[w][g][0] = m[g];
        red[w][g][1] = l[g];
      }
#pragma unroll
      for (int e = 0; e < CH; ++e) red[w][g][2 + CH * c + e] = acc[g][e];
    }
  }
  __syncthreads();
  for (int idx = tid; idx < GQ * D; idx += 256) {
    const int g = idx / D, d = idx - g * D;
    if (g >= nq) continue;
    float mstar = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) mstar = fmaxf(mstar, red[ww][g][0]);
    const float mu = (mstar == -INFINITY) ? 0.f : mstar;
    float a = 0.f, ls = 0.f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      const float f = __builtin_amdgcn_exp2f(red[ww][g][0] - mu);
      a += f * red[ww][g][2 + d];
      ls += f * red[ww][g][1];
    }
    const int64_t row = ((int64_t)split * p.B + b) * p.Hq + hq0 + g;
    p.ws_acc[row * D + d] = a;
    if (d == 0) {
      p.ws_ml[2 * row] = mstar;
      p.ws_ml[2 * row + 1] = ls;
    }
  }
}

}  // namespace af
