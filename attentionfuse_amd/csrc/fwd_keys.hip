// Launcher of the key-split forward for small grids (fwd_keys_kernel).
#include "fwd_keys_kernel.hpp"
#include "launch.hpp"

namespace af {

namespace {

template <class E, int D, bool ROPE, int KW>
int go(const FwdKeysParams& P, hipStream_t s) {
  const dim3 grid((unsigned)(P.f.n_mblocks * P.f.B * P.f.Hq));
  hipLaunchKernelGGL((fwd_keys_kernel<E, D, ROPE, KW>), grid, dim3(KW * 64), 0, s, P);
  return 0;
}

template <class E, int D>
int pick(const FwdKeysParams& P, int kw, bool rope, hipStream_t s) {
  if (kw == 4) return rope ? go<E, D, true, 4>(P, s) : go<E, D, false, 4>(P, s);
  if (kw == 8) return rope ? go<E, D, true, 8>(P, s) : go<E, D, false, 8>(P, s);
  return -1;
}

template <class E>
int pick_d(const FwdKeysParams& P, int d, int kw, bool rope, hipStream_t s) {
  switch (d) {
    case 32: return pick<E, 32>(P, kw, rope, s);
    case 64: return pick<E, 64>(P, kw, rope, s);
    case 128: return pick<E, 128>(P, kw, rope, s);
  }
  return -1;
}

}  // namespace

int launch_fwd_keys(const FwdParams& p, int dtype, int d, int mask, int bias, bool rope, int kw, hipStream_t s) {
  FwdKeysParams P;
  P.f = p;
  P.f.n_mblocks = (p.Nq + 31) / 32;
  P.mask = mask;
  P.alibi = bias == BIAS_ALIBI;
  return dtype == AF_F16 ? pick_d<F16>(P, d, kw, rope, s) : pick_d<BF16>(P, d, kw, rope, s);
}

}  // namespace af
