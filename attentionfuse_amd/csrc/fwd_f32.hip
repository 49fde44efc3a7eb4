// Launchers of the fp32 forward (fwd_f32_kernel) and its key rotation.
#include "fwd_f32_kernel.hpp"
#include "launch.hpp"

namespace af {

template <int D, int KW>
static int go(const FwdF32Params& p, int blocks, hipStream_t s) {
  FwdF32Params q = p;
  q.f.n_mblocks = blocks;
  hipLaunchKernelGGL((fwd_f32_kernel<D, KW>), dim3((unsigned)(blocks * p.f.B * p.f.Hq)),
                     dim3((KW > 1 ? KW : kF32Waves) * 64), 0, s, q);
  return 0;
}

template <int D>
static int pick_kw(const FwdF32Params& p, hipStream_t s) {
  const int blocks32 = (p.f.Nq + 31) / 32;   // of one head
  switch (f32_key_waves(D, (int64_t)blocks32 * p.f.B * p.f.Hq)) {
    case 8:
      if constexpr (D <= 64) return go<D, 8>(p, blocks32, s);
      return -1;
    case 4: return go<D, 4>(p, blocks32, s);
    case 2: return go<D, 2>(p, blocks32, s);
  }
  return go<D, 1>(p, (p.f.Nq + kF32BlockM - 1) / kF32BlockM, s);
}

int launch_fwd_f32(const FwdF32Params& p, int head_dim, hipStream_t s) {
  switch (head_dim) {
    case 32: return pick_kw<32>(p, s);
    case 64: return pick_kw<64>(p, s);
    case 128: return pick_kw<128>(p, s);
  }
  return -1;
}

int launch_rope_f32(const float* x, float* out, const float* cs, const float* sn, const int64_t* xs, int64_t rs,
                    int H, int N, int64_t rows, int head_dim, hipStream_t s) {
  const int64_t threads = rows * (head_dim / 2);
  const int64_t blocks = (threads + 255) / 256;
  if (blocks <= 0) return 0;
  switch (head_dim) {
    case 32:
      hipLaunchKernelGGL((rope_f32_kernel<32>), dim3((unsigned)blocks), dim3(256), 0, s, x, out, cs, sn, xs[0], xs[1],
                         xs[2], rs, H, N, rows);
      return 0;
    case 64:
      hipLaunchKernelGGL((rope_f32_kernel<64>), dim3((unsigned)blocks), dim3(256), 0, s, x, out, cs, sn, xs[0], xs[1],
                         xs[2], rs, H, N, rows);
      return 0;
    case 128:
      hipLaunchKernelGGL((rope_f32_kernel<128>), dim3((unsigned)blocks), dim3(256), 0, s, x, out, cs, sn, xs[0],
                         xs[1], xs[2], rs, H, N, rows);
      return 0;
  }
  return -1;
}

}  // namespace af
