"""Forward on both sides of the line between the key-split kernel of small
grids (8 or 4 waves on one 32-row query block) and the 128-row kernel.

Head counts put the grid on each side of every step of the rule; lengths
leave ragged last tiles and blocks and waves with no visible tile.  Outputs
and the log-sum-exp against the fp32 oracle at the tolerances of the other
forward tests (the merge of the waves adds a few roundings of 2^-24).
"""
import pytest
import torch

import attnfuse as af
import oracle as O
from attentionfuse_amd.runtime.dispatch import run_attention
from attnfuse.rope_utils import build_rope_cache
from test_fwd_gpu import LSE_TOL, TOL, make, oracle_kwargs, run_case, variant

pytestmark = pytest.mark.gpu
DTYPES = [torch.float16, torch.bfloat16]

# (heads, head dim) at N = 161 (6 blocks of 32 rows a head): 8 waves, 4
# waves, past the dense line, past the causal one
GRIDS = [(2, 32), (60, 32), (120, 32), (180, 32), (2, 64), (60, 64), (100, 64), (135, 64),
         (2, 128), (44, 128), (70, 128), (90, 128)]


@pytest.mark.parametrize("dtype", DTYPES, ids=["f16", "bf16"])
@pytest.mark.parametrize("H,D", GRIDS)
@pytest.mark.parametrize("name", ["dense", "causal", "sw", "sw_causal_alibi", "rope_causal_alibi"])
def test_both_sides_of_the_line(name, H, D, dtype):
    print(f"[fwd] {name} {dtype} H={H} D={D} N=161", flush=True)
    N = 161
    Q, K, V = make(1, H, H, N, N, D, dtype, seed=H)
    kw, rope = {}, None
    if name.startswith("rope"):
        cos, sin = build_rope_cache(N, D, device="cuda", dtype=dtype)
        kw, rope = dict(cos=cos, sin=sin), (cos[0, 0].cpu(), sin[0, 0].cpu())
    out = af.attention(variant(name, H))(Q, K, V, **kw)
    torch.cuda.synchronize()
    # Against q~, k~ rounded to the input type, which is how the path defines
    # them: over millions of outputs that rounding alone, 2^-11 of each
    # operand, moves a fp16 logit of 10 by up to 2^-10 * 10 and an output by
    # 2e-3, the whole bound of the other cases.
    want = O.naive_attention(Q.cpu(), K.cpu(), V.cpu(), rope_round=dtype if rope else None,
                             **oracle_kwargs(name, H, Q, rope=rope))
    assert (out.float().cpu() - want).abs().max().item() <= TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=["f16", "bf16"])
@pytest.mark.parametrize("Nq,Nkv", [(1, 31), (2, 33), (31, 1), (33, 1000), (100, 257), (3, 4097)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_few_rows(D, Nq, Nkv, dtype):
    print(f"[fwd] dense {dtype} D={D} {Nq}x{Nkv}", flush=True)
    assert run_case("dense", 1, 4, 2, Nq, D, dtype, Nkv=Nkv) <= TOL[dtype]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("name", ["causal", "sw", "rope_dense"])
def test_strided_views_lse_and_coverage(name, D):
    """(B, N, H, D) projections as strided views, the saved log-sum-exp and
    the tile-visit counters, on a grid of 8 waves a block."""
    B, H, N, dtype, W = 2, 6, 203, torch.float16, 40
    Q, K, V = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in make(B, H, H // 2, N, N, D, dtype, seed=5))
    kw, rope = {}, None
    if name.startswith("rope"):
        cos, sin = build_rope_cache(N, D, device="cuda", dtype=dtype)
        kw, rope = dict(cos=cos, sin=sin), (cos[0, 0].cpu(), sin[0, 0].cpu())
    g = af.attention(variant(name, H, window=W))(Q, K, V, return_graph=True)
    L = torch.empty(B, H, N, device="cuda")
    cov = torch.zeros(B, H, -(-N // 32), -(-N // 64), dtype=torch.int32, device="cuda")
    out = run_attention(g, Q, K, V, save_lse=L, coverage=cov, **kw)
    torch.cuda.synchronize()
    okw = oracle_kwargs(name, H, Q, window=W, rope=rope)
    want, want_l = O.naive_attention(Q.cpu(), K.cpu(), V.cpu(), return_lse=True, **okw)
    assert (out.float().cpu() - want).abs().max().item() <= TOL[dtype]
    assert (L.cpu() - want_l).abs().max().item() <= LSE_TOL[dtype]
    wc = O.expected_coverage(N, N, mask={"causal": "causal", "sw": "sliding_window"}.get(name, "full"), window=W)
    assert torch.equal(cov.cpu(), wc.expand(B, H, *wc.shape))
