"""The float32 kernels on cut bf16 pieces (fa_f32.hpp, and the key-split forward
of small grids) at the edges of their tiles: O, LSE and the gradients within
1e-5 of max|oracle| as the other float32 cases, and no further from float64 than
the float32 matrix instruction's own rounding; infinities stay infinities."""
import pytest
import torch

from flash_attention_v100 import _lib
from helpers import assert_parity, c_keep_mask, compare, make_inputs

pytestmark = pytest.mark.gpu

CASES = [
    # B, Sq, Sk, H, Hkv, D, causal, p
    (1, 1, 1, 1, 1, 32, False, 0.0),
    (1, 31, 33, 2, 1, 64, False, 0.0),
    (2, 129, 129, 4, 2, 128, True, 0.0),
    (1, 130, 65, 3, 3, 32, True, 0.1),
    (4, 127, 257, 64, 16, 64, False, 0.0),   # 256 forward workgroups, grouped heads
    (2, 200, 200, 64, 64, 32, True, 0.2),    # 256 workgroups, dropout
    (4, 100, 161, 64, 64, 128, False, 0.1),  # 256 workgroups
    (2, 257, 96, 48, 48, 128, True, 0.0),    # fewer keys than queries
]


@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_f32_parity(case, stored):
    B, Sq, Sk, H, Hkv, D, causal, p = case
    if stored and p == 0:
        pytest.skip("no mask to store")
    print(f"case: f32 {case} stored={stored}", flush=True)
    q, k, v, do = make_inputs(B, Sq, H, D, torch.float32, Sk=Sk, Hkv=Hkv, seed=Sq + D, device="cuda")
    scale = D ** -0.5
    bits = _lib.alloc_keep_bits(B, H, Sq, Sk, q.device) if stored else None
    o, lse, _ = _lib.fwd(q, k, v, causal, scale, p, 77, 5, keep_bits=bits)
    dq, dk, dv = _lib.bwd(q, k, v, o, do, lse, causal, scale, p, 77, 5, keep_bits=bits)
    torch.cuda.synchronize()
    keep = torch.from_numpy(c_keep_mask(77, 5, B, H, Sq, Sk, p)).cuda() if p > 0 else None
    assert_parity(compare(q, k, v, do, causal, scale, (o, lse, dq, dk, dv), keep=keep, p=p), torch.float32, str(case))


@pytest.mark.parametrize("B", [1, 64])  # the key-split forward, and fwd32_kernel
def test_f32_range(B):
    # values whose lower pieces matter (1 + 2^-23), huge and infinite ones
    g = torch.Generator("cpu").manual_seed(3)
    q, k = (torch.randn(B, 64, 4, 64, generator=g).cuda() for _ in range(2))
    v = torch.full((B, 64, 4, 64), 1.0 + 2.0 ** -23, device="cuda")
    v[:, :, 1] = 1e34  # (sums before the normalisation reach 64 * 2^8 times it)
    v[:, 3, 2, 5] = float("inf")
    v[:, 4, 2, 6] = -float("inf")
    o, _, _ = _lib.fwd(q, k, v, False, 0.125)
    # a convex combination of equal values: 64 products and sums of relative
    # error 2^-24 each, and the normalisation's
    assert ((o[:, :, 0].double() / (1.0 + 2.0 ** -23)) - 1).abs().max().item() < 70 * 2.0 ** -24
    assert ((o[:, :, 1].double() / 1e34) - 1).abs().max().item() < 70 * 2.0 ** -24
    assert (o[:, :, 2, 5] == float("inf")).all() and (o[:, :, 2, 6] == -float("inf")).all()
    cols = [c for c in range(64) if c not in (5, 6)]
    assert torch.isfinite(o[:, :, 2][..., cols]).all()
    # a key of -inf in every column met by positive q gets no weight
    kk = k.clone()
    kk[:, 7] = -float("inf")
    o, lse, _ = _lib.fwd(q.abs() + 0.1, kk, v[:, :, :1].expand_as(v).contiguous(), False, 0.125)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
