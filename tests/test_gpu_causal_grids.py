"""Causal grids of one to two 128-row workgroups per CU, at the lines where the
launchers change kernels (key-split forward and dQ, the 8-wave dK/dV, the
combined backward): O, LSE, dQ, dK, dV against the float64 oracle with the
tolerance of the other parity tests, and the whole backward equal to its two
passes bit for bit."""
import ctypes

import pytest
import torch

from flash_attention_v100 import _lib
from helpers import assert_parity, compare, make_inputs

pytestmark = pytest.mark.gpu

CASES = [
    # B, Sq, Sk, H, Hkv, D, dtype: workgroups of 128 queries / keys
    (4, 512, 512, 16, 16, 64, torch.bfloat16),    # 256 / 256: combined backward
    (8, 513, 513, 8, 8, 64, torch.float16),       # 320 / 320
    (2, 1000, 1000, 16, 16, 128, torch.bfloat16),  # 256 / 256
    (3, 1024, 1024, 16, 4, 128, torch.float16),   # 384 / 96: grouped heads
    (1, 1600, 1600, 24, 24, 128, torch.bfloat16),  # 312 / 312: 8-wave dK/dV
    (1, 2100, 2100, 20, 20, 64, torch.float16),   # 340 / 340: long chains, slices that straddle XCDs
    (2, 2050, 2050, 8, 8, 64, torch.float16),     # 272 / 272: the same with key-split dQ and forward
    (1, 2100, 2100, 24, 24, 64, torch.bfloat16),  # 408 / 408: whole slices per XCD
    (1, 2048, 2304, 32, 32, 64, torch.bfloat16),  # 512 / 576: the last of the rules, keys no query sees
    (1, 2049, 2049, 32, 32, 32, torch.bfloat16),  # 544: past them
    (2, 512, 512, 32, 32, 32, torch.float16),     # 256 at D = 32
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_causal_grid_parity(case):
    B, Sq, Sk, H, Hkv, D, dt = case
    print(f"case: causal grid {case}", flush=True)
    q, k, v, do = make_inputs(B, Sq, H, D, dt, Sk=Sk, Hkv=Hkv, seed=Sq + H, device="cuda")
    scale = D ** -0.5
    o, lse, _ = _lib.fwd(q, k, v, True, scale)
    grads = _lib.bwd(q, k, v, o, do, lse, True, scale)
    torch.cuda.synchronize()
    assert_parity(compare(q, k, v, do, True, scale, (o, lse) + tuple(grads)), dt, str(case))
    # the passes one by one (delta, then dK/dV and dQ)
    lib, stream = _lib.load(), _lib._stream(q)
    two = [torch.empty_like(t) for t in grads]
    a = _lib.bwd_args(q, k, v, o, do, lse, *two, True, scale, 0.0, 0, 0)
    n = lib.fa_bwd_workspace_size(ctypes.byref(a))
    ws = torch.empty(n, device="cuda", dtype=torch.uint8)
    for stage in (0, 1, 2):
        assert lib.fa_bwd_stage(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), n, stage, stream) == 0
    torch.cuda.synchronize()
    for x, y in zip(grads, two):
        assert torch.equal(x, y)
