"""The key-split forward with a staged 16-bit bias (D <= 64, rows of whole 16-byte
chunks), at the lines of its rule and the edges of its tiles, against the float64
oracle with the tolerance of the other bias tests; masks of -inf keys and rows."""
import pytest
import torch

import test_gpu_bias as tb
from helpers import make_inputs

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, B, Sq, Sk, H, Hkv, D, causal, bias shape
    (torch.bfloat16, 1, 1, 72, 2, 2, 64, False, (1, 2, 1, 72)),          # one query, 8 keys past a tile
    (torch.float16, 2, 130, 136, 3, 1, 64, True, (2, 3, 130, 136)),      # three tiles for two splits
    (torch.bfloat16, 1, 200, 64, 2, 2, 32, False, (1, 1, 200, 64)),      # one tile: not split
    (torch.float16, 4, 300, 328, 20, 20, 64, False, (1, 20, 300, 328)),  # 240 workgroups
    (torch.bfloat16, 2, 500, 504, 32, 32, 32, False, (1, 32, 500, 504)),  # 256: the last without a mask
    (torch.bfloat16, 2, 1024, 1024, 20, 10, 64, True, (1, 20, 1024, 1024)),  # causal, 320, split
    (torch.float16, 2, 512, 520, 40, 40, 64, True, (2, 1, 512, 520)),    # causal, 320, short: not split
    (torch.bfloat16, 1, 257, 257, 4, 4, 64, True, (1, 4, 257, 257)),     # rows not whole chunks: not staged
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_bias_split(case):
    dt, B, Sq, Sk, H, Hkv, D, causal, shape = case
    print(f"case: staged bias split {case}", flush=True)
    q, k, v, do = make_inputs(B, Sq, H, D, dt, Sk=Sk, Hkv=Hkv, seed=Sq + Sk)
    bias = tb.make_bias(shape, dt, seed=Sq)
    bias[..., Sk // 3] = float("-inf")  # a masked key
    if Sk > 64 and (not causal or Sq > 64):
        bias[..., -1, :64] = float("-inf")  # a row with nothing in its first tile
    outs = tb.run_kernels(q, k, v, do, causal, D ** -0.5, bias)
    tb.check(q, k, v, do, causal, D ** -0.5, bias, [t.cpu() for t in outs], label=str(case))
