"""The stored dropout mask at the edges of its kernel: rows that end inside a
64-key set, steps of one to four sets, odd row counts, and counters whose low
32-bit word wraps inside a step (offsets just below multiples of 2^32), against
the C oracle's mask, bit for bit on every pair the attention sees."""
import numpy as np
import pytest
import torch

from flash_attention_v100 import _lib
from helpers import c_keep_mask

pytestmark = pytest.mark.gpu

WRAP = 2 ** 32
CASES = [
    # B, H, Sq, Sk, causal, seed, offset
    (1, 1, 1, 1, False, 7, 0),
    (1, 3, 5, 63, False, 8, 1),
    (2, 1, 3, 64, True, 2 ** 63 + 9, 12345),
    (1, 1, 7, 65, False, 10, WRAP - 100),        # the wrap inside the second row
    (1, 1, 9, 129, False, 11, WRAP - 129 * 4 - 64),  # at a set's first key
    (1, 2, 130, 193, True, 12, 3 * WRAP - 5000),
    (1, 1, 300, 257, True, 13, WRAP - 1),        # at the first key of all
    (2, 2, 259, 259, True, 14, 2 ** 64 - 2000),  # the 64-bit counter wraps too
    (1, 1, 4, 1000, False, 15, WRAP - 1000 - 767),
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_keep_bits_edges(case):
    B, H, Sq, Sk, causal, seed, offset = case
    print(f"case: keep bits {case}", flush=True)
    g = torch.Generator("cpu").manual_seed(1)
    q = torch.randn(B, Sq, H, 32, generator=g).half().cuda()
    k = torch.randn(B, Sk, H, 32, generator=g).half().cuda()
    p = 0.3
    bits = _lib.alloc_keep_bits(B, H, Sq, Sk, q.device)
    _lib.fwd(q, k, k, causal, 0.2, p, seed, offset, keep_bits=bits)
    torch.cuda.synchronize()
    words = bits.cpu().numpy().view(np.uint32).reshape(B, H, Sq, -1)
    got = ((words[..., None] >> np.arange(32, dtype=np.uint32)) & 1).reshape(B, H, Sq, -1)[..., :Sk]
    want = c_keep_mask(seed, offset, B, H, Sq, Sk, p)
    seen = np.tril(np.ones((Sq, Sk), dtype=bool)) if causal else np.ones((Sq, Sk), dtype=bool)
    assert np.array_equal(got[..., seen], want[..., seen])
    # the mask drawn inside the kernels (no stored bits) is the same one
    assert torch.equal(_lib.dropout_mask(seed, offset, B, H, Sq, Sk, p).cpu(), torch.from_numpy(want))
