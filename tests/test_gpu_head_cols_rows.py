"""Head dims between the compiled ones through rows that follow each other
closer than the kernel's columns (heads-first storage passed transposed, a
single head, a single KV head): the row behind the last key or query starts
inside the span a full-width last row would have.  It is filled with NaN here
(the unfilled part of a cache); nothing of it may reach a result, so O, LSE,
dQ, dK and dV equal the zero-padded run's on contiguous copies bit for bit, on
every routing, at lengths that are no tile multiple."""
import pytest
import torch

from flash_attention_v100 import _lib

pytestmark = pytest.mark.gpu

CASES = [
    # D, B, Sq, Sk, H, Hkv, dtype, causal
    (40, 1, 300, 333, 2, 2, torch.float16, False),        # D = 64 kernels, few rows, combined backward
    (40, 8, 700, 500, 8, 8, torch.bfloat16, False),       # 128-row kernels
    (80, 1, 1, 3001, 8, 2, torch.bfloat16, False),        # D = 96, one query, split keys
    (72, 2, 130, 130, 3, 1, torch.float16, True),         # one KV head
    (80, 1, 200, 100, 1, 1, torch.bfloat16, True),        # one head
    (80, 4, 1025, 1025, 16, 16, torch.bfloat16, False),   # ping-pong kernels
    (72, 1, 3100, 3100, 48, 24, torch.float16, True),     # causal ping-pong, grouped heads
    (104, 1, 2, 2049, 4, 1, torch.float16, False),        # D = 128, few rows
    (104, 4, 513, 513, 32, 32, torch.bfloat16, False),    # ping-pong
    (120, 2, 257, 300, 4, 1, torch.float16, True),        # small grid
    (136, 1, 200, 201, 2, 2, torch.bfloat16, True),       # D = 256
    (200, 2, 333, 129, 4, 1, torch.float16, False),
]


def _rows(t):
    """t (B, S, h, D) as a view of heads-first storage with 5 rows of NaN behind each head's."""
    B, S, h, D = t.shape
    buf = torch.full((B, h, S + 5, D), float("nan"), device=t.device, dtype=t.dtype)
    buf[:, :, :S] = t.transpose(1, 2)
    return buf.transpose(1, 2)[:, :S]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_row_behind_the_last_is_not_read(case):
    D, B, Sq, Sk, H, Hkv, dt, causal = case
    print(f"case: head cols rows {case}", flush=True)
    g = torch.Generator("cuda").manual_seed(D + Sq)

    def randn(S, h):
        return torch.randn(B, S, h, D, generator=g, device="cuda").to(dt)

    q, do, k, v = randn(Sq, H), randn(Sq, H), randn(Sk, Hkv), randn(Sk, Hkv)
    scale, dp = D ** -0.5, _lib.padded_head_dim(D, dt)
    pad = [torch.nn.functional.pad(t, (0, dp - D)) for t in (q, k, v, do)]
    op, lsep, _ = _lib.fwd(*pad[:3], causal, scale)
    want = (op, lsep) + tuple(_lib.bwd(*pad[:3], op, pad[3], lsep, causal, scale))
    qr, kr, vr, dor = (_rows(t) for t in (q, k, v, do))
    assert qr.stride(1) == D and kr.stride(1) == D
    o, lse, _ = _lib.fwd(qr, kr, vr, causal, scale)
    got = (o, lse) + tuple(_lib.bwd(qr, kr, vr, _rows(o), dor, lse, causal, scale))
    torch.cuda.synchronize()
    for name, t, r in zip(("O", "LSE", "dQ", "dK", "dV"), got, want):
        assert torch.equal(t, r if name == "LSE" else r[..., :D]), name
