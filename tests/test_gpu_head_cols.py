"""Head dims between the compiled ones without padded copies (``fa_fwd_cols`` /
``fa_bwd_cols``): the kernels read and write only the columns that exist.  On
zero-padded tensors the same products gain exact zeros, in the same order, so
O, LSE, dQ, dK and dV equal the padded run's bit for bit -- at the edges of the
column classes (96, 128, 256), on every routing (few rows, small grids,
128-query and ping-pong kernels), with q, k, v interleaved in one buffer (a read
past the columns meets a neighbour) and outputs in wider rows whose other
columns must stay untouched."""
import ctypes

import pytest
import torch

from flash_attention_v100 import _lib

pytestmark = pytest.mark.gpu

CASES = [
    # D, B, Sq, Sk, H, Hkv, dtype, causal
    (40, 2, 300, 300, 4, 4, torch.float16, True),        # D = 64 kernels, small grid
    (56, 4, 700, 500, 16, 8, torch.bfloat16, False),     # D = 64, 128-query kernels
    (72, 1, 130, 130, 3, 3, torch.bfloat16, True),       # D = 96, few rows
    (80, 4, 1025, 1025, 16, 16, torch.bfloat16, False),  # D = 96, ping-pong kernels
    (88, 1, 3100, 3100, 48, 24, torch.float16, True),    # D = 96, causal ping-pong, grouped heads
    (96, 2, 1000, 1000, 8, 2, torch.float16, True),      # D = 96, every column exists
    (96, 1, 1, 3000, 8, 2, torch.bfloat16, False),       # one query: split keys
    (104, 4, 513, 513, 32, 32, torch.bfloat16, False),   # D = 128, ping-pong
    (120, 2, 257, 300, 4, 1, torch.float16, True),       # D = 128, small grid
    (136, 1, 200, 200, 2, 2, torch.bfloat16, True),      # D = 256
    (248, 2, 333, 129, 4, 2, torch.float16, False),      # D = 256
]


def _padded(t, dp):
    return torch.nn.functional.pad(t, (0, dp - t.shape[-1])).contiguous()


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_columns_equal_the_padded_run(case):
    D, B, Sq, Sk, H, Hkv, dt, causal = case
    print(f"case: head cols {case}", flush=True)
    g = torch.Generator("cuda").manual_seed(D + Sq)

    def inter(S, h):  # rows of a buffer that holds other tensors' columns beside these
        return torch.randn(B, S, h, 3 * D, generator=g, device="cuda").to(dt)[..., D:2 * D]

    q, do, k, v = inter(Sq, H), inter(Sq, H), inter(Sk, Hkv), inter(Sk, Hkv)
    dp = _lib.padded_head_dim(D, dt)
    scale = D ** -0.5
    lib, stream = _lib.load(), _lib._stream(q)

    # the padded run, through the plain entry points
    qp, kp, vp, dop = (_padded(t, dp) for t in (q, k, v, do))
    op, lsep, _ = _lib.fwd(qp, kp, vp, causal, scale)
    gp = _lib.bwd(qp, kp, vp, op, dop, lsep, causal, scale)

    # the columns, into rows of D + 8
    def out(S, h):
        return torch.full((B, S, h, D + 8), 77.0, device="cuda", dtype=dt)

    bufs = [out(Sq, H), out(Sq, H), out(Sk, Hkv), out(Sk, Hkv)]
    o, dq, dk, dv = (t[..., :D] for t in bufs)
    lse = torch.empty(B, H, Sq, device="cuda")
    a = _lib.fwd_args(q, k, v, o, lse, None, causal, scale, 0.0, 0, 0, head_dim=dp)
    n = lib.fa_fwd_workspace_size(ctypes.byref(a))
    ws = torch.empty(max(n, 16), device="cuda", dtype=torch.uint8)
    assert lib.fa_fwd_cols(ctypes.byref(a), D, ws.data_ptr(), n, stream) == 0
    ba = _lib.bwd_args(q, k, v, o, do, lse, dq, dk, dv, causal, scale, 0.0, 0, 0, head_dim=dp)
    n = lib.fa_bwd_workspace_size(ctypes.byref(ba))
    ws = torch.empty(n, device="cuda", dtype=torch.uint8)
    assert lib.fa_bwd_cols(ctypes.byref(ba), D, ws.data_ptr(), n, stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(lse, lsep)
    for name, t, r, buf in zip(("O", "dQ", "dK", "dV"), (o, dq, dk, dv), (op,) + gp, bufs):
        assert torch.equal(t, r[..., :D]), name
        assert (buf[..., D:] == 77.0).all(), name

    # and through the Python entry points
    o2, lse2, _ = _lib.fwd(q, k, v, causal, scale)
    g2 = _lib.bwd(q, k, v, o2, do, lse2, causal, scale)
    torch.cuda.synchronize()
    for t, r in zip((o2, lse2) + g2, (o, lse, dq, dk, dv)):
        assert torch.equal(t, r)


def test_columns_refused():
    lib = _lib.load()
    q = torch.zeros(1, 64, 2, 128, device="cuda", dtype=torch.bfloat16)
    lse = torch.empty(1, 2, 64, device="cuda")
    a = _lib.fwd_args(q, q, q, torch.empty_like(q), lse, None, False, 0.1, 0.0, 0, 0)
    for cols in (0, -8, 64, 100, 136):  # none, negative, the class below, no whole chunk, too many
        assert lib.fa_fwd_cols(ctypes.byref(a), cols, None, 0, _lib._stream(q)) == -3
    d = _lib.fwd_args(q, q, q, torch.empty_like(q), lse, None, False, 0.1, 0.1, 0, 0)
    assert lib.fa_fwd_cols(ctypes.byref(d), 104, None, 0, _lib._stream(q)) == -3
