"""The few-row forward (rows of a KV head's query heads in 32-row tiles, keys
split over waves and workgroups) at the edges of its tiles, splits and routing
rules: O, LSE and the row maxima against the float64 oracle with the tolerance
of the other parity tests, through strided caches, and equal on every call."""
import pytest
import torch

from flash_attention_v100 import _lib
from helpers import assert_parity, compare, make_inputs

pytestmark = pytest.mark.gpu

CASES = [
    # B, Sq, Sk, H, Hkv, D, dtype, causal
    (2, 1, 4096, 8, 2, 128, torch.bfloat16, False),   # one query, grouped heads, several splits
    (1, 1, 257, 4, 4, 64, torch.float16, False),      # a tile of one key at the end
    (3, 1, 1000, 8, 1, 32, torch.bfloat16, False),    # ragged keys, one KV head
    (1, 5, 2049, 12, 4, 64, torch.float16, False),    # rows cross heads inside a row tile (15 rows)
    (1, 33, 700, 4, 2, 128, torch.bfloat16, False),   # 66 rows: three row tiles, heads meet inside one
    (1, 11, 12000, 3, 1, 128, torch.float16, False),  # 33 rows: a last row tile of one row, many splits
    (2, 32, 65, 2, 2, 64, torch.bfloat16, False),     # two tiles, one key in the second
    (1, 65, 65, 2, 2, 64, torch.float16, True),       # causal: the diagonal in every tile
    (2, 300, 300, 4, 2, 128, torch.bfloat16, True),   # causal, grouped heads, 600 rows
    (1, 1500, 1500, 2, 1, 128, torch.float16, True),  # causal with splits, some of them empty for early rows
    (1, 700, 300, 4, 4, 64, torch.bfloat16, True),    # causal, fewer keys than queries
    (1, 100, 5000, 2, 2, 32, torch.bfloat16, True),   # causal, more keys than any query sees
    (1, 513, 513, 16, 16, 64, torch.float16, False),  # 272 units: two workgroups per CU
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(str(x) for x in c) for c in CASES])
def test_few_rows_parity(case):
    B, Sq, Sk, H, Hkv, D, dt, causal = case
    print(f"case: few rows {case}", flush=True)
    q, k, v, do = make_inputs(B, Sq, H, D, dt, Sk=Sk, Hkv=Hkv, seed=Sq + Sk + H, device="cuda")
    # a cache with room behind the keys: a strided view, garbage past Sk
    room = [torch.full((B, Sk + 70, Hkv, D), float("nan"), device="cuda", dtype=dt) for _ in range(2)]
    for r, t in zip(room, (k, v)):
        r[:, :Sk] = t
    kc, vc = (r[:, :Sk] for r in room)
    scale = D ** -0.5
    o, lse, mx = _lib.fwd(q, kc, vc, causal, scale, want_max=True)
    dq, dk, dv = _lib.bwd(q, k, v, o, do, lse, causal, scale)
    again = _lib.fwd(q, kc, vc, causal, scale, want_max=True)
    torch.cuda.synchronize()
    assert_parity(compare(q, k, v, do, causal, scale, (o, lse, dq, dk, dv)), dt, str(case))
    for a, b in zip((o, lse, mx), again):
        assert torch.equal(a, b)
    # row maxima of the scaled scores: sums of D products of 16-bit values in
    # float32, D * 2^-24 of sum |q k| scale, which D * 2^-24 * D * 16 * scale
    # bounds for these N(0, 1) draws (|q k| below 16 on average per product)
    kr = k.double().repeat_interleave(H // Hkv, dim=2)
    s = torch.einsum("bihd,bjhd->bhij", q.double().cpu(), kr.cpu()) * scale
    if causal:
        s = s.masked_fill(torch.ones(Sq, Sk, dtype=torch.bool).triu(1), float("-inf"))
    assert (mx.cpu().double() - s.amax(-1)).abs().max().item() <= D * 2.0 ** -24 * D * 16 * scale


def test_split_plan_needs_its_workspace():
    # the plan's workspace: none for short key loops, and refused when missing
    import ctypes
    lib = _lib.load()
    q = torch.zeros(1, 1, 8, 128, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(1, 16384, 8, 128, device="cuda", dtype=torch.bfloat16)
    o, lse = torch.empty_like(q), torch.empty(1, 8, 1, device="cuda")
    a = _lib.fwd_args(q, k, k, o, lse, None, False, 0.1, 0.0, 0, 0)
    n = lib.fa_fwd_workspace_size(ctypes.byref(a))
    assert n > 0
    assert lib.fa_fwd_ws(ctypes.byref(a), None, 0, _lib._stream(q)) == -8
    short = _lib.fwd_args(q, k[:, :300], k[:, :300], o, lse, None, False, 0.1, 0.0, 0, 0)
    assert lib.fa_fwd_workspace_size(ctypes.byref(short)) == 0
    assert lib.fa_fwd_ws(ctypes.byref(short), None, 0, _lib._stream(q)) == 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("D", [32, 64, 128])
def test_causal_rows_do_not_meet_later_keys(D):
    # grouped heads whose length is no multiple of the 32-row tiles: NaN in the
    # keys and values of the last rows reaches no row before their 64-key tile
    print(f"case: few rows, later keys {D}", flush=True)
    g = torch.Generator("cuda").manual_seed(D)
    q, k, v = (torch.randn(2, 200, h, D, generator=g, device="cuda").to(torch.bfloat16) for h in (8, 2, 2))
    want = _lib.fwd(q, k, v, True, D ** -0.5)
    k[:, 150:], v[:, 150:] = float("nan"), float("nan")
    got = _lib.fwd(q, k, v, True, D ** -0.5)
    torch.cuda.synchronize()
    assert torch.equal(got[0][:, :128], want[0][:, :128]) and torch.equal(got[1][:, :, :128], want[1][:, :, :128])
