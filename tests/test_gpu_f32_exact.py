"""float32 without a bias on bf16 pieces keeps what float32 products give:
exact zeros, NaN, infinities, values far below and above one, and the accuracy
of rows that see few keys.  On the key-split forward (small grids) and the
128-row kernels (B H ceil(Sq / 128) >= 256), forward and backward."""
import struct

import pytest
import torch

from flash_attention_v100 import _lib
from helpers import c_keep_mask

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # relative error of one float32 rounding
GRIDS = [(1, 2), (8, 32)]  # B, H: few workgroups, and 256 or more


def _inputs(B, H, S, D, Sk=None, Hkv=None, seed=0):
    g = torch.Generator("cpu").manual_seed(seed)
    return [torch.randn(B, s, h, D, generator=g).cuda() for s, h in
            ((S, H), (Sk or S, Hkv or H), (Sk or S, Hkv or H), (S, H))]


def _exact(q, k, v, do, causal, keep=None, p=0.0):
    """O, dQ, dK, dV and sum |P V| (the scale of O's rounding errors) in float64."""
    B, Sq, H, D = q.shape
    Hkv = k.shape[2]
    q, do = (t.double().transpose(1, 2).contiguous() for t in (q, do))
    k, v = (t.double().transpose(1, 2).repeat_interleave(H // Hkv, dim=1).contiguous() for t in (k, v))
    scale = D ** -0.5
    s = q @ k.transpose(2, 3).contiguous() * scale
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    pr = torch.softmax(s, -1)
    drop = torch.ones_like(pr) if keep is None else keep.to(pr) / (1 - p)
    pd = pr * drop
    o = pd @ v
    dp = (do @ v.transpose(2, 3).contiguous()) * drop
    ds = pr * (dp - (do * o).sum(-1, keepdim=True))
    dq = ds @ k * scale
    dk = (ds.transpose(2, 3).contiguous() @ q) * scale
    dv = pd.transpose(2, 3).contiguous() @ do

    def kv(t):
        return t.view(B, Hkv, H // Hkv, *t.shape[2:]).sum(2).transpose(1, 2)

    return o.transpose(1, 2), dq.transpose(1, 2), kv(dk), kv(dv), (pd @ v.abs()).transpose(1, 2)


def _run(q, k, v, do, causal, p=0.0, bits=None):
    scale = q.shape[-1] ** -0.5
    o, lse, _ = _lib.fwd(q, k, v, causal, scale, p, 9, 1, keep_bits=bits)
    return (o, lse) + tuple(_lib.bwd(q, k, v, o, do, lse, causal, scale, p, 9, 1, keep_bits=bits))


def _rel(got, want):
    return (got.double() - want).norm().item() / want.norm().item()


@pytest.mark.parametrize("B,H", GRIDS)
@pytest.mark.parametrize("D", [32, 64, 128])
def test_zeros_stay_zeros(B, H, D):
    print(f"case: f32 zeros {B} {H} {D}", flush=True)
    q, k, v, do = _inputs(B, H, 130, D)
    v[..., 3] = 0
    do[:, 7] = 0
    o, _, dq, dk, dv = _run(q, k, v, do, False)
    assert (o[..., 3] == 0).all() and (dq[:, 7] == 0).all()
    assert o[..., 4].abs().min().item() > 0
    z = torch.zeros_like
    o, _, dq, dk, dv = _run(q, k, z(v), do, True)
    assert not o.any() and not dq.any() and not dk.any()
    o, _, dq, dk, dv = _run(q, k, v, z(do), True)
    assert not dq.any() and not dk.any() and not dv.any()


@pytest.mark.parametrize("B,H", GRIDS)
@pytest.mark.parametrize("bits", [0x7FC00000, 0x7F800001, 0xFF800100])
def test_nan_stays_nan(B, H, bits):
    # (payloads in the lower half of the word among them)
    print(f"case: f32 NaN {B} {H} {bits:x}", flush=True)
    q, k, v, do = _inputs(B, H, 130, 64)
    nan = torch.tensor([struct.unpack("i", struct.pack("I", bits))[0]], dtype=torch.int32).cuda()
    v.view(torch.int32)[:, 5, 1, 6:7] = nan
    o, _, dq, dk, dv = _run(q, k, v, do, False)
    assert torch.isnan(o[:, :, 1, 6]).all()
    o[:, :, 1, 6] = 0
    assert torch.isfinite(o).all()
    assert torch.isnan(dq[:, :, 1]).all() and torch.isfinite(dq[:, :, 0]).all()


@pytest.mark.parametrize("B,H", GRIDS)
@pytest.mark.parametrize("causal,p,stored", [(False, 0.0, False), (True, 0.0, False), (True, 0.2, False), (False, 0.2, True)])
def test_infinities(B, H, causal, p, stored):
    # an infinite V gives its column, an infinite K takes its key out of the
    # rows whose score it makes -inf; every other result as without them
    print(f"case: f32 infinities {B} {H} {causal} {p} {stored}", flush=True)
    S, D = 161, 64
    q, k, v, do = _inputs(B, H, S, D, Hkv=H // 2)
    bits = _lib.alloc_keep_bits(B, H, S, S, q.device) if stored else None
    q[:, :, 0] = q[:, :, 0].abs() + 0.1
    q[:, :, 1] = q[:, :, 1].abs() + 0.1
    plain = _run(q, k, v, do, causal, p, bits)
    k2, v2 = k.clone(), v.clone()
    k2[:, 9, 0] = -float("inf")  # KV head 0: query heads 0 and 1
    if H > 2:
        v2[:, 0, 1, 5] = float("inf")  # key 0 of KV head 1: query heads 2 and 3
    got = _run(q, k2, v2, do, causal, p, bits)
    keep = torch.from_numpy(c_keep_mask(9, 1, B, H, S, S, p)).cuda() if p > 0 else None
    if H > 2:
        o = got[0][:, :, 2:4]
        seen = keep[:, 2:4, :, 0].bool().transpose(1, 2) if p > 0 else torch.ones_like(o[..., 5], dtype=torch.bool)
        # a dropped weight of zero times infinity is NaN, as in float32
        assert (o[..., 5][seen] == float("inf")).all() and torch.isnan(o[..., 5][~seen]).all()
        assert _rel(o[..., 6:], plain[0][:, :, 2:4, 6:].double()) < 3e-6
        for t, r in zip(got[:3], plain[:3]):  # heads that meet neither
            d = 2 if t.dim() == 4 else 1
            assert torch.equal(t.narrow(d, 4, H - 4), r.narrow(d, 4, H - 4))
    kz = k.clone()
    kz[:, 9, 0] = -1e30 / D  # scores of about -1e29: no weight either
    want = _exact(q, kz, v, do, causal, keep, p)
    assert _rel(got[0][:, :, :2], want[0][:, :, :2]) < 3e-6
    assert torch.isfinite(got[1][:, :2]).all()
    # dV of the other keys (key 9 meets the zeros behind the last query: 0 times infinity)
    others = [j for j in range(S) if j != 9]
    assert _rel(got[4][:, others, 0], want[3][:, others, 0]) < 3e-6


@pytest.mark.parametrize("B,H", GRIDS)
@pytest.mark.parametrize("mag", [1e-36, 1e-31, 1e-20, 1e8, 1e12])
def test_magnitudes(B, H, mag):
    # V and dO far from one, products of both in range: every result keeps
    # float32's relative accuracy (2-norm; the bound of the other f32 cases)
    print(f"case: f32 magnitude {B} {H} {mag}", flush=True)
    q, k, v, do = _inputs(B, H, 130, 64)
    s = 2.0 ** round(torch.tensor(mag).log2().item())  # powers of two: the same mantissas
    o, lse, *_ = _run(q, k, v * s, do, True)
    want = _exact(q, k, v * s, do, True)
    assert _rel(o, want[0]) < 2e-6
    o, lse, dq, dk, dv = _run(q, k, v, do * s, True)
    want = _exact(q, k, v, do * s, True)
    # (P below one scales some terms: those under 2^-126 are denormal in float32 too)
    for name, t, r in zip(("dq", "dk", "dv"), (dq, dk, dv), want[1:]):
        assert _rel(t / s, r / s) < 4e-6, name


@pytest.mark.parametrize("B,H", GRIDS)
@pytest.mark.parametrize("D", [32, 64, 128])
def test_few_visible_keys(B, H, D):
    # causal rows 0 .. 7 see one to eight keys: n products and sums of P V, the
    # exponentials (their argument's rounding included: |s - max| below 16 here)
    # and the normalisation, each some roundings of U of sum |P V|; over 256 heads
    # no more than the float32 instruction makes of them (the same call with a
    # bias of zero) and half of one rounding's root mean square (0.3 U)
    print(f"case: f32 few keys {B} {H} {D}", flush=True)
    q, k, v, do = _inputs(B, H, 136, D, seed=D)
    want = _exact(q, k, v, do, True)
    o, *_ = _run(q, k, v, do, True)
    ob, *_ = _lib.fwd(q, k, v, True, D ** -0.5, bias=torch.zeros(136, 136, device="cuda"))
    for n in range(1, 9):
        err = (o[:, n - 1].double() - want[0][:, n - 1]).abs()
        errb = (ob[:, n - 1].double() - want[0][:, n - 1]).abs()
        size = want[4][:, n - 1]
        assert (err / size).max().item() <= (40 if n > 1 else 4) * U, n
        if B * H >= 256:
            assert err.norm().item() <= errb.norm().item() + 0.15 * U * size.norm().item(), n


@pytest.mark.parametrize("B,H", GRIDS)
def test_products_of_one_term(B, H):
    # scores of a single product (the row maximum is the score itself), also
    # where every lower piece is as large as it can be: the products of lower
    # pieces cut at the last place of the first (2 U at most), those left out (U)
    print(f"case: f32 one term {B} {H}", flush=True)
    q, k, v, _ = _inputs(B, H, 130, 32)
    bits = torch.randint(0, 1 << 23, q.shape[:3], generator=torch.Generator("cpu").manual_seed(5), dtype=torch.int32)
    bits[0, :4, 0] = torch.tensor([0xFFFF, 0x7FFFFF, 0x8000, 0x7FFF])
    q[..., 1:], k[:] = 0, 0
    q[..., 0] = (bits | 0x3F800000).view(torch.float32).cuda()
    k[:, 77, :, 0] = (torch.tensor(0x3F80FFFF, dtype=torch.int32)).view(torch.float32).cuda()
    _, _, mx = _lib.fwd(q, k, v, False, 1.0, want_max=True)
    want = (q[..., 0].double() * k[:, 77, None, :, 0].double()).transpose(1, 2)
    assert ((mx.double() - want).abs() / want).max().item() <= 3 * U
