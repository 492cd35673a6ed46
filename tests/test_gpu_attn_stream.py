"""The streaming decode attention (grids of >= 1024 chunk blocks, FP8 row caches) against the
oracle, at the edges of its steps (32 positions), chunks (64 .. 512) and cache blocks, and the
block lengths it leaves to the general kernels.

Tolerance: max-abs-rel 2e-2, the bf16 bound of the other attention tests (probabilities rounded to
bf16, kept in fp32 for FP8, and a bf16 output).  The same logical cache through block lengths 16 / 32 /
64 (streaming) and 24 (general kernels) differs only by the two kernels' summation orders and their
bf16 roundings of the probabilities: held to 1e-2.
"""
import math

import pytest
import torch

from conftest import max_abs_rel
from oracle import ref
from test_gpu_kv_formats import _call, _rope_rows, bf

pytestmark = pytest.mark.gpu


def _run(mk, dev, fp8, blk, B, nq, nkv, d, NT, P, seed=3):
    """The operator and the oracle on one case: (out, oracle out), both [B, nq, d, NT]."""
    g = torch.Generator().manual_seed(seed + B + P)
    H, gqa = 128, nq // nkv
    S_max = P + NT + 5 if not blk else (P + NT + blk - 1) // blk * blk
    S_ctx = S_max if blk else P + NT           # a block cache's mask covers its whole table
    prior = S_ctx - NT
    X = bf(torch.randn(B, NT, H, generator=g))
    W = bf(0.05 * torch.randn(H, d * (nq + 2 * nkv), generator=g))
    K = torch.randn(B, nkv, S_max, d, generator=g)
    V = torch.randn(B, nkv, S_max, d, generator=g)
    ks = vs = None
    if fp8:
        K, V = ref.kv_fp8_quant(K, 8.0), ref.kv_fp8_quant(V, 8.0)
        ks = vs = torch.full((1, 1), 8.0)
    else:
        K, V = bf(K), bf(V)
    # ragged lengths, single masked positions and a whole masked 64-position stretch
    lens = torch.randint(max(P // 2, 0), P + 1, (B,), generator=g)
    lens[0] = P
    keep = (torch.arange(prior)[:, None] < lens[None, :])[:, :, None, None].expand(prior, B, nq, NT).clone()
    keep &= torch.rand(prior, B, nq, NT, generator=g) < 0.9
    keep[P // 2: P // 2 + 64] = False
    mask = torch.cat([keep, torch.ones(NT, B, nq, NT, dtype=torch.bool)]).to(torch.uint8)
    cos, sin = _rope_rows(B, NT, P, d)
    upd = torch.full((B, 1), 0xFFFFFFFF, dtype=torch.int64)
    scale = d ** -0.5 / (8.0 if fp8 else 1.0)
    table = None
    Kd, Vd = K, V
    if blk:
        nb = S_max // blk
        table = torch.randperm(B * nb, generator=g).to(torch.int32).reshape(B, nb)
        pool = [torch.empty(B * nb, blk, nkv, d, dtype=K.dtype) for _ in range(2)]
        for t, p in ((K, pool[0]), (V, pool[1])):
            p.view(torch.uint8)[table.reshape(-1).long()] = \
                t.transpose(1, 2).reshape(B * nb, blk, nkv, d).contiguous().view(torch.uint8)
        Kd, Vd = pool
    Kg, Vg = Kd.contiguous().to(dev), Vd.contiguous().to(dev)
    out, _, _ = _call(mk, dev, X, W, None, None, None, cos, sin, Kg, Vg, mask, None, upd, table, False,
                      ks, vs, scale)
    torch.cuda.synchronize()
    attn = torch.zeros(B * NT, nq * d)
    for h in range(nkv):
        cols = torch.cat([torch.arange(h * gqa * d, (h + 1) * gqa * d), nq * d + h * d + torch.arange(d),
                          (nq + nkv) * d + h * d + torch.arange(d)])
        o, _, _ = ref.attention_block_tkg(
            X.float(), W.float()[:, cols], None, 1e-6, None, None, None, 1e-6, cos, sin, K[:, h].clone(),
            V[:, h].clone(), mask[:, :, h * gqa:(h + 1) * gqa].float(), None, False, upd, None, None,
            softmax_scale=scale, k_scale=8.0 if fp8 else None, v_scale=8.0 if fp8 else None)
        attn[:, h * gqa * d:(h + 1) * gqa * d] = o
    return out, attn.reshape(B, NT, nq, d).permute(0, 2, 3, 1)


@pytest.mark.parametrize("blk,B,nq,nkv,d,NT,P", [
    (0, 1, 8, 1, 128, 1, 0), (0, 1, 8, 1, 128, 1, 1), (0, 2, 4, 2, 64, 1, 31), (0, 1, 16, 1, 128, 1, 32),
    (16, 2, 2, 2, 64, 1, 63), (64, 1, 8, 1, 128, 3, 64), (0, 3, 8, 2, 64, 8, 129), (32, 4, 8, 4, 128, 1, 500),
    (24, 2, 8, 2, 128, 1, 100), (64, 64, 16, 8, 64, 1, 640), (0, 64, 16, 16, 64, 2, 300)])
def test_fp8_stream_matches_oracle(mk, dev, blk, B, nq, nkv, d, NT, P):
    print(f"fp8 stream blk={blk} B={B} nq={nq} nkv={nkv} d={d} NT={NT} P={P}", flush=True)
    out, want = _run(mk, dev, True, blk, B, nq, nkv, d, NT, P)
    assert max_abs_rel(out, want) < 2e-2


@pytest.mark.parametrize("d,a,b", [(128, 11, 15), (64, 12, 13), (64, 8, 9)])
def test_fp8_probabilities_keep_fp32(mk, dev, d, a, b):
    """Two positions of probability 1 and r = a / b (unnormalised; scores ln(b / a) and 0) with values
    -16 a and 16 b, and a new token of zeros: the head's output is 16 b (r - a / b) / (1 + 2 r), which
    shows r's own error.  In fp32 that is expf's 2^-23 r and 2^-24 ln(b / a) r of the scale, and the sum
    of terms up to 16 a rounds three times by at most 2^-24 of it.  (r as two bf16 terms: 2^-18, 6 to 12
    times the bound.)"""
    nq, S = 4, 16
    X, W = torch.zeros(1, 1, 128), torch.zeros(128, d * (nq + 2))
    X[..., 0] = 1.0
    W[0, 0:nq * d:d] = 1.0                       # q = e0 for every head; k = v = 0
    K, V = torch.zeros(1, S, d), torch.zeros(1, S, d)
    K[0, 1, 0] = 1.0
    V[0, 0], V[0, 1] = 16.0 * b, -16.0 * a
    K, V = K.to(torch.float8_e4m3fn), V.to(torch.float8_e4m3fn)
    ones, one = torch.ones(d // 2, 1, 1), torch.ones(1, 1)
    out, _, _ = _call(mk, dev, bf(X), bf(W), None, None, None, ones, 0 * ones, K.to(dev), V.to(dev),
                      torch.ones(3, 1, nq, 1, dtype=torch.uint8), None, torch.tensor([[-1]], dtype=torch.int32),
                      None, False, one, one, math.log(b / a))
    r = a / b
    bound = (16 * b * r * (2.0 ** -23 + 2.0 ** -24 * math.log(b / a)) + 3 * 2.0 ** -24 * 16 * a) / (1 + 2 * r)
    assert out.float().abs().max().item() <= bound, (out.float().abs().max().item(), bound)


# >= 1024 blocks of 256 positions: the streaming kernel; from 2048 blocks of 512: its larger chunk
@pytest.mark.parametrize("blk,B,nq,nkv,d,NT,P", [
    (0, 64, 16, 16, 64, 1, 255), (16, 64, 32, 16, 64, 1, 300), (64, 64, 16, 8, 128, 1, 511),
    (0, 64, 8, 8, 128, 2, 257), (32, 128, 16, 16, 64, 1, 513)])
def test_bf16_stream_matches_oracle(mk, dev, blk, B, nq, nkv, d, NT, P):
    print(f"bf16 stream blk={blk} B={B} nq={nq} nkv={nkv} d={d} NT={NT} P={P}", flush=True)
    out, want = _run(mk, dev, False, blk, B, nq, nkv, d, NT, P)
    assert max_abs_rel(out, want) < 2e-2


@pytest.mark.parametrize("fp8", [False, True])
def test_stream_equals_general_path(mk, dev, fp8):
    """The same logical cache (192 positions per table) in blocks of 16 / 32 / 64 rows and, through the
    general kernels, of 24."""
    outs = [_run(mk, dev, fp8, blk, 128, 16, 8, 64, 1, 191)[0] for blk in (16, 32, 64, 24)]
    for o in outs[:3]:
        assert max_abs_rel(o, outs[3].float()) < 1e-2


@pytest.mark.parametrize("blk", [0, 16])
@pytest.mark.parametrize("form", ["int64", "strided", "bf16 rope", "mask bool", "mask bf16"])
def test_operand_forms_agree(mk, dev, blk, form):
    """Write positions, block tables, masks and RoPE tables in the other dtypes and strides the operator
    takes give bit for bit the result of their plain forms, out-of-range entries included."""
    g = torch.Generator().manual_seed(9)
    B, H, nq, nkv, d, S = 3, 256, 8, 2, 64, 48
    X, W = bf(torch.randn(B, 1, H, generator=g)), bf(0.05 * torch.randn(H, d * (nq + 2 * nkv), generator=g))
    shape = (B * 3, 16, nkv, d) if blk else (B, nkv, S, d)
    K, V = bf(torch.randn(shape, generator=g)), bf(torch.randn(shape, generator=g))
    cos, sin = [bf(t).float() for t in _rope_rows(B, 1, S - 1, d)]
    mask = (torch.rand(S, B, nq, 1, generator=g) < 0.8).to(torch.uint8)
    upd = torch.tensor([5, -1, 40], dtype=torch.int32)[:, None]
    table = torch.arange(B * 3, dtype=torch.int32).reshape(B, 3) if blk else None
    if blk:
        table[1, 2], table[2, 0] = -7, B * 3 + 100           # no such blocks: rows read as zero

    def call(cos, sin, mask, upd, table):
        Kg, Vg = K.to(dev), V.to(dev)
        from nki_moe_megakernel_amd.common_types import QuantizationType as QT
        out, _, _ = mk.attention_block_tkg(
            X.to(dev), None, False, 1e-6, None, W.to(dev), None, QT.NONE, None, None, False, 1e-6, None, None,
            cos, sin, True, False, 1e-6, None, None, False, table, Kg, Vg, mask, None, True, upd, None, None,
            QT.NONE, None, None, False, False)
        return out, Kg, Vg
    tb = table.to(dev) if blk else None
    base = call(cos.to(dev), sin.to(dev), mask.to(dev), upd.to(dev), tb)
    c, s, m, u = cos.to(dev), sin.to(dev), mask.to(dev), upd.to(dev)
    if form == "int64":
        u = torch.tensor([5, 0xFFFFFFFF, 40], device=dev)[:, None]
        tb = tb.long() if blk else None
        if blk:
            tb[2, 0] = (1 << 33) + 1                          # its low 32 bits name a block
    elif form == "strided":
        c = torch.cat([c, c], 2)[:, :, :1]
        s = s.permute(1, 2, 0).contiguous().permute(2, 0, 1)
        u = torch.cat([u, u], 1).long()[:, 1:]
        tb = torch.cat([tb, tb], 1).long()[:, 3:] if blk else None
        m = torch.cat([m, m], 3)[..., :1]
    elif form == "bf16 rope":
        c, s = c.bfloat16(), s.bfloat16()
    else:
        m = m.to(torch.bool if form == "mask bool" else torch.bfloat16)
    got = call(c, s, m, u, tb)
    for a, b in zip(got, base):
        assert torch.equal(a, b)


def test_router_writes_callers_tensors(mk, dev):
    """Outputs of the kernels' own layout are written in place; strided or otherwise typed ones get the
    same values."""
    g = torch.Generator().manual_seed(4)
    T, H, E, k = 33, 256, 128, 8
    x, w = torch.randn(T, H, generator=g).to(dev), bf(torch.randn(H, E, generator=g)).float().to(dev)

    def call(lg, af, ix):
        r = mk.router_topk(x, w, None, lg, af, ix, mk.RouterActFnType.SOFTMAX, k, 1, 0, True, True)
        assert r[0] is lg and r[1] is ix and r[2] is af
        return lg, af, ix
    a = call(torch.empty(T, E, device=dev), torch.empty(T, E, device=dev),
             torch.empty(T, k, dtype=torch.int32, device=dev))
    b = call(torch.empty(E, T, device=dev).t(), torch.empty(T * E + 1, device=dev)[1:].reshape(T, E),
             torch.empty(T, k, dtype=torch.int64, device=dev))
    for p, q in zip(a, b):
        assert torch.equal(p, q.to(p.dtype))


def test_router_outputs_behave_like_copies(mk, dev):
    """Writing in place keeps what copy_ did: version counters move, a leaf that requires grad is refused,
    an output that shares memory with another output or the input gets the later one's values."""
    g = torch.Generator().manual_seed(5)
    T, H, E, k = 16, 128, 128, 4
    x, w = torch.randn(T, H, generator=g).to(dev), bf(torch.randn(H, E, generator=g)).float().to(dev)

    def call(x, lg, af, ix):
        mk.router_topk(x, w, None, lg, af, ix, mk.RouterActFnType.SOFTMAX, k, 1, 0, True, True)
        return lg, af, ix

    def outs():
        return (torch.empty(T, E, device=dev), torch.empty(T, E, device=dev),
                torch.empty(T, k, dtype=torch.int32, device=dev))
    want = call(x, *outs())
    fresh = outs()
    before = [t._version for t in fresh]
    call(x, *fresh)
    assert all(t._version > v for t, v in zip(fresh, before))
    for i in range(2):
        o = list(outs())
        o[i].requires_grad_(True)
        with pytest.raises(RuntimeError, match="leaf Variable that requires grad"):
            call(x, *o)
    lg, _, ix = outs()
    call(x, lg, lg, ix)                                          # affinities are stored last
    assert torch.equal(lg, want[1]) and torch.equal(ix, want[2])
    xi = x.clone()                                               # logits over the input
    _, af, ix = outs()
    call(xi, xi, af, ix)
    assert torch.equal(xi, want[0]) and torch.equal(af, want[1]) and torch.equal(ix, want[2])
    both = torch.empty(2 * T * E, device=dev)                    # parts of one buffer, apart and overlapping
    got = call(x, both[:T * E].view(T, E), both[T * E:].view(T, E), ix)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    call(x, both[E:E + T * E].view(T, E), both[:T * E].view(T, E), ix)
    assert torch.equal(both[:T * E].view(T, E), want[1]) and torch.equal(both[T * E:T * E + E], want[0][-1])


def test_router_chunks_land_in_their_rows(mk, dev):
    """Above 4096 tokens the operator makes a call per 4096: the last call's rows (odd counts, into rows
    of outputs with a guard after them) equal those of the same tokens alone, a call of the same form."""
    g = torch.Generator().manual_seed(6)
    T, H, E, k = 4096 + 133, 128, 24, 3
    x, w = bf(torch.randn(T, H, generator=g)).to(dev), bf(torch.randn(H, E, generator=g)).to(dev)

    def call(x):
        n = x.shape[0]
        lg, af = torch.full((n + 1, E), 7.0, device=dev), torch.full((n + 1, E), 7.0, device=dev)
        ix = torch.full((n + 1, k), 7, dtype=torch.int32, device=dev)
        mk.router_topk(x, w, None, lg[:n], af[:n], ix[:n], mk.RouterActFnType.SOFTMAX, k, 1, 0, True, True)
        assert all(bool((t[n] == 7).all()) for t in (lg, af, ix))
        return lg[:n], af[:n], ix[:n]
    whole, first, last = call(x), call(x[:4096]), call(x[4096:])
    for t, a, b in zip(whole, first, last):
        assert torch.equal(t[:4096], a) and torch.equal(t[4096:], b)
