"""lbw_attention_chain through the C ABI: explicit piece counts, fp32 output, per-batch key counts,
the running triple, and every refusal."""
import ctypes

import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(B, Lq, H, lens, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    return r(B, Lq, H, 128), [r(B, n, H, 128) for n in lens], [r(B, n, H, 128) for n in lens]


def _triple(B, H, Lq):
    return (torch.empty(B, H, Lq, 128, device=DEV), torch.empty(B, H, Lq, device=DEV),
            torch.empty(B, H, Lq, device=DEV))


def _chain(lib, p, state, ws_bytes=None):
    from lbw_amd import _lib
    n = lib.lbw_attention_chain_workspace_size(ctypes.byref(p), int(state is not None))
    assert n > 0, lib.lbw_last_error()
    n = n if ws_bytes is None else ws_bytes
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device=DEV)
    sp = [None] * 3 if state is None else [t.data_ptr() for t in state]
    rc = lib.lbw_attention_chain(ctypes.byref(p), *sp, ws.data_ptr(), n, _lib.stream_ptr())
    torch.cuda.synchronize()
    return rc


@pytest.mark.parametrize("splits", [0, 1, 2, 15, 40])
@pytest.mark.parametrize("B,Lq,H,lens,k_lens", [
    (1, 300, 3, [1000, 700], None),        # six units: up to 90 items, one per CU
    (2, 40, 70, [330, 520], [200, 300]),   # 140 units: from two pieces on more items than CUs
])
def test_pieces_triple_and_fp32_output(lib, B, Lq, H, lens, k_lens, splits):
    """A first call without a state (written straight into the triple, or merged from its pieces), one
    that joins it, and the last into fp32: the triple equals the oracle's partials (m the true row
    max) and the output its attention over all keys, within the bf16 rounding of P. k_lens counts
    the keys of each call's own segment."""
    from lbw_amd import _lib
    q, ks, vs = _inputs(B, Lq, H, lens, seed=Lq + splits)
    qd = q.to(DEV)
    kl = None if k_lens is None else torch.tensor(k_lens, dtype=torch.int32)
    kld = None if kl is None else kl.to(DEV)
    print(f"case B={B} Lq={Lq} H={H} splits={splits}", flush=True)
    dev = [(k.to(DEV), v.to(DEV)) for k, v in zip(ks, vs)]
    state = _triple(B, H, Lq)
    p = _lib.attn_params(qd, None, [dev[0]], k_lens=kld, num_splits=splits, parts=state)
    _lib.check(_chain(lib, p, None), "first")
    _, (ro, rm, rl) = O.attention_ref(q, ks[0], vs[0], k_lens=kl, return_partials=True)
    joined = _triple(B, H, Lq)
    p = _lib.attn_params(qd, None, [dev[1]], k_lens=kld, num_splits=splits, parts=joined)
    _lib.check(_chain(lib, p, state), "joined")
    out = torch.empty(B, Lq, H, 128, device=DEV)
    p = _lib.attn_params(qd, out, [dev[1]], k_lens=kld, num_splits=splits)
    _lib.check(_chain(lib, p, state), "last")

    def cut(x, n):
        return x[:, :n]
    if kl is None:
        kk, vv = torch.cat(ks, 1), torch.cat(vs, 1)
        ref, (jo, jm, jl) = O.attention_ref(q, kk, vv, return_partials=True)
    else:   # per batch, the valid keys of both segments
        parts = [O.attention_ref(q[b:b + 1], torch.cat([cut(k[b:b + 1], n) for k in ks], 1),
                                 torch.cat([cut(v[b:b + 1], n) for v in vs], 1),
                                 return_partials=True) for b, n in enumerate(k_lens)]
        ref = torch.cat([r for r, _ in parts])
        jo, jm, jl = (torch.cat([t[i] for _, t in parts]) for i in range(3))
    for (po, pm, pl), (xo, xm, xl) in ((state, (ro, rm, rl)), (joined, (jo, jm, jl))):
        assert torch.allclose(pm.cpu(), xm, rtol=1e-5, atol=1e-4)
        assert torch.allclose(pl.cpu(), xl, rtol=5e-3, atol=1e-3)
        assert torch.allclose((po / pl[..., None]).cpu(), xo / xl[..., None], atol=1e-2)
    assert float((out.cpu() - ref).abs().max()) <= 1e-2
    assert torch.allclose(out.permute(0, 2, 1, 3), joined[0] / joined[2][..., None], atol=1e-5)


def test_refusals(lib):
    """Every refusal comes before a launch, with its code and a message; the outputs keep what they
    held."""
    from lbw_amd import _lib
    B, Lq, H = 1, 40, 2
    q, ks, vs = _inputs(B, Lq, H, [300], seed=3)
    qd, seg = q.to(DEV), (ks[0].to(DEV), vs[0].to(DEV))
    state = tuple(t.fill_(1.0) for t in _triple(B, H, Lq))
    new = tuple(t.fill_(7.0) for t in _triple(B, H, Lq))
    out = torch.full((B, Lq, H, 128), 7.0, dtype=torch.bfloat16, device=DEV)

    def params(parts=None, out=None, **kw):
        return _lib.attn_params(qd, out, [seg], num_splits=2, parts=parts, **kw)

    def call(p, s, ws=True):
        n = lib.lbw_attention_chain_workspace_size(ctypes.byref(params(new)), 1)
        w = torch.empty(n, dtype=torch.uint8, device=DEV)
        rc = lib.lbw_attention_chain(ctypes.byref(p), *s, w.data_ptr() if ws else None, n,
                                     _lib.stream_ptr())
        return rc, lib.lbw_last_error()

    so, sm, sl = (t.data_ptr() for t in state)
    assert call(params(new), (so, None, sl))[0] == 1            # a state in parts
    assert call(params(new), (so + 4, sm, sl))[0] == 1          # misaligned
    for parts in (state, (new[0], state[1], new[2]), (new[0], new[1], state[2]),
                  (state[0], new[1], new[2]), (new[0], state[0][0, 0, 5], new[2])):
        rc, msg = call(params(parts), (so, sm, sl))             # the triple over the state
        assert rc == 1 and b"overlaps" in msg
    rc, msg = call(params(new), (so, sm, sl), ws=False)
    assert rc == 4 and b"workspace" in msg
    assert _chain(lib, params(None, out), state, ws_bytes=64) == 4
    bias = torch.zeros(300, device=DEV)
    p = params(None, out)
    p.key_bias = bias.data_ptr()
    rc, msg = call(p, (so, sm, sl))
    assert rc == 2 and b"key_bias" in msg
    p = params(new)
    p.part_m = None
    assert call(p, (so, sm, sl))[0] == 1                        # a new triple in parts
    torch.cuda.synchronize()
    for t in (*new, out):
        assert bool((t == 7.0).all())
    for t in state:
        assert bool((t == 1.0).all())
