"""Backward of the attention-family and row-encoder operators (GPU).

Each operator's gradients, taken through ``torch.autograd`` on the
``mantisnet::*`` operator, are compared with autograd through the CPU fp32
oracle's formulation of the same forward (oracle/model_ref.py: the segment
softmax, the window-latent read and broadcast, masked SDPA, the row
encoder; each pinned by literal loops in tests/test_oracle_model.py), on a
real encoded batch.  Tolerances: 1e-4 for fp32 operands (fp32 sums in
another order; the reference's own gradient tests use 1e-4,
tests/test_relay.py:116-134), 2e-2 for 16-bit operands (one rounding of each
gradient to the operand dtype).  Two backward passes agree bitwise.
"""

from __future__ import annotations

import pytest
import torch

import mantisnet  # noqa: F401  registers the operators
from mantisnet import collate_positions, synthetic
from oracle import model_ref as R

pytestmark = pytest.mark.gpu
OPS = torch.ops.mantisnet


@pytest.fixture(scope="module")
def batch():
    return collate_positions(synthetic.random_games(1, 6, start=40))


def _grads(fn, inputs, seed_grad):
    leaves = [t.detach().clone().requires_grad_(True) for t in inputs]
    out = fn(*leaves)
    out.backward(seed_grad)
    return [t.grad for t in leaves]


def _close(got, exp, dt):
    tol = dict(rtol=1e-4, atol=1e-4) if dt == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    for g, e in zip(got, exp):
        torch.testing.assert_close(g.float().cpu(), e.float(), **tol)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("with_vcls", [True, False])
def test_cell_attention_backward(device, batch, dt, with_vcls):
    b = batch
    n_w, n_c = b.window_feat.numel(), b.cell_pos.shape[0]
    t = R.cell_tables_full(b.dec_cell, b.dec_window, b.dec_class, n_w, 726, n_c)
    gen = torch.Generator().manual_seed(21)
    q = torch.randn(n_c, 4, 32, generator=gen).to(dt)
    k, v = (torch.randn(n_w, 4, 32, generator=gen).to(dt) for _ in range(2))
    bias = 0.3 * torch.randn(4, 726, generator=gen)
    vcls = 0.1 * torch.randn(726, 128, generator=gen)
    seed = torch.randn(n_c, 4, 32, generator=gen)
    views = [t["cell_ptr"], t["edge_window"], t["edge_class"], t["edge_cell"], t["win_ptr"], t["edge_wcell"],
             t["edge_wclass"], t["cls_ptr"], t["cedge_cell"]]
    dviews = [x.to(device) for x in views]

    if with_vcls:
        def op(q_, k_, v_, b_, c_):
            return OPS.cell_attention(q_, k_, v_, b_, c_, *dviews)[0]

        def ref(q_, k_, v_, b_, c_):
            return R.cell_attention(q_, k_, v_, b_, c_, t["edge_window"], t["edge_class"], t["edge_cell"])

        inputs = [q, k, v, bias, vcls]
    else:
        def op(q_, k_, v_, b_):
            return OPS.cell_attention_plain(q_, k_, v_, b_, *dviews)[0]

        def ref(q_, k_, v_, b_):
            return R.cell_attention(q_, k_, v_, b_, None, t["edge_window"], t["edge_class"], t["edge_cell"])

        inputs = [q, k, v, bias]
    got = _grads(op, [x.to(device) for x in inputs], seed.to(device))
    mantisnet.ops.raise_on_device_error(device)
    exp = _grads(ref, [x.float() for x in inputs], seed)
    assert got[0].dtype == dt and got[3].dtype == torch.float32
    _close(got, exp, dt)
    again = _grads(op, [x.to(device) for x in inputs], seed.to(device))
    assert all(torch.equal(a, c) for a, c in zip(got, again))


def test_window_latent_backward(device, batch):
    b = batch
    p = b.attn_valid.shape[0]
    window_pos = b.window_slot // b.value_valid.shape[1]
    n_w = window_pos.numel()
    offsets, order = R.window_layout(window_pos, p)
    layout = [x.to(device) for x in (window_pos, offsets, order)]
    gen = torch.Generator().manual_seed(22)
    q = torch.randn(p, 4, 4, 32, generator=gen)
    k, v = (torch.randn(n_w, 4, 32, generator=gen) for _ in range(2))
    seed = torch.randn(p, 4, 4, 32, generator=gen)
    got = _grads(lambda a, c, d: OPS.window_latent_read(a, c, d, *layout)[0], [x.to(device) for x in (q, k, v)],
                 seed.to(device))
    exp = _grads(lambda a, c, d: R.latent_read(a, c, d, offsets, order), [q, k, v], seed)
    _close(got, exp, torch.float32)
    qb = torch.randn(n_w, 4, 32, generator=gen)
    kb, vb = (torch.randn(p, 4, 4, 32, generator=gen) for _ in range(2))
    seed = torch.randn(n_w, 4, 32, generator=gen)
    got = _grads(lambda a, c, d: OPS.window_latent_broadcast(a, c, d, *layout)[0],
                 [x.to(device) for x in (qb, kb, vb)], seed.to(device))
    exp = _grads(lambda a, c, d: R.latent_broadcast(a, c, d, window_pos), [qb, kb, vb], seed)
    _close(got, exp, torch.float32)
    mantisnet.ops.raise_on_device_error(device)


@pytest.mark.parametrize("n_k,dt,with_vcls", [(400, torch.float32, True), (19, torch.float32, False),
                                              (18, torch.float16, True), (5, torch.float32, True),
                                              (4, torch.bfloat16, False), (1, torch.float32, True)])
def test_cell_attention_backward_run_lengths(device, n_k, dt, with_vcls):
    """300 entries over few or many source rows: mean source runs either side
    of 16 and 64 entries (one, 4 or 16 lane groups per row), query runs of 0
    to over 16 entries, one class owning most entries."""
    gen = torch.Generator().manual_seed(27 + n_k)
    n_q, n_e = 33, 300
    dst = torch.cat([torch.full((40,), 7), torch.randint(8, n_q, (n_e - 40,), generator=gen)])
    src = torch.randint(0, n_k, (n_e,), generator=gen)
    cls = torch.where(torch.rand(n_e, generator=gen) < 0.7, 2, torch.randint(0, 5, (n_e,), generator=gen))
    t = R.edge_tables_full(src, dst, cls, torch.zeros(0, dtype=torch.long), n_k, n_q, 5, False)
    views = [t[n].to(device) for n in ("dst_ptr", "edge_src", "edge_class", "edge_dst", "source_ptr", "edge_sdst",
                                       "edge_sclass", "cls_ptr", "cedge_dst")]
    inputs = [torch.randn(n, 4, 32, generator=gen).to(dt) for n in (n_q, n_k, n_k)]
    inputs += [0.3 * torch.randn(4, 5, generator=gen)] + ([0.1 * torch.randn(5, 128, generator=gen)] if with_vcls else [])
    seed = torch.randn(n_q, 4, 32, generator=gen)
    op = OPS.cell_attention if with_vcls else OPS.cell_attention_plain

    def ref(q, k, v, b, c=None):
        return R.cell_attention(q, k, v, b, c, t["edge_src"], t["edge_class"], t["edge_dst"])

    got = _grads(lambda *x: op(*x, *views)[0], [x.to(device) for x in inputs], seed.to(device))
    mantisnet.ops.raise_on_device_error(device)
    _close(got, _grads(ref, [x.float() for x in inputs], seed), dt)
    again = _grads(lambda *x: op(*x, *views)[0], [x.to(device) for x in inputs], seed.to(device))
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_attention_backward_without_classes_or_query_ids(device, dt):
    """The module-level forms that the operators do not take: untyped entries
    are entries of one class without a bias, and without the entries' query
    ids the query pass itself finishes the bias gradient's terms."""
    gen = torch.Generator().manual_seed(29)
    n_q, n_k, n_e = 21, 13, 160
    dst, src = torch.randint(3, n_q, (n_e,), generator=gen), torch.randint(0, n_k, (n_e,), generator=gen)
    q, k, v = (torch.randn(n, 4, 32, generator=gen).to(device, dt) for n in (n_q, n_k, n_k))
    go = torch.randn(n_q, 4, 32, generator=gen).to(device)
    back = mantisnet.ops.attention_backward
    for n_cls in (1, 3):
        t = R.edge_tables_full(src, dst, torch.randint(0, n_cls, (n_e,), generator=gen), dst[:0], n_k, n_q, n_cls, False)
        bias = torch.zeros(4, n_cls, device=device)
        views = [t[n].to(device) for n in ("dst_ptr", "edge_src", "edge_class", "edge_dst", "source_ptr", "edge_sdst",
                                           "edge_sclass", "cls_ptr", "cedge_dst")]
        _, m, l = OPS.cell_attention_plain(q, k, v, bias, *views)
        full = OPS.cell_attention_plain_backward(q, k, v, bias, *views, m, l, go)
        seg, es, ec, _, sseg, sqid, scls, cptr, cedge = views
        no_qid = back(q, k, v, bias, None, go, m, l, seg, es, ec, None, sseg, sqid, scls, cptr, cedge)
        assert all(torch.equal(a, b) for a, b in zip(no_qid[:3], full))
        # fp32 sums of 160 terms of up to about 5 each
        torch.testing.assert_close(no_qid[3], full[3], rtol=0, atol=5e-5)
        untyped = back(q, k, v, None, None, go, m, l, seg, es, None, None, sseg, sqid, None, None, None)
        assert all(torch.equal(a, b) for a, b in zip(untyped[:3], full)) and untyped[3] is None and untyped[4] is None
    mantisnet.ops.raise_on_device_error(device)


@pytest.mark.parametrize("counts,dt,shuffled", [
    ([0], torch.float32, False), ([1], torch.float32, False), ([63, 64, 65], torch.float32, True),
    ([3, 0, 700, 17], torch.float32, True), ([130, 1, 0], torch.bfloat16, False), ([16, 15, 257], torch.float16, True),
])
def test_window_latent_backward_layouts(device, counts, dt, shuffled):
    """Runs around the lane groups and the split of a position's windows,
    positions without windows, and windows whose order is not the identity."""
    p, n_w = len(counts), sum(counts)
    gen = torch.Generator().manual_seed(25 + n_w)
    window_pos = torch.repeat_interleave(torch.arange(p), torch.tensor(counts))
    if shuffled:
        window_pos = window_pos[torch.randperm(n_w, generator=gen)]
    offsets, order = R.window_layout(window_pos, p)
    layout = [x.to(device) for x in (window_pos, offsets, order)]
    shapes = [(p, 4, 4, 32), (n_w, 4, 32)]
    for read in (True, False):
        sq, sk = shapes if read else shapes[::-1]
        q, k, v = (torch.randn(*s, generator=gen).to(dt) for s in (sq, sk, sk))
        seed = torch.randn(*sq, generator=gen)
        op = OPS.window_latent_read if read else OPS.window_latent_broadcast
        got = _grads(lambda a, c, d: op(a, c, d, *layout)[0], [x.to(device) for x in (q, k, v)], seed.to(device))
        ref = (lambda a, c, d: R.latent_read(a, c, d, offsets, order)) if read else (
            lambda a, c, d: R.latent_broadcast(a, c, d, window_pos))
        exp = _grads(ref, [x.float() for x in (q, k, v)], seed) if n_w else [torch.zeros(s) for s in (sq, sk, sk)]
        _close(got, exp, dt)
        assert all(g.dtype == dt for g in got)
    mantisnet.ops.raise_on_device_error(device)


def test_window_latent_backward_takes_any_order(device):
    """An order that is not a permutation: the latent rows sum over the order's
    runs, the window rows come from each window's own position."""
    gen = torch.Generator().manual_seed(26)
    window_pos = torch.tensor([0, 1, 1, 0, 1])
    offsets, order = torch.tensor([0, 3, 5]), torch.tensor([0, 0, 2, 1, 4])  # window 3 unnamed, 0 twice, 2 misplaced
    layout = [x.to(device) for x in (window_pos, offsets, order)]
    q, k, v = (torch.randn(*s, generator=gen).to(device) for s in ((2, 4, 4, 32), (5, 4, 32), (5, 4, 32)))
    go = torch.randn(2, 4, 4, 32, generator=gen).to(device)
    out, m, l = OPS.window_latent_read(q, k, v, *layout)
    dq, dk, dv = OPS.window_latent_read_backward(q, k, v, *layout, out, m, l, go)
    sc = 32 ** -0.5
    delta = (go * out).sum(-1)

    def terms(w, p):  # alpha, dscore: (slots, heads)
        al = torch.exp((q[p] * k[w]).sum(-1) * sc - m[p]) / l[p]
        return al, al * ((go[p] * v[w]).sum(-1) - delta[p])

    for p in range(2):
        exp = sum(terms(w, p)[1][..., None] * k[w] * sc for w in order[offsets[p]:offsets[p + 1]].tolist())
        torch.testing.assert_close(dq[p], exp, rtol=1e-4, atol=1e-4)
    for w in range(5):
        p = int(window_pos[w])
        al, ds = terms(w, p)
        torch.testing.assert_close(dv[w], (al[..., None] * go[p]).sum(0), rtol=1e-4, atol=1e-4)
        torch.testing.assert_close(dk[w], (ds[..., None] * q[p]).sum(0) * sc, rtol=1e-4, atol=1e-4)
    mantisnet.ops.raise_on_device_error(device)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("read", [True, False])
@pytest.mark.parametrize("which", [0, 1])
def test_window_latent_backward_keeps_non_finite_scores(device, read, which, value):
    """A non-finite query or key element: the rows whose softmax it leaves
    undefined get NaN gradients for all of their head's dims and pass NaN to
    their head's dims of every key they meet, where autograd through the oracle
    has NaN; the other positions and heads stay finite.  (Such a row's output
    can be 0.)"""
    gen = torch.Generator().manual_seed(33)
    counts = [70, 0, 3, 18]
    window_pos = torch.repeat_interleave(torch.arange(4), torch.tensor(counts))
    window_pos = window_pos[torch.randperm(len(window_pos), generator=gen)]
    offsets, order = R.window_layout(window_pos, 4)
    layout = [x.to(device) for x in (window_pos, offsets, order)]
    sq, sk = ((4, 4, 4, 32), (91, 4, 32)) if read else ((91, 4, 32), (4, 4, 4, 32))
    ins = [torch.randn(*s, generator=gen) for s in (sq, sk, sk)]
    # where the forward's own sums are the oracle's: the read's lane groups skip a
    # NaN score that they meet alone and make a lone -inf a NaN
    p = 0 if value != value else 2
    w = int((window_pos == p).nonzero()[1])
    at = (p, 1, 3, 5) if (which == 0) == read else (w, 3, 5)  # a latent's or a window's head 3
    ins[which][at] = value
    go = torch.randn(*sq, generator=gen)
    op = OPS.window_latent_read if read else OPS.window_latent_broadcast
    got = _grads(lambda *x: op(*x, *layout)[0], [x.to(device) for x in ins], go.to(device))
    mantisnet.ops.raise_on_device_error(device)
    ref = (lambda *x: R.latent_read(*x, offsets, order)) if read else (lambda *x: R.latent_broadcast(*x, window_pos))
    exp = _grads(ref, ins, go)
    for g, e in zip(got[:2], exp):
        assert torch.isnan(e).any() and torch.equal(torch.isnan(g.cpu()), torch.isnan(e))
    torch.testing.assert_close(got[0].cpu(), exp[0], rtol=1e-4, atol=1e-4, equal_nan=True)
    torch.testing.assert_close(got[1].cpu(), exp[1], rtol=1e-4, atol=1e-4, equal_nan=True)
    assert torch.isfinite(got[2]).all()


def test_latent_read_backward_without_the_forward_output(device):
    # the module-level call as it was: m, l and the gradient, out formed again
    gen = torch.Generator().manual_seed(28)
    window_pos = torch.tensor([0] * 70 + [2] * 9)
    offsets, order = R.window_layout(window_pos, 3)
    q, k, v, go = (torch.randn(*s, generator=gen).to(device) for s in ((3, 4, 4, 32), (79, 4, 32), (79, 4, 32),
                                                                     (3, 4, 4, 32)))
    layout = [x.to(device) for x in (window_pos, offsets, order)]
    out, m, l = OPS.window_latent_read(q, k, v, *layout)
    got = mantisnet.ops.latent_read_backward(q, k, v, *layout, m, l, go)
    assert all(torch.equal(a, b) for a, b in zip(got, OPS.window_latent_read_backward(q, k, v, *layout, out, m, l, go)))


def test_action_row_encode_backward(device, batch):
    b = batch
    n_w, n_c = b.window_feat.numel(), b.cell_pos.shape[0]
    t = R.cell_tables_full(b.dec_cell, b.dec_window, b.dec_class, n_w, 726, n_c)
    gen = torch.Generator().manual_seed(23)
    pre = torch.randn(n_w, 128, generator=gen)
    table = torch.randn(729, 128, generator=gen)
    cls = torch.randint(0, 729, (t["edge_cell"].numel(),), generator=gen)
    seed = torch.randn(n_c, 128, generator=gen)
    # edge_rev: the window-major order of the cell-major entries (the batch's act_rev)
    edge_rev = torch.argsort(t["edge_window"], stable=True)
    idx = [x.to(device) for x in (t["edge_window"], cls, t["edge_cell"], edge_rev)]
    got = _grads(lambda a, c: OPS.action_row_encode(a, c, *idx, n_c), [pre.to(device), table.to(device)],
                 seed.to(device))
    exp = _grads(lambda a, c: R.encode_rows(a, c, t["edge_window"], cls, t["edge_cell"], n_c), [pre, table], seed)
    _close(got, exp, torch.float32)
    mantisnet.ops.raise_on_device_error(device)


@pytest.mark.parametrize("heads,hd,dt", [(4, 32, torch.float16), (8, 32, torch.float16), (4, 32, torch.bfloat16),
                                         (3, 16, torch.float16), (4, 16, torch.bfloat16), (2, 64, torch.float16),
                                         (4, 64, torch.bfloat16)])
def test_fused_attention_backward(device, heads, hd, dt):
    gen = torch.Generator().manual_seed(24 + hd)
    p, t = 5, 140
    lens = torch.tensor([140, 4, 65, 64, 0], dtype=torch.int32)
    q, k, v = (torch.randn(p, t, heads, hd, generator=gen).to(dt).transpose(1, 2) for _ in range(3))
    seed = torch.randn(p, heads, t, hd, generator=gen)
    valid = torch.arange(t)[None, :] < lens[:, None]
    seed = seed.masked_fill(~valid[:, None, :, None], 0.0)  # pad rows carry no gradient in either form
    ld = lens.to(device)
    got = _grads(lambda a, c, d: OPS.fused_attention(a, c, d, ld)[0], [x.to(device) for x in (q, k, v)],
                 seed.to(device, dt))
    mantisnet.ops.raise_on_device_error(device)
    exp = _grads(lambda a, c, d: R.stone_attention(a, c, d, lens), [x.float() for x in (q, k, v)],
                 seed.to(dt).float())
    _close(got, exp, dt)
    assert all(g.dtype == dt for g in got)
    # pad keys and rows: zero gradients
    for g in got:
        assert torch.count_nonzero(g.cpu().float().masked_fill(valid[:, None, :, None], 0.0)) == 0
    # two backward passes agree bitwise
    again = _grads(lambda a, c, d: OPS.fused_attention(a, c, d, ld)[0], [x.to(device) for x in (q, k, v)],
                   seed.to(device, dt))
    assert all(torch.equal(a.cpu(), b.cpu()) for a, b in zip(got, again))


@pytest.mark.parametrize("hd,dt,grad_scale", [(16, torch.bfloat16, 1.0), (32, torch.bfloat16, 1.0),
                                              (64, torch.bfloat16, 1.0), (16, torch.float16, 1.0),
                                              (32, torch.float16, 1e-3), (64, torch.float16, 1.0)])
def test_fused_attention_backward_tiles(device, hd, dt, grad_scale):
    """Lengths around the 16-row sub-tiles and the 64-row tiles and chunks, T
    off a tile, at small gradients too: within one rounding of the gradients
    of float64 attention (2^-9 bf16, 2^-12 fp16 relative, and the forward's
    rounded output and normaliser in delta, a few times that on the sums)."""
    gen = torch.Generator().manual_seed(40 + hd)
    lens = torch.tensor([0, 1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 201], dtype=torch.int32)
    p, t, heads = len(lens), 201, 3
    q, k, v, go = (torch.randn(p, t, heads, hd, generator=gen).to(dt).transpose(1, 2) for _ in range(4))
    go = (go.float() * grad_scale).to(dt)
    valid = (torch.arange(t)[None, :] < lens[:, None])[:, None, :, None]
    go = go.masked_fill(~valid, 0.0)
    got = _grads(lambda a, b, c: OPS.fused_attention(a, b, c, lens.to(device))[0], [x.to(device) for x in (q, k, v)],
                 go.to(device))

    def ref(a, b, c):  # float64; a position without live rows has no keys
        s = (a @ b.transpose(2, 3)) / hd ** 0.5
        s = s.masked_fill(~valid.transpose(2, 3), -1e30)
        return (s.softmax(-1) @ c).masked_fill(~valid, 0.0)

    exp = _grads(ref, [x.double() for x in (q, k, v)], go.double())
    tol = 2 ** -9 if dt == torch.bfloat16 else 2 ** -12
    for g, e in zip(got, exp):
        g, e = g.cpu().double(), e.masked_fill(~valid, 0.0)
        assert float((g - e).norm() / e.norm()) < 2 * tol + 1e-7 / grad_scale
        assert torch.count_nonzero(g.masked_fill(valid, 0.0)) == 0


def _attention_backward_terms(q, k, v, lens, lse, go, out, scale):
    """P, dS (heads, L, L) and the live rows of each position in float64."""
    for p, n in enumerate(lens.tolist()):
        a, b, c, g, o = (x[p, :, :n].double() for x in (q, k, v, go, out))
        pr = torch.exp(a @ b.transpose(1, 2) * scale - lse[p, :, :n].double()[..., None])
        yield p, n, a, b, g, pr, pr * (g @ c.transpose(1, 2) - (o * g).sum(-1)[..., None])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [16, 32, 64])
def test_fused_attention_backward_keeps_fp32_probabilities(device, hd, dt):
    """Queries in pairs a few 16-bit steps apart with opposite gradients: dv and
    dk are 2^-7 and less of their terms, so what a product loses of P or dS
    shows through the output's rounding.  Past half a rounding step the error
    stays within 2^-20 of the terms' root sum of squares: fp32 operands leave
    2^-22 of the exponent's argument and 2^-25 of the sums, operands of 16
    significant bits leave 2^-17."""
    gen = torch.Generator().manual_seed(50 + hd)
    lens = torch.tensor([2, 8, 64, 66, 128], dtype=torch.int32)
    p, t, heads, scale = len(lens), 130, 2, hd ** -0.5
    q, go = (torch.randn(p, heads, t // 2, hd, generator=gen).repeat_interleave(2, 2) for _ in range(2))
    q[:, :, 1::2] += 2 ** -9 * torch.randn(p, heads, t // 2, hd, generator=gen)
    go[:, :, 1::2] *= -1
    k, v = (torch.randn(p, heads, t, hd, generator=gen) for _ in range(2))
    q, k, v, go = (x.to(dt) for x in (q, k, v, go))
    out, lse = torch.zeros_like(q), torch.zeros(p, heads, t)
    for i, n in enumerate(lens.tolist()):
        s = q[i, :, :n].double() @ k[i, :, :n].double().transpose(1, 2) * scale
        lse[i, :, :n] = s.logsumexp(-1).float()
        out[i, :, :n] = (s.softmax(-1) @ v[i, :, :n].double()).to(dt)
    dq, dk, dv = (x.cpu().double() for x in OPS.fused_attention_backward(
        *(x.to(device) for x in (q, k, v, lens, out, lse, go))))
    half = 2 ** -8 if dt == torch.bfloat16 else 2 ** -11
    worst = {}
    for i, n, a, b, g, pr, ds in _attention_backward_terms(q, k, v, lens, lse, go, out, scale):
        for name, got, x, rows, f in (("dv", dv, pr.transpose(1, 2), g, 1.0),
                                      ("dk", dk, ds.transpose(1, 2), a, scale), ("dq", dq, ds, b, scale)):
            exp = x @ rows * f
            terms = f * ((x ** 2) @ (rows ** 2)).sqrt()
            over = ((got[i, :, :n] - exp).abs() - half * exp.abs() - 2 ** -25).clamp(min=0)  # (fp16 below 2^-14)
            worst[name, n] = float((over ** 2).mean().sqrt() / (terms ** 2).mean().sqrt())
    print(hd, dt, {k: f"{v:.1e}" for k, v in worst.items()}, flush=True)
    assert max(worst.values()) < 2 ** -20, worst


@pytest.mark.parametrize("hd", [16, 32, 64])
def test_fused_attention_backward_of_a_masked_key(device, hd):
    """A key of -inf scores (P = 0 on every row) gets zero gradients, and the
    rows past the prefix bring none to it; an infinite P leaves infinities of
    the gradient's sign."""
    gen = torch.Generator().manual_seed(60 + hd)
    n, t, scale = 3, 70, hd ** -0.5
    lens = torch.tensor([n], dtype=torch.int32)
    q, k, v, go = (torch.randn(1, 1, t, hd, generator=gen).bfloat16() for _ in range(4))
    q[..., 0] = q[..., 0].abs() + 1
    k[0, 0, 1, 0] = float("-inf")
    s = q[0, 0, :n].double() @ k[0, 0, :n].double().t() * scale
    lse, out = torch.zeros(1, 1, t), torch.zeros_like(q)
    lse[0, 0, :n] = s.logsumexp(-1).float()
    out[0, 0, :n] = (s.softmax(-1) @ v[0, 0, :n].double()).bfloat16()
    args = [x.to(device) for x in (q, k, v, lens, out, lse, go)]
    dq, dk, dv = (x.cpu().double() for x in OPS.fused_attention_backward(*args))
    assert not dk[0, 0, 1].any() and not dv[0, 0, 1].any()
    for i, m, a, b, g, pr, ds in _attention_backward_terms(q, k, v, lens, lse, go, out, scale):
        torch.testing.assert_close(dv[i, :, :m], pr.transpose(1, 2) @ g, rtol=2 ** -8, atol=1e-6)
        torch.testing.assert_close(dk[i, :, :m], ds.transpose(1, 2) @ a * scale, rtol=2 ** -8, atol=1e-6)
        torch.testing.assert_close(dq[i, :, :m, 1:], (ds @ b * scale)[..., 1:], rtol=2 ** -8, atol=1e-6)
    args[3], args[5] = torch.ones_like(args[3]), torch.full_like(args[5], -500.0)
    dv = OPS.fused_attention_backward(*args)[2].cpu().float()
    assert torch.equal(dv[0, 0, 0], torch.copysign(torch.tensor(float("inf")), go[0, 0, 0].float()))
