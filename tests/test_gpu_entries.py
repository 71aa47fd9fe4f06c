"""GPU: the read of many rows by entries (the routed (row, chunk) pairs grouped by chunk,
csrc/entries.hip) against the fp64 oracle and against the dense 128-row tiles it replaces: both
tile heights, every slot-group split of a page, ragged libraries (fewer chunks than top_k, no rows),
fewer columns than column groups, one entry per row, untied values, the linear read, slot blocks
and their all-masked tails, and the gradient through the read, the routing and an outside use of
the weights.  fp16 operands with fp32 sums: the prefill tests' bars."""

from __future__ import annotations

import pytest
import torch

import oracle as O
from kv_skill_v2_amd import ops, synth

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


def _close(got, ref, what):
    got, ref = got.double().cpu(), ref.double()
    err, scale = (got - ref).abs().max().item(), ref.abs().max().item()
    rel = ((got - ref).norm() / ref.norm().clamp_min(1e-30)).item()
    assert rel <= 2e-3 and err <= 1e-2 * max(scale, 1e-30), (what, rel, err, scale)


def _oracle(P, q, rows, top_k, softmax, untied):
    r, w, at = [], [], 0
    cmax = max(P.n_chunks)
    for g, T in enumerate(rows):
        K, M, S = P.library(g)
        v = K.double().roll(1, -1) if untied else None
        rg, wg = O.branch_read(q[None, at:at + T], K.double(), M, S.double(), top_k=top_k, read_softmax=softmax, V=v)
        r.append(rg[0])
        w.append(torch.nn.functional.pad(wg[0], (0, cmax - wg.shape[-1])))
        at += T
    return torch.cat(r), torch.cat(w)


CASES = [
    # (d, N, chunks per library, rows per library, top_k, softmax, untied)
    (64, 64, [5, 3], [70, 33], 2, True, False),          # 1 k step for 8 column groups
    (256, 512, [4], [64], 2, True, False),
    (320, 128, [9, 2, 4], [40, 0, 129], 3, True, False),  # a library of 2 chunks, one without rows
    (512, 192, [7], [130], 3, False, True),
    (256, 320, [6, 12], [65, 100], 4, True, True),        # 5 of 8 slot groups
    (128, 256, [3], [97], 1, True, False),                # one entry per row
    (2048, 512, [3], [66], 0, True, False),               # every chunk
]


# (64-row tiles take pages of more than 128 slots)
@pytest.mark.parametrize("d,N,counts,rows,top_k,softmax,untied,tile",
                         [(*c, t) for c in CASES for t in (32, 64) if t == 32 or c[1] > 128])
def test_entries_read_and_gradient(dev, monkeypatch, d, N, counts, rows, top_k, softmax, untied, tile):
    say("entries", dict(d=d, N=N, counts=counts, rows=rows, top_k=top_k, softmax=softmax, untied=untied, tile=tile))
    P = synth.pool(counts, N, d, device="cpu", tail_lo=1)
    lib = ops.PagedLibrary(*(t.to(dev) for t in (P.pages, P.chunk_page, P.chunk_nvalid, P.chunk_ptr, P.S)),
                           n_chunks=P.n_chunks, nvalid=P.nvalid,
                           values=P.pages.roll(1, -1).to(dev) if untied else None)   # columns moved by one
    M = sum(rows)
    q = synth.queries(M, d, device="cpu", seed=5)
    g = torch.Generator().manual_seed(3)
    up, uw = torch.randn(M, d, generator=g), torch.randn(M, lib.cmax, generator=g)
    plan = lib.plan(rows)

    q64 = q.double().requires_grad_()
    r64, w64 = _oracle(P, q64, rows, top_k, softmax, untied)
    d64, = torch.autograd.grad((r64 * up.double()).sum() + (w64 * uw.double()).sum(), q64, retain_graph=True)
    d64r, = torch.autograd.grad((r64 * up.double()).sum(), q64)

    monkeypatch.setattr(ops, "_entry_tile", lambda *a: tile)
    for with_w, ref in ((True, d64), (False, d64r)):
        qd = q.to(dev).requires_grad_()
        r, w = ops.library_read(qd, lib, plan, top_k=top_k, read_softmax=softmax)
        loss = (r * up.to(dev)).sum() + ((w * uw.to(dev)).sum() if with_w else 0.0)
        dq, = torch.autograd.grad(loss, qd)
        _close(r.detach(), r64.detach(), "r")
        _close(w.detach(), w64.detach(), "w")
        _close(dq, ref, "dq")
    monkeypatch.setattr(ops, "_entry_tile", lambda *a: 0)
    qd = q.to(dev).requires_grad_()
    r0, w0 = ops.library_read(qd, lib, plan, top_k=top_k, read_softmax=softmax)
    assert torch.equal(w0, w)                      # the routing is the same kernels'
    _close(r.detach(), r0.detach().cpu().double(), "r vs dense")
    wq = q.to(dev).requires_grad_()                # only w reaches the loss
    monkeypatch.setattr(ops, "_entry_tile", lambda *a: tile)
    _, w1 = ops.library_read(wq, lib, plan, top_k=top_k, read_softmax=softmax)
    dw, = torch.autograd.grad((w1 * uw.to(dev)).sum(), wq)
    d64w, = torch.autograd.grad((_oracle(P, q64, rows, top_k, softmax, untied)[1] * uw.double()).sum(), q64)
    _close(dw, d64w, "dq of w")


@pytest.mark.parametrize("d,N,C,M,top_k,softmax,nv", [
    (64, 192, 3, 9, 2, True, 192), (256, 512, 5, 40, 3, True, 130), (512, 320, 1, 70, 0, True, 64),
    (320, 448, 4, 33, 0, True, 449 - 65), (256, 512, 6, 65, 2, False, 512), (1024, 64, 2, 31, 1, True, 3)])
def test_entries_without_gradient(dev, monkeypatch, d, N, C, M, top_k, softmax, nv):
    """branch_read and read_rows by entries (few tiles: pages over 128 slots in 128-slot blocks, the
    last chunk of nv slots leaving whole blocks masked) against the oracle and the dense tiles."""
    say("entries no grad", dict(d=d, N=N, C=C, M=M, top_k=top_k, softmax=softmax, nv=nv))
    P = synth.pool([C], N, d, device="cpu", tail_lo=1)
    P.nvalid[-1] = nv
    P.chunk_nvalid[-1] = nv
    lib = ops.PagedLibrary(*(t.to(dev) for t in (P.pages, P.chunk_page, P.chunk_nvalid, P.chunk_ptr, P.S)),
                           n_chunks=P.n_chunks, nvalid=P.nvalid)
    q = 3.0 * synth.queries(M, d, device="cpu", seed=6)   # sharper scores: block maxima far apart
    K = P.pages[P.chunk_page.long()].double()
    mask = torch.arange(N)[None] < P.chunk_nvalid[:, None]
    r64, w64 = O.branch_read(q[None].double(), K, mask, P.S.double(), top_k=top_k, read_softmax=softmax)
    out = {}
    for tile in (32, 0):
        monkeypatch.setattr(ops, "_entry_tile", lambda *a: tile)
        r, w = ops.branch_read(q.to(dev), lib, top_k, 12.0, 10.0, softmax)
        _close(r, r64[0], f"r tile {tile}")
        _close(w, w64[0], "w")
        _, idx, wsel = ops.route_rows(q.to(dev), lib, top_k)
        out[tile] = (w, ops.read_rows(q.to(dev), w, idx, wsel, lib, 12.0, softmax))
        _close(out[tile][1], r64[0], f"read_rows tile {tile}")
    assert torch.equal(out[0][0], out[32][0])
    empty, _ = ops.branch_read(q[:0].to(dev), lib, top_k)
    assert empty.shape == (0, d)


def test_entries_rule(dev):
    """Routed launches read by entries, large dense ones by 128-row tiles."""
    assert ops._entry_tile_of(48, 3, 333 * 4, 16, 16, 4, 512, 2048) == 32
    assert ops._entry_tile_of(1024, 16, 2048 * 8, 64, 64, 8, 512, 2048) == 64
    assert ops._entry_tile_of(2048, 64, 8192 * 32, 128, 32, 32, 512, 2048) == 0


CHECKS = ("test_schema", "test_autograd_registration", "test_faketensor", "test_aot_dispatch_dynamic")


def test_entries_operators(dev, monkeypatch):
    """opcheck (schema, fakes, autograd, AOT dispatch with the backward) of the operators; saved tensors
    packed and unpacked by hooks; a gradient of the gradient-free outputs; no gradient at all."""
    say("entries operators")
    P = synth.pool([4, 3], 128, 128, device="cpu", tail_lo=1)
    lib = ops.PagedLibrary(*(t.to(dev) for t in (P.pages, P.chunk_page, P.chunk_nvalid, P.chunk_ptr, P.S)),
                           n_chunks=P.n_chunks, nvalid=P.nvalid)
    plan = lib.plan([70, 66])
    q = synth.queries(plan.M, lib.d, device=dev, seed=4).requires_grad_(True)
    fk, fv, fvs, fkr, chunk_ptr, chunk_page, chunk_nvalid, row_ptr, *_ = ops._prefill_operands(lib, plan)
    args = (q, lib.S, chunk_ptr, row_ptr, plan.logit_tiles, plan.route_tiles, plan.n_logit, plan.n_route, 2, 10.0,
            lib.cmax, 2, fk, fv, fvs, fkr, chunk_page, chunk_nvalid, 70, 32, 128, 12.0, True)
    # (a list's tail past its chunk's count is never written, so whole outputs are not compared here)
    torch.library.opcheck(torch.ops.xenc.library_read_entries.default, args, test_utils=CHECKS[:3])
    r, w, idx, _, p, lst, count = torch.ops.xenc.library_read_entries(*args)
    assert r.requires_grad and w.requires_grad and not any(t.requires_grad for t in (idx, p, lst, count))
    g = torch.randn(r.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(1))
    want, = torch.autograd.grad(r, q, g, retain_graph=True)
    from functorch.compile import aot_function, nop
    traced = aot_function(lambda *a: torch.ops.xenc.library_read_entries(*a)[:2], nop, nop)
    rt, wt = traced(*args)
    got, = torch.autograd.grad(rt, q, g)
    assert torch.equal(rt, r) and torch.equal(wt, w) and torch.equal(got, want)
    bargs = (g, w.detach(), idx, p, torch.randn_like(w), lib.S, lst, count, fvs, fkr, chunk_ptr, chunk_page, chunk_nvalid,
             row_ptr, 70, 32, 128, 12.0, True, 10.0)
    torch.library.opcheck(torch.ops.xenc.library_read_entries_bwd.default, bargs,
                          test_utils=("test_schema", "test_faketensor"))
    for i, blocks in ((None, 1), (idx, 1)):
        rargs = (q.detach(), w.detach(), i, fk, fv, chunk_ptr, row_ptr, chunk_page, chunk_nvalid, 70, 32, blocks, 128, 12.0,
                 True)
        torch.library.opcheck(torch.ops.xenc.read_entries.default, rargs, test_utils=CHECKS)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(), lambda t: t.to(dev)):
        r2 = torch.ops.xenc.library_read_entries(*args)[0]
        got, = torch.autograd.grad(r2, q, g)
    assert len(packed) == 13 and torch.equal(got, want)
    monkeypatch.setattr(ops, "_entry_tile", lambda *a: 32)
    with torch.no_grad():
        r3, w3 = ops.library_read(q, lib, plan, top_k=2)
    assert torch.equal(r3, r.detach()) and not r3.requires_grad and torch.equal(w3, w.detach())
    with torch.inference_mode():
        assert torch.equal(ops.library_read(q.detach().clone(), lib, plan, top_k=2)[0], r3)
    dq, = torch.autograd.grad(w.sum() * 0.0 + r.sum() * 0.0, q)
    assert float(dq.abs().max()) == 0.0
