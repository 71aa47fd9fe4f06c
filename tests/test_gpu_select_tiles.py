"""GPU: the slot-selection kernels for the common shapes against the general ones, bit for bit: scores
of 64 / 128 / 256-wide heads against the same vectors zero-padded to a width the general kernel takes,
and the top-k of rows whose keys fit in registers against the same rows padded past that size.  Plus
the row plan's offset tables from kernel arguments."""

from __future__ import annotations

import pytest
import torch

import oracle as O
from kv_skill_v2_amd import ops, synth

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.mark.parametrize("hd,n_kv,G,S", [(64, 1, 1, 1), (64, 2, 8, 33), (128, 3, 3, 130), (128, 1, 2, 257),
                                         (256, 4, 4, 64), (256, 2, 7, 19), (256, 1, 1, 100)])
@pytest.mark.parametrize("pool", ["max", "mean"])
def test_scores_equal_the_general_kernel(dev, hd, n_kv, G, S, pool):
    say("select scores", dict(hd=hd, n_kv=n_kv, G=G, S=S, pool=pool))
    g = torch.Generator().manual_seed(hd + S)
    q, keys = torch.randn(2, n_kv * G, hd, generator=g), torch.randn(S, n_kv, hd, generator=g)
    valid = torch.rand(S, generator=g) > 0.2
    pad = lambda t: torch.nn.functional.pad(t, (0, 320 - hd))  # noqa: E731
    got = ops.select_scores(q.to(dev), keys.to(dev), valid.to(dev), pool)
    want = ops.select_scores(pad(q).to(dev), pad(keys).to(dev), valid.to(torch.int64).to(dev), pool)
    assert torch.equal(got, want)
    ref = O.select_scores(q.double(), keys.double(), valid, pool)
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(got).cpu(), fin)
    if fin.any():
        # hd products of unit normals: |error| <= hd eps sum |q k| < hd * 2^-24 * 4 hd, far below this
        assert float((got.cpu().double() - ref)[fin].abs().max()) < 1e-3


@pytest.mark.parametrize("S,k", [(1, 1), (63, 63), (1024, 256), (1025, 257), (8192, 64), (8192, 1024), (8193, 100),
                                 (32768, 1000), (32767, 1), (5000, 0)])
def test_topk_equals_the_general_kernel(dev, S, k):
    say("topk", dict(S=S, k=k))
    g = torch.Generator().manual_seed(S + k)
    sc = torch.randn(4, S, generator=g)
    sc[1] = torch.randint(-3, 3, (S,), generator=g).float() / 4          # ties at the edge
    sc[2, ::3] = float("-inf")
    sc[3] = 0.0
    sc[3, ::2] = -0.0
    sc[3, S // 2] = float("inf")
    sc[3, S // 3] = float("nan")
    idx, vals = ops.topk_rows(sc.to(dev), k)
    wide = torch.nn.functional.pad(sc, (0, 40000 - S), value=float("-inf")).to(dev)
    want_idx, want = ops.topk_rows(wide, k)
    assert torch.equal(idx, want_idx)
    assert torch.equal(vals.view(torch.int32), want.view(torch.int32))
    order = O.topk_order(sc[:3], k)
    assert torch.equal(idx[:3].cpu().long(), order)


@pytest.mark.parametrize("n_lib", [1, 3, 80])
def test_row_plan_tables(dev, n_lib):
    """The offset tables (kernel arguments up to 256 integers, a copy beyond)."""
    counts = [1 + i % 3 for i in range(n_lib)]
    P = synth.pool(counts, 64, 64, device="cpu")
    lib = ops.PagedLibrary(*(t.to(dev) for t in (P.pages, P.chunk_page, P.chunk_nvalid, P.chunk_ptr, P.S)),
                           n_chunks=P.n_chunks, nvalid=P.nvalid)
    rows = [(37 * i) % 300 for i in range(n_lib)]
    plan = ops.row_plan(lib, rows)
    tiles = lambda t, n: -(-t // n)  # noqa: E731
    want = {"row_ptr": rows, "score_tiles": [tiles(t, 128) * c for t, c in zip(rows, counts)],
            "readout_tiles": [tiles(t, 128) for t in rows], "route_tiles": [tiles(t, 16) for t in rows],
            "logit_tiles": [tiles(t, 32) * tiles(c, 32) for t, c in zip(rows, counts)]}
    for name, per in want.items():
        t = getattr(plan, name)
        assert t.is_cuda and t.dtype == torch.int32
        assert t.cpu().tolist() == [sum(per[:i]) for i in range(n_lib + 1)], name


@pytest.mark.parametrize("M,C,d", [(300, 9, 2048), (512, 5, 2048), (513, 33, 2048), (1030, 16, 1024), (2050, 40, 2048)])
def test_route_topk_is_one_result(dev, M, C, d):
    """Routing with a workgroup per row and split over waves: either side of the line the same bits as calls
    of fewer than 256 rows."""
    say("route topk rows", dict(M=M, C=C, d=d))
    P = synth.pool([C], 64, d, device="cpu")
    lib = ops.PagedLibrary(*(t.to(dev) for t in (P.pages, P.chunk_page, P.chunk_nvalid, P.chunk_ptr, P.S)),
                           n_chunks=P.n_chunks, nvalid=P.nvalid)
    q = synth.queries(M, d, device=dev, seed=8)
    got = ops.route_topk(q, lib, None, 3)
    want = [torch.cat(t) for t in zip(*(ops.route_topk(x, lib, None, 3) for x in q.split(200)))]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
