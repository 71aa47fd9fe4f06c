"""GPU: the row kernels of a hooked layer (norm, unit, residual add) against fp64, and a decode step's
whole layer as one operator against the same layer taken part by part: the same bits, and the long
way kept wherever a part is replaced or the operator does not apply (more rows, other layouts and
types, gradients, autocast, a padded pool, untied values)."""

from __future__ import annotations

import pytest
import torch

from kv_skill_v2_amd import _lib, injector as xi
from kv_skill_v2_amd.depth import DEPTHS, injection_layers
from kv_skill_v2_amd.injector import LibraryInjector
from kv_skill_v2_amd.interface import ModelInterface
from kv_skill_v2_amd.library import Library
from tiny import TinyLM, close, oracle_forward, randomize, skill_rho

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.mark.parametrize("M,d", [(1, 4), (3, 20), (64, 1024), (5, 8192), (2, 8196), (7, 12288)])
def test_row_kernels(dev, M, d):
    say("hook rows", dict(M=M, d=d))
    g = torch.Generator().manual_seed(d)
    h, dl = torch.randn(M, d + 4, generator=g)[:, :d].to(dev), 0.1 * torch.randn(M, d, generator=g).to(dev)
    h[0, 0] = 0.0
    L, st = _lib.lib(), _lib.stream_handle(dev)
    hn, ratio = torch.empty(M, d, device=dev), torch.empty(M, device=dev)
    _lib.check(L.xenc_hook_norm(h.data_ptr(), h.stride(0), M, d, 1e-6, hn.data_ptr(), st), "norm")
    h64 = h.double()
    want = h64 * torch.rsqrt(h64.square().mean(-1, keepdim=True) + 1e-6)
    # fp32: one sum of d squares (relative error < 2^-24 (d / 1024 + 16)) under a square root, two roundings
    tol = 2.0 ** -24 * (d / 1024 + 20)
    assert float(((hn.double() - want).abs() / want.abs().clamp_min(1e-30)).max()) < tol
    q = dl.clone()
    _lib.check(L.xenc_hook_unit(q.data_ptr(), q.stride(0), M, d, 1e-6, st), "unit")
    want = dl.double() / (dl.double().norm(dim=-1, keepdim=True) + 1e-6)
    assert float(((q.double() - want).abs() / want.abs().clamp_min(1e-30)).max()) < tol
    out = torch.empty(M, d, device=dev)
    _lib.check(L.xenc_hook_add(h.data_ptr(), h.stride(0), dl.data_ptr(), d, M, d, out.data_ptr(), ratio.data_ptr(), st),
               "add")
    assert torch.equal(out, h + dl)
    want = dl.double().norm(dim=-1) / (h64.norm(dim=-1) + 1e-6)
    assert float(((ratio.double() - want).abs() / want).max()) < 2 * tol
    assert L.xenc_hook_norm(h.data_ptr(), d + 2, M, d, 1e-6, hn.data_ptr(), st) == -1
    assert L.xenc_hook_unit(q.data_ptr() + 4, d, M, d, 1e-6, st) == -3


def _setup(dev, d=48, d_s=64, ns=(5, 70, 3), top_k=2, cls=LibraryInjector):
    reader = TinyLM(d=d, n_layers=8).to(dev)
    layers = injection_layers(reader, DEPTHS)
    itf = ModelInterface(d, d_s, layers).to(dev)
    randomize(itf, seed=3)
    inj = cls(reader, itf, top_k=top_k)
    lib = Library([skill_rho(d_s, DEPTHS, n=n, seed=i) for i, n in enumerate(ns)], layers, DEPTHS)
    inj.load_library(lib)
    tensors = {li: (lib.K[li].cpu(), lib.mask[li].cpu(), lib.S[li].cpu()) for li in lib.layers}
    return reader, inj, tensors


def _count(monkeypatch):
    calls = []
    real = torch.ops.xenc.hook_layer
    monkeypatch.setattr(torch.ops.xenc, "hook_layer", lambda *a: calls.append(1) or real(*a))
    return calls


class _PartByPart(LibraryInjector):
    def _pos_mask(self, h):     # a replaced part: the long way
        return None


@pytest.mark.parametrize("rows", [1, 4, 8, 9])
def test_whole_layer_equals_its_parts(dev, monkeypatch, rows):
    say("hook layer", dict(rows=rows))
    calls = _count(monkeypatch)
    x = torch.randn(rows, 1, 48, generator=torch.Generator().manual_seed(rows)).to(dev)
    outs = []
    for cls in (LibraryInjector, _PartByPart):
        reader, inj, tensors = _setup(dev, cls=cls)
        n0 = len(calls)
        with torch.no_grad():
            outs.append((reader(x), inj.last_route, [float(m) for m in inj.mag_terms]))
        used = len(calls) - n0
        assert used == (len(inj.itf.inject_layers) if cls is LibraryInjector and rows <= 8 else 0)
        if cls is LibraryInjector:
            ref, _ = oracle_forward(reader, x.cpu(), inj.itf, tensors, top_k=2)
            assert close(outs[0][0], ref)[0]
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]) and outs[0][2] == outs[1][2]
    assert outs[0][1].shape == (rows, 1, 3)


def test_whole_layer_is_left_out(dev, monkeypatch):
    say("hook layer guards")
    calls = _count(monkeypatch)
    reader, inj, _ = _setup(dev)
    x = torch.randn(4, 1, 48, generator=torch.Generator().manual_seed(1)).to(dev)
    with torch.no_grad():
        want = reader(x)
    n0 = len(calls)
    assert n0 > 0
    reader(x)                                                    # grad mode: the autograd path
    assert len(inj.route_terms) > 0
    inj.route_terms.clear()
    with torch.no_grad():
        h = x.transpose(0, 2).contiguous().transpose(0, 2)      # hidden rows strided by layout
        assert inj._whole_layer(h, inj.itf.inject_layers[0]) is None or h.is_contiguous()
        assert inj._whole_layer(x.half(), inj.itf.inject_layers[0]) is None
        assert inj._whole_layer(x[..., :46], inj.itf.inject_layers[0]) is None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert inj._whole_layer(x, inj.itf.inject_layers[0]) is None
        inj._branch = lambda h, li: torch.zeros_like(h)          # an instance's own branch is called
        assert inj._whole_layer(x, inj.itf.inject_layers[0]) is None
        del inj._branch
        inj.record_attn = True
        assert inj._whole_layer(x, inj.itf.inject_layers[0]) is None
        inj.record_attn = False
    assert len(calls) == n0
    with torch.no_grad():
        assert torch.equal(reader(x), want)
    padded, inj2, t2 = _setup(dev, d_s=24)                      # a pool padded to 64 columns
    with torch.no_grad():
        n1 = len(calls)
        ref, _ = oracle_forward(padded, x.cpu(), inj2.itf, t2, top_k=2)
        assert close(padded(x), ref)[0]
        assert len(calls) == n1
    with pytest.raises(ValueError):
        torch.ops.xenc.hook_layer(x[:, 0], [], None, None, [], [], [], True, torch.empty(1, dtype=torch.uint8, device=dev))
    assert xi._rows_fp32(x.cpu()) is None
