"""GPU: the many-row D18 read (d18_tile_kernel: 64-column tiles of rows x query heads; one wave per
output in the merge) against the fp64 oracle, at the edges of its tiles: the first row count that
takes it, ragged columns (T * G not a multiple of 16 or 64), key splits shorter than a tile or
empty, every head dim and key type, the causal diagonal of the own rows, queries in other layouts,
and a non-finite own row that only later rows see.  The tolerance is the few-row test's: fp32 sums
of products kept to 2^-22."""

from __future__ import annotations

import pytest
import torch

from kv_skill_v2_amd import ops
from test_gpu_d18 import _case, _check, _oracle, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ns,T,P,Hkv,G,hd,dtype,skip,top_k,nsplit", [
    ([40], 16, 0, 1, 1, 32, torch.bfloat16, 0, 0, None),           # one 16-column group
    ([33, 31, 1, 64], 17, 3, 2, 3, 64, torch.float16, 5, 2, 3),    # tile edges, a one-key document
    ([100, 500], 33, 90, 1, 7, 128, torch.bfloat16, 16, 0, 5),     # ragged columns, own splits
    ([16, 17, 300], 21, 40, 2, 8, 256, torch.float32, 2, 2, 4),    # fp32 keys, 16-key tiles
    ([700], 40, 0, 4, 8, 256, torch.bfloat16, 600, 0, 2),          # skip inside a later split
    ([20, 9], 64, 600, 1, 4, 128, torch.float32, 0, 1, 32),        # most splits empty
    ([260] * 5, 130, 7, 2, 2, 64, torch.float16, 4, 3, None),
])
def test_d18_many_rows_match_oracle(dev, Ns, T, P, Hkv, G, hd, dtype, skip, top_k, nsplit):
    say("d18 rows", dict(Ns=Ns, T=T, P=P, Hkv=Hkv, G=G, hd=hd, dtype=str(dtype), skip=skip, top_k=top_k, nsplit=nsplit))
    qd, qo, docs, Kown, Vown = _case(Ns, T, P, Hkv, G, hd, dtype, sum(Ns) + T)
    scale = hd ** -0.5
    dd = [(K.to(dev), V.to(dev)) for K, V in docs]
    args = (dd, Kown.to(dev), Vown.to(dev), scale)
    kw = dict(skip=skip, beta=1.3, top_k=top_k, nsplit=nsplit)
    got = ops.d18_read(qd.to(dev), qo.to(dev), *args, **kw)
    _check(got, _oracle(qd, qo, docs, Kown, Vown, P, scale, skip=skip, beta=1.3, top_k=top_k), 2e-5)
    # rows outermost, and rows at an unaligned base: other layouts of the same queries, the same bits
    flip = lambda t: t.transpose(-2, -3).contiguous().transpose(-2, -3)  # noqa: E731
    shift = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)  # noqa: E731
    for f in (flip, shift):
        again = ops.d18_read(f(qd.to(dev)), f(qo.to(dev)), *args, **kw)
        assert all(torch.equal(got[k], again[k]) for k in ("o", "w", "r", "rmax", "n"))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_d18_rows_do_not_see_later_own_rows(dev, bad):
    """A non-finite value row of own row j reaches rows t >= j only, as in the few-row read."""
    say("d18 causal", dict(bad=bad))
    T, P, j = 40, 5, 23
    qd, qo, docs, Kown, Vown = _case([50, 70], T, P, 2, 2, 64, torch.bfloat16, 9)
    ref = _oracle(qd, qo, docs, Kown, Vown, P, 0.125)
    Vown[:, P + j, 7] = bad
    got = ops.d18_read(qd.to(dev), qo.to(dev), [(K.to(dev), V.to(dev)) for K, V in docs], Kown.to(dev), Vown.to(dev),
                       0.125)
    o, want = got["o"].double().cpu(), ref["o"]
    assert float((o[:j] - want[:j]).abs().max()) <= 2e-5
    hit = torch.zeros(64, dtype=torch.bool)
    hit[7] = True
    cols = hit.repeat(4)
    assert not torch.isfinite(o[j:][:, cols]).any() and torch.isfinite(o[j:][:, ~cols]).all()
    assert float((o[j:][:, ~cols] - want[j:][:, ~cols]).abs().max()) <= 2e-5
