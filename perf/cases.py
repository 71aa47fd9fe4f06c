"""The work that programs have this package do, as cases that can be timed and compared.

A case is one call (or one training step) through the package's public entry points, at a size
that a program meets: the smallest calls, where latency and launches count, ordinary ones, and
the largest.  Each kind of case below says what in real use it stands for; `listed` gives the
sizes of the package's own workloads and of ordinary programs, `draw` further ones of the same
ranges.  Inputs are synthetic: unit-norm fp16 slot rows, ragged last chunks, shuffled page tables
and queries that point at one slot of their library, so that the softmax over a chunk is neither
flat nor one-hot.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from kv_skill_v2_amd import ops
from kv_skill_v2_amd.decode_reader import DecodeReader
from kv_skill_v2_amd.injector import LibraryInjector
from kv_skill_v2_amd.interface import ModelInterface
from kv_skill_v2_amd.library import Library
from kv_skill_v2_amd.multi_depth import MultiDepthDecode

DEV = "cuda"
READ_TEMP, ROUTE_TEMP = 12.0, 10.0
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


# ------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # One sequence's decode step over one document of 8,192 slots: the smallest call.
        dict(name="single_decode", kind="decode", rows=1, lo=16, hi=16, slots=512, d=2048, top_k=4),
        # A serving batch: 64 sequences, each with a library of its own of 8 to 64 chunks.
        dict(name="batched_decode", kind="decode", rows=64, lo=8, hi=64, slots=512, d=2048, top_k=8),
        # A decode step whose selector spreads the read over 2 of 8 depths for each of 32 tokens.
        dict(name="multi_depth", kind="multi_depth", rows=32, depths=8, chunks=64, slots=512, d=2560, d_r=5120,
             k_sel=2, top_k=8),
        # One hooked decode step of a reader: 4 tokens, 4 injection layers.
        dict(name="injector_step", kind="injector", rows=4, depths=4, chunks=16, slots=512, d=2560, d_r=5120, top_k=4),
        # Registration training: 4 documents x 2,048 tokens, every chunk read, forward and gradient.
        dict(name="train_4x2048", kind="train", libs=4, rows=2048, ragged=False, lo=32, hi=32, slots=512, d=2048,
             top_k=0, softmax=True),
        # The same step at its smallest: 64 tokens, 4 chunks, top-2 routing.
        dict(name="train_tiny", kind="train", libs=1, rows=64, ragged=False, lo=4, hi=4, slots=512, d=256, top_k=2,
             softmax=True),
        # A user's question (a prompt) read against one document with routing, no gradient.
        dict(name="prompt", kind="prompt", rows=333, chunks=16, slots=512, d=2048, top_k=4, softmax=True),
        # The serving plugin's joint read: 32 requests, each over its own 16k-row operator.
        dict(name="op_b_batch", kind="op_b", rows=32, hq=16, hkv=4, d=256, block=16, keys=16384, own=64, even=True,
             chunk=0, dtype="bf16"),
        # A few requests with documents of different lengths, the reader's default split.
        dict(name="op_b_ragged", kind="op_b", rows=5, hq=32, hkv=8, d=128, block=16, keys=5000, own=77, even=False,
             chunk=1024, dtype="fp16"),
        # The multi-document read of one decode token, and of a question's tokens.
        dict(name="d18_decode", kind="d18", rows=1, docs=6, keys=2048, own=512, hkv=2, g=8, hd=256, skip=16, top_k=0,
             dtype="bf16"),
        dict(name="d18_prompt", kind="d18", rows=130, docs=4, keys=1500, own=0, hkv=2, g=8, hd=256, skip=16, top_k=2,
             dtype="bf16"),
        # Slot selection for a question (64 of 8,192 slots), then its tokens' read of those slots.
        dict(name="slot_topk", kind="slot_topk", rows=200, chunks=16, slots=512, d=2048, k=64, n_q=16, n_kv=4, hd=256),
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    def mult(lo, hi, m):
        return max(lo, log(lo, hi) // m * m)

    kind = rng.choice(list(KINDS))
    if kind == "decode":      # pages of any length, widths in steps of 8
        hi = log(2, 64)
        return dict(kind=kind, rows=log(1, 64), lo=rng.randint(1, hi), hi=hi, slots=rng.randint(40, 512),
                    d=mult(128, 2048, 8), top_k=rng.randint(1, 8))
    if kind == "multi_depth":
        return dict(kind=kind, rows=log(1, 32), depths=rng.randint(3, 8), chunks=log(4, 64), slots=rng.randint(64, 512),
                    d=mult(256, 2560, 64), d_r=mult(512, 5120, 64), k_sel=rng.randint(1, 2), top_k=rng.randint(1, 8))
    if kind == "injector":
        return dict(kind=kind, rows=log(1, 32), depths=rng.randint(2, 4), chunks=log(2, 32), slots=rng.randint(40, 512),
                    d=mult(256, 2560, 64), d_r=mult(512, 5120, 64), top_k=rng.randint(0, 4))
    if kind == "train":
        hi = log(2, 32)
        return dict(kind=kind, libs=rng.randint(1, 4), rows=log(64, 2048), ragged=rng.random() < 0.7,
                    lo=rng.randint(max(1, hi // 2), hi), hi=hi, slots=64 * rng.randint(1, 8), d=mult(256, 2048, 64),
                    top_k=rng.choice([0, 0, 2, 4]), softmax=rng.random() < 0.8)
    if kind == "prompt":
        return dict(kind=kind, rows=log(9, 2048), chunks=log(1, 64), slots=64 * rng.randint(1, 8),
                    d=mult(256, 2048, 64), top_k=rng.choice([0, 2, 4, 8]), softmax=rng.random() < 0.8)
    if kind == "op_b":
        hq, hkv, d = rng.choice([(16, 4, 256), (32, 8, 128), (8, 2, 128), (16, 2, 256), (28, 4, 128), (12, 2, 64)])
        return dict(kind=kind, rows=log(1, 32), hq=hq, hkv=hkv, d=d, block=rng.choice([16, 32]), keys=log(200, 16384),
                    own=log(1, 512), even=rng.random() < 0.3, chunk=rng.choice([0, 1024]),
                    dtype=rng.choice(["bf16", "fp16"]))
    if kind == "d18":
        return dict(kind=kind, rows=log(1, 256), docs=rng.randint(1, 8), keys=log(128, 4096),
                    own=rng.choice([0, log(1, 1024)]), hkv=rng.choice([1, 2, 4]), g=rng.choice([1, 4, 7, 8]),
                    hd=rng.choice([64, 128, 256]), skip=rng.choice([0, 16]), top_k=rng.choice([0, 2]),
                    dtype=rng.choice(["bf16", "fp16", "fp32"]))
    n_kv = rng.choice([1, 2, 4])
    return dict(kind=kind, rows=log(1, 1024), chunks=log(2, 64), slots=rng.randint(64, 512), d=mult(256, 2048, 64),
                k=log(8, 100), n_q=n_kv * rng.choice([1, 4, 8]), n_kv=n_kv, hd=rng.choice([64, 128, 256]))


# ------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _spread(n, lo, hi):
    """n whole numbers spread evenly over [lo, hi], the same for every seed."""
    return [hi if n == 1 else lo + round((hi - lo) * i / (n - 1)) for i in range(n)]


def _unit(x):
    return x / (torch.linalg.vector_norm(x, dim=-1, keepdim=True) + 1e-6)


def _pool(counts, slots, d, g):
    """Libraries of counts[i] chunks in one page pool: fp16 unit rows, the last chunk of each
    library cut short, pages in shuffled order, S = L2(mean of the valid rows)."""
    total = sum(counts)
    valid = []
    for i, c in enumerate(counts):
        valid += [slots] * (c - 1) + [max(1, slots - (37 * (i + 1)) % max(1, 3 * slots // 4))]
    page = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    nv = torch.tensor(valid, dtype=torch.int32, device=DEV)
    pages = torch.empty(total, slots, d, dtype=torch.float16, device=DEV)
    S = torch.empty(total, d, device=DEV)
    at = torch.arange(slots, device=DEV)
    for c0 in range(0, total, 64):
        c1 = min(total, c0 + 64)
        rows = _unit(torch.randn(c1 - c0, slots, d, generator=g, device=DEV)).half()
        rows *= (at < nv[c0:c1, None])[..., None]
        pages[page[c0:c1].long()] = rows
        S[c0:c1] = _unit(rows.float().sum(1) / nv[c0:c1, None])
    ptr = [0]
    for c in counts:
        ptr.append(ptr[-1] + c)
    return SimpleNamespace(pages=pages, page=page, valid=nv, ptr=torch.tensor(ptr, dtype=torch.int32, device=DEV), S=S,
                           counts=list(counts), valid_list=valid, first=ptr)


def _paged(p):
    return ops.PagedLibrary(p.pages, p.page, p.valid, p.ptr, p.S, n_chunks=p.counts, nvalid=p.valid_list)


def _queries(p, lib, n, g):
    """n unit rows, each half way to one valid slot of library `lib`."""
    first, count = p.first[lib], p.counts[lib]
    chunk = first + torch.randint(count, (n,), generator=g, device=DEV)
    slot = (torch.rand(n, generator=g, device=DEV) * p.valid[chunk]).long()
    near = p.pages[p.page[chunk].long(), slot].float()
    return _unit(0.5 * near + _unit(torch.randn(n, near.shape[1], generator=g, device=DEV)))


# ------------------------------------------------------------------------------------- 64 bits
def _route64(q, S, top_k):
    """(dense weights, kept chunks in rank order, their weights) of rows q over summaries S."""
    logit = q @ S.T * ROUTE_TEMP
    C = logit.shape[-1]
    k = C if top_k <= 0 or top_k >= C else top_k
    order = torch.sort(logit, dim=-1, descending=True, stable=True).indices[:, :k]
    if k == C:
        order = torch.arange(C, device=q.device).expand_as(logit)
    w = torch.zeros_like(logit).scatter(-1, order, torch.softmax(logit.gather(-1, order), -1))
    return w, order, w.gather(-1, order)


def _keys64(p, c):
    n = p.valid_list[c]
    return p.pages[int(p.page[c])][:n].double()


def _attend64(q, K, softmax=True):
    s = q @ K.T
    return torch.softmax(s * READ_TEMP, -1) if softmax else s / math.sqrt(K.shape[0])


def _read64(p, lib, q, w, softmax=True):
    """The read of rows q of one library: the sum over its chunks of w[:, c] times the chunk's read."""
    r = torch.zeros_like(q)
    for c in range(p.counts[lib]):
        rows = w[:, c].nonzero()[:, 0]
        if rows.numel():
            K = _keys64(p, p.first[lib] + c)
            r[rows] += w[rows, c, None] * (_attend64(q[rows], K, softmax) @ K)
    return r


# ------------------------------------------------------------------------------------- decode
# A decode step: every sequence's query row is routed over its own library's chunks and reads the
# kept ones (ops.route_read_decode).
class Decode:
    @staticmethod
    def inputs(c, seed):
        g = _gen(seed)
        p = _pool(_spread(c["rows"], c["lo"], c["hi"]), c["slots"], c["d"], g)
        return p, torch.cat([_queries(p, i, 1, g) for i in range(c["rows"])])

    @staticmethod
    def prepare(c, seed):
        p, q = Decode.inputs(c, seed)
        return SimpleNamespace(lib=_paged(p), q=q, group=torch.arange(c["rows"], dtype=torch.int32, device=DEV),
                               top_k=c["top_k"])

    @staticmethod
    def run(s):
        return ops.route_read_decode(s.q, s.lib, s.group, top_k=s.top_k, route_temp=ROUTE_TEMP, read_temp=READ_TEMP)

    @staticmethod
    def exact(c, seed):
        p, q = Decode.inputs(c, seed)
        kk = max(n if c["top_k"] >= n else c["top_k"] for n in p.counts)
        w = torch.zeros(c["rows"], max(p.counts), dtype=torch.float64, device=DEV)
        wsel = torch.zeros(c["rows"], kk, dtype=torch.float64, device=DEV)
        r = torch.zeros(c["rows"], c["d"], dtype=torch.float64, device=DEV)
        for i, n in enumerate(p.counts):
            a = p.first[i]
            wi, _, ws = _route64(q[i:i + 1].double(), p.S[a:a + n].double(), c["top_k"])
            w[i, :n], wsel[i, :ws.shape[1]] = wi[0], ws[0]
            r[i] = _read64(p, i, q[i:i + 1].double(), wi)[0]
        return w, None, wsel, r

    @staticmethod
    def work(c):
        counts = _spread(c["rows"], c["lo"], c["hi"])
        read = sum(min(c["top_k"], n) for n in counts) * c["slots"]
        return {"bytes": read * c["d"] * 2 + sum(counts) * c["d"] * 4 + c["rows"] * c["d"] * 8, "flops": 4 * read * c["d"]}


# ------------------------------------------------------------------------------------- multi-depth
# A decode step whose selector keeps k_sel of the candidate depths per token: selection, routing and
# read of the kept (token, depth) rows, write-back through each depth's map (MultiDepthDecode).
class MultiDepth:
    @staticmethod
    def inputs(c, seed):
        g = _gen(seed)
        L, B = c["depths"], c["rows"]
        p = _pool([c["chunks"]] * L, c["slots"], c["d"], g)
        q = torch.stack([_queries(p, i, B, g) for i in range(L)])
        rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
        h = rnd(B, c["d_r"])
        return SimpleNamespace(p=p, q=q, z=rnd(B, L), h=h, hn=h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6),
                               B=rnd(L, c["d_r"], c["d"]) / c["d"] ** 0.5, gate_w=rnd(c["d_r"]) / c["d_r"] ** 0.5,
                               gate_b=rnd(L) - 2.0, log_gain=0.1 * rnd(L), log_alpha=torch.full((), math.log(0.02), device=DEV))

    @staticmethod
    def prepare(c, seed):
        x = MultiDepth.inputs(c, seed)
        step = MultiDepthDecode(_paged(x.p), x.B, x.gate_w, x.gate_b, x.log_gain, x.log_alpha, k_sel=c["k_sel"],
                                top_k=c["top_k"], route_temp=ROUTE_TEMP, read_temp=READ_TEMP)
        return SimpleNamespace(step=step, x=x)

    @staticmethod
    def run(s):
        return s.step(s.x.z, s.x.q, s.x.h, s.x.hn)

    @staticmethod
    def exact(c, seed):
        x = MultiDepth.inputs(c, seed)
        p, k = x.p, c["k_sel"]
        top = torch.sort(x.z, dim=-1, descending=True, stable=True).indices[:, :k]
        wt = torch.softmax(x.z.double().gather(-1, top), -1)
        out = torch.zeros(c["rows"], c["d_r"], dtype=torch.float64, device=DEV)
        h, hn = x.h.double(), x.hn.double()
        for l in range(c["depths"]):
            tok, rank = (top == l).nonzero(as_tuple=True)
            if not tok.numel():
                continue
            q = x.q[l][tok].double()
            w, _, _ = _route64(q, p.S[p.first[l]:p.first[l + 1]].double(), c["top_k"])
            r = _read64(p, l, q, w)
            scale = torch.exp(x.log_gain[l].double()) * torch.sigmoid(hn[tok] @ x.gate_w.double() + x.gate_b[l].double())
            delta = scale[:, None] * (r @ x.B[l].double().T)
            rel = delta.norm(dim=-1, keepdim=True) / (h[tok].norm(dim=-1, keepdim=True) + 1e-6)
            out.index_add_(0, tok, wt[tok, rank, None] * delta / (rel + 1e-6) * torch.exp(x.log_alpha.double()))
        return out, None, None

    @staticmethod
    def work(c):
        rows, kk = c["rows"] * c["k_sel"], min(c["top_k"], c["chunks"])
        used = c["depths"] * (1 - (1 - c["k_sel"] / c["depths"]) ** c["rows"])           # depths some token keeps
        each = rows / used
        chunks = used * c["chunks"] * (1 - (1 - kk / c["chunks"]) ** each)               # chunks some row routes
        return {"bytes": chunks * c["slots"] * c["d"] * 2 + used * c["d"] * (c["chunks"] * 4 + c["d_r"] * 4)
                + rows * c["d"] * 4 + 3 * c["rows"] * c["d_r"] * 4,
                "flops": rows * (4 * kk * c["slots"] * c["d"] + 2 * c["d"] * c["d_r"])}


# ------------------------------------------------------------------------------------- injector
# One decode step (T = 1) of a reader with a LibraryInjector: at each injection layer the query map,
# routing and read of that layer's library, gate, gain and write map, added to the residual.  The
# reader's own blocks pass their input through: what is timed is the injector's share of a step.
class _Reader(torch.nn.Module):
    def __init__(self, n, d):
        super().__init__()
        self.model = torch.nn.Module()
        self.model.layers = torch.nn.ModuleList(torch.nn.Identity() for _ in range(n))
        self.config = SimpleNamespace(num_hidden_layers=n, hidden_size=d)
        self.device = torch.device(DEV, torch.cuda.current_device())

    def forward(self, x):
        for block in self.model.layers:
            x = block(x)
        return x


class Injector:
    @staticmethod
    def inputs(c, seed):
        g = _gen(seed)
        rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
        L = c["depths"]
        lengths = [c["slots"]] * (c["chunks"] - 1) + [max(1, 2 * c["slots"] // 3)]
        depths = [(i + 1) / L for i in range(L)]
        chunks = [{"K": {rho: _unit(rnd(n, c["d"])).half() for rho in depths}} for n in lengths]
        return SimpleNamespace(chunks=chunks, depths=depths, x=rnd(c["rows"], 1, c["d_r"]),
                               A=rnd(c["d"], c["d_r"]) / c["d_r"] ** 0.5, B=0.3 * rnd(c["d_r"], c["d"]),
                               gate_w=0.3 * rnd(c["d_r"]) / c["d_r"] ** 0.5, gate_b=rnd(L) - 1.0, log_gain=0.1 * rnd(L))

    @staticmethod
    def prepare(c, seed):
        x = Injector.inputs(c, seed)
        L = c["depths"]
        reader = _Reader(L, c["d_r"])
        itf = ModelInterface(c["d_r"], c["d"], list(range(L))).to(DEV).requires_grad_(False)
        with torch.no_grad():
            for name, v in (("A.weight", x.A), ("B.weight", x.B), ("gate_w", x.gate_w), ("gate_b", x.gate_b),
                            ("log_gain", x.log_gain)):
                itf.get_parameter(name).copy_(v)
        inj = LibraryInjector(reader, itf, read_temp=READ_TEMP, route_temp=ROUTE_TEMP, top_k=c["top_k"])
        inj.load_library(Library(x.chunks, list(range(L)), x.depths, device=DEV))
        return SimpleNamespace(reader=reader, inj=inj, x=x.x)

    @staticmethod
    def run(s):
        s.inj.mag_terms.clear()
        with torch.no_grad():
            return s.reader(s.x)

    @staticmethod
    def exact(c, seed):
        x = Injector.inputs(c, seed)
        h = x.x[:, 0].double()
        for i, rho in enumerate(x.depths):
            hn = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6)
            q = hn @ x.A.double().T
            q = q / (q.norm(dim=-1, keepdim=True) + 1e-6)
            Ks = [ch["K"][rho].double() for ch in x.chunks]
            m = torch.stack([K.mean(0) for K in Ks])
            w, _, _ = _route64(q, m / (m.norm(dim=-1, keepdim=True) + 1e-6), c["top_k"])
            r = sum(w[:, j, None] * (_attend64(q, K) @ K) for j, K in enumerate(Ks))
            gate = torch.sigmoid(hn @ x.gate_w.double() + x.gate_b[i].double())[:, None]
            h = h + torch.exp(x.log_gain[i].double()) * gate * (r @ x.B.double().T)
        return h[:, None]

    @staticmethod
    def work(c):
        C, L = c["chunks"], c["depths"]
        kk = min(c["top_k"] or C, C)
        touched = C * (1 - (1 - kk / C) ** c["rows"])
        # (the one A and one B are read again at each layer: a layer needs the one before it)
        return {"bytes": L * (touched * c["slots"] * c["d"] * 2 + C * c["d"] * 4 + 2 * c["d"] * c["d_r"] * 4)
                + 2 * c["rows"] * c["d_r"] * 4,
                "flops": L * c["rows"] * (4 * kk * c["slots"] * c["d"] + 4 * c["d"] * c["d_r"])}


# ------------------------------------------------------------------------------------- training
# A registration-training step of the read: forward with autograd, then the gradient of the query
# rows for an upstream gradient (ops.library_read and its backward).
class Train:
    @staticmethod
    def rows(c):
        return _spread(c["libs"], max(1, c["rows"] // 3), c["rows"]) if c["ragged"] else [c["rows"]] * c["libs"]

    @staticmethod
    def inputs(c, seed):
        g = _gen(seed)
        p = _pool(_spread(c["libs"], c["lo"], c["hi"]), c["slots"], c["d"], g)
        q = torch.cat([_queries(p, i, n, g) for i, n in enumerate(Train.rows(c))])
        return p, q, torch.randn(q.shape, generator=g, device=DEV)

    @staticmethod
    def prepare(c, seed):
        p, q, up = Train.inputs(c, seed)
        lib = _paged(p)
        return SimpleNamespace(lib=lib, plan=lib.plan(Train.rows(c)), q=q.requires_grad_(), up=up, top_k=c["top_k"],
                               softmax=c["softmax"])

    @staticmethod
    def run(s):
        r, w = ops.library_read(s.q, s.lib, s.plan, top_k=s.top_k, read_temp=READ_TEMP, route_temp=ROUTE_TEMP,
                                read_softmax=s.softmax)
        dq, = torch.autograd.grad(r, s.q, s.up)
        return r.detach(), w.detach(), dq

    @staticmethod
    def exact(c, seed):
        p, q, up = Train.inputs(c, seed)
        r, dq = torch.zeros_like(q, dtype=torch.float64), torch.zeros_like(q, dtype=torch.float64)
        wd = torch.zeros(q.shape[0], max(p.counts), dtype=torch.float64, device=DEV)
        at = 0
        for i, n in enumerate(Train.rows(c)):
            S = p.S[p.first[i]:p.first[i + 1]].double()
            for t in range(at, at + n, 512):
                e = slice(t, min(at + n, t + 512))
                x, u = q[e].double(), up[e].double()
                w, _, _ = _route64(x, S, c["top_k"])
                wd[e, :w.shape[1]] = w
                gam = torch.zeros_like(w)
                for j in range(p.counts[i]):
                    K = _keys64(p, p.first[i] + j)
                    a, v = _attend64(x, K, c["softmax"]), u @ K.T
                    r[e] += w[:, j, None] * (a @ K)
                    gam[:, j] = (a * v).sum(-1)
                    da = READ_TEMP * a * (v - gam[:, j, None]) if c["softmax"] else v / math.sqrt(K.shape[0])
                    dq[e] += w[:, j, None] * (da @ K)
                dq[e] += ROUTE_TEMP * (w * (gam - (w * gam).sum(-1, keepdim=True))) @ S
            at += n
        return r, wd, dq

    @staticmethod
    def work(c):
        pairs, chunks, rows = 0, 0, Train.rows(c)
        for n, C in zip(rows, _spread(c["libs"], c["lo"], c["hi"])):
            pairs += n * min(c["top_k"] or C, C) * c["slots"]
            chunks += C
        return {"bytes": chunks * c["slots"] * c["d"] * 2 + chunks * c["d"] * 4 + 4 * sum(rows) * c["d"] * 4,
                "flops": 8 * pairs * c["d"]}


# ------------------------------------------------------------------------------------- prompt
# The tokens of a prompt read against one document's library with no gradient: routing and the
# read at one injection layer (ops.branch_read).
class Prompt:
    @staticmethod
    def inputs(c, seed):
        g = _gen(seed)
        p = _pool([c["chunks"]], c["slots"], c["d"], g)
        return p, _queries(p, 0, c["rows"], g)

    @staticmethod
    def prepare(c, seed):
        p, q = Prompt.inputs(c, seed)
        return SimpleNamespace(lib=_paged(p), q=q, top_k=c["top_k"], softmax=c["softmax"])

    @staticmethod
    def run(s):
        return ops.branch_read(s.q, s.lib, s.top_k, READ_TEMP, ROUTE_TEMP, s.softmax)

    @staticmethod
    def exact(c, seed):
        p, q = Prompt.inputs(c, seed)
        w, _, _ = _route64(q.double(), p.S.double(), c["top_k"])
        return _read64(p, 0, q.double(), w, c["softmax"]), w

    @staticmethod
    def work(c):
        C, M = c["chunks"], c["rows"]
        kk = min(c["top_k"] or C, C)
        return {"bytes": C * (1 - (1 - kk / C) ** M) * c["slots"] * c["d"] * 2 + C * c["d"] * 4 + 2 * M * c["d"] * 4,
                "flops": 4 * M * kk * c["slots"] * c["d"]}


# ------------------------------------------------------------------------------------- joint decode read
# The serving plugin's decode step: each request's query heads over its document operator's rows
# and its own rows, both paged (DecodeReader).
class OpB:
    @staticmethod
    def lengths(c):
        n = [c["keys"]] * c["rows"] if c["even"] else _spread(c["rows"], max(1, c["keys"] // 5), c["keys"])
        return n, [c["own"]] * c["rows"] if c["even"] else _spread(c["rows"], 1, c["own"])

    @staticmethod
    def inputs(c, seed):
        g, dt = _gen(seed), DTYPES[c["dtype"]]
        parts = []
        for lens in OpB.lengths(c):
            width = -(-max(lens) // c["block"])
            blocks = width * c["rows"]
            bt = torch.randperm(blocks, generator=g, device=DEV).to(torch.int32).view(c["rows"], width)
            k, v = (torch.randn(blocks, c["block"], c["hkv"], c["d"], generator=g, device=DEV).to(dt) for _ in range(2))
            parts += [k, v, bt, torch.tensor(lens, dtype=torch.int32, device=DEV)]
        return torch.randn(c["rows"], c["hq"], c["d"], generator=g, device=DEV).to(dt), parts

    @staticmethod
    def prepare(c, seed):
        q, parts = OpB.inputs(c, seed)
        dec = DecodeReader(c["rows"], c["hq"], c["hkv"], c["d"], max_keys=c["keys"] + c["own"], device=DEV + ":0",
                           chunk=c["chunk"] or None)
        return SimpleNamespace(dec=dec, q=q, parts=parts, scale=c["d"] ** -0.5)

    @staticmethod
    def run(s):
        return s.dec(s.q, *s.parts, s.scale)

    @staticmethod
    def exact(c, seed):
        q, (ok, ov, obt, _, wk, wv, wbt, _) = OpB.inputs(c, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        hkv, d = c["hkv"], c["d"]
        for i, (n, m) in enumerate(zip(*OpB.lengths(c))):
            K = torch.cat([ok[obt[i].long()].view(-1, hkv, d)[:n], wk[wbt[i].long()].view(-1, hkv, d)[:m]]).double()
            V = torch.cat([ov[obt[i].long()].view(-1, hkv, d)[:n], wv[wbt[i].long()].view(-1, hkv, d)[:m]]).double()
            for h in range(c["hq"]):
                j = h // (c["hq"] // hkv)
                out[i, h] = torch.softmax(K[:, j] @ q[i, h].double() * d ** -0.5, 0) @ V[:, j]
        return out

    @staticmethod
    def work(c):
        keys = sum(sum(x) for x in OpB.lengths(c))
        return {"bytes": keys * c["hkv"] * c["d"] * 4 + c["rows"] * c["hq"] * c["d"] * 6,
                "flops": 4 * keys * c["hq"] * c["d"]}


# ------------------------------------------------------------------------------------- multi-document read
# The attention core of the multi-document read: rows of a reader over several documents'
# operators and their own rows, with routing over the documents (ops.d18_read).
class D18:
    @staticmethod
    def inputs(c, seed):
        g, dt, T = _gen(seed), DTYPES[c["dtype"]], c["rows"]
        rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
        docs = [tuple(rnd(c["hkv"], n, c["hd"]).to(dt) for _ in range(2))
                for n in _spread(c["docs"], max(1, 2 * c["keys"] // 3), c["keys"])]
        hq = c["hkv"] * c["g"]
        return SimpleNamespace(docs=docs, qd=rnd(c["docs"], hq, T, c["hd"]), qo=rnd(hq, T, c["hd"]),
                               ko=rnd(c["hkv"], c["own"] + T, c["hd"]), vo=rnd(c["hkv"], c["own"] + T, c["hd"]))

    @staticmethod
    def prepare(c, seed):
        x = D18.inputs(c, seed)
        x.docs = ops.d18_pack(x.docs)
        x.args = (c["hd"] ** -0.5, c["skip"], 1.0, c["top_k"])
        return x

    @staticmethod
    def run(s):
        return ops.d18_read(s.qd, s.qo, s.docs, s.ko, s.vo, *s.args)

    @staticmethod
    def exact(c, seed):
        x = D18.inputs(c, seed)
        T, P, G, hkv, hd = c["rows"], c["own"], c["g"], c["hkv"], c["hd"]
        D = c["docs"]
        f64 = dict(dtype=torch.float64, device=DEV)
        O, r, rmax = (torch.empty(hkv, G, T, D, *s, **f64) for s in ((hd,), (), ()))
        hide = torch.arange(P + T, device=DEV)[None] > P + torch.arange(T, device=DEV)[:, None]
        for h in range(hkv):
            ko, vo = x.ko[h].double(), x.vo[h].double()
            for e in range(G):
                so = (x.qo[h * G + e].double() @ ko.T * hd ** -0.5).masked_fill(hide, float("-inf"))
                for j, (K, V) in enumerate(x.docs):
                    s = x.qd[j, h * G + e].double() @ K[h].double().T * hd ** -0.5
                    a = torch.softmax(torch.cat([s, so], 1), -1)
                    O[h, e, :, j] = a[:, :s.shape[1]] @ V[h].double() + a[:, s.shape[1]:] @ vo
                    content = s[:, c["skip"]:] if s.shape[1] > c["skip"] else s
                    r[h, e, :, j], rmax[h, e, :, j] = torch.logsumexp(content, -1), content.amax(-1)
        logit = r
        if 0 < c["top_k"] < D:
            keep = torch.sort(r, dim=-1, descending=True, stable=True).indices[..., :c["top_k"]]
            logit = torch.full_like(r, float("-inf")).scatter(-1, keep, r.gather(-1, keep))
        w = torch.softmax(logit, -1)
        o = (w[..., None] * O).sum(-2).reshape(hkv * G, T, hd).transpose(0, 1).reshape(T, hkv * G * hd)
        return {"o": o, "w": w, "r": r, "rmax": rmax, "n": None}

    @staticmethod
    def work(c):
        T, hq = c["rows"], c["hkv"] * c["g"]
        keys = sum(_spread(c["docs"], max(1, 2 * c["keys"] // 3), c["keys"]))
        size = torch.empty(0, dtype=DTYPES[c["dtype"]]).element_size()
        own = c["own"] + T
        return {"bytes": keys * c["hkv"] * c["hd"] * 2 * size + own * c["hkv"] * c["hd"] * 8
                + (c["docs"] + 2) * T * hq * c["hd"] * 4 + 3 * hq * T * c["docs"] * 4,
                "flops": 4 * T * hq * c["hd"] * (keys + c["own"] + (T + 1) / 2)}


# ------------------------------------------------------------------------------------- slot selection
# The question-dependent read: the reader's attention query picks k slots of the library, which are
# gathered, and the question's rows read them (ops.select_scores, topk_rows, gather_library,
# read_rows: what one selection and one injection layer of TopKLibraryInjector run).
class SlotTopK:
    @staticmethod
    def inputs(c, seed):
        g = _gen(seed)
        p = _pool([c["chunks"]], c["slots"], c["d"], g)
        n = c["chunks"] * c["slots"]
        valid = (torch.arange(c["slots"], device=DEV)[None] < p.valid[:, None]).reshape(-1)
        return SimpleNamespace(p=p, q=_queries(p, 0, c["rows"], g), valid=valid,
                               qs=torch.randn(1, c["n_q"], c["hd"], generator=g, device=DEV),
                               keys=torch.randn(n, c["n_kv"], c["hd"], generator=g, device=DEV))

    @staticmethod
    def prepare(c, seed):
        x = SlotTopK.inputs(c, seed)
        one = torch.ones(c["rows"], 1, device=DEV)
        return SimpleNamespace(x=x, lib=_paged(x.p), k=min(c["k"], sum(x.p.valid_list)), slots=c["slots"], one=one,
                               first=torch.zeros(c["rows"], 1, dtype=torch.int32, device=DEV))

    @staticmethod
    def run(s):
        scores = ops.select_scores(s.x.qs, s.x.keys, s.x.valid)
        idx, top = ops.topk_rows(scores, s.k)
        sel = ops.gather_library(s.lib, idx, s.slots)
        with torch.no_grad():
            return scores, idx, top, ops.read_rows(s.x.q, s.one, s.first, s.one, sel, READ_TEMP)

    @staticmethod
    def exact(c, seed):
        x = SlotTopK.inputs(c, seed)
        q = x.qs[0].double().view(c["n_kv"], -1, c["hd"])
        s = torch.stack([x.keys[:, j].double() @ q[j].T for j in range(c["n_kv"])]).amax((0, 2))
        s = s.masked_fill(~x.valid, float("-inf"))
        k = min(c["k"], sum(x.p.valid_list))
        idx = torch.sort(s, dim=-1, descending=True, stable=True).indices[:k]
        K = x.p.pages[x.p.page.long()[idx // c["slots"]], idx % c["slots"]].double()
        return s[None], None, s[idx][None], _attend64(x.q.double(), K) @ K

    @staticmethod
    def work(c):
        n = c["chunks"] * c["slots"]
        k = min(c["k"], n)
        return {"bytes": n * c["n_kv"] * c["hd"] * 4 + n * 4 + k * c["d"] * 2 + 2 * c["rows"] * c["d"] * 4,
                "flops": 2 * n * c["n_q"] * c["hd"] + 4 * c["rows"] * k * c["d"]}


KINDS = {"decode": Decode, "multi_depth": MultiDepth, "injector": Injector, "train": Train, "prompt": Prompt,
         "op_b": OpB, "d18": D18, "slot_topk": SlotTopK}


# ------------------------------------------------------------------------------------- the entry points
def prepare(case, seed):
    s = KINDS[case["kind"]].prepare(case, seed)
    s.kind = case["kind"]
    return s


def run(state):
    return KINDS[state.kind].run(state)


def work(case):
    return KINDS[case["kind"]].work(case)


def exact(case, seed):
    with torch.no_grad():
        return KINDS[case["kind"]].exact(case, seed)


# About four times the error against `exact`: 3e-8 to 9e-7 where sums are in fp32, 2.2e-4 to 4e-4
# where the read's operands and probabilities are fp16.
FP32, FP16 = {"rel": 5e-6}, {"rel": 1.6e-3}
TOLERANCE = {"decode": FP32, "multi_depth": FP32, "injector": FP32, "op_b": FP32, "d18": FP32,
             "train": FP16, "prompt": FP16, "slot_topk": FP16}


def tolerance(case):
    return TOLERANCE[case["kind"]]
