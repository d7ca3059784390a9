"""Preconditioner cycles and numeric updates recorded into a caller's graph, in every
order with eager ones. What a cycle reads beside the levels (the matrix of the coarse
end, the FP64 tiles, the fused sweep's values) has to be the current operator's
whichever of the two sides changed it; every result is compared in bits with a fresh
hierarchy that had the same values by eager calls alone.

The grids put the coarse end's matrix at level 0 and below other levels."""
import numpy as np
import pytest
import torch

from matrices import impes_like
from test_gpu_solver import to_dev

pytestmark = pytest.mark.gpu

GRIDS = [(12, 10, 10), (30, 24, 10)]
SIGMAS = (1.0, 1.3, 0.7, 1.1)


class Operators:
    """One pattern, several values, and what a fresh hierarchy makes of each."""

    def __init__(self, dims, kind, dev, graphs):
        self.dims, self.kind, self.graphs = dims, kind, graphs
        self.csr = [to_dev(impes_like(*dims, seed=8, sigma=s)[0], dev) for s in SIGMAS]
        self.st = [[torch.tensor(a, dtype=torch.float64, device=dev) for a in impes_like(*dims, seed=8, sigma=s)[1:]]
                   for s in SIGMAS]
        self.v = torch.tensor(np.random.default_rng(0).standard_normal(int(np.prod(dims))), device=dev)
        # the buffers that a recorded update reads
        self.now = [t.clone() for t in (self.st[0] if kind == "st7" else [self.csr[0][2]])]

    def load(self, q):
        for a, b in zip(self.now, self.st[q] if self.kind == "st7" else [self.csr[q][2]]):
            a.copy_(b)

    def setup(self):
        import impes_hip as H

        h = H.AmgHierarchy()
        if self.kind == "st7":
            h.setup_st7(self.dims, *self.st[0])
        else:
            h.setup_csr(*self.csr[0])
        h.set_graphs(self.graphs)
        return h

    def update(self, h):
        (h.update_st7 if self.kind == "st7" else h.update_csr)(*self.now)

    def results(self, h, precisions=(64, 32)):
        out = [h.precondition(self.v, precision=p) for p in precisions]
        return out + [h.vcycle(self.v, precision=p) for p in precisions]

    def reference(self, q, precisions=(64, 32)):
        h = self.setup()
        if q:
            self.load(q)
            self.update(h)
        return self.results(h, precisions)


def record(fn):
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    return g


def same(got, ref, what):
    torch.cuda.synchronize()
    for k, (a, b) in enumerate(zip(got, ref)):
        assert torch.equal(a, b), f"{what}: result {k} differs by {((a - b).norm() / b.norm()).item():.1e}"


params = pytest.mark.parametrize("precision", [64, 32])
grids = pytest.mark.parametrize("dims", GRIDS)
kinds = pytest.mark.parametrize("kind", ["csr", "st7"])
graphs_ = pytest.mark.parametrize("graphs", [True, False])  # eager cycles replayed from a graph of their own


@params
@grids
@kinds
@graphs_
def test_recorded_cycle_after_eager_updates(dev, dims, kind, precision, graphs):
    """Warm up, record, update eagerly, replay."""
    op = Operators(dims, kind, dev, graphs)
    refs = [op.reference(q, (precision,))[0] for q in range(3)]
    h = op.setup()
    z = h.precondition(op.v, precision=precision).clone()
    g = record(lambda: h.precondition(op.v, precision=precision, out=z))
    for q in (1, 2, 1):
        op.load(q)
        op.update(h)
        z.zero_()
        g.replay()
        same([z], [refs[q]], f"replay after update {q}")
        same([h.precondition(op.v, precision=precision)], [refs[q]], f"eager cycle after update {q}")


@params
@grids
@kinds
@graphs_
def test_recorded_update_with_eager_cycles(dev, dims, kind, precision, graphs):
    """Record an update, run an eager cycle, replay the update with new values, run an
    eager cycle; the update recorded with no cycle before it, after one of this
    precision, and after one of the other."""
    op = Operators(dims, kind, dev, graphs)
    refs = [op.reference(q) for q in range(4)]
    for warm in ((), (precision,), (96 - precision,)):
        h = op.setup()
        for p in warm:
            op.results(h, (p,))
        op.load(0)
        g = record(lambda: op.update(h))
        same(op.results(h), refs[0], f"warmed up {warm}: recorded, not run")
        for q in (1, 2):
            op.load(q)
            g.replay()
            same(op.results(h), refs[q], f"warmed up {warm}: replay {q}")
        op.load(3)
        op.update(h)
        same(op.results(h), refs[3], f"warmed up {warm}: eager update")
        op.load(1)
        g.replay()
        same(op.results(h), refs[1], f"warmed up {warm}: replay after it")


@params
@grids
@kinds
@graphs_
def test_recorded_cycle_as_the_first_call(dev, dims, kind, precision, graphs):
    """The first cycle after a setup goes into a graph: nothing is allocated in it, and
    it serves the operators of later updates."""
    op = Operators(dims, kind, dev, graphs)
    refs = [op.reference(q, (precision,))[0] for q in range(3)]
    h = op.setup()
    z = torch.empty_like(op.v)
    g = record(lambda: h.precondition(op.v, precision=precision, out=z))
    same([h.precondition(op.v, precision=precision)], [refs[0]], "eager cycle before the first replay")
    for q in (0, 1, 2):
        if q:
            op.load(q)
            op.update(h)
        z.zero_()
        g.replay()
        same([z], [refs[q]], f"replay {q}")
        same([h.precondition(op.v, precision=precision)], [refs[q]], f"eager cycle {q}")


@params
@grids
@kinds
@graphs_
def test_update_and_cycles_in_one_graph(dev, dims, kind, precision, graphs):
    """An update with two cycles behind it, recorded after a warm-up, and a graph of
    cycles alone beside it."""
    op = Operators(dims, kind, dev, graphs)
    refs = [op.reference(q, (precision,))[0] for q in range(3)]
    h = op.setup()
    z = [h.precondition(op.v, precision=precision).clone() for _ in range(3)]
    op.load(0)

    def body():
        op.update(h)
        for k in range(2):
            h.precondition(op.v, precision=precision, out=z[k])

    both = record(body)
    alone = record(lambda: h.precondition(op.v, precision=precision, out=z[2]))
    for q in (1, 2, 0, 1):
        op.load(q)
        for a in z:
            a.zero_()
        both.replay()
        alone.replay()
        same(z, [refs[q]] * 3, f"replay {q}")
        same([h.precondition(op.v, precision=precision)], [refs[q]], f"eager cycle {q}")
