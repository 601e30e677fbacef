"""A solve in hipGraphs takes its turn among the operators' other calls: projections from another thread and
stream during its replays, and a second solve, give the bits that they give alone, and so does the solve."""
import threading

import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["operator", "batch", "separate"])
def test_projections_beside_a_graph_solve(kind):
    import torch

    import elsa_amd as E

    g = oracle.circle_geometry(3, (64, 64, 64), 90, 360, 6400.0, 320.0, det=(96, 96))
    # operators of one kind run fused passes; the batch of two kinds runs its operators one by one
    classes = {"operator": [E.JosephsMethodCUDA], "batch": [E.JosephsMethodCUDA] * 2,
               "separate": [E.JosephsMethodCUDA, E.SiddonsMethodCUDA]}[kind]
    ops = [c(*geom_to_descriptors(g)) for c in classes]
    gen = torch.Generator(device="cuda").manual_seed(1)
    bs = [torch.rand(g.sino_shape, device="cuda", generator=gen) for _ in ops]
    if kind == "operator":
        A, b = ops[0], bs[0]
    else:
        A = E.ProjectorBatch(ops)
        assert A.fused == (kind == "batch")
        b = A.pack(bs, adjoint_space=True)
    alone = E.CGLS(A, b, tol=0.0, graph=True).solve(30).clone()
    # data of different sizes, so that one call's scale would not do for another
    xs = [torch.rand(g.vol_shape, device="cuda", generator=gen) * 10.0 ** k for k in range(4)]
    ys = [torch.rand(g.sino_shape, device="cuda", generator=gen) * 10.0 ** k for k in range(4)]
    ref = [[(op.apply(x).clone(), op.applyAdjoint(y).clone()) for x, y in zip(xs, ys)] for op in ops]
    torch.cuda.synchronize()
    done, found = threading.Event(), []

    def solves():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(3):
                    found.append(E.CGLS(A, b, tol=0.0, graph=True).solve(30))
                torch.cuda.synchronize()
        finally:
            done.set()

    threads = [threading.Thread(target=solves) for _ in range(2)]
    for t in threads:
        t.start()
    stream, outs = torch.cuda.Stream(), []
    with torch.cuda.stream(stream):
        for k in range(200):
            op, i = k % len(ops), k % len(xs)
            outs.append((op, i, ops[op].apply(xs[i]), ops[op].applyAdjoint(ys[i])))
            if k >= 20 and done.is_set():
                break
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert len(found) == 6
    for x in found:
        assert torch.equal(x, alone)
    for op, i, fwd, adj in outs:
        assert torch.equal(fwd, ref[op][i][0]) and torch.equal(adj, ref[op][i][1]), (op, i)
