"""Calls captured into graphs: their replays come after, and beside, calls
that grow, trim and use the device's arena and drop its pass tables."""
import time

import numpy as np
import pytest

import eithot_amd as E
from gpu_graph import GLOBAL, RELAXED, THREAD_LOCAL, Graph
from gpu_util import assert_bitexact
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

# (dims, perm, elem): cut cycles with boundary cells, three passes with two
# tables, cycles of small cells, cycles beside a segmented tile, one pass
# without scratch or table, a whole pass, staged rows
CASES = [([2, 2048, 512, 2], [1, 3, 2, 4], 4), ([32, 48, 64, 40], [4, 2, 3, 1], 4),
         ([31, 279, 1213], [1, 3, 2], 4), ([7000, 501], [2, 1], 4), ([64, 64, 64], [3, 2, 1], 4),
         ([500, 500], [2, 1], 4), ([5, 2, 60001, 14], [3, 2, 1, 4], 2)]


class Case:
    def __init__(self, torch, dims, perm, elem, seed):
        self.dims, self.perm, self.elem = dims, perm, elem
        host = O.fill(int(np.prod(dims)), elem, seed, 1)
        self.want = O.permute(host, dims, [p - 1 for p in perm], elem)
        self.src = torch.from_numpy(host.copy()).to("cuda:0")
        self.buf = self.src.clone()

    def call(self, stream=None):
        E.transpose_ptr(self.buf.data_ptr(), self.dims, self.perm, self.elem, stream=stream)

    def check(self, what):
        assert_bitexact(self.buf.cpu().numpy(), self.want, f"{self.dims} {what}")


@pytest.mark.parametrize("dims,perm,elem", CASES)
def test_replays_after_and_beside_other_calls(torch_cuda, dims, perm, elem):
    torch = torch_cuda
    print(f"capture dims={dims} perm={perm} elem={elem}", flush=True)
    a, b = Case(torch, dims, perm, elem, 3), Case(torch, dims, perm, elem, 4)
    # the same passes on another tensor, and a call with more scratch
    c, big = Case(torch, dims, perm, elem, 5), Case(torch, [2, 3001, 5003, 2], [1, 3, 2, 4], 4, 6)
    torch.cuda.synchronize()
    E.lib().eithot_release()
    graphs = [Graph(a.call)]  # nothing is uploaded or allocated before
    for what in (b, big):
        what.call()
    graphs.append(Graph(b.call, GLOBAL))
    big.call()  # a larger arena; the others' tables make room
    E.lib().eithot_release()
    for k in range(3):
        for x, g in ((a, graphs[0]), (b, graphs[1])):
            x.buf.copy_(x.src)
            torch.cuda.synchronize()
            g.replay()
            g.wait()
            x.check(f"replay {k}")
        c.buf.copy_(c.src)
        big.buf.copy_(big.src)
        torch.cuda.synchronize()
        c.call()
        c.check(f"eager {k}")
        big.call()
        big.check(f"eager {k}")
    # two graphs and a plain call at once, several times over, with host work only
    side = torch.cuda.Stream()
    for k in range(5):
        for x in (a, b, c):
            x.buf.copy_(x.src)
        torch.cuda.synchronize()
        graphs[0].replay()
        graphs[1].replay()
        c.call(side.cuda_stream)
        torch.cuda.synchronize()
        for x, g in ((a, graphs[0]), (b, graphs[1])):
            g.wait()
            x.check(f"beside {k}")
        c.check(f"beside {k}")
    for g in graphs:
        g.close()


def test_graphs_give_their_memory_back(torch_cuda):
    # the memory lives as long as the executable graph, not the graph it was
    # made from, and goes back with the next call
    torch = torch_cuda
    x = Case(torch, [2, 4096, 1024, 2], [1, 3, 2, 4], 4, 7)
    alpha = 0.05
    _, need = E.plan_describe(x.dims, x.perm, x.elem, alpha=alpha)
    assert need > 0
    E.lib().eithot_release()
    small = Case(torch, [64, 64], [2, 1], 4, 8)
    graphs = [Graph(x.call, RELAXED) for _ in range(64)]
    assert E.last_peak_extra_bytes() >= need
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    graphs[0].replay()
    graphs[0].wait()
    x.check("replay")
    for g in graphs:
        g.close()
    for _ in range(100):  # graphs are torn down behind the calls that end them
        small.call()
        if torch.cuda.mem_get_info()[0] >= free + 32 * need:
            break
        time.sleep(0.05)
    assert torch.cuda.mem_get_info()[0] >= free + 32 * need


def test_capture_after_a_graph_has_ended(torch_cuda):
    # memory that an ended graph has let go of waits for a call outside the capture
    torch = torch_cuda
    x = Case(torch, CASES[0][0], CASES[0][1], 4, 14)
    for mode in (THREAD_LOCAL, GLOBAL, RELAXED):
        g = Graph(x.call, mode)
        g.close()
        torch.cuda.synchronize()
        time.sleep(0.3)
        g = Graph(x.call, mode)
        for k in range(3):
            x.buf.copy_(x.src)
            torch.cuda.synchronize()
            g.replay()
            g.wait()
            x.check(f"replay {k}")
        g.close()


def test_capture_mode_is_left_as_it_was(torch_cuda):
    # two calls in one capture, beside torch's own work
    torch = torch_cuda
    x, y = Case(torch, CASES[0][0], CASES[0][1], 4, 9), Case(torch, CASES[1][0], CASES[1][1], 4, 10)

    def both(stream):
        x.call(stream)
        y.call(stream)

    for mode in (THREAD_LOCAL, GLOBAL):
        g = Graph(both, mode)
        for k in range(3):
            x.buf.copy_(x.src)
            y.buf.copy_(y.src)
            torch.cuda.synchronize()
            g.replay()
            g.wait()
            x.check(f"replay {k}")
            y.check(f"replay {k}")
        g.close()


def test_batch_run_on_a_captured_stream(torch_cuda):
    # the batch's own graph is launched, not captured, and resident passes of
    # other streams, during the capture and after it, are no part of it either
    torch = torch_cuda
    a, b, c = (Case(torch, [1021, 523], [2, 1], 4, k) for k in (11, 12, 13))
    batch = E.Batch()
    batch.add(a.buf.data_ptr(), a.dims, a.perm, a.elem)
    batch.add(b.buf.data_ptr(), b.dims, b.perm, b.elem)
    batch.build()
    side = torch.cuda.Stream()
    c.call(side.cuda_stream)
    torch.cuda.synchronize()
    for k in range(3):
        for x in (a, b, c):
            x.buf.copy_(x.src)
        torch.cuda.synchronize()

        def calls(stream):
            batch.run(stream=stream, sync=False)
            c.call(side.cuda_stream)

        print(f"batch on a captured stream {k}", flush=True)
        g = Graph(calls)
        nodes = g.nodes
        g.close()
        torch.cuda.synchronize()
        assert nodes == 0
        c.check(f"during {k}")
        c.buf.copy_(c.src)
        torch.cuda.synchronize()
        c.call(None if k else side.cuda_stream)
        torch.cuda.synchronize()
        c.check(f"after {k}")
        a.buf.copy_(a.src)
        b.buf.copy_(b.src)
        torch.cuda.synchronize()
        batch.run()
        a.check(f"batch {k}")
        b.check(f"batch {k}")
