"""Block admission rounds under a small budget (host logic only): a round's own batches stay
resident until its solves have run; blocks that do not fit beside them follow."""
import collections
import queue

from femorax_amd import serve


class Handle:
    def __init__(self, n):
        self.n, self.open = n, True

    def close(self):
        self.open = False

    free = close

    def zero(self):
        assert self.open


class Mesh:
    def __init__(self, n):
        self.neq = n

    def params_for(self, model):
        return None


def test_a_round_does_not_evict_its_own_blocks(monkeypatch):
    calls = []

    def cg_many(ctx, batches, bs, xs, rtol):
        assert all(h.open for h in (*batches, *bs, *xs))
        calls.append([b.n for b in batches])
        return [dict(converged=1, iterations=b.n) for b in batches]

    class Array(Handle):
        def __init__(self, ctx, n):
            super().__init__(n)

        @classmethod
        def from_host(cls, ctx, a):
            return cls(ctx, a)

    monkeypatch.setattr(serve.core, "Batch", lambda ctx, mesh, params, **kw: Handle(mesh.neq))
    monkeypatch.setattr(serve.core, "DeviceArray", Array)
    monkeypatch.setattr(serve.core, "cg_many", cg_many)
    monkeypatch.setattr(serve, "_block_bytes", lambda neq, mixed: 10)

    class Problems:
        def get(self, n):
            return {}, Mesh(n), n

    class Request:
        def __init__(self, n):
            self.n, self.result = n, None

    w = serve.BlockWorker.__new__(serve.BlockWorker)
    w.problems, w.mixed, w.rtol, w.keep_x, w.used = Problems(), False, 1e-8, False, 0
    resident = collections.OrderedDict()
    for budget, groups in ((25, [[4, 5], [6, 7]]), (5, [[4], [5], [6], [7]]), (100, [[4, 5, 6, 7]])):
        w.budget = budget
        calls.clear()
        rs = [Request(n) for n in (4, 5, 6, 7)]
        w._solve_round(None, resident, rs)
        assert calls == groups
        assert [r.result["iterations"] for r in rs] == [4, 5, 6, 7]


def test_a_failed_part_leaves_the_solved_results(monkeypatch):
    """A round of two parts whose second solve fails: the first part's requests keep their results."""
    def cg_many(ctx, batches, bs, xs, rtol):
        if any(b.n >= 6 for b in batches):
            raise RuntimeError("no room")
        return [dict(converged=1, iterations=b.n) for b in batches]

    class Array(Handle):
        def __init__(self, ctx, n):
            super().__init__(n)

        @classmethod
        def from_host(cls, ctx, a):
            return cls(ctx, a)

    class Problems:
        def get(self, n):
            return {}, Mesh(n), n

    class Request:
        def __init__(self, n):
            self.n, self.result, self.start, self.end = n, {"of": "an earlier run"}, None, None

    monkeypatch.setattr(serve.core, "Context", lambda device: Handle(device))
    monkeypatch.setattr(serve.core, "Batch", lambda ctx, mesh, params, **kw: Handle(mesh.neq))
    monkeypatch.setattr(serve.core, "DeviceArray", Array)
    monkeypatch.setattr(serve.core, "cg_many", cg_many)
    monkeypatch.setattr(serve, "_block_bytes", lambda neq, mixed: 10)
    inbox, done = queue.Queue(), queue.Queue()
    rs = [Request(n) for n in (4, 5, 6, 7)]
    for r in (*rs, None):
        inbox.put(r)
    serve.BlockWorker(0, Problems(), inbox, done, budget=25, mixed=False, rounds=True).run()
    assert [done.get_nowait() for _ in rs] == rs
    assert [r.result.get("iterations") for r in rs] == [4, 5, None, None]
    assert ["error" in r.result for r in rs] == [False, False, True, True]
