"""The tuner's own runs do not try the cell tile, which the library accepts without effect: the tile it would pick
was the noise of equal runs."""
from iwf_mfree_gpu_3d_amd import _lib, autotune, serve


class Recorded:
    """Stands in for serve.Instance: keeps the choices it was made with."""
    choices = []

    def __init__(self, req, stream=0, choice=(), max_neighbours=0):
        Recorded.choices.append(tuple(choice))

    def advance(self, steps):
        return steps

    def finish(self):
        pass

    def release(self):
        pass


def test_own_runs_leave_the_tile_alone(monkeypatch):
    monkeypatch.setattr(serve, "Instance", Recorded)
    Recorded.choices = []
    reqs = serve.sweep_requests(count=12, batched=True, n_min=5e3, n_max=2e5, steps=(10, 10), seed=4)
    table = autotune.tune(reqs)
    assert Recorded.choices and all(c[2] == 0 for c in Recorded.choices)
    assert len(Recorded.choices) == len(table.choice) * (len(autotune.CANDIDATES) + len(autotune.BLOCKS))
    assert all(c[2] == 0 for c in table.choice.values())


def test_batches_are_not_run_for_nothing(monkeypatch):
    monkeypatch.setattr(serve, "Instance", Recorded)
    Recorded.choices = []
    reqs = serve.sweep_requests(count=12, batched=True, n_min=5e3, n_max=2e5, steps=(10, 10), seed=4)
    table = autotune.Table()
    table.batch_tile[_lib.MFG_FP64] = 8  # of a table made before
    assert autotune.tune_batched(reqs, table=table) is table
    assert not Recorded.choices and table.batch_tile == {_lib.MFG_FP64: 8}
