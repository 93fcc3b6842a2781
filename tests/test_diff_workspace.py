"""The workspace of the differentiable sums is memory that a call can do
without: where it cannot be had, the calls go on with a null one."""
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from amuse_amd import diff  # noqa: E402

LIMIT = 1 << 20


class Entries:
    """Stands for the entry points of one dtype; notes their workspaces."""
    size = 4

    def __init__(self, values):
        self.values = values
        self.seen = []

    def forces_values(self, n):
        return self.values

    adjoint_values = forces_values

    def forces_ws(self, n, *args):
        self.seen.append(args[6:8])
        return 0

    def adjoint_ws(self, n, *args):
        self.seen.append(args[9:11])
        return 0

    def _step(self, *args):
        return 0

    step_predict = step_correct = step_correct_t = step_predict_t = _step


@pytest.fixture
def calls(monkeypatch):
    """Entry points as diff binds them, and an allocator of LIMIT values."""
    new_empty = torch.Tensor.new_empty

    def limited(t, size, *args, **kw):
        if isinstance(size, int) and size > LIMIT:
            raise torch.OutOfMemoryError("no room")
        return new_empty(t, size, *args, **kw)

    def with_values(values):
        k = Entries(values)
        monkeypatch.setattr(diff, "_entries", lambda dtype: k)
        monkeypatch.setattr(diff, "_stream", lambda t: 0)
        monkeypatch.setattr(diff, "_check", lambda t, name: t)
        monkeypatch.setattr(torch.Tensor, "new_empty", limited)
        return k
    return with_values


@pytest.mark.parametrize("n,values", [(70, 0), (70, 1000), (70, LIMIT + 1), (0, 0)])
def test_workspace_is_optional(calls, n, values):
    k = calls(values)
    x, v, g = (torch.zeros(n, 3) for _ in range(3))
    m = torch.zeros(n)
    ctx = SimpleNamespace(save_for_backward=lambda *t: None)
    diff.PairForce.forward(ctx, x, v, m, 1e-4)
    diff.HermiteStep.forward(ctx, x, v, x, v, m, 0.1, 1e-4)
    ctx.saved_tensors = (x, v, m)
    diff.PairForce.backward(ctx, g, g)
    diff.HermiteStep.backward(ctx, g, g, g, g)
    assert len(k.seen) == 4
    for ws, size in k.seen:
        if values == 1000:
            assert ws and size == 4 * values
        else:
            assert not ws and size == 0


def test_no_room_for_the_results_is_an_error(calls):
    k = calls(8)
    with pytest.raises(torch.OutOfMemoryError):
        diff._room(torch.zeros(3), LIMIT + 1, k.values)
