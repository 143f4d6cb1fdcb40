"""The workspace cache of the sampling and acceptance calls, on the CPU: one buffer per
(name, stream), buffers of captured calls apart and kept, the number of eager ones bounded."""
import torch

from batchspec_amd import _util

DEV = torch.device("cpu")


def test_workspaces_by_stream_and_capture(monkeypatch):
    capturing = [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    cache = {}

    def get(nbytes, stream, name="a"):
        return _util.workspace(DEV, nbytes, cache, name, stream)

    one = get(1000, 1)
    assert one.numel() >= 1000 and get(900, 1) is one
    two, other = get(1000, 2), get(1000, 1, "b")
    assert len({t.data_ptr() for t in (one, two, other)}) == 3
    assert get(5000, 1).numel() >= 5000 and get(1000, 2) is two
    assert not cache.get("__retired__")  # an outgrown eager buffer goes back
    capturing[0] = True
    cap = get(1000, 2)
    assert cap is not two and get(1000, 2) is cap
    grown = get(4000, 2)
    assert [t is c for t, c in zip(cache["__retired__"], (cap, grown))] == [True, True]
    capturing[0] = False
    assert get(1000, 2) is two
    for s in range(3, 3 + 2 * _util._MAX_WORKSPACES):
        get(256, s)
    assert sum(not k[3] for k in cache if k != "__retired__") <= _util._MAX_WORKSPACES
    capturing[0] = True
    assert get(4000, 2) is grown  # captured ones are not dropped
