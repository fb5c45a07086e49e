"""The Python launch layer's K-split workspaces (rocknpu_amd/hip.py) on the
CPU: which buffers stay alive and how large they grow. Host logic only, with
torch's stream calls and the device allocation replaced."""
import types
import weakref

import pytest
import torch

from rocknpu_amd import hip

CASES = [("_workspaces", hip.workspace_for, 1 << 20), ("_gemv_workspaces", hip.gemv_workspace_for, 1 << 16)]


@pytest.fixture
def on_cpu(monkeypatch):
    """hip.py with host tensors for its workspaces; .stream is the current
    stream's handle, .capturing whether it is being captured."""
    s = types.SimpleNamespace(stream=7, capturing=False)
    zeros = torch.zeros
    monkeypatch.setattr(hip.torch, "zeros", lambda n, dtype, device: zeros(n, dtype=dtype))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *_: types.SimpleNamespace(cuda_stream=s.stream))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: s.capturing)
    for name, _, _ in CASES:
        monkeypatch.setattr(hip, name, {})
    monkeypatch.setattr(hip, "_retired", [])
    return s


@pytest.mark.parametrize("name,get,least", CASES)
def test_a_replaced_workspace_stays_alive(on_cpu, name, get, least):
    """A graph captured with a stream's workspace holds its raw address: the
    buffer must outlive the larger one that a later call on the stream makes."""
    dev = torch.device("cuda", 0)
    sizes = [least, least + 1, 5 * least, 5 * least, 23 * least]
    seen = []
    for n in sizes:
        on_cpu.capturing = False
        ws = get(dev, n)  # the eager call before a capture
        on_cpu.capturing = True
        assert get(dev, n) is ws and ws.numel() >= n and not ws.any()
        seen.append((ws.data_ptr(), weakref.ref(ws)))
        del ws
    assert all(ref() is not None and ref().data_ptr() == at for at, ref in seen)
    # growing by doubling keeps what was replaced smaller than what is in use
    kept = {ref().data_ptr(): ref().numel() for _, ref in seen}
    current = getattr(hip, name)[(0, 7)].numel()
    assert sum(kept.values()) - current < current


@pytest.mark.parametrize("name,get,least", CASES)
def test_streams_keep_workspaces_of_their_own(on_cpu, name, get, least):
    dev = torch.device("cuda", 0)
    a = get(dev, 4 * least)
    on_cpu.stream = 8
    b = get(dev, least)
    assert b is not a and b.numel() == least
    on_cpu.stream = 7
    assert get(dev, least) is a and len(getattr(hip, name)) == 2


def _aligned(nbytes):
    t = torch.zeros(nbytes + 256, dtype=torch.uint8)
    return t[-t.data_ptr() % 256:][:nbytes]


RAGGED = [(4, 2, 8192, [8192, 1000, 1000]), (4, 2, 8192, [5000, 5000]), (6, 8, 8192, [2728, 2728]),
          (6, 5, 5632, [1000, 1048]), (4, 3, 5632, [17, 17, 17]), (6, 1, 14336, [1, 1, 1, 1])]


@pytest.mark.skipif(torch.cuda.is_available(), reason="host buffers: without a GPU no launch can read them")
@pytest.mark.parametrize("kind,m,k,ns", RAGGED)
def test_ragged_groups_fit_the_workspace_asked_for(monkeypatch, kind, m, k, ns):
    """Groups whose members end inside a 16-row tile: the launch takes the
    workspace that the module makes for it, and one of the size the query
    gives for the members' rows summed; one byte less is refused. Without a
    GPU an accepted call ends as a failed launch (-3), a refused one as an
    invalid argument (-1)."""
    made = []

    def exact(device, nbytes):
        made.append(_aligned(nbytes))
        return made[-1]

    monkeypatch.setattr(hip, "_stream", lambda: None)
    monkeypatch.setattr(hip, "gemv_workspace_for", exact)
    tiled = [torch.empty(hip.gemv_tiled_bytes(kind, k, n), dtype=torch.uint8) for n in ns]
    x = torch.zeros(m, k)
    summed = hip.gemv_tiled_workspace_bytes(kind, m, k, sum(ns))
    assert summed > 0
    for workspace, status in ((None, -3), (_aligned(summed), -3), (_aligned(summed - 1), -1)):
        with pytest.raises(hip.LaunchError, match=f"status {status}$"):
            hip.gemv_q_f32_tiled(kind, tiled, k, ns, x, workspace=workspace)
    # what the module makes holds every tile of one launch: no falling back to one a member
    assert made[0].numel() == hip.gemv_tiled_workspace_bytes(kind, m, k, sum(-(-n // 16) * 16 for n in ns))
