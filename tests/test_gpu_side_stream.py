"""The second stream of a PairFormerStack's call: the library's own, for every stream of a caller, beside captures of
other threads, and given back."""
import threading

import pytest
import torch

from gpu_util import lib  # noqa: F401

import of3pair
from of3pair import functional as F3

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _stack(n, no_blocks=3):
    torch.manual_seed(31)
    m = of3pair.PairFormerStack(384, 128, 24, 16, 128, 32, 4, no_blocks=no_blocks)
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 2:
                p.normal_(std=p.shape[1] ** -0.5)
    m = m.to(DEV).to(torch.bfloat16).eval()
    s, z = torch.randn(1, n, 384, device=DEV).to(torch.bfloat16), torch.randn(1, n, n, 128, device=DEV).to(torch.bfloat16)
    m(s, z, None, None)
    want = m(s, z, None, None)  # the stack's own call
    torch.cuda.synchronize()
    return m, s, z, want


def test_side_stream_is_nobody_elses():
    lib()
    pool = {torch.cuda.Stream().cuda_stream for _ in range(64)}  # all of torch's pool, twice
    seen = set()
    for _ in range(20):
        caller = torch.cuda.Stream()
        with torch.cuda.stream(caller):
            seen.add(F3._side_stream(caller.device, caller.cuda_stream))
    assert seen.isdisjoint(pool | {None, 0, torch.cuda.default_stream().cuda_stream})
    assert len(seen) <= F3._MAX_SIDES


def test_stack_beside_a_capture_of_another_thread():
    """Another thread captures on one stream of torch's pool after the other while this one issues stack calls."""
    lib()
    m, s, z, want = _stack(40)
    x = torch.zeros(256, device=DEV)
    failed, graphs = [], []
    open_, done = threading.Event(), threading.Event()

    def capture():
        try:
            for _ in range(32):
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode="thread_local"):
                    x.add_(1.0)
                    open_.set()
                    done.wait(60)
                    done.clear()
                graphs.append(g)
        except Exception as e:  # noqa: BLE001
            failed.append(e)
        finally:
            open_.set()

    t = threading.Thread(target=capture)
    t.start()
    for _ in range(32):
        assert open_.wait(60)
        open_.clear()
        got = m(s, z, None, None)
        done.set()
    t.join(60)
    assert not t.is_alive() and not failed, failed
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    for g in graphs:
        g.replay()
    torch.cuda.synchronize()
    assert float(x[0]) == 32.0


def test_many_callers_streams_and_release():
    lib()
    m, s, z, want = _stack(33)
    callers = [torch.cuda.Stream() for _ in range(F3._MAX_SIDES + 4)]
    outs = []
    for c in callers:
        c.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(c):
            outs.append(m(s, z, None, None))
    torch.cuda.synchronize()
    assert all(torch.equal(a, want[0]) and torch.equal(b, want[1]) for a, b in outs)
    F3.release_workspaces()
    assert not F3._sides and not any(F3._own_streams.values())
    got = m(s, z, None, None)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_release_under_a_capture_keeps_the_streams():
    lib()
    m, s, z, want = _stack(33)
    x = torch.zeros(64, device=DEV)
    kept = {d: list(own) for d, own in F3._own_streams.items()}
    assert any(kept.values())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1.0)
        F3.release_workspaces()
    assert F3._own_streams == kept
    for _ in range(3):
        graph.replay()
        got = m(s, z, None, None)
        torch.cuda.synchronize()
    assert float(x[0]) == 3.0 and torch.equal(got[0], want[0])
    F3.release_workspaces()
    assert not any(F3._own_streams.values())
