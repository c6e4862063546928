"""Workspaces of the functional operators: which calls may share one."""
import threading

import numpy as np
import pytest
import torch

from deploy3d_amd import plugin

HOST = torch.device("cpu")


@pytest.fixture
def capturing(monkeypatch):
    state = dict(now=False)
    monkeypatch.setattr(plugin, "_capturing", lambda: state["now"])
    monkeypatch.setattr(plugin, "_scratch", plugin._Scratch())
    return state


def test_one_buffer_per_thread_and_stream(capturing):
    """Calls of one thread on one stream run in order and share a buffer that grows; other streams, and other threads on the
    same stream, whose launches interleave with them, have their own."""
    a = plugin.scratch(100, HOST, 1)
    assert plugin.scratch(60, HOST, 1) is a and plugin.scratch(100, HOST, 2) is not a
    b = plugin.scratch(101, HOST, 1)
    assert b is not a and b.numel() >= 101 and plugin.scratch(1, HOST, 1) is b
    seen = []
    t = threading.Thread(target=lambda: seen.append(plugin.scratch(10, HOST, 1)))
    t.start()
    t.join()
    assert seen[0].data_ptr() != b.data_ptr() and plugin.scratch(10, HOST, 1) is b


def test_a_captured_call_has_memory_of_its_own(capturing):
    """What a graph reads and writes on every replay is no buffer that other calls get, before or after."""
    before = plugin.scratch(100, HOST, 1)
    capturing["now"] = True
    captured = [plugin.scratch(n, HOST, 1) for n in (50, 100, 200)]
    capturing["now"] = False
    after = plugin.scratch(150, HOST, 1)
    at = [t.data_ptr() for t in [before, after] + captured]
    assert len(set(at)) == len(at)
    assert [t.numel() for t in captured] == [50, 100, 200] and plugin.scratch(150, HOST, 1) is after


@pytest.mark.gpu
def test_captured_calls_survive_larger_calls_on_the_same_stream(engine):
    """bev_densify and simple_mean_encoder captured on a stream, then calls on it that need far more workspace: every
    replay still gives the eager result, with the memory that used to back the smaller workspace handed out and
    overwritten in between."""
    g = torch.Generator(device="cuda").manual_seed(5)
    rows, grid = 500, (2, 24, 24)
    cells = torch.randperm(int(np.prod(grid)), generator=g, device="cuda")[:rows].sort().values
    coords = torch.stack([cells * 0, cells // 576, cells // 24 % 24, cells % 24], dim=1).int().contiguous()
    feats = torch.randn((rows, 16), generator=g, device="cuda").half()
    num = torch.tensor([rows], dtype=torch.int32, device="cuda")
    shape = torch.empty((1, 0) + grid, dtype=torch.int32, device="cuda")
    points = torch.rand((6000, 4), generator=g, device="cuda") * 2.4
    batch = torch.zeros(6000, dtype=torch.int32, device="cuda")
    config = torch.tensor([0, 0, 0, 0.1, 0.1, 1.2], device="cuda")
    big_shape = torch.empty((1, 0, 41, 800, 800), dtype=torch.int32, device="cuda")

    def small():
        return (engine.bev_densify(feats, coords, num, shape, 32),) + \
            engine.simple_mean_encoder(points, batch, config, shape, 2000)

    def large():
        return engine.spconv_index(coords, num, big_shape, (3, 3, 3), (2, 2, 2), (1, 1, 1), (1, 1, 1), (0, 0, 0),
                                   8 * rows, False, False)

    want = [t.clone() for t in small()]
    index = [t.clone() for t in large()[1:4]]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        small()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = small()
        for _ in range(4):
            got = large()
            filler = [torch.full((1 << 18,), 0x5a, dtype=torch.uint8, device="cuda") for _ in range(64)]
            for t in out:
                t.zero_()
            graph.replay()
            stream.synchronize()
            assert all(int((f != 0x5a).sum()) == 0 for f in filler)
            assert torch.equal(out[0], want[0]) and torch.equal(out[3], want[3])
            n = int(want[3].item())
            assert torch.equal(out[2][:n], want[2][:n])
            torch.testing.assert_close(out[1][:n], want[1][:n], rtol=1e-5, atol=1e-6)  # sums of atomics: any order
            assert torch.equal(got[1], index[0]) and torch.equal(got[3], index[2])
            del filler
