"""Which pass a recorded schedule holds, on the CPU: the operators and the schedule are replaced by stand-ins that run on host
tensors (a convolution fills its output with one more than the mean of its input, so every result names the input it came
from), everything else - buffers, keys, what is recorded when and what is handed out - is the product's own code."""
import ctypes
import weakref

import numpy as np
import pytest
import torch

from deploy3d_amd import layers, onnx_graph, plugin, synth

GRID = (4, 8, 8)


def _apply(op, inputs, outputs):
    if op.name == "SPConvMM":
        outputs[0].fill_(float(inputs[0].float().mean()) + 1)


def _bytes_of(t):
    """The elements at a tensor's address in memory order: all that a step of a schedule knows of a tensor."""
    if t is None or t.numel() == 0:
        return None
    raw = (ctypes.c_byte * (t.numel() * t.element_size())).from_address(t.data_ptr())
    return torch.frombuffer(raw, dtype=t.dtype)


class _HostSchedule(plugin.Schedule):
    def __init__(self, lanes=1, **options):
        super().__init__(lanes=1, **options)  # one lane needs no device
        self._steps = []

    def add(self, op, in_descs, out_descs, inputs, outputs, workspace=None, lane=0, after=()):
        ins, outs = [_bytes_of(t) for t in inputs], [_bytes_of(t) for t in outputs]
        self._steps.append(lambda: _apply(op, ins, outs))
        return super().add(op, in_descs, out_descs, inputs, outputs, workspace, 0, after)

    def add_sum(self, a, b, out, lane=0, after=()):
        x, y, z = _bytes_of(a), _bytes_of(b), _bytes_of(out)
        self._steps.append(lambda: torch.add(x, y, out=z))
        return super().add_sum(a, b, out, 0, after)

    def add_cast(self, a, out, lane=0, after=()):
        x, y = _bytes_of(a), _bytes_of(out)
        self._steps.append(lambda: y.copy_(x))
        return super().add_cast(a, out, 0, after)

    def run(self, stream=None):
        for step in self._steps:
            step()


@pytest.fixture
def host(monkeypatch):
    """The stand-ins; ``host.capturing`` is what the stream is asked."""
    class State:
        capturing = False
    monkeypatch.setattr(plugin.Launch, "__call__", lambda self, ins, outs, ws, stream: _apply(self.plugin, ins, outs))
    monkeypatch.setattr(plugin.Plugin, "configure", lambda self, *a: None)
    monkeypatch.setattr(plugin.Plugin, "set_option", lambda self, *a: None)
    monkeypatch.setattr(plugin.Plugin, "link_rulebook", lambda self, *a: None)
    monkeypatch.setattr(plugin.Plugin, "enqueue", lambda self, ind, outd, ins, outs, ws=None, stream=None:
                        _apply(self, ins, outs))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: State.capturing)
    for module in (layers, onnx_graph):
        monkeypatch.setattr(module, "Schedule", _HostSchedule)
    monkeypatch.setattr(layers, "current_stream", lambda *a: 0)
    return State


def _specs(last_sum=False):
    p = dict(padding=(1, 1, 1))
    specs = [synth.layer("a", "s", True, (3, 3, 3), 4, 4, **p), synth.layer("b", "s", True, (3, 3, 3), 4, 4, **p)]
    if last_sum:
        specs.append(synth.layer("c", "s", True, (3, 3, 3), 4, 4, src="b+input", **p))
    return specs


def _net(specs, rows=16):
    weights = [synth.layer_weights(0, i, s) for i, s in enumerate(specs)]
    net = layers.SparseBackbone(specs, weights, [rows] * len(specs), dtype=torch.float32, device="cpu", overlap=False,
                                extensions=False)
    for lyr in net.layers:  # one lane of host tensors
        lyr.device = "cpu"
    return net


def _input(value, rows=16):
    coords = np.zeros((rows, 4), np.int32)
    return layers.make_input(coords, np.full((rows, 4), value, np.float32), GRID, dtype=torch.float32, device="cpu")


def _expect(y, value, convolutions=2):
    assert float(y.feats.min()) == float(y.feats.max()) == value + convolutions


@pytest.mark.parametrize("between", ["capture", "scheduled", "build", "steps"])
def test_a_recorded_pass_reads_its_own_input(host, between):
    """Warm up on ``a``, make one pass on other buffers in another way, go on with ``a``: every result is of its input."""
    net, a, static = _net(_specs()), _input(10.0), _input(500.0)
    _expect(net.forward(a), 10.0)
    _expect(net.forward(a), 10.0)
    if between == "capture":
        host.capturing = True
        _expect(net.forward(static), 500.0)
        host.capturing = False
    elif between == "scheduled":
        _expect(net.forward_scheduled(static), 500.0)
    elif between == "build":
        net.build_schedule(static)
    else:
        net._forward_steps(static)
    for _ in range(6):
        y = net.forward(a)
        _expect(y, 10.0)
        assert y.coors is a.coors and net.outputs["input"].feats is a.feats
    assert any(net._plans.values())  # the pass did become a schedule


def test_a_scheduled_pass_hands_out_its_own_tensors(host):
    net, a, b = _net(_specs()), _input(10.0), _input(500.0)
    net.forward_scheduled(a)
    _expect(net.forward(b), 500.0)
    y = net.forward_scheduled(a)
    _expect(y, 10.0)
    assert y.coors is a.coors and net.inputs["a"].feats is a.feats


def test_a_schedule_is_not_reused_for_other_shapes_at_the_same_address(host):
    net, whole = _net(_specs()), _input(10.0, rows=32)
    part = layers.SparseTensor(whole.feats[:16], whole.coors[:16], whole.num_act, GRID)
    for x in (whole, part, whole):
        net.forward_scheduled(x)
        assert net.inputs["a"].feats.shape == x.feats.shape


def test_a_sum_of_strided_features_is_not_recorded(host):
    """torch adds views of any stride; a schedule's sum step reads memory in order, so such a pass stays step by step."""
    net, x = _net(_specs(last_sum=True)), _input(0.0)
    wide = torch.zeros(16, 8)
    wide[:, :4] = 10.0
    wide[:, 4:] = 1000.0
    x.feats = wide[:, :4]
    for _ in range(5):
        y = net.forward(x)
        assert float(y.feats.max()) == 10.0 + 2 + 10.0 + 1
    assert not any(net._plans.values())


@pytest.mark.parametrize("node", ["Cast", "Add"])
@pytest.mark.parametrize("view", ["columns", "transposed", "plain"])
def test_elementwise_nodes_of_graph_inputs_that_are_views(host, node, view):
    """Runs on one binding become a schedule from the third on; a Cast or an Add of a strided view stays what torch makes
    of it, run after run, with contents that change in between.  Dense tensors do become steps."""
    base = torch.empty(16, 16)
    x = {"columns": base[:, 4:8], "transposed": base.t(), "plain": base}[view]
    elem = onnx_graph.FLOAT
    make = onnx_graph.Node("Cast", ["x"], ["y"], dict(to=onnx_graph.FLOAT16)) if node == "Cast" else \
        onnx_graph.Node("Add", ["x", "z"], ["y"])
    names = ["x"] if node == "Cast" else ["x", "z"]
    model = onnx_graph.Model([make], [onnx_graph.Value(n, elem, list(x.shape)) for n in names],
                             [onnx_graph.Value("y", elem, list(x.shape))])
    ex = onnx_graph.GraphExecutor(model, device="cpu")
    z = torch.arange(float(x.numel())).reshape(x.shape)
    for i in range(8):
        base.copy_(torch.randn(16, 16, generator=torch.Generator().manual_seed(i)))
        y = ex.run(**dict(x=x, z=z) if node == "Add" else dict(x=x))["y"]
        assert torch.equal(y, x.half() if node == "Cast" else x + z)
    assert (ex._bound["native"] is not None) == (view == "plain")


def test_a_view_of_other_strides_at_the_same_address_is_bound_anew(host):
    base = torch.randn(16, 16, generator=torch.Generator().manual_seed(0))
    model = onnx_graph.Model([onnx_graph.Node("Cast", ["x"], ["y"], dict(to=onnx_graph.FLOAT16))],
                             [onnx_graph.Value("x", onnx_graph.FLOAT, [16, 16])],
                             [onnx_graph.Value("y", onnx_graph.FLOAT16, [16, 16])])
    ex = onnx_graph.GraphExecutor(model, device="cpu")
    for x in (base, base.t(), base, base.t()):
        assert torch.equal(ex.run(x=x)["y"], x.half())


def test_a_captured_run_of_an_imported_graph_is_enqueued_operator_by_operator(host, monkeypatch):
    """Also where the run before was on the same buffers or has become a schedule: neither is captured nor run."""
    model = onnx_graph.Model([onnx_graph.Node("Cast", ["x"], ["y"], dict(to=onnx_graph.FLOAT16))],
                             [onnx_graph.Value("x", onnx_graph.FLOAT, [16, 16])],
                             [onnx_graph.Value("y", onnx_graph.FLOAT16, [16, 16])])
    ex, x = onnx_graph.GraphExecutor(model, device="cpu"), torch.rand(16, 16)
    monkeypatch.setattr(_HostSchedule, "capture", lambda *a: pytest.fail("captured as a schedule's steps"))
    for eager in (2, 4):
        for _ in range(eager):
            ex.run(x=x)
        host.capturing = True
        ex._bound["values"]["y"].zero_()
        with monkeypatch.context() as m:
            m.setattr(_HostSchedule, "run", lambda *a: pytest.fail("a schedule does not run under capture"))
            assert torch.equal(ex.run(x=x)["y"], x.half())
        host.capturing = False


def test_results_are_the_callers_own_objects(host):
    """Rebinding tensors on what a pass returned, on its outputs or rulebooks, or on the input afterwards, reaches neither
    the recorded pass nor a later result - while passes run step by step, when they are recorded, and after."""
    net, x = _net(_specs(last_sum=True)), _input(10.0)
    seen = []
    for _ in range(8):
        y = net.forward(x)
        assert y is net.outputs["c"] and net.outputs["input"] is x and net.inputs["b"] is net.outputs["a"]
        _expect(y, 10.0, 2 + 10 + 1)
        assert all(y is not s for s in seen)
        seen.append(y)
        y.feats = y.feats.double() * 0 - 1                 # a float copy, say
        net.outputs["a"].feats = torch.full((16, 4), 99.0)
        net.outputs["b"].coors = None
        net.rulebooks["s"].num_act_in = None
        net.outputs.clear()
    assert any(net._plans.values())
    feats, same = x.feats, layers.SparseTensor(x.feats, x.coors, x.num_act, GRID)
    net = _net(_specs())
    net.forward(x)
    net.forward(x)
    x.feats = torch.full((16, 4), 700.0)                   # the object now names other features, `same` the old ones
    for _ in range(4):
        _expect(net.forward(same), float(feats[0, 0]))


def test_a_recorded_pass_does_not_keep_a_dropped_input(host):
    """The three tensors of an input that became a schedule are freed with the caller's last reference and the next pass,
    and a schedule whose input is gone is dropped, also when another input comes to lie at the same addresses."""
    net, other = _net(_specs(last_sum=True)), _input(500.0)
    memory = torch.empty(16 * 4 * 8)

    def at_the_same_address(value):
        feats = torch.from_numpy(memory.numpy()[:64]).view(16, 4)   # a storage of its own over the same bytes
        feats.fill_(value)
        x = _input(0.0)
        return layers.SparseTensor(feats, x.coors, x.num_act, GRID)

    for value in (10.0, 20.0, 30.0):
        x = at_the_same_address(value)
        for _ in range(5):
            _expect(net.forward(x), value, 2 + value + 1)
        assert any(net._plans.values())
        gone = [weakref.ref(t) for t in (x.feats, x.coors, x.num_act)]
        del x
        net.forward(other)
        assert all(r() is None for r in gone)
        net.forward(other)
        assert not any(net._plans.values())
    for _ in range(5):
        y = net.forward(other)
    assert any(net._plans.values()) and y.coors is other.coors and y.num_act is other.num_act
    assert net.rulebooks["s"].in_coors is other.coors and net.inputs["a"] is other
