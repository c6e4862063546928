"""Which operator instance ``spconv_mm`` runs for the weights it is handed with a call (no GPU)."""
import importlib

import numpy as np
import pytest

from deploy3d_amd import EngineError, Plugin
from deploy3d_amd.spconv_index import index_blob

mm = importlib.import_module("deploy3d_amd.spconv_mm")
ATTRIBUTES = ((3, 3, 3), 4, 8, 100, True, False, False, 1.0, 1.0)


def _weights(seed, n=27 * 4 * 8):
    return np.random.default_rng(seed).standard_normal(n).astype(np.float32)


@pytest.fixture
def fresh(monkeypatch):
    monkeypatch.setattr(mm, "_by_sample", {})
    monkeypatch.setattr(mm, "_plugins", {})


def test_the_instance_of_a_set_of_values(fresh, monkeypatch):
    """Equal values find their operator without packing a blob, in whatever array they come; any difference - a weight that
    is not sampled, the bias, its absence, an attribute - is another operator; the one used last is asked first."""
    w, b = _weights(0), _weights(1, 8)
    other = w.copy()
    other[1] = np.nextafter(other[1], np.float32(9))       # not among the sampled weights
    sets = [(w, b), (other, b), (w, b + 1), (w, None), (other, None)]
    ops = [mm._plugin_of(ATTRIBUTES, *s) for s in sets]
    assert len(set(map(id, ops))) == len(ops)
    assert len(mm._by_sample) == 1                          # all five share the sampled weights
    shorter = mm._plugin_of(((3, 3, 3), 4, 8, 99) + ATTRIBUTES[4:], w, b)
    assert all(shorter is not o for o in ops)
    monkeypatch.setattr(mm, "mm_blob", lambda *a: pytest.fail("packed a blob for known values"))
    for i in (3, 0, 4, 1, 1, 2):
        weight, bias = sets[i]
        copies = weight.reshape(27, 4, 8).astype(np.float64), None if bias is None else list(bias)
        assert mm._plugin_of(ATTRIBUTES, *copies) is ops[i]
        assert next(iter(mm._by_sample.values()))[0] is ops[i]


def test_no_second_copy_of_the_weights_stays(fresh):
    held = [mm._plugin_of(ATTRIBUTES, _weights(seed), None) for seed in range(20)]
    assert len(set(map(id, held))) == 20
    kept = [x for known in mm._by_sample.values() for x in known]
    assert all(type(p) is Plugin for p in kept) and len(kept) == 20
    assert max(len(sample) for _, sample in mm._by_sample) <= 17 * 4


def test_operators_without_weights_are_refused():
    p = Plugin("SPConvIdx3d", index_blob((3,) * 3, (1,) * 3, (1,) * 3, (1,) * 3, (0,) * 3, 64, True, False))
    with pytest.raises(EngineError):
        p.holds_weights(_weights(0), None)
