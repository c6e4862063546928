"""Rulebooks of millions of rows.  Where the pairs of every (tap, 512 inputs) go is worked out by one workgroup per tap, which
takes 8192 of those blocks a turn (4 194 304 inputs), or 4096 beside a table probe (2 097 152): capacities and live rows on
either side of one turn."""
import numpy as np
import pytest
import torch

from helpers import check_index_structure
from oracle import oracle

pytestmark = pytest.mark.gpu


def cloud(rng, n, grid):
    """About n rows (0, z, y, x) in random order, unique, uniform over the grid."""
    cells = int(np.prod(grid))
    at = rng.permutation(np.flatnonzero(rng.random(cells, dtype=np.float32) < n / cells))
    coords = np.zeros((len(at), 4), np.int32)
    for dim in (3, 2, 1):
        coords[:, dim] = at % grid[dim - 1]
        at = at // grid[dim - 1]
    return coords


@pytest.mark.parametrize("subm", [True, False])
def test_pair_places_beyond_one_turn(engine, subm):
    from deploy3d_amd import spconv_index_nd
    grid, cap, max_out = (41, 1000, 1000), 4300000, 4300000 if subm else 7000000
    geometry = ((3, 1, 1), (1, 1, 1), (1, 0, 0), (1, 1, 1)) if subm else ((3, 1, 1), (2, 1, 1), (0, 0, 0), (1, 1, 1))
    coords = cloud(np.random.default_rng(41), 4250000, grid)
    c = torch.zeros((cap, 4), dtype=torch.int32, device="cuda")
    c[:len(coords)] = torch.from_numpy(coords).cuda()
    host = c.cpu().numpy()
    shape = torch.empty((1, 0) + grid, dtype=torch.int32, device="cuda")
    for n in (len(coords), 4194304, 5000):
        assert n <= len(coords)
        out = spconv_index_nd(c, torch.tensor([n], dtype=torch.int32, device="cuda"), shape, *geometry, (0, 0, 0), max_out, subm, False)
        index, num_index = out[0].cpu().numpy(), int(out[1].item())
        out_grid = list(grid) if subm else list(out[4].shape[2:])
        ref = oracle.rulebook(host, n, [1] + out_grid, *geometry, max_out, subm)
        assert num_index == ref["num_index"]
        if subm:
            np.testing.assert_array_equal(index, ref["index"])
            continue
        # outputs are numbered another way than the oracle's: gather rows and taps as they lie, coordinates through their rows
        live, n_out = ref["index"][2] >= 0, ref["num_act_out"]
        assert int(out[3].item()) == n_out < max_out
        np.testing.assert_array_equal(index[[0, 2]], ref["index"][[0, 2]])
        oc = out[2].cpu().numpy()
        np.testing.assert_array_equal(oc[index[1][live]], ref["out_coors"][ref["index"][1][live]])
        assert len(np.unique(oc[:n_out].astype(np.int64) @ [0, grid[1] * grid[2], grid[2], 1])) == n_out
    check_index_structure(index, num_index, 3, cap)


def test_table_probe_beyond_one_turn(engine):
    """As test_large_strided_operator_on_a_strided_operators_map, with more than one turn of inputs: the linked operator's
    index tensor and table against those of the unlinked one."""
    from deploy3d_amd import spconv_index_nd, spconv_mm
    from deploy3d_amd.spconv_index import index_plugin
    grid, max1, max2 = (41, 1440, 1440), 2600000, 1500000
    rng = np.random.default_rng(43)
    geometry = ((3, 3, 3), (2, 2, 2), (1, 1, 1), (1, 1, 1), (0, 0, 0))
    c = torch.from_numpy(cloud(rng, 800000, grid)).cuda()
    shape = torch.empty((1, 0) + grid, dtype=torch.int32, device="cuda")
    producer, consumer = index_plugin(*geometry, max1, False, False), index_plugin(*geometry, max2, False, False)
    weight = rng.standard_normal(27 * 32 * 64).astype(np.float32) * 0.1
    feats = torch.randn((max1, 32), dtype=torch.float16, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    for n in (len(c), len(c), 60000):   # (a table is written from the first linked convolution on)
        num = torch.tensor([n], dtype=torch.int32, device="cuda")
        got = []
        for linked in (True, False):
            consumer.link_coords(producer if linked else None)
            _, _, oc, no, osh = spconv_index_nd(c, num, shape, *geometry, max1, False, False)
            index, num_index, oc2, no2, _ = spconv_index_nd(oc, no, osh, *geometry, max2, False, False)
            out = spconv_mm(feats, no, no2, index, num_index, (3, 3, 3), 32, 64, max2, False, False, weight,
                            rulebook=consumer if linked else None)
            assert (int(no.item()) > 1 << 21) == (n > 60000) and int(no.item()) <= max1 and int(no2.item()) <= max2
            got.append([index, num_index, oc2[:int(no2.item())], no2, out])
        for a, b in zip(*got):
            assert torch.equal(a, b)
    consumer.link_coords(None)
