"""int8 convolution (this build's extension: the reference accepts fp16 only, trt/spconv/mm_trt.cu:184) through the
C ABI against the CPU oracle: int32 accumulation of int8 products and the requantize rule
q = clamp(rint(float(acc) * m[c] + bq[c])), bit-exact.  Parity is pinned by that written rule, not by the reference."""
import numpy as np
import pytest
import torch

from chain import oracle_chain
from helpers import gpu_rulebook, random_cloud
from oracle import oracle

pytestmark = pytest.mark.gpu


def run_int8(n, grid, ksize, stride, padding, cin, cout, subm, relu, with_bias=True, seed=0, cap_extra=0):
    from deploy3d_amd import spconv_mm
    rng = np.random.default_rng(seed + 31 * cin + cout + n)
    coords = random_cloud(rng, n, grid, 1)
    n = len(coords)
    kvol = int(np.prod(ksize))
    max_out = n + cap_extra if subm else 8 * n
    rb = gpu_rulebook(coords, n, grid, 1, ksize, stride, padding, (1,) * len(ksize), max_out, subm, cap=n + cap_extra)
    n_out = n if subm else rb["num_act_out"]
    x_q = rng.integers(-128, 128, (n + cap_extra, cin)).astype(np.int8)
    w = (rng.standard_normal((kvol, cin, cout)) / np.sqrt(kvol * cin)).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32) if with_bias else None
    s_in, s_out = np.float32(0.043), np.float32(0.057)
    w_q, s_w = oracle.quantize_weights(w)
    m, bq = oracle.requant_params(s_in, s_w, s_out, b)
    acc = oracle.conv_i8(x_q, w_q, rb["index"], rb["num_index"], max_out)
    want = oracle.requantize(acc, m, bq, relu)
    num_in = rb["num_act_in"]
    num_out = num_in if subm else rb["dev"][3]
    y = spconv_mm(torch.from_numpy(x_q).cuda(), num_in, num_out, rb["dev"][0], rb["dev"][1], ksize, cin, cout, max_out,
                  subm, False, w, b, relu=relu, act_scale_in=float(s_in), act_scale_out=float(s_out))
    torch.cuda.synchronize()
    assert y.dtype == torch.int8
    got = y.cpu().numpy()
    np.testing.assert_array_equal(got[:n_out], want[:n_out])
    # rows past the live outputs hold the requantized bias alone
    if max_out > n_out:
        tail = oracle.requantize(np.zeros((1, cout), np.int32), m, bq, relu)
        np.testing.assert_array_equal(got[n_out:], np.broadcast_to(tail, got[n_out:].shape))
    assert np.abs(got[:n_out].astype(np.int32)).max() > 30      # the case exercises the value range


@pytest.mark.parametrize("cin,cout", [(5, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
                                      (128, 16), (20, 64), (100, 32)])
@pytest.mark.parametrize("relu", [False, True])
def test_int8_subm_bit_exact(engine, cin, cout, relu):
    run_int8(3000, (10, 36, 30), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, cout, True, relu)


@pytest.mark.parametrize("cin,cout", [(1, 16), (3, 32), (5, 16), (8, 32), (9, 16), (16, 16), (16, 32), (32, 16), (32, 32), (32, 64)])
def test_int8_rows_of_at_most_32_bytes(engine, cin, cout):
    """Two or four taps per MFMA (conv_taps.h): 16-row groups, kernel volumes around a multiple of four and 32, rows that
    begin at any byte."""
    for n in (15, 16, 17, 2500):
        run_int8(n, (10, 36, 30), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, cout, True, n == 17)
    for ksize in ((1, 1, 1), (2, 2, 2), (1, 5, 5), (2, 2, 7), (1, 2, 15), (2, 4, 4), (1, 3, 11)):
        run_int8(333, (10, 36, 30), ksize, (1, 1, 1), tuple((k - 1) // 2 for k in ksize), cin, cout, False, False)
    run_int8(2500, (10, 36, 30), (3, 3, 3), (2, 2, 2), (1, 1, 1), cin, cout, False, True)


@pytest.mark.parametrize("cin,cout", [(16, 32), (32, 64), (64, 128), (128, 128)])
def test_int8_strided_bit_exact(engine, cin, cout):
    run_int8(3000, (10, 36, 30), (3, 3, 3), (2, 2, 2), (1, 1, 1), cin, cout, False, True)
    run_int8(2000, (10, 36, 30), (3, 1, 1), (2, 1, 1), (0, 0, 0), cin, cout, False, False, with_bias=False)


@pytest.mark.parametrize("cfg", ["4,8,2", "2,8,3", "2,8,2", "4,4,2", "4,4,3"])
def test_int8_staged_configurations(engine, monkeypatch, cfg):
    monkeypatch.setenv("D3D_CONV_STAGED", cfg)
    run_int8(3001, (10, 36, 30), (3, 3, 3), (1, 1, 1), (1, 1, 1), 64, 64, True, True)
    run_int8(3001, (10, 36, 30), (3, 3, 3), (1, 1, 1), (1, 1, 1), 128, 32, True, False)


@pytest.mark.parametrize("ksize", [(2, 4, 4), (1, 3, 11), (4, 4, 4)])
def test_int8_staged_kernel_volumes_from_32(engine, ksize):
    """32 to 64 taps on the barrier-per-tap kernel: its mask of the taps that occur has its 32nd bit set."""
    run_int8(333, (10, 36, 30), ksize, (1, 1, 1), tuple((k - 1) // 2 for k in ksize), 32, 64, False, False)


@pytest.mark.parametrize("shape", ["32,4", "48,4"])
@pytest.mark.parametrize("cin,cout", [(64, 128), (128, 128)])
def test_int8_pipelined_tile_shapes(engine, monkeypatch, shape, cin, cout):
    """Layers with rows of 64 bytes and more run the software-pipelined kernel; for 128 output channels it chooses
    between two workgroup shapes (and a third for few rows) by row count.  Each forced on a SubM layer with spare capacity and
    a strided one, and once on a layer with more tiles than workgroups, where the pipeline runs across tiles."""
    monkeypatch.setenv("D3D_CONV_PIPE_SHAPE", shape)
    run_int8(9001, (12, 48, 40), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, cout, True, True, cap_extra=51)
    if cin == 64:
        run_int8(5000, (12, 48, 40), (3, 3, 3), (2, 2, 2), (1, 1, 1), cin, cout, False, False)
        run_int8(70000, (16, 200, 200), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, cout, True, True)


@pytest.mark.parametrize("cin", [64, 128])
def test_int8_rows_past_the_live_ones(engine, cin):
    """One capacity with a third to four fifths of it live: the tiles of live rows are dealt out first, the others take their
    bias alone."""
    for n in (30000, 60000):
        run_int8(n, (16, 128, 128), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, 128, True, True, cap_extra=76011 - n)


@pytest.mark.parametrize("cin", [64, 128])
def test_int8_output_channels_shared_out_by_row_count(engine, cin):
    """128 output channels in workgroups of 32 or 64 of them: row counts on both sides of the lines of the shapes."""
    for n in (32 * 256, 32 * 256 + 1, 64 * 256 + 1, 96 * 256 + 1, 128 * 256 + 1):
        run_int8(n, (16, 120, 120), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, 128, True, True)


@pytest.mark.parametrize("cin,cout", [(64, 32), (64, 64), (128, 64), (128, 128)])
def test_int8_pipelined_and_barrier_per_tap_kernels_agree_with_the_oracle(engine, monkeypatch, cin, cout):
    """The same layer on the pipelined kernel (the default from 64 input channels up), across several tiles per
    workgroup, and with the pipelined kernel switched off, which leaves the barrier-per-tap kernel."""
    run_int8(40000, (16, 120, 120), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, cout, True, True)
    monkeypatch.setenv("D3D_CONV_PIPE", "0")
    run_int8(3001, (10, 36, 30), (3, 3, 3), (1, 1, 1), (1, 1, 1), cin, cout, True, False)


@pytest.mark.parametrize("cout", [16, 32])
def test_int8_narrow_rows_of_3_gb(engine, cout):
    """Rows of 8 channels whose offsets no longer fit the kernel that reads them as stored are widened: three gathers, the
    last row among them, from 402.7 million rows."""
    from deploy3d_amd.plugin import Plugin
    from deploy3d_amd.spconv_mm import mm_blob, run_mm
    rows, cin, n_out = 3 << 27, 8, 20
    rng = np.random.default_rng(8)
    x = torch.zeros((rows, cin), dtype=torch.int8, device="cuda")
    picks = [rows - 1, 5, (1 << 28) + 77]
    values = rng.integers(-128, 128, (3, cin)).astype(np.int8)
    for r, v in zip(picks, values):
        x[r] = torch.from_numpy(v).cuda()
    index = np.full((3, 128), -1, np.int32)
    index[:, :3] = [picks, [0, 17, 9], [0, 0, 0]]
    w = rng.standard_normal((1, cin, cout)).astype(np.float32)
    s_in, s_out = np.float32(0.043), np.float32(0.057)
    w_q, s_w = oracle.quantize_weights(w)
    acc = np.zeros((n_out, cout), np.int32)
    acc[[0, 17, 9]] = values.astype(np.int32) @ w_q[0].astype(np.int32)
    want = oracle.requantize(acc, *oracle.requant_params(s_in, s_w, s_out, None), False)
    num = torch.tensor([n_out], dtype=torch.int32, device="cuda")
    plugin = Plugin("SPConvMM", mm_blob((1, 1, 1), cin, cout, n_out, False, False, w, None, act_scale_in=float(s_in),
                                        act_scale_out=float(s_out)))
    out = run_mm(plugin, x, num, num, torch.from_numpy(index).cuda(), torch.tensor([128], dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), want)
    plugin.close()


def test_int8_unsupported_channels_report_status(engine):
    from deploy3d_amd import EngineError
    with pytest.raises(EngineError) as e:
        run_int8(500, (10, 36, 30), (3, 3, 3), (1, 1, 1), (1, 1, 1), 16, 24, True, True)
    assert e.value.status == -1
