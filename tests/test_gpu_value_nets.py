"""The leaf-network kernels at the edges of their tiles, through the C ABI.

Float32: bit-identical to the oracle's CPU loop at every tile size the
dispatch takes (few, some and many rows), with inputs, hidden widths and heads
that fill no tile, no 16-byte run and no k tile, from buffers that 16-byte
loads may not read, and with infinite weights behind zero inputs.
"""
import ctypes as C
import sys

import numpy as np
import pytest

import oracle as O
import warchest_wave as ww
import workloads as W
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def forward_on_device(ex, v, x, heads, offset):
    """mlp_noalloc with both buffers `offset` floats past a 256-byte boundary."""
    hip = Hip()
    rows = x.shape[0]
    xd, od = hip.alloc((x.size + offset) * 4), hip.alloc((rows * heads + offset) * 4)
    try:
        hip.to_dev(xd + 4 * offset, x)
        ex.mlp_noalloc(v, rows, xd + 4 * offset, od + 4 * offset)
        out = np.zeros((rows, heads), np.float32)
        hip.to_host(out, od + 4 * offset)
        return out
    finally:
        hip.free(xd)
        hip.free(od)


# rows x outputs cross the lines between the four tile sizes
@pytest.mark.parametrize("inputs,hidden,layers,heads,rows,offset", [
    (101, 50, 2, 7, 1, 0), (130, 64, 1, 1, 17, 1), (512, 384, 3, 22, 64, 0), (97, 130, 2, 567, 333, 3),
    (160, 384, 2, 33, 1500, 2), (132, 384, 1, 567, 3100, 1),
    (132, 384, 1, 65, 5500, 0), (31, 391, 1, 22, 6001, 1)])
def test_float32_net_edges(inputs, hidden, layers, heads, rows, offset):
    say(f"case float32 net: {rows} rows, {inputs} -> {layers}x{hidden} -> {heads}, buffers + {offset} floats")
    net = ww.synth_weights(ww.mlp_dims(inputs, hidden, layers, heads, pool=8), seed=rows)
    x = ww.synth_features(rows, inputs, seed=rows + 1)
    ex = ww.Executor(0, ww.WC_PRECISE)
    got = forward_on_device(ex, ex.publish(net), x, heads, offset)
    ex.close()
    keys = np.tile(np.arange(heads, dtype=np.uint32), (rows, 1))
    np.testing.assert_array_equal(got, O.mlp(x, keys, net, O.NET_F32))


def test_float32_net_skips_zero_inputs_of_infinite_weights():
    say("case float32 net: infinite and NaN weights behind zero and non-zero inputs")
    net = ww.synth_weights(ww.mlp_dims(36, 40, 2, 5, pool=8), seed=3)
    x = ww.synth_features(50, 36, seed=4)
    x[:25, 7] = 0.0
    net.w[7 * 40 + 11] = np.inf
    net.w[7 * 40 + 12] = np.nan
    ex = ww.Executor(0, ww.WC_PRECISE)
    got = ex.mlp(ex.publish(net), x, heads=5)
    ex.close()
    keys = np.tile(np.arange(5, dtype=np.uint32), (50, 1))
    want = O.mlp(x, keys, net, O.NET_F32)
    assert np.isfinite(want[:25]).all() and not np.isfinite(want[25:]).all()
    np.testing.assert_array_equal(got, want)


def test_float32_bank_holds_its_weights_once():
    """Device memory a published float32 network takes: its matrices and biases, and no copy of them beside."""
    say("case float32 bank: device memory of a 2048 -> 3x2048 -> 64 net")
    net = ww.synth_weights(ww.mlp_dims(2048, 2048, 3, 64, pool=8), seed=1)
    size = 4 * (net.w.size + net.b.size)
    ex = ww.Executor(0, ww.WC_PRECISE)
    ex.publish(ww.synth_weights(ww.mlp_dims(32, 32, 1, 1, pool=8), seed=1))  # (what a first publish sets up)
    free, total = C.c_size_t(), C.c_size_t()
    L = Hip().L
    L.hipMemGetInfo.argtypes, L.hipMemGetInfo.restype = [C.POINTER(C.c_size_t)] * 2, C.c_int
    assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    before = free.value
    ex.publish(net)
    assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    ex.close()
    say(f"  {size} bytes of weights, {before - free.value} bytes of memory")
    assert size <= before - free.value < 1.25 * size


# one pass per row block, several blocks per pass with a short last one, full passes; buffers off 16 bytes
@pytest.mark.parametrize("precision", [ww.WC_F16, ww.WC_BF16])
@pytest.mark.parametrize("inputs,hidden,layers,heads,rows,offset", [
    (512, 384, 3, 567, 1, 0), (32, 32, 1, 1, 17, 1), (512, 384, 3, 22, 250, 3), (96, 352, 2, 130, 4113, 0),
    (480, 128, 8, 64, 9000, 2), (512, 384, 3, 64, 32000, 0)])
def test_fused_net_from_rows_equals_the_planned_passes(precision, inputs, hidden, layers, heads, rows, offset):
    say(f"case fused net {precision}: {rows} rows, {inputs} -> {layers}x{hidden} -> {heads}, buffers + {offset} floats")
    net = ww.synth_weights(ww.mlp_dims(inputs, hidden, layers, heads, pool=8), seed=rows)
    x = ww.synth_features(rows, inputs, seed=rows + 1)
    ex = ww.Executor(0, precision)
    v = ex.publish(net)
    got = forward_on_device(ex, v, x, heads, offset)
    want = ex.mlp(v, x, heads=heads)
    ex.close()
    np.testing.assert_array_equal(got, want)


# the same launches against the oracle's model of the operand rounding (which shares nothing with them), within the
# bounds of the other comparisons with it: the products' float32 sums run in another order, and where that moves an
# activation across a rounding boundary it moves by one unit of the operand's last place
@pytest.mark.parametrize("precision,mode,bound", [(ww.WC_F16, O.NET_F16, 2e-3), (ww.WC_BF16, O.NET_BF16, 1e-2)])
@pytest.mark.parametrize("inputs,hidden,layers,heads,rows,offset", [
    (512, 384, 3, 567, 250, 3), (96, 352, 2, 130, 1713, 0), (480, 128, 8, 64, 2100, 2), (512, 384, 3, 22, 33, 1)])
def test_fused_net_from_rows_tracks_the_operand_model(precision, mode, bound, inputs, hidden, layers, heads, rows,
                                                      offset):
    say(f"case fused net {precision} against the model: {rows} rows, {inputs} -> {layers}x{hidden} -> {heads}")
    net = ww.synth_weights(ww.mlp_dims(inputs, hidden, layers, heads, pool=8), seed=rows)
    x = ww.synth_features(rows, inputs, seed=rows + 1)
    ex = ww.Executor(0, precision)
    got = forward_on_device(ex, ex.publish(net), x, heads, offset)
    ex.close()
    want = O.mlp(x, np.tile(np.arange(heads, dtype=np.uint32), (rows, 1)), net, mode)
    say(f"  max error {np.abs(got - want).max() / np.abs(want).max():.1e} of the largest value")
    assert np.abs(got - want).max() <= bound * np.abs(want).max()


# in place, out ahead of and behind x by part of a row and by many rows, and end to end; shared head columns,
# one pass and many, rows more and less wide than the head
@pytest.mark.parametrize("precision", [ww.WC_F16, ww.WC_BF16, ww.WC_F16X, ww.WC_PRECISE])
@pytest.mark.parametrize("inputs,hidden,layers,heads,rows,xo,oo", [
    (512, 384, 3, 567, 250, 0, 0), (512, 384, 3, 64, 5000, 0, 0), (96, 128, 2, 567, 3000, 40, 0),
    (480, 384, 3, 22, 4000, 0, 100), (512, 384, 3, 64, 5000, 160000, 0), (160, 64, 1, 33, 700, 0, 160 * 700)])
def test_net_on_overlapping_buffers(precision, inputs, hidden, layers, heads, rows, xo, oo):
    say(f"case overlap {precision}: {rows} rows, {inputs} -> {layers}x{hidden} -> {heads}, x + {xo}, out + {oo} floats")
    net = ww.synth_weights(ww.mlp_dims(inputs, hidden, layers, heads, pool=8), seed=rows)
    x = ww.synth_features(rows, inputs, seed=rows + 1)
    ex = ww.Executor(0, precision)
    v = ex.publish(net)
    hip = Hip()
    at = hip.alloc(4 * max(xo + rows * inputs, oo + rows * heads))
    got = np.zeros((rows, heads), np.float32)
    try:
        hip.to_dev(at + 4 * xo, x)
        ex.mlp_noalloc(v, rows, at + 4 * xo, at + 4 * oo)
        hip.to_host(got, at + 4 * oo)
        want = ex.mlp(v, x, heads=heads)
    finally:
        hip.free(at)
        ex.close()
    np.testing.assert_array_equal(got, want)


# one to four row blocks per pass, two rounds of passes, widths that leave wavefronts idle
@pytest.mark.parametrize("inputs,hidden,layers,heads,rows,offset", [
    (512, 384, 3, 567, 1, 0), (32, 32, 1, 1, 17, 1), (160, 352, 8, 130, 250, 3), (512, 384, 3, 22, 5100, 0),
    (96, 128, 2, 140, 16000, 2), (64, 64, 1, 33, 26000, 0)])
def test_compensated_fused_net(inputs, hidden, layers, heads, rows, offset):
    """From rows and from planned passes alike, and within the compensated operands' rounding of float64: each
    layer's pairs hold 22 bits (2^-22 of the operand), its float32 sum of K terms rounds by at most K 2^-24 of
    the sum of magnitudes; 1e-5 of the largest value covers eight such layers of up to 512 terms."""
    say(f"case compensated fused net: {rows} rows, {inputs} -> {layers}x{hidden} -> {heads}, buffers + {offset} floats")
    net = ww.synth_weights(ww.mlp_dims(inputs, hidden, layers, heads, pool=8), seed=rows)
    x = ww.synth_features(rows, inputs, seed=rows + 1)
    ex = ww.Executor(0, ww.WC_F16X)
    v = ex.publish(net)
    got = forward_on_device(ex, v, x, heads, offset)
    want = ex.mlp(v, x, heads=heads)
    ex.close()
    np.testing.assert_array_equal(got, want)
    h, at, k = x[:500].astype(np.float64), 0, inputs
    for layer in range(layers):
        w = net.w[at:at + k * hidden].reshape(k, hidden).astype(np.float64)
        h, at, k = np.maximum(h @ w + net.b[layer * hidden:(layer + 1) * hidden], 0.0), at + k * hidden, hidden
    ref = h @ net.w[at:].reshape(heads, hidden).T.astype(np.float64) + net.b[layers * hidden:]
    assert np.abs(got[:500] - ref).max() <= 1e-5 * np.abs(ref).max()


# both sides of the lines: a block per CU and more, heads about as wide as a CU should stream, two rounds of passes
@pytest.mark.parametrize("inputs,hidden,layers,heads,rows", [
    (512, 384, 1, 1536, 33), (512, 384, 1, 1540, 33), (96, 64, 2, 1024, 4100), (96, 64, 2, 1030, 4100),
    (96, 64, 1, 830, 20000), (96, 64, 1, 850, 20000)])
def test_compensated_net_under_a_wide_head(inputs, hidden, layers, heads, rows):
    """Planned passes where the fused net pays and layer by layer where it does not, bit for bit the launch from device
    rows, which is always fused."""
    say(f"case compensated wide head: {rows} rows, {inputs} -> {layers}x{hidden} -> {heads}")
    net = ww.synth_weights(ww.mlp_dims(inputs, hidden, layers, heads, pool=8), seed=rows)
    x = ww.synth_features(rows, inputs, seed=rows + 1)
    ex = ww.Executor(0, ww.WC_F16X)
    v = ex.publish(net)
    got, want = ex.mlp(v, x, heads=heads), forward_on_device(ex, v, x, heads, 0)
    ex.close()
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("info,fused", [(1500, True), (2000, False)])
def test_compensated_wave_under_a_wide_head(info, fused):
    """The same line inside a wave, by the widths its row blocks need: leaf values at the initial reach against the
    oracle's model of the compensated operands, within the bound of the other probes of this mode."""
    say(f"case compensated wave: lists of up to {info} configs")
    dims = ww.mlp_dims(inputs=96, hidden=64, layers=1, heads=info, pool=16)
    jobs = ww.synth_jobs(dims, seed=info, trees=2, nodes_lo=12, nodes_hi=20, act_lo=2, act_hi=3, collapse=0.2,
                         chance=1, draw_lo=2, draw_hi=2, info_fixed=info, dirichlet=1, iters=2, depth=2, snapshots=1,
                         nroots=1, **W.DCFR)
    net = ww.synth_weights(dims, seed=info + 1)
    ex = ww.Executor(0, ww.WC_F16X)
    v = ex.publish(net)
    wave = ww.Wave(jobs)
    for p in (0, 1):
        widest = int(wave.array(f"head_rb_n{p}").max())
        assert (widest <= 1536) == fused and widest > 1024
        got, _ = ex.leaf_probe(wave, v, p)
        want = np.concatenate([O.leaf_probe(j, net, O.NET_F16X, p)[0] for j in jobs])
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    wave.close()
    ex.close()


# idle wavefronts, one to four feature blocks each, one to three layers; few rows and several blocks per pass
@pytest.mark.parametrize("precision,mode,bound", [(ww.WC_F16, O.NET_F16, 2e-3), (ww.WC_BF16, O.NET_BF16, 1e-2)])
@pytest.mark.parametrize("inputs,width,layers,trees,nodes", [
    (160, 32, 1, 1, 12), (192, 96, 2, 2, 60), (512, 288, 3, 3, 90), (256, 512, 2, 12, 400), (512, 416, 1, 40, 400)])
def test_fused_public_tower(precision, mode, bound, inputs, width, layers, trees, nodes):
    """The wave's leaf values at the initial reach against the oracle's model of the operand rounding, within the
    bounds of the full waves' leaf probes."""
    say(f"case fused tower {precision}: {inputs} -> {layers}x{width}, {trees} trees of {nodes} nodes")
    dims = ww.two_tower_dims(inputs=inputs, width=width, pub_layers=layers, priv_in=32, priv_layers=1, pool=64)
    jobs = ww.synth_jobs(dims, seed=width, trees=trees, nodes_lo=nodes, nodes_hi=nodes + 9, act_lo=3, act_hi=8,
                         collapse=0.6, chance=1, draw_lo=2, draw_hi=3, info_fixed=9, dirichlet=1, iters=2, depth=2,
                         snapshots=1, nroots=1, **W.DCFR)
    net = ww.synth_weights(dims, seed=layers)
    ex = ww.Executor(0, precision)
    wave = ww.Wave(jobs)
    got, _ = ex.leaf_probe(wave, ex.publish(net), 0)
    rows = wave.stats()["rows"]
    wave.close()
    ex.close()
    want = np.concatenate([O.leaf_probe(j, net, mode, 0)[0] for j in jobs])
    say(f"  {rows} rows, max error {np.abs(got - want).max() / np.abs(want).max():.1e} of the largest value")
    assert np.abs(got - want).max() <= bound * np.abs(want).max()
