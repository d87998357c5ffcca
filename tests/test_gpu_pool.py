"""The leaf-input kernels at the edges of their lists, through the C ABI: waves
whose config lists cross the line between one wavefront and one workgroup, the
chunks and the batches, with pooled widths that are no multiple of 8 or 64.

The masses and the network's values at the initial reach against the oracle's
leaf probe: float32 bit-identical; 16-bit nets within the operand rounding's
bound that the leaf probes of the full waves use (2e-3 of the largest value
for f16 and 1e-5 for the compensated mode; masses within 2e-6 relative, a
float32 sum in another order).
"""
import sys

import numpy as np
import pytest

import oracle as O
import warchest_wave as ww
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,mode,bound", [
    (ww.WC_PRECISE, O.NET_F32, 0.0), (ww.WC_F16, O.NET_F16A, 2e-3), (ww.WC_F16X, O.NET_F16X, 1e-5)])
@pytest.mark.parametrize("info,pool", [(1, 64), (15, 24), (16, 20), (17, 72), (33, 64), (63, 64), (65, 12), (191, 64),
                                       (193, 64), (257, 72), (320, 20)])
def test_pool_list_edges(precision, mode, bound, info, pool):
    print(f"case pool: precision {precision}, lists of up to {info} configs, {pool} pooled columns", flush=True)
    sys.stdout.flush()
    dims = ww.mlp_dims(inputs=256, hidden=64, layers=1, heads=max(info, 2), pool=pool)
    jobs = ww.synth_jobs(dims, seed=info, trees=3, nodes_lo=20, nodes_hi=40, act_lo=2, act_hi=5, collapse=0.6,
                         chance=1, draw_lo=2, draw_hi=3, info_fixed=info, dirichlet=1, iters=2, depth=2, snapshots=1,
                         nroots=1, **W.DCFR)
    net = ww.synth_weights(dims, seed=info + 1)
    ex = ww.Executor(0, precision)
    v = ex.publish(net)
    wave = ww.Wave(jobs)
    for p in (0, 1):
        got, mass = ex.leaf_probe(wave, v, p)
        want = [O.leaf_probe(j, net, mode, p) for j in jobs]
        ref, ref_mass = np.concatenate([a for a, _ in want]), np.concatenate([m for _, m in want])
        if bound == 0.0:
            np.testing.assert_array_equal(got, ref)
            np.testing.assert_array_equal(mass.reshape(-1), ref_mass.reshape(-1))
        else:
            assert np.abs(got - ref).max() <= bound * np.abs(ref).max()
            np.testing.assert_allclose(mass.reshape(-1), ref_mass.reshape(-1), rtol=2e-6, atol=1e-30)
    wave.close()
    ex.close()


@pytest.mark.parametrize("info,pool", [(1, 20), (17, 72), (64, 64), (81, 12), (257, 130)])
def test_float32_pool_with_wide_offsets(monkeypatch, info, pool):
    """The path of an embedding table of 4 GiB or more (WC_EMB_WIDE=1 forces it), against the oracle's leaf probe."""
    print(f"case wide pool: lists of up to {info} configs, {pool} pooled columns", flush=True)
    sys.stdout.flush()
    monkeypatch.setenv("WC_EMB_WIDE", "1")
    dims = ww.mlp_dims(inputs=300, hidden=64, layers=1, heads=max(info, 2), pool=pool)
    jobs = ww.synth_jobs(dims, seed=info, trees=3, nodes_lo=20, nodes_hi=40, act_lo=2, act_hi=5, collapse=0.6,
                         chance=1, draw_lo=2, draw_hi=3, info_fixed=info, dirichlet=1, iters=2, depth=2, snapshots=1,
                         nroots=1, **W.DCFR)
    net = ww.synth_weights(dims, seed=info + 1)
    ex = ww.Executor(0, ww.WC_PRECISE)
    v = ex.publish(net)
    wave = ww.Wave(jobs)
    for p in (0, 1):
        got, mass = ex.leaf_probe(wave, v, p)
        want = [O.leaf_probe(j, net, O.NET_F32, p) for j in jobs]
        np.testing.assert_array_equal(got, np.concatenate([a for a, _ in want]))
        np.testing.assert_array_equal(mass.reshape(-1), np.concatenate([m for _, m in want]).reshape(-1))
    wave.close()
    ex.close()


@pytest.mark.parametrize("precision,pool", [(ww.WC_F16, 64), (ww.WC_BF16, 20), (ww.WC_F16X, 72)])
def test_long_lists_that_fill_the_device(precision, pool):
    """More than 16 lists of over 192 configs per CU take a wavefront each instead of a workgroup: the same sums in the
    same order, so a wave of them solves as its parts do, which have few enough for workgroups."""
    print(f"case pool: long lists that fill the device, precision {precision}, {pool} pooled columns", flush=True)
    sys.stdout.flush()
    dims = ww.mlp_dims(inputs=160, hidden=32, layers=1, heads=567, pool=pool)
    jobs = ww.synth_jobs(dims, seed=9, trees=110, nodes_lo=200, nodes_hi=250, act_lo=2, act_hi=3, collapse=0.2,
                         chance=1, draw_lo=2, draw_hi=2, info_fixed=567, dirichlet=1, iters=2, depth=2, snapshots=1,
                         nroots=1, **W.DCFR)
    ex = ww.Executor(0, precision)
    v = ex.publish(ww.synth_weights(dims, seed=pool))

    def solve(part):
        wave = ww.Wave(part)
        lists = [wave.array(f"pool_grp{p}").reshape(-1, 36)[:, 1] for p in (0, 1)]
        out = ex.solve(wave, v)
        wave.close()
        return out, [int((n > 192).sum()) for n in lists]

    whole, long = solve(jobs)
    assert min(long) > 16 * 256
    for lo in range(0, len(jobs), 55):
        part, long = solve(jobs[lo:lo + 55])
        assert 1024 < max(long) < 16 * 256
        for got, want in zip(whole[lo:], part):
            np.testing.assert_array_equal(got.strategy, want.strategy)
            np.testing.assert_array_equal(got.root_values, want.root_values)
            np.testing.assert_array_equal(got.carries, want.carries)
    ex.close()
