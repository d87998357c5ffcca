"""The CFR row kernels at the edges of their four-element batches, through the
C ABI, bit-identical to the oracle in float32: decision rows of 1 to 40 cells
(past the rows kept in registers), draws and reach gathers of every remainder,
with cells that have no successor, in subtree units with and without staged
windows and in top regions.
"""
import numpy as np
import pytest

import oracle as O
import warchest_wave as ww
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("acts,draws,info,trees,nodes,lds", [
    ((1, 4), (1, 2), 5, 3, 40, "1"), ((2, 9), (2, 5), 40, 4, 200, "1"), ((4, 13), (3, 9), 9, 2, 300, "1"),
    ((12, 40), (7, 17), 20, 2, 400, "1"), ((3, 12), (2, 6), 300, 2, 300, "1"), ((3, 14), (2, 6), 60, 2, 200, "0")])
def test_row_edges_bit_exact(monkeypatch, acts, draws, info, trees, nodes, lds):
    print(f"case rows: {acts} actions, {draws} draws, {info} configs, {trees} trees of {nodes} nodes, windows in LDS "
          f"{lds}", flush=True)
    dims = ww.mlp_dims(inputs=64, hidden=32, layers=1, heads=max(info, 2), pool=8)
    jobs = ww.synth_jobs(dims, seed=info, trees=trees, nodes_lo=nodes, nodes_hi=nodes + 30, act_lo=acts[0],
                         act_hi=acts[1], collapse=0.6, chance=1, draw_lo=draws[0], draw_hi=draws[1], info_fixed=info,
                         legal_p=0.8, notrans_p=0.2, terminal_p=0.3, dirichlet=1, iters=5, depth=2, snapshots=1,
                         nroots=2, **W.DCFR)
    net = ww.synth_weights(dims, seed=info + 1)
    monkeypatch.setenv("WC_UNIT_LDS", lds)
    ex = ww.Executor(0, ww.WC_PRECISE)
    wave = ww.Wave(jobs)
    for got, job in zip(ex.solve(wave, ex.publish(net)), jobs):
        want = O.solve(job, net, O.NET_F32)
        np.testing.assert_array_equal(got.strategy, want["strategy"])
        np.testing.assert_array_equal(got.root_values, want["roots"])
        np.testing.assert_array_equal(got.carries, want["carries"].astype(np.float16))
    wave.close()
    ex.close()
