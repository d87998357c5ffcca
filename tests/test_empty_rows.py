"""Decision rows without actions and chance rows without outcomes, which the
job contract accepts: such a config's value is zero and none of its cells
exist, so its kernels may write nothing but that value. Its neighbours' cells
start where its own would.

Jobs are edited so that in every decision node the first, the last and most of
the rows between hold no action (their cells go to a neighbouring row, so that
rows of one to several dozen actions remain) and likewise every chance node's
rows. Results bit-identical to the oracle in float32.
"""
import sys

import numpy as np
import pytest

import oracle as O
import warchest_wave as ww
import wcj8
import workloads as W


def regroup(off, lo, n):
    """Empties rows lo .. lo + n - 1 of an offset list except every third, in place; the old row -> new row map."""
    kept = [k for k in range(n) if k % 3 == 1 and k < n - 1] or [0]
    owner = np.array([max((x for x in kept if x <= k), default=kept[0]) for k in range(n)])
    start, end = int(off[lo]), int(off[lo + n])
    ends = {k: int(off[lo + int(np.flatnonzero(owner == k)[-1]) + 1]) for k in kept}
    at = start
    for k in range(n):
        off[lo + k] = at
        at = ends.get(k, at)
    assert at == end == off[lo + n]
    return owner


def emptied(job: bytes) -> bytes:
    d = wcj8.decode(job)
    place = np.arange(d["ncells"], dtype=np.uint32)  # each cell's new place
    for i in range(d["nodes"]):
        me = int(d["node_player"][i])
        n = int(d["cfg_off"][2 * i + me + 1] - d["cfg_off"][2 * i + me])
        if d["node_kind"][i] == 0 and n > 1:
            row0 = int(d["legal_row_of"][i])
            owner = regroup(d["legal_off"], row0, n)
            cells = slice(int(d["soff"][i]), int(d["soff"][i + 1]))
            d["cell_row"][cells] = owner[d["cell_row"][cells]]
            order = np.lexsort((d["legal_action"][cells], d["cell_row"][cells]))  # a row's cells, in action order
            for name in ("legal_action", "legal_child", "legal_trans", "cell_row"):
                d[name][cells] = d[name][cells][order]
            place[cells] = cells.start + np.argsort(order)
        elif d["node_kind"][i] == 1 and n > 1:
            owner = regroup(d["draw_row_start"], int(d["draw_row_off"][i]), n)
            ch = int(d["node_child"][d["node_child_start"][i]])
            row0, rows = int(d["rvd_row_of"][ch]), int(d["cfg_off"][2 * ch + me + 1] - d["cfg_off"][2 * ch + me])
            src = slice(int(d["rvd_start"][row0]), int(d["rvd_start"][row0 + rows]))
            d["rvd_src"][src] = owner[d["rvd_src"][src]]
    d["rev_cell"] = place[d["rev_cell"]]
    d["rev_src"] = d["cell_row"][d["rev_cell"]]
    return wcj8.encode(d)


# actions and outcomes per row, configs per list, trees, nodes, seed, unit slots, windows in LDS
CASES = [
    ((1, 4), (1, 3), 5, 3, 40, 5, "4096", "1"),     # short rows, staged units
    ((2, 9), (2, 5), 40, 4, 200, 40, "4096", "1"),  # rows of every length up to several dozen
    ((2, 9), (2, 5), 12, 3, 200, 12, "4096", "0"),  # units without staged windows
    ((1, 5), (2, 3), 9, 4, 250, 9, "256", "1"),     # small units: top regions, swept per depth
    ((1, 2), (1, 2), 3, 2, 30, 0, "4096", "1"),     # cells a multiple of 64: the last row's would be another array's
]


def case_jobs(case):
    acts, draws, info, trees, nodes, seed = case[:6]
    dims = ww.mlp_dims(inputs=64, hidden=32, layers=1, heads=info, pool=8)
    make = lambda s: [emptied(j) for j in ww.synth_jobs(  # noqa: E731
        dims, seed=s, trees=trees, nodes_lo=nodes, nodes_hi=nodes + 30, act_lo=acts[0], act_hi=acts[1], collapse=0.6,
        chance=1, draw_lo=draws[0], draw_hi=draws[1], info_fixed=info, legal_p=0.8, notrans_p=0.2, terminal_p=0.3,
        dirichlet=1, iters=5, depth=2, snapshots=1, nroots=2, **W.DCFR)]
    jobs = make(seed)
    if seed == 0:
        last = lambda j: np.diff(wcj8.decode(j[-1])["legal_off"])[-1]  # noqa: E731
        jobs = next(j for s in range(1, 2000) for j in [make(s)]
                    if last(j) == 0 and sum(wcj8.decode(b)["ncells"] for b in j) % 64 == 0)
    return jobs, ww.synth_weights(dims, seed=info + 1)


@pytest.mark.parametrize("case", CASES)
def test_jobs_with_empty_rows_are_accepted(case, monkeypatch):
    monkeypatch.setenv("WC_UNIT_SLOTS", case[6])
    jobs, net = case_jobs(case)
    for j in jobs:
        ww.job_validate(j)
        lens = np.diff(wcj8.decode(j)["legal_off"])
        assert (lens == 0).sum() * 2 > len(lens)
        assert np.isfinite(O.solve(j, net, O.NET_F32)["strategy"]).all()
    assert lens[-1] == 0  # the wave's last row
    wave = ww.Wave(jobs)  # (checks it)
    assert wave.stats()["top_levels"] > 0 or case[6] != "256"
    wave.close()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_empty_rows_bit_exact(case, monkeypatch):
    print(f"case empty rows: {case}", flush=True)
    sys.stdout.flush()
    monkeypatch.setenv("WC_UNIT_SLOTS", case[6])
    monkeypatch.setenv("WC_UNIT_LDS", case[7])
    jobs, net = case_jobs(case)
    ex = ww.Executor(0, ww.WC_PRECISE)
    wave = ww.Wave(jobs)
    for got, job in zip(ex.solve(wave, ex.publish(net)), jobs):
        want = O.solve(job, net, O.NET_F32)
        np.testing.assert_array_equal(got.strategy, want["strategy"])
        np.testing.assert_array_equal(got.root_values, want["roots"])
        np.testing.assert_array_equal(got.carries, want["carries"].astype(np.float16))
    wave.close()
    ex.close()


def without_configs(job: bytes) -> bytes:
    """The job's tree with no config at any node."""
    d = wcj8.decode(job)
    for name in ("cfg_off", "reach_off", "soff", "legal_off", "draw_off", "draw_row_start", "rev_start", "rvd_start",
                 "leaf_coff", "snap_coff"):
        d[name] = np.zeros_like(d[name])
    for name in ("legal_action", "legal_child", "legal_trans", "cell_row", "draw_to", "draw_p", "rev_src", "rev_cell",
                 "rvd_src", "rvd_p", "leaf_cidx", "cphi", "cplayer"):
        d[name] = d[name][:0]
    d["ncfg"] = d["ncells"] = 0
    d["root"] = [r[:0] for r in d["root"]]
    d["carried"] = [[r[:0] for r in c] for c in d["carried"]]
    return wcj8.encode(d)


def configless_jobs(pool):
    """Jobs without configs, and their network: pooled columns past the end of such a wave's tables."""
    dims = ww.mlp_dims(inputs=2 * pool + 8, hidden=16, layers=1, heads=3, pool=pool)
    jobs = ww.synth_jobs(dims, seed=pool, trees=2, nodes_lo=20, nodes_hi=30, act_lo=2, act_hi=4, collapse=0.6, chance=1,
                         draw_lo=1, draw_hi=3, info_fixed=3, dirichlet=1, iters=3, depth=2, snapshots=1, nroots=2,
                         **W.DCFR)
    return [without_configs(j) for j in jobs], jobs, ww.synth_weights(dims, seed=pool + 1)


def test_jobs_without_configs_are_accepted():
    for j in configless_jobs(64)[0]:
        ww.job_validate(j)
    wave = ww.Wave(configless_jobs(64)[0])  # (checks it)
    assert wave.stats()["rows"] > 0 and wave.stats()["table_bytes"] < 1 << 16
    wave.close()


@pytest.mark.gpu
@pytest.mark.parametrize("wide", ["0", "1"])
def test_waves_without_configs_read_no_embedding(wide, monkeypatch):
    """Their embedding table is empty, and so is every leaf's pooled belief; beside other jobs they change nothing."""
    monkeypatch.setenv("WC_EMB_WIDE", wide)
    bare, jobs, net = configless_jobs(20000)
    print(f"case waves without configs, wide offsets {wide}", flush=True)
    ex = ww.Executor(0, ww.WC_PRECISE)
    v = ex.publish(net)
    for wave_jobs in (bare, [bare[0], jobs[0], bare[1], jobs[1]]):
        wave = ww.Wave(wave_jobs)
        for p in (0, 1):
            got, mass = ex.leaf_probe(wave, v, p)
            want = [O.leaf_probe(j, net, O.NET_F32, p) for j in wave_jobs]
            np.testing.assert_array_equal(got, np.concatenate([a for a, _ in want]))
            np.testing.assert_array_equal(mass.reshape(-1), np.concatenate([m for _, m in want]).reshape(-1))
        for got, job in zip(ex.solve(wave, v), wave_jobs):
            want = O.solve(job, net, O.NET_F32)
            np.testing.assert_array_equal(got.strategy, want["strategy"])
            np.testing.assert_array_equal(got.root_values, want["roots"])
        wave.close()
    ex.close()
