"""Flags that a step in the middle of a chunk raises, where the next step's kernels close it: a displacement beyond
the bound of the lists (decided by the closing) and cells or LJ rows that a later rebuild fills (raised by the
binning and the list build of the next step).  Every step's record names the same flags
whichever launch closes it, the chunk that holds the first one fails, and so does every chunk after it.

A cluster flies at the sheet.  Displacement: 0.037 a step from a rebuild on, so the fifth step after one is at
0.185, below the skin rule's 0.2, and the bound 0.2 + 0.01 lies within its next step.  Capacities: enough for the
first list, too small once the cluster is nearer."""
import ctypes as C

import numpy as np
import pytest

import surfacegrowthconsole_amd as sg
from surfacegrowthconsole_amd import _native as N
from surfacegrowthconsole_amd.engine import record_dicts

pytestmark = pytest.mark.gpu

OVERFLOW, DISPLACEMENT = -4, -7
LAYOUTS = ([1] * 30, [30], [17, 13], [4, 26])


def _system(speed, delta_f, ux=8, uy=7):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=100, temperature=20.0, geometry="sphere", seed=3, gap=6.0,
                       velocities="maxwell", step_equil=0, step_cool=2, delta_f=delta_f)
    s.v[:100] = 0.0
    s.v[:100, 2] = -speed
    return s


def _engine(s, prec, chunks, graphs, cfg):
    with sg.Engine(s.params, precision=prec, use_graphs=graphs, **cfg) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        recs, codes = [], []
        for n in chunks:
            buf = (N.SgkRecord * n)()
            codes.append(eng.lib.sgk_run(eng.h, n, 0, buf))
            recs += record_dicts(buf)
        return recs, codes


def _batch(systems, prec, chunks, cfg):
    with sg.Batch([s.params for s in systems], precision=prec, **cfg) as b:
        for k, s in enumerate(systems):
            b.upload(k, s.r, s.v, s.a)
            b.set_run_state(k, 0, 1, 0.0)
        recs, codes = [[] for _ in systems], []
        for n in chunks:
            buf = (N.SgkRecord * (n * len(systems)))()
            codes.append(b.lib.sgk_batch_run(b.h, n, 0, buf))
            for k, x in enumerate(recs):
                x += record_dicts(buf)[k * n : (k + 1) * n]
        return recs, codes


def _expected(codes_of_steps, chunks):
    """A chunk's result is that of its last step."""
    out, at = [], 0
    for n in chunks:
        at += n
        out.append(codes_of_steps[at - 1])
    return out


def _middle(recs):
    first = next(k for k, r in enumerate(recs) if r["errors"])
    assert 3 <= first < 27, first
    assert all(r["errors"] == recs[first]["errors"] for r in recs[first:])


def _same(got, want):
    """The same flags at every step, and up to the first one the same records: a cell or a row that is too small keeps
    the atoms that came first, which are others in another run."""
    first = next((k for k, r in enumerate(want) if r["errors"]), len(want))
    assert [r["errors"] for r in got] == [r["errors"] for r in want]
    assert got[:first] == want[:first]


CASES = {
    "displacement": (7.4, dict(close_margin=0.01), DISPLACEMENT),
    "cells": (6.0, dict(cell_capacity=16), OVERFLOW),
}


@pytest.mark.parametrize("delta_f", [0.0, 1e-4])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
def test_one_system(gpu, case, prec, delta_f):
    speed, cfg, code = CASES[case]
    s = _system(speed, delta_f)
    want, codes = _engine(s, prec, LAYOUTS[0], True, cfg)
    _middle(want)
    assert codes == [code if r["errors"] else 0 for r in want]
    for chunks in LAYOUTS[1:]:
        for graphs in (True, False):
            got, rcs = _engine(s, prec, chunks, graphs, cfg)
            _same(got, want)
            assert rcs == _expected(codes, chunks), (chunks, graphs)


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
def test_rows_that_fill_later(gpu, prec):
    s = _system(6.0, 0.0)
    cfg = dict(lj_capacity=1)  # none is needed at first: the cluster is out of reach of the sheet
    want, codes = _engine(s, prec, LAYOUTS[0], True, cfg)
    _middle(want)
    assert codes == [OVERFLOW if r["errors"] else 0 for r in want]
    for chunks in LAYOUTS[1:]:
        got, rcs = _engine(s, prec, chunks, True, cfg)
        _same(got, want)
        assert rcs == _expected(codes, chunks), chunks


@pytest.mark.parametrize("sync", [0, 1])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
def test_one_replica_of_three(gpu, case, prec, sync):
    speed, cfg, code = CASES[case]
    systems = [_system(0.0, 0.0, 7, 7), _system(speed, 0.0), _system(0.0, 0.0, 7, 8)]
    if case == "cells":  # at rest, these have fuller cells from the start
        systems = [systems[1]]
    cfg = dict(cfg, sync_rebuilds=sync)
    want, codes = _batch(systems, prec, LAYOUTS[0], cfg)
    hit = min(1, len(systems) - 1)
    _middle(want[hit])
    assert all(not r["errors"] for k, x in enumerate(want) if k != hit for r in x)
    assert codes == [code if r["errors"] else 0 for r in want[hit]]
    for chunks in LAYOUTS[1:]:
        got, rcs = _batch(systems, prec, chunks, cfg)
        for x, y in zip(got, want):
            _same(x, y)
        assert rcs == _expected(codes, chunks), chunks
