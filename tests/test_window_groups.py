"""Window loops in groups of iterations and of rows: every reduction over
windows that do and do not divide into groups, over an input (ring or direct
reads) and a computed value (ring in LDS or scratch), for chunks around the
group's rows, with missing values, ties, zeros of both signs and infinities.
The generated kernels run on the CPU against the oracle, bit for bit."""
import numpy as np
import pytest

from emu.emu import EmuModule
from kunquant_amd.codegen import hip
from kunquant_amd.codegen.program import program_text
from kunquant_amd.Driver import compileit
from kunquant_amd.Op import Builder, Input, Output
from kunquant_amd.Stage import Function
from kunquant_amd.ops import (DecayLinear, TsArgMax, TsArgMin, TsRank, WindowedCorrelation, WindowedMax, WindowedMin,
                              WindowedStddev)
from oracle.kun_oracle import OracleProgram
from tests.helpers import assert_bit_exact


def _graph(w):
    b = Builder()
    with b:
        a, c = Input("a"), Input("c")
        x = a * c
        for n, v in (("in", a), ("val", x)):
            for op in (WindowedStddev, TsRank, TsArgMax, TsArgMin, WindowedMin, WindowedMax, DecayLinear):
                Output(op(v, w), f"{op.__name__}_{n}")
        Output(WindowedCorrelation(x, w, a), "corr")
        Output(TsRank(TsRank(a, w), w), "chain")
    return Function(b.ops)


def _rows(T, S, dt, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((T, S))
    a[:, 1] = np.round(a[:, 1] * 2)
    a[:, 2] = rng.choice([0.0, -0.0], T)
    a[:, 3] = rng.choice([np.inf, -np.inf, 0.5], T)
    a[:, 4] = np.where(rng.random(T) < 0.02, np.nan, a[:, 4])
    a[:, 5] = np.where(np.arange(T) == T // 2, np.nan, 1.0)
    a[:, 6] = -np.inf
    a[:, 7] = np.arange(T)
    return np.ascontiguousarray(a.astype(dt))


@pytest.mark.parametrize("dtype", ["float", "double"])
@pytest.mark.parametrize("w,lds", [(2, None), (3, None), (10, None), (13, 1024), (23, None), (37, 4096)])
def test_groups_equal_the_oracle(dtype, w, lds):
    m = compileit(_graph(w), f"groups{w}_{dtype}", input_layout="TS", output_layout="TS", dtype=dtype,
                  options={"no_fast_stat": True})
    S, T, start = 9, 2 * w + 50, 2
    L = T - start
    dt = np.float32 if dtype == "float" else np.float64
    ins = {"a": _rows(T, S, dt, w), "c": _rows(T, S, dt, w + 1)}
    with np.errstate(all="ignore"):
        exp = OracleProgram(program_text(m)).run(ins, S, T, start, L, nthreads=2, temps=True)
    emu = EmuModule(m, lds)
    for st in m.stages:
        for chunk in (0, 1, 3, 5, 22):
            got = {**ins, **exp}
            for b in st.out_bufs:
                got[b.name] = np.full_like(exp[b.name], 12345.0)
            emu.run_stage(st.idx, got, S, T, start, L, chunk)
            for b in st.out_bufs:
                assert_bit_exact(got[b.name], exp[b.name], f"{b.name} chunk {chunk}")


@pytest.mark.parametrize("dtype", ["float", "double"])
@pytest.mark.parametrize("lds", [None, 1024, 3072, 4096, 8192])
def test_scratch_does_not_grow_with_the_rows_of_a_group(dtype, lds, monkeypatch):
    """Groups of four rows need three more slots a ring; a component whose
    rings would then spill more than with two rows keeps to two."""
    m = compileit(_graph(37), f"spill_{dtype}_{lds}", input_layout="TS", output_layout="TS", dtype=dtype,
                  options={"no_fast_stat": True})

    def comps():
        out = []
        for st in m.stages:
            plan = hip.stage_plan(m, st)
            for level in plan.levels:
                for c in level.comps:
                    out.append(hip.CompEmitter(m, st, plan, c, level.kind, lds))
        return [e for e in out if e.interleave]

    now = comps()
    monkeypatch.setattr(hip, "INTERLEAVE_MIN", 2)
    monkeypatch.setattr(hip, "INTERLEAVE_MAX", 2)
    two = comps()
    assert len(now) == len(two) > 0
    for e, t in zip(now, two):
        assert t.interleave == 2 and e.interleave in (2, 4)
        assert e.spill_bytes == t.spill_bytes if e.interleave == 2 else e.spill_bytes <= t.spill_bytes
