"""Sorted windows (quantile, and the skip-list forms of rank, extremes and
position) in row chunks: the generated kernels run on the CPU against the
oracle bit for bit, for chunks around the window's length, with missing
values, ties, zeros of both signs and infinities."""
import numpy as np
import pytest

from emu.emu import EmuModule
from kunquant_amd.codegen.hip import rows_splittable, stage_plan
from kunquant_amd.codegen.plan import is_window_sorted
from kunquant_amd.codegen.program import program_text
from kunquant_amd.Driver import compileit
from kunquant_amd.Op import Builder, Input, Output
from kunquant_amd.Stage import Function
from kunquant_amd.ops import BackRef, ExpMovingAvg, SkipListQuantile, SkipListState, WindowedQuantile
from kunquant_amd.ops.MiscOp import SkipListArgMin, SkipListMax, SkipListMin, SkipListRank
from oracle.kun_oracle import OracleProgram
from tests.helpers import assert_bit_exact


def _graph(w):
    b = Builder()
    with b:
        a = Input("a")
        Output(WindowedQuantile(a, w, 0.3), "q")
        Output(WindowedQuantile(a * 2 - BackRef(a, 2), w, 0.8), "q_computed")
        st = SkipListState(BackRef(a, w), a, w)
        Output(SkipListRank(st, a), "rank")
        Output(SkipListMin(st), "min")
        Output(SkipListMax(st), "max")
        Output(SkipListArgMin([st], []), "argmin")
    return Function(b.ops)


def _rows(T, S, dt):
    rng = np.random.default_rng(T + S)
    a = rng.standard_normal((T, S))
    a[:, 1] = np.round(a[:, 1] * 2)                                     # ties
    a[:, 2] = rng.choice([0.0, -0.0, 1.0], T)
    a[:, 3] = rng.choice([np.inf, -np.inf, 0.5, np.nan], T)
    a[:, 4] = np.where(rng.random(T) < 0.1, np.nan, a[:, 4])
    a[:, 5] = np.nan
    a[:, 6] = np.inf
    a[:, 7] = np.arange(T)
    return np.ascontiguousarray(a.astype(dt))


@pytest.mark.parametrize("dtype", ["float", "double"])
@pytest.mark.parametrize("w", [1, 2, 7, 150])
def test_row_chunks_equal_the_oracle(dtype, w):
    """150 rows: the values and row indices of the one state exceed the
    registers, sit in scratch columns and keep walking every row."""
    m = compileit(_graph(w), f"sorted{w}_{dtype}", input_layout="TS", output_layout="TS", dtype=dtype,
                  options={"no_fast_stat": "no_warn"})
    S, T, start = 9, 2 * w + 40, 3
    L = T - start
    a = _rows(T, S, np.float32 if dtype == "float" else np.float64)
    exp = OracleProgram(program_text(m)).run({"a": a}, S, T, start, L, nthreads=2, temps=True)
    emu = EmuModule(m)
    for st in m.stages:
        for chunk in {0, 1, max(1, w - 1), w, w + 1, 16}:
            got = {"a": a, **exp}
            for b in st.out_bufs:
                got[b.name] = np.full_like(exp[b.name], 12345.0)
            emu.run_stage(st.idx, got, S, T, start, L, chunk)
            for b in st.out_bufs:
                assert_bit_exact(got[b.name], exp[b.name], f"{b.name} chunk {chunk}")


def test_only_pure_windows_are_split():
    """A state fed something else than its own value a window ago, and one
    beside a recurrence over all rows, keep walking every row."""
    b = Builder()
    with b:
        a = Input("a")
        good = SkipListState(BackRef(a, 9), a, 9)
        other = SkipListState(BackRef(a, 8), a, 9)
        Output(SkipListQuantile(good, 0.5), "good")
        Output(SkipListQuantile(other, 0.5), "other")
        Output(ExpMovingAvg(a, 5), "ema")
    m = compileit(Function(b.ops), "t", input_layout="TS", output_layout="TS", dtype="double",
                  options={"no_fast_stat": "no_warn"})
    (st,) = m.stages
    plan = stage_plan(m, st)
    split = {}
    for level in plan.levels:
        for c in level.comps:
            for op in c.ops:
                if isinstance(op, Output):
                    split[op.attrs["name"]] = rows_splittable(plan, c)
                if op.__class__.__name__ == "SkipListState":
                    assert is_window_sorted(op) == (op.inputs[0].attrs["window"] == 9)
    assert split == {"good": True, "other": False, "ema": False}


@pytest.mark.parametrize("dtype", ["float", "double"])
@pytest.mark.parametrize("w", [1, 2, 7, 150])
def test_any_leaving_value_equals_the_oracle(dtype, w):
    """States whose leaving value is not the value that entered a window ago:
    only what is found leaves. `a` and `c` are the same series but for cells
    missing from one of them, so that a value leaves that never entered, or
    one that entered stays (at most one a stock: no window ever holds more
    than w + 1 values); a lag of w + 1 holds w values only where one of them
    is missing. In registers, and (150 rows) in scratch columns."""
    b = Builder()
    with b:
        a, c = Input("a"), Input("c")
        for name, st in (("other", SkipListState(BackRef(c, w), a, w)),
                         ("longer", SkipListState(BackRef(a, w + 1), a, w)),
                         ("computed", SkipListState(BackRef(c * 2, w), a * 2, w))):
            assert not is_window_sorted(st)
            Output(SkipListQuantile(st, 0.3), f"q_{name}")
            Output(SkipListMin(st), f"min_{name}")
            Output(SkipListMax(st), f"max_{name}")
            Output(SkipListArgMin([st], []), f"argmin_{name}")
    m = compileit(Function(b.ops), f"leaving{w}_{dtype}", input_layout="TS", output_layout="TS", dtype=dtype,
                  options={"no_fast_stat": "no_warn"})
    S, T = 9, 4 * w + 40
    dt = np.float32 if dtype == "float" else np.float64
    rng = np.random.default_rng(w)
    x = rng.standard_normal((T, S))
    x[:, 1] = np.round(x[:, 1] * 2)
    a, c = x.astype(dt), x.astype(dt)
    for s in range(S):
        gone = rng.choice(np.arange(1, T), 3 + T // (w + 3), replace=False)
        a[gone[1:], s] = np.nan             # leaves without having entered
        if s % 3:
            c[:, s] = np.where(np.isin(np.arange(T), gone[2:]), np.nan, c[:, s])
            c[gone[0], s] = np.nan          # entered and stays
    exp = OracleProgram(program_text(m)).run({"a": a, "c": c}, S, T, 0, T, nthreads=2, temps=True)
    for name in ("q_other", "q_longer", "q_computed"):
        assert np.isfinite(exp[name][T // 2:]).sum() >= 10, name
    emu = EmuModule(m)
    for st in m.stages:
        for chunk in (0, 16):
            got = {"a": a, "c": c, **exp}
            for o in st.out_bufs:
                got[o.name] = np.full_like(exp[o.name], 12345.0)
            emu.run_stage(st.idx, got, S, T, 0, T, chunk)
            for o in st.out_bufs:
                assert_bit_exact(got[o.name], exp[o.name], f"{o.name} chunk {chunk}")


@pytest.mark.parametrize("dtype", ["float", "double"])
def test_windows_that_grow_keep_to_their_columns(dtype):
    """A state whose leaving values are never in its window grows with every
    row. In scratch columns it keeps to its own w + 1 slots: the window in the
    next columns is that of a module without it."""
    w, S, T = 150, 9, 600

    def graph(grow):
        b = Builder()
        with b:
            a, c = Input("a"), Input("c")
            first = SkipListArgMin([SkipListState(BackRef(c, w), a, w)], [])
            second = SkipListArgMin([SkipListState(BackRef(a, w), a, w)], [])
            Output(second, "second")
            Output(first + second if grow else c - second, "joint")
        return Function(b.ops)

    dt = np.float32 if dtype == "float" else np.float64
    rng = np.random.default_rng(3)
    a = rng.standard_normal((T, S)).astype(dt)
    ins = {"a": a, "c": a + dt(1000)}
    opt = dict(input_layout="TS", output_layout="TS", dtype=dtype, options={"no_fast_stat": "no_warn"})
    exp = OracleProgram(program_text(compileit(graph(False), "g", **opt))).run(ins, S, T, 0, T)
    m = compileit(graph(True), f"grow_{dtype}", **opt)
    emu = EmuModule(m)
    (st,) = m.stages
    got = {**ins, **{o.name: np.full((T, S), 12345.0, dt) for o in st.out_bufs}}
    emu.run_stage(st.idx, got, S, T, 0, T, 0)
    assert_bit_exact(got["second"], exp["second"], "second")
    assert np.isnan(got["joint"][w + 1:]).all()
