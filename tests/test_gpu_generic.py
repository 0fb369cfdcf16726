"""Generic cross-sectional op (a GenericCrossSectionalOp's body compiled as
device code, one thread per row) between time-series stages:
DiffWithWeightedSum(a - b, c), its 5-row average and its rank.

  * TS fp32 module: equal to the reference's own outputs
    (tests/golden/ref_generic_f32.npz) bit for bit;
  * STs fp64 module: equal to the oracle bit for bit;
  * stream module: tick by tick equal to the reference's batch outputs;
  * generic ops with two computed inputs (fp32 TS): equal to the oracle bit for
    bit as a plain run, a batch of jobs, a graph of them and without allocations;
  * session pools refuse the module (the body runs in stream contexts).

Bar: bit-exact (NaN positions equal, NaN payload bits ignored)."""
import os

import numpy as np
import pytest

from kunquant_amd.codegen.program import program_text
from kunquant_amd.runner import KunRunner as kr
from kunquant_amd.workloads import catalog
from oracle.kun_oracle import OracleProgram
from tests.test_zz_no_alloc import _no_alloc, capi  # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")


@pytest.fixture(scope="module")
def executor():
    return kr.createSingleThreadExecutor()


@pytest.fixture(scope="module")
def golden():
    z = np.load(os.path.join(GOLD, "ref_generic_f32.npz"))
    ins = {k[3:]: z[k] for k in z.files if k.startswith("in_")}
    outs = {k[4:]: z[k] for k in z.files if k.startswith("out_")}
    return ins, outs, [int(x) for x in z["meta"]]


def _same(a, b):
    return np.array_equal(a, b, equal_nan=True)


def test_ts_module_matches_reference(executor, golden):
    ins, outs, (S, T, start, L) = golden
    _, mod = catalog.load("generic_f32")
    got = kr.runGraph(executor, mod, ins, start, L)
    bad = [k for k in outs if not _same(got[k], outs[k])]
    assert not bad, bad


def _to_sts(x, b):
    T, S = x.shape
    return np.ascontiguousarray(x.reshape(T, S // b, b).transpose(1, 0, 2))


def test_sts_module_matches_oracle(executor):
    _, mod = catalog.load("generic_f64_sts")
    S, T = 48, 40
    rng = np.random.default_rng(61)
    ins = {k: _to_sts(rng.random((T, S)), 4) for k in ("a", "b", "c")}
    ins["c"][2, 7, 1] = np.nan
    got = kr.runGraph(executor, mod, ins, 0, T)
    exp = OracleProgram(program_text(catalog.module_ir("generic_f64_sts"))).run(ins, S, T, 0, T)
    bad = [k for k in exp if not _same(got[k], exp[k])]
    assert not bad, bad


def test_stream_module_matches_reference(executor, golden):
    ins, outs, (S, T, start, L) = golden
    _, mod = catalog.load("generic_stream_f32")
    st = kr.StreamContext(executor, mod, S)
    h = {k: st.queryBufferHandle(k) for k in list(ins) + list(outs)}
    for t in range(T):
        for k in ins:
            st.pushData(h[k], np.ascontiguousarray(ins[k][t]))
        st.run()
        for k in outs:
            assert _same(st.getCurrentBuffer(h[k]), outs[k][t]), (k, t)


@pytest.mark.parametrize("S,T", [(64, 40), (800, 500)])
def test_two_computed_inputs_match_oracle(executor, capi, S, T):
    torch = pytest.importorskip("torch")
    _, mod = catalog.load("generic_pair_f32")
    prog = OracleProgram(program_text(catalog.module_ir("generic_pair_f32")))
    rng = np.random.default_rng(S + T)
    jobs, exp = [], []
    for _ in range(2):
        ins = {k: rng.standard_normal((T, S)).astype(np.float32) for k in ("a", "b", "c")}
        ins["c"][T // 2, 1] = np.nan
        dev = {k: torch.from_numpy(v).cuda() for k, v in ins.items()}
        out = {k: torch.empty((T, S), device="cuda") for k in mod.getOutputNames()}
        jobs.append((mod, dev, out))
        exp.append(prog.run(ins, S, T, 0, T, nthreads=4))
        got = kr.runGraph(executor, mod, ins, 0, T)
        assert not [k for k in exp[-1] if not _same(got[k], exp[-1][k])]
    tuples = [(m, {k: v.data_ptr() for k, v in {**i, **o}.items()}, S, T, 0, T) for m, i, o in jobs]
    graph = kr.BatchGraph(executor, tuples)
    ways = dict(batch=lambda: kr.runGraphBatchDevice(executor, tuples), graph=graph.launch, replay=graph.launch,
                device=lambda: [kr.runGraphDevice(executor, *t) for t in tuples],
                no_alloc=lambda: [_no_alloc(capi, executor, m, t[1], S, T) for m, t in zip((mod, mod), tuples)])
    for way, call in ways.items():
        for _, _, out in jobs:
            for v in out.values():
                v.fill_(12345.0)
        torch.cuda.synchronize()
        call()
        executor.synchronize()
        torch.cuda.synchronize()
        for (_, _, out), e in zip(jobs, exp):
            bad = [k for k in e if not _same(out[k].cpu().numpy(), e[k])]
            assert not bad, (way, bad)


def test_pool_refuses_generic_stage(executor):
    _, mod = catalog.load("generic_stream_f32")
    with pytest.raises(RuntimeError, match="generic cross-sectional"):
        kr.StreamPool(executor, mod, capacity_stocks=128, max_sessions=2)
