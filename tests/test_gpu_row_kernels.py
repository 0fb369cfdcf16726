"""Scale and Rank row kernels at the sizes and on the rows where their
tiles, binades and buckets end, against the oracle (bit for bit)."""
import numpy as np
import pytest

from kunquant_amd.codegen.program import program_text
from kunquant_amd.runner import KunRunner as kr
from kunquant_amd.workloads import catalog
from oracle import kun_oracle as ko
from oracle.kun_oracle import OracleProgram
from tests.helpers import assert_bit_exact

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def executor():
    return kr.createMultiThreadExecutor(4)


def _check(executor, module, a, b):
    _, mod = catalog.load(module)
    T, S = a.shape
    ins = {"a": a, "b": b}
    got = kr.runGraph(executor, mod, ins, 0, T)
    exp = OracleProgram(program_text(catalog.module_ir(module))).run(ins, S, T, 0, T, nthreads=4)
    for k in exp:
        assert_bit_exact(got[k], exp[k], f"{module} {k} S={S}")


def _sum_rows(S, dt, seed):
    """Rows whose running sum of |x| meets ties, binades and limits."""
    rng = np.random.default_rng(seed)
    f = np.finfo(dt)
    one = rng.integers(0, 1 << 20, S).astype(np.float64)
    with np.errstate(all="ignore"):
        rows = [
            # every other cell is half a unit of the sum: the tie goes by the sum's last bit
            np.concatenate([[1024.0], rng.integers(0, 4, max(0, S - 1)) * 512.0 * f.eps])[:S],
            np.concatenate([[1024.0 * (1 + f.eps)], np.full(max(0, S - 1), 512.0 * f.eps)])[:S],
            one * (1 if dt == np.float32 else 2.0 ** 26 + 0.5),          # whole numbers past the mantissa
            2.0 ** (np.arange(S) % 60 - 30.0),                            # many binades, up and down
            np.minimum(2.0 ** np.minimum(np.arange(S) / 5.0, 200.0), 1e30),
            rng.integers(0, 1 << 12, S) * float(f.smallest_subnormal),    # subnormal sums, into the normal ones
            np.full(S, float(f.max) / 3.0),                               # overflow to infinity
            np.where(np.arange(S) == S // 3, np.inf, 1.0),
            np.where(np.arange(S) % 7 == 0, np.nan, rng.standard_normal(S)),
            np.zeros(S),
            np.exp(rng.standard_normal(S) * 3.0),
            rng.standard_normal(S),
        ]
    return np.ascontiguousarray(np.stack(rows).astype(dt))


@pytest.mark.parametrize("module", ["cs_f32", "cs_f64"])
@pytest.mark.parametrize("S", [1, 15, 17, 1023, 1024, 1025, 2049, 3071, 9000])
def test_scale_sums_in_order(executor, module, S):
    dt = catalog.load(module)[1].dtype
    _check(executor, module, _sum_rows(S, dt, S), _sum_rows(S, dt, S + 1))


def _rank_rows(S, dt, seed):
    """Rows whose buckets are empty, deep, mixed, or at the ends of the key range."""
    rng = np.random.default_rng(seed)
    f = np.finfo(dt)
    i = np.arange(S)
    with np.errstate(all="ignore"):
        rows = [
            rng.standard_normal(S),
            100.0 * np.exp(rng.standard_normal(S) * 0.6),
            rng.integers(0, 10, S).astype(np.float64),                            # deep tie groups
            np.where(i % 2 == 0, 0.0, rng.random(S)),                             # half of them zero
            np.where(i % 2 == 0, 100.0 * (1 + (i % 97) * float(f.eps)), 50.0 + 150.0 * rng.random(S)),  # deep and mixed
            np.where(i == S // 2, -float(f.max), rng.random(S)),                  # one outlier
            np.where(i % 3 == 0, np.inf, np.where(i % 3 == 1, -np.inf, rng.standard_normal(S))),
            np.where(i % 2 == 0, np.nan, -rng.random(S)),
            np.full(S, 7.5),
            np.where(i == 0, 1.0, np.nan),
            np.full(S, np.nan),
            rng.integers(-50, 50, S) * float(f.smallest_subnormal),
            rng.standard_normal(S) * 10.0 ** rng.uniform(-30, 30, S),
            1.0 + rng.integers(0, 4 * S, S) * float(f.eps),                       # dense: neighbouring values
            np.sort(rng.standard_normal(S)),
            np.where(rng.random(S) < 0.5, -0.0, 0.0) + np.where(i % 5 == 0, rng.standard_normal(S), 0.0),
        ]
    return np.ascontiguousarray(np.stack(rows).astype(dt))


@pytest.mark.parametrize("module", ["cs_f32", "cs_f64"])
@pytest.mark.parametrize("S", [1, 2, 255, 256, 257, 513, 1025, 2048, 2049, 4097, 8191, 8193, 16383])
def test_rank_buckets(executor, module, S):
    dt = catalog.load(module)[1].dtype
    _check(executor, module, _rank_rows(S, dt, S), _rank_rows(S, dt, S + 1)[::-1].copy())


@pytest.mark.parametrize("rank_inputs", [False, True])
@pytest.mark.parametrize("S,T,n", [(1, 1, 1), (5, 9, 2), (127, 8, 3), (128, 7, 1), (129, 17, 17), (256, 64, 33), (1000, 5, 2)])
def test_corr_tiles(executor, S, T, n, rank_inputs):
    """Rows and tiles that do not fill up, more inputs than one launch takes,
    signed zeros, a missing cell."""
    rng = np.random.default_rng(S * 100 + T + n)
    y = rng.standard_normal((T, S)).astype(np.float32)
    y[0] = -0.0
    xs = [rng.standard_normal((T, S)).astype(np.float32) for _ in range(n)]
    xs[0][T // 2, S // 2] = np.nan
    outs = [np.full(T, 7.0, np.float32) for _ in range(n)]
    kr.corrWith(executor, xs, y, outs, "TS", rank_inputs=rank_inputs)
    for x, o in zip(xs, outs):
        assert_bit_exact(o, ko.corr_with(x, y, rank_inputs=rank_inputs), f"S={S} T={T} n={n}")


def _cluster_rows(S, dt, seed):
    """Rows that crowd few buckets: clusters beside distant values, clusters
    within clusters (which end in the sort), with ties and missing cells."""
    rng = np.random.default_rng(seed)
    eps = float(np.finfo(dt).eps)
    i = np.arange(S)
    far = lambda x, *v: np.where(i < len(v), np.resize(v, S), x)
    rows = [
        far(100 * (1 + 1e-4 * rng.random(S)), 1e30),
        far(100 * (1 + 1e-4 * rng.random(S)), -1e30, np.inf, -np.inf),
        far(1 + eps * rng.integers(0, 3 * S, S), 1e30),                                 # neighbouring values
        far(1 + eps * rng.integers(0, 9, S), 1e30, -1e30),                              # few of them
        far(np.where(i % 2, 1.0, 1 + 64 * eps * rng.integers(0, S, S)), 1e30),          # half of them equal
        far(np.where(rng.random(S) < 0.02, np.nan, -3 * (1 + 1e-5 * rng.random(S))), 1e25),
        far(np.where(i % 2, 1 + eps * rng.integers(0, 2 * S, S), rng.random(S) * 1e4), 1e30),
        far(1e-3 + np.where(i % 3, 0, 1e-30) * rng.random(S), 1e30, 1e-30),
    ]
    return np.ascontiguousarray(np.stack(rows).astype(dt))


@pytest.mark.parametrize("module", ["cs_f32", "cs_f64"])
@pytest.mark.parametrize("S", [67, 256, 513, 2049, 8191, 8192, 8193, 16384])
def test_rank_clusters(executor, module, S):
    dt = catalog.load(module)[1].dtype
    _check(executor, module, _cluster_rows(S, dt, S), _cluster_rows(S, dt, S + 1)[::-1].copy())


@pytest.mark.parametrize("module", ["cs_f32", "cs_f64"])
@pytest.mark.parametrize("S", [16, 112, 113, 127, 128, 129, 144, 145, 2048, 2050, 3073, 4097])
def test_scale_heads(executor, module, S):
    """Rows that end in, at and after the cells added one by one."""
    dt = catalog.load(module)[1].dtype
    _check(executor, module, _sum_rows(S, dt, S), _sum_rows(S, dt, S + 1))
