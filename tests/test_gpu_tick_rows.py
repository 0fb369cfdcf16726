"""Rows of a stream context that join the tick's copies to the host: what a
read returns, whatever was read, pushed or written on the device before."""
import numpy as np
import pytest
import torch

from kunquant_amd.runner import KunRunner as kr
from kunquant_amd.workloads import catalog

pytestmark = pytest.mark.gpu


class _Row:
    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr=typestr, data=(ptr, False), version=2)


@pytest.mark.parametrize("name", ["stream_f32", "stream_f64"])
@pytest.mark.parametrize("stocks", [8, 40, 1032, 8192])
def test_reads_equal_those_of_a_context_that_never_reads_twice(name, stocks):
    """One context reads every output after every tick (copies join the
    tick), one reads each output only after ticks that follow an unread tick
    (copied when read); inputs are read back, too."""
    _, mod = catalog.load(name)
    ex = kr.createSingleThreadExecutor()
    every, rare = kr.StreamContext(ex, mod, stocks), kr.StreamContext(ex, mod, stocks)
    (inp,), outs = mod.getInputNames(), mod.getOutputNames()
    hi, ho = every.queryBufferHandle(inp), [every.queryBufferHandle(k) for k in outs]
    rng = np.random.default_rng(stocks)
    held = None
    for t in range(7):
        row = rng.standard_normal(stocks).astype(mod.dtype)
        row[rng.random(stocks) < 0.05] = np.nan
        for c in (every, rare):
            c.pushData(hi, row)
            c.run()
        if held is not None:  # a row read before stays until it is read again
            assert np.array_equal(held[0], held[1], equal_nan=True)
        assert np.array_equal(every.getCurrentBuffer(hi), row, equal_nan=True)
        got = [every.getCurrentBuffer(h).copy() for h in ho]
        held = (every.getCurrentBuffer(ho[0]), got[0])
        if t % 2:
            for g, h in zip(got, ho):
                assert np.array_equal(g, rare.getCurrentBuffer(h), equal_nan=True)
        # a pushed row is seen at once
        every.pushData(hi, row + 1)
        assert np.array_equal(every.getCurrentBuffer(hi), row + 1, equal_nan=True)
    # a row written through its device pointer is seen, before and after ticks
    dev = torch.as_tensor(_Row(every.getCurrentDeviceBuffer(hi), stocks, np.dtype(mod.dtype).str), device="cuda")
    for v in (3.0, 4.0):
        every.run()
        dev.fill_(v)
        torch.cuda.synchronize()
        assert np.all(every.getCurrentBuffer(hi) == v)
