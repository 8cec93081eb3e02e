"""A reset puts every buffer of a run back on the device: the state holds the
reference's 1e-24 everywhere, the outputs zeros, and a second run gives the
first one's bits.  Buffer sizes with every remainder of the 16-byte stores (odd
numbers of steps and elements' nodes), each scheme's buffers, both precisions.
"""
import numpy as np
import pytest

from nexd_amd import batch, capi, layout, problem

pytestmark = pytest.mark.gpu

TINY = np.float64(np.float32(1e-24))


@pytest.mark.parametrize("timeint", [2, 3, 4])
@pytest.mark.parametrize("order,nt", [(1, 9), (2, 10), (3, 11)])
def test_reset_restores_every_buffer(order, nt, timeint):
    p = problem.layered_box(4, 3, 3, order=order, nt=nt, pml_cells=1, nrec_side=1, attenuation=True, timeint=timeint)
    print(f"[gpu reset] N={order} nt={nt} timeint={timeint}", flush=True)
    with capi.Context(layout.reference_arrays(p), energy=True) as ctx:
        ctx.reset()
        q0 = ctx.state()
        assert np.all(q0 == TINY)
        en = np.array(ctx.run(1, nt, want_energy=True))
        first = ctx.seismograms().copy()
        ctx.reset()
        assert not np.any(ctx.seismograms())
        q1 = ctx.state()
        assert np.all(q1 == TINY)
        assert np.array_equal(np.array(ctx.run(1, nt, want_energy=True)), en)
        assert np.array_equal(ctx.seismograms(), first) and np.any(first)
    sb = batch.ShotBatch(p, [p, p, p], True)
    for precision, comp in ((capi.NEXD_FP32, timeint != 4), (capi.NEXD_FP32, False), (capi.NEXD_FP64, False)):
        with capi.BatchContext(sb, precision=precision, compensated=comp, energy=True) as b:
            b.reset()
            b.run(1, nt)
            first = [(b.seismograms(k).copy(), np.array(b.energy(k))) for k in range(3)]
            b.reset()
            assert not any(np.any(b.seismograms(k)) or np.any(b.energy(k)) for k in range(3))
            b.run(1, nt)
            for k in range(3):
                assert np.array_equal(b.seismograms(k), first[k][0]) and np.array_equal(b.energy(k), first[k][1])
