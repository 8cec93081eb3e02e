"""FP32 batches on straight-sided meshes run kernels of their own (one product
per element, geometry per element); meshes whose metric varies within an
element by more than 1e-6 run the general ones.

Every order from 2, with and without attenuation and PML, RK2 and RK3, both
block shapes, element counts that leave a part of the last block empty: the
mesh as it is, and the same mesh with one node's metric term changed by 1e-5
(far from the source), which takes the general kernels, each within the FP32
bound 1e-4 of the FP64 run on the same arrays; and the two routes differ.
"""
import dataclasses

import numpy as np
import pytest

from nexd_amd import batch, capi, layout, problem

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return float(np.max(np.linalg.norm(a - b, axis=-1) / np.maximum(np.linalg.norm(b, axis=-1), 1e-300)))


@pytest.mark.parametrize("order", [2, 3, 4, 5])
@pytest.mark.parametrize("att,pml", [(False, 0), (True, 0), (False, 1), (True, 1)])
def test_affine_and_general_route(order, att, pml):
    for timeint in (2, 3):
        p = problem.layered_box(4, 3, 3, order=order, nt=40, pml_cells=pml, nrec_side=2, attenuation=att, timeint=timeint)
        rx = p.geom.rx.reshape(p.nelem, -1).copy()
        rx[0, 0] *= 1 + 1e-5
        bent = dataclasses.replace(p, geom=dataclasses.replace(p.geom, rx=rx.reshape(p.geom.rx.shape)))
        got = {}
        for name, q in (("straight", p), ("bent", bent)):
            print(f"[gpu affine] N={order} att={att} pml={pml} timeint={timeint} {name}", flush=True)
            with capi.Context(layout.reference_arrays(q), energy=False) as ctx:
                ctx.reset()
                ctx.run(1, q.nt)
                ref = ctx.seismograms()
            sb = batch.ShotBatch(q, [q, q, q], True)
            for tile in (0, 1):
                with capi.BatchContext(sb, precision=capi.NEXD_FP32, compensated=tile == 0) as b:
                    b.set_tile(tile)
                    b.reset()
                    b.run(1, q.nt)
                    got[name, tile] = [b.seismograms(k) for k in range(3)]
                assert rel_l2(got[name, tile][2], ref) <= 1e-4
                assert np.array_equal(got[name, tile][0], got[name, tile][2])
        assert not np.array_equal(got["straight", 0][0], got["bent", 0][0])


@pytest.mark.parametrize("order,cells", [(2, (3, 3, 3)), (2, (8, 7, 7)), (2, (12, 11, 11)), (3, (3, 3, 3)), (3, (8, 8, 8)),
                                         (3, (12, 11, 11)), (4, (3, 3, 3)), (4, (5, 5, 5)), (4, (9, 8, 7)), (5, (3, 3, 3)),
                                         (5, (6, 5, 5)), (5, (9, 8, 7))])
@pytest.mark.parametrize("att,pml", [(False, 0), (True, 0), (False, 1), (True, 1)])
def test_affine_and_general_route_fp64(order, cells, att, pml):
    """FP64 single shots take the route for meshes whose metric is one
    pattern times a constant per element to 1e-11; a change of 1e-10 in one
    metric value takes the general kernels.  Mesh sizes on each side of the
    lines between the block shapes; RK2, RK3 and the low-storage RK4 on the
    smallest.  The two runs differ by that change and by 1e-11 of the metric:
    1e-9 of the seismograms' (and energies') norm.
    """
    for timeint in (2, 3, 4) if cells == (3, 3, 3) else (2,):
        p = problem.layered_box(*cells, order=order, nt=24, pml_cells=pml, nrec_side=2, attenuation=att, timeint=timeint)
        rx = p.geom.rx.reshape(p.nelem, -1).copy()
        rx[0, 0] += 1e-10 * np.abs(rx[0]).max()
        bent = dataclasses.replace(p, geom=dataclasses.replace(p.geom, rx=rx.reshape(p.geom.rx.shape)))
        got = []
        for q in (p, bent):
            print(f"[gpu affine fp64] N={order} {cells} att={att} pml={pml} timeint={timeint}", flush=True)
            with capi.Context(layout.reference_arrays(q), energy=True) as ctx:
                ctx.reset()
                en = ctx.run(1, q.nt, want_energy=True)
                got.append((ctx.seismograms(), np.asarray(en)))
        assert np.linalg.norm(got[1][0]) > 0
        for a, b in zip(*got):   # (the energy of a run without PML is zero)
            assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
        assert not np.array_equal(got[0][0], got[1][0])
