"""TVD RK2 with attenuation or PML: the kernels whose second stage forms the
element-local stage-1 values again instead of loading them.

The reference keeps every stage-1 value (src/rungekuttaMod.f90:90-120), as the
oracle does, so every combination of attenuation and PML at every order is
compared with it: block remainders, the last element inside and outside the
PML (its fluxes drive every PML node's update), both FP32 block shapes.
FP64 within the parity bound 1e-10, FP32 within its bound 1e-4.
"""
import dataclasses

import numpy as np
import pytest

from nexd_amd import batch, capi, layout, problem
from oracle import oracle

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return float(np.max(np.linalg.norm(a - b, axis=-1) / np.maximum(np.linalg.norm(b, axis=-1), 1e-300)))


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("att,pml,last_in_pml", [(True, 1, True), (True, 1, False), (False, 1, True), (True, 0, False)])
def test_rk2_recomputed_stage_values(order, att, pml, last_in_pml):
    p = problem.layered_box(5, 4, 3, order=order, nt=60, pml_cells=pml, nrec_side=2, attenuation=att)
    if pml and not last_in_pml:
        # the last element keeps its coefficients but leaves the PML list
        check = p.pml.pmlcheck.copy()
        check[-1] = 0
        p = dataclasses.replace(p, pml=dataclasses.replace(p.pml, pmlcheck=check))
    print(f"[gpu recompute] N={order} att={att} pml={pml} last in PML {last_in_pml} nelem={p.nelem}", flush=True)
    arrs = layout.reference_arrays(p)
    so, eo, _ = oracle.run(arrs, compat=3)
    with capi.Context(arrs) as ctx:
        ctx.reset()
        e = np.concatenate([ctx.run(1, 25, want_energy=True), ctx.run(26, p.nt, want_energy=True)])
        assert rel_l2(ctx.seismograms(), so) <= 1e-10
    if pml:
        assert float(np.max(np.abs(e - eo) / np.abs(eo))) <= 1e-10
    sb = batch.ShotBatch(p, [p, p], True)
    for tile in (0, 1):
        with capi.BatchContext(sb, precision=capi.NEXD_FP32, compensated=tile == 0) as b:
            b.set_tile(tile)
            b.reset()
            b.run(1, p.nt)
            assert rel_l2(b.seismograms(1), so) <= 1e-4
