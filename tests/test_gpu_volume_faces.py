"""The conforming face term inside the volume kernel against the volume kernel
followed by the element-ordered face launch: the same bits at every order,
precision, layout and flux, on a refined octree whose element count fills no
batch evenly, with a normal velocity of zero on the x-faces (UPWIND's tie), a
Coriolis parameter varying in space, and values that are not finite."""
import numpy as np
import pytest

from drifter_amd import _lib, faces, synth
from drifter_amd.mesh import OctreeAdapter
from drifter_amd.solver import CoriolisParameter, PrimitiveEquationsSolver

pytestmark = pytest.mark.gpu

LAYOUTS = {"packed": _lib.LAYOUT_PACKED, "soa": _lib.LAYOUT_SOA, "lines": _lib.LAYOUT_LINES,
           "blocks": _lib.LAYOUT_BLOCKS}


def _state(case, layout):
    E, n, nd = case.E, case.n, case.nd
    if layout == "soa":
        return synth.to_soa(case.U, E, nd)
    if layout == "lines":
        return synth.to_lines(case.U, E, n)
    if layout == "blocks":
        return synth.to_blocks(case.U, E, n, _lib.load().drf_layout_block_elements(case.order))
    return case.U


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("prec", [_lib.PREC_FP64, _lib.PREC_MIXED])
@pytest.mark.parametrize("kind,params", [(faces.LF_ADV, (0.3, -0.2, 0.1, 0.6)),
                                         (faces.UPWIND, (0.0, -0.2, 0.1, 0.0))])
def test_volume_faces_are_the_element_launch(order, prec, kind, params):
    import torch

    m = OctreeAdapter(0.0, 10000.0, 0.0, 10000.0, -1.0, 0.0)
    m.build_uniform(8, 4, 4)
    m.refine([0, 37, 90], [7, 3, 1])
    bounds, levels, _ = m.elements()
    case = synth.make_case_on(bounds, order, 10000.0, "seamount")
    s = PrimitiveEquationsSolver(order, prec)
    s.initialize(case.E, case.h, coriolis=CoriolisParameter(1e-4, 2e-11, 0.0), y_positions=case.y)
    plan = faces.FacePlan(s, bounds, levels, m.build_face_connections(two_to_one=True), kind=kind,
                          params=params)
    plan.attach()
    dt = torch.float64 if prec == _lib.PREC_FP64 else torch.float32
    for name, layout in LAYOUTS.items():
        U = torch.from_numpy(np.ascontiguousarray(_state(case, name))).cuda().to(dt)
        for bad in (None, float("inf"), float("nan")):
            print(f"[volume faces] order={order} prec={prec} kind={kind} {name} {bad}", flush=True)
            if bad is not None:
                U[U.numel() // 3] = bad
                U[U.numel() // 2] = bad
            plan.set_conforming_mode(faces.BY_ELEMENT)
            want = torch.zeros_like(U)
            s.compute_rhs_dev(U, want, layout)
            plan.set_conforming_mode(faces.IN_VOLUME)
            for lines, remap in ((128, True), (256, False), (512, True)):
                s.set_launch(0, remap, lines)
                got = torch.zeros_like(U)
                s.compute_rhs_dev(U, got, layout)
                torch.cuda.synchronize()
                assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want)), (lines, remap)
                assert torch.equal(torch.isnan(got), torch.isnan(want)), (lines, remap)
    plan.detach()
    plan.close()
    s.close()


@pytest.mark.parametrize("kind", [faces.LF_ADV, faces.UPWIND])
def test_parameters_that_are_not_finite(kind):
    """v n of the scalar fluxes sums all three axes, so one infinite velocity
    makes every face's flux NaN, in the volume kernel as in the element launch."""
    import torch

    print(f"[volume faces] infinite velocity kind={kind}", flush=True)
    m = OctreeAdapter(0.0, 10000.0, 0.0, 10000.0, -1.0, 0.0)
    m.build_uniform(4, 4, 2)
    bounds, levels, _ = m.elements()
    case = synth.make_case_on(bounds, 2, 10000.0, "seamount")
    s = PrimitiveEquationsSolver(2)
    s.initialize(case.E, case.h, coriolis=CoriolisParameter(1e-4, 0.0, 0.0))
    plan = faces.FacePlan(s, bounds, levels, m.build_face_connections(two_to_one=True), kind=kind,
                          params=(0.3, float("inf"), 0.1, 0.6))
    plan.attach()
    U = torch.from_numpy(np.ascontiguousarray(_state(case, "lines"))).cuda()
    out = []
    for mode in (faces.BY_ELEMENT, faces.IN_VOLUME):
        plan.set_conforming_mode(mode)
        out.append(torch.zeros_like(U))
        s.compute_rhs_dev(U, out[-1], _lib.LAYOUT_LINES)
    torch.cuda.synchronize()
    assert torch.isnan(out[0]).any()
    assert torch.equal(torch.isnan(out[0]), torch.isnan(out[1]))
    assert torch.equal(torch.nan_to_num(out[0]), torch.nan_to_num(out[1]))
    plan.detach()
    plan.close()
    s.close()
