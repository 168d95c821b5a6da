"""Whole Runge-Kutta steps in one launch (the volume kernel's step modes)
against the same scheme composed of right-hand sides and vector updates, at
every order, precision and layout, on element counts around one workgroup's
batch (128 grid lines: 128 // (N + 1)^2 elements) and past it.

Tolerance, field by field: both sides evaluate the same expressions and differ
in FMA contraction and in the rounding of the stage states.  A stage's
combination rounds a few times at the size of the field, and a rounding of the
stage state by eps |U| or of a contraction's terms moves the field's tendency by
eps times the size of its terms (_term_size: the largest row sum of |D| times
the fluxes, the pressure gradient and the diffusion), which enters times dt: 8
eps (max |U_f| + stages dt terms_f).  dt is half the CFL step, so that every
field's update and, against the Euler step, some field's stages exceed that
tolerance many times; both are asserted.
"""
import numpy as np
import pytest

from drifter_amd import _lib, synth
from drifter_amd.solver import CoriolisParameter, PrimitiveEquationsSolver

pytestmark = pytest.mark.gpu

SCHEMES = {"euler": _lib.RK_EULER, "rk2": _lib.RK_RK2, "ssprk3": _lib.RK_SSPRK3,
           "rk4": _lib.RK_RK4, "lsrk45": _lib.RK_LSRK45}
LAYOUTS = (_lib.LAYOUT_PACKED, _lib.LAYOUT_SOA, _lib.LAYOUT_LINES, _lib.LAYOUT_BLOCKS)


def _composed(k, U, scheme, dt):
    if scheme == "euler":
        return U + dt * k(U)
    if scheme == "rk2":
        return U + dt * k(U + (0.5 * dt) * k(U))
    if scheme == "ssprk3":
        a = U + dt * k(U)
        b = 0.75 * U + 0.25 * (a + dt * k(a))
        return (1.0 / 3.0) * U + (2.0 / 3.0) * (b + dt * k(b))
    if scheme == "rk4":
        k1 = k(U)
        k2 = k(U + (0.5 * dt) * k1)
        k3 = k(U + (0.5 * dt) * k2)
        return U + (dt / 6.0) * (((k1 + 2.0 * k2) + 2.0 * k3) + k(U + dt * k3))
    A = (0.0, -0.4178904745, -1.192151694643, -1.697784692471, -1.514183444257)
    B = (0.1496590219993, 0.3792103129999, 0.8229550293869, 0.6994504559488, 0.1530572479681)
    Y, r = U, 0.0 * U
    for a, b in zip(A, B):
        r = a * r + dt * k(Y)
        Y = Y + b * r
    return Y


STAGES = {"euler": 1, "rk2": 2, "ssprk3": 3, "rk4": 4, "lsrk45": 5}


def _fields(V, layout, E, n, block):
    """The flat state as (E, 5, nd) float64 on the host."""
    A = V.double().cpu().numpy()
    if layout == _lib.LAYOUT_SOA:
        A = synth.from_soa(A, E, n ** 3)
    elif layout == _lib.LAYOUT_LINES:
        A = synth.from_lines(A, E, n)
    elif layout == _lib.LAYOUT_BLOCKS:
        A = synth.from_blocks(A, E, n, block)
    return A.reshape(E, 5, n ** 3)


def _term_size(P, h, order):
    """Sizes of the terms of each field's tendency, and half the CFL step."""
    n = order + 1
    D = np.zeros(n * n)
    _lib.load().drf_basis(order, None, None, _lib.dptr(D))
    row = np.abs(D).reshape(n, n).sum(axis=1).max()
    H = P[:, 2] + h
    Hm = np.abs(H).max()
    q = np.abs(P).max(axis=(0, 2))
    u, v = np.abs(P[:, 0] / H).max(), np.abs(P[:, 1] / H).max()
    grad = 9.81 * Hm * row * q[2]  # g H times a derivative of eta
    terms = np.array([row * q[0] * (u + v) + grad + 2 * Hm * row ** 2 * u,
                      row * q[1] * (u + v) + grad + 2 * Hm * row ** 2 * v,
                      row * (q[0] + q[1]), row * q[3] * (u + v), row * q[4] * (u + v)])
    return terms, 0.5 * (2.0 / n) / (np.sqrt(9.81 * Hm) + max(u, v))


@pytest.mark.parametrize("order", range(1, 9))
@pytest.mark.parametrize("prec", [_lib.PREC_FP64, _lib.PREC_MIXED])
@pytest.mark.parametrize("scheme", sorted(SCHEMES))
def test_step_is_the_composed_scheme(order, prec, scheme):
    import torch

    n = order + 1
    batch = max(1, 128 // (n * n))
    block = _lib.load().drf_layout_block_elements(order)
    full = synth.make_case(5, 5, 8, order, 10000.0, "seamount")
    nd, dtype = n ** 3, torch.float64 if prec == _lib.PREC_FP64 else torch.float32
    eps = float(np.finfo(np.float64 if prec == _lib.PREC_FP64 else np.float32).eps)
    for q, E in enumerate(sorted({1, max(1, batch - 1), batch, batch + 1, 3 * batch + 2})):
        E = min(E, full.E)
        layout = LAYOUTS[(q + order) % 4]
        print(f"[step] order={order} prec={prec} {scheme} E={E} layout={layout}", flush=True)
        s = PrimitiveEquationsSolver(order, prec)
        beta = 2e-11 if q % 2 else 0.0
        s.initialize(E, full.h[:E * nd], coriolis=CoriolisParameter(1e-4, beta, 0.0),
                     y_positions=full.y[:E * nd])
        P = full.U[:E * 5 * nd]
        terms, dt = _term_size(P.reshape(E, 5, nd), full.h[:E * nd].reshape(E, nd), order)
        if layout == _lib.LAYOUT_SOA:
            P = synth.to_soa(P, E, nd)
        elif layout == _lib.LAYOUT_LINES:
            P = synth.to_lines(P, E, n)
        elif layout == _lib.LAYOUT_BLOCKS:
            P = synth.to_blocks(P, E, n, block)
        U = torch.from_numpy(np.ascontiguousarray(P)).cuda().to(dtype)

        def k(V):
            R = torch.zeros_like(V)
            s.compute_rhs_dev(V.contiguous(), R, layout)
            return R

        want = _composed(k, U, scheme, dt)
        euler = _composed(k, U, "euler", dt)
        got = U.clone()
        s.rk_step_dev(SCHEMES[scheme], 0.0, dt, got, layout)
        torch.cuda.synchronize()
        W, A, B, G = (_fields(V, layout, E, n, block) for V in (want, U, euler, got))
        size = np.abs(A).max(axis=(0, 2))
        tol = 8 * eps * (size + STAGES[scheme] * dt * terms)
        err = np.abs(G - W).max(axis=(0, 2)) / tol
        print("  error / tolerance", np.round(err, 3), flush=True)
        assert (err <= 1.0).all(), err
        # what the tolerance tells apart
        assert (np.abs(W - A).max(axis=(0, 2)) >= 20 * tol).all()
        if scheme != "euler":
            assert (np.abs(W - B).max(axis=(0, 2)) / tol).max() >= 10.0
        s.close()


@pytest.mark.parametrize("order,mesh,E", [(6, (32, 16, 16), 6145), (7, (16, 16, 16), 4095),
                                          (8, (16, 16, 16), 3331)])
@pytest.mark.parametrize("layout", [_lib.LAYOUT_PACKED, _lib.LAYOUT_LINES])
def test_steps_of_resident_workgroups(order, mesh, E, layout):
    """FP64 steps from order 6 run resident workgroups that loop over several
    batches each, in place, on meshes of more batches than fit the card at once.
    The right-hand side is element-local: the step equals, bit for bit, steps of
    300 of the elements at a time, whose batches get a workgroup each.  A
    workgroup holds two elements at orders 6 and 7 and one at order 8, and at
    most four fit a CU, so the batches fill the card three times and the last
    one is part-filled."""
    import torch

    n, nd = order + 1, (order + 1) ** 3
    full = synth.make_case(*mesh, order, 10000.0, "seamount")
    assert full.E >= E
    h = full.h[:E * nd]
    P = torch.from_numpy(full.U[:E * 5 * nd].reshape(E, 5, n * n, n)).cuda()

    def flat(V):
        return V.permute(1, 3, 0, 2).contiguous() if layout == _lib.LAYOUT_LINES else V.clone()

    def step(V, hs, scheme):
        s = PrimitiveEquationsSolver(order)
        s.initialize(V.shape[0], hs, coriolis=CoriolisParameter(1e-4, 0.0, 0.0))
        U = flat(V)
        s.rk_step_dev(SCHEMES[scheme], 0.0, 2e-3, U.view(-1), layout)
        torch.cuda.synchronize()
        s.close()
        return U.permute(2, 0, 3, 1) if layout == _lib.LAYOUT_LINES else U

    for scheme in sorted(SCHEMES):
        print(f"[resident steps] order={order} E={E} layout={layout} {scheme}", flush=True)
        got = step(P, h, scheme)
        for e in range(0, E, 300):
            c = slice(e, min(E, e + 300))
            assert torch.equal(got[c], step(P[c], h[c.start * nd:c.stop * nd], scheme)), e
        assert not torch.equal(got, P)


@pytest.mark.parametrize("order,E", [(1, 64 * 3 + 1), (2, 27), (3, 16 * 2049 + 3), (4, 10 * 2048),
                                     (6, 11), (8, 3 * 2048 + 1)])
@pytest.mark.parametrize("layout", [_lib.LAYOUT_SOA, _lib.LAYOUT_LINES])
def test_wave_speed_at_batch_edges(order, E, layout):
    """The maximum sits in the last element's last node: every batch of every
    workgroup (one or two rounds) counts.  max and sqrt are exact."""
    import torch

    n, nd = order + 1, (order + 1) ** 3
    print(f"[wave] order={order} E={E} layout={layout}", flush=True)
    s = PrimitiveEquationsSolver(order)
    s.initialize(E, np.full(E * nd, 50.0), coriolis=CoriolisParameter(1e-4, 0.0, 0.0))
    P = torch.zeros((E, 5, n * n, n), dtype=torch.float64, device="cuda")
    P[:, 0] = 3.0
    P[-1, 1, -1, -1] = -250.0
    perm = (1, 0, 2, 3) if layout == _lib.LAYOUT_SOA else (1, 3, 0, 2)
    U = P.permute(*perm).contiguous().view(-1)
    assert s.max_wave_speed_dev(U, layout) == float(np.sqrt(9.81 * 50.0) + 250.0 * (1.0 / 50.0))
    out = torch.zeros(1, dtype=torch.float64, device="cuda")
    s.max_wave_speed_noalloc_dev(U, out, layout)
    assert float(out[0]) == s.max_wave_speed_dev(U, layout)
    s.close()
