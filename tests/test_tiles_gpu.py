"""Densities and the V_xc build against the FP64 oracle at basis sizes on both sides of every tile
edge (16-wide blocks, tiles of up to four blocks, a ragged last tile), with one spin and two, a
short grid (one chunk an item) and a longer one, on random AO planes: no symmetry, no cancellation.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# FP64: sums of up to 1300 points and 210 functions in another order, 1e-13 expected.  FP32: planes,
# D and the potentials each round by 2^-24 and sums over the basis add a few of them (1e-6 expected);
# the bar is the mixed-precision gate.
TOL = {"fp64": 1e-11, "fp32": 1e-5}


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _molecule(n, npts, seed, polarised):
    from graddft_amd.molecule import Grid, Molecule
    rng = np.random.default_rng(seed)
    rows, cols = (npts + 63) // 64 * 64, (n + 15) // 16 * 16
    planes = np.zeros((5, rows, cols))
    planes[:, :npts, :n] = rng.normal(size=(5, npts, n)) / np.sqrt(n)
    w = np.zeros(rows)
    w[:npts] = rng.uniform(0.1, 1.0, npts)
    D = []
    for s in range(2):
        c = rng.normal(size=(n, max(2, n // 3)))
        D.append(c @ c.T * 0.3)
    rdm1 = np.stack(D if polarised else [D[0], D[0]])
    dev = lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
    z = dev(np.zeros((n, n)))
    mol = Molecule(grid=Grid(dev(np.zeros((npts, 3))), dev(w[:npts]), dev(w)), atom_index=torch.ones(1),
                   nuclear_pos=dev(np.zeros((1, 3))), ao_planes=dev(planes), rdm1=dev(rdm1), nuclear_repulsion=0.0,
                   h1e=z, s1e=z, mo_coeff=dev(np.zeros((2, n, n))), mo_occ=dev(np.zeros((2, n))),
                   mo_energy=dev(np.zeros((2, n))), restricted=not polarised)
    return mol, planes[:, :npts, :n], w[:npts], rdm1


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,npts", [(1, 70), (16, 300), (17, 1300), (33, 300), (49, 1300), (64, 64), (65, 300),
                                    (81, 1300), (97, 300), (113, 1300), (128, 300), (129, 300), (150, 64), (177, 1300),
                                    (192, 300), (193, 300), (209, 1300)])
def test_densities_and_vxc_at_tile_edges(n, npts, precision):
    from graddft_amd import B3LYP_GRID
    from oracle import xc as X
    for polarised in (False, True):
        print(f"case: n={n} npts={npts} {precision} polarised={polarised}", flush=True)
        mol, p, w, D0 = _molecule(n, npts, n + npts, polarised)
        d2 = np.repeat(p[4][..., None] / 3.0, 3, axis=-1)
        inp = X.to_inputs(p[0], np.moveaxis(p[1:4], 0, -1), d2, w)
        E0, gD0, _ = X.xc_value_and_grads("b3lyp", inp, D0)
        D = mol.rdm1.detach().clone().requires_grad_(True)
        E = B3LYP_GRID.xc_energy(None, mol, precision, rdm1=D)
        (gD,) = torch.autograd.grad(E, [D])
        assert _rel(gD.cpu().numpy(), gD0) <= TOL[precision]
        # FP32: rho is exact to 2^-31, the gradients and the kinetic term are rounded by 2^-24 a point
        assert abs(float(E.detach()) - E0) <= (1e-11 if precision == "fp64" else 1e-6) * abs(E0)
        # densities of a matrix that is not symmetric
        A = D0 + 0.1 * np.random.default_rng(n).normal(size=D0.shape)
        if not polarised:
            A[1] = A[0]
        T = torch.as_tensor(A)
        dens = B3LYP_GRID.plan(mol, precision).densities(T.cuda()).cpu().numpy()
        for got, ref in [(dens[:, :, 0], X.density(T, inp.ao)), (dens[:, :, 1:4], X.grad_density(T, inp.ao, inp.grad_ao)),
                         (dens[:, :, 4], X.kinetic_density(T, inp.grad_ao)),
                         (dens[:, :, 5], X.lapl_density(T, inp.ao, inp.grad_ao, inp.d2_ao))]:
            assert _rel(got, ref.numpy()) <= TOL[precision]
