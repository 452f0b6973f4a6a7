"""FP32 plans at the ends of the range: values that FP64 takes and FP32 took before its products were
split into bf16 terms."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("restricted", [True, False])
def test_potentials_past_the_range_of_fp32(restricted):
    """Grid weights of 1e42 over small AO values: the potentials of the kinetic term exceed FP32's largest
    number, their products with the AO derivatives do not."""
    from graddft_amd import B3LYP_GRID
    from graddft_amd.molecule import Grid, Molecule
    print(f"case: large potentials, restricted={restricted}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    n, npts = 40, 512
    planes = torch.zeros((5, npts, 48), dtype=torch.float64, device="cuda")
    planes[:, :, :n] = torch.randn((5, npts, n), dtype=torch.float64, device="cuda", generator=g) * 1e-15
    w = (torch.rand(npts, dtype=torch.float64, device="cuda", generator=g) + 0.1) * 1e42
    c = torch.randn((n, n // 3), dtype=torch.float64, device="cuda", generator=g)
    D = torch.stack([c @ c.T] * 2) * 1e28
    z = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    m = Molecule(grid=Grid(torch.zeros((npts, 3), dtype=torch.float64, device="cuda"), w, w), atom_index=torch.ones(1),
                 nuclear_pos=torch.zeros((1, 3)), ao_planes=planes, rdm1=D, nuclear_repulsion=0.0, h1e=z, s1e=z,
                 mo_coeff=torch.zeros((2, n, n)), mo_occ=torch.zeros((2, n)), mo_energy=torch.zeros((2, n)),
                 restricted=restricted)
    out = {}
    for p in ("fp64", "fp32"):
        Dg = D.detach().requires_grad_(True)
        E = B3LYP_GRID.xc_energy(None, m, p, rdm1=Dg)
        out[p] = (E.detach(), *torch.autograd.grad(E, [Dg]))
    assert torch.isfinite(out["fp64"][1]).all()
    assert abs(float(out["fp32"][0] / out["fp64"][0]) - 1) <= 1e-6
    assert _rel(out["fp32"][1], out["fp64"][1]) <= 1e-5


def _water_and_network():
    from graddft_amd import MLPSpec, NeuralFunctional
    from graddft_amd.interface import geometry
    from graddft_amd.interface.builder import molecule_from_geometry
    sym, xyz = geometry.water(np.random.default_rng(0))
    return (molecule_from_geometry(sym, xyz, "sto-3g", 0), NeuralFunctional(MLPSpec(nc=6, h=32, n_hidden=3, nd=4)),
            [0, 6 * 32 + 32, 6 * 32 + 32 + 32 * 32 + 32])


@pytest.mark.parametrize("precision", ["fp32", "bf16x6"])
@pytest.mark.parametrize("layer,weight,exact", [(k, w, w) for k in (0, 1, 2) for w in (np.inf, -np.inf, np.nan)] +
                         [(1, 1e39, np.inf), (2, 1e39, np.inf), (1, -1e39, -np.inf), (2, 3.395e38, 3.395e38)])
def test_weights_that_saturate_the_network(layer, weight, exact, precision):
    """A weight past the range (FP32's largest number, or bf16's, 3.39e38) drives units to ELU(-inf) = -1
    and coefficients to 0 or 2: a finite energy, the one that FP64 has of an infinite weight."""
    print(f"case: weight {weight} in layer {layer}, {precision}", flush=True)
    m, f, first = _water_and_network()
    e = {}
    for p, w in (("fp64", exact), (precision, weight)):
        theta = f.init(seed=4)
        theta[first[layer] + 5] = w
        e[p] = float(f.xc_energy(theta, m, p).detach())
    print("  ", e, flush=True)
    # saturated units are exact, the others' roundings are those of any FP32 network
    assert abs(e[precision] - e["fp64"]) <= 1e-6 * abs(e["fp64"])
    assert (e["fp64"] == 0.0) == bool(np.isnan(weight))   # (the energy's clip takes a NaN for zero)
