"""Every width class of the coefficient MLP through the device paths, against the FP64 oracle: the
hidden-layer products pick a kernel by width (feature blocks a wave, tiles past the last feature,
k steps that are not whole) and by the row count (the last row tile)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# FP32: a K <= 256 sum rounds by a few 2^-24 and six products are chained (three layers, forward and
# backward): 6e-8 x 6 x 4 = 1.4e-6 on dE/dtheta.  dE/dD also carries the FP32 rounding of D, which
# the cancellation near the nuclei amplifies; its bar is the mixed-precision gate.  Second order:
# ten times the first.  FP64: the device path's own bars.
TOL = {"fp64": (1e-8, 1e-8, 1e-8), "fp32": (1e-5, 2e-6, 1e-4), "bf16x6": (1e-5, 2e-6, 1e-4)}


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x6"])
@pytest.mark.parametrize("h,layers", [(16, 1), (16, 3), (32, 2), (48, 3), (64, 3), (80, 2), (96, 3), (128, 2), (144, 3),
                                      (192, 2), (208, 2), (256, 3)])
def test_width_first_and_second_order(h, layers, precision):
    print(f"case: h={h} layers={layers} {precision}", flush=True)
    from graddft_amd import MLPSpec, NeuralFunctional, XCEnergyVxcFn
    from graddft_amd.interface import geometry
    from graddft_amd.interface.builder import molecule_from_geometry
    from oracle.ao import eval_ao
    from oracle.scf_grad import xc_hvp
    from oracle.xc import MLPSpec as OSpec, to_inputs, xc_value_and_grads
    rng = np.random.default_rng(h + layers)
    sym, xyz = geometry.water(rng)
    # rows a multiple of 64 but not of 128, so that the last row tile of the larger tilings is ragged
    mol = molecule_from_geometry(sym, xyz, "sto-3g", 0, npts_align=64)
    if mol.npts_pad % 128 == 0:
        mol = molecule_from_geometry(sym, xyz, "sto-3g", 0, npts_align=mol.npts_pad + 64)
    assert mol.npts_pad % 128 == 64
    f = NeuralFunctional(MLPSpec(nc=6, h=h, n_hidden=layers, nd=4))
    theta = f.init(seed=h)
    theta = theta + 0.05 * torch.as_tensor(rng.normal(size=theta.shape), device="cuda")
    direction = torch.as_tensor(rng.normal(size=(2, mol.nao, mol.nao)), device="cuda") * 0.1
    direction = direction + direction.transpose(1, 2)
    g = torch.as_tensor(0.7, dtype=torch.float64, device="cuda")
    ao, gr, d2 = eval_ao(mol.basis, mol.grid.coords.cpu().numpy())
    inp = to_inputs(ao, gr, d2, mol.grid.weights.cpu().numpy())
    spec = OSpec(6, h, layers, 4)
    D0, th0 = mol.rdm1.cpu().numpy(), theta.cpu().numpy()
    E0, gD0, gth0 = xc_value_and_grads("neural_b3lyp", inp, D0, th0, spec)
    _, _, hD0, hth0 = xc_hvp("neural_b3lyp", inp, D0, th0, spec, direction.cpu().numpy(), 0.7)
    D = mol.rdm1.detach().clone().requires_grad_(True)
    th = theta.detach().clone().requires_grad_(True)
    E = f.xc_energy(th, mol, precision, rdm1=D)
    gD, gth = torch.autograd.grad(E, [D, th])
    E2, V = XCEnergyVxcFn.apply(D, th, f.plan(mol, precision))
    hD, hth = torch.autograd.grad([E2, V], [D, th], [g, direction])
    tD, tth, th2 = TOL[precision]
    got = (abs(float(E) - E0), _rel(gD.cpu().numpy(), gD0), _rel(gth.cpu().numpy(), gth0),
           _rel(V.detach().cpu().numpy(), gD0), _rel(hD.cpu().numpy(), hD0), _rel(hth.cpu().numpy(), hth0))
    print("  |dE| %.1e dD %.1e dth %.1e V %.1e hD %.1e hth %.1e" % got, flush=True)
    # FP32: the energy of a grid of one FP32 rounding common to all points (a hidden layer's bias), 6e-7 Ha
    assert got[0] <= (1e-9 if precision == "fp64" else 2.0 ** -24 * abs(E0))
    assert 2.0 ** -24 * abs(E0) <= 1e-6
    assert got[1] <= tD and got[3] <= tD
    assert got[2] <= tth
    assert got[4] <= th2 and got[5] <= th2
