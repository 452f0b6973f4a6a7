"""The V_xc build under different chunkings of the same sums: a molecule in a plan of its own and in a
batch plan, whose items have other point chunks and, in FP32, other slabs; and the entry point that tells
its output tile (gdx_xc_autotune), which answers with the one that runs.

Cases: propane def2-SVP (n_pad 96: 2 x 2 tiles) and naphthalene def2-SVP (n_pad 192: 3 x 3), level-1
grids; B3LYP (one spin in a plan of its own, two in the batch) and the neural functional; FP64 and FP32.
Bars between the two: FP64 1e-12 relative, FP32 1e-6 relative.
"""
import ctypes

import numpy as np
import pytest
import torch


def _say(msg):
    print(msg, flush=True)


def _mol(name):
    from graddft_amd.interface import geometry
    from graddft_amd.interface.builder import molecule_from_geometry
    rng = np.random.default_rng(17)
    sym, xyz = geometry.alkane(rng, 3) if name == "propane" else geometry.naphthalene(rng)
    return molecule_from_geometry(sym, xyz, "def2-svp", 1, npts_align=256)


def test_entry_point_answers_with_the_tile_that_runs():
    from graddft_amd import _lib
    lib = _lib.load()
    d = _lib.XCDesc()
    d.npts, d.npts_pad, d.nao, d.nao_pad = 100, 128, 30, 32
    held = ctypes.create_string_buffer(16)   # the pointers are checked, not read
    for precision in (_lib.GDX_FP64, _lib.GDX_FP32, _lib.GDX_BF16X6):
        d.precision = precision
        for asked, rc in ((0, 0), (64, 0), (128, 0), (0, 0), (96, -1)):
            v = ctypes.c_int32(asked)
            assert lib.gdx_xc_autotune(0, ctypes.byref(d), ctypes.addressof(held), ctypes.addressof(held),
                                       ctypes.byref(v)) == rc
            assert v.value == (64 if rc == 0 else asked)


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", ["propane", "naphthalene"])
def test_vxc_chunkings_agree(name, precision):
    from graddft_amd import B3LYP_GRID, MLPSpec, NeuralFunctional
    from graddft_amd.batch import XCBatchPlan
    mol = _mol(name)
    _say(f"case: V_xc alone and in a batch, {name} (n_pad {mol.nao_pad}), {precision}")
    nf = NeuralFunctional(MLPSpec(nc=6, h=32, n_hidden=3, nd=4))
    one = torch.ones(1, dtype=torch.float64, device="cuda")
    tol = 1e-12 if precision == "fp64" else 1e-6
    for f, theta, m in ((B3LYP_GRID, None, mol), (nf, nf.init(seed=2), mol.replace(restricted=False))):
        plan = f.plan(m, precision)
        batch = XCBatchPlan(f, [m], precision, restricted=False)
        out = []
        for p, D in ((plan, m.rdm1.contiguous()), (batch, batch.concat([m.rdm1]))):
            e = torch.empty(1, dtype=torch.float64, device="cuda")
            dD = torch.empty_like(D)
            dth = None if theta is None else torch.empty_like(theta)
            p.forward(D, theta, e)
            p.backward(*((D, theta, one, dD, dth, plan.generation) if p is plan else (theta, one, dD, dth)))
            out.append((e.item(), dD.cpu().numpy().ravel(), None if dth is None else dth.cpu().numpy()))
        batch.close()
        (e1, d1, t1), (e2, d2, t2) = out
        _say(f"  kind {f.kind}: dE {abs(e1 - e2):.2e} dD rel {_rel(d1, d2):.2e}, equal bits: {np.array_equal(d1, d2)}")
        assert not np.array_equal(d1, d2)   # the chunks do differ: otherwise this compares nothing
        assert abs(e1 - e2) <= tol * abs(e2)
        assert _rel(d1, d2) <= tol
        if theta is not None:
            assert _rel(t1, t2) <= tol
