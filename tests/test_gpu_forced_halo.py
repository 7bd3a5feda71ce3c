"""What a forced step's forcing sees of the halo: the one that the reference's
in-place friction leaves (integrate.f90:59-82), where under a rigid lid the
harmonic pass clears w from level nz up, halo points included (:63)."""
import dataclasses

import numpy as np
import pytest

from conftest import interior
from test_gpu_lee_wave import _forcing

pytestmark = pytest.mark.gpu

HARMONIC = dict(Avbi=0.0, Kvbi=0.0)
BIHARMONIC = dict(Ah=0.0, Av=0.0, Kh=0.0, Kv=0.0, Avbi=0.0, Kvbi=0.0)
NAMES = ("u", "v", "w", "b")


@pytest.mark.parametrize("lid", [True, False])
@pytest.mark.parametrize("ops", [HARMONIC, BIHARMONIC, {}], ids=["harmonic", "biharmonic_h", "all"])
@pytest.mark.parametrize("size", [(2, 2, 2), (32, 24, 12), (72, 10, 6)])
def test_hook_sees_the_reference_friction(size, ops, lid):
    """The fields inside a hook, halo included, against the oracle's friction
    operators on the state before the step: two steps, bit for bit."""
    import oracle
    from ps3d_amd import configs
    from ps3d_amd.model import Model
    nx, ny, nz = size
    print(f"hook {nx}x{ny}x{nz} lid={lid} {sorted(ops)}", flush=True)
    prm, fields = configs.random_state(nx, ny, nz, lid=lid, **ops)
    gpu = Model(prm)
    orc = oracle.OracleModel(prm)
    for n, a in fields.items():
        gpu.f[n][...] = a
    gpu.push()
    seen = {}

    def hook(m, itt, tau, stream):
        m.synchronize()
        m.pull(NAMES)
        for n in NAMES:
            seen[n] = m.f[n].copy()

    gpu.set_forcing(hook)
    for step in range(2):
        gpu.pull(NAMES)
        for n in NAMES:
            orc.f[n][...] = gpu.f[n]
        gpu.run(1)
        for n in NAMES:
            H, V, Hb, Vb = ((prm.Ah, prm.Av, prm.Ahbi, prm.Avbi) if n != "b" else
                            (prm.Kh, prm.Kv, prm.Khbi, prm.Kvbi))
            if H > 0 or V > 0:
                orc.harmonic(n, H, V)
                if n == "w" and lid:
                    orc.f["w"][:, :, nz + 1:] = 0.0
            if Hb > 0:
                orc.biharmonic_h(n, Hb)
            if Vb > 0:
                orc.biharmonic_v(n, Vb)
                if n == "w" and lid:
                    orc.f["w"][:, :, nz + 1:] = 0.0
            assert np.array_equal(seen[n], orc.f[n]), (step, n)
    gpu.set_forcing(None)
    gpu.close()
    orc.close()


def _w_above_the_lid(prm, fields, seed):
    """w as a caller may hand it over, not zero at the lid's level"""
    from ps3d_amd import configs
    w = np.zeros(prm.shape, order="F")
    w[2:2 + prm.nx, 2:2 + prm.ny, 2:2 + prm.nz] = 1e-3 * configs.uniform(seed, "w", prm.nx, prm.ny, prm.nz)
    configs.border_exchg(w)
    return {**fields, "w": w}


@pytest.mark.parametrize("size", [(32, 24, 12), (72, 10, 5)])
def test_background_flow_over_w_at_the_lid(size):
    """The background flow's advection of w reads w(nz) along x up to the
    halo: a first state with w(nz) other than zero, against the oracle bit for
    bit, fields and tendency slots."""
    import oracle
    from ps3d_amd import configs
    from ps3d_amd.model import Model
    print(f"background flow, w at the lid, {size}", flush=True)
    prm, fields = configs.random_state(*size, seed=6, lid=True, **HARMONIC)
    fields = _w_above_the_lid(prm, fields, 3)
    ub, bb, force = _forcing(prm)
    gpu = Model(prm)
    orc = oracle.OracleModel(prm)
    for n, a in fields.items():
        gpu.f[n][...] = a
        orc.f[n][...] = a
    gpu.push()
    gpu.set_background_flow(ub, bb)
    gpu.set_body_force(force)
    orc.set_background(ub, bb, force)
    gpu.run(3)
    orc.run(3)
    gpu.pull()
    for n in NAMES + ("p",):
        assert np.array_equal(gpu.f[n], orc.f[n]), n
    for n in ("du", "dv", "dw", "db"):
        for slot in range(3):
            assert np.array_equal(interior(gpu.f[n][..., slot], prm), interior(orc.f[n][..., slot], prm)), (n, slot)
    gpu.close()
    orc.close()


@pytest.mark.parametrize("mixed", [False, True])
def test_forced_members_over_w_at_the_lid(mixed):
    """Forced members from such a state follow single models bit for bit."""
    from ps3d_amd import configs
    from ps3d_amd.ensemble import Ensemble
    from ps3d_amd.model import Model
    from ps3d_amd.params import PS3D_FP64, PS3D_MIXED
    print(f"forced members, w at the lid, mixed={mixed}", flush=True)
    members = []
    for s, seed in (((32, 24, 12), 6), ((16, 16, 16), 8)):
        prm, fields = configs.random_state(*s, seed=seed, lid=True, **HARMONIC)
        members.append((dataclasses.replace(prm, precision=PS3D_MIXED if mixed else PS3D_FP64),
                        _w_above_the_lid(prm, fields, seed)))
    ens = Ensemble([p for p, _ in members])
    for i, (prm, fields) in enumerate(members):
        for n, a in fields.items():
            ens.set(i, n, a)
        ub, bb, force = _forcing(prm, seed=i + 1)
        ens.set_background_flow(i, ub, bb)
        ens.set_body_force(i, force)
    ens.run(4)
    for i, (prm, fields) in enumerate(members):
        m = Model(prm)
        for n, a in fields.items():
            m.f[n][...] = a
        m.push()
        ub, bb, force = _forcing(prm, seed=i + 1)
        m.set_background_flow(ub, bb)
        m.set_body_force(force)
        m.run(4)
        m.pull()
        for n in NAMES + ("p",):
            assert np.array_equal(ens.get(i, n), m.f[n]), (i, n)
        m.close()
    ens.close()
