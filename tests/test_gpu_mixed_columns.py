"""The mixed form's column solve at the edges of its compiled-in bounds (12,
24, 40, 64, 96, 128 levels, and past the last): the untuned model against the
form that solves on the fly in LDS, and a member of an ensemble, whose tallest
member picks its kernel, against the untuned model, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = ("u", "v", "w", "b", "p")


@pytest.mark.parametrize("nz", [2, 12, 13, 25, 41, 64, 65, 97, 127, 129])
def test_mixed_column_solve_lengths(nz, tmp_path):
    from ps3d_amd import configs
    from ps3d_amd.ensemble import Ensemble
    from ps3d_amd.model import Model
    from ps3d_amd.params import PS3D_MIXED
    print(f"mixed columns of {nz} levels", flush=True)
    kw = dict(lid=True, Avbi=0.0, Kvbi=0.0, precision=PS3D_MIXED)
    prm, fields = configs.random_state(32, 16, nz, seed=43, **kw)
    shape = f"32x16x{nz}:lid:mixed"
    cache = tmp_path / "plan.txt"
    cache.write_text(f"friction_ab {shape} 8\ntendency {shape} 8\nthomas {shape} 32\n"
                     f"fft_plan_x {shape} 0\nfft_plan_y {shape} 0\n")
    state = {}
    for form in ("untuned", "on the fly"):
        m = Model(prm)
        for n, a in fields.items():
            m.f[n][...] = a
        m.push()
        if form == "on the fly":
            m.tune(str(cache), reps=1)
            assert f"thomas {shape} 32" in m.tuning()
        m.run(3)
        m.pull()
        state[form] = {n: m.f[n].copy() for n in NAMES}
        m.close()
    for n in NAMES:
        assert np.isfinite(state["untuned"][n]).all(), n
        assert np.array_equal(state["untuned"][n], state["on the fly"][n]), n
    if nz < 4:   # an ensemble's members have at least four levels
        return
    small, sf = configs.random_state(16, 8, 5, seed=9, **kw)
    ens = Ensemble([prm, small])
    for n in fields:
        ens.set(0, n, fields[n])
        ens.set(1, n, sf[n])
    ens.run(3)
    for n in NAMES:
        assert np.array_equal(ens.get(0, n), state["untuned"][n]), n
    ens.close()
