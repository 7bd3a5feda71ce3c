"""The tiled stencil kernels at the edges of their tiles and chunks.

The tendency and friction kernels own 64 x 8 columns and march up chunks of
levels whose planes go to LDS in 16-byte loads (4-byte ones where rows do not
start at 16-byte boundaries: FP32 with nx % 4 == 2).  Sizes: the smallest
grid, extents below, at and just past a tile, remainders of a chunk.  FP64
follows the oracle bit for bit; the mixed form stays within the 1e-5 that its
FP32 stencils are allowed elsewhere.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(2, 2, 2), (4, 4, 4), (6, 4, 5), (60, 16, 9), (64, 8, 3), (64, 10, 17), (72, 18, 6), (128, 6, 35)]


def _pair(make, precision=None):
    import oracle
    from ps3d_amd.model import Model
    prm, fields = make
    gpu = Model(prm if precision is None else prm.replace(precision=precision))
    orc = oracle.OracleModel(prm)
    for n, a in fields.items():
        gpu.f[n][...] = a
        orc.f[n][...] = a
    gpu.push()
    return prm, gpu, orc


@pytest.mark.parametrize("lid", [True, False])
@pytest.mark.parametrize("size", SIZES)
def test_fused_step_bitwise(size, lid):
    from ps3d_amd import configs
    nx, ny, nz = size
    if not lid:
        nz += nz % 2
    print(f"steps {nx}x{ny}x{nz} lid={lid}", flush=True)
    prm, gpu, orc = _pair(configs.random_state(nx, ny, nz, lid=lid, Avbi=0.0, Kvbi=0.0))
    gpu.run(4)
    orc.run(4)
    gpu.pull()
    for n in ("u", "v", "w", "b", "p"):
        assert np.array_equal(gpu.f[n], orc.f[n]), n
    gpu.close()
    orc.close()


@pytest.mark.parametrize("size", [(16, 8, 4), (30, 8, 5), (30, 30, 6), (64, 10, 17), (80, 16, 9)])
def test_mixed_step(size):
    from ps3d_amd import configs, diagnose
    from ps3d_amd.params import PS3D_MIXED
    print(f"mixed steps {size}", flush=True)
    prm, gpu, orc = _pair(configs.jets(*size, seed=4), PS3D_MIXED)
    gpu.run(4)
    orc.run(4)
    gpu.pull()
    err = diagnose.compare(gpu.f, {n: orc.f[n] for n in ("u", "v", "w", "b", "p")}, prm)
    for k in ("u", "v", "w", "b"):
        assert err[k] <= 1e-5, (k, err[k])
    gpu.close()
    orc.close()


OPS = {
    "all": {},
    "vertical_only": dict(Ah=0.0, Av=0.0, Kh=0.0, Kv=0.0, Ahbi=0.0, Khbi=0.0),
    "harmonic_and_vertical_of_uvw": dict(Ahbi=0.0, Khbi=0.0, Kh=0.0, Kv=0.0, Kvbi=0.0),
    "biharmonic_of_b": dict(Ah=0.0, Av=0.0, Ahbi=0.0, Avbi=0.0, Kh=0.0, Kv=0.0),
}


@pytest.mark.parametrize("lid", [True, False])
@pytest.mark.parametrize("ops", list(OPS))
@pytest.mark.parametrize("size", [(2, 2, 2), (4, 4, 4), (30, 10, 5), (64, 8, 9), (128, 18, 12)])
def test_friction_block_bitwise(size, ops, lid):
    """The friction operators in their launches (two, where the halo can be
    carried along) against the oracle's single ones, twice in a row, halo
    included -- a halo that is not the interior's image."""
    from ps3d_amd import configs
    nx, ny, nz = size
    if not lid:
        nz += nz % 2
    print(f"friction {nx}x{ny}x{nz} {ops} lid={lid}", flush=True)
    prm, gpu, orc = _pair(configs.random_state(nx, ny, nz, lid=lid, **OPS[ops]))
    rng = np.random.default_rng(3)
    for n in ("u", "v", "w", "b"):
        a = gpu.f[n] + 1e-3 * rng.standard_normal(gpu.f[n].shape)
        gpu.f[n][...] = a
        orc.f[n][...] = a
    gpu.push(["u", "v", "w", "b"])
    for _ in range(2):
        gpu.friction()
        for n in ("u", "v", "w", "b"):
            H, V, Hb, Vb = (prm.Ah, prm.Av, prm.Ahbi, prm.Avbi) if n != "b" else (prm.Kh, prm.Kv, prm.Khbi, prm.Kvbi)
            if H > 0 or V > 0:
                orc.harmonic(n, H, V)
                if n == "w" and lid:
                    orc.f["w"][:, :, nz + 1:] = 0.0   # integrate.f90:63
            if Hb > 0:
                orc.biharmonic_h(n, Hb)
            if Vb > 0:
                orc.biharmonic_v(n, Vb)
                if n == "w" and lid:
                    orc.f["w"][:, :, nz + 1:] = 0.0   # integrate.f90:73
        gpu.pull(["u", "v", "w", "b"])
        for n in ("u", "v", "w", "b"):
            assert np.array_equal(gpu.f[n], orc.f[n]), n
    gpu.close()
    orc.close()


@pytest.mark.parametrize("ops", list(OPS))
def test_steps_with_vertical_friction_bitwise(ops):
    from ps3d_amd import configs
    print(f"steps {ops}", flush=True)
    prm, gpu, orc = _pair(configs.random_state(72, 10, 13, lid=True, **OPS[ops]))
    gpu.run(4)
    orc.run(4)
    gpu.pull()
    for n in ("u", "v", "w", "b", "p"):
        assert np.array_equal(gpu.f[n], orc.f[n]), n
    gpu.close()
    orc.close()


@pytest.mark.parametrize("nz", [4, 12, 13, 24, 25, 41, 63, 65, 97, 127, 129])
def test_column_solve_lengths(nz):
    """The column solve at the edges of its compiled-in bounds (12, 24, 40, 64,
    96, 128 levels, and past the last): FP64 bit for bit like the oracle, alone
    and as a member of an ensemble, whose tallest member picks its kernel."""
    from ps3d_amd import configs
    from ps3d_amd.ensemble import Ensemble
    print(f"columns of {nz} levels", flush=True)
    prm, gpu, orc = _pair(configs.random_state(16, 10, nz, lid=True, Avbi=0.0, Kvbi=0.0))
    small, fields = configs.random_state(16, 8, 5, seed=9, lid=True, Avbi=0.0, Kvbi=0.0)
    ens = Ensemble([prm, small])
    for n in fields:
        ens.set(0, n, orc.f[n])
        ens.set(1, n, fields[n])
    gpu.run(3)
    orc.run(3)
    ens.run(3)
    gpu.pull()
    for n in ("u", "v", "w", "b", "p"):
        assert np.array_equal(gpu.f[n], orc.f[n]), n
        assert np.array_equal(ens.get(0, n), orc.f[n]), n
    ens.close()
    gpu.close()
    orc.close()
