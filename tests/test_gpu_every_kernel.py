"""Every compiled form of the tiled kernels against the oracle, or against
another form of the same operation, bit for bit: halos 2 to 11, tile sides 8 to
64, both strip heights, first, middle and last launches of a solve, alone and
batched.  They are instances of a few templates, and each is compiled anew:
the wave tiles lean on what the compiler does with their registers
(own_register in csrc/pfs_wave_kernels.h), so none goes untried."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from probabilistic_fluid_simulation_amd import fluid, scenes  # noqa: E402
from probabilistic_fluid_simulation_amd.batch import Batch  # noqa: E402
from probabilistic_fluid_simulation_amd.fluid import VPField  # noqa: E402

from gpu_util import assert_bitexact, gpu_run, oracle_run, to_dev  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset():
    yield
    fluid.set_step_path("auto")
    fluid.set_precise_schedule()


# The step's side of the square tiles, by field; wave tiles of 2 rows a wave
# past side 24, of 4 from (1001, 980) on.
SIDES = {8: (101, 83), 12: (181, 150), 16: (251, 240), 20: (311, 300), 24: (371, 330),
         32: (500, 401), 36: (601, 430), 40: (621, 600), 48: (761, 700), 56: (881, 870),
         64: (1001, 980)}


@pytest.mark.parametrize("side", list(SIDES))
def test_step(orc, side):
    w, h = SIDES[side]
    assert fluid.get_step_side(w, h, 8, True) == side
    s = scenes.random_scene(w, h, w, h, seed=side, dt=0.5, visc=0.15, vel_scale=30.0)
    for k in [*range(1, 12), 16, 17, 18, 19, 20]:
        assert_bitexact(gpu_run(s, 1, iters=k, combined=True), oracle_run(orc, s, 1, iters=k),
                        [f"{n} K={k}" for n in ("vp", "tmp", "image", "itmp")])


@pytest.mark.parametrize("shape", [(521, 403), (1201, 803)], ids=["2-rows", "4-rows"])
def test_step_many_launches(orc, shape):
    """Sweeps in chunks of 10 (first field: tiles leave CUs idle) and of 8."""
    s = scenes.random_scene(*shape, *shape, seed=7, dt=0.5, visc=0.15, vel_scale=30.0)
    for k in [*range(11, 31), 41, 42]:
        assert_bitexact(gpu_run(s, 1, iters=k, combined=True), oracle_run(orc, s, 1, iters=k),
                        [f"{n} K={k}" for n in ("vp", "tmp", "image", "itmp")])


@pytest.mark.parametrize("shape", [(331, 403), (1001, 980)], ids=["2-rows", "4-rows"])
def test_operators(shape):
    """Several sweeps a launch against a launch per sweep."""
    s = scenes.random_scene(*shape, 1, 1, seed=8, dt=0.5, visc=0.15)
    for k in range(5, 32):
        out = []
        for path in ("auto", "per_op"):
            fluid.set_step_path(path)
            a, b = VPField.from_numpy(s.vp), VPField.from_numpy(s.tmp)
            fluid.diffuse(a, b, s.visc, s.dt, k)
            d = a.data.clone(), b.data.clone()
            fluid.computePressure(a, b, s.dt, k)
            out.append((*d, a.data, b.data))
        assert all(torch.equal(p, q) for p, q in zip(*out)), k


def _precise(s, k, chunk, tile):
    fluid.set_precise_schedule(chunk, tile)
    vp, tmp = VPField.from_numpy(s.vp), VPField.from_numpy(s.tmp)
    fluid.simulate_fluid_step_precise(vp, tmp, s.dt, s.visc, max_iters=k, tol=0.0, report=False)
    return vp.data, tmp.data


@pytest.mark.parametrize("chunk", [4, 8])
@pytest.mark.parametrize("shape", [(203, 150), (331, 403), (1201, 803)], ids=["small", "2-rows", "4-rows"])
def test_precise_diffusion(shape, chunk):
    """Square tiles of 16 (tile 16) against wave tiles (tiles 32 and 64), which
    have the same results whatever the launches; one count near the FP64 twin."""
    s = scenes.make_scene(*shape, 4, 4, kind="tg", seed=9, dt=1 / 60, visc=0.1)
    for k in range(1, 2 * chunk + 2):
        want = _precise(s, k, chunk, 16)
        for tile in (32, 64):
            got = _precise(s, k, chunk, tile)
            assert all(torch.equal(p, q) for p, q in zip(got, want)), (k, tile)
    v64, t64 = (torch.from_numpy(a).cuda().double() for a in (s.vp, s.tmp))
    fluid.simulate_fluid_step_f64(v64, t64, s.dt, s.visc, 2 * chunk + 1, 2 * chunk + 1)
    assert float((want[0][..., :2].double() - v64[..., :2]).abs().max() / v64[..., :2].abs().max()) < 2e-6


@pytest.mark.parametrize("shape", [(250, 240), (311, 300), (350, 340), (500, 400), (601, 430), (621, 600),
                                   (761, 700), (881, 870), (1201, 803)],
                         ids=["16", "20", "24", "32", "36", "40", "48", "56", "64"])
def test_precise_pressure_sides(shape):
    """The automatic side of the precision form's pressure against side 16."""
    s = scenes.make_scene(*shape, 4, 4, kind="tg", seed=10, dt=1 / 60, visc=0.1)
    for chunk, k in ((8, 5), (8, 17), (4, 3), (4, 10)):
        want = _precise(s, k, chunk, 16)
        got = _precise(s, k, chunk, 0)
        assert all(torch.equal(p, q) for p, q in zip(got, want)), (chunk, k)


@pytest.mark.parametrize("tile", [16, 32, 64], ids=["t16", "t32", "t64"])
@pytest.mark.parametrize("shape", [(203, 150), (1200, 900)], ids=["2-rows", "4-rows"])
def test_batch(orc, shape, tile):
    """A scene of every sweep count from 1 to 24, each a group of its own."""
    if tile == 16 and shape[0] > 500:
        pytest.skip("square tiles of 16 have one form")
    b = Batch()
    sc = [scenes.random_scene(*shape, *shape, seed=500 + k, dt=0.5, visc=0.15, iters=k, vel_scale=30.0)
          for k in range(1, 25)]
    slots = [b.add(*to_dev(s), s.dt, s.visc, s.iters) for s in sc]
    b.set_tile(tile)
    b.step(2)
    b.sync()
    for slot, s in zip(slots, sc):
        assert_bitexact([t.cpu().numpy() for t in b.buffers(slot)], oracle_run(orc, s, 2),
                        [f"{n} K={s.iters}" for n in ("vp", "tmp", "image", "itmp")])
    b.close()
