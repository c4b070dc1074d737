"""The streaming temporally blocked step (k_step_ts) against the CPU oracle,
value for value, on lattices that the built-in choice gives to it: one strip
and very many rows, very wide and flat, and ragged in both directions; zero
and periodic edges; the reference's solid mask; every operator it runs; steps
that leave a 4-step launch and single steps over."""
import numpy as np
import pytest

from chemsim_amd import Lattice, Params, capi
from chemsim_amd import workloads as W
from oracle import pyoracle as O
from test_gpu_temporal import OPERATORS, gpu_params, rand_state, random_flags

pytestmark = pytest.mark.gpu

# (w, h): a part strip; 18 strips of ragged width; a run of rows per wave with one column over
SHAPES = [(101, 30011), (2003, 2300), (24641, 163)]


@pytest.mark.parametrize("edge", [O.EDGE_ZERO, O.EDGE_PERIODIC])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=[f"{w}x{h}" for w, h in SHAPES])
def test_bgk_matches_oracle(ctx, shape, masked, edge):
    w, h = shape
    rng = np.random.default_rng(61)
    f = rand_state(rng, h, w)
    flags = random_flags(rng, h, w) if masked else None
    if masked:
        flags[:, w // 3:] = 0  # strips and rows with and without solid cells
        flags[h // 2:] = 0
    op = O.params(w, h, tau=0.62, edge=edge)
    with Lattice(ctx, w, h, "f32", gpu_params(op), flags) as lat:
        assert lat.temporal_steps() == 8
        lat.upload(f)
        lat.step(21)  # two 8-step launches, one of 4, one step
        np.testing.assert_array_equal(lat.download(), O.run(op, f, 21, flags))


@pytest.mark.parametrize("edge", [O.EDGE_ZERO, O.EDGE_PERIODIC])
@pytest.mark.parametrize("shape", SHAPES, ids=[f"{w}x{h}" for w, h in SHAPES])
def test_halfway_matches_oracle(ctx, shape, edge):
    w, h = shape
    rng = np.random.default_rng(68)
    f = rand_state(rng, h, w)
    flags = random_flags(rng, h, w)
    flags[:, w // 3:] = 0
    flags[h // 2:] = 0
    op = O.params(w, h, tau=0.62, edge=edge, boundary=O.BB_HALFWAY, lid=(0.02, -0.03))
    with Lattice(ctx, w, h, "f32", gpu_params(op), flags) as lat:
        assert lat.temporal_steps() == 8
        lat.upload(f)
        lat.step(13)
        np.testing.assert_array_equal(lat.download(), O.run(op, f, 13, flags))


@pytest.mark.parametrize("storage", ["f32", "f32dev"])
def test_channel_matches_oracle(ctx, storage):
    ch = W.Channel(w=3001, h=1802, circles=[(900, 700, 160), (400, 2000, 90)], re=60.0, u_in=0.05)
    flags = ch.flags()
    op = O.params(ch.w, ch.h, tau=max(ch.tau, 0.55), boundary=O.BB_HALFWAY, inlet=ch.inlet(), outlet_rho=1.0)
    rho, ux, uy = W.rest_state(ch.w, ch.h)
    with Lattice(ctx, ch.w, ch.h, storage, gpu_params(op), flags) as lat:
        lat.init_equilibrium(rho, ux, uy)
        lat.step(20)
        if storage == "f32":
            f0 = O.equilibrium(op, rho, ux, uy).astype(np.float32)
            np.testing.assert_array_equal(lat.download(), O.run(op, f0, 20, flags))
        else:
            g0 = O.equilibrium_dev(op, rho, ux, uy)
            np.testing.assert_array_equal(lat.download_raw(), O.run_devf32(op, g0, 20, flags))


@pytest.mark.parametrize("coll", ["trt", "regularized"])
def test_operators_match_oracle(ctx, coll):
    w, h = SHAPES[1]
    rng = np.random.default_rng(62)
    f = rand_state(rng, h, w)
    flags = random_flags(rng, h, w)
    flags[:, w // 2:] = 0
    op = O.params(w, h, edge=O.EDGE_PERIODIC, **OPERATORS[coll])
    with Lattice(ctx, w, h, "f32", gpu_params(op), flags) as lat:
        lat.upload(f)
        lat.step(9)
        np.testing.assert_array_equal(lat.download(), O.run(op, f, 9, flags))


@pytest.mark.parametrize("edge", [O.EDGE_ZERO, O.EDGE_PERIODIC])
def test_deviations_match_oracle(ctx, edge):
    w, h = SHAPES[1]
    rng = np.random.default_rng(63)
    op = O.params(w, h, tau=0.7, edge=edge)
    rho = (1 + 0.01 * rng.standard_normal((h, w))).astype(np.float32)
    u = (0.03 * rng.standard_normal((2, h, w))).astype(np.float32)
    with Lattice(ctx, w, h, "f32dev", gpu_params(op)) as lat:
        lat.init_equilibrium(rho, u[0], u[1])
        lat.step(12)
        np.testing.assert_array_equal(lat.download_raw(), O.run_devf32(op, O.equilibrium_dev(op, rho, u[0], u[1]), 12))


def test_unusual_densities_match_oracle(ctx):
    """Densities that take the reciprocal's IEEE branch: zero, subnormal, huge
    and all-ones significands beside ordinary ones."""
    w, h = SHAPES[1]
    rng = np.random.default_rng(64)
    f = rand_state(rng, h, w)
    for k, v in enumerate([0.0, 1e-40, 3e37, 2.0 - 2.0 ** -23]):
        f[:, 100 + 40 * k:110 + 40 * k, 200:230] = 0
        f[0, 100 + 40 * k:110 + 40 * k, 200:230] = v
    op = O.params(w, h, tau=0.8, edge=O.EDGE_PERIODIC)
    with Lattice(ctx, w, h, "f32", gpu_params(op)) as lat:
        lat.upload(f)
        lat.step(8)
        np.testing.assert_array_equal(lat.download(), O.run(op, f, 8))


F64_SHAPES = [(1100, 1001), (49, 22001), (65601, 17)]


@pytest.mark.parametrize("edge", [O.EDGE_ZERO, O.EDGE_PERIODIC])
@pytest.mark.parametrize("mode", ["fluid", "reference", "halfway"])
@pytest.mark.parametrize("shape", F64_SHAPES, ids=[f"{w}x{h}" for w, h in F64_SHAPES])
def test_f64_matches_oracle(ctx, shape, mode, edge):
    w, h = shape
    rng = np.random.default_rng(65)
    f = rand_state(rng, h, w).astype(np.float64)
    flags = None
    if mode != "fluid":
        flags = random_flags(rng, h, w)
        flags[:, w // 2:] = 0
        flags[h // 2:] = 0
    kw = dict(boundary=O.BB_HALFWAY, lid=(0.02, -0.03)) if mode == "halfway" else {}
    op = O.params(w, h, tau=0.62, edge=edge, **kw)
    with Lattice(ctx, w, h, "f64", gpu_params(op), flags) as lat:
        assert lat.temporal_steps() == 8
        lat.upload(f)
        lat.step(13)  # 8 steps, 4 steps, one step
        np.testing.assert_array_equal(lat.download(np.float64), O.run(op, f, 13, flags))


@pytest.mark.parametrize("coll", ["trt", "regularized"])
def test_f64_operators_match_oracle(ctx, coll):
    w, h = F64_SHAPES[0]
    rng = np.random.default_rng(66)
    f = rand_state(rng, h, w).astype(np.float64)
    op = O.params(w, h, edge=O.EDGE_ZERO, **OPERATORS[coll])
    with Lattice(ctx, w, h, "f64", gpu_params(op)) as lat:
        lat.upload(f)
        lat.step(8)
        np.testing.assert_array_equal(lat.download(np.float64), O.run(op, f, 8))


def test_f64_channel_matches_one_step(ctx):
    """Inlet, outlet, obstacle and walls: eight steps in one launch equal eight
    one-step launches."""
    ch = W.Channel(w=2100, h=512, circles=[(200, 700, 60)], re=60.0, u_in=0.05)
    p = Params(tau=ch.tau, boundary=capi.CS_BB_HALFWAY, inlet_uy=ch.u_in, outlet_rho=1.0)
    out = []
    try:
        for k in (capi.CS_TEMPORAL_AUTO, 0):
            capi.call("cs_set_temporal_steps", k)
            with Lattice(ctx, ch.w, ch.h, "f64", p, ch.flags()) as lat:
                lat.init_equilibrium(*[a.astype(np.float64) for a in W.rest_state(ch.w, ch.h)])
                lat.step(24)
                out.append(lat.download(np.float64))
    finally:
        capi.call("cs_set_temporal_steps", capi.CS_TEMPORAL_AUTO)
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("edge", [O.EDGE_ZERO, O.EDGE_PERIODIC])
@pytest.mark.parametrize("masked", [None, "reference", "halfway"])
@pytest.mark.parametrize("rounding", [capi.CS_ROUND_NEAREST, capi.CS_ROUND_STOCHASTIC], ids=["nearest", "stochastic"])
@pytest.mark.parametrize("storage", ["bf16", "f16"])
def test_16bit_matches_one_step(ctx, storage, rounding, masked, edge):
    """Every stored value, NaNs and infinities included, of 21 steps (two 8-step
    launches and five single ones) against 21 one-step launches.  A NaN's sign
    and payload are not compared: the one-step kernels with 1 and with 4 cells
    per lane already differ in them."""
    w, h = 3001, 3003
    rng = np.random.default_rng(67)
    rho = (1 + 0.01 * rng.standard_normal((h, w))).astype(np.float32)
    u = (0.03 * rng.standard_normal((2, h, w))).astype(np.float32)
    rho[1000, 1000], rho[2000, 50] = np.nan, 1e8
    flags = random_flags(rng, h, w) if masked else None
    if masked:
        flags[:, w // 3:] = 0
    p = Params(tau=0.7, edge=edge, rounding=rounding, seed=9, lid_uy=0.03,
               boundary=capi.CS_BB_HALFWAY if masked == "halfway" else capi.CS_BB_REFERENCE)
    out = []
    try:
        for k in (capi.CS_TEMPORAL_AUTO, 0):
            capi.call("cs_set_temporal_steps", k)
            with Lattice(ctx, w, h, storage, p, flags) as lat:
                assert lat.temporal_steps() == (1 if k == 0 else 8)
                lat.init_equilibrium(rho, u[0], u[1])
                lat.step(21)
                raw = lat.download_raw()
                nan = np.uint16(0x7FC0 if storage == "bf16" else 0x7E00)
                out.append(np.where((raw & 0x7FFF) > (0x7F80 if storage == "bf16" else 0x7C00), nan, raw))
    finally:
        capi.call("cs_set_temporal_steps", capi.CS_TEMPORAL_AUTO)
    np.testing.assert_array_equal(out[0], out[1])
