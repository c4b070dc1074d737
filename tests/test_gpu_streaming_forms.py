"""The streaming step against the one-step kernels (which the oracle tests pin),
value for value, in the forms that test_gpu_streaming.py leaves out: every
operator with every edge and boundary mode, walls, lids, inlets and outlets in
the last strip and the last rows, 16-bit storage with inlets and outlets."""
import numpy as np
import pytest

from chemsim_amd import Lattice, Params, capi
from chemsim_amd import workloads as W
from test_gpu_temporal import random_flags

pytestmark = pytest.mark.gpu

EDGES = {"zero": capi.CS_EDGE_ZERO, "periodic": capi.CS_EDGE_PERIODIC}


def values(raw, storage):
    """Stored values as floats, NaN for every NaN pattern."""
    if storage == "f16":
        return raw.view(np.float16)
    if storage == "bf16":
        return (raw.astype(np.uint32) << 16).view(np.float32)
    return raw


def compare(ctx, w, h, storage, p, flags, steps, seed=71):
    rng = np.random.default_rng(seed)
    dt = np.float64 if storage == "f64" else np.float32
    rho = (1 + 0.01 * rng.standard_normal((h, w))).astype(dt)
    u = (0.03 * rng.standard_normal((2, h, w))).astype(dt)
    out = []
    try:
        for k in (capi.CS_TEMPORAL_AUTO, 0):
            capi.call("cs_set_temporal_steps", k)
            with Lattice(ctx, w, h, storage, p, flags) as lat:
                assert lat.temporal_steps() == (8 if k else 1)
                lat.init_equilibrium(rho, u[0], u[1])
                lat.step(steps)
                out.append(values(lat.download_raw(), storage))
    finally:
        capi.call("cs_set_temporal_steps", capi.CS_TEMPORAL_AUTO)
    np.testing.assert_array_equal(out[0], out[1])


def ends(w, h, seed=72):
    """Random walls and lids, but only in the last 140 columns and the last 20 rows
    (the ragged last strips and the last runs of rows)."""
    flags = random_flags(np.random.default_rng(seed), h, w)
    flags[:max(0, h - 20), :max(0, w - 140)] = 0
    return flags


@pytest.mark.parametrize("edge", EDGES)
@pytest.mark.parametrize("mode", ["fluid", "reference", "halfway"])
@pytest.mark.parametrize("storage,coll", [(s, c) for s in ("f32", "f64") for c in ("bgk", "trt", "regularized")] +
                         [("f32dev", "bgk")])
def test_operators_in_every_form(ctx, storage, coll, mode, edge):
    w, h = (1100, 1001) if storage == "f64" else (2003, 2300)
    p = Params(tau=0.7, edge=EDGES[edge], lid_ux=0.02, lid_uy=-0.03,
               boundary=capi.CS_BB_HALFWAY if mode == "halfway" else capi.CS_BB_REFERENCE)
    if coll == "trt":
        p.collision, p.tau_minus = capi.CS_COLL_TRT, 0.9
    elif coll == "regularized":
        p.collision = capi.CS_COLL_REGULARIZED
    compare(ctx, w, h, storage, p, None if mode == "fluid" else ends(w, h), 13)


@pytest.mark.parametrize("mode", ["reference", "halfway"])
@pytest.mark.parametrize("shape", [(101, 30011), (24641, 163), (2001, 1499)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_f32_ends_of_ragged_shapes(ctx, shape, mode):
    """(2001, 1499) with the reference mask takes regions; 24641 leaves one column
    to the last strip."""
    w, h = shape
    if mode == "reference" and shape == (2001, 1499):
        w, h = 2003, 2300
    p = Params(tau=0.62, lid_ux=0.02, lid_uy=-0.03,
               boundary=capi.CS_BB_HALFWAY if mode == "halfway" else capi.CS_BB_REFERENCE)
    compare(ctx, w, h, "f32", p, ends(w, h), 21)


@pytest.mark.parametrize("rounding", [capi.CS_ROUND_NEAREST, capi.CS_ROUND_STOCHASTIC], ids=["nearest", "stochastic"])
@pytest.mark.parametrize("storage", ["bf16", "f16"])
def test_16bit_ends_of_a_ragged_shape(ctx, storage, rounding):
    w, h = 3001, 3003
    p = Params(tau=0.7, boundary=capi.CS_BB_HALFWAY, lid_ux=0.02, lid_uy=-0.03, rounding=rounding, seed=5)
    compare(ctx, w, h, storage, p, ends(w, h), 11)


@pytest.mark.parametrize("rounding", [capi.CS_ROUND_NEAREST, capi.CS_ROUND_STOCHASTIC], ids=["nearest", "stochastic"])
@pytest.mark.parametrize("storage", ["bf16", "f16"])
def test_16bit_channel(ctx, storage, rounding):
    """Zou-He cells followed by the rounding of every level; a lid on one wall."""
    w, h = 101, 30011
    p = Params(tau=0.7, boundary=capi.CS_BB_HALFWAY, inlet_uy=0.05, inlet_ux=0.01, outlet_rho=1.01, lid_uy=0.02,
               rounding=rounding, seed=6)
    flags = np.zeros((h, w), np.uint8)
    flags[:, 0], flags[:, -1] = W.INLET, W.OUTLET
    flags[0, :], flags[-1, :] = W.WALL, W.LID
    flags[200:240, 30:50] = W.WALL
    compare(ctx, w, h, storage, p, flags, 19)


@pytest.mark.parametrize("storage,shape", [("f64", (2100, 1024)), ("f32", (4100, 3001)), ("f32dev", (4100, 3001))],
                         ids=["f64", "f32", "f32dev"])
def test_channel_with_a_lid(ctx, storage, shape):
    """Inlet, outlet, walls, an obstacle and a moving lid, 8-, 4- and one-step launches."""
    w, h = shape
    flags = W.Channel(w=w, h=h, circles=[(h // 2, w // 3, h // 8), (h // 3, w - 90, 40)], re=60.0, u_in=0.05).flags()
    flags[-1, 1:-1] = W.LID
    p = Params(tau=0.62, boundary=capi.CS_BB_HALFWAY, inlet_uy=0.05, outlet_rho=1.0, lid_uy=0.04)
    compare(ctx, w, h, storage, p, flags, 21)


@pytest.mark.parametrize("value", [5, 128, 255])
@pytest.mark.parametrize("at", [0, -1, 1234])
def test_flags_out_of_range_are_refused(ctx, value, at):
    """Any cell, any value above CS_OUTLET; the lattice keeps the flags it had."""
    w, h = 61, 47
    good = ends(w, h)
    bad = good.copy()
    bad.ravel()[at] = value
    p = Params(tau=0.7, boundary=capi.CS_BB_HALFWAY, lid_uy=0.03)
    out = []
    for again in (False, True):
        with Lattice(ctx, w, h, "f32", p, good) as lat:
            lat.init_equilibrium(*W.rest_state(w, h))
            if again:
                with pytest.raises(capi.ChemsimError, match="flag value out of range"):
                    lat.set_flags(bad)
            lat.step(9)
            out.append(lat.download())
    np.testing.assert_array_equal(out[0], out[1])


def test_buffers_above_4_gib(ctx):
    """FP64 strips address rows from 64-bit bases: a population buffer of 4.4e9
    bytes, eight steps in one launch and four in another against twelve one-step
    launches, every cell's density and velocity."""
    w, h = 7800, 7800
    y, x = np.arange(h)[:, None], np.arange(w)[None, :]
    rho = 1 + 0.01 * np.sin(0.013 * y + 0.011 * x)
    ux, uy = 0.03 * np.cos(0.017 * y) * np.sin(0.012 * x), 0.03 * np.sin(0.009 * y) * np.cos(0.014 * x)
    flags = np.zeros((h, w), np.uint8)
    flags[-2:, ::97] = W.WALL
    out = []
    try:
        for k in (capi.CS_TEMPORAL_AUTO, 0):
            capi.call("cs_set_temporal_steps", k)
            with Lattice(ctx, w, h, "f64", Params(tau=0.7, edge=capi.CS_EDGE_PERIODIC), flags) as lat:
                assert lat.temporal_steps() == (8 if k else 1)
                lat.init_equilibrium(rho, ux, uy)
                lat.step(12)
                out.append(lat.moments_f64())
    finally:
        capi.call("cs_set_temporal_steps", capi.CS_TEMPORAL_AUTO)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
