"""GPU parity: the HIP path (through the C ABI) against the oracle, the
reference's golden vectors and size-independent properties."""

import math

import numpy as np
import pytest

from conftest import GOLDEN
from pyradiance_amd import scenes

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def L():
    from pyradiance_amd import _lib
    _lib.lib()
    return _lib


def _ctx(L, rad, builder=None):
    c = L.Context(0)
    c.load_text(rad)
    if builder is not None:
        c.set_bvh_builder(builder)
    c.commit()
    return c


def _rc_params(L, **kw):
    p = L.default_params(True)
    for k, v in kw.items():
        setattr(p, k, v)
    return p


def _sky_mods(L, mf=1):
    m = L.RgModifier()
    m.name, m.bin_kind, m.nbins, m.mf, m.rhs = b"skyglow", 1, scenes.reinhart_nbins(mf), float(mf), 1.0
    m.nrm[:] = (0, 0, -1)
    m.up[:] = (0, 1, 0)
    g = L.RgModifier()
    g.name, g.bin_kind, g.nbins, g.cbin = b"groundglow", 0, 1, 0
    return [m, g]


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_config1_irradiance_matches_reference(L, oracle, seed):
    _say(f"config1 seed {seed}")
    g = np.load(GOLDEN / f"c1_seed{seed}.npz")
    rad, sens, _ = scenes.config1(seed)
    c = _ctx(L, rad)
    p = L.default_params(False)
    p.ambounce, p.dstrsrc, p.srcsizerat = 0, 0.0, 0.0
    c.set_params(p)
    out = c.trace(sens, L.RT_IMM_IRRAD)
    ref = g["values"]
    assert np.abs(out - ref).max() <= 1e-4 * ref.max()
    orc, nr = oracle.Scene(rad).trace(sens, oracle.params(ambounce=0, dstrsrc=0.0, srcsizerat=0.0), 8)
    assert np.abs(out - orc).max() <= 1e-6 * orc.max()
    assert c.last_nrays() == nr          # ray counts: bit-exact
    assert c.last_nrays() == int(g["nrays"])   # the reference's own counter (rt/raytrace.c:606)


def _mixed_scene():
    return ("void plastic m 0 0 5 .5 .5 .5 0 0\n"
            "void glass g 0 0 3 .8 .8 .8\n"
            "m sphere s1 0 0 4 0 0 0 1\n"
            "m bubble s2 0 0 4 3 0 0 0.7\n"
            "m polygon floor 0 0 12 -6 -6 -2 6 -6 -2 6 6 -2 -6 6 -2\n"
            "m polygon tri 0 0 9 -3 -3 0 -1 -3 0 -2 -1 1\n"
            "g polygon pane 0 0 12 -4 2 -1 -2 2 -1 -2 2 1 -4 2 1\n"
            "m ring r1 0 0 8 0 3 0 0 1 0 0.2 1.2\n"
            "m cylinder c1 0 0 7 -3 0 -2 -3 0 2 0.5\n"
            "m tube t1 0 0 7 3 3 -2 3 3 2 0.6\n"
            "m cone k1 0 0 8 0 -3 -2 0 -3 1 1.0 0.2\n"
            "m cup k2 0 0 8 2 -3 -2 2 -3 0 0.1 0.8\n")


@pytest.mark.parametrize("builder", ["sah", "lbvh"])
def test_closest_hit_matches_brute_force(L, oracle, builder):
    _say(f"closest hit, mixed primitives, {builder} tree")
    kind = {"sah": L.BVH_SAH, "lbvh": L.BVH_LBVH}[builder]
    rad = _mixed_scene()
    rng = np.random.default_rng(7)
    n = 4000
    org = rng.uniform(-5, 5, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    rays = np.hstack([org, d])
    prim, t = oracle.Scene(rad).closest(rays)
    # GPU: primary rays into an all-black scene carrying one tracked modifier
    # per primitive would need bins; instead compare through rtrace -i, whose
    # value is non-zero exactly when a primitive is hit under a bright sky.
    sky = "void glow skyglow 0 0 4 1 1 1 0\nskyglow source sky 0 0 4 0 0 1 360\n"
    c = _ctx(L, rad + sky, kind)
    p = L.default_params(False)
    c.set_params(p)
    out = c.trace(rays, 0)
    o2, _ = oracle.Scene(rad + sky).trace(rays, oracle.params(), 0)
    same = np.isclose(out, o2, rtol=1e-6, atol=1e-9).all(1)
    assert same.mean() >= 0.999
    # rays that escape see the sky (value 1), hits on plastic with -ab 0 are black
    escaped = prim < 0
    assert np.allclose(out[escaped], 1.0)


@pytest.mark.parametrize("builder", ["sah", "lbvh"])
def test_first_hit_matches_reference(L, builder):
    """rg_first_hit against rtrace -oLN / -os of the reference: distance,
    unflipped normal and surface for sphere, bubble, polygons, rings,
    cylinders, tubes, cones and cups."""
    _say(f"first hit vs reference, {builder} tree")
    g = np.load(GOLDEN / "prims.npz")
    c = _ctx(L, str(g["scene"]), {"sah": L.BVH_SAH, "lbvh": L.BVH_LBVH}[builder])
    t, nrm, prim = c.first_hit(g["rays"])
    hit = g["t"] < 1e9
    assert np.array_equal(prim >= 0, hit)
    assert np.allclose(t[hit], g["t"][hit], rtol=1e-5, atol=0)
    assert np.all(t[~hit] == 1e10)
    assert np.allclose(nrm, g["normal"], rtol=0, atol=2e-6)
    names = np.array([ln.split()[2] for ln in str(g["scene"]).splitlines() if ln.split()[1] not in
                      ("plastic", "glass")])
    assert np.array_equal(np.where(prim >= 0, names[np.maximum(prim, 0)], "*"), g["name"])
    c.close()


def test_local_sources_metal_trans_glass_match_reference(L):
    """Deterministic shading against the reference rtrace: polygon, sphere
    and ring light sources, a proximity glow, metal, trans, glass and
    mirror-smooth metal (-ab 0 -dj 0 -ds 0 -dt 0 -st 1), radiance and -I."""
    _say("shading vs reference")
    g = np.load(GOLDEN / "shading.npz")
    c = _ctx(L, str(g["scene"]))
    p = L.default_params(False)
    p.ambounce, p.dstrsrc, p.srcsizerat, p.specthresh, p.maxdepth, p.minweight = 0, 0.0, 0.0, 1.0, 8, 1e-4
    p.ambval[:] = (0.0, 0.0, 0.0)
    c.set_params(p)
    v = c.trace(g["rays"], 0)
    assert np.allclose(v, g["values"], rtol=1e-5, atol=1e-9)
    e = c.trace(g["sensors"], L.RT_IMM_IRRAD)
    assert np.allclose(e, g["irradiance"], rtol=1e-5, atol=1e-9)
    c.close()


def test_rcontrib_matches_oracle_same_samples(L, oracle):
    _say("rcontrib -ab 2 vs oracle")
    rng = np.random.default_rng(1)
    room = scenes.Room()
    rad = scenes.room_rad(room) + scenes.furniture_rad(rng, 5, room, 1, 1) + scenes.sky_rad((1, 1, 1), (1, 1, 1))
    pts = np.array([[1.0, 1.0, 0.8, 0, 0, 1], [3.0, 2.0, 0.8, 0, 0, 1], [5.0, 3.0, 1.5, 0, 0, 1],
                    [3.0, 0.5, 1.5, 0, -1, 0]])
    rays = np.repeat(pts, 8, axis=0)
    mods = _sky_mods(L)
    c = _ctx(L, rad)
    c.set_params(_rc_params(L, ambounce=2, ambdiv=256, minweight=1e-3, seed=3))
    out = c.contrib(rays, mods, 1, L.RT_IMM_IRRAD)
    omods = [oracle.mod("skyglow", 1, 145), oracle.mod("groundglow", 0, 1)]
    orc, nr = oracle.Scene(rad).contrib(rays, oracle.params(ambounce=2, ambdiv=256, minweight=1e-3, dstrsrc=0.9,
                                                            specthresh=0.02, seed=3), omods, 1, 8)
    # identical samples: totals agree tightly, entries agree except where a
    # sample's path diverged on an FP32-vs-FP64 edge decision
    assert np.allclose(out.sum(1), orc.sum(1), rtol=2e-3)
    close = np.isclose(out, orc, rtol=1e-4, atol=1e-7)
    assert close.mean() > 0.99
    assert abs(c.last_nrays() - nr) <= 0.002 * nr


def test_rtrace_ambient_matches_oracle(L, oracle):
    _say("rtrace -I -ab 1 with sun and sky vs oracle")
    rad, sens, _ = scenes.config1(0)
    c = _ctx(L, rad)
    p = L.default_params(False)
    p.ambounce, p.ambdiv, p.dstrsrc = 1, 128, 0.5
    p.seed = 9
    c.set_params(p)
    out = c.trace(sens, L.RT_IMM_IRRAD)
    orc, nr = oracle.Scene(rad).trace(sens, oracle.params(ambounce=1, ambdiv=128, dstrsrc=0.5, seed=9), 8)
    assert np.allclose(out.sum(1), orc.sum(1), rtol=1e-3, atol=1e-6)


def test_uniform_sky_pi(L):
    _say("uniform sky = pi")
    c = _ctx(L, scenes.sky_rad((1, 1, 1), ground=(1, 1, 1)))
    c.set_params(_rc_params(L, ambounce=1, ambdiv=4096, minweight=1e-4))
    rays = np.array([[0, 0, 1.0, 0, 0, 1], [5, 5, 0, 0, 0, 1], [0, 0, 0, 1, 0, 0]], float)
    out = c.contrib(rays, _sky_mods(L), 1, L.RT_IMM_IRRAD)
    assert np.allclose(out[:, 0::3].sum(1), math.pi, rtol=1e-6)
    assert np.allclose(out[2, -3], math.pi / 2, rtol=0.02)    # half the hemisphere is ground


@pytest.mark.parametrize("mf", [1, 2, 4])
def test_bins_match_reference(L, mf):
    _say(f"Reinhart MF {mf} bins")
    g = np.load(GOLDEN / "bins_reinhart.npz")
    d = g["dirs"]
    c = _ctx(L, "void glow skyglow 0 0 4 1 1 1 0\nskyglow source sky 0 0 4 0 0 1 180\n")
    c.set_params(_rc_params(L, ambounce=0))
    out = c.contrib(np.hstack([np.zeros_like(d), d]), _sky_mods(L, mf)[:1], 1, 0)
    v = out[:, 0::3]
    got = np.where(v.max(1) > 0.5, v.argmax(1), -1)
    assert np.array_equal(got, g[f"mf{mf}"])


def test_klems_bins_match_reference(L):
    _say("Klems bins")
    g = np.load(GOLDEN / "bins_klems.npz")
    d = g["dirs"]
    c = _ctx(L, "void glow skyglow 0 0 4 1 1 1 0\nskyglow source sky 0 0 4 0 0 1 360\n")
    c.set_params(_rc_params(L, ambounce=0))
    for name, nrm, up in (("kbinS", (0, 1, 0), (0, 0, 1)), ("kbinD", (0, 0, -1), (0, 1, 0))):
        m = L.RgModifier()
        m.name, m.bin_kind, m.nbins, m.rhs = b"skyglow", 2, 145, 1.0
        m.nrm[:], m.up[:] = nrm, up
        out = c.contrib(np.hstack([np.zeros_like(d), d]), [m], 1, 0)[:, 0::3]
        got = np.where(out.max(1) > 0.5, out.argmax(1), -1)
        assert np.array_equal(got, g[name]), name


def test_sah_tree_independent_of_host_threads(L, monkeypatch):
    """The host SAH build splits the top of the tree on one thread and hands
    the subtrees below to the host threads; every range is split and
    numbered as the one-thread build does it, so first hits (distance,
    normal, primitive) agree bit for bit whatever the thread count.  150k
    random triangles, above the size the build starts threads at."""
    _say("sah threads")
    rng = np.random.default_rng(5)
    n = 150_000
    c0 = rng.random((n, 3)) * 20.0
    parts = ["void plastic m 0 0 5 .5 .5 .5 0 0"]
    for i in range(n):
        v = c0[i] + rng.normal(0, 0.15, (3, 3))
        parts.append(f"m polygon t{i} 0 0 9 " + " ".join(f"{x:.9g}" for x in v.ravel()))
    rad = "\n".join(parts) + "\n"
    rays = np.hstack([rng.random((20_000, 3)) * 20.0, rng.normal(0, 1, (20_000, 3))])
    out = []
    for threads in ("1", "16"):
        monkeypatch.setenv("RG_BVH_THREADS", threads)
        c = _ctx(L, rad, L.BVH_SAH)
        out.append(c.first_hit(rays))
        c.close()
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)
    assert (out[0][2] >= 0).mean() > 0.3


def test_dcsky_against_fp64(L):
    _say("dcsky")
    rng = np.random.default_rng(0)
    for (M, K, N) in [(37, 19, 51), (250, 146, 877), (64, 2305, 96), (300, 77, 130), (129, 33, 257),
                      (513, 160, 1203), (130, 64, 2048)]:
        A = rng.random((M, K, 3), dtype=np.float32)
        B = rng.lognormal(0, 1, (K, N, 3)).astype(np.float32)
        ref = np.einsum("mkc,knc->mnc", A.astype(np.float64), B.astype(np.float64), optimize=True)
        c32 = L.dcsky(A, B, 0)
        e32 = np.abs(c32 - ref).max() / np.abs(ref).max()
        assert e32 < 1e-5, (M, K, N, e32)
        # automatic, direct, LDS-staged and (K <= 160) short-K split-BF16 products
        for mode in ((1, 2, 3, 4) if K <= 160 else (1, 2, 3)):
            cbf = L.dcsky(A, B, mode)
            ebf = (np.abs(cbf - ref) / np.abs(ref)).max()
            assert ebf < 1e-4, (M, K, N, mode, ebf)


def test_config2_full_size_properties(L):
    """Full config-2 workload: every record is a valid irradiance split
    (non-negative, total <= pi per unit sky), repeatable for a fixed seed."""
    _say("config2 full size")
    rad, sens = scenes.config2(0)
    c = _ctx(L, rad)
    assert c.info()["primitives"] == 8 + 200 * 6 * 21 - 1
    c.set_params(_rc_params(L, ambounce=4, ambdiv=4096, minweight=1e-4, seed=1))
    out = c.contrib(sens, _sky_mods(L), 1, L.RT_IMM_IRRAD)
    n1 = c.last_nrays()
    assert out.shape == (2500, 438)
    assert (out >= 0).all()
    tot = out.sum(1) / 3
    assert (tot <= math.pi * 1.02).all() and tot.max() > 0.01
    out2 = c.contrib(sens, _sky_mods(L), 1, L.RT_IMM_IRRAD)
    assert c.last_nrays() == n1
    assert np.allclose(out, out2, rtol=1e-9, atol=1e-15)
    assert n1 > 2500 * 4096


def test_contrib_on_device_buffers_matches_host_buffers(L):
    """rg_contrib_device (rays and output resident on the GPU) gives the same
    records as rg_contrib for the same seed, also when records average
    several rays."""
    import torch
    _say("contrib on device buffers")
    rad, sens = scenes.config2(2)
    c = _ctx(L, rad)
    c.set_params(_rc_params(L, ambounce=2, ambdiv=256, minweight=1e-3, seed=5))
    mods = _sky_mods(L)
    for accum in (1, 3):
        rays = np.repeat(sens[:300], accum, axis=0)
        host = c.contrib(rays, mods, accum, L.RT_IMM_IRRAD)
        n_host = c.last_nrays()
        d_rays = torch.from_numpy(rays).cuda()
        d_out = torch.full(host.shape, -1.0, dtype=torch.float64, device="cuda")
        c.contrib_device(d_rays.data_ptr(), rays.shape[0] // accum, mods, d_out.data_ptr(), accum, L.RT_IMM_IRRAD)
        assert c.last_nrays() == n_host
        assert np.allclose(d_out.cpu().numpy(), host, rtol=1e-12, atol=1e-15)
    c.close()


def test_config5_full_size_properties(L):
    """Full config-5 scene (10-storey office, 2,495,700 quads = 5 M
    triangles) under a Reinhart MF:4 sky (2305 + 1 bins), -ab 5 -ad 8192
    -lw 5e-5, on every 100th of its 20,000 sensors: every record a valid
    irradiance split (non-negative, total <= pi per unit sky), the four-wide
    and the binary walks agree, and the rays exceed the first bounce."""
    _say("config5 full size")
    rad, sens = scenes.config5(0)
    c = _ctx(L, rad)
    del rad
    assert c.info()["primitives"] == 2_495_700
    sub = sens[::100]
    mods = _sky_mods(L, 4)
    c.set_params(_rc_params(L, ambounce=5, ambdiv=8192, minweight=5e-5, seed=3))
    out = c.contrib(sub, mods, 1, L.RT_IMM_IRRAD)
    n1 = c.last_nrays()
    assert out.shape == (200, 3 * 2306)
    assert (out >= 0).all()
    tot = out.sum(1) / 3
    assert (tot <= math.pi * 1.02).all() and tot.max() > 0.01
    assert n1 > 200 * 8192
    c.set_tuning(wide=0)
    out2 = c.contrib(sub, mods, 1, L.RT_IMM_IRRAD)
    assert c.last_nrays() == n1
    assert np.allclose(out, out2, rtol=1e-9, atol=1e-15)
    c.close()


def test_sah_and_lbvh_trees_give_the_same_contributions(L):
    """The two spatial indexes change only the traversal order: closest hits,
    and so every sample, agree (up to coincident-surface ties)."""
    _say("config2 subset, SAH vs LBVH")
    rad, sens = scenes.config2(0)
    sens = sens[::5]
    outs, nrs = [], []
    for kind in (L.BVH_SAH, L.BVH_LBVH):
        c = _ctx(L, rad, kind)
        c.set_params(_rc_params(L, ambounce=2, ambdiv=512, minweight=1e-3, seed=5))
        outs.append(c.contrib(sens, _sky_mods(L), 1, L.RT_IMM_IRRAD))
        nrs.append(c.last_nrays())
        c.close()
    assert abs(nrs[0] - nrs[1]) <= 1e-4 * nrs[0]
    close = np.isclose(outs[0], outs[1], rtol=1e-6, atol=1e-12).all(1)
    assert close.mean() >= 0.99
    assert np.allclose(outs[0].sum(), outs[1].sum(), rtol=1e-3)


def test_persistent_and_per_thread_traversal_agree(L):
    """The persistent dynamic-fetch kernel (four-wide and binary walks) and
    the one-ray-per-thread kernel trace the same rays: same ray count, same
    contributions (up to the order of the FP64 additions), also with small
    refill thresholds and windows that split the generations."""
    _say("persistent vs per-thread traversal")
    rad, sens = scenes.config2(1)
    sens = sens[::5]
    res = []
    for kw in ({"trace_kernel": 0}, {"trace_kernel": 1}, {"trace_kernel": 1, "wide": 0},
               {"trace_kernel": 1, "refill": 1, "window": 50000},
               {"trace_kernel": 1, "refill": 64, "blocks_per_cu": 1, "wide": 0}):
        c = _ctx(L, rad)
        c.set_tuning(**kw)
        c.set_params(_rc_params(L, ambounce=2, ambdiv=512, minweight=1e-3, seed=7))
        res.append((c.contrib(sens, _sky_mods(L), 1, L.RT_IMM_IRRAD), c.last_nrays()))
        c.close()
    for out, nr in res[1:]:
        assert nr == res[0][1]
        assert np.allclose(out, res[0][0], rtol=1e-12, atol=1e-15)


def test_python_api_bytes(L, tmp_path):
    _say("python API")
    from pyradiance_amd import Rcontrib, rtrace
    rad, sens, _ = scenes.config1(0)
    f = tmp_path / "room.rad"
    f.write_text(rad)
    inp = "\n".join(" ".join(f"{v:.10g}" for v in r) for r in sens[:5]).encode()
    out = rtrace(inp, f, irradiance=True, params=["-ab", "0", "-dj", "0", "-ds", "0"])
    head, _, body = out.partition(b"\n\n")
    assert head.startswith(b"#?RADIANCE") and b"FORMAT=ascii" in head
    lines = body.decode().strip("\n").split("\n")
    assert len(lines) == 5 and all(len(ln.split("\t")) == 4 for ln in lines)
    g = np.load(GOLDEN / "c1_seed0.npz")
    vals = np.array(body.split(), float).reshape(-1, 3)
    assert np.allclose(vals, g["values"][:5], rtol=1e-5, atol=1e-9)
    raw = rtrace(inp, f, header=False, irradiance=True, outform="f", params=["-ab", "0", "-dj", "0", "-ds", "0"])
    assert len(raw) == 5 * 3 * 4
    sky = tmp_path / "sky.rad"
    sky.write_text(scenes.sky_rad((1, 1, 1), (1, 1, 1)))
    rc = Rcontrib(b"0 0 0 0 0 1\n", sky, params=["-I+", "-ab", "1", "-ad", "1024", "-lw", "1e-4", "-h"])
    rc.add_modifier(modifier="skyglow", calfile="reinhartb.cal", param="MF=1", nbins="Nrbins", binv="rbin")
    rc.add_modifier(modifier="groundglow", nbins="1", binv="0")
    res = rc()
    v = np.array(res.split(), float)
    assert v.size == 146 * 3 and abs(v[0::3].sum() - math.pi) < 1e-4


def test_errors_are_status_codes(L):
    c = L.Context(0)
    with pytest.raises(RuntimeError, match="undefined modifier"):
        c.load_text("nosuch polygon p 0 0 9 0 0 0 1 0 0 0 1 0\n")
    c2 = L.Context(0)
    c2.load_text("void mirror mm 0 0 3 1 1 1\nmm polygon p 0 0 9 0 0 0 1 0 0 0 1 0\n")
    with pytest.raises(RuntimeError, match="not supported"):
        c2.commit()


def test_batched_scenes_match_individual_runs(L):
    """Several scenes in one wavefront give each scene's standalone result
    (scene k of a batch draws the samples of seed + k)."""
    _say("batched scenes vs individual")
    sc = scenes.config3(5, nscenes=4, prims=(600, 6000), sensors=(20, 200))
    ctxs = [_ctx(L, rad) for rad, _ in sc]
    p = _rc_params(L, ambounce=2, ambdiv=256, minweight=1e-3, seed=21)
    ctxs[0].set_params(p)
    mods = _sky_mods(L)
    res = L.contrib_batch(ctxs, [s for _, s in sc], mods, 1, L.RT_IMM_IRRAD)
    nb = ctxs[0].last_nrays()
    total = 0
    # fresh contexts: each first call counts its scene's shadow-cache rays,
    # as the batch did
    ctxs = [_ctx(L, rad) for rad, _ in sc]
    for k, (c, (_, sens)) in enumerate(zip(ctxs, sc)):
        p.seed = 21 + k
        c.set_params(p)
        single = c.contrib(sens, mods, 1, L.RT_IMM_IRRAD)
        total += c.last_nrays()
        assert single.shape == res[k].shape
        # coefficient bins accumulate in fixed point: bit for bit
        assert np.array_equal(single, res[k]), k
    assert nb == total


def test_bins_repeat_bit_for_bit_across_launch_shapes(L):
    """rcontrib coefficients add up in 64-bit fixed point, so the order in
    which deposits arrive (launch shape, persistent refill, window size,
    child order, windows in flight) leaves every record unchanged to the
    last bit."""
    _say("bin accumulation: identical across launch shapes")
    rad, sens = scenes.config2(0, nboxes=40)
    sens = sens[::10]
    c = _ctx(L, rad)
    c.set_params(_rc_params(L, ambounce=2, ambdiv=512, minweight=1e-3, seed=5))
    mods = _sky_mods(L)
    outs = []
    for shape in (dict(trace_kernel=1, refill=16, window=1 << 21), dict(trace_kernel=1, refill=48, window=1 << 12),
                  dict(trace_kernel=0, window=1 << 14, child_order=0),
                  dict(trace_kernel=1, refill=32, window=1 << 13, child_order=1, inflight=2)):
        c.set_tuning(**shape)
        outs.append(c.contrib(sens, mods, 1, L.RT_IMM_IRRAD))
    for o in outs[1:]:
        assert np.array_equal(outs[0], o)
    assert outs[0].sum() > 0
    c.close()


def test_batched_rtrace_config1_sun_positions(L):
    """Config 1 for many sun positions in one launch equals the reference
    fixtures scene by scene (deterministic at -ab 0 -dj 0)."""
    _say("batched rtrace, config-1 suns")
    ctxs, rays = [], []
    for seed in range(3):
        rad, sens, _ = scenes.config1(seed)
        ctxs.append(_ctx(L, rad))
        rays.append(sens)
    p = L.default_params(False)
    p.ambounce, p.dstrsrc, p.srcsizerat = 0, 0.0, 0.0
    ctxs[0].set_params(p)
    res = L.trace_batch(ctxs, rays, L.RT_IMM_IRRAD)
    for seed in range(3):
        ref = np.load(GOLDEN / f"c1_seed{seed}.npz")["values"]
        assert np.abs(res[seed] - ref).max() <= 1e-4 * ref.max()


def test_empty_and_smallest_inputs(L, tmp_path):
    """Zero rays, zero records and 1 x 1 x 1 products are valid calls: empty
    results, no error (the reference programs print only their header for an
    empty ray stream)."""
    import torch
    from pyradiance_amd import rt
    _say("empty and smallest inputs")
    rad, _ = scenes.config2(0, nboxes=10)
    c = _ctx(L, rad)
    assert c.trace(np.zeros((0, 6)), L.RT_IMM_IRRAD).shape == (0, 3)
    t, nrm, prim = c.first_hit(np.zeros((0, 6)))
    assert t.shape == (0,) and prim.shape == (0,)
    mods = _sky_mods(L)
    c.set_params(_rc_params(L, ambounce=1, ambdiv=64, seed=1))
    assert c.contrib(np.zeros((0, 6)), mods, 1, L.RT_IMM_IRRAD).shape == (0, 438)
    assert c.last_nrays() == 0
    c.contrib_device(0, 0, mods, 0, 1, L.RT_IMM_IRRAD)
    assert c.last_nrays() == 0
    # one ray, one record, records of several rays
    one = np.array([[3.0, 2.0, 0.8, 0.0, 0.0, 1.0]])
    assert c.trace(one, L.RT_IMM_IRRAD).shape == (1, 3)
    r3 = c.contrib(np.repeat(one, 3, axis=0), mods, 3, L.RT_IMM_IRRAD)
    assert r3.shape == (1, 438) and (r3 >= 0).all()
    c.close()
    # the Python entry points on an empty ray stream
    (tmp_path / "room.rad").write_text(rad)
    out = rt.rtrace(b"", tmp_path / "room.rad", params=["-ab", "0"])
    assert out.endswith(b"\n\n") and out.startswith(b"#?RADIANCE")
    assert rt.rtrace(b"", tmp_path / "room.rad", header=False) == b""
    # 1 x 1 x 1 and 1 x K x 1 products
    A = np.full((1, 1, 3), 2.0, dtype=np.float32)
    B = np.full((1, 1, 3), 3.0, dtype=np.float32)
    for mode in (0, 1, 2, 3, 4):
        assert np.allclose(L.dcsky(A, B, mode), 6.0, rtol=1e-5)
    A = np.ones((1, 300, 3), dtype=np.float32)
    B = np.ones((300, 1, 3), dtype=np.float32)
    for mode in (1, 3):
        assert np.allclose(L.dcsky(A, B, mode), 300.0, rtol=1e-5)


def test_child_order_changes_only_the_order(L):
    """Handing a spawn's hemisphere children out in 8 x 8 blocks of strata
    instead of by stratum row changes which rays share a wavefront, not
    which samples are drawn: same records (to summation order), same rays."""
    _say("child order: blocks of strata vs rows")
    rad, sens = scenes.config2(0)
    c = _ctx(L, rad)
    c.set_params(_rc_params(L, ambounce=3, ambdiv=1024, minweight=1e-3, seed=8))
    res = []
    for order in (0, 1):
        c.set_tuning(child_order=order)
        res.append((c.contrib(sens[::25], _sky_mods(L), 1, L.RT_IMM_IRRAD), c.last_nrays()))
    c.close()
    assert res[0][1] == res[1][1]
    assert np.allclose(res[0][0], res[1][0], rtol=1e-9, atol=1e-15)


@pytest.fixture(scope="module")
def mirror_room(L):
    """A room whose trees hold every kind of child at once: hemispheres,
    single rays, mirror and pane continuations and shadow rays of a sun."""
    room = scenes.Room()
    rad = (scenes.room_rad(room) + "void metal mirror_mat\n0\n0\n5 .8 .8 .8 .9 0\n"
           + scenes.box_quads_rad("mirror_mat", "mbox", (2.0, 1.5, 0.01), (3.1, 2.4, 1.7), 2, 2)
           + scenes.furniture_rad(np.random.default_rng(3), 6, room)
           + scenes.sun_rad(scenes.sun_direction(35.0, 170.0)) + scenes.sky_rad((1, 1, 1), ground=(1, 1, 1)))
    sens = np.zeros((600, 6))
    rng = np.random.default_rng(9)
    sens[:, 0], sens[:, 1], sens[:, 2] = rng.uniform(0.1, 5.9, 600), rng.uniform(0.1, 3.9, 600), 0.8
    sens[:, 5] = 1.0
    c = _ctx(L, rad)
    c.set_params(_rc_params(L, ambounce=3, ambdiv=96, minweight=1e-3, seed=4))
    mods = _sky_mods(L)
    full = c.contrib(sens, mods, 1, L.RT_IMM_IRRAD)
    yield c, mods, sens, full, c.last_nrays()
    c.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 129, 255, 256, 257, 600])
@pytest.mark.parametrize("window", [1 << 10, 1 << 15, 1 << 24])
def test_records_do_not_depend_on_the_batch_around_them(L, mirror_room, n, window):
    """A sensor's samples follow from its index alone, so its record is the
    same bit for bit however many sensors share the call and however the
    rays fall into segments, chunks and windows (window 1024 splits every
    generation, 2^15 some of them, 2^24 none)."""
    _say(f"records of {n} sensors, window {window}")
    c, mods, sens, full, _ = mirror_room
    c.set_tuning(window=window)
    got = c.contrib(sens[:n], mods, 1, L.RT_IMM_IRRAD)
    c.set_tuning(window=1 << 24)
    assert np.array_equal(got, full[:n])


@pytest.mark.parametrize("shape", [dict(window=1 << 10), dict(window=1 << 12, inflight=2), dict(trace_kernel=0),
                                   dict(refill=1), dict(refill=64, blocks_per_cu=1)])
def test_ray_count_does_not_depend_on_the_launch_shape(L, mirror_room, shape):
    """Every admitted ray is traced and counted once, whichever windows,
    wavefronts and units of work it falls into."""
    _say(f"ray count at {shape}")
    c, mods, sens, full, nrays = mirror_room
    c.set_tuning(**shape)
    got = c.contrib(sens, mods, 1, L.RT_IMM_IRRAD)
    count = c.last_nrays()
    c.set_tuning(window=1 << 24, inflight=1, trace_kernel=1, refill=16, blocks_per_cu=4)
    again = c.contrib(sens, mods, 1, L.RT_IMM_IRRAD)
    assert np.array_equal(got, full) and np.array_equal(again, full)
    assert count == c.last_nrays()


def test_path_records_follow_their_rays_through_every_window(L):
    """The adjoint's gradient with every generation split into windows of
    1,024 children equals the one of whole generations (FP64 atomics: to
    summation order)."""
    from pyradiance_amd.adjoint import DiffScene
    _say("adjoint over split windows")
    rad, sens, groups = scenes.config4(nsensors=40)
    sc = DiffScene(rad, sens, groups, _sky_mods(L), _rc_params(L, ambounce=2, ambdiv=128, minweight=1e-3, seed=2))
    rng = np.random.default_rng(1)
    dlde, sky = rng.normal(size=(40, 3)), rng.uniform(0.5, 2.0, (146, 3))
    res = []
    for shape in (dict(window=1 << 24), dict(window=1 << 10), dict(window=1 << 11, inflight=2)):
        sc.ctx.set_tuning(**shape)
        res.append(sc.adjoint(dlde, sky))
    sc.close()
    scale = np.abs(res[0]).max()
    assert scale > 0
    for g in res[1:]:
        assert np.abs(g - res[0]).max() <= 1e-11 * scale


@pytest.mark.parametrize("m,k,n", [(1, 257, 1), (127, 288, 129), (128, 289, 128), (129, 320, 127), (300, 2306, 4),
                                   (33, 384, 1157), (130, 161, 260), (2049, 352, 2051), (1500, 578, 1408)])
def test_long_k_product_at_tile_and_split_edges(L, m, k, n):
    """The ring form of the K > 160 product (mode 3, whatever the size would
    choose): tile remainders in both directions, K steps that do and do not fill a group of four, K shared by
    many blocks and by one, sky columns that do and do not allow 16-byte
    stores.  Operands are positive, so every term's relative error bounds the
    sum's: the dropped lo x lo part and the rounding of lo are each at most
    2^-16 of a term (hi and lo hold 8 bits each), twice over both operands,
    and the FP32 sum adds at most K 2^-24."""
    import torch
    _say(f"long-K product {m} x {k} x {n}")
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    a = torch.rand((m, k, 3), generator=g, device="cuda")
    b = torch.exp(torch.randn((k, n, 3), generator=g, device="cuda"))
    c = torch.full((m, n, 3), float("nan"), device="cuda")
    torch.cuda.synchronize()
    L.dcsky_device(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, k, n, 3)
    for ch in range(3):
        ref = a[:, :, ch].double().contiguous() @ b[:, :, ch].double().contiguous()
        rel = ((c[:, :, ch].double() - ref) / ref).abs().max().item()
        assert rel <= 3 * 2.0 ** -16 + k * 2.0 ** -24, (ch, rel)


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (15, 32, 33), (16, 33, 31), (127, 64, 2048), (129, 65, 130), (128, 146, 128),
                                   (257, 160, 1001), (2500, 146, 97), (130, 20, 8192), (130, 64, 8196),
                                   (257, 96, 6148), (200, 128, 8196), (300, 146, 8196), (2500, 146, 1000),
                                   (129, 100, 8193), (129, 160, 8191)])
def test_short_k_product_at_chunk_and_slab_edges(L, m, k, n):
    """The short-K form (mode 4, whatever the size would choose): rows that do
    and do not fill a wavefront's 16 or a slab's 128, sky columns around the
    32-column chunks, one and several chunks to a block, and every number of
    K steps with columns that do and do not allow 16-byte stores (which wait
    for the next chunk's loads in different places).  The bound is the long-K
    test's."""
    import torch
    _say(f"short-K product {m} x {k} x {n}")
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    a = torch.rand((m, k, 3), generator=g, device="cuda")
    b = torch.exp(torch.randn((k, n, 3), generator=g, device="cuda"))
    c = torch.full((m + 1, n, 3), -1.0, device="cuda")
    torch.cuda.synchronize()
    L.dcsky_device(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, k, n, 4)
    assert (c[m] == -1.0).all()                    # nothing past the last row
    for ch in range(3):
        ref = a[:, :, ch].double().contiguous() @ b[:, :, ch].double().contiguous()
        rel = ((c[:m, :, ch].double() - ref) / ref).abs().max().item()
        assert rel <= 3 * 2.0 ** -16 + k * 2.0 ** -24, (ch, rel)


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (67, 41, 5), (3, 15, 300), (4, 16, 255), (4, 1024, 1024), (5, 1025, 30),
                                   (9, 146, 8760), (101, 289, 257), (14000, 578, 1), (63, 513, 256),
                                   (4, 1024, 1025), (128, 257, 255), (129, 257, 255), (3, 1024, 2730),
                                   (3, 1024, 2731), (4, 1024, 4096), (4, 1024, 4097), (1200, 146, 96)])
def test_small_product_against_fp64(L, m, k, n):
    """The one-launch form: fewer K than wavefronts, row groups cut short,
    columns that end inside a block, either side of its lines (K 1024; 2^22
    multiply-adds, where rows are grouped; 2^23 with fewer than 256 columns or
    4 rows; 2^24 with more), past which the product is the split form's bit
    for bit.  FP32 sums of positive terms: K 2^-24 relative; the split forms
    add the long-K test's bound."""
    import torch
    _say(f"small product {m} x {k} x {n}")
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    a = torch.rand((m, k, 3), generator=g, device="cuda")
    b = torch.exp(torch.randn((k, n, 3), generator=g, device="cuda"))
    c = torch.full((m + 1, n, 3), -1.0, device="cuda")
    torch.cuda.synchronize()
    L.dcsky_device(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, k, n)
    assert (c[m] == -1.0).all()
    split = k > 1024 or m * k * n > (1 << 24 if n >= 256 and m >= 4 else 1 << 23)
    if m * n >= 100:
        forced = torch.empty((m, n, 3), device="cuda")
        L.dcsky_device(a.data_ptr(), b.data_ptr(), forced.data_ptr(), m, k, n, 4 if k <= 160 else 3)
        assert torch.equal(c[:m], forced) == split
    for ch in range(3):
        ref = a[:, :, ch].double().contiguous() @ b[:, :, ch].double().contiguous()
        rel = ((c[:m, :, ch].double() - ref) / ref).abs().max().item()
        assert rel <= (3 * 2.0 ** -16 if split else 0) + (k + 1) * 2.0 ** -24, (ch, rel)


def test_tracked_modifiers_belong_to_the_call_and_the_scene(L):
    """Which modifiers are tracked changes from call to call on one context,
    and a batch's scenes number the same names differently: every column is
    that of its modifier, bit for bit, and an unknown name's stays zero."""
    _say("tracked modifiers per call and per scene")
    sky = ("void glow sky 0 0 4 1 1 1 0\nsky source up 0 0 4 0 0 1 180\n",
           "void glow ground 0 0 4 1 1 1 0\nground source down 0 0 4 0 0 -1 180\n",
           "void plastic wall 0 0 5 .5 .5 .5 0 0\nwall polygon w 0 0 12 1 -1 -1 1 1 -1 1 1 1 1 -1 1\n"
           "wall polygon v 0 0 12 -2 -1 1 -2 1 1 -2 1 -1 -2 -1 -1\n",
           "void plastic roof 0 0 5 .3 .3 .3 0 0\nroof polygon r 0 0 12 -1 -1 2 -1 1 2 0 1 2 0 -1 2\n")
    texts = ["".join(sky), "".join(reversed(sky)), sky[0] + sky[2]]
    rng = np.random.default_rng(3)
    sens = [np.hstack([rng.uniform(-.5, .5, (n, 3)), np.tile([0., 0., 1.], (n, 1))]) for n in (7, 65, 1)]
    p = _rc_params(L, ambounce=2, ambdiv=128, minweight=1e-3, seed=4)
    names = ["roof", "sky", "nobody", "wall", "ground"]

    def mods(ns):
        out = [L.RgModifier() for _ in ns]
        for m, n in zip(out, ns):
            m.name, m.bin_kind, m.nbins, m.cbin = n.encode(), 0, 1, 0
        return out

    single = []
    for k, (t, s) in enumerate(zip(texts, sens)):
        c = _ctx(L, t)
        p.seed = 4 + k
        c.set_params(p)
        full = c.contrib(s, mods(names), 1, L.RT_IMM_IRRAD).reshape(len(s), -1, 3)
        assert not full[:, 2].any() and full[:, 1].any() and full[:, 3].any()
        for ns in (["wall"], ["ground", "sky"], names[::-1]):
            got = c.contrib(s, mods(ns), 1, L.RT_IMM_IRRAD).reshape(len(s), -1, 3)
            assert np.array_equal(got, full[:, [names.index(n) for n in ns]]), (k, ns)
        single.append(full)
    assert single[0][:, 0].any() and not single[2][:, 0].any()
    ctxs = [_ctx(L, t) for t in texts]
    p.seed = 4
    ctxs[0].set_params(p)
    for got, want in zip(L.contrib_batch(ctxs, sens, mods(names), 1, L.RT_IMM_IRRAD), single):
        assert np.array_equal(got.reshape(want.shape), want)


@pytest.mark.parametrize("shape", [dict(), dict(window=1 << 10), dict(window=1 << 12, inflight=2),
                                   dict(inflight=2)])
def test_batch_of_rooms_with_and_without_room_sized_primitives(L, shape):
    """Rooms whose walls are tested ahead of the walk, one whose walls all lie
    in its tree and one of a single triangle pair, in one call: every record is
    that of the room alone, bit for bit, whichever windows its rays share and
    whether one or two of them are under way."""
    _say(f"batch of rooms with and without room-sized primitives, {shape}")
    rng = np.random.default_rng(12)
    room = scenes.Room()
    walls = scenes.room_rad(room) + scenes.furniture_rad(rng, 3, room) + scenes.sky_rad((1, 1, 1), ground=(1, 1, 1))
    bare = ("void plastic grey 0 0 5 .5 .5 .5 0 0\ngrey polygon a 0 0 9 0 0 2 4 0 2 0 4 2\n"
            "grey polygon b 0 0 9 0 0 1 4 0 1 0 4 1.5\n" + scenes.sky_rad((1, 1, 1), ground=(1, 1, 1)))
    ctxs, sens = [], []
    for text, big, n in ((walls, 8, 40), (walls, 0, 33), (bare, 0, 7), (walls, 8, 65)):
        c = L.Context(0)
        c.load_text(text)
        c.set_tuning(max_big=big)
        c.commit()
        ctxs.append(c)
        sens.append(np.hstack([rng.uniform(.5, 3.5, (n, 2)), np.full((n, 1), .8), np.tile([0., 0., 1.], (n, 1))]))
    p = _rc_params(L, ambounce=3, ambdiv=128, minweight=1e-3, seed=9)
    single = []
    for k, (c, s) in enumerate(zip(ctxs, sens)):
        p.seed = 9 + k
        c.set_params(p)
        single.append(c.contrib(s, _sky_mods(L), 1, L.RT_IMM_IRRAD))
        assert single[-1].any()
    p.seed = 9
    ctxs[0].set_params(p)
    ctxs[0].set_tuning(**shape)
    got = L.contrib_batch(ctxs, sens, _sky_mods(L), 1, L.RT_IMM_IRRAD)
    assert ctxs[0].last_stats()["wide"]
    for k, (a, b) in enumerate(zip(got, single)):
        assert np.array_equal(a, b), k


def test_rays_that_are_not_numbers_meet_nothing_in_either_tree(L):
    """A ray without a direction (or an origin) bounds no box: the four-wide
    walk leaves it without a hit, as the binary walk does, and its neighbours
    in the wavefront are not touched.  The scene's rings would take any
    distance that is not a number for a hit."""
    _say("rays that are not numbers")
    text = ("void plastic grey 0 0 5 .5 .5 .5 0 0\nvoid glow lamp 0 0 4 3 2 1 0\nvoid glow sky 0 0 4 1 1 1 0\n"
            "sky source up 0 0 4 0 0 1 180\n"
            "grey polygon floor 0 0 12 -5 -5 -1 5 -5 -1 5 5 -1 -5 5 -1\n")
    for i in range(64):
        x, y = i % 8 - 3.5, i // 8 - 3.5
        text += f"{'lamp' if i % 3 else 'grey'} ring r{i} 0 0 8 {x} {y} 1 0 0 -1 0 .3\n"
    c = _ctx(L, text)
    c.set_params(_rc_params(L, ambounce=0, seed=1))
    rng = np.random.default_rng(8)
    rays = np.hstack([rng.uniform(-4, 4, (300, 2)), np.zeros((300, 1)), rng.normal(size=(300, 3))])
    got = {}
    for k in ("good", "direction", "origin"):
        r = rays.copy()
        if k != "good":
            r[::7, 3 if k == "direction" else 0:6 if k == "direction" else 3] = np.nan
        res = []
        for wide in (1, 0):
            c.set_tuning(wide=wide)
            res.append((c.trace(r, 0), c.last_nrays()))
        c.set_tuning(wide=1)
        assert np.array_equal(res[0][0], res[1][0], equal_nan=True) and res[0][1] == res[1][1], k
        got[k] = res[0][0]
    rest = np.arange(300) % 7 != 0
    assert (got["good"] == [3, 2, 1]).all(axis=1).any()
    for k in ("direction", "origin"):
        assert np.array_equal(got[k][rest], got["good"][rest])
        assert not (got[k][~rest] == [3, 2, 1]).all(axis=1).any()      # no ring


def test_stats_tell_the_tree_that_was_walked(L):
    """last_stats() names the walk that ran, not the one a builder's trees
    usually take, and counts the room-sized primitives tested ahead of the
    four-wide walk apart from its leaves; the binary walks test both in one."""
    _say("the tree of last_stats()")
    room = scenes.Room()
    rad = scenes.room_rad(room) + scenes.furniture_rad(np.random.default_rng(2), 2, room) + scenes.sky_rad((1, 1, 1))
    sens = scenes.config1(0)[1]
    res = {}
    for name, builder, shape in [("wide", L.BVH_SAH, {}), ("asked for binary", L.BVH_SAH, dict(wide=0)),
                                 ("per thread", L.BVH_SAH, dict(trace_kernel=0)), ("lbvh", L.BVH_LBVH, {})]:
        c = _ctx(L, rad, builder)
        c.set_params(_rc_params(L, ambounce=0, seed=1))
        c.set_tuning(**shape)
        c.set_profiling(2)
        c.trace(sens, 0)
        res[name] = c.last_stats()
        c.trace(sens[:0], 0)
        assert not c.last_stats()["wide"] and not c.last_stats()["prims"]
        c.close()
    for name, st in res.items():
        assert st["wide"] == (name == "wide") and st["prims"] > 0 and st["node_bytes"] == 64
        assert 0 < st["big_prims"] < st["prims"] if st["wide"] else st["big_prims"] == 0
