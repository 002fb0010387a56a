"""The pair pass (4, 8 or 16 lanes per particle, one walk over the list) against plain numpy.

Small clouds whose particle counts and list lengths straddle the pass's units: 4 to 16 lanes per
particle, 4 to 16 particles per wavefront, 16 to 64 per workgroup; lists of 0 to 8 neighbours and long ones,
odd capacities.  Tool particles (their volume and mechanics left out, their temperature not) and
unequal smoothing lengths are among them; unlocked grids take the ordered sums.  The reference is the brute-force
sum over all pairs in numpy's 64 bits, B inverted per particle, the corrected gradient used pair by
pair.  Tolerances from the arithmetic: FP64 sums of at most 300 terms of a few roundings each, the
inverse of a well-conditioned B: 1e-12 of the largest value; FP32 terms, 2^-24 each with a handful of
operations and cancellation of the stress sum by up to ten: 2e-5.
"""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api

pytestmark = pytest.mark.gpu

DX, RHO0, K, G = 5e-4, 4.43, 1.2, 0.4
MASS = DX ** 3 * RHO0
EPS_X, ALPHA, BETA, ETA = 0.5, 1.0, 2.0, 0.1


def constants(heat, cspm, single_sqrt, h, cap):
    api.reset_globals()
    api.constants_reset()
    api.set_options(cspm=cspm, heat=heat, single_sqrt=single_sqrt, max_neighbours=cap)
    ph = api.make_phys_constants()
    ph.rho0, ph.K, ph.G, ph.mass = RHO0, K, G, MASS
    co = api.make_corr_constants()
    co.wdeltap, co.stresseps, co.xspheps, co.alpha, co.beta, co.eta = 1e8, 0.3, EPS_X, ALPHA, BETA, ETA
    t = api.make_trml_constants()
    t.cp, t.k, t.alpha, t.T_init = 5e-6, 7e-13, 3e-8, 300.0
    tool = api.make_trml_constants()
    tool.cp, tool.k, tool.alpha, tool.T_init = 5e-6, 7e-13, 9e-8, 300.0
    api.actions_setup_physical_constants(ph)
    api.actions_setup_corrector_constants(co)
    api.actions_setup_thermal_constants_wp(t)
    api.interactions_setup_physical_constants(ph)
    api.interactions_setup_corrector_constants(co)
    api.interactions_setup_thermal_constants_workpiece(t)
    api.interactions_setup_thermal_constants_tool(tool, None)
    return 3e-8, 9e-8


def cloud(n, seed, spread):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = (g * spread + rng.uniform(-0.2, 0.2, g.shape)) * DX
    S = rng.uniform(-5e-3, 5e-3, (n, 6))
    tool = (rng.uniform(size=n) < 0.15).astype(float)
    tool[0] = 0.0
    return dict(pos=pos, vel=rng.uniform(-2e-3, 2e-3, (n, 3)), rho=RHO0 * (1 + rng.uniform(-5e-3, 5e-3, n)),
                T=300 + rng.uniform(0, 400, n), h=1.5 * DX * rng.uniform(0.9, 1.0, n), tool=tool,
                S9=S[:, [0, 3, 5, 3, 1, 4, 5, 4, 2]])


def reference(c, heat, cspm, single_sqrt, alphas):
    """x_t, v_t, v_der, S_der, T_t of every particle over all pairs, artificial stress zero."""
    n = len(c["rho"])
    x, v, rho, T, h = c["pos"], c["vel"], c["rho"], c["T"], c["h"]
    wp = c["tool"] == 0
    d = x[:, None] - x[None]
    r2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
    near = (r2 >= 1e-8) & (r2 < 4 * (h * h)[:, None])
    r = np.where(near, r2, 1.0)
    r = np.sqrt(r.astype(np.float32)).astype(np.float64) if single_sqrt else np.sqrt(r)
    q = r / h[:, None]
    fac = 1 / (np.pi * h ** 3)[:, None]
    W = np.where(q > 1, 0.25 * (2 - q) ** 3, 1 - 1.5 * q * q * (1 - 0.5 * q)) * fac * near
    dW = np.where(q > 1, -0.75 * (2 - q) ** 2, -3 * q * (1 - 0.75 * q)) * fac / h[:, None] / r * near
    w0 = dW[..., None] * d
    vol = MASS / rho
    mech = near & wp[:, None] & wp[None]
    B = -np.einsum("ij,j,ija,ijb->iab", (near & wp[None]).astype(float), vol, d, w0)
    inv = np.tile(np.eye(3), (n, 1, 1))
    ok = (np.linalg.det(B) > 1e-8) & wp & bool(cspm)
    inv[ok] = np.linalg.inv(B[ok])
    w = np.einsum("iba,ija->ijb", inv, w0)
    p = K / RHO0 * (rho - RHO0)
    if single_sqrt:
        c0 = float(np.sqrt(np.float32(K / RHO0)))
        p = c0 * c0 * (rho - RHO0)
    A = (c["S9"].reshape(n, 3, 3) - np.where(wp, p, 0.0)[:, None, None] * np.eye(3)) / (rho * rho)[:, None, None]
    vij = v[:, None] - v[None]
    mw = w * mech[..., None]
    v_der = -np.einsum("ija,j,ijb->iab", vij, vol, mw)
    S_der = MASS * np.einsum("ijab,ijb->iab", A[:, None] + A[None], mw)
    cs = K / rho
    cs = np.sqrt(cs.astype(np.float32)).astype(np.float64) if single_sqrt else np.sqrt(cs)
    vx = np.einsum("ija,ija->ij", vij, d)
    hij, rij = 0.5 * (h[:, None] + h), 0.5 * (rho[:, None] + rho)
    mu = hij * vx / (r2 + ETA ** 2 * hij * hij)
    Pi = np.where(vx < 0, (-ALPHA * 0.5 * (cs[:, None] + cs) * mu + BETA * mu * mu) / rij, 0.0)
    v_t = -MASS * np.einsum("ij,ija->ia", Pi, mw)
    x_t = -EPS_X * MASS * np.einsum("ij,ija->ia", W * mech / rij, vij)
    T_t = np.zeros(n)
    if heat == _lib.MFG_HEAT_BROOKSHAW:
        rr = np.where(near, r2, 1.0)
        T_t = np.where(wp, *alphas) * 2 * np.einsum("j,ij,ija,ija->i", vol, near * (T[:, None] - T) / rr, d, w)
    return x_t, v_t, v_der.reshape(n, 9), S_der.reshape(n, 9), T_t


# (particles, lattice spacing in dx: 2.2 gives short lists, 1 long ones, 5 empty ones, list capacity)
CLOUDS = [(1, 1.0, 0), (2, 1.0, 8), (5, 1.0, 0), (15, 2.2, 0), (16, 2.2, 0), (17, 1.0, 20), (63, 2.2, 0), (64, 1.0, 0),
          (65, 1.0, 0), (130, 5.0, 0), (257, 1.0, 0), (515, 0.8, 0)]


@pytest.mark.parametrize("single_sqrt", [True, False], ids=["sqrtf", "sqrt"])
@pytest.mark.parametrize("cspm", [True, False], ids=["cspm", "plain"])
@pytest.mark.parametrize("heat", [_lib.MFG_HEAT_NONE, _lib.MFG_HEAT_BROOKSHAW], ids=["none", "brookshaw"])
@pytest.mark.parametrize("precision,locked", [(_lib.MFG_FP64, True), (_lib.MFG_FP64, False),
                                              (_lib.MFG_FP32_KAHAN, True), (_lib.MFG_FP32_WIDE, False)],
                         ids=["fp64", "fp64_unlocked", "kahan", "wide_unlocked"])
def test_pair_sums_against_all_pairs(hip_device, precision, locked, heat, cspm, single_sqrt):
    tol = 1e-12 if precision == _lib.MFG_FP64 else 2e-5
    for n, spread, cap in CLOUDS:
        c = cloud(n, 100 + n, spread)
        alphas = constants(heat, cspm, single_sqrt, c["h"].max(), cap)
        p = api.particle_gpu(c["pos"], c["vel"], c["rho"], c["T"], c["h"], None, c["tool"], c["S9"], precision=precision)
        if locked:
            g = api.grid_gpu_green(n, c["pos"].min(0) - DX, c["pos"].max(0) + DX, float(c["h"].max()))
        else:
            g = api.grid_gpu_green(100000, n)
            g.update_geometry(p)
        g.sort(p)
        order = p.download(_lib.F_ID).astype(int)
        api.material_eos(p)
        api.interactions_monaghan(p, g)
        got = [p.download(f) for f in (_lib.F_POS_T, _lib.F_VEL_T, _lib.F_V_DER, _lib.F_S_DER, _lib.F_T_T)]
        ref = reference(c, heat, cspm, single_sqrt, alphas)
        for name, a, b in zip(("x_t", "v_t", "v_der", "S_der", "T_t"), got, ref):
            if name in ("x_t", "v_t"):  # kept as they were for tool particles
                a, b = a * (c["tool"][order] == 0)[:, None], b
            b = b[order]
            scale = np.abs(b).max()
            err = np.abs(a - b).max() / scale if scale > 0 else np.abs(a).max()
            assert err <= tol, (n, spread, name, err)


def many_clouds(n, spread, total, precision):
    """Copies of a cloud too far apart to meet, `total` particles; (inputs, fields by id)."""
    copies = -(-total // n)
    one = cloud(n, 900 + n, spread)
    step = np.ptp(one["pos"][:, 0]) + 8 * DX
    c = {k: np.concatenate([v] * copies)[:total] for k, v in one.items()}
    c["pos"] = c["pos"] + np.repeat(np.arange(copies) * step, n)[:total, None] * [1.0, 0.0, 0.0]
    alphas = constants(_lib.MFG_HEAT_BROOKSHAW, True, False, c["h"].max(), 0)
    p = api.particle_gpu(c["pos"], c["vel"], c["rho"], c["T"], c["h"], None, c["tool"], c["S9"], precision=precision)
    g = api.grid_gpu_green(total, c["pos"].min(0) - DX, c["pos"].max(0) + DX, float(c["h"].max()))
    g.sort(p)
    place = np.argsort(p.download(_lib.F_ID).astype(int))
    api.material_eos(p)
    api.interactions_monaghan(p, g)
    got = [p.download(f)[place] for f in (_lib.F_POS_T, _lib.F_VEL_T, _lib.F_V_DER, _lib.F_S_DER, _lib.F_T_T)]
    return c, alphas, got


@pytest.mark.parametrize("total", [4095, 4096])
def test_fp64_lanes(hip_device, total):
    """Both sides of the size where 16 lanes a particle become 4: the first and the last cloud against
    all pairs."""
    for n, spread in ((65, 1.0), (257, 1.0), (515, 2.2)):
        c, alphas, got = many_clouds(n, spread, total, _lib.MFG_FP64)
        for lo in (0, (total - 1) // n * n):
            part = slice(lo, min(lo + n, total))
            ref = reference({k: v[part] for k, v in c.items()}, _lib.MFG_HEAT_BROOKSHAW, True, False, alphas)
            for name, a, b in zip(("x_t", "v_t", "v_der", "S_der", "T_t"), got, ref):
                a = a[part]
                if name in ("x_t", "v_t"):
                    a = a * (c["tool"][part] == 0)[:, None]
                scale = np.abs(b).max()
                err = np.abs(a - b).max() / scale if scale > 0 else np.abs(a).max()
                assert err <= 1e-12, (n, lo, name, err)


@pytest.mark.parametrize("precision", [_lib.MFG_FP32_KAHAN, _lib.MFG_FP32_WIDE], ids=["kahan", "wide"])
def test_fp32_lanes_give_the_same_sums(hip_device, precision):
    """Both sides of the size where 8 lanes a particle become 4: every particle that the two sets share
    with all its neighbours has the same sums, to the bit."""
    for n, spread in ((65, 1.0), (257, 1.0), (515, 2.2)):
        _, _, small = many_clouds(n, spread, 24 * 1024 - 1, precision)
        _, _, large = many_clouds(n, spread, 24 * 1024, precision)
        whole = (24 * 1024 - 1) // n * n
        for a, b in zip(small, large):
            assert np.array_equal(a[:whole], b[:whole]), (n, spread)
