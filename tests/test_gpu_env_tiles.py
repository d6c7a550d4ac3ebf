"""Environment projection and irradiance at the edges of the projection's tiling.

Maps narrower than, as wide as and one texel past a 256-column tile, single rows and columns, more
rows than a block's angle table, and every lmax, against the same sum in FP64. The projection reads
cell (phi, theta) from texel floor(k / n * n) and takes its angles as first + k step, both evaluated
in FP32, as the reference does; the sum over those cells is what FP64 checks."""
import numpy as np
import pytest


pytestmark = pytest.mark.gpu


def basis64(w, lmax):
    """Real SH in FP64 (z the pole, Condon-Shortley phase) from the associated Legendre recurrences."""
    from math import factorial, pi, sqrt
    x, y, z = w[..., 0], w[..., 1], w[..., 2]
    r, phi = np.hypot(x, y), np.arctan2(y, x)   # (sqrt(1 - z^2) loses its digits near the poles)
    P = {(0, 0): np.ones_like(z)}
    for m in range(1, lmax + 1):
        P[m, m] = -(2 * m - 1) * r * P[m - 1, m - 1]
    for m in range(lmax):
        P[m + 1, m] = (2 * m + 1) * z * P[m, m]
    for m in range(lmax + 1):
        for lev in range(m + 2, lmax + 1):
            P[lev, m] = ((2 * lev - 1) * z * P[lev - 1, m] - (lev + m - 1) * P[lev - 2, m]) / (lev - m)
    out = []
    for lev in range(lmax + 1):
        for m in range(-lev, lev + 1):
            k = sqrt((2 * lev + 1) / (4 * pi) * factorial(lev - abs(m)) / factorial(lev + abs(m)))
            v = k * P[lev, abs(m)]
            out.append(v if m == 0 else sqrt(2) * v * (np.cos(m * phi) if m > 0 else np.sin(-m * phi)))
    return np.stack(out, -1)


@pytest.mark.parametrize("W,H", [(1, 1), (1, 700), (2, 1), (3, 5), (64, 31), (255, 2), (256, 128), (257, 129), (300, 1),
                                 (513, 517), (1031, 40)])
@pytest.mark.parametrize("lmax", range(5))
def test_projection_and_irradiance(ctx, W, H, lmax):
    rng = np.random.default_rng(W * 1000 + H)
    env = (rng.random((H, W, 3)) ** 4 * 20).astype(np.float32)
    got = ctx.sh_project_env(env, lmax)
    np.testing.assert_array_equal(ctx.sh_project_env_noalloc(env, lmax), got)
    f = np.float32
    th = (f(np.pi) / f(H) / f(2) + np.arange(H, dtype=f) * (f(np.pi) / f(H))).astype(np.float64)
    ph = (f(2) * f(np.pi) / f(W) / f(2) + np.arange(W, dtype=f) * (f(2) * f(np.pi) / f(W))).astype(np.float64)
    at = [np.floor(np.arange(n, dtype=np.float32) / np.float32(n) * np.float32(n)).astype(int) for n in (W, H)]
    T, P = np.meshgrid(th, ph, indexing="ij")
    Y = basis64(np.stack([np.sin(T) * np.cos(P), np.cos(T), np.sin(T) * np.sin(P)], -1), lmax)
    terms = (Y * (np.sin(T) * (np.pi / H) * (2 * np.pi / W))[..., None])[..., None] * \
        env.astype(np.float64)[at[1]][:, at[0]][:, :, None, :]
    # 40 roundings per term (angles, basis, weight), one per addition: at most 256 rows in a thread,
    # then 32 + 3 in the block and 16 + 6 over the blocks
    tol = (40 + 256 + 35 + 22) * 2.0 ** -24 * np.abs(terms).sum((0, 1))
    assert np.all(np.abs(got - terms.sum((0, 1))) <= tol + 1e-30)
    n = 257
    nrm = rng.normal(size=(n, 3))
    nrm = (nrm / np.linalg.norm(nrm, axis=1, keepdims=True)).astype(np.float32)
    nrm[0] = (0, 0, 1)
    nrm[1] = (0, 0, -1)
    irr = ctx.sh_irradiance(lmax, got, nrm)
    lam = np.concatenate([np.full(2 * lev + 1, [0.8862268925, 1.0233267546, 0.4954159260, 0.0, -0.1107783690][lev] *
                                  np.sqrt(4 * np.pi / (2 * lev + 1)) * 0.7 / np.pi) for lev in range(lmax + 1)])
    part = basis64(nrm.astype(np.float64), lmax)[:, :, None] * (got.astype(np.float64) * lam[:, None])[None]
    # near the poles the basis of sh_evaluate divides by sqrt(1 - z^2), whose relative rounding error
    # is up to 2^-24 / (1 - z^2)
    s2 = np.maximum(1 - nrm[:, 2].astype(np.float64) ** 2, 2.0 ** -24)
    tol = (60 + 4 * lmax / s2)[:, None] * 2.0 ** -24 * np.abs(part).sum(1)
    assert np.all(np.abs(irr - part.sum(1)) <= tol + 1e-30)
