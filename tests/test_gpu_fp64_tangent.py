"""Binary64 difference form on the sphere: what the rounding of a point's tangent velocity U leaves along its
position p adds tan(separation / 2) (p.U) to du_L of every pair of the point, all alike.  One point moves among
20000 at rest, far from it: the sum's error against the reference's formula in extended precision (on the same
positions and local bases), over the sum of the tangents, is that residual.

Bound: one component's rounding, at most half a unit in the last place of U_k times p_k, and |U_k p_k| <= |U| / 2
for a tangent U: 2^-54 |u|; a fifth more for the other roundings, which differ from pair to pair (2^-53 /
cos(separation / 2) each, over the root of 20000)."""
import numpy as np
import pytest

import _oracle
from test_gpu_parity import gpu_hist

pytestmark = pytest.mark.gpu
LD = np.longdouble


def _frame(x):
    """Positions and local bases as the records hold them: binary64 sines and cosines of the degrees."""
    s = np.array([_oracle.sincosd(v) for v in x.ravel()]).reshape(2, -1, 2)
    (sl, cl), (sp, cp) = (s[0].T, s[1].T)
    p = np.stack([cp * cl, cp * sl, sp])
    return p, np.stack([-sl, cl, 0 * sl]), np.stack([-sp * cl, -sp * sl, cp])


def test_normal_residual(ctx):
    rng = np.random.default_rng(8)
    n = 20000
    worst = 0.0
    for _ in range(40):
        a = rng.normal(size=3)
        a /= np.linalg.norm(a)
        v = rng.normal(size=(3, 12 * n))
        v /= np.linalg.norm(v, axis=0)
        c = a @ v
        v = v[:, (c < np.cos(2.6)) & (c > np.cos(3.0))][:, :n]
        v = np.concatenate([a[:, None], v], axis=1)
        x = np.degrees(np.stack([np.arctan2(v[1], v[0]), np.arcsin(v[2])]))
        u = np.zeros((2, v.shape[1]))
        u[:, 0] = rng.normal(size=2)
        s, cnt = gpu_hist(ctx, x, u, np.array([2.55, 3.05]), (0, 1, 0), geometry="deg", prec="fp64")
        p, E, N = _frame(x)
        p, E, N = p.astype(LD), E.astype(LD), N.astype(LD)
        U = u[0, 0].astype(LD) * E[:, :1] + u[1, 0].astype(LD) * N[:, :1]
        d = p[:, 1:] - p[:, :1]
        w = np.cross(p[:, 0], d.T).T
        sin = np.sqrt((w * w).sum(0))
        t = d - (d * p[:, :1]).sum(0) * p[:, :1]
        L = -(t * U).sum(0) / sin
        tan = np.sqrt((d * d).sum(0) / ((p[:, 1:] + p[:, :1]) ** 2).sum(0))
        # (pairs of two points at rest add zero; those of the axis' only bin and the moving point are all here)
        assert int(cnt.sum()) >= v.shape[1] - 1
        worst = max(worst, abs(float((LD(float(s.sum())) - L.sum()) / tan.sum())) / np.hypot(*u[:, 0]))
    assert worst <= 1.2 * 2.0 ** -54
