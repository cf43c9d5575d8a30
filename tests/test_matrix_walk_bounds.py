"""Soundness of the raster's matrix path (CPU property test).

The path evaluates a prim's three scaled edge functions and its depth plane at
a quadrant's samples from f32 coefficients (walk_rows in k_raster_q), summed by
a matrix instruction whose error is taken as at most 8u times the sum of the
terms' magnitudes (u = 2^-24; 3.2u was measured). For random triangles --
ordinary, slivers, huge, tiny, partly off the screen -- that sum must lie within
WALK_TOL of the reference's own f32 edge value times the scale, and, where all
three edges are past the tolerance, the plane within WALK_EZ of the depth the
reference interpolates there (mod.rs:225-253). The lowered plane of the depth
culls must stay below that depth at every covered sample.
"""
import numpy as np
import pytest

from tests.test_cull_bounds import RGSS, clamp01, covered_depths, setup

F = np.float32
U = 2.0 ** -24
TOL, EZ = 2.0 ** -16, 2.0 ** -17


def fma(a, b, c):
    a, b, c = (np.asarray(v, np.float64) for v in (a, b, c))
    return (a * b + c).astype(np.float32)


def scale_of(p, n, bbox):
    """walk_scale() in k_setup (f32)."""
    x0, x1, y0, y1 = (F(v) for v in bbox)
    m = F(0)
    for k in range(3):
        dx = F(max(abs(F(x0 - p[k][0])), abs(F(x1 - p[k][0]))) + F(8))
        dy = F(max(abs(F(y0 - p[k][1])), abs(F(y1 - p[k][1]))) + F(8))
        m = max(m, F(F(abs(n[k][0]) * dx) + F(abs(n[k][1]) * dy)))
    v10 = (F(p[1][0] - p[0][0]), F(p[1][1] - p[0][1]))
    v20 = (F(p[2][0] - p[0][0]), F(p[2][1] - p[0][1]))
    area = F(F(v10[0] * v20[1]) - F(v20[0] * v10[1]))
    e = F(F(m * F(40.0 * U)) + F(abs(area) * F(2.0 ** -20)))
    return F(F(TOL) / e)


def plane_of(p, n, inv, z, bbox):
    """depth_plane_bound() in k_setup (f64): the plane about point 2 lowered
    below every interpolated depth, its slopes, and whether the plane itself
    is close enough for the matrix path."""
    x0, x1, y0, y1 = bbox
    z0, z1, z2 = (float(v) for v in z)
    dz0, dz1 = z0 - z2, z1 - z2
    (n1x, n1y), (n2x, n2y) = [tuple(float(c) for c in v) for v in (n[1], n[2])]
    inv = float(inv)
    far = [[max(abs(x0 - float(q[0])), abs(x1 - float(q[0]))), max(abs(y0 - float(q[1])), abs(y1 - float(q[1])))]
           for q in p]
    px, py = inv * (n1x * dz0 + n2x * dz1), inv * (n1y * dz0 + n2y * dz1)
    m1, m2 = abs(n1x) * far[1][0] + abs(n1y) * far[1][1], abs(n2x) * far[2][0] + abs(n2y) * far[2][1]
    d = 12 * U * max(m1, m2) * abs(inv) + 2 * U
    slack = (3 * d + 16 * U) * (abs(z0) + abs(z1) + abs(z2))
    rise = abs(px) * (far[2][0] + 8) + abs(py) * (far[2][1] + 8)
    lo = z2 - 2 * (slack + 8 * U * (abs(z2) + rise) + 1e-30)
    zm = max(abs(z0), abs(z1), abs(z2)) + rise
    ez = U * (18 * zm + 2 * (abs(dz0) + abs(dz1)) + 8 * abs(inv) * (m1 * abs(dz0) + m2 * abs(dz1)))
    return F(lo), F(px), F(py), ez <= 0.9375 * EZ


def rows(nx, ny, ax, ay, rs, z2, qx, qy):
    """The candidate's coefficients about the quadrant's centre, then walk_rows():
    A, B and the constant of each (half, sample). z2: None for an edge."""
    s8 = F(rs * F(0.125))
    a, b = F(nx * s8), F(ny * s8)
    c0 = fma(ny, F(F(qy + 4) - ay), F(nx * F(F(qx + 4) - ax)))
    c0 = F(c0 * rs) if z2 is None else F(c0 + z2)
    p, q = fma(F(-3), b, a), fma(F(3), a, b)
    c = {}
    for h in (0, 1):
        base = fma(F(32 * h - 16), b, c0)
        for k, v in ((0, F(base + p)), (1, F(base + q)), (2, F(base - p)), (3, F(base - q))):
            c[h, k] = v
    return float(a), float(b), c


def triangles(kind, rng):
    w, h = 1920.0, 1080.0
    c = rng.uniform(0, 1, 2) * (w, h)
    size = {"ordinary": rng.uniform(3, 80), "huge": rng.uniform(500, 2500), "tiny": rng.uniform(0.05, 2.0),
            "sliver": rng.uniform(50, 600)}[kind]
    p = c + rng.uniform(-1, 1, (3, 2)) * size
    if kind == "sliver":
        p[2] = p[1] + rng.uniform(-0.5, 0.5, 2)
    p = np.clip(p, 0, (w, h)).astype(np.float32)
    v = (p[1] - p[0]).astype(np.float64), (p[2] - p[0]).astype(np.float64)
    if v[0][0] * v[1][1] - v[1][0] * v[0][1] < 0:
        p[[1, 2]] = p[[2, 1]]
    z = (rng.uniform(0, 1) + rng.uniform(-1, 1, 3) * rng.choice([0.5, 0.05, 1e-3])).clip(0, 1).astype(np.float32)
    return p, z


@pytest.mark.parametrize("kind", ["ordinary", "huge", "tiny", "sliver"])
def test_matrix_path_margins(kind):
    rng = np.random.default_rng({"ordinary": 1, "huge": 2, "tiny": 3, "sliver": 4}[kind])
    fast = edges = inside = below = 0
    for _ in range(250):
        p, z = triangles(kind, rng)
        with np.errstate(all="ignore"):
            n, inv = setup(p, z)
        if not (0 < inv < np.finfo(np.float32).max):
            continue
        bbox = (int(np.floor(p[:, 0].min())), int(np.ceil(p[:, 0].max())),
                int(np.floor(p[:, 1].min())), int(np.ceil(p[:, 1].max())))
        if bbox[0] >= bbox[1] or bbox[2] >= bbox[3]:
            continue
        pz0, pzx, pzy, ok = plane_of(p, n, inv, z, bbox)
        tie = [bool((nx > 0) or (not (nx < 0) and ny < 0)) for nx, ny in n]
        cx, cy, cz = covered_depths(p, n, inv, z, bbox, tie) if (bbox[1] - bbox[0]) * (bbox[3] - bbox[2]) < 10**5 else \
            [np.zeros(0, np.float32)] * 3
        bound = fma(pzy, (cy - p[2][1]).astype(np.float32), (pzx * (cx - p[2][0]).astype(np.float32)).astype(np.float32))
        bound = (bound + pz0).astype(np.float32)
        assert (cz >= bound).all(), kind
        below += cz.size
        rs = scale_of(p, n, bbox)
        fast += ok
        qs = [(x, y) for x in range(bbox[0] // 8 * 8, bbox[1], 8) for y in range(bbox[2] // 8 * 8, bbox[3], 8)]
        for qx, qy in [qs[i] for i in rng.permutation(len(qs))[:4]]:
            fn = [rows(n[k][0], n[k][1], p[k][0], p[k][1], rs, None, qx, qy) for k in range(3)]
            fn.append(rows(pzx, pzy, p[2][0], p[2][1], F(1), z[2], qx, qy))
            X, Y = np.meshgrid(np.arange(8), np.arange(8))
            for k in range(4):
                sx = ((qx + X).astype(np.float32) + RGSS[k, 0]).astype(np.float32)
                sy = ((qy + Y).astype(np.float32) + RGSS[k, 1]).astype(np.float32)
                val, err, ref = [], [], []
                for f in range(4):
                    a, b, c = fn[f]
                    cc = np.where(Y < 4, float(c[0, k]), float(c[1, k]))
                    tx, ty = a * (8 * X - 28), b * (8 * (Y % 4) - 12)
                    val.append(tx + ty + cc)
                    err.append(8 * U * (abs(tx) + abs(ty) + abs(cc)))
                for f in range(3):
                    e = (n[f][0] * (sx - p[f][0]).astype(np.float32) +
                         n[f][1] * (sy - p[f][1]).astype(np.float32)).astype(np.float32)
                    ref.append(e)
                    assert (abs(val[f] - e.astype(np.float64) * float(rs)) + err[f] <= TOL).all(), (kind, f)
                    edges += e.size
                if not ok:
                    continue
                sure = np.minimum(np.minimum(val[0], val[1]), val[2]) > TOL
                b0, b1 = clamp01((ref[1] * inv).astype(np.float32)), clamp01((ref[2] * inv).astype(np.float32))
                b2 = clamp01(((F(1) - b0) - b1).astype(np.float32))
                zr = ((b0 * z[0] + b1 * z[1]).astype(np.float32) + b2 * z[2]).astype(np.float64)
                bad = sure & (abs(val[3] - zr) + err[3] > EZ)
                assert not bad.any(), (kind, abs(val[3] - zr)[bad].max() / U)
                inside += int(sure.sum())
    assert edges > 10_000 and fast > 20 and inside > 100 and below > 100, (kind, edges, fast, inside, below)
