"""The algebra of the PCG by sectors (csrc/sect.hip) in numpy: with D constant along x and mirror-symmetric
in y and z, the x transform and the parities of y and z turn A = D + aK into independent operators on
quarter planes, whose weighted dots add up to the whole dots.  Odd and even counts, down to three nodes."""
import math

import numpy as np
import pytest


def bases(n):
    k = np.arange(n)
    V = math.sqrt(2 / n) * np.cos(math.pi * k[None, :] * (k[:, None] + 0.5) / n)
    V[:, 0] = 1 / math.sqrt(n)
    U = -math.sqrt(2 / n) * np.sin(math.pi * k[None, 1:] * (k[:-1, None] + 1) / n)
    return V, U, 2 * np.sin(math.pi * k / (2 * n))


def half(n, par, edge):
    """Points of parity `par` on the half axis of n nodes (edge: of its n - 1 edges, the parity of the wave
    number, opposite to the values')."""
    return n // 2 if par else (n + 1) // 2 - edge


def weights(n, par, edge):
    w = np.full(half(n, par, edge), 2.0)
    if w.size and ((not edge and n % 2 == 1 and not par) or (edge and n % 2 == 0 and par)):
        w[-1] = 1.0
    return w


def whole(P, D, a):
    d = lambda x, ax: np.diff(x, axis=ax)  # noqa: E731

    def back(x, ax):
        z = np.zeros(x.shape[:ax] + (1,) + x.shape[ax + 1:])
        return np.diff(np.concatenate([z, x, z], ax), axis=ax)
    px, py, pz = P
    hx, hy, hz = d(pz, 1) - d(py, 2), d(px, 2) - d(pz, 0), d(py, 0) - d(px, 1)
    q = (back(hz, 1) - back(hy, 2), back(hx, 2) - back(hz, 0), back(hy, 0) - back(hx, 1))
    return [dd * x + a * y for dd, x, y in zip(D, P, q)]


def sectors(f, n):
    Vx, Ux, _ = bases(n[0])
    out = {}
    for c in range(3):
        h = np.tensordot((Ux if c == 0 else Vx).T, f[c], axes=(1, 0))
        if c == 0:
            h = np.concatenate([np.zeros((1,) + h.shape[1:]), h], 0)
        for py in (0, 1):
            for pz in (0, 1):
                g = (h + (1 - 2 * (py ^ (c == 1))) * h[:, ::-1]) / 2
                g = (g + (1 - 2 * (pz ^ (c == 2))) * g[:, :, ::-1]) / 2
                out[c, py, pz] = g[:, :half(n[1], py, c == 1), :half(n[2], pz, c == 2)]
    return out


def operator(X, Y, Z, s, a, D, ny, nz, py, pz):
    """k_sect_cg's operator on one sector: mirrored values past the last node (even count, odd parity) and
    past the last edge (odd count, even parity)."""
    gn = lambda n, p: -1.0 if n % 2 == 0 and p else 0.0  # noqa: E731
    ge = lambda n, p: -1.0 if n % 2 == 1 and not p else 0.0  # noqa: E731

    def diff(F, ax, n, p):
        up = np.concatenate([np.take(F, range(1, F.shape[ax]), ax), gn(n, p) * np.take(F, [-1], ax)], ax) - F
        return np.take(up, range(half(n, p, 1)), ax)

    def back(h, ax, n, p):
        z = np.zeros_like(np.take(h, [0], ax))
        up = np.concatenate([h, ge(n, p) * np.take(h, [-1], ax)], ax)
        up = np.take(up, range(half(n, p, 0)), ax)
        return up - np.concatenate([z, np.take(h, range(half(n, p, 0) - 1), ax)], ax)
    hz = s * Y - diff(X, 0, ny, py)
    hy = diff(X, 1, nz, pz) - s * Z
    hx = diff(Z, 0, ny, py) - diff(Y, 1, nz, pz)
    return (D[0] * X + a * (back(hz, 0, ny, py) - back(hy, 1, nz, pz)), D[1] * Y + a * (back(hx, 1, nz, pz) + s * hz),
            D[2] * Z + a * (-s * hy - back(hx, 0, ny, py)))


@pytest.mark.parametrize("n", [(5, 7, 3), (6, 8, 4), (7, 6, 5), (4, 9, 6), (3, 3, 3), (6, 4, 3), (4, 3, 8)])
def test_sector_operators_are_the_whole_one(n):
    rng = np.random.default_rng(sum(n))
    nx, ny, nz = n
    sh = ((nx - 1, ny, nz), (nx, ny - 1, nz), (nx, ny, nz - 1))
    P = [rng.standard_normal(s) for s in sh]
    D = []
    for s in sh:
        d = rng.random(s[1:])
        d = d + d[::-1]
        D.append(np.broadcast_to((d + d[:, ::-1])[None], s))
    SP, SQ = sectors(P, n), sectors(whole(P, D, 0.7), n)
    _, _, sx = bases(nx)
    dot = 0.0
    for py in (0, 1):
        for pz in (0, 1):
            for mx in range(nx):
                x = [SP[c, py, pz][mx] for c in range(3)]
                q = operator(*x, sx[mx], 0.7, [D[c][0][:v.shape[0], :v.shape[1]] for c, v in enumerate(x)], ny, nz, py, pz)
                for c in range(3):
                    if c or mx:
                        assert np.abs(q[c] - SQ[c, py, pz][mx]).max(initial=0.0) < 1e-13
                    w = weights(ny, py, c == 1)[:, None] * weights(nz, pz, c == 2)[None]
                    dot += (w * x[c] ** 2).sum()
    assert abs(dot - sum((p * p).sum() for p in P)) < 1e-11
