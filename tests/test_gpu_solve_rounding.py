"""The rounding of the banded solves against extended precision (80 bit) on the
same operators: no larger than that of a substitution in doubles that subtracts
each row's products one after the other, nearest row first (one fused multiply-
add per product and component, as the device has them).  Bar: 1.1 times its rms
over 64 channels; a channel's error scatters by a third, so that the rms of 64
is known to 4% on either side.  (Subtracted farthest row first, the products are
rounded at the size of the right-hand side: 1.15 to 1.3 times.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD, CLD = np.longdouble, np.clongdouble


def _round(x):
    return x.astype(np.complex128).astype(CLD)


def _keep(x):
    return x


def _msub(a, c, y, rnd):
    """a - c y: per component two fused multiply-adds (one for a real c)"""
    if np.iscomplexobj(c) and rnd is _round:
        a = rnd(a - c.real * y)
        return rnd(a - 1j * c.imag * y)
    return rnd(a - c * y)


def _solve(mult, low, diag, z, rnd):
    """x = (L D L^T)^-1 (B z) for every channel: mult (nch, N, p+1) the band of B, low L's columns, diag 1 / D;
    every operation rounded by rnd."""
    nch, N = z.shape
    p = mult.shape[-1] - 1
    v = np.zeros_like(z)
    for j in range(p, 0, -1):  # the band product, lower neighbours first
        v[:, j:] = _msub(v[:, j:], -mult[:, :N - j, j], z[:, :N - j], rnd)
    for j in range(p + 1):
        v[:, :N - j] = _msub(v[:, :N - j], -mult[:, :N - j, j], z[:, j:], rnd)
    y = v
    for i in range(N):
        for j in range(1, min(p, i) + 1):
            y[:, i] = _msub(y[:, i], low[:, i - j, j], y[:, i - j], rnd)
    y = rnd(diag * y)
    for i in range(N - 1, -1, -1):
        for j in range(1, min(p, N - 1 - i) + 1):
            y[:, i] = _msub(y[:, i], low[:, i, j], y[:, i + j], rnd)
    return y


def _err(x, t):
    d = np.sqrt((np.abs(x - t) ** 2).sum(1)) / np.sqrt((np.abs(t) ** 2).sum(1))
    return float(np.sqrt((d ** 2).mean()))


@pytest.mark.parametrize("p", [7, 8])
@pytest.mark.parametrize("N", [240, 800])
def test_solves_round_no_worse_than_nearest_row_first(N, p):
    import qpc_gpu
    L = 64
    print(f"case: rounding of solves N={N} p={p}", flush=True)
    rmax = 0.2 * (N + 2 - p)
    st = qpc_gpu.Setup(N, p, L, 1, 0, 0.05, 0.0, rmax, 1.0, 1.0, rmax - 8.0, rmax, 0.125)
    prop = qpc_gpu.Propagator(N, p, L, 1, 0, 0.05)
    prop.upload_setup(st)
    rng = np.random.default_rng(N + p)
    i = np.arange(N)
    c = np.zeros((L, N), np.complex128)
    for _ in range(2):
        x0, w = rng.uniform(0.3, 0.7, (L, 1)) * N, rng.uniform(0.03, 0.06, (L, 1)) * N
        q, f = rng.uniform(-0.25, 0.25, (L, 1)), rng.uniform(0, 6.28, (L, 1))
        c += rng.uniform(0.3, 1.0, (L, 1)) * np.exp(-((i - x0) / w) ** 2 + 1j * (q * i + f))

    def band(what, n=1):
        return np.array(st.get(what)).reshape(-1, N, p + 1)[:n]

    chol = band(qpc_gpu.SETUP_CHOL)
    ld = band(qpc_gpu.SETUP_LOWER, L)  # D on the diagonal, L below it
    ops = {  # (B, L unit lower by columns, 1 / D)
        "mask": (band(qpc_gpu.SETUP_MASK), chol.astype(LD) / chol[:, :, :1].astype(LD), 1 / chol[:, :, 0].astype(LD) ** 2),
        "free": (band(qpc_gpu.SETUP_UPPER, L), ld, 1 / ld[:, :, 0].astype(CLD))}
    for kind, (b, low, diag) in ops.items():
        prop.set_state(c.ravel())
        prop.mask() if kind == "mask" else prop.propagate()
        got = prop.get_state().reshape(L, N)
        wide = CLD if kind == "free" else LD
        t = _solve(b.astype(wide), low.astype(wide), diag, c.astype(CLD), _keep)
        dbl = np.complex128 if kind == "free" else np.float64
        near = _solve(b.astype(wide), low.astype(dbl).astype(wide), diag.astype(dbl).astype(wide), c.astype(CLD), _round)
        e, ref = _err(got, t), _err(near, t)
        print(f"  {kind}: {e:.3e}, nearest row first {ref:.3e} ({e / ref:.2f})", flush=True)
        assert e <= 1.1 * ref
    prop.close()
