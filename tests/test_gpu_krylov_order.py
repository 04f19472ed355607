"""The Lanczos tridiagonal bit for bit: every sum of the Krylov chain (H u, the
inner products, S^-1, the orthogonalisation, the norm) keeps its order and its
fused multiply-adds, whatever the launch shape.

Estimates far below the tolerance are rounding of these sums, and a controller
reads them: its steps, and with them a controlled run's state (by up to 4e-7),
move with any other order.  The operators and the state are dyadic rationals and
their Cholesky factor comes from plain sums, products, quotients and roots, so
the inputs are the same bits everywhere.  Wanted: tests/golden/
krylov_tridiagonals.npz (recorded on an MI355X), equal in every bit."""
import math
import os

import numpy as np
import pytest

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "krylov_tridiagonals.npz")

# N around one row block, one and two waves of partitions, a cut channel (more
# than 64 partitions), chunks of more than 256 rows in the inner products,
# subspaces of more than 128 vectors
CASES = [dict(N=18, p=7, L=1, M=1, m0=0, kmax=8), dict(N=250, p=7, L=5, M=1, m0=0, kmax=64),
         dict(N=400, p=8, L=3, M=3, m0=-1, kmax=64), dict(N=900, p=7, L=2, M=1, m0=0, kmax=150),
         dict(N=1300, p=7, L=2, M=1, m0=0, kmax=24), dict(N=1700, p=8, L=2, M=1, m0=0, kmax=24),
         dict(N=1700, p=7, L=20, M=1, m0=0, kmax=24)]


def case_name(c):
    return "N{N}_p{p}_L{L}_M{M}".format(**c)


def _dyadic(rng, shape):
    return rng.integers(-2 ** 20, 2 ** 20, shape) / 2.0 ** 20


def operators(c):
    """S (diagonally dominant), its Cholesky factor, 1/r, d/dr, H per l, y10, q10 and a state, none of them physical."""
    N, p, L, M, m0 = c["N"], c["p"], c["L"], c["M"], c["m0"]
    rng = np.random.default_rng(1000 * N + 10 * p + L)
    ne, nl = p + 1, max(abs(m0), abs(m0 + M - 1)) + L
    inside = np.arange(N)[:, None] + np.arange(ne) < N
    decay = 0.5 ** np.arange(ne)

    def band():
        return np.where(inside, _dyadic(rng, (N, ne)) * decay, 0.0)

    S, F, G = band(), band(), band()
    S[:, 0] = 3.0 + S[:, 0]
    G[:, 0] = 0.0
    H = np.stack([band() for _ in range(nl)])
    ch = S.tolist()  # plain floats: one rounding per operation
    for i in range(N):
        d = ch[i][0] = math.sqrt(ch[i][0])
        for j in range(1, ne):
            ch[i][j] /= d
        for j in range(1, min(ne, N - i)):
            for k in range(j, min(ne, N - i)):
                ch[i + j][k - j] -= ch[i][j] * ch[i][k]
    z = _dyadic(rng, (M * L, N)) + 1j * _dyadic(rng, (M * L, N))
    return S, np.array(ch), F, G, H, _dyadic(rng, M * L), _dyadic(rng, M * L), z.ravel()


def tridiagonal(qpc_gpu, c):
    S, ch, F, G, H, y10, q10, z = operators(c)
    prop = qpc_gpu.Propagator(c["N"], c["p"], c["L"], c["M"], c["m0"], 0.05)
    prop.upload_radial(S, ch, F, G, F, S)
    prop.upload_krylov(H, y10, q10)
    prop.set_state(z)
    m, _, ab = prop.krylov_step_adaptive(0.75, 0.03125, c["kmax"], c["kmax"], 0.0)
    prop.close()
    return ab


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=case_name)
def test_tridiagonal_keeps_its_bits(c):
    import qpc_gpu
    print(f"case: tridiagonal {case_name(c)}", flush=True)
    ab = tridiagonal(qpc_gpu, c)
    with np.load(GOLDEN) as g:
        ref = g[case_name(c)]
    print(f"  {len(ab)} vectors, largest difference {np.abs(ab - ref).max():.1e}", flush=True)
    assert np.array_equal(ab, ref)
