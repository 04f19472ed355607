"""The last rows of a band array have entries past the matrix (row i, diagonal
j with i + j >= N).  Whatever a caller's arrays hold there, the observables and
the Lanczos vectors are those of the matrix: the same bits as with zeros."""
import numpy as np
import pytest

from _cfg import make_oracle, mixed_state, shape, upload_from_oracle

pytestmark = pytest.mark.gpu


def with_tail(band, N, p, value):
    b = np.array(band, np.float64).reshape(-1, N, p + 1)
    b[:, np.arange(N)[:, None] + np.arange(p + 1) >= N] = value
    return b.ravel()


@pytest.mark.parametrize("p", [7, 8])
@pytest.mark.parametrize("N", [40, 1024, 1030])
def test_observables_do_not_see_entries_past_the_matrix(N, p):
    import pyoracle as po
    import qpc_gpu
    cfg = shape(N, 3, 0.2 * N, M=3, m0=-1, p=p)
    print(f"case: band tails, observables N={N} p={p}", flush=True)
    o = make_oracle(cfg)
    st = qpc_gpu.Setup(N, p, 3, 3, -1, cfg["dt"], 0.0, cfg["rmax"], 1.0, 1.0, cfg["mask_rmin"], cfg["mask_rmax"],
                       cfg["mask_fact"])
    c = mixed_state(o, seed=N + p, amp=0.4)
    out = []
    for value in (0.0, np.nan):
        prop = qpc_gpu.Propagator(N, p, 3, 3, -1, cfg["dt"])
        upload_from_oracle(prop, o)
        prop.upload_radial(*[with_tail(o.get(k), N, p, value if k in (po.QOR_RPOW1, po.QOR_S) else 0.0)
                             for k in (po.QOR_S, po.QOR_CHOL, po.QOR_RINV, po.QOR_RDIF, po.QOR_RPOW1, po.QOR_MASK)])
        prop.upload_outer(with_tail(st.get(qpc_gpu.SETUP_SOUTER), N, p, value))
        prop.upload_accel(with_tail(o.get(po.QOR_DVDR), N, p, value))
        prop.set_state(c)
        prop.record(qpc_gpu.REC_ALL, 1)
        prop.run(np.zeros(1), 0, 0, 1, use_mask=False)
        out.append(prop.record_read()[0].copy())
        prop.close()
    print(f"  {out[0]}\n  {out[1]}", flush=True)
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("c", [dict(N=250, p=7, L=5, M=1, m0=0, kmax=64), dict(N=400, p=8, L=3, M=3, m0=-1, kmax=64)],
                         ids=lambda c: "N{N}_p{p}".format(**c))
def test_lanczos_vectors_do_not_see_entries_past_the_matrix(c):
    import qpc_gpu
    from test_gpu_krylov_order import operators
    N, p = c["N"], c["p"]
    print(f"case: band tails, Krylov N={N} p={p}", flush=True)
    S, ch, F, G, H, y10, q10, z = operators(c)
    out = []
    for value in (0.0, np.nan):
        prop = qpc_gpu.Propagator(N, p, c["L"], c["M"], c["m0"], 0.05)
        prop.upload_radial(*[with_tail(b, N, p, value) for b in (S, ch, F, G, F, S)])
        prop.upload_krylov(with_tail(H, N, p, value), y10, q10)
        prop.set_state(z)
        m, _, ab = prop.krylov_step_adaptive(0.75, 0.03125, c["kmax"], c["kmax"], 0.0)
        out.append(np.concatenate([ab.ravel(), prop.get_state().view(np.float64).ravel()]))
        prop.close()
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])
