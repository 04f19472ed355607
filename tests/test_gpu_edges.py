"""Steps at the sizes where the partitioned kernels have edges, against the
oracle: fewer rows than one partition (24), whole and ragged last partitions,
grids shorter than the factorisation's restart and the carry, one and two wave
groups of partitions (1536 rows), both spline orders.  Bar: relative L2 <=
1e-12 per call, the parity bar of single steps."""
import numpy as np
import pytest

from _cfg import make_oracle, mixed_state, rel_l2, shape, upload_from_oracle

pytestmark = pytest.mark.gpu


def _pair(N, p, L, M=1, m0=0):
    import qpc_gpu
    cfg = shape(N, L, 0.2 * N, M=M, m0=m0, p=p)
    o = make_oracle(cfg)
    prop = qpc_gpu.Propagator(N, p, L, M, m0, cfg["dt"])
    upload_from_oracle(prop, o)
    return o, prop


@pytest.mark.parametrize("p", [7, 8])
@pytest.mark.parametrize("N", [18, 23, 24, 25, 48, 71, 97, 145, 191, 1535, 1536, 1537])
def test_steps_at_partition_edges(N, p):
    print(f"case: edges N={N} p={p}", flush=True)
    o, prop = _pair(N, p, 3)
    c = mixed_state(o, seed=N + p, amp=0.3)
    prop.set_state(c)
    for kind, a in (("vg", (0.7, 0.9)), ("vg", (0.9, -0.4)), ("free", None), ("lg", (0.05, 0.03)), ("mask", None)):
        ref = np.ascontiguousarray(prop.get_state())
        if kind == "vg":
            o.step(ref, *a)
            prop.propagate(*a)
        elif kind == "lg":
            o.step_lg(ref, *a)
            prop.propagate_lg(*a)
        elif kind == "free":
            o.step_free(ref)
            prop.propagate()
        else:
            o.mask(ref)
            prop.mask()
        err = rel_l2(prop.get_state(), ref)
        print(f"  {kind} {a}: rel L2 {err:.2e}", flush=True)
        assert err <= 1e-12
    prop.close()


@pytest.mark.parametrize("gauge", ["vgwr", "lgwr"])
@pytest.mark.parametrize("M,L,N,isub", [(2, 4, 32, -1), (3, 3, 31, -1), (3, 5, 33, 2), (7, 9, 95, -1), (8, 8, 64, 3),
                                        (5, 13, 48, -1), (5, 13, 50, 2), (13, 11, 40, 3)])
def test_rotations_at_tile_edges(M, L, N, isub, gauge):
    """Channel counts around the rotations' 64-row tiles and 8-term slices,
    row lengths around their 64 columns, each sub-block (row groups that are
    empty, of a few rows, of several tiles)."""
    import pyoracle as po
    print(f"case: rotation edges M={M} L={L} N={N} isub={isub} {gauge}", flush=True)
    m0 = -(M // 2)
    o, prop = _pair(N, 7, L, M, m0)
    c = mixed_state(o, seed=N + M, amp=0.3)
    if isub > 0:
        c = np.where(np.repeat([il % 2 == isub - 2 for _ in range(M) for il in range(L)], N), c, 0.0)
    c = np.ascontiguousarray(c / np.sqrt(o.norm(c)))
    prop.set_state(c)
    if gauge == "vgwr":
        ang, f = po.ep_angular(M, L, m0), (0.9, 1.1, -0.5, 0.3)
        o.set_ep(ang, isub=isub)
        prop.upload_angular_ep(ang, isub=isub)
        o.step_ep(c, *f)
        prop.propagate_ep(*f)
    else:
        ang, f = po.lgwr_angular(M, L, m0), (0.05, 0.06, -0.03, 0.02)
        o.set_lgwr(ang, isub=isub)
        prop.upload_angular_lgwr(ang, isub=isub)
        o.step_lgwr(c, *f)
        prop.propagate_lgwr(*f)
    err = rel_l2(prop.get_state(), c)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err <= 1e-12
    prop.close()


@pytest.mark.parametrize("p", [7, 8])
def test_batched_and_single_time_points_agree(p):
    """The tables of a run's time points are factorised together, those of
    single steps one time point at a time, by different kernels: 16 steps
    either way (20 R-part tables and 40 D-part tables of 25 partitions)."""
    N, L, nt = 600, 40, 16
    print(f"case: batched against single time points N={N} L={L} p={p}", flush=True)
    o, prop = _pair(N, p, L)
    a = 0.8 * np.sin(0.3 * np.arange(nt + 1)) + 0.1
    c = mixed_state(o, seed=p, amp=0.3)
    prop.set_state(c)
    prop.run(a, nt, 0, nt, use_mask=False)
    ref = prop.get_state().copy()
    prop.set_state(c)
    for k in range(nt):
        prop.propagate(a[k], a[k + 1])
    err = rel_l2(prop.get_state(), ref)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err <= 1e-12
    prop.close()


@pytest.mark.parametrize("gauge", ["vgwr", "lgwr"])
def test_queued_elliptical_steps_match_the_run(gauge):
    """Elliptical steps called one by one return when queued, each call's
    tables in the other of two sets: seven steps in a row against the run's."""
    import pyoracle as po
    M, L, N, n = 5, 6, 150, 7
    print(f"case: queued elliptical steps {gauge}", flush=True)
    o, prop = _pair(N, 7, L, M, -2)
    f = 0.6 if gauge == "vgwr" else 0.05
    ax, ay = (f * np.cos(0.4 * np.arange(n + 1) + ph) for ph in (0.0, 1.1))
    if gauge == "vgwr":
        prop.upload_angular_ep(po.ep_angular(M, L, -2))
        step, run = prop.propagate_ep, prop.run_ep
    else:
        prop.upload_angular_lgwr(po.lgwr_angular(M, L, -2))
        step, run = prop.propagate_lgwr, prop.run_lgwr
    c = mixed_state(o, seed=3, amp=0.3)
    prop.set_state(c)
    run(ax, ay, n, 0, n, use_mask=True)
    ref = prop.get_state().copy()
    prop.set_state(c)
    for k in range(n):
        step(ax[k], ax[k + 1], ay[k], ay[k + 1])
        prop.mask()
    err = rel_l2(prop.get_state(), ref)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err <= 1e-12
    prop.close()


@pytest.mark.parametrize("p", [7, 8])
@pytest.mark.parametrize("N,L,kmax", [(18, 1, 1), (33, 2, 3), (127, 3, 8), (128, 3, 9), (129, 2, 8), (255, 1, 8),
                                      (256, 3, 2), (257, 3, 8), (700, 2, 12)])
def test_krylov_step_at_tile_edges(N, L, kmax, p):
    """The Lanczos vector's kernels around their tiles of 128 and 256 rows
    (with p rows on either side), one channel and several, subspaces from one
    vector on.  Bar: 1e-10, as the other sizes' in test_gpu_parity."""
    import pyoracle as po
    print(f"case: krylov edges N={N} L={L} p={p} kmax={kmax}", flush=True)
    o, prop = _pair(N, p, L)
    prop.upload_krylov(o.get(po.QOR_H), o.get(po.QOR_Y10), o.get(po.QOR_Q10))
    c = mixed_state(o, seed=N + p, amp=0.3)
    ref = c.copy()
    _, m_o, eps_o, ab_o = o.krylov_step(ref, 0.7, 0.002, kmax=kmax)
    prop.set_state(c)
    _, m, eps = prop.krylov_step(0.7, 0.002, kmax=kmax)
    err = rel_l2(prop.get_state(), ref)
    print(f"  m={m}/{m_o} eps={eps:.2e}/{eps_o:.2e} rel L2 {err:.2e}", flush=True)
    assert m == m_o
    assert err <= 1e-10
    prop.close()


@pytest.mark.parametrize("p", [7, 8])
@pytest.mark.parametrize("N", [18, 40, 1023, 1024, 1025, 1031, 2049])
def test_recorded_observables_at_block_edges(N, p):
    """All eight recorded observables of a state around the 1024 rows that a
    block takes at a time (with p rows after them), three m blocks.  Bars as
    the single observables' in test_gpu_observe."""
    import pyoracle as po
    import qpc_gpu
    print(f"case: observables edges N={N} p={p}", flush=True)
    L, M, m0 = 3, 3, -1
    cfg = shape(N, L, 0.2 * N, M=M, m0=m0, p=p)
    o, prop = _pair(N, p, L, M, m0)
    st = qpc_gpu.Setup(N, p, L, M, m0, cfg["dt"], 0.0, cfg["rmax"], 1.0, 1.0, cfg["mask_rmin"], cfg["mask_rmax"],
                       cfg["mask_fact"])
    prop.upload_outer(st.get(qpc_gpu.SETUP_SOUTER))
    prop.upload_accel(o.get(po.QOR_DVDR))
    c = mixed_state(o, seed=N + p, amp=0.5)
    prop.set_state(c)
    prop.record(qpc_gpu.REC_ALL, 1)
    prop.run(np.zeros(2), 0, 0, 1, use_mask=False)
    h = prop.record_read()[0]
    ref = [o.norm(c), o.dipole_z(c, 0), o.dipole_z(c, 1), o.outer_norm(c, cfg["mask_rmin"]), *o.dipole_xy(c, 0),
           *o.dipole_xy(c, 1)]
    for g, r in zip(h, ref):
        assert abs(g - r) <= 1e-12 * max(1.0, abs(r))
    prop.close()


@pytest.mark.parametrize("p", [7, 8])
@pytest.mark.parametrize("N", [192, 745, 767, 768, 769, 793])
def test_steps_where_the_solve_changes_kernel(N, p):
    """Channels of up to 32 partitions (768 rows) have eight lanes per
    partition in the solves, longer ones one: steps on either side of the line
    against the oracle, and the same bits however the channel is segmented."""
    print(f"case: solve kernels N={N} p={p}", flush=True)
    o, prop = _pair(N, p, 3, M=3, m0=-1)
    c = mixed_state(o, seed=N + p, amp=0.3)
    ref = c.copy()
    out = []
    for seg in (0, 1, 3):
        prop.set_tune(seg_add=seg)
        prop.set_state(c)
        for a in ((0.7, 0.9), (0.9, -0.4)):
            prop.propagate(*a)
        prop.propagate()
        prop.mask()
        out.append(prop.get_state().copy())
    for a in ((0.7, 0.9), (0.9, -0.4)):
        o.step(ref, *a)
    o.step_free(ref)
    o.mask(ref)
    err = rel_l2(out[0], ref)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err <= 1e-12
    assert all(np.array_equal(x, out[0]) for x in out[1:])
    prop.close()


@pytest.mark.parametrize("N,p", [(769, 7), (1000, 8), (1537, 7), (1801, 8), (2305, 7)])
def test_steps_whichever_solve_kernel_runs(N, p):
    """Long channels on small grids are cut into segments with eight lanes per
    partition, on large ones run with one: the same bits either way, and the
    oracle's steps."""
    print(f"case: solve kernels on long channels N={N} p={p}", flush=True)
    o, prop = _pair(N, p, 3, M=3, m0=-1)
    c = mixed_state(o, seed=N + p, amp=0.3)
    ref = c.copy()
    out = []
    for seg, grid in ((0, 512), (3, 512), (0, 0), (1, 0)):
        prop.set_tune(seg_add=seg, stage_grid=grid)
        prop.set_state(c)
        for a in ((0.7, 0.9), (0.9, -0.4)):
            prop.propagate(*a)
        prop.propagate()
        prop.mask()
        out.append(prop.get_state().copy())
    for a in ((0.7, 0.9), (0.9, -0.4)):
        o.step(ref, *a)
    o.step_free(ref)
    o.mask(ref)
    err = rel_l2(out[0], ref)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err <= 1e-12
    assert all(np.array_equal(x, out[0]) for x in out[1:])
    prop.close()


@pytest.mark.parametrize("p", [7, 8])
def test_tables_have_the_same_bits_however_many_are_factorised(p):
    """A run factorises its time points' tables together (17 time points of 20
    and 40 tables), a step one time point's, by different kernels.  With a
    recorded observable the run hands the whole state over between steps as the
    single calls do, so that equal tables give equal states in every bit."""
    import qpc_gpu
    N, L, nt = 600, 40, 16
    print(f"case: bits of batched and single tables N={N} L={L} p={p}", flush=True)
    o, prop = _pair(N, p, L)
    a = 0.8 * np.sin(0.3 * np.arange(nt + 1)) + 0.1
    c = mixed_state(o, seed=p, amp=0.3)
    prop.set_state(c)
    prop.record(qpc_gpu.REC_NORM, nt)
    prop.run(a, nt, 0, nt, use_mask=False)
    ref = prop.get_state().copy()
    prop.set_state(c)
    for k in range(nt):
        prop.propagate(a[k], a[k + 1])
    got = prop.get_state()
    print(f"  rel L2 {rel_l2(got, ref):.2e}", flush=True)
    assert np.array_equal(got, ref)
    prop.close()


@pytest.mark.parametrize("gauge", ["vg", "lg"])
def test_refused_step_leaves_the_next_one_right(gauge):
    """A step with a non-finite field value is refused; the loop goes on from
    the step before it, whose last time point's tables and scalars are kept."""
    import qpc_gpu
    N, L = 240, 4
    print(f"case: refused step {gauge}", flush=True)
    o, prop = _pair(N, 7, L)
    step, ref_step = (prop.propagate, o.step) if gauge == "vg" else (prop.propagate_lg, o.step_lg)
    f = 0.9 if gauge == "vg" else 0.05
    c = mixed_state(o, seed=5, amp=0.3)
    prop.set_state(c)
    step(f, 0.8 * f)
    for bad in ((0.5 * f, np.nan), (np.inf, 0.5 * f), (0.8 * f, np.nan)):
        with pytest.raises(qpc_gpu.QpcError):
            step(*bad)
    step(0.8 * f, 0.6 * f)
    for a in ((f, 0.8 * f), (0.8 * f, 0.6 * f)):
        ref_step(c, *a)
    err = rel_l2(prop.get_state(), c)
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err <= 1e-12
    prop.close()
