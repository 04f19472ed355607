"""ShotBuckets.get_states hands every shot an array of its own: a caller that
keeps one shot does not keep its bucket's whole block, and may resize it."""
import numpy as np

import qpc_gpu


class _Block:
    """Stands for a bucket's context: its state is the channel numbers."""

    def __init__(self, nch, N):
        self.state = np.repeat(np.arange(nch, dtype=np.complex128), N)

    def get_state(self):
        return self.state.copy()


def test_states_own_their_data():
    N, ldim = 5, [3, 1, 4, 2, 4]
    b = object.__new__(qpc_gpu.ShotBuckets)
    b.N, b.ldim = N, ldim
    b.groups = qpc_gpu.bucket_shots(ldim, 2)
    b.Lb = [max(ldim[k] for k in g) for g in b.groups]
    b.props = [_Block(len(g) * Lb, N) for g, Lb in zip(b.groups, b.Lb)]
    out = b.get_states()
    for g, Lb in zip(b.groups, b.Lb):
        for q, k in enumerate(g):
            assert np.array_equal(out[k], np.repeat(np.arange(q * Lb, q * Lb + ldim[k]), N))
    for x in out:
        assert x.base is None and x.flags.owndata and x.flags.writeable
    out[0].resize(2 * N, refcheck=False)
