"""Per-bead getters of a replica whose slots the spatial reorder has permuted."""
import threading

import numpy as np
import pytest

import decks
import tild

pytestmark = pytest.mark.gpu


def test_threads_read_one_reordered_engine(tmp_path):
    # positions, forces and restart displacement go through one device buffer: threads that
    # read the engine together each get the array they asked for
    text, d = decks.melt3d(tmp_path, n_chains=600, N=10, box=(12.0, 12.0, 12.0), grid=(24, 24, 24), integrator="GJF",
                           delt=0.01)
    s = tild.System(text, d)
    e = tild.Engine(s, device=0, seed=3, reorder_every=4)
    e.step(10)
    f = e.forces()
    want = {"positions": e.positions(), "state": e.state()[1], "forces": f}
    get = {"positions": e.positions, "state": lambda: e.state()[1], "forces": e.get_forces}
    wrong = []

    def read(name):
        for _ in range(50):
            if not np.array_equal(get[name](), want[name]):
                wrong.append(name)

    threads = [threading.Thread(target=read, args=(k,)) for k in want for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    e.close()
    assert not wrong, wrong
