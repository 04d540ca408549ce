"""Several host threads read the fields of one engine at a time: every read
gives that field."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scatter", ["colored", "gather"])
def test_threads_read_one_engine(scatter):
    from specfempp_amd import Engine2D, meshes

    n = 24
    mesh = meshes.quad_mesh(n, n, 0, n * 20.0, 0, n * 20.0, materials=[meshes.elastic(2400.0, 3000.0, 1732.0)])
    e = Engine2D(mesh, [], [], 1e-3, 4, 1, (), scatter=scatter)
    e.initialize()
    rng = np.random.default_rng(1)
    want = {k: rng.standard_normal(e.field(k).shape).astype(np.float32)
            for k in ("displacement", "velocity", "acceleration")}
    for k, v in want.items():
        e.set_field(k, v)
    print(f"[case] threads {scatter}", flush=True)
    wrong = []

    def read(k):
        for _ in range(20):
            if not np.array_equal(e.field(k), want[k]):
                wrong.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    e.close()
    assert not wrong
