"""Host arrays through the pinned buffers, which start small, grow with a
larger transfer and are shared by the contexts of every thread: what an upload
writes a download returns bit for bit, halos included, for one field of one
chunk, of two, and whole states, small boxes before and after large ones, alone
and from several threads at once."""
import threading

import numpy as np
import pytest

import astr_gpu_amd as ag

pytestmark = pytest.mark.gpu

# fields of one chunk of 512 KB (16^3, 24^3), of two (32x31x33, 40x32x36), more
DIMS = [(16, 16, 16), (24, 24, 24), (40, 32, 36), (64, 70, 60), (32, 31, 33), (17, 16, 19)]


def roundtrip(dims, seed, reps=2):
    p = ag.default_params(dims)
    s = ag.AstrSolver(p)
    rng = np.random.default_rng(seed)
    shp = ag.haloed_shape(p)
    for _ in range(reps):
        st = {nm: np.asfortranarray(rng.standard_normal(shp + ext)) for nm, ext in
              (("q", (5,)), ("rho", ()), ("vel", (3,)), ("prs", ()), ("tmp", ()))}
        s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
        out = s.download_state()
        for nm in st:
            assert np.array_equal(out[nm], st[nm]), (dims, nm)
        # one field up and one down: linear, so twice the field is twice the
        # derivative exactly
        a, b = s.central(2, st["rho"]), s.central(2, 2.0 * st["rho"])
        assert np.array_equal(2.0 * a, b), dims
    s.close()


def test_sizes_in_turn_without_another_context():
    for n, dims in enumerate(DIMS + DIMS[::-1]):
        print(f"case transfer {dims}", flush=True)
        roundtrip(dims, n)


def test_sizes_while_a_context_holds_the_buffers():
    keep = ag.AstrSolver(ag.default_params((16, 16, 16)))
    for n, dims in enumerate(DIMS + DIMS[::-1]):
        roundtrip(dims, n)
    keep.close()


def test_threads():
    errors = []

    def work(n):
        try:
            for k in range(3):
                roundtrip(DIMS[(n + k) % len(DIMS)], 10 * n + k, 1)
        except BaseException as e:  # handed to the test's thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(n,)) for n in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
