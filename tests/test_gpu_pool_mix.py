"""Serving pools: a request's results do not depend on the requests beside it, bit for bit, also

* where another request's smoothing lengths outgrow their search radii in a step (its force pass
  then walks for its own candidates), in both precisions;
* where the requests are so small that several of them together fit one walk group."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("r", "v", "a", "h", "u", "rho", "gpot")


def run(params, precision, requests, nsteps, fields):
    from gandalf_amd.gpu import GpuPool
    pool = GpuPool(params, precision, max_particles=1 << 16)
    ids = [pool.admit(q["r"], q["v"], q["m"], q["u"], nsteps) for q in requests]
    for _ in range(nsteps):
        pool.step()
    return [{f: pool.get(i, f) for f in fields} for i in ids]


def check(params, precision, requests, nsteps, fields=FIELDS):
    mix = run(params, precision, requests, nsteps, fields)
    for k, q in enumerate(requests):
        (alone,) = run(params, precision, [q], nsteps, fields)
        for f in fields:
            assert np.all(np.isfinite(alone[f])), (k, f)
            assert np.array_equal(alone[f], mix[k][f]), \
                (k, f, float(np.max(np.abs(alone[f] - mix[k][f]))))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", [0, 1])
def test_quiet_request_beside_an_expanding_one(precision, order):
    """Steps of 0.03: the expanding spheres' smoothing lengths grow by 15 % a step, past the search
    radius of 1.05 h, and need a retry; the quiet ones' do not."""
    from gandalf_amd import serving as S
    params = dict(S.class_params("sphere"), fixed_dt=0.03)
    quiet, wild = (S.make_request_ic("sphere", n, seed) for n, seed in ((3000, 5), (2000, 6)))
    third = S.make_request_ic("sphere", 1500, 7)
    wild["v"] = 5.0 * wild["r"]
    requests = [quiet, wild, third] if order == 0 else [wild, quiet, third]
    check(params, precision, requests, 3)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_quiet_request_beside_one_that_outgrows_its_lists(precision):
    """The same with candidate lists of one batch to start with, which the first step has to grow;
    its length is the Courant step of the set-up, here a long one that needs retries as well."""
    from gandalf_amd import serving as S
    params = dict(S.class_params("sphere"), fixed_dt=0.03, cand_batches_init=1, courant_mult=1.0)
    quiet, wild = (S.make_request_ic("sphere", n, seed) for n, seed in ((3000, 5), (2000, 6)))
    wild["v"] = 5.0 * wild["r"]
    check(params, precision, [quiet, wild], 3)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,sizes", [("plummer", (2, 20, 40, 3)), ("plummer", (64, 64, 65)),
                                        ("sphere", (20, 24, 40, 20))])
def test_requests_smaller_than_a_walk_group(kind, sizes, precision):
    from gandalf_amd import serving as S
    requests = [S.make_request_ic(kind, n, 50 + k) for k, n in enumerate(sizes)]
    check(S.class_params(kind), precision, requests, 2,
          ("r", "v", "a", "gpot") if kind == "plummer" else FIELDS)
