"""Serving pools: a request's results do not depend on the requests beside it, bit for bit, also where
the requests are so small that several of them together fit one walk group."""
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
@pytest.mark.parametrize("kind,sizes", [("plummer", (2, 20, 40, 3)), ("plummer", (64, 64, 65)),
                                        ("sphere", (20, 24, 40, 20))])
def test_requests_smaller_than_a_walk_group(kind, sizes, precision):
    from gandalf_amd import serving as S
    requests = [S.make_request_ic(kind, n, 50 + k) for k, n in enumerate(sizes)]
    check(S.class_params(kind), precision, requests, 2,
          ("r", "v", "a", "gpot") if kind == "plummer" else FIELDS)
