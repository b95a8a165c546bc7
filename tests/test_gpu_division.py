"""FP64 populations far from 1 and the reciprocal division (fused.h div_by,
div_safe): where it does not apply -- tiny, zero, huge or non-finite
populations, rates beyond its divisors -- the IEEE division is taken, and
both give the oracle's arithmetic bit for bit."""
import numpy as np
import pytest

from oracle.oracle import LDC, TGV, CONFIG, FAITHFUL, Oracle

pytestmark = pytest.mark.gpu

N = (36, 20, 3)  # tiled
SMALL = (12, 10, 9)  # structure of arrays


def fields(n, seed):
    r = np.random.default_rng(seed)
    return r.uniform(0.5, 1.5, (27, n[2], n[1], n[0])) * r.choice([-1.0, 1.0], (27, n[2], n[1], n[0]))


# 2^-1060: products and remainders of the reciprocal form are subnormal; 2^-601
# and 2^401: just outside div_safe, 2^-600 and 2^400 just inside; 0: every wavefront
# on the IEEE side; "mixed": one wavefront in a few has a tiny population
@pytest.mark.parametrize("scale", [2.0 ** -1060, 2.0 ** -1000, 2.0 ** -601, 2.0 ** -599, 1e-30, 2.0 ** 399, 2.0 ** 401, "mixed", 0.0])
@pytest.mark.parametrize("n", [N, SMALL])
@pytest.mark.parametrize("storage", ["pull", "aa"])
def test_scaled_populations(scale, n, storage):
    from imexlb_amd import LBM
    print(f"[case] division scale {scale} {n} {storage}", flush=True)
    f = fields(n, 7)
    if scale == "mixed":
        f[3, :, ::7, ::5] *= 2.0 ** -900
    else:
        f *= scale
    # one step from the same post-collision populations in every address mode
    # that the oracle's tests check, and by hand
    out = []
    for am in (-1, 2):
        g = LBM(*n, 0.013, u0=0.05, storage=storage, addr_mode=am)
        g.Initialize()
        g.set_f(f)
        g.step(1)
        out.append((g.get_f(), g.moments()))
        g.close()
    with np.errstate(all="ignore"):
        want, mom = by_hand(f, 0.013)
    for got, m in out:
        for a, b in zip(m, mom):
            assert np.array_equal(a, b, equal_nan=True)
        assert np.array_equal(got, want, equal_nan=True)


def by_hand(f, tau0):
    """One TGV step in the oracle's order of operations."""
    from oracle import oracle_np as O
    g = np.empty_like(f)
    for q in range(27):
        e = O.E[q]
        g[q] = np.roll(f[q], (int(e[2]), int(e[1]), int(e[0])), axis=(0, 1, 2))
    p = np.zeros(g.shape[1:])
    u, v, w = np.zeros_like(p), np.zeros_like(p), np.zeros_like(p)
    for q in range(27):
        p = p + g[q] / 3.0
        for s, a in ((0, "u"), (1, "v"), (2, "w")):
            if O.E[q, s] == 0:
                continue
            d = g[q] if O.E[q, s] > 0 else -g[q]
            if a == "u":
                u = u + d
            elif a == "v":
                v = v + d
            else:
                w = w + d
    udu = u * u + v * v + w * w
    out = np.empty_like(g)
    for q in range(27):
        terms = [(u, v, w)[s] if O.E[q, s] > 0 else -(u, v, w)[s] for s in range(3) if O.E[q, s] != 0]
        edu = np.zeros_like(p)
        for k, t in enumerate(terms):
            edu = t if k == 0 else edu + t
        t = O.W[q]
        feq = t * p * 3.0 + t * (3.0 * edu + 4.5 * (edu * edu) - 1.5 * udu)
        out[q] = g[q] - (g[q] - feq) / (tau0 + 0.5)
    return out, [p, u, v, w]


@pytest.mark.parametrize("tau0", [-0.4999, -0.4, 0.0, 0.25, 1.0 / 3.0, 7.0, 3e9])
@pytest.mark.parametrize("case,mode", [(TGV, FAITHFUL), (LDC, CONFIG)])
def test_rates(tau0, case, mode):
    from imexlb_amd import LBM
    print(f"[case] division tau0 {tau0} case {case}", flush=True)
    g = LBM(*N, tau0, u0=0.05, case=case, mode=mode, storage="aa")
    o = Oracle(case, *N, tau0=tau0, u0=0.05, mode=mode, lid_u=0.1)
    g.Initialize()
    o.Initialize()
    g.step(3)
    o.run(3)
    for a, b in zip(o.moments(), g.moments()):
        assert np.array_equal(a, b, equal_nan=True)
    g.close()
