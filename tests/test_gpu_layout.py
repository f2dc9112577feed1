"""Launches whose LDS is sized by the decoded expressions, against the CPU oracle
(the sizes themselves: tests/test_layout.py)."""
import numpy as np
import pytest

from cusr_amd.benchmark import popio
from oracle import lm_oracle
from tests.helpers import f64

pytestmark = pytest.mark.gpu

VAR, CONST, UN, BIN = popio.NODE_VAR, popio.NODE_CONST, popio.NODE_UFUNC, popio.NODE_BFUNC
ADD, MUL, SIN = 1, 3, 14


def _tree(k, D):
    """sin(c0 + ... + c_{k-1}) * x_{D-1}"""
    nt = [BIN, UN] + [BIN] * (k - 1) + [CONST] * k + [VAR]
    nv = [float(MUL), float(SIN)] + [float(ADD)] * (k - 1) + [0.0] * k + [float(D - 1)]
    return nt, nv, [-1] * (k + 1) + list(range(k)) + [-1]


@pytest.mark.parametrize("D", [3, 12])     # fast and wide programs
@pytest.mark.parametrize("k_max", [0, 2])
def test_evaluate_with_understated_k_max(co, D, k_max):
    """The header's K_max is no bound on the expressions' own: constants and C's
    values keep their place beside the rows."""
    rng = np.random.default_rng(5)
    xs = rng.uniform(-2, 2, (700, D)).astype(np.float32)
    slots = [(*_tree(k, D), rng.standard_normal(k).astype(np.float32)) for k in (1, 3, 7, 16, 20)]
    pop = popio.build_pop(slots, xs, np.zeros((len(slots), 700)))
    c0, x64, _ = f64(pop)
    under = dict(pop, K_max=k_max)
    print(f"evaluate D={D} K_max={k_max} of {pop['K_max']}", flush=True)
    want = lm_oracle.eval_pop(pop, c=c0, xs=x64)
    assert np.array_equal(co.evaluate(under, c0, x64), want)
    # fp32: k - 1 sums, each within 2^-24 of a partial sum of at most sum |c|, go through
    # the sine (slope at most 1) and the factor x; the sine, the product and the
    # operands' own rounding are a few 2^-24 of |x|
    single = co.evaluate(under, c0, x64, precision=1)
    for m, (_, _, _, c) in enumerate(slots):
        bound = (len(c) * np.abs(c).sum() + 8) * 2.0 ** -24 * np.abs(x64[:, D - 1])
        assert np.all(np.abs(single[m] - want[m]) <= bound), m


@pytest.mark.parametrize("opts", [dict(), dict(ad_mode=1), dict(partitions=8),
                                  dict(partitions=1, precision=1)])
def test_constants_alone_in_padded_kernels(co, opts):
    """Expressions without variables in groups of K bins: a scalar area and no rows,
    whose tangents a padded kernel reads up to its own K."""
    rng = np.random.default_rng(11)
    xs = rng.uniform(-2, 2, (1100, 3)).astype(np.float32)
    slots = []
    for k in (1, 1, 2, 3, 5, 7, 9, 11, 13, 14, 20):
        nt, nv, ci = _tree(k, 3)
        slots.append((nt[1:-1], nv[1:-1], ci[1:-1], rng.standard_normal(k).astype(np.float32)))
        slots.append((*_tree(k, 3), rng.standard_normal(k).astype(np.float32)))
    y = rng.standard_normal((len(slots), 1100)).astype(np.float32)
    pop = popio.build_pop(slots, xs, y)
    print(f"constants alone M={pop['M']} {opts}", flush=True)
    g = co.optimize_ex(pop, 6, **opts)
    o = lm_oracle.fit(pop, max_iter=6, **opts)
    if opts.get("precision"):
        # fp32 partials: each step's path may differ; the fp64 losses at the start do not
        assert np.array_equal(g["loss_init"], o["loss_init"])
        return
    for k in ("status", "loss_init", "loss_final", "iters", "c_final"):
        assert np.array_equal(g[k], o[k], equal_nan=True), k


def test_long_tape_beside_staged_expressions(co):
    """Reverse AD near the LDS limit: a chain whose tape nearly fills it beside an
    expression whose staged rows and scalars pass its plain program's. Each fits by
    itself, and so does their launch (areas by their largest each: 164,416 bytes of
    the 163,840; the plain programs: 161,040)."""
    rng = np.random.default_rng(3)
    N = 1000
    xs = rng.uniform(-1, 1, (N, 1)).astype(np.float32)
    chain = ([UN] * 260 + [BIN, CONST, VAR],
             [float(SIN if i % 2 else 15) for i in range(260)] + [float(MUL), 0.0, 0.0],
             [-1] * 261 + [0, -1], rng.standard_normal(1).astype(np.float32))
    # 17 constants: sin(c c) x, then c f(x) and c with f in sin, cos, square
    nt, nv, ci, K = [BIN] * 17 + [BIN, UN, BIN, CONST, CONST, VAR], [float(ADD)] * 17, [], 2
    nv += [float(MUL), float(SIN), float(MUL), 0.0, 0.0, 0.0]
    ci = [-1] * 20 + [0, 1, -1]
    for i in range(15):
        nt += [BIN, CONST, UN, VAR]
        nv += [float(MUL), 0.0, float((SIN, 15, 34)[i % 3]), 0.0]
        ci += [-1, K, -1, -1]
        K += 1
    nt += [UN, UN, VAR, VAR]
    nv += [float(SIN), float(SIN), 0.0, 0.0]
    ci += [-1, -1, -1, -1]
    slots = [chain, (nt, nv, ci, (0.3 * rng.standard_normal(K)).astype(np.float32))]
    pop = popio.build_pop(slots, xs, rng.standard_normal((2, N)).astype(np.float32))
    print("long tape beside staged rows", flush=True)
    g = co.optimize_ex(pop, 5, ad_mode=1, partitions=1)
    o = lm_oracle.fit(pop, max_iter=5, ad_mode=1, partitions=1)
    for k in ("status", "loss_init", "loss_final", "iters", "c_final"):
        assert np.array_equal(g[k], o[k], equal_nan=True), k
