"""Grouped launches: bins of few expressions run in the padded kernel of their
group's largest K. The same expressions, alone (grouped) and repeated until
every bin is launched by itself, must give the same bits. At 70 points a pass is one
batch, in which constant subtrees are not staged; at 1,100 (two partitions of nine
granules) they are."""
import numpy as np
import pytest

from cusr_amd.benchmark import gen_synth, popio
from oracle import lm_oracle

pytestmark = pytest.mark.gpu

KS = (0, 1, 3, 4, 5, 8, 9, 11, 12, 13, 15, 16)   # both ends of every group
KEYS = ("status", "loss_init", "loss_final", "iters")


def _constant_operators(nt):
    """Operators of a prefix tree over constants alone."""
    stack, n = [], 0
    for t in reversed(nt):
        arity = {popio.NODE_BFUNC: 2, popio.NODE_UFUNC: 1}.get(int(t), 0)
        alone = all([stack.pop() for _ in range(arity)]) if arity else t == popio.NODE_CONST
        n += bool(arity and alone)
        stack.append(alone)
    return n


def _pops(N, copies, per_k=6):
    cfg = gen_synth.scaled(gen_synth.CONFIGS["C3"], M=per_k, N=N)
    rng = np.random.default_rng(77)
    xs = rng.uniform(-2, 2, (N, cfg.D)).astype(np.float32)
    slots = []
    for K in KS:
        cfg.k_lo = cfg.k_hi = K
        for _ in range(per_k):
            nt, nv, ci, k = gen_synth.random_tree(rng, cfg)
            slots.append((nt, nv, ci, rng.standard_normal(k).astype(np.float32)))
    for ks in ((1, 3, 4), (5, 8), (9, 11, 12), (13, 15)):   # every group has some to stage
        assert sum(_constant_operators(nt) for nt, _, _, c in slots if len(c) in ks) > 0, ks
    y = rng.standard_normal((len(slots), N)).astype(np.float32)
    one = popio.build_pop(slots, xs, y)
    return one, popio.build_pop(slots * copies, xs, np.tile(y, (copies, 1)))


@pytest.mark.parametrize("N", [70, 1100])
@pytest.mark.parametrize("opts", [dict(), dict(ad_mode=1), dict(precision=1),
                                  dict(ad_mode=1, precision=1), dict(partitions=8),
                                  dict(partitions=8, ad_mode=1, precision=1)])
def test_grouped_bins_equal_single_bins(co, opts, N):
    # wavefronts per bin: 6 or 12 (48) alone; from 1,080 (1,080 x 8 on the split path) repeated
    one, many = _pops(N, 180)
    print(f"grouped N={N} M={one['M']} against M={many['M']} {opts}", flush=True)
    a, b = co.optimize_ex(one, 4, **opts), co.optimize_ex(many, 4, **opts)
    M, C = one["M"], one["total_c"]
    for k in KEYS:
        assert np.array_equal(a[k], b[k][:M], equal_nan=True), k
        assert np.array_equal(b[k][:M], b[k][-M:], equal_nan=True), k
    assert np.array_equal(a["c_final"], b["c_final"][:C], equal_nan=True)
    if not opts.get("precision"):
        o = lm_oracle.fit(one, max_iter=4, **opts)
        assert np.array_equal(a["status"], o["status"])
        assert np.array_equal(a["loss_final"], o["loss_final"], equal_nan=True)
