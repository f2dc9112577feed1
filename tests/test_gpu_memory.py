"""A handle when device memory runs out (an allocation is refused, nothing else), and
fits whose V workspace passes the limit."""
import ctypes

import numpy as np
import pytest

from cusr_amd.benchmark import popio
from cusr_amd.kernel import co_inproc as ci
from oracle import lm_oracle
from tests.helpers import f64

pytestmark = pytest.mark.gpu

KEYS = ("c_final", "status", "loss_init", "loss_final", "iters")
VAR, CONST, UN, BIN = popio.NODE_VAR, popio.NODE_CONST, popio.NODE_UFUNC, popio.NODE_BFUNC
ADD, MUL, SIN = 1, 3, 14
N = 1_000_000


def _say(msg):
    print(f"[memory] {msg}", flush=True)


def _hip():
    """The HIP runtime that the library runs on."""
    with open("/proc/self/maps") as f:
        paths = {line.split()[-1] for line in f if "libamdhip64" in line}
    assert len(paths) == 1, paths
    return ctypes.CDLL(paths.pop())


def _memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value, total.value


def _pop(copies):
    """copies of four expressions f(x0) c0 + sin(x1) c1 + sin(x0 x1) c2, which keep three
    V columns each, and one target."""
    rng = np.random.default_rng(9)
    xs = rng.uniform(-2, 2, (N, 2)).astype(np.float32)
    nt = [BIN, BIN, BIN, UN, VAR, CONST, BIN, UN, VAR, CONST, BIN, UN, BIN, VAR, VAR, CONST]
    nv = [ADD, ADD, MUL, SIN, 0, 0, MUL, SIN, 1, 0, MUL, SIN, MUL, 0, 1, 0]
    ranks = [-1, -1, -1, -1, -1, 0, -1, -1, -1, 1, -1, -1, -1, -1, -1, 2]
    slots = [(nt, nv[:3] + [f] + nv[4:], ranks, rng.standard_normal(3).astype(np.float32))
             for f in (14, 15, 33, 34)]
    y = rng.standard_normal((1, N)).astype(np.float32)
    one = popio.build_pop(slots, xs, np.broadcast_to(y, (4, N)))
    M = 4 * copies
    many = dict(one, M=M, total_nodes=M * 16, total_c=M * 3, nt=np.tile(one["nt"], copies),
                nv=np.tile(one["nv"], copies), ci=np.tile(one["ci"], copies),
                c_init=np.tile(one["c_init"], copies), ym=y, shared_y=True,
                metas=np.array([(16 * m, 16, 3 * m, 3) for m in range(M)], np.int32))
    return one, many


@pytest.fixture()
def own():
    """A handle whose buffers no other test has grown."""
    with ci.InProcessCO(device_id=0, variant="ad") as co:
        yield co


def test_call_after_a_refused_allocation(own):
    """An allocation beyond the device is refused, and the next calls are not."""
    one, _ = _pop(1)
    x, y = np.zeros(1), np.zeros(1)
    _say("data set of 4 TB refused")
    rc = own._lib.co_data_upload(own._handle, 2**31 - 1, 255, x.ctypes.data_as(ctypes.c_void_p),
                                 y.ctypes.data_as(ctypes.c_void_p))
    assert rc == ci.CO_ERR_OOM
    c0, x64, _ = f64(one)
    assert np.array_equal(own.evaluate(one, c0, x64), lm_oracle.eval_pop(one, c=c0, xs=x64))


@pytest.mark.parametrize("opts", [dict(), dict(partitions=2), dict(ad_mode=1),
                                  dict(precision=1), dict(precision=1, partitions=4),
                                  dict(ad_mode=1, precision=1)])
def test_fits_without_workspaces(own, opts):
    """V run in every pass gives the bits that its kept values give: four expressions
    whose columns take 96 MB, and 500 copies whose columns would take 48 GB."""
    _, few = _pop(1)
    _, many = _pop(500)
    own.upload_data(*f64(many)[1:])
    kept = own.optimize_data(few, 4, **opts)
    free, total = _memory()
    assert 8 * 3 * N * many["M"] > total // 8
    _say(f"fit without workspaces {opts}")
    run = own.optimize_data(many, 4, **opts)
    assert free - _memory()[0] < 4 << 30
    for k in KEYS:
        assert np.array_equal(run[k].reshape(500, -1), np.tile(kept[k], (500, 1)),
                              equal_nan=True), k
