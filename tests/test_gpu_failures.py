"""GPU: calls of the runtime that fail on the host (a launch, an allocation, a
thread), and devices of few CUs, forced by a shim between the library and the
HIP runtime.  The library must then stand as before the call, and go on."""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

HEADER = """
import ctypes, os, sys
sys.path[:0] = [{root!r}, os.path.join({root!r}, "tests")]
shim = ctypes.CDLL({shim!r}, mode=ctypes.RTLD_GLOBAL)
shim.shim_fail_launch.argtypes = [ctypes.c_long]
shim.shim_launches_left.restype = ctypes.c_long
shim.shim_fail_malloc.argtypes = [ctypes.c_size_t, ctypes.c_long]
import numpy as np
from conftest import make_corpus
from lda_sc20_amd import ezlda
from oracle import binding as ob

def context(off, words, V, K, seed=21, **kw):
    ctx = ezlda.Context(K=K, alpha=50.0 / K, beta=0.01, seed=seed, **kw)
    ctx.load(ezlda.Corpus(V, off, words))
    return ctx

def failing(call):
    try:
        call()
    except ezlda.EzldaError:
        return True
    return False
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    cc = shutil.which("g++")
    if cc is None:
        pytest.skip("no C++ compiler")
    so = tmp_path_factory.mktemp("shim") / "libshim.so"
    subprocess.run([cc, "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", os.path.join(ROOT, "tests", "hip_shim.cpp"),
                    "-o", str(so), "-ldl", "-lpthread"], check=True)
    return str(so)


def _run(shim, body):
    """The body in a process of its own, with the shim between the library and the runtime."""
    r = subprocess.run([sys.executable, "-c", HEADER.format(root=ROOT, shim=shim) + body], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-3000:]
    return r.stdout


# every launch of a sweep fails once: the sweep is as if it had not been asked
# for (the sampler's launch is the last), its number included
@pytest.mark.parametrize("call", ["ctx.sweep(1)", "ctx.time_sweeps(1, use_graph=False)"])
def test_a_failed_launch_leaves_the_sweep_undone(shim, call):
    out = _run(shim, f"""
off, words = make_corpus(3, 120, 200, 60)
orc = ob.Oracle(64, float(np.float32(50.0 / 64)), 0.01, 21, 200, off, words)
want = []
for s in range(3):
    orc.sweep(1)
    want.append((orc.get_topics(), orc.loglik()))
j = 0
while True:
    ctx = context(off, words, 200, 64)
    ctx.loglik()
    ctx.sweep(1)
    shim.shim_fail_launch(j)
    if not failing(lambda: {call}):
        assert shim.shim_launches_left() == 0, "no launch failed"
        break
    assert ctx.info().sweep == 1, j
    assert np.array_equal(ctx.get_topics(), want[0][0]), j
    assert abs(ctx.loglik() - want[0][1]) <= 1e-9 * abs(want[0][1]), j
    for s in (1, 2):
        ctx.sweep(1)
        assert ctx.info().sweep == s + 1 and np.array_equal(ctx.get_topics(), want[s][0]), (j, s)
    j += 1
print("launches", j)
""")
    assert int(out.split("launches")[1]) >= 4


# a device of 4 CUs (a partition): every queue of the samplers is still drained
@pytest.mark.parametrize("K", [10000, 2000, 64])
def test_a_device_of_few_cus(shim, K):
    _run(shim, f"""
shim.shim_cus(4)
off, words = make_corpus(5, 150, 400, 60, zipf=1.15)
ctx = context(off, words, 400, {K})
orc = ob.Oracle({K}, float(np.float32(50.0 / {K})), 0.01, 21, 400, off, words)
for s in range(2):
    ctx.sweep(1)
    orc.sweep(1)
    assert np.array_equal(ctx.get_topics(), orc.get_topics()), s
assert abs(ctx.loglik() - orc.loglik()) <= 1e-9 * abs(orc.loglik())
""")


# threads that cannot be started: the caller does their part (the readback of a resident and of a chunked corpus, and
# the layout)
@pytest.mark.parametrize("kw", ["{}", "{'num_chunks': 3}"])
def test_threads_that_cannot_be_started(shim, kw):
    _run(shim, f"""
rng = np.random.default_rng(7)
n = 1100000
off = np.arange(0, n + 1, 100, dtype=np.int64)
words = rng.integers(0, 500, n).astype(np.int32)
z = rng.integers(0, 9, n).astype(np.uint16)
for failing_load in (0, 1):
    shim.shim_fail_threads(failing_load)
    ctx = ezlda.Context(K=9, alpha=0.5, beta=0.01, seed=1, **{kw})
    ctx.load(ezlda.Corpus(500, off, words), z0=z)
    for on in (1, 0):
        shim.shim_fail_threads(on)
        assert np.array_equal(ctx.get_topics(), z), on
    ctx.close()
""")


# the readback's own buffers (4 bytes a token, pinned pieces) are no condition: without them, when loading or given
# back to a later allocation, the topics come through the host
@pytest.mark.parametrize("n", [70001, (1 << 19) + 70001])
@pytest.mark.parametrize("when", ["order", "pinned", "later", "server"])
def test_readback_without_its_buffers(shim, n, when):
    _run(shim, f"""
n, when = {n}, {when!r}
rng = np.random.default_rng(n)
off = np.append(np.arange(0, n, 97, dtype=np.int64), n)
words = rng.integers(0, 300, n).astype(np.int32)
one = n <= 1 << 19
order = (n + 3) // 4 * 4 * (6 if one else 4)  # its allocation, no other of this size
ref = context(off, words, 300, 16)
if when == "order":
    shim.shim_fail_malloc(order, 1)
elif when == "pinned":
    shim.shim_fail_pinned(1)
ctx = context(off, words, 300, 16)
shim.shim_fail_pinned(0)
gone = when == "order" or (when == "pinned" and not one)
assert ref.info().device_bytes - ctx.info().device_bytes == (order if gone else 0)
ctx.sweep(1)
ref.sweep(1)
z, aux = ref.get_topics(), ref.get_aux()
if when == "later":  # the records of get_aux
    shim.shim_fail_malloc(4 * n, 1)
elif when == "server":  # its pool
    shim.shim_fail_malloc(300 * 16 * 4, 1)
    srv = ezlda.Server(ctx, max_slots=4, sweeps=2, hbm_budget_bytes=1 << 20, seed=3)
    srv.submit(1, words[:50])
    srv.wait(1)
    srv.close()
if when == "server":  # its creation renews the top topics that the records are of
    ref.loglik()
    aux = ref.get_aux()
assert np.array_equal(ctx.get_aux(), aux)
if when in ("later", "server"):
    assert ref.info().device_bytes - ctx.info().device_bytes == order
assert np.array_equal(ctx.get_topics(), z)
ctx.sweep(1)
ref.sweep(1)
assert np.array_equal(ctx.get_topics(), ref.get_topics())
assert ctx.loglik() == ref.loglik()
""")


# half wavefronts of words of few tokens on one CU, where a handful of such words is enough for them
@pytest.mark.parametrize("K", [8192, 8193, 10000, 16383])
def test_words_of_few_tokens_on_one_cu(shim, K):
    _run(shim, f"""
shim.shim_cus(1)
from test_gpu_edges import test_words_of_few_tokens_at_large_k as test
for odd in (0, 1):
    for kw in (dict(), dict(shortcut=0), dict(block_dim=64, run_cap=1)):
        test({K}, kw, odd)
""")
