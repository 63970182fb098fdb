"""The GPU library's host code on the CPU, above all its failure paths:
allocations that fail in the middle of a call.  Each case runs in a process of its own in which
tests/fake_hip/fake_hip.c stands in for the HIP runtime (nothing is launched,
a download fills its destination with a byte)."""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_live.restype = ctypes.c_size_t
fake.fake_fail_next.argtypes = [ctypes.c_int, ctypes.c_size_t]
DEVICE, PINNED = 0, 1
sys.path.insert(0, sys.argv[2])
import numpy as np
import se2dr_fork_amd as S
from se2dr_fork_amd import scenarios as SC
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("gcc is not installed")
    if not os.path.exists(os.path.join(ROOT, "se2dr_fork_amd", "lib", "libse2w_hip.so")):
        pytest.skip("libse2w_hip.so is not built")
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-o", so,
                    os.path.join(ROOT, "tests", "fake_hip", "fake_hip.c")], check=True)

    def run(body):
        env = dict(os.environ, SE2W_AUTOTUNE="0", OMP_NUM_THREADS="2")
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, so, ROOT], capture_output=True, text=True, timeout=120,
                           env=env)
        assert r.returncode == 0 and "case ok" in r.stdout, r.stdout[-2000:] + r.stderr[-4000:]

    return run


def test_ensemble_rows_after_a_record_buffer_that_could_not_grow(fake):
    """The second member's pinned record buffer cannot grow: the run fails,
    and the first member's rows are then downloaded, not read from a buffer
    that no copy of this run has filled."""
    fake("""
builts = [SC.build(SC.small(mx=6, my=5, p=3, nt=20, seed=i, nrec=n)) for i, n in ((1, 2), (2, 5))]
ens = S.Ensemble([b.solver for b in builts])
dts = [b.dt for b in builts]
ens.advance(4, dts)
fake.fake_fail_next(PINNED, 6 * 5 * (6 + 2 * 4) * 8)
try:
    ens.advance(6, dts)
    raise SystemExit("the run did not fail")
except S.Se2wError as e:
    assert "hipHostMalloc" in str(e), e
fake.fake_fill(0x3f)
n = fake.fake_downloads()
rows = builts[0].solver.ctx.receivers()
assert fake.fake_downloads() == n + 1
assert rows.shape == (6, 2, 7) and (rows[..., :6] == np.frombuffer(b"\\x3f" * 8)[0]).all()
rows = builts[1].solver.ctx.receivers()
assert fake.fake_downloads() == n + 2
print("case ok")
""")


def test_gradient_buffers_after_a_training_that_could_not_grow_them(fake):
    """The buffer of the batches' squared errors cannot grow for an epoch: the
    training fails, and the buffer of one batch, which the loss of a gradient
    is written to, is still there."""
    fake("""
net = S.Mlp([66, 64, 192], batch=64, seed=1)
x, t = np.zeros((4 * 64, 66), np.float32), np.zeros((4 * 64, 192), np.float32)
net.set_data(x, t)
parts = (64 // 16) * (192 // 16)  # workgroups of the last product
before = fake.fake_live(DEVICE)
fake.fake_fail_next(DEVICE, 8 * 4 * parts)
try:
    net.train(1)
    raise SystemExit("the training did not fail")
except S.Se2wError as e:
    assert "hipMalloc" in str(e), e
assert fake.fake_live(DEVICE) == before
net.gradient(x[:64], t[:64])
net.train(1)
net.close()
assert fake.fake_live(DEVICE) == 0 and fake.fake_live(PINNED) == 0
print("case ok")
""")


def test_training_data_needs_no_second_copy_in_host_memory(fake):
    """Rows of one input are padded to 64 on the device; on the way there the
    host holds a few megabytes of padded rows, not all of them (512 MB)."""
    fake("""
import resource
net = S.Mlp([1, 64, 64], batch=64, seed=1)
n = 1 << 21
x, t = np.ones((n, 1), np.float32), np.zeros((n, 64), np.float32)  # t's pages are never touched
before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
net.set_data(x, t)
grown = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before
assert grown < 100 << 10, grown  # KB
net.close()
print("case ok")
""")


def test_a_network_pins_a_bounded_amount_of_host_memory(fake):
    """Five pieces of input rows and four chunks of output rows, about 1 MB
    each, whatever the width and the batch (5 x 134 MB of inputs here), and
    more only for rows that are longer than that."""
    fake("""
net = S.Mlp([8192, 64, 64], batch=4096, seed=1)
assert fake.fake_live(PINNED) <= 9 << 20, fake.fake_live(PINNED)
net.forward(np.zeros((3 * 4096 + 5, 8192), np.float32))
assert fake.fake_live(PINNED) <= 9 << 20, fake.fake_live(PINNED)
net.close()
net = S.Mlp([1 << 19, 64], batch=64, seed=1)
assert fake.fake_live(PINNED) <= (5 * 2 << 20) + (4 << 20), fake.fake_live(PINNED)
net.close()
assert fake.fake_live(PINNED) == 0
print("case ok")
""")


def test_tuning_with_one_candidate_runs_no_trial(fake):
    """In FP64 from p = 5 up only the column kernel is left to a tuner: it is
    set without trials unless the caller asks for its time."""
    fake("""
builts = [SC.build(SC.small(mx=mx, my=my, p=p, nt=20)) for mx, my, p in ((7, 6, 6), (7, 6, 4), (20, 17, 6))]
ctx, ctx4, ctx6 = [b.solver.ctx for b in builts]
ctx.set_kernel(S.KERNEL_LDS)
best, n = ctypes.c_int32(), fake.fake_launches()
assert ctx._hip.se2w_autotune(ctx._handle, 20, 3, ctypes.byref(best), None) == 0
assert best.value == ctx.kernel() == S.KERNEL_COL
assert fake.fake_launches() == n
assert ctx4._hip.se2w_autotune(ctx4._handle, 20, 3, ctypes.byref(best), None) == 0
assert fake.fake_launches() > n
n = fake.fake_launches()
assert ctx6.autotune()[1] > 0 and fake.fake_launches() > n
print("case ok")
""")


def test_tuning_does_not_charge_the_first_candidate_with_a_cold_gpu(fake):
    """Kernels of equal time, of which the first is tried while the GPU is
    still at half its clocks: the first one stays the choice."""
    fake("""
b = SC.build(SC.small(mx=7, my=6, p=4, nt=20))
ctx, best = b.solver.ctx, ctypes.c_int32()
fake.fake_slow(12)  # two times are taken of each trial run
assert ctx._hip.se2w_autotune(ctx._handle, 20, 3, ctypes.byref(best), None) == 0
assert best.value == S.KERNEL_REG64, best.value
print("case ok")
""")
