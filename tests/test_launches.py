"""The library's host side without a GPU: what it allocates and launches, on a
HIP runtime whose kernels do nothing (tests/host_checks/fake_hip.c)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

HEAD = """
import ctypes, os, numpy as np
fake = ctypes.CDLL(os.environ["FAKE_HIP"])
fake.fake_hip_log.restype = ctypes.c_char_p
fake.fake_hip_limit.argtypes = [ctypes.c_size_t]
import patchyparticles_amd as pp
def log():
    return [w.split() for w in fake.fake_hip_log().decode().splitlines()]
def launches():
    # (kernel, threads along x)
    return [(w[1], int(w[2]) * int(w[5])) for w in log() if w[0] == "launch"]
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    src = os.path.join(ROOT, "tests", "host_checks", "fake_hip.c")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", src, "-o", so], check=True)
    env = dict(os.environ, FAKE_HIP=so, PYTHONPATH=ROOT, LD_PRELOAD=" ".join(filter(None, [os.environ.get("LD_PRELOAD"), so])))

    def go(script):
        res = subprocess.run([sys.executable, "-c", HEAD + script], env=env, cwd=ROOT, capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stdout + res.stderr
        return res.stdout
    return go


@pytest.mark.parametrize("replicas,ensemble", [(26, "NPT"), (40, "NVT")])
def test_systems_of_many_cells_start(run, replicas, ensemble):
    """Replicas of 138^3 cells (122^3 in NVT), more than 2^26 in all: a launch
    of a thread per word of the cells' records would pass 2^32 threads, which
    HIP refuses."""
    run(f"""
one = [np.full((1, 3), 1.0)] * {replicas}, [np.eye(3)[None]] * {replicas}, [np.full(3, 137.9)] * {replicas}
prm = [dict(T=0.11, P=0.02, ensemble=pp.{ensemble}, rescale_factor_max=0.01)] * {replicas}
with pp.System.batch(*one, prm, trials_per_cell=16) as s:
    if "{ensemble}" == "NVT":
        s.do_ensemble(2)
got = launches()
assert len(got) > 10 and max(n for _, n in got) < 1 << 32
cells = [int(w[1]) for w in log() if w[0] == "malloc"]
assert max(cells) >= 8 * (1 << 23) * 256  # the records
""")


def test_snapshot_clears_no_records(run):
    """A snapshot's context never sweeps: of what creation clears, none is as
    large as the records (64 words a cell; here 32 x 32 x 32 cells)."""
    run("""
rng = np.random.default_rng(1)
r = rng.uniform(0, 36.0, (2000, 3))
pp.energy_snapshot(r, np.broadcast_to(np.eye(3), (2000, 3, 3)), np.full(3, 36.0))
cleared = [n for k, n in launches() if "fill" in k or "clear" in k]
assert cleared and sum(cleared) < 2 * 32 ** 3 + 8192, cleared  # (two tables of a word a cell)
""")


def test_only_loss_grad_pins_its_results(run):
    """Pinning host memory is dear: a network that is evaluated or trained pins
    none, the first loss_grad call its gradients and losses, later ones of no
    more rows nothing."""
    run("""
r, O, box = pp.generate(500, 0.1, 1)
x, t = np.zeros((100, 84), np.float32), np.zeros((100, 6), np.float32)
with pp.System(r, O, box, T=0.1) as s, pp.ProposalNet(seed=1) as net:
    pins = lambda: [int(w[1]) for w in log() if w[0] == "hostmalloc"]
    fake.fake_hip_clear()
    net.forward(x)
    s.train(net, steps=2, batch=1000)
    assert pins() == []
    net.loss_grad(x, t)
    assert pins() == [4 * (49152 + 416 + 1024)]
    net.forward(np.zeros((1024, 84), np.float32))
    net.loss_grad(np.zeros((1024, 84), np.float32), np.zeros((1024, 6), np.float32))
    assert len(pins()) == 1
    net.loss_grad(np.zeros((1025, 84), np.float32), np.zeros((1025, 6), np.float32))
    assert pins()[1:] == [4 * (49152 + 416 + 1056)]
""")


def test_download_without_device_memory(run):
    """A context that leaves no device memory is downloaded all the same, and
    the allocation that failed is no later call's error.  (One particle: its
    index is 0, as the memory that no kernel has written.)"""
    run("""
with pp.System(np.ones((1, 3)), np.eye(3)[None], np.full(3, 9.0), T=0.1) as s:
    fake.fake_hip_limit(0)
    for _ in range(2):
        r, O, box = s.state()
        assert box.tolist() == [9.0] * 3
        s.do_ensemble(1)
    fake.fake_hip_limit(1 << 30)
    fake.fake_hip_clear()
    s.state()
    assert "k_unpack" in fake.fake_hip_log().decode()
""")


def test_a_failed_allocation_is_no_later_call_s_error(run):
    run("""
r, O, box = pp.generate(2000, 0.1, 1)
x = np.zeros((4000, 84), np.float32)
with pp.ProposalNet(seed=1) as net:
    for refused in (lambda: pp.System(r, O, box, T=0.1), lambda: net.forward(np.zeros((40000, 84), np.float32))):
        fake.fake_hip_limit(1 << 16)
        try:
            refused()
            assert False
        except pp.PPError as e:
            assert e.status == 7, e  # PP_ERR_NOMEM
        fake.fake_hip_limit(1 << 30)
        with pp.System(r, O, box, T=0.1) as s:
            s.do_ensemble(1)
        assert net.forward(x).shape == (4000, 26)
""")


@pytest.mark.gpu
def test_systems_of_many_cells_move():
    """The same 40 replicas with a few particles each: replica k moves as in a
    batch of the first two."""
    import patchyparticles_amd as pp
    rng = np.random.default_rng(1)
    r = np.arange(6)[:, None] * 1.15 + rng.uniform(0, 0.05, (6, 3))
    O = np.linalg.qr(rng.normal(size=(6, 3, 3)))[0]
    got = []
    for copies in (2, 40):
        with pp.System.batch([r] * copies, [O] * copies, [np.full(3, 137.9)] * copies, [dict(T=0.11)] * copies, seed=3,
                             trials_per_cell=16) as s:
            assert s.grid()[0] == [122] * 3
            s.do_ensemble(3)
            got.append([s.state(k) + (s.counters(k),) for k in (0, 1)])
            assert s.counters_all()["tries"][-1, 0] > 0
    for a, b in zip(*got):
        assert all(np.array_equal(x, y) for x, y in zip(a[:3], b[:3])) and a[3] == b[3]
