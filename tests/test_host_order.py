"""Order and recovery of libhk.so's host code, on the CPU: the library runs in
a child process over the runtime of ``_fake_hip.cpp`` (no kernel runs there),
which finishes queued work as late as HIP may, fails the calls that a scenario
names, and counts the uses that a wait is missing for."""

import os
import subprocess
import sys
from pathlib import Path

import pytest

TESTS = Path(__file__).resolve().parent

PREAMBLE = """
import ctypes, os, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before libhk.so: its calls go here
import numpy as np
from runtime import hip
from runtime.experts import GgmlExperts, coli_init, coli_matmul
from runtime.qwen_engine import QwenDecoderEngine
from runtime.synthetic import SMOLLM2_135M, SyntheticModel

def engine(w8=False, context=256):
    shape = dict(SMOLLM2_135M, layers=2, hidden_size=128, intermediate_size=256, attention_heads=2, kv_heads=1,
                 vocab_size=512)
    return QwenDecoderEngine(SyntheticModel(shape, seed=0), context_length=context, w8=w8)

def fails(call):
    try:
        call()
    except RuntimeError:
        return
    raise AssertionError("the call was meant to fail")

def settled():
    n = fake.fake_early_sources()
    assert n == 0, f"{n} staged inputs changed or freed before their copy was done"
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    lib = tmp_path_factory.mktemp("fake") / "libfakehip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(TESTS / "_fake_hip.cpp"), "-o", str(lib)], check=True)

    def run(script, **env):
        path = os.pathsep.join([str(TESTS.parent), str(TESTS.parent / "hawkpoint-npu-llm_amd")])
        done = subprocess.run([sys.executable, "-c", PREAMBLE + script, str(lib)], capture_output=True, text=True,
                              env={**os.environ, "PYTHONPATH": path, "HK_EAGER": "1", **env}, timeout=120)
        assert done.returncode == 0, done.stdout + done.stderr

    return run


@pytest.mark.parametrize("launch", [0, 3, 9])
def test_engine_call_after_one_that_failed(child, launch):
    """A call that fails after its inputs were queued leaves their copy in
    flight; the next call's inputs wait for it."""
    child(f"""
e = engine()
e.prefill(np.arange(70))
fake.fake_fail_launch({launch})
fails(lambda: e.prefill(np.arange(70) + 7))
e.prefill(np.arange(70) + 200)
settled()
if {launch} < 9:
    fake.fake_fail_launch({launch})
    fails(lambda: e.step(np.full(128, 0x3f80, np.uint16), 70))
e.step(np.full(128, 0x4000, np.uint16), 70)
settled()
""")


def test_prompt_of_two_chunks(child):
    """The second chunk's token ids wait for the first one's copy."""
    child("""
e = engine(context=5120)
e.prefill(np.arange(5000) % 512)
settled()
""")


def test_expert_call_after_one_that_failed(child):
    """The same for the expert calls, whose staging may also be replaced by a
    larger one meanwhile."""
    child("""
rng = np.random.default_rng(0)
hip.init(0)
s = GgmlExperts(rng.normal(size=(8, 64, 256)).astype(np.float32))
x = rng.normal(size=(2, 256)).astype(np.float32)
fake.fake_fail_launch(0)
fails(lambda: s.mul_mat_id(x, [0, 1]))
s.mul_mat_id(-x, [0, 1])
settled()
coli_init()
matmul = lambda n: coli_matmul(rng.normal(size=(n, n)).astype(np.float32), None, 0, rng.normal(size=n), n, n)
for n in (64, 64, 256):
    fake.fake_fail_launch(0)
    fails(lambda: matmul(n))
matmul(256)
settled()
""")


def test_expert_call_after_a_failed_reservation(child):
    """A set whose scratch could not be had at its creation reserves it again
    with a call, which then succeeds: the old failure is not reported again."""
    child("""
rng = np.random.default_rng(0)
hip.init(0)
w = rng.normal(size=(8, 64, 256)).astype(np.float32)
x = rng.normal(size=(2, 256)).astype(np.float32)
fake.fake_fail_malloc_after(2)  # (int8 rows and their scales first)
s = GgmlExperts(w)
s.mul_mat_id(x, [0, 1])
fake.fake_fail_malloc_after(0)
fails(lambda: GgmlExperts(w))
s.mul_mat_id(x, [0, 1])
""")


def test_first_prefill_waits_for_its_cleared_workspace(child):
    """The workspace's tickets and tags are cleared on the null stream, which
    the engine's stream does not wait for by itself."""
    child("""
e = engine()
assert fake.fake_early_launches() == 0
e.prefill(np.arange(70))
assert fake.fake_early_launches() == 0, "kernels launched before the workspace was cleared"
stream = ctypes.c_void_p()
hip.check(hip.lib().hk_stream_create(ctypes.byref(stream)), "stream")
b = [hip.DeviceBuffer(1 << 16) for _ in range(7)]
hip.check(hip.lib().hk_attention_decode(*[x.ptr for x in b[:5]], 300, 512, 4, 2, 64, b[5].ptr, stream.value), "attention")
assert fake.fake_early_launches() == 0, "attention launched before its tickets were cleared"
""")


@pytest.mark.parametrize("ring", ["1", "0"])
def test_bf16_copies_only_where_the_ring_reads_them(child, ring):
    """A W8 prompt of more than 64 tokens makes bf16 copies of the projections
    for the ring GEMM; without the ring (HK_GEMM_RING=0) nothing reads them."""
    child(f"""
e = engine(w8=True)
e.prefill(np.arange(40))
before = fake.fake_device_bytes()
e.prefill(np.arange(70), 40)
per_layer = (2 + 2 * 1) * 64 * 128 + 128 * 128 + 3 * 256 * 128
assert fake.fake_device_bytes() - before == ({ring} and 2 * 2 * per_layer), fake.fake_device_bytes() - before
""", HK_GEMM_RING=ring)
