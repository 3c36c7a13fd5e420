"""The vision tower's host side without a GPU: which products run on fp16 parts and which in fp32,
by what each tensor's measuring found and whether it came to its end.  tests/host/vision_host.cpp
stands in for the device and the kernels (linked with this build's own api_vision.o)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import exn_vision_oracle as vo

HERE = os.path.dirname(os.path.abspath(__file__))
OBJ = os.path.join(HERE, "..", "ex-nihilo_amd", "_build", "api_vision.o")
OK, F32 = 0, 0
DATA = np.zeros(4608 * 4608, np.float32)


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if not os.path.exists(OBJ):
        pytest.skip("the library's objects are not here")
    d = tmp_path_factory.mktemp("vision_host")
    o, so = str(d / "vision_host.o"), str(d / "vision_host.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-c",
                    os.path.join(HERE, "host", "vision_host.cpp"), "-o", o], check=True)
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", so, o, OBJ], check=True)
    L = ctypes.CDLL(so)
    L.vh_encode.restype = ctypes.c_char_p
    L.vh_ctx.restype = ctypes.c_void_p
    L.vh_spread.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_double]
    L.vh_spread(0, 0, 1.0, 1.0)
    L.vh_facts.argtypes = [ctypes.c_float, ctypes.c_double, ctypes.c_int, ctypes.c_int]
    return L


class Tower:
    def __init__(self, L):
        self.L, self.h = L, ctypes.c_void_p()
        self.shapes = dict(vo.vision_expected(vo.VShape()))
        assert L.exn_vision_create(ctypes.c_void_p(L.vh_ctx()), ctypes.byref(self.h)) == OK

    def set(self, name, mx=1.0, norm=1.0, inexact=0, fail=0):
        """Store tensor NAME; its measuring finds MX, NORM and INEXACT, or fails: 1 its
        statistics, 2 a matrix's fp16 rows, 3 their flag's way back."""
        self.L.vh_facts(mx, norm * norm, inexact, fail)
        shape = self.shapes[name]
        return self.L.exn_vision_set(self.h, name.encode(), F32, DATA.ctypes.data_as(ctypes.c_void_p),
                                     (ctypes.c_int64 * len(shape))(*shape), len(shape))

    def encode(self):
        """The kernels of each block (its LayerNorms, products and attention) and of each merger; a
        merger after block i runs behind block i + 1's first LayerNorm, which finishes block i's rows."""
        log = self.L.vh_encode(self.h).decode().split()
        assert log[0] == "mm/f", log      # the patch embedding
        blocks, mergers = [], []
        for i, a in enumerate(k for k, what in enumerate(log) if what.startswith("heads")):
            after = i - 1 in (8, 16, 24)
            blocks.append([log[a - (5 if after else 2)]] + log[a - 1:a + 6])
            if after:
                mergers.append(log[a - 4:a - 1])
        mergers.append(log[-3:])
        assert len(log) == 1 + 27 * 8 + 4 * 3
        return blocks, mergers


SPLIT = ["ln/s", "mm/s", "heads/s", "attend/s", "mm/s", "ln/s", "mm/s", "mm/s"]


@pytest.fixture
def tower(host):
    t = Tower(host)
    for name in t.shapes:
        assert t.set(name) == OK
    yield t
    host.exn_vision_destroy(t.h)


def test_every_product_runs_split(tower):
    blocks, mergers = tower.encode()
    assert blocks == [SPLIT] * 27 and mergers == [["ln/s", "mm/s", "mm/s"]] * 4


FP32 = ["ln/f", "mm/f", "heads/f", "attend/f", "mm/f", "ln/f", "mm/f", "mm/f"]
FP32_QKV = FP32[:5] + SPLIT[5:]
FP32_OUT = SPLIT[:4] + ["mm/f"] + SPLIT[5:]
FP32_MLP = SPLIT[:5] + FP32[5:]


@pytest.mark.parametrize("tensor,steps", [("attn_qkv.weight", 4), ("attn_out.weight", 4), ("ffn_down.weight", 4),
                                          ("attn_qkv.bias", 1), ("ln1.weight", 1), ("ffn_down.bias", 1)])
def test_a_tensor_whose_measuring_failed_runs_in_fp32(tower, tensor, steps):
    """A replaced tensor whose measuring fails, at whichever step, has no fp16 rows and bounds
    nothing: its block runs in fp32, the others as before.  Measured again, all is as it was."""
    name = "v.blk.3." + tensor
    for fail in range(1, steps + 1):
        assert tower.set(name, fail=fail) != OK
        tower.L.vh_facts(1.0, 1.0, 0, 0)
        blocks, mergers = tower.encode()
        assert blocks[3] == FP32, fail
        assert blocks[:3] + blocks[4:] == [SPLIT] * 26 and mergers == [["ln/s", "mm/s", "mm/s"]] * 4
        assert tower.set(name) == OK
        assert tower.encode()[0] == [SPLIT] * 27


def test_values_that_fp16_does_not_hold_run_in_fp32(tower):
    assert tower.set("v.blk.5.ffn_up.weight", inexact=1) == OK
    assert tower.set("mm.2.weight", inexact=1) == OK
    blocks, mergers = tower.encode()
    assert blocks[5] == FP32_MLP and blocks[:5] + blocks[6:] == [SPLIT] * 26
    assert mergers == [["ln/s", "mm/s", "mm/s"]] * 3 + [["ln/f", "mm/f", "mm/f"]]


def test_bounds_that_are_not_finite_run_in_fp32(tower):
    assert tower.set("v.blk.0.ln1.bias", mx=float("nan"), norm=float("nan")) == OK
    assert tower.encode()[0][0] == FP32_QKV


def test_values_too_small_for_a_scale_run_in_fp32(tower):
    """A q | k | v matrix of values near 2^-75 (no bias): no scale of at most 2^60 brings its rows to
    where two fp16 parts hold them, and their norms are no zeros in fp32's own squares."""
    assert tower.set("v.blk.2.attn_qkv.bias", mx=0.0, norm=0.0) == OK
    assert tower.set("v.blk.2.attn_qkv.weight", mx=2.0 ** -75, norm=2.0 ** -71) == OK
    assert tower.encode()[0][2] == SPLIT[:2] + FP32_QKV[2:]


@pytest.mark.parametrize("rows,cols,bound,want", [
    (3456, 1152, 1152 ** 0.5 + 1, FP32[:2] + SPLIT[2:]),
    (4304, 1152, 1152 ** 0.5 + 1, FP32_MLP),
    (1152, 4304, 1.001 * 1.001 * 1152 ** 0.5 + 2.003, FP32_MLP),
    (1152, 1152, 64 * (1.001 * 1.001 * 1152 ** 0.5 + 2.003), FP32_OUT),
])
def test_bounds_far_above_the_inputs_run_in_fp32(tower, rows, cols, bound, want):
    """A product whose scale's bound is over 2^17 times its outputs' own size per unit of weight (2^11
    for attn_out, whose inputs attention averages) runs in fp32, one 10% below runs split; every
    tensor's largest value and row norm are 1, which makes BOUND."""
    for spread, kernels in ((2 ** 17 / bound * 0.9, SPLIT), (2 ** 17 / bound * 1.1, want)):
        tower.L.vh_spread(rows, cols, spread, 1.0)
        assert tower.set("v.blk.6.ln1.bias") == OK
        tower.L.vh_spread(0, 0, 1.0, 1.0)
        blocks, _ = tower.encode()
        assert blocks[6] == kernels and blocks[:6] + blocks[7:] == [SPLIT] * 26
    assert tower.set("v.blk.6.ln1.bias") == OK
    assert tower.encode()[0][6] == SPLIT


def test_scores_and_mergers_far_below_their_bounds_run_in_fp32(tower):
    """q and k 2^30 times smaller than their bound: their scores stay under 1 and the split's error
    with them (they run split); 2^20 times larger than ordinary ones with the same bound: no finite
    scores (a mean square of NaN): fp32.  A merger whose second product's inputs are far below."""
    tower.L.vh_spread(0, 0, 1.0, 2.0 ** -60)
    assert tower.set("v.blk.0.ln2.bias") == OK and tower.encode()[0][0] == SPLIT
    tower.L.vh_spread(0, 0, 1.0, float("nan"))
    assert tower.set("v.blk.0.ln2.bias") == OK and tower.encode()[0][0] == SPLIT[:2] + FP32_QKV[2:]
    tower.L.vh_spread(4096, 4608, 2.0 ** 14, 1.0)
    assert tower.set("v.deepstack.16.fc1.bias") == OK
    tower.L.vh_spread(0, 0, 1.0, 1.0)
    assert tower.encode()[1] == [["ln/s", "mm/s", "mm/s"], ["ln/f", "mm/f", "mm/f"]] + [["ln/s", "mm/s", "mm/s"]] * 2
