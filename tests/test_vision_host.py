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


BROKEN = {   # the block's kernels without the tensor's facts
    "attn_qkv.weight": ["ln/f", "mm/f", "heads/f", "attend/f", "mm/f"] + SPLIT[5:],
    "attn_qkv.bias": SPLIT[:2] + ["heads/f", "attend/f", "mm/f"] + SPLIT[5:],
    "ln1.weight": ["ln/f", "mm/f", "heads/f", "attend/f", "mm/f"] + SPLIT[5:],
    "attn_out.weight": SPLIT[:4] + ["mm/f"] + SPLIT[5:],
    "ffn_up.bias": SPLIT[:5] + ["ln/f", "mm/f", "mm/f"],
    "ffn_down.weight": SPLIT[:5] + ["ln/f", "mm/f", "mm/f"],
    "ffn_down.bias": SPLIT,
}


@pytest.mark.parametrize("tensor,fail", [(t, 1) for t in BROKEN] + [(t, f) for t in BROKEN if t.count("_") and "weight" in t
                                         for f in (2, 3)])
def test_a_tensor_whose_measuring_failed_runs_in_fp32(tower, tensor, fail):
    """A replaced tensor whose measuring fails has no fp16 rows and no bounds of its own: its product
    and those that its bounds reach run in fp32, the other blocks as before.  Measured again, all is
    as it was."""
    name = "v.blk.3." + tensor
    assert tower.set(name, fail=fail) != OK
    tower.L.vh_facts(1.0, 1.0, 0, 0)
    blocks, mergers = tower.encode()
    # past step 1 the new values' bounds are known, so the attention on them may stay split
    assert blocks[3] == (["ln/f", "mm/f"] + SPLIT[2:] if fail > 1 and tensor == "attn_qkv.weight" else BROKEN[tensor])
    assert blocks[:3] + blocks[4:] == [SPLIT] * 26 and mergers == [["ln/s", "mm/s", "mm/s"]] * 4
    assert tower.set(name) == OK
    assert tower.encode()[0] == [SPLIT] * 27


def test_values_that_fp16_does_not_hold_run_in_fp32(tower):
    assert tower.set("v.blk.5.ffn_up.weight", inexact=1) == OK
    assert tower.set("mm.2.weight", inexact=1) == OK
    blocks, mergers = tower.encode()
    assert blocks[5] == SPLIT[:5] + ["ln/f", "mm/f", "mm/f"] and blocks[:5] + blocks[6:] == [SPLIT] * 26
    assert mergers == [["ln/s", "mm/s", "mm/s"]] * 3 + [["ln/f", "mm/f", "mm/f"]]


def test_bounds_that_are_not_finite_run_in_fp32(tower):
    assert tower.set("v.blk.0.ln1.bias", mx=float("nan"), norm=float("nan")) == OK
    assert tower.encode()[0][0] == BROKEN["ln1.weight"]


def test_values_too_small_for_a_scale_run_in_fp32(tower):
    """A q | k | v matrix of values near 2^-75 (no bias): no scale of at most 2^60 brings its rows to
    where two fp16 parts hold them, and their norms are no zeros in fp32's own squares."""
    assert tower.set("v.blk.2.attn_qkv.bias", mx=0.0, norm=0.0) == OK
    assert tower.set("v.blk.2.attn_qkv.weight", mx=2.0 ** -75, norm=2.0 ** -71) == OK
    assert tower.encode()[0][2] == SPLIT[:2] + ["heads/f", "attend/f", "mm/f"] + SPLIT[5:]
