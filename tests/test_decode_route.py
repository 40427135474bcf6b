"""The rule that picks a decode call's form (csrc/decode_route.h), built for the CPU.

The points are shapes measured on both sides of each line: a form other than the plain one (all of the plan's
heads per wave, four waves; one head and eight waves up to one (sequence, head) pair per CU) has to be no
slower for equal lengths and for lengths spread over a factor of eight.
"""

import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-practice_amd", "csrc")


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "route.cpp").write_text(
        '#include "decode_route.h"\n'
        'extern "C" int route(int b, int h, int kvh, int plan, int kv, int f32, int cus) {\n'
        "    const femto::DecodeRoute r = femto::decode_route(b, h, kvh, plan, kv, f32, cus);\n"
        "    return r.nrep_tile * 100 + r.waves * 10 + r.split;\n}\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(d / "route.cpp"),
                    "-o", str(d / "route.so")], check=True)
    lib = ctypes.CDLL(str(d / "route.so"))

    def call(seqs, heads, kv_heads, keys, dtype="bf16", cus=256):
        v = lib.route(seqs, heads, kv_heads, plan(heads // kv_heads, dtype), keys, dtype == "f32", cus)
        return v // 100, v // 10 % 10, bool(v % 10)

    return call


def plan(n_rep, dtype):
    """Query heads per wave of plan_paged_decode."""
    return next(r for r in ((4, 2, 1) if dtype == "f32" else (8, 4, 2, 1)) if n_rep % r == 0)


POINTS = [
    # 16-bit, at most one workgroup per CU
    ((8, 32, 8, 100), (1, 8, False)), ((16, 32, 8, 1024), (2, 8, False)), ((8, 64, 8, 1024), (2, 8, False)),
    ((16, 64, 8, 512), (4, 4, False)), ((16, 64, 8, 1024), (4, 8, False)), ((32, 32, 8, 768), (4, 4, False)),
    ((18, 16, 8, 1024), (2, 8, False)), ((32, 16, 8, 384), (2, 4, False)), ((256, 2, 1, 1024), (2, 4, False)),
    ((21, 24, 2, 1024), (4, 8, False)), ((21, 24, 2, 512), (4, 4, False)),
    # more workgroups
    ((64, 16, 8, 512), (2, 4, False)), ((64, 32, 8, 512), (4, 4, False)), ((64, 16, 16, 512), (1, 4, False)),
    # eight heads per KV head
    ((17, 64, 8, 512), (8, 4, False)), ((64, 64, 8, 128), (4, 4, False)), ((64, 64, 8, 512), (4, 4, False)),
    ((512, 8, 1, 512), (8, 4, False)), ((187, 16, 2, 512), (8, 4, False)), ((100, 64, 8, 128), (4, 4, False)),
    ((100, 64, 8, 1024), (8, 4, True)), ((200, 64, 8, 32), (8, 4, True)), ((1000, 8, 1, 257), (8, 4, False)),
    # f32
    ((8, 16, 8, 900, "f32"), (1, 8, True)), ((8, 16, 8, 896, "f32"), (1, 8, False)),
    ((8, 16, 16, 900, "f32"), (1, 8, False)), ((8, 8, 1, 900, "f32"), (1, 8, False)),
    ((4, 32, 8, 900, "f32"), (1, 8, True)), ((16, 4, 1, 900, "f32"), (1, 8, False)),
    ((2048, 1, 1, 128, "f32"), (1, 4, False)), ((128, 16, 16, 128, "f32"), (1, 4, False)),
    ((2048, 2, 1, 128, "f32"), (2, 4, False)), ((100, 64, 8, 128, "f32"), (4, 4, True)),
    ((200, 32, 8, 1024, "f32"), (4, 4, True)), ((96, 64, 8, 128, "f32"), (4, 4, False)),
]


@pytest.mark.parametrize("shape,form", POINTS, ids=str)
def test_measured_points(route, shape, form):
    assert route(*shape) == form


def test_forms_exist_for_every_shape(route):
    """Heads per wave divide the plan's, eight waves come with at most four heads (f32: one), and the plain
    form is kept for plain shapes."""
    rng = np.random.default_rng(1)
    for _ in range(20000):
        kv_heads = int(rng.choice([1, 2, 3, 4, 8, 16]))
        n_rep = int(rng.choice([1, 2, 3, 4, 5, 6, 7, 8, 12, 16, 24]))
        dtype = str(rng.choice(["f32", "bf16"]))
        seqs, keys = int(2.0 ** rng.uniform(0, 17)), int(rng.integers(0, 1500))
        cus = int(rng.choice([1, 32, 64, 128, 256, 304]))
        r, waves, split = route(seqs, n_rep * kv_heads, kv_heads, keys, dtype, cus)
        assert plan(n_rep, dtype) % r == 0 and waves in (4, 8)
        assert waves == 4 or r <= (1 if dtype == "f32" else 4)
        assert not split or kv_heads >= 4 or (dtype == "f32" and seqs * n_rep * kv_heads <= cus / 2)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_lines_follow_the_compute_units(route, dtype):
    """Half the sequences on half the CUs take the same form (from nine sequences up: f32 has a line at four)."""
    rng = np.random.default_rng(2)
    for _ in range(5000):
        heads, kv_heads = [(16, 8), (32, 8), (64, 8), (16, 16), (8, 1), (24, 2)][int(rng.integers(6))]
        seqs, keys = 2 * int(2.0 ** rng.uniform(3.4, 11)), int(rng.integers(1, 1025))
        assert route(seqs, heads, kv_heads, keys, dtype, 256) == route(seqs // 2, heads, kv_heads, keys, dtype, 128)
