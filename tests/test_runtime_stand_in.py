"""The library's host code on the CPU, over a stand-in for the HIP runtime
(fake_hip.cpp): each test is a program of its own in which the stand-in's functions,
loaded first, take the place of the runtime's. Kernels do not run.
"""

import shutil
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
PKG = HERE.parent / "differentiable-rasterizer_amd"

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_pinned_bytes.restype = ctypes.c_size_t
fake.fake_malloc_fails.argtypes = [ctypes.c_size_t]
fake.fake_launches.restype = ctypes.c_char_p
sys.modules["torch"] = None  # its runtime is not wanted here
sys.path.insert(0, {pkg!r})
import numpy as np
from diffrast import _lib

MIB = 1 << 20

def launched(f):
    fake.fake_launches()
    f()
    return fake.fake_launches().decode().split()

def addr(a):  # device memory is host memory here
    return a.ctypes.data

def code(f):
    try:
        f()
    except _lib.DiffrastError as e:
        return e.code
    return 0

ctx = _lib.Context()
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    so = tmp_path_factory.mktemp("fake") / "libfake_hip.so"
    # the headers want the platform named where hipcc does not compile them
    subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(HERE / "fake_hip.cpp"), "-o", str(so)], check=True)

    def run(text):
        body = PRELUDE.format(fake=str(so), pkg=str(PKG)) + textwrap.dedent(text)
        res = subprocess.run([sys.executable, "-c", body], capture_output=True, text=True, timeout=100)
        assert res.returncode == 0, res.stderr

    return run


def test_timed_out_calls_return(program):
    """A wait that times out ends the call with the time-out; nothing waits without a limit."""
    program("""
        v = np.linspace(0, 1, 1000, dtype=np.float32)
        target, init = np.zeros((24, 24, 3), np.float32), np.full((5, 10), .5, np.float32)
        fit = _lib.Fitter(ctx, target, init, np.zeros(3, np.float32), iters=4)
        fake.fake_stuck(1)
        assert code(lambda: ctx.encode_srgb(v)) == 2
        assert code(lambda: ctx.render(init[None], 24, 24, .01)) == 2
        assert code(lambda: ctx.fused_loss_backward(init[None], target[None], .01, want_images=True)) == 2
        assert code(lambda: _lib.Fitter(ctx, target, init, np.zeros(3, np.float32), iters=4)) == 2
        assert code(fit.step) == 2
        assert code(lambda: ctx.resize_lanczos3(np.zeros((30, 30, 3), np.uint8), 7, 8)) == 2
        assert fake.fake_unbounded_waits() == 0
        parked = fake.fake_pinned_bytes()
        fake.fake_stuck(0)
        # the parked buffers are used again
        ctx.encode_srgb(v)
        assert fake.fake_pinned_bytes() == parked
        fit.close()
        ctx.clear_pool()
        assert fake.fake_pinned_bytes() == 0
    """)


def test_parked_buffers_are_bounded(program):
    program("""
        fake.fake_stuck(1)
        v = np.zeros(3 * MIB, np.float32)  # 15 MiB both ways: a buffer of 16
        for _ in range(4):
            assert code(lambda: ctx.encode_srgb(v)) == 2
        assert fake.fake_unbounded_waits() == 0 and fake.fake_pinned_bytes() == 64 * MIB
        code(lambda: ctx.encode_srgb(v))  # no buffer is left: copied as it is
        assert fake.fake_pinned_bytes() == 64 * MIB
        fake.fake_stuck(0)
        ctx.encode_srgb(v)
        ctx.clear_pool()
        assert fake.fake_pinned_bytes() == 0
    """)


@pytest.mark.parametrize("stuck", [0, 1])
@pytest.mark.parametrize("copy", [0, 1, 2, 4])
def test_call_that_fails_half_way(program, copy, stuck):
    """The failed copy's error is the call's, also where the wait for the others times out."""
    program(f"""
        init, target = np.full((1, 5, 10), .5, np.float32), np.zeros((1, 24, 24, 3), np.float32)
        call = lambda: ctx.fused_loss_backward(init, target, .01)  # three copies in, two out
        fake.fake_copy_fails({copy})
        fake.fake_stuck({stuck})
        rc = code(call)
        assert rc == ({copy} < 3 and 3 or 4), (rc, _lib.last_error())
        assert "stand-in error" in _lib.last_error()
        assert fake.fake_unbounded_waits() == 0
        fake.fake_stuck(0)
        assert code(call) == 0
        assert fake.fake_pinned_bytes() == MIB
    """)


@pytest.mark.parametrize("n", [10, 12800, 1 << 20, 5 << 20])
def test_arrays_go_through_the_buffer_or_past_it(program, n):
    """Adam's arrays in and out unchanged (its kernel does not run): all of them staged, the
    first four of eight, none."""
    program(f"""
        fake.fake_polls(5)
        n = {n} // 10 * 10
        p, g, m, v, lr = (np.random.default_rng(i).random((n // 10, 10), dtype=np.float32) for i in range(5))
        want = p.copy(), m.copy(), v.copy()
        for _ in range(2):
            out = ctx.adam_project_step(p, g, m, v, lr, step=1)
            for a, b in zip((p, m, v), want):
                assert np.array_equal(a, b)
        assert fake.fake_pinned_bytes() <= 16 * MIB
    """)


def test_free_buffers_are_bounded_and_given_back(program):
    program("""
        import threading
        fake.fake_polls(3)
        for n in (1, MIB // 4, MIB // 2, MIB, 3 * MIB, 20 * MIB):
            ctx.encode_srgb(np.zeros(n, np.float32))
        assert fake.fake_pinned_bytes() == 31 * MIB  # a buffer each of 1, 2, 4, 8 and 16
        ctx.clear_pool()
        assert fake.fake_pinned_bytes() == 0
        ctx.encode_srgb(np.zeros(5, np.float32))
        ctx.close()
        assert fake.fake_pinned_bytes() == 0
    """)


@pytest.mark.parametrize("B,H,W,T", [(1, 520, 500, 300), (2, 1000, 1000, 128), (8, 256, 256, 200)])
def test_call_without_room_for_row_lists(program, B, H, W, T):
    """The tile rows' lists only save time: a call that finds no memory for them scans every
    triangle."""
    program(f"""
        B, H, W, T = {B}, {H}, {W}, {T}
        params, bg = np.full((B, T, 10), .5, np.float32), np.zeros((B, 3), np.float32)
        img, losses, grads = np.zeros((B, H, W, 3), np.float32), np.zeros(B, np.float32), np.zeros((B, T, 10), np.float32)
        render = lambda: ctx.render_ptr(addr(params), addr(bg), B, T, H, W, .002, addr(img))
        fused = lambda: ctx.fused_ptr(addr(params), addr(bg), addr(img), B, T, H, W, .002, addr(losses), addr(grads))
        rows = 2 * B * ((H + 15) // 16)
        for call in (render, fused):
            listed = launched(call)
            ctx.clear_pool()
            fake.fake_malloc_fails(rows * T * 8 + rows * 4)
            scanned = launched(call)
            fake.fake_malloc_fails(0)
            assert len(scanned) == len(listed) and scanned != listed, (scanned, listed)
            assert launched(call) == listed
            ctx.clear_pool()
    """)


# waves a tile of fused_seg_kernel (0: another kernel) for one call of drh_fused_loss_backward and of
# drh_fused_loss_backward_noalloc; tiles are 8x8, four to a 16x16 block
@pytest.mark.parametrize("B,H,W,T,pooled,noalloc", [
    (1, 64, 64, 15, 0, 0), (1, 64, 64, 16, 8, 8), (1, 64, 64, 1024, 8, 8), (1, 64, 64, 1025, 0, 0),
    (3, 128, 128, 16, 8, 8), (4, 128, 96, 16, 8, 8), (4, 128, 112, 16, 4, 4), (1, 224, 240, 150, 4, 4),
    (8, 128, 128, 16, 4, 4), (1, 256, 512, 300, 4, 4), (1, 272, 496, 300, 0, 0),
    # a batch past 2048 tiles, from 48 triangles
    (9, 128, 128, 16, 0, 0), (9, 128, 128, 47, 0, 0), (9, 128, 128, 48, 4, 4), (10, 128, 128, 300, 4, 4),
    (11, 128, 128, 47, 0, 0), (11, 128, 128, 48, 2, 2), (12, 128, 128, 512, 2, 2), (12, 128, 128, 513, 4, 4),
    (13, 128, 128, 200, 2, 0), (16, 128, 128, 32, 0, 0), (16, 128, 128, 128, 2, 0), (16, 128, 128, 1024, 4, 0),
    (5, 256, 256, 512, 2, 0), (6, 256, 256, 128, 0, 0), (23, 128, 128, 128, 2, 0), (24, 128, 128, 128, 0, 0),
])
def test_waves_per_tile(program, B, H, W, T, pooled, noalloc):
    """Which kernel a gradient call takes, also without atomics (no batch past 2048 tiles) and in
    the IEEE mode."""
    program(f"""
        import re
        B, H, W, T = {B}, {H}, {W}, {T}
        params, bg = np.full((B, T, 10), .5, np.float32), np.zeros((B, 3), np.float32)
        img, losses, grads = np.zeros((B, H, W, 3), np.float32), np.zeros(B, np.float32), np.zeros((B, T, 10), np.float32)
        def waves(call, flags):
            names = launched(lambda: call(addr(params), addr(bg), addr(img), B, T, H, W, .002, addr(losses),
                                          addr(grads), flags=flags))
            found = [re.search(r"fused_seg_kernelILi\\d+ELb\\dELb\\dELi(\\d)E", n) for n in names]
            return sum(int(m.group(1)) for m in found if m)
        tiles = 4 * B * ((H + 15) // 16) * ((W + 15) // 16)
        for flags in (0, _lib.EXACT_MATH, _lib.DETERMINISTIC):
            off = flags == _lib.DETERMINISTIC and tiles > 2048
            assert waves(ctx.fused_ptr, flags) == (0 if off else {pooled}), flags
            assert waves(ctx.fused_noalloc_ptr, flags) == (0 if off else {noalloc}), flags
        bwd = lambda p, b, i, B, T, H, W, s, l, g, flags: ctx.from_grad_ptr(p, b, i, B, T, H, W, s, g, flags=flags)
        assert waves(bwd, 0) == {pooled}
    """)


@pytest.mark.parametrize("B,H,W,T,render,fused", [
    (1, 512, 512, 63, 0, 0), (1, 512, 512, 64, 0, 1), (1, 512, 512, 127, 0, 1), (1, 512, 512, 128, 1, 1),
    (1, 40, 4096, 128, 1, 1), (6, 256, 256, 64, 0, 1), (16, 256, 256, 64, 0, 1), (17, 256, 256, 64, 0, 1),
    # up to 512 tile rows in all, past them from 2048 triangles times a scene's rows
    (24, 128, 128, 64, 0, 1), (32, 128, 128, 64, 0, 1), (33, 128, 128, 127, 0, 0), (33, 128, 128, 128, 1, 1),
    (64, 64, 128, 128, 1, 1), (96, 64, 64, 128, 0, 0), (96, 64, 64, 255, 0, 0), (96, 64, 64, 256, 1, 1),
    (65, 64, 128, 255, 0, 0), (128, 32, 128, 128, 1, 1), (512, 32, 32, 511, 0, 0), (512, 32, 32, 512, 1, 1),
    (128, 64, 64, 4096, 1, 1), (128, 64, 64, 32800, 0, 0),  # 256 MiB of lists at most
])
def test_row_lists_rule(program, B, H, W, T, render, fused):
    """Whether a render and a fused call outside the segmented kernel's share list the tile rows."""
    program(f"""
        import re
        B, H, W, T = {B}, {H}, {W}, {T}
        params, bg = np.zeros((B, T, 10), np.float32), np.zeros((B, 3), np.float32)
        img, losses, grads = np.zeros((B, H, W, 3), np.float32), np.zeros(B, np.float32), np.zeros((B, T, 10), np.float32)
        names = launched(lambda: ctx.render_ptr(addr(params), addr(bg), B, T, H, W, .002, addr(img)))
        lists = [re.search(r"forward_kernelILi\\d+ELb\\dELb\\dELb(\\d)E", n) for n in names]
        assert [int(m.group(1)) for m in lists if m] == [{render}], names
        names = launched(lambda: ctx.fused_ptr(addr(params), addr(bg), addr(img), B, T, H, W, .002, addr(losses),
                                               addr(grads)))
        lists = [re.search(r"fused_tile_kernelILi\\d+ELb\\dELb(\\d)E", n) for n in names]
        lists = [int(m.group(1)) for m in lists if m]
        assert lists == [{fused}] or not lists and T > 1024, names
    """)


SEG, ONE_WAVE, ONE_WAVE_ROWS = "fused_seg_kernel", r"fused_tile_kernelILi\\d+ELb\\dELb0E", r"fused_tile_kernelILi\\d+ELb\\dELb1E"
SPLIT = r"forward_kernelILi\\d+ELb\\dELb1E"  # with checkpoints


@pytest.mark.parametrize("name,B,H,W,T,segments,entry,kernel", [
    ("split backward", 6, 128, 128, 128, False, "fused_ptr", SPLIT),
    ("split backward from gradients", 6, 128, 128, 128, False, "from_grad_ptr", SPLIT),
    ("merged lists", 1, 480, 512, 300, True, "fused_noalloc_ptr", ONE_WAVE),
    ("merged lists, full region", 1, 480, 512, 304, True, "fused_noalloc_ptr", ONE_WAVE),
    ("merged lists of rows", 1, 480, 512, 304, True, "fused_ptr", ONE_WAVE_ROWS),
    ("ordered", 4, 160, 200, 100, True, "fused_ptr", SEG),
    ("ordered, split", 4, 160, 200, 100, False, "fused_ptr", SPLIT),
    ("backward-ordered, split", 3, 200, 208, 300, False, "fused_ptr", SPLIT),
    ("large-block-order", 2, 720, 768, 40, True, "fused_ptr", ONE_WAVE),
    ("many-triangles", 2, 256, 256, 1100, True, "fused_ptr", SPLIT),
    ("tile-order", 6, 250, 256, 100, True, "fused_ptr", ONE_WAVE_ROWS),
    ("tile-order-row-lists", 6, 256, 245, 300, True, "fused_ptr", ONE_WAVE_ROWS),
    ("tail, 48 scenes", 48, 40, 56, 20, False, "fused_ptr", ONE_WAVE),
    ("tail, 1254 blocks", 1, 600, 520, 40, False, "fused_ptr", ONE_WAVE),
    ("tail, odd", 2, 301, 333, 47, False, "fused_ptr", ONE_WAVE),
], ids=lambda v: v if isinstance(v, str) and " " in v else None)
def test_gpu_tests_reach_their_kernels(program, name, B, H, W, T, segments, entry, kernel):
    """The sizes of GPU tests that name a kernel launch it."""
    program(f"""
        import os, re
        if not {segments}:
            os.environ["DRH_NO_SEGMENTS"] = "1"
        B, H, W, T = {B}, {H}, {W}, {T}
        params, bg = np.zeros((B, T, 10), np.float32), np.zeros((B, 3), np.float32)
        img, losses, grads = np.zeros((B, H, W, 3), np.float32), np.zeros(B, np.float32), np.zeros((B, T, 10), np.float32)
        out = (addr(grads),) if "{entry}" == "from_grad_ptr" else (addr(losses), addr(grads))
        names = launched(lambda: ctx.{entry}(addr(params), addr(bg), addr(img), B, T, H, W, .002, *out))
        assert any(re.search("{kernel}", n) for n in names), names
    """)
