"""The register-march stage (fv2d_amd/csrc/fv2d_march.h), run lane by lane on the host
(tests/emu/march_emu.cpp), against the CPU oracle: bitwise-equal dt, reset counts and fields
over the switch combinations and at the edges of its strips (60 output columns per wave) and
row segments; the FP32 form close to the oracle. A sanitized build of one class checks every
global index and slot of the same code."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import emu as EMU
import test_emulated_kernel as T
from fv2d_amd.capi import FP32, FP32_STATE64, FP64, PLM, Params

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
FLAGS = ["-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-fno-fast-math", "-Wno-unknown-pragmas"]
SAN = ["-O1", "-DMARCH_EMU_FEW", "-fsanitize=address,undefined", "-fno-sanitize-recover=all"]


def build(name, flags):
    out = os.path.join(HERE, name)
    csrc = os.path.join(HERE, "..", "..", "fv2d_amd", "csrc")
    deps = [os.path.join(HERE, f) for f in ("march_emu.cpp", "tile_emu.cpp", "tile_emu.h")]
    deps += [os.path.join(csrc, f) for f in ("fv2d_march.h", "fv2d_stage.h", "fv2d_math.h", "fv2d_params.h")]
    if not os.path.exists(out) or os.path.getmtime(out) < max(os.path.getmtime(d) for d in deps):
        subprocess.run(["g++", *FLAGS, *flags, "-o", out, os.path.join(HERE, "march_emu.cpp")], check=True)
    return out


def load(path):
    lib, dp = C.CDLL(path), C.POINTER(C.c_double)
    lib.emu_create.restype = C.c_void_p
    lib.emu_create.argtypes = [C.POINTER(Params), C.c_char_p]
    lib.emu_destroy.argtypes = [C.c_void_p]
    lib.emu_set_prim.argtypes = [C.c_void_p, dp]
    lib.emu_compute_dt.restype = C.c_double
    lib.emu_compute_dt.argtypes = [C.c_void_p, dp]
    lib.emu_step.argtypes = [C.c_void_p, C.c_double, C.POINTER(C.c_uint64)]
    lib.emu_get_prim.argtypes = [C.c_void_p, dp]
    lib.emu_get_cons.argtypes = [C.c_void_p, dp]
    return lib


@pytest.fixture(scope="module")
def march_lib():
    return load(build("libmarch_emu.so", ["-O2"]))


def test_switch_combinations_bitwise(march_lib, oracle_lib):
    for n, c in enumerate(T.COMBOS):
        if n % 5 == 0:
            p, q0 = T.make(n, *c)
            T.compare(p, q0, march_lib, oracle_lib, steps=2)


SHAPES = [(2, 2, 0), (3, 5, 0), (59, 33, 4), (60, 4, 0), (61, 9, 4), (62, 7, 0), (120, 66, 8), (121, 130, 12), (130, 7, 4),
          (5, 301, 0), (63, 45, 20)]
CLASSES = [(1, 1, PLM, 1, 1, 1, 1, 1, 1), (2, 0, PLM, 0, 0, 0, 1, 0, 0), (0, 2, 0, 2, 1, 1, 0, 2, 1)]


@pytest.mark.parametrize("Nx,Ny,seg", SHAPES)
def test_grid_shapes_bitwise(Nx, Ny, seg, march_lib, oracle_lib):
    for n, c in enumerate(CLASSES):
        p, q0 = T.make(n, *c, Nx=Nx, Ny=Ny)
        T.compare(p.copy(seg_rows=seg), q0, march_lib, oracle_lib, steps=2)


@pytest.mark.parametrize("precision", [FP64, FP32, FP32_STATE64])
@pytest.mark.parametrize("Nx,Ny,seg,banded", [
    (2, 2, 0, False), (512, 8, 0, False), (1024, 1024, 0, False), (60, 70, 4, False), (4096, 4096, 0, True),
    (2048, 2048, 0, True), (4097, 4099, 0, True), (60, 40001, 0, None), (70000, 301, 0, True), (2048, 2048, 64, False)])
def test_tasks_cover_the_grid_once(Nx, Ny, seg, banded, precision, march_lib):
    """Every (strip, row) belongs to one task, in the uniform and in the banded long-then-short split."""
    p = Params.defaults(Nx=Nx, Ny=Ny, seg_rows=seg, precision=precision)
    march_lib.emu_march_tasks.argtypes = [C.POINTER(Params), C.POINTER(C.c_int), C.POINTER(C.c_int)]
    bands = C.c_int()
    n = march_lib.emu_march_tasks(C.byref(p), None, C.byref(bands))
    out = np.zeros((n, 3), dtype=np.int32)
    march_lib.emu_march_tasks(C.byref(p), out.ctypes.data_as(C.POINTER(C.c_int)), C.byref(bands))
    if banded is not None:  # (60 x 40001: 10 rows per wave of an FP64 grid, 6.5 of an FP32 one)
        assert bands.value == (8 if banded else 1)
    live = out[out[:, 2] > out[:, 1]]
    assert (live[:, 0] % 60 == 0).all() and live[:, 0].max() < Nx and live[:, 1].min() == 0 and live[:, 2].max() == Ny
    nsx = -(-Nx // 60)
    edge = np.zeros((nsx, Ny + 1), dtype=np.int64)
    np.add.at(edge, (live[:, 0] // 60, live[:, 1]), 1)
    np.add.at(edge, (live[:, 0] // 60, live[:, 2]), -1)
    assert (np.cumsum(edge, axis=1)[:, :Ny] == 1).all()


def test_resets_nan_and_fp32(march_lib, oracle_lib):
    T.test_reset_and_nan_counts(0, march_lib, oracle_lib)
    T.fp32_close(march_lib, oracle_lib, N=64, steps=8)


def test_sanitized_bounds(oracle_lib):
    """ASan / UBSan in a child interpreter: a bad index aborts it."""
    lib = build("libmarch_emu_san.so", SAN)
    code = ("import sys; sys.path[:0] = %r\n"
            "import test_emulated_march as M, test_emulated_kernel as T\n"
            "from oracle import oracle as OR\n"
            "lib, olib = M.load(%r), OR.load()\n"
            "for Nx, Ny, seg in M.SHAPES:\n"
            "    for n, c in enumerate(((1, 1, 2, 1, 1, 1, 1, 1, 1), (2, 0, 2, 1, 0, 1, 1, 0, 0))):\n"
            "        p, q0 = T.make(n, *c, Nx=Nx, Ny=Ny)\n"
            "        T.compare(p.copy(seg_rows=seg), q0, lib, olib, steps=2)\n"
            "T.fp32_close(lib, olib, N=24, steps=4)\n"
            "print('ok')\n" % ([os.path.dirname(os.path.abspath(__file__)), os.path.dirname(os.path.dirname(HERE)), HERE],
                                lib))
    pre = ":".join(subprocess.run(["g++", f"-print-file-name=lib{n}.so"], capture_output=True, text=True).stdout.strip()
                   for n in ("asan", "ubsan"))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=1200,
                       env=dict(os.environ, LD_PRELOAD=pre, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and "ok" in r.stdout, r.stderr[-3000:]
