"""The shared library loads without a GPU and exports every symbol include/metis_hip.h declares."""
import ctypes
import os
import re
import subprocess
import sys
import threading
import time

import numpy as np
import pytest
import torch

from metis_hip import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header():
    text = open(os.path.join(ROOT, "include", "metis_hip.h")).read()
    return re.sub(r"/\*.*?\*/", "", text, flags=re.S)


def _declared():
    return sorted(set(re.findall(r"\b(metis_[a-z0-9_]+)\s*\(", _header())))


def test_every_declared_symbol_is_exported_and_bound():
    lib = _lib.load()
    names = _declared()
    assert len(names) >= 12
    for n in names:
        assert hasattr(lib, n), f"{n} declared in metis_hip.h but not exported"
        assert n in _lib.SIGNATURES, f"{n} has no ctypes signature"
    assert sorted(_lib.SIGNATURES) == names


def test_host_only_calls():
    lib = _lib.load()
    assert lib.metis_version() >= 0x100
    assert b"16" in lib.metis_error_string(_lib.E_SHAPE)
    assert lib.metis_nvfp4_workspace_bytes(8192, 4096) >= 8192 * 4096 // 16 * 2
    assert lib.metis_nvfp4_workspace_bytes(0, 0) > 0


def test_size_helpers_of_the_one_pass_entry_points_need_no_device():
    """The workspace and buffer sizes a caller asks for before it allocates: pure host arithmetic (a 256-CU device is
    assumed when none is present).  K slices only while the row tiles alone leave compute units idle, never more than 16,
    never fewer than four 256-element steps each; the deferred buffer holds 2048 partial maxima and one bf16 per block."""
    from metis_hip import _lib
    L = _lib.load()
    ws = L.metis_lowrank_project_rows_workspace_bytes
    assert ws(8192, 64, 4096) == 0 and ws(16384, 64, 18944) == 0          # 256 row tiles or more: one slice
    assert ws(1024, 64, 18944) == 16 * 1024 * 64 * 4                       # 32 row tiles, 74 steps: 16 slices
    assert ws(4096, 32, 8960) == 4 * 4096 * 32 * 4                         # 128 row tiles: 4 slices
    assert ws(4096, 32, 1536) == 0                                          # 6 steps: fewer than four per slice
    assert ws(0, 64, 4096) == 0 and ws(1024, 0, 4096) == 0
    for rows, cols in ((256, 64), (8192, 4096), (300, 192)):
        nb = rows * cols // 16
        assert L.metis_nvfp4_deferred_bytes(rows, cols) == 2048 * 4 + (nb * 2 + 255) // 256 * 256
        assert L.metis_nvfp4_workspace_bytes(rows, cols) >= 16384 + nb * 4
    assert L.metis_nvfp4_deferred_bytes(0, 64) == 0


def test_compiled_calls_take_the_arguments_that_the_abi_declares():
    """_lib.call reaches its entry points through their declarations in metis_hip.h; what Python passes is counted and its kinds looked at before
    anything is allocated on a device or launched.  (No call of this test gets that far.)"""
    with pytest.raises(KeyError):
        _lib.call("metis_no_such_entry", 0, (), ())
    source = open(os.path.join(os.path.dirname(_lib.LIB_PATH), "..", "csrc", "host_calls.cpp")).read()
    names = re.findall(r"METIS_ENTRY\((metis_\w+)\)", source)
    assert len(names) > 30 and len(set(names)) == len(names)
    for name in names:
        args = _lib.SIGNATURES[name][1]
        for n in (len(args) - 1, len(args) + 1):
            with pytest.raises(TypeError, match=rf"{name} takes {len(args)} arguments"):
                _lib.call(name, 0, (), (0,) * n)
        with pytest.raises(TypeError):
            _lib.call(name, 0, (), (0.5,) * len(args))              # a float for a pointer
        with pytest.raises(TypeError):
            _lib.call(name, 0, (), (0,) * (len(args) - 1) + ("0",))  # a new tensor that is not there
    with pytest.raises(ValueError):
        _lib.call("metis_rmsnorm", 0, ((7, 1),), (0,) * 7)


def test_compiled_calls_take_every_argument_by_its_declared_kind():
    """What ctypes refused for an integer, a float or an address is refused here too, what it took for one has the same value, and an array of
    structures is as long as its number says.  (No call gets beyond the entry points' own argument checks.)"""
    source = open(os.path.join(os.path.dirname(_lib.LIB_PATH), "..", "csrc", "host_calls.cpp")).read()
    structures = {"metis_linear_member": 12, "metis_lowrank_factor": 3}
    words = {kind: (None,) * 5 + (0, None, None, 0, 0, 0, None) if n == 12 else (None, None, 0) for kind, n in structures.items()}
    header = _header()
    for name in re.findall(r"METIS_ENTRY\((metis_\w+)\)", source):
        declared = [" ".join(a.split()) for a in re.search(rf"\b{name}\(([^)]*)\)", header).group(1).split(",")]
        types = _lib.SIGNATURES[name][1]
        assert len(declared) == len(types)
        arrays = {i: kind for i, a in enumerate(declared) for kind in structures if kind in a}
        good = []
        for i, t in enumerate(types):
            good.append([words[arrays[i]]] if i in arrays else 1 if i - 1 in arrays else None if t is ctypes.c_void_p else 0.0 if t is ctypes.c_float else 0)

        def call(i, value):
            return _lib.call(name, 0, (), tuple(good[:i] + [value] + good[i + 1:]))

        for i, t in enumerate(types):
            if i in arrays:
                bad = [None, 0, torch.zeros(4), (), "0", [()], [words[arrays[i]][1:]], [words[arrays[i]] + (0,)], [list(words[arrays[i]])]]
                bad += [[words[arrays[i]][:k] + (0.5,) + words[arrays[i]][k + 1:]] for k in range(len(words[arrays[i]]))]
                with pytest.raises(ValueError, match=f"{name}: 2 structures for 1"):
                    call(i, [words[arrays[i]]] * 2)
            elif t is ctypes.c_void_p:
                bad = [0.5, np.int64(16), "00", "0", (), [words["metis_lowrank_factor"]]]
            elif t is ctypes.c_float:
                bad = [None, "1", torch.zeros(2), ()]
            else:
                bad = [None, 0.5, "1", torch.zeros(2, dtype=torch.int64), torch.tensor(0.5), (), [words["metis_lowrank_factor"]]]
            for value in bad:
                with pytest.raises((TypeError, ValueError, RuntimeError)):
                    call(i, value)
    # numbers of other libraries, and tensors that hold one: 33 columns are no whole blocks, 32 without a tensor are an argument error
    row = "metis_nvfp4_quant_row"
    for columns in (33, np.int64(33), np.uint8(33), torch.tensor(33), torch.tensor([33])):
        assert _lib.call(row, 0, (), (None, 16, columns, 64, 0, None, None, None, None, 0, None)) == _lib.E_SHAPE
    assert _lib.call(row, 0, (), (None, 16, 32, 64, 0, None, None, None, None, 0, None)) == _lib.E_ARG


def test_compiled_calls_allocate_tensors_of_any_number_of_dimensions():
    """(The device does not exist: the allocation itself fails, not what is asked of it.)"""
    with pytest.raises(RuntimeError):
        _lib.call("metis_nvfp4_roundtrip", 99, ((_lib.F32, *(1,) * 11, 16),), (None, 1, 16, 0, "0", None, 0, 0, None))


def test_compiled_calls_give_up_the_interpreter_while_they_allocate():
    """No thread is made to hand over the interpreter here, so another one runs only where the calls let it.  (The device does not exist: every
    call ends in its allocation.)"""
    args = ("metis_nvfp4_roundtrip", 99, ((_lib.F32, 1, 16),), (None, 1, 16, 0, "0", None, 0, 0, None))
    turns, stop = [0], False

    def other():
        while not stop:
            turns[0] += 1
            time.sleep(0)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    with pytest.raises(RuntimeError):
        _lib.call(*args)
    sys.setswitchinterval(1000.0)
    try:
        thread.start()
        while not turns[0]:
            time.sleep(0.001)
        before = turns[0]
        for _ in range(20000):
            try:
                _lib.call(*args)
            except RuntimeError:
                pass
            if turns[0] > before + 10:
                break
        ran = turns[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop = True
        thread.join()
    assert ran > 10


def test_the_library_builds_without_torch():
    """What `make` would run: the library and the probes for any interpreter, Python's way into the library for the one that has torch."""
    csrc = os.path.join(os.path.dirname(_lib.LIB_PATH), "..", "csrc")
    for python, has_torch in ((sys.executable, True), (f"{sys.executable} -S -I", False), ("no-such-interpreter", False)):
        run = subprocess.run(["make", "-B", "-n", "-C", csrc, f"PYTHON={python}"], capture_output=True, text=True)
        assert run.returncode == 0, run.stderr
        assert "libmetis_hip.so" in run.stdout and "libmetis_ceilings.so" in run.stdout
        assert ("host_calls.cpp" in run.stdout) == has_torch
