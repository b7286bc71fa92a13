"""CPU tests of the C ABI: libflashrt_moe.so loads, exports every entry point include/flashrt_moe.h
declares (and the Python mirror binds exactly those), and the host-only entry points (sizes,
version, argument checks that fail before any device work) behave as documented. No kernel is
launched here."""
from __future__ import annotations

import ctypes as C
import os
import re

import pytest

from flashrt_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions() -> set[str]:
    text = open(os.path.join(ROOT, "include", "flashrt_moe.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return set(re.findall(r"\b(frt_[a-z0-9_]+)\s*\(", text))


def test_header_matches_bindings():
    assert header_functions() == set(_lib.SIGNATURES)


def test_library_exports_every_symbol():
    L = _lib.lib()
    for name in header_functions():
        assert hasattr(L, name), name


def test_host_entry_points():
    L = _lib.lib()
    assert L.frt_version().decode().startswith("flashrt")
    assert L.frt_q2_mat_bytes(512, 2048) == 294912
    assert L.frt_q2_expert_bytes(2048, 512) == 884736
    assert L.frt_q2_expert_bytes(2560, 640) == 1382400
    assert L.frt_moe_q2_workspace_bytes(2048, 10, 2048, 512, 512) > 0
    assert L.frt_moe_dispatch_workspace_bytes(2048, 10, 512) > 0


def _layer(E, n, ff, K, dense=None, shared_ff=0, norm=0):
    """A layer description for the size functions (its pointers are never read)."""
    d = _lib.FrtMoeLayer(1, 1 << 30, E, 1, 1, 0, 1, n, ff, K, norm)
    if dense is not None:
        d.shared_dense, d.shared_type, d.shared_ff = 1, dense, shared_ff
        d.shared_gate = d.shared_up = d.shared_down = 1
    return d


@pytest.mark.parametrize("n,ff", [(2048, 512), (2560, 640), (4096, 256), (512, 128), (2560, 2048)])
@pytest.mark.parametrize("K", [1, 10, 15, 31, 32])
def test_dense_layer_workspace_grows_with_tokens(n, ff, K):
    """A workspace sized for a longer call of a layer with a dense shared expert holds every shorter one,
    across the window, slot and grouped paths."""
    for gtype in (0, 8, 30):
        for shared_ff in (64, 640, 4096):
            d = _layer(512, n, ff, K, gtype, shared_ff)
            b = [_lib.lib().frt_moe_layer_workspace_bytes(C.byref(d), T) for T in range(1, 65)]
            assert b == sorted(b), (gtype, shared_ff, [T for T in range(1, 64) if b[T - 1] > b[T]])


def test_noalloc_scratch_holds_dense_windows():
    """Every window the allocation-free entry takes (T <= 4, T * K <= 63) of a layer with the widest dense shared
    expert fits its static scratch."""
    L = _lib.lib()
    worst = max((L.frt_moe_layer_workspace_bytes(C.byref(_layer(1024, n, ff, K, gtype, 4096, 1)), T), n, ff, K, gtype, T)
                for n in (512, 2560, 4096) for ff in (256, 640, 1024) for gtype in (0, 8) for T in (1, 2, 3, 4)
                for K in range(1, 33) if T * K <= 63)
    assert 0 < worst[0] <= L.frt_noalloc_scratch_bytes(), worst


@pytest.mark.parametrize("E,K", [(1, 1), (2, 2), (7, 3), (8, 8), (64, 8), (128, 1), (512, 10), (1025, 1)])
def test_grouped_workspaces_grow_with_tokens(E, K):
    """The workspaces of the dispatch alone, the grouped expert products and a prefill layer never shrink as the
    tokens grow, across the tile sizes that the number of slots selects (1536 slots)."""
    L = _lib.lib()
    T = range(9, 2 * 1536 // K + 70)
    d = _layer(E, 512, 128, K)
    for size in (lambda t: L.frt_moe_dispatch_workspace_bytes(t, K, E), lambda t: L.frt_moe_q2_workspace_bytes(t, K, 128, 128, E),
                 lambda t: L.frt_moe_layer_workspace_bytes(C.byref(d), t)):
        b = [size(t) for t in T]
        assert b == sorted(b), [(t, x, y) for t, x, y in zip(T, b, b[1:]) if x > y]


def test_stack_workspace_holds_every_layer():
    """A stack whose layers have shared experts of different kinds and widths: its workspace holds the largest
    layer's, whichever comes first, and the two activation buffers."""
    L = _lib.lib()
    kinds = [(None, 0), (8, 64), (8, 640), (0, 4096)]
    for n, ff, K in ((512, 2048, 15), (2048, 512, 10), (2560, 640, 10)):
        for a in kinds:
            for b in kinds:
                two = (_lib.FrtMoeLayer * 2)(_layer(16, n, ff, K, *a), _layer(16, n, ff, K, *b))
                one = [L.frt_moe_layer_workspace_bytes(C.byref(d), 1) for d in two]
                assert L.frt_moe_stack_workspace_bytes(two, 2) == max(one) + 2 * 4 * n, (n, ff, a, b, one)


def test_argument_errors_before_device_work():
    """Shape and null-pointer errors are reported with a status and a message, as the reference's
    std::runtime_error would be, without touching a device."""
    L = _lib.lib()
    rc = L.frt_moe_route_topk(None, None, 1, 512, 10, None, None, None, None, 1 << 30)
    assert rc != 0 and L.frt_last_error()
    rc = L.frt_moe_route_topk(None, None, 1, 512, 0, None, None, None, None, 1 << 30)
    assert rc != 0
    with pytest.raises(_lib.FrtError):
        _lib.check(L.frt_moe_q2_run(None, 0, 512, 2048, 512, None, None, 16, 10, None, None, 0, None, 1, 0))


@pytest.mark.parametrize("T", [1, 4, 8, 9, 20])
@pytest.mark.parametrize("gtype", [0, 8])
@pytest.mark.parametrize("norm", [0, 1])
def test_dense_layer_refuses_shapes_before_any_launch(T, gtype, norm):
    """A layer with a dense shared expert whose n is a multiple of 128 but not of 512: the grouped products
    would take it, the router does not. The call is refused for its shape before it launches anything (a
    launch would report FRT_ERR_HIP here, where there is no device)."""
    L = _lib.lib()
    d = _layer(16, 640, 128, 2, gtype, 64, norm)
    n = L.frt_moe_layer_workspace_bytes(C.byref(d), T)
    ws = C.create_string_buffer(n + 256)
    before = ws.raw
    rc = L.frt_moe_layer_forward(C.byref(d), 256, T, None, 256, None, None, None, (C.addressof(ws) + 255) // 256 * 256, n, None)
    assert rc == -1, (rc, L.frt_last_error())
    assert ws.raw == before


def test_q2_repack_matches_reference_fixture():
    """The product's host repack (frt_q2_repack) reproduces the reference's compiled repack on the
    golden blocks bit for bit (tests/golden/q2_format.npz, 8 rows x 4096), and repack_expert places
    gate | up | down back to back (quant/q2_0/q2_0.cpp:64-80); bad shapes are refused."""
    import numpy as np
    import flashrt_amd as F
    g = np.load(os.path.join(ROOT, "tests", "golden", "q2_format.npz"))
    assert np.array_equal(F.q2_repack(g["repack_in"], 8, 4096), g["repack_out"])
    rng = np.random.default_rng(1)
    n, ff = 256, 128
    mats = [rng.integers(0, 256, r * (c // 64) * 18, dtype=np.uint8) for r, c in ((ff, n), (ff, n), (n, ff))]
    blob = F.q2_repack_expert(*mats, n, ff)
    want = np.concatenate([F.q2_repack(mats[0], ff, n), F.q2_repack(mats[1], ff, n), F.q2_repack(mats[2], n, ff)])
    assert np.array_equal(blob, want)
    with pytest.raises(F.FrtError):
        F.q2_repack(mats[0], ff, 100)


def test_load_experts_reports_io_errors():
    """A missing shard file is an FRT_ERR_IO error with its path in the message (checked before any
    device work)."""
    import flashrt_amd as F
    arena = F._lib.FrtArena(C.c_void_p(1), F.expert_bytes(1024, 256), 0, 1, 1)
    a = F.ExpertArena(arena)
    with pytest.raises(F.FrtError) as e:
        F.load_experts(["/nonexistent/model.gguf"], [(0, 0)] * 3, 1024, 256, a, threads=1)
    assert e.value.code == -5 and "/nonexistent/model.gguf" in str(e.value)


def test_product_does_not_use_the_oracle():
    """The product package never imports or loads anything under oracle/."""
    pkg = os.path.join(ROOT, "flashrt_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".cpp", ".hip", ".hpp", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert not re.search(r"(import\s+oracle|from\s+oracle|liboracle|libfrref|oracle/)", text), \
                    os.path.join(dirpath, f)


def test_cpp_mirror_host():
    """The C++ mirror (include/flashrt_moe.hpp) compiles into a client and maps status codes to
    std::runtime_error (built by `make -C flashrt_amd/csrc`)."""
    import subprocess
    exe = os.path.join(ROOT, "tests", "cpp", "_build", "test_shim")
    assert os.path.exists(exe), "build first: make -C flashrt_amd/csrc"
    r = subprocess.run([exe, "--host"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "all passed" in r.stdout, r.stdout + r.stderr
