"""The C-ABI library loads and exports every symbol include/*.h declares; pure
host-side argument validation works without a GPU (no compute calls here)."""
import ctypes
import glob
import hashlib
import os
import random
import re
import shutil
import subprocess
import sys

import pytest

from mindspeed_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    names = set()
    for header in glob.glob(os.path.join(ROOT, "include", "*.h")):
        text = open(header).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names.update(re.findall(r"\b(ms_[a-z0-9_]+)\s*\(", text))
    return names


def test_header_and_binding_agree():
    assert declared_symbols() == set(_lib.EXPORTED_SYMBOLS)


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    for name in sorted(declared_symbols()):
        assert hasattr(lib, name), name
    assert lib.ms_version() == _lib.ABI_VERSION


def test_the_version_moves_with_the_entry_points(tmp_path):
    """The names that a version stands for, and what a build of the version before says when it is loaded: that it has to
    be built again (and not which symbol it lacks)."""
    names = " ".join(sorted(declared_symbols()))
    assert (_lib.ABI_VERSION, hashlib.sha256(names.encode()).hexdigest()[:16]) == (104, "357be616bd29ac47")
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    stale = tmp_path / "stale.so"
    subprocess.run([cc, "-shared", "-fPIC", "-x", "c", "-", "-o", str(stale)], input=f"int ms_version(void) {{ return {_lib.ABI_VERSION - 1}; }}",
                   text=True, check=True)
    res = subprocess.run([sys.executable, "-c", "from mindspeed_amd import _lib; _lib.load()"], capture_output=True, text=True,
                         cwd=ROOT, env=dict(os.environ, MINDSPEED_AMD_LIB=str(stale)))
    assert res.returncode != 0 and "rebuild it" in res.stderr and "undefined symbol" not in res.stderr


def test_workspace_size_and_validation_are_host_only():
    lib = _lib.load()
    n = ctypes.c_size_t(123)
    assert lib.ms_moe_token_permute_workspace_size(4096, 2, 8, ctypes.byref(n)) == 0 and n.value == 0
    assert lib.ms_moe_token_permute_workspace_size(8192, 8, 64, ctypes.byref(n)) == 0 and n.value == 64 * 64 * 4
    assert lib.ms_moe_token_permute_workspace_size(8192, 8, 0, ctypes.byref(n)) == 0 and n.value == 64 * 1024 * 4
    assert lib.ms_moe_token_permute_workspace_size(8, 2, 5000, ctypes.byref(n)) != 0
    assert b"exceeds" in lib.ms_last_error()
    assert lib.ms_gmm_workspace_size(8, 8192, 0, ctypes.byref(n)) == 0 and n.value >= 8 * 40
    assert lib.ms_gmm_workspace_size(0, 8192, 0, ctypes.byref(n)) != 0
    # the second query adds room for partial sums only where tail tiles may be split: split on rows, 16-bit output,
    # few rounds of tiles over a long reduction
    base, m2 = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert lib.ms_gmm_workspace_size(8, 8192, 0, ctypes.byref(base)) == 0
    BF16, FP32 = 0, 2
    assert lib.ms_gmm_workspace_size_split(8, 8192, 14336, 4096, 0, BF16, BF16, 0, ctypes.byref(m2)) == 0
    assert base.value + (16 << 20) <= m2.value <= base.value + (32 << 20) + 4096       # fc2 forward of the Mixtral shape
    for args in [(8, 8192, 4096, 28672, 0, BF16, BF16, 0),      # many rounds of tiles
                 (8, 8192, 2048, 4096, 0, BF16, BF16, 0),       # short reduction
                 (8, 8192, 14336, 4096, 2, BF16, BF16, 0),      # split on the reduction dim
                 (8, 8192, 14336, 4096, 0, BF16, FP32, 1),      # fp32 accumulate form
                 (8, 8192, 14336, 4096, 0, FP32, FP32, 0),      # fp32 operands
                 (4, 600, 8192, 512, 0, BF16, BF16, 0)]:        # far less than a round of tiles
        assert lib.ms_gmm_workspace_size_split(*args, ctypes.byref(m2)) == 0
        assert lib.ms_gmm_workspace_size(args[0], args[1], args[4], ctypes.byref(base)) == 0
        assert m2.value == base.value, args
    assert lib.ms_gmm_workspace_size_split(0, 8192, 14336, 4096, 0, BF16, BF16, 0, ctypes.byref(m2)) != 0
    # bad arguments are rejected before anything is launched
    rc = lib.ms_gmm(None, None, 1, 1, None, 1, 1, 1, None, 1, None, 0, 1, 8, 16, 16, 16, 0, 0, 0, None, 0)
    assert rc != 0 and b"group_type" in lib.ms_last_error()
    rc = lib.ms_gmm(None, None, 1, 1, None, 1, 1, 1, None, 1, None, 0, 0, 8, 16, 16, 16, 7, 7, 0, None, 0)
    assert rc != 0 and b"dtype" in lib.ms_last_error()
    rc = lib.ms_swiglu(None, None, None, 0, -1, 16, 0, None)
    assert rc != 0
    rc = lib.ms_moe_token_unpermute(None, None, None, None, 0, 4, 0, 16, 0, 8, None)
    assert rc != 0 and b"topk" in lib.ms_last_error()
    with pytest.raises(_lib.MindSpeedAmdError):
        _lib.check(rc, "ms_moe_token_unpermute")
    # probabilities and token numbers of routing-map rows come with the rows (no pointer here is ever followed)
    for probs, permuted_probs, ids in ((64, 64, None), (None, None, 64)):
        rc = lib.msi_routing_map_permute(None, None, 64, 4, 2, 8, BF16, 4, 0, None, 64, 64, None, probs, FP32, permuted_probs, ids, 64, 1 << 20)
        assert rc != 0 and b"with the rows only" in lib.ms_last_error()


def test_tile_order_visits_every_tile_once():
    """The order in which the grouped-matmul kernels walk the tiles of a group (blocks of 4 row tiles x 8 column
    panels, partly filled blocks at both edges, a single left-over row tile joining the last block) is a bijection
    for every group shape up to 40 x 40, and where the sides are multiples of 4 and 8 every run of 32 consecutive
    indices is one 4 x 8 block."""
    lib = _lib.load()
    row, col = ctypes.c_int(-1), ctypes.c_int(-1)
    for R in range(1, 41):
        for C in range(1, 41):
            seen = set()
            order = []
            for i in range(R * C):
                assert lib.ms_gmm_tile_order(R, C, i, ctypes.byref(row), ctypes.byref(col)) == 0
                assert 0 <= row.value < R and 0 <= col.value < C, (R, C, i, row.value, col.value)
                seen.add((row.value, col.value))
                order.append((row.value, col.value))
            assert len(seen) == R * C, (R, C)
            if R % 4 == 0 and C % 8 == 0:
                for b in range(0, R * C, 32):
                    chunk = order[b:b + 32]
                    assert len({r for r, _ in chunk}) == 4 and len({c for _, c in chunk}) == 8, (R, C, b)
    assert lib.ms_gmm_tile_order(4, 4, 16, ctypes.byref(row), ctypes.byref(col)) != 0
    assert lib.ms_gmm_tile_order(0, 4, 0, ctypes.byref(row), ctypes.byref(col)) != 0


def _cdiv(a, b):
    return -(-a // b)


def _slots_needed_split_on_rows(counts, m, k, n):
    """Slots per XCD of the tables the schedule kernel can write for these group sizes (256 x 256 tiles): the common table,
    the common table with every small tail tile cut in parts, and the per-XCD lists (None where they are not taken)."""
    cols = _cdiv(n, 256)
    row_tiles = [_cdiv(c, 256) for c in counts]
    tiles = sum(row_tiles) * cols
    zero_fill = _cdiv(m - sum(counts), 256) * cols               # rows past the last group are written as zeros
    tail_tiles = sum(1 for c in counts if 1 <= (c - 1) % 256 + 1 <= 128 and c > 0) * cols
    parts = min(256 // tail_tiles, k // 2048, 4) if tail_tiles else 1
    split = tiles + max(parts - 1, 0) * tail_tiles
    lists = None
    if 16 <= len(counts) <= 256 and max(row_tiles) <= 8:
        load = [0] * 8
        for rank, t in enumerate(sorted(row_tiles, reverse=True)):
            load[7 - rank % 8 if rank // 8 % 2 else rank % 8] += t * cols
        if tiles > 0 and max(load) * 800 <= tiles * 103:
            lists = max(load) + _cdiv(zero_fill, 8)
    return _cdiv(tiles + zero_fill, 8), _cdiv(split + zero_fill, 8), lists


def test_launch_has_slots_for_every_table_the_schedule_can_write():
    """Workgroups per XCD of a grouped-matmul launch (exactly what is launched) against the slots that the tables of many
    group lists need, evaluated on the host: ragged, equal and empty groups, fewer rows than groups, rows past the last
    group, split tail tiles, whole groups per XCD.  The launch carries no workgroup beyond its bound either: a workgroup
    without a tile still waits for a compute unit."""
    lib = _lib.load()
    slots = ctypes.c_int64(0)

    def launched(G, m, k, n, group_type, lists, split):
        assert lib.ms_gmm_launch_slots(G, m, k, n, group_type, lists, split, ctypes.byref(slots)) == 0
        return slots.value

    # Split on the reduction dim: every group has all its tiles, also an empty one, so the common table needs an eighth of
    # them.  Per-XCD lists: the XCD with the most groups holds ceil(G / 8) output blocks, e.g. 3 of 17.
    for G in (1, 8, 16, 17, 20, 23, 24, 31, 33, 64, 100, 255, 256, 4096):
        for k, n in ((2048, 8192), (2880, 2880), (256, 256), (4096, 4096), (8, 8), (1000, 520)):
            out_tiles = _cdiv(k, 256) * _cdiv(n, 256)
            assert launched(G, 4096, k, n, 2, 0, 0) == _cdiv(G * out_tiles, 8)
            assert launched(G, 4096, k, n, 2, 1, 0) == _cdiv(G, 8) * out_tiles

    # Split on rows: at most ceil(m / 256) + G + 1 row tiles (every group and the zero-fill pseudo-group may end in a partly
    # filled one) and at most one per row.
    rng = random.Random(0)
    with_lists = fullest = 0
    for trial in range(4000):
        G = rng.choice([1, 2, 3, 8, 16, 17, 20, 24, 33, 64, 100, 255, 256, 300])
        k, n = rng.choice([72, 2048, 4096, 14336]), rng.choice([8, 264, 1408, 4096, 28672])
        kind = rng.randrange(5)
        if kind == 0:
            counts = [rng.randrange(0, 3) for _ in range(G)]                  # fewer rows than groups, many empty
        elif kind == 1:
            counts = [rng.choice([1, 257, 513, 128, 129]) for _ in range(G)]   # every last tile nearly empty
        elif kind == 2:
            counts = [rng.randrange(1, 9) * 256] * G                           # equal groups of whole tiles
        elif kind == 3:
            counts = [int(rng.expovariate(1 / 700)) for _ in range(G)]
        else:
            counts = [256 * rng.randrange(1, 4) + rng.randrange(256) for _ in range(G)]
        m = max(sum(counts) + rng.choice([0, 0, 1, 255, 257, 3000]), 1)
        common, split, lists = _slots_needed_split_on_rows(counts, m, k, n)
        got = launched(G, m, k, n, 0, 0, 0)
        assert common <= got, (counts, m, n, common, got)
        assert got == _cdiv(min(_cdiv(m, 256) + G + 1, m) * _cdiv(n, 256), 8)
        assert split <= launched(G, m, k, n, 0, 0, 1), (counts, m, k, n, split, slots.value)
        if lists is not None:
            with_lists += 1
            assert max(lists, common) <= launched(G, m, k, n, 0, 1, 0), (counts, m, n, lists, slots.value)
        fullest = max(fullest, common / got)
    assert with_lists > 300 and fullest > 0.95           # the lists were met, and the bound is nearly reached
    assert lib.ms_gmm_launch_slots(0, 1, 1, 1, 0, 0, 0, ctypes.byref(slots)) != 0
    assert lib.ms_gmm_launch_slots(8, 1, 1, 1, 1, 0, 0, ctypes.byref(slots)) != 0


def _stub(path, interface, version=_lib.ABI_VERSION):
    """A library with every name that this package binds, built from other declarations."""
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    names = (set(_lib._SIGNATURES) | set(_lib._INTERNAL) | {"ms_last_error"}) - {"ms_version"}
    code = "".join(f"int {n}(void) {{ return 0; }}\n" for n in sorted(names))
    code += f"int ms_version(void) {{ return {version}; }}\n"
    if interface is not None:
        code += f'const char *msi_interface(void) {{ return "{interface}"; }}\n'
    subprocess.run([cc, "-shared", "-fPIC", "-x", "c", "-", "-o", str(path)], input=code, text=True, check=True)
    return str(path)


@pytest.mark.parametrize("interface", ["0123456789abcdef", None])
def test_the_native_side_refuses_a_library_of_other_declarations(interface, tmp_path):
    """_host.so passes arguments by the declarations it was compiled with: another build's may differ in them without a name
    missing."""
    lib = _stub(tmp_path / "other.so", interface)
    code = f"import torch; from mindspeed_amd import _host; _host.bind({lib!r}, RuntimeError)"
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT)
    assert res.returncode != 0 and "rebuild" in res.stderr, res.stderr
    # ... and the library of this tree is the one it was built with
    code = "import torch; from mindspeed_amd import _host, _lib; _host.bind(_lib.LIB_PATH, RuntimeError); print('bound')"
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT)
    assert res.returncode == 0 and "bound" in res.stdout, res.stderr


@pytest.mark.parametrize("interface", ["0123456789abcdef", None])
def test_the_python_binding_refuses_a_library_of_other_declarations(interface, tmp_path):
    lib = _stub(tmp_path / "other.so", interface)
    res = subprocess.run([sys.executable, "-c", "from mindspeed_amd import _lib; _lib.load()"], capture_output=True, text=True,
                         cwd=ROOT, env=dict(os.environ, MINDSPEED_AMD_LIB=lib))
    assert res.returncode != 0 and "rebuild it" in res.stderr, res.stderr


def test_the_interface_hash_follows_declarations_and_not_comments(tmp_path, monkeypatch):
    from mindspeed_amd import build
    copies = []
    for f in build.INTERFACE_HEADERS:
        copies.append(str(tmp_path / os.path.basename(f)))
        shutil.copy(f, copies[-1])
    before = build.interface_hash()
    monkeypatch.setattr(build, "INTERFACE_HEADERS", tuple(copies))
    assert build.interface_hash() == before and _lib.load().msi_interface().decode() == before
    text = open(copies[1]).read()
    open(copies[1], "w").write("/* a comment */\n\n" + text + "// and another\n")
    assert build.interface_hash() == before
    open(copies[1], "w").write(text.replace("int drop_and_pad", "int64_t drop_and_pad"))
    assert build.interface_hash() != before


@pytest.mark.parametrize("args,force", [([], True), (["--incremental"], False)])
def test_the_build_command_makes_the_library_and_its_native_side(args, force, monkeypatch):
    from mindspeed_amd import build
    made = []
    monkeypatch.setattr(build, "build", lambda force, verbose: made.append(("library", force)))
    monkeypatch.setattr(build, "build_host", lambda verbose, force: made.append(("host", force)))
    build.main(args)
    assert sorted(made) == [("host", force), ("library", force)]
