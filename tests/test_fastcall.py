"""The extension that the kernel libraries are called through (csrc/python/fastcall.c) against ctypes: the same C functions, the same
arguments, each signature length that it passes in another way (up to 16, 32 and 64 integers), floats between the integers."""
import ctypes
import random
import shutil
import subprocess

import numpy as np
import pytest

from flexible_llm_sharding_amd import _native

TYPES = {"p": ctypes.c_void_p, "i": ctypes.c_int, "l": ctypes.c_longlong, "f": ctypes.c_float}
SIGS = ["i", "p", "fi", "pipipippiiffiiiiiiippliillp"[:26] + "p", "f" * 8 + "i" * 16, "if" * 8 + "p" * 9, "pl" * 16, "ppi" * 21 + "f", "l" * 64]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("no gcc")
    c = {"p": "const void*", "i": "int", "l": "long long", "f": "float"}
    src = "#include <stdio.h>\nstatic char out[8192];\nconst char* seen(void) { return out; }\n"
    for n, sig in enumerate(SIGS):
        put = "".join(f"n += sprintf(out + n, \"{'%a' if k == 'f' else '%lld'} \", {'(double)a' if k == 'f' else '(long long)a'}{i});" for i, k in enumerate(sig))
        src += f"int f{n}({', '.join(f'{c[k]} a{i}' for i, k in enumerate(sig))}) {{ int n = 0; {put} return -n; }}\n"
    d = tmp_path_factory.mktemp("fastcall")
    (d / "f.c").write_text(src)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w", str(d / "f.c"), "-o", str(d / "f.so")], check=True)
    lib = ctypes.CDLL(str(d / "f.so"))
    lib.seen.restype = ctypes.c_char_p
    for n, sig in enumerate(SIGS):
        _native._bind(lib, f"f{n}", ctypes.c_int, *(TYPES[k] for k in sig))
    return lib


def test_same_arguments_as_ctypes(lib):
    quick, rng = _native._Quick(lib), random.Random(0)
    for n, sig in enumerate(SIGS):
        for _ in range(20):
            args = [rng.choice((None, 0, rng.getrandbits(47))) if k == "p" else rng.randint(-2 ** 31, 2 ** 31 - 1) if k == "i"
                    else rng.randint(-2 ** 63, 2 ** 63 - 1) if k == "l" else rng.choice((rng.uniform(-1e3, 1e3), 3, float("inf"))) for k in sig]
            want = (getattr(lib, f"f{n}")(*args), lib.seen())
            assert (getattr(quick, f"f{n}")(*args), lib.seen()) == want


def test_other_arguments_go_to_ctypes(lib):
    quick = _native._Quick(lib)
    buf = ctypes.create_string_buffer(8)
    assert quick.f1(buf) == lib.f1(buf)                              # (an address that only ctypes knows how to take)
    for call in ((quick.f0, "x"), (quick.f0, None), (quick.f0, 1.5), (quick.f2, "x", 1), (quick.f0,), (quick.f2, 1.0)):
        with pytest.raises((ctypes.ArgumentError, TypeError)):
            call[0](*call[1:])


def test_refuses_what_it_cannot_pass():
    f = _native._fastcall().function
    for sig in ("d", "f" * 9, "i" * 65):
        with pytest.raises(ValueError):
            f(1, sig, None)
    with pytest.raises(ValueError):
        f(0, "i", None)


def test_a_library_of_other_signatures_is_refused(tmp_path):
    """A kernel library built before fls_moe_gemm lost an argument says so by its version, and is refused with what to do about it."""
    if shutil.which("gcc") is None:
        pytest.skip("no gcc")
    (tmp_path / "old.c").write_text("int fls_kernels_version(void) { return 33; }")
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "old.c"), "-o", str(tmp_path / "old.so")], check=True)
    with pytest.raises(RuntimeError, match="stale build"):
        _native._load_kernels(str(tmp_path / "old.so"))


def test_token_lists_to_int32():
    int32s, rng = _native.host().int32s, random.Random(1)
    for n in (0, 1, 7, 1000):
        v = [rng.randint(-2 ** 31, 2 ** 31 - 1) for _ in range(n)]
        for seq in (v, tuple(v)):
            out = np.full(n + 2, 5, np.int32)
            assert int32s(out[1:n + 1], seq) is True
            assert out.tolist() == [5] + v + [5]
    out = np.zeros(2, np.int32)
    for seq in ([1, 2 ** 31], [1, -2 ** 31 - 1], [1, 2.0], [1, True], [1, np.int32(2)], [1], [1, 2, 3], np.array([1, 2]), range(2), "12", [1, 10 ** 30]):
        assert int32s(out, seq) is False                             # (left to numpy, which takes or refuses them)
    with pytest.raises((ValueError, BufferError)):
        int32s(np.zeros(4, np.int32)[::2], [1, 2])


@pytest.mark.parametrize("lens,pos0,ps", [([1], [0], 16), ([3, 40, 1], [0, 7, 100], 16), ([64, 64], [0, 64], 64), ([500, 33, 2], [1, 0, 30], 7)])
def test_step_rows(lens, pos0, ps):
    B, cu = len(lens), np.cumsum([0] + lens).astype(np.int32)
    T, p0 = int(cu[-1]), np.asarray(pos0, np.int32)
    P = max((a + n - 1) // ps for a, n in zip(pos0, lens)) + 1
    table = np.random.default_rng(0).permutation(4 * B * P)[:B * P].reshape(B, P).astype(np.int32)
    seq, pos, slot = (np.zeros(T, np.int32) for _ in range(3))
    rows = _native.host().step_rows
    assert rows(cu, p0, table, ps, seq, pos, slot) is True
    b = np.repeat(np.arange(B), lens)
    at = np.arange(T) - cu[b] + p0[b]
    assert (seq == b).all() and (pos == at).all() and (slot == table[b, at // ps] * ps + at % ps).all()
    for hole in ((0, 0 if pos0[0] < ps else pos0[0] // ps), (B - 1, (pos0[-1] + lens[-1] - 1) // ps)):
        bad = table.copy()
        bad[hole] = -1
        assert rows(cu, p0, bad, ps, seq, pos, slot) is False
    assert rows(cu, p0 + P * ps, table, ps, seq, pos, slot) is False     # (past the table)
    for args in ((cu[:-1], p0, table, ps, seq, pos, slot), (cu, p0, table, 0, seq, pos, slot), (cu, p0, table, ps, seq[1:], pos, slot),
                 (cu, p0, table, ps, seq, pos, slot.astype(np.int64)), (cu[::-1].copy(), p0, table, ps, seq, pos, slot), (cu, p0 - 200, table, ps, seq, pos, slot)):
        with pytest.raises(ValueError):
            rows(*args)
