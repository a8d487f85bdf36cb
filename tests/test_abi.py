"""The C-ABI library loads and exports every symbol include/mkgpu.h declares
(no compute calls: runs without a GPU)."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "mkgpu.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(mk_[a-z0-9_]+)\s*\(", txt)))


def test_header_declares_symbols():
    syms = declared_symbols()
    assert "mk_map2tod_f32" in syms and "mk_t2m_plan_create" in syms
    assert len(syms) >= 20


def test_library_exports_every_declared_symbol():
    from minkasi_amd.lib import mkgpu
    missing = [s for s in declared_symbols() if not hasattr(mkgpu.lib, s)]
    assert not missing, missing
    assert mkgpu.lib.mk_version() >= 1
    assert mkgpu.lib.mk_reduce_workspace_bytes() > 0


def test_bindings_cover_header():
    from minkasi_amd.lib import mkgpu
    missing = [s for s in declared_symbols() if s not in mkgpu._SIGS]
    assert not missing, missing


def test_workspace_of_the_largest_call_serves_the_others():
    """Workspace sizes of the split sums never fall as a size grows."""
    from minkasi_amd.lib import mkgpu
    lib = mkgpu.lib
    ns = sorted({8192 * k + d for k in (1, 2, 15, 16, 51, 52, 63, 64, 127, 128, 255, 256, 511, 512, 513) for d in (-1, 0, 1)}
                | {1, 2, 1023, 1025, 2049, 4097, 1 << 23})
    ms = [1, 2, 8, 9, 63, 64, 65, 128, 129, 215, 511, 512, 513, 700, 1024]
    for size in (lambda n, m: lib.mk_gram_workspace_bytes(m, n), lambda n, m: lib.mk_cross_workspace_bytes(m, 5, n),
                 lambda n, m: lib.mk_cross_workspace_bytes(65, m, n),
                 lambda n, m: lib.mk_design_dots_workspace_bytes(n, 6, m)):
        for m in ms:
            got = [size(n, m) for n in ns]
            assert got == sorted(got), m
        for n in ns:
            got = [size(n, m) for m in ms]
            assert got == sorted(got), n
