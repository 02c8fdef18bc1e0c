"""The C ABI boundary without a GPU: the built library loads, exports every
function that include/iwhisper_amd.h declares, the ctypes binding matches the
header's argument counts, and argument validation reports errors through
iw_last_error() before any device work."""
import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "iwhisper_amd.h"


def _declarations():
    """name -> number of parameters, for every function the header declares."""
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    decls = {}
    for m in re.finditer(r"\b(?:int64_t|int|const char\s*\*)\s*(iw_\w+)\s*\(([^)]*)\)\s*;", text):
        params = m.group(2).strip()
        decls[m.group(1)] = 0 if params in ("", "void") else len(params.split(","))
    return decls


@pytest.fixture(scope="module")
def lib(iw):
    path = iw._lib.LIB_PATH
    if not path.exists():
        import __graft_entry__

        __graft_entry__._build_lib()
    return ctypes.CDLL(str(path))


def test_header_declares_the_api():
    decls = _declarations()
    assert len(decls) >= 29
    for name in ("iw_linear8", "iw_attention", "iw_attention_decode_cache", "iw_linear8_qkv_cache",
                 "iw_greedy_advance", "iw_last_error", "iw_abi_version"):
        assert name in decls


def test_library_exports_every_declared_function(lib):
    missing = [name for name in _declarations() if not hasattr(lib, name)]
    assert not missing, f"declared but not exported: {missing}"


def test_binding_matches_header(iw):
    decls = _declarations()
    sigs = dict(iw._lib.SIGNATURES)
    sigs.update({name: argtypes for name, (argtypes, _) in iw._lib.VALUE_FUNCS.items()})
    assert set(sigs) | {"iw_abi_version", "iw_last_error"} == set(decls)
    for name, argtypes in sigs.items():
        assert len(argtypes) == decls[name], name


def test_validation_errors_reach_iw_last_error(iw, lib):
    lib.iw_last_error.restype = ctypes.c_char_p
    fn = lib.iw_layernorm32
    fn.argtypes = iw._lib.SIGNATURES["iw_layernorm32"]
    fn.restype = ctypes.c_int
    # an unsupported width is rejected before any device call
    rc = fn(None, None, None, 1, 1, 1, 1, 13, None, 2, 100, False, None)
    assert rc != 0
    assert b"unsupported LayerNorm hidden size" in lib.iw_last_error()
    lib.iw_abi_version.restype = ctypes.c_int
    assert lib.iw_abi_version() == iw._lib.ABI_VERSION


def test_frag_bytes(iw):
    """Size of a fragment-major image: rows rounded up to 32, columns to 320."""
    v = iw._lib.value
    assert v("iw_frag_bytes", 128, 1280) == 128 * 1280
    assert v("iw_frag_bytes", 5, 384) == 32 * 640
    assert v("iw_frag_bytes", 33, 5120) == 64 * 5120
    assert v("iw_frag_bytes", 51865, 1280) == 51872 * 1280
    assert v("iw_frag_bytes", 1, 5121) == 0 and v("iw_frag_bytes", -1, 4) == 0


LLVM = Path("/opt/rocm/llvm/bin")


@pytest.fixture(scope="module")
def code_objects(lib, tmp_path_factory):
    """The gfx950 code objects of the built library."""
    if not (LLVM / "llvm-objdump").exists():
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(lib._name, d / "lib.so")
    subprocess.run([LLVM / "llvm-objdump", "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    return sorted(d.glob("*gfx950*"))


def test_lds_loads_keep_their_wait_state(code_objects):
    """A load into LDS takes its address from M0 and needs one wait state after a write of it. The
    compiler inserts none within inline assembly, so the built kernels are looked through."""
    loads, bad = 0, []
    for code in code_objects:
        out = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", code], check=True,
                             capture_output=True, text=True)
        before = ""
        for line in out.stdout.splitlines():
            op = line.split("//")[0].strip()
            if re.match(r"(global|buffer|scratch)_load_lds", op):
                loads += 1
                if re.match(r"s_\w+ m0\b", before):
                    bad.append(op)
            before = op
    assert loads > 0 and not bad


def test_decode_cache_attention_keeps_its_loads_in_registers(code_objects):
    """A spilled operand load waits for its data before the next one is issued."""
    spills = {}
    for code in code_objects:
        out = subprocess.run([LLVM / "llvm-readelf", "--notes", code], check=True, capture_output=True, text=True)
        for m in re.finditer(r"\.name: +(\S*attn_decode_cache_kernel\S*).*?\.vgpr_spill_count: (\d+)", out.stdout, re.S):
            spills[m[1]] = int(m[2])
    assert len(spills) >= 7 and not any(spills.values()), spills
