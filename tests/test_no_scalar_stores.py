"""Static check (CPU only) of the built gfx950 code objects: what their kernels may do through the scalar data cache,
and which instructions may write memory. Scalar memory instructions are told by their encoding (bits 31-26 of the
first word 110000, the SMEM format) and must be loads or clock reads, nothing else of that format; every store and
atomic must be a vector-memory or LDS instruction."""
import re
import subprocess

import pytest

from .test_code_objects import UNITS, _co, _tool

_SMEM_ALLOWED = re.compile(r"s_(load_dword(x2|x4|x8|x16)?|buffer_load_dword(x2|x4|x8|x16)?|memtime|memrealtime)$")
_WRITE_ALLOWED = re.compile(r"(global|buffer|flat|scratch|ds)_")
_LINE = re.compile(r"^\s+([a-z]\w*)(?:\s[^/]*)?//\s*[0-9A-F]+:\s*([0-9A-F]{8})", re.M)


def refused(disasm):
    """Instructions of a disassembly that are not on the lists."""
    bad = set()
    for name, word in _LINE.findall(disasm):
        if int(word, 16) >> 26 == 0b110000:
            if not _SMEM_ALLOWED.match(name):
                bad.add(name)
        elif re.search(r"store|atomic", name) and not _WRITE_ALLOWED.match(name):
            bad.add(name)
    return bad


def test_pattern_matches_planted_lines():
    planted = ("\ts_load_dwordx2 s[0:1], s[2:3], 0x0                       // 000000001000: C0060001 00000000\n"
               "\ts_unlisted s1, s[2:3], 0x0                               // 000000001008: C0420041 00000000\n"
               "\tglobal_store_dword v0, v1, s[0:1]                        // 000000001010: DC708000 00000100\n"
               "\tv_unlisted_atomic v0, v1                                 // 000000001018: 7E000301\n"
               "\ts_endpgm                                                 // 000000001020: BF810000\n")
    assert refused(planted) == {"s_unlisted", "v_unlisted_atomic"}


@pytest.mark.parametrize("unit", UNITS)
def test_no_scalar_cache_writes(unit):
    out = subprocess.run([_tool("llvm-objdump"), "-d", "--mcpu=gfx950", str(_co(unit))], capture_output=True,
                         text=True, check=True).stdout
    assert "s_endpgm" in out
    lines = _LINE.findall(out)
    assert sum(n.startswith(("global_store", "buffer_store", "flat_store")) for n, _ in lines) > 0 or unit == "calib"
    hits = refused(out)
    assert not hits, f"{unit}: {sorted(hits)}"
