"""Static check of the gfx950 code of every HIP source (CPU only): nothing
writes through the scalar data cache.  All device writes in this library are
vector stores (buffer/global); this keeps it that way.

It is an allow-list: every scalar mnemonic in the listing must be scalar
arithmetic, control flow or a wait, or, of those that touch memory, a load or a
clock read.  Anything else fails, known to this file or not, and so do raw
words in a function's body, which could encode an instruction.
"""
import os
import re
import shutil
import subprocess

import pytest

from fmha_native_amd import build

_SOURCES = sorted(f for f in os.listdir(build.CSRC) if f.endswith(".hip"))
_TYPE = r"(?:_[iub](?:8|16|32|64)){0,2}"
_ALLOWED = re.compile(
    r"s_(?:"
    r"(?:add|addc|addk|sub|subb|mul|mul_hi|mulk|min|max|abs|absdiff|and|or|xor|xnor|nand|nor|andn[12]|orn[12]|not|"
    r"lshl|lshr|ashr|lshl[1-4]_add|bfe|bfm|bcnt[01]|ff[01]|flbit|sext|brev|bitset[01]|bitcmp[01]|pack_[lh][lh]|mov|"
    r"movk|cmov|cmovk|cselect|cmpk?_(?:eq|lg|gt|ge|lt|le)|(?:and|or|xor|xnor|nand|nor|andn[12]|orn[12])_saveexec)" + _TYPE +
    r"|branch|cbranch_(?:scc[01]|vccn?z|execn?z)|endpgm|nop|waitcnt|barrier|setprio|sleep"
    r"|(?:load|buffer_load)_dword(?:x2|x4|x8|x16)?|memtime|memrealtime)")


def _device_asm(tmp_path, name):
    out = tmp_path / (name + ".s")
    cmd = [build.HIPCC, *[f for f in build.HIP_FLAGS if f != "-fPIC"], "--cuda-device-only", "-S",
           os.path.join(build.CSRC, name), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    return out.read_text()


def not_allowed(asm):
    """Scalar mnemonics outside the list, and data directives between a
    function's label and its end."""
    bad = {m for m in re.findall(r"^\s*(s_[a-z0-9_]+)", asm, re.M) if not _ALLOWED.fullmatch(m)}
    for name in re.findall(r"^\s*\.type\s+(\S+),@function", asm, re.M):
        start = re.search(r"^" + re.escape(name) + r":", asm, re.M).end()
        bad |= set(re.findall(r"^\s*(\.(?:byte|short|hword|long|word|int|quad|octa|ascii|string|fill|inst)\b)",
                              asm[start:asm.index(".Lfunc_end", start)], re.M))
    return sorted(bad)


@pytest.mark.parametrize("name", _SOURCES)
def test_no_scalar_cache_writes(tmp_path, name):
    if shutil.which(build.HIPCC) is None and not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not available")
    assert not_allowed(_device_asm(tmp_path, name)) == []


def test_every_built_source_is_checked():
    with open(build.__file__) as f:
        built = set(re.findall(r'"(\w+\.hip)"', f.read()))
    assert built and built <= set(_SOURCES)


def test_checker_flags_what_is_not_on_the_list():
    ok = "\ts_load_dwordx2 s[0:1], s[2:3], 0x0\n\ts_add_u32 s0, s1, s2\n\ts_and_saveexec_b64 s[0:1], vcc\n" \
         "\ts_cbranch_scc1 .LBB0_1\n\tbuffer_store_dwordx2 v[0:1], v2, s[4:7], 0 offen\n\tglobal_atomic_add v0, v1, s[0:1]\n"
    assert not_allowed(ok) == []
    for word in ("s_madeup_dword", "s_buffer_madeup_dwordx2", "s_load_madeup", "s_dword", "s_addx_u32", "s_mov_b3"):
        assert not_allowed(ok + f"\t{word} s0, s[2:3], 0x0\n") == [word]
    fn = "\t.type\tf,@function\nf:\n\ts_nop 0\n{}.Lfunc_end0:\n\t.long 1\n"
    assert not_allowed(fn.format("")) == []
    assert not_allowed(fn.format("\t.long 0xc0000000\n")) == [".long"]
