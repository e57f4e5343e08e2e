"""The compiled device code: kernels call no functions.

A helper that the compiler does not inline takes its register arrays through scratch memory and makes its caller save
the registers in use; a fused x pass with one such call site is slower by half."""
import os
import struct

import pytest

from tarang_amd import _lib


def _bundled(blob):
    """The gfx950 code objects of a host library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        n, p = struct.unpack_from("<Q", blob, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + length] and size:
                yield blob[at + off:at + off + size]
            p += 24 + length
        at += len(magic)


def _functions(elf):
    """Names of the functions and of the kernels (those with a descriptor) of a code object."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    functions, kernels = set(), set()
    for s in sections:
        if s[1] not in (2, 11):   # .symtab, .dynsym
            continue
        names = sections[s[6]][4]
        for o in range(s[4], s[4] + s[5], 24):
            name, info, _, section = struct.unpack_from("<IBBH", elf, o)
            text = elf[names + name:elf.index(b"\0", names + name)].decode()
            if text.endswith(".kd"):
                kernels.add(text[:-3])
            elif info & 15 == 2 and section:
                functions.add(text)
    return functions, kernels


def test_kernels_call_no_functions():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    kernels, called = set(), set()
    for elf in _bundled(blob):
        f, k = _functions(elf)
        kernels |= k
        called |= f - k
    assert any("k_x_mhd" in k for k in kernels) and any("k_x_nlin" in k for k in kernels)
    assert not called, sorted(called)[:8]
