"""A decoder layer's kernels stay in the instruction cache.

Two CUs share 64 KB of it, and a token cycles through its layer's kernels at 3
to 12 us a launch: when their code did not fit, the token's time changed by 4%
with where the linker had put them.  The kernels that a layer launches (the
widths of the 4B decoder, whose launch shapes launch_matvec picks) may take
three quarters of it, whatever else is built."""
import os
import re
import struct

import pytest

import vkv

ICACHE = 64 * 1024
ATTENTION = [r"k_decodeI\w*FmtF16\w*ELi4ELb1ELi4ELi2E", r"9k_combineE"]


def code_objects(path):
    """the gfx950 ELF images bundled in a library"""
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + ln]
            p += 24 + ln
            if b"gfx950" in name:
                yield data[at + off:at + off + size]
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def kernel_sizes(path):
    """mangled name -> bytes of code, from the images' symbol tables"""
    out = {}
    for elf in code_objects(path):
        shoff, = struct.unpack_from("<Q", elf, 40)
        shentsize, shnum = struct.unpack_from("<HH", elf, 58)
        sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
        for s in sections:
            if s[1] not in (2, 11):   # SHT_SYMTAB, SHT_DYNSYM
                continue
            names = sections[s[6]][4]
            for at in range(s[4], s[4] + s[5], 24):
                name, info, _, _, _, size = struct.unpack_from("<IBBHQQ", elf, at)
                if info & 15 == 2:    # STT_FUNC
                    end = elf.index(b"\0", names + name)
                    out[elf[names + name:end].decode()] = size
    return out


def matvec(shape, kind):
    """k_matvec<S, D4, D6, ONE, false, kind...>, or the shape's only kernel"""
    def args(v):
        return "".join(f"L{'b' if isinstance(x, bool) else 'i'}{int(x)}E" for x in v)
    return f"k_matvecI{args(shape + (False,))}({args(kind)})?EEv"


# (steps, units in flight, all at once), (formats, norm, SwiGLU): Q/K/V, O, W1/W3, W2
LAYERS = {
    "Q4_K and Q6_K": [((1, 3, 2, True), (3, True, 0)), ((1, 3, 2, True), (0, False, 0)),
                      ((1, 4, 4, False), (0, True, 1)), ((3, 2, 2, False), (1, False, 0))],
    "Q8_0": [((1, 3, 2, True), (2, True, 0)), ((1, 6, 3, True), (2, False, 0)),
             ((1, 4, 4, False), (2, True, 1)), ((3, 2, 2, False), (2, False, 0))],
}


@pytest.mark.parametrize("formats", LAYERS)
def test_a_decoder_layers_kernels_fit_the_instruction_cache(formats):
    sizes = kernel_sizes(os.path.join(os.path.dirname(vkv.__file__), "libvkv.so"))
    found = {}
    for pattern in [matvec(*k) for k in LAYERS[formats]] + ATTENTION:
        hits = {n: s for n, s in sizes.items() if re.search(pattern, n)}
        assert len(hits) == 1, (pattern, sorted(hits))
        found.update(hits)
    assert sum(found.values()) <= ICACHE * 3 // 4, found
