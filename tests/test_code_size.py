"""A layer's kernels stay in the instruction cache.

Two CUs share 64 KB of it, and a decoder token or a 4-frame encoder chunk
cycles through its layer's kernels at 3 to 12 us a launch: when their code did
not fit, the times changed by 2 to 4% with where the linker had put them.  The
kernels that a layer launches (at the 4B model's widths, whose launch shapes
launch_matvec and launch_gemm_kq pick) may take three quarters of it, whatever
else is built."""
import os
import re
import struct

import pytest

import vkv

ICACHE = 64 * 1024


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


def args(v):
    return "".join(f"L{'b' if isinstance(x, bool) else 'i'}{int(x)}E" for x in v)


def matvec(shape, kind):
    """k_matvec<steps, units in flight (2), all at once, no argmax, formats, norm, SwiGLU>"""
    return f"k_matvecI{args(shape + (False,))}({args(kind)})?EEv"


def gemm(waves, fmt, epilogue):
    """k_gemm_kq<waves, one column tile, input quantized inside, formats, epilogue>"""
    return f"k_gemm_kqI{args((waves, 1, True))}({args((fmt, epilogue))})?EEv"


DECODE = [r"k_decodeI\w*FmtF16\w*ELi4ELb1ELi4ELi2E", r"9k_combineE"]
WINDOW = [r"\d\dk_window_mfma_f32_64_splitE", r"k_window_mergeI"]
# Q/K/V, O, W1/W3, W2 and the attention
LAYERS = {
    "decoder, Q4_K and Q6_K": [matvec((1, 3, 2, True), (3, True, 0)), matvec((1, 3, 2, True), (0, False, 0)),
                               matvec((1, 4, 4, False), (0, True, 1)), matvec((3, 2, 2, False), (1, False, 0)),
                               *DECODE],
    "decoder, Q8_0": [matvec((1, 3, 2, True), (2, True, 0)), matvec((1, 6, 3, True), (2, False, 0)),
                      matvec((1, 4, 4, False), (2, True, 1)), matvec((3, 2, 2, False), (2, False, 0)), *DECODE],
    # (O and W2 in one kernel)
    "encoder chunk, Q8_0": [gemm(8, 2, 0), gemm(16, 2, 0), gemm(8, 2, 1), *WINDOW],
}


@pytest.mark.parametrize("layer", LAYERS)
def test_a_layers_kernels_fit_the_instruction_cache(layer):
    sizes = kernel_sizes(os.path.join(os.path.dirname(vkv.__file__), "libvkv.so"))
    found = {}
    for pattern in LAYERS[layer]:
        hits = {n: s for n, s in sizes.items() if re.search(pattern, n)}
        assert len(hits) == 1, (pattern, sorted(hits))
        found.update(hits)
    assert sum(found.values()) <= ICACHE * 3 // 4, found
