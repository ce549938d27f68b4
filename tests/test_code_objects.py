"""The built device code calls no function: every kernel is one inlined body.  A device function the
compiler leaves out of line returns through s[30:31], and where its code is longer than a branch
reaches, the compiler's long branches overwrote that pair (the mixed-type 256 x 256 GEMM never
returned); out of line its uniform operands also came back from memory as vector values."""
import struct

from gguf_hip import _lib


def _code_objects(blob):
    """The AMDGPU ELF images embedded in a library built by hipcc (uncompressed bundles)."""
    at = blob.find(b"\x7fELF", 4)
    while at >= 0:
        if blob[at + 4] == 2 and struct.unpack_from("<H", blob, at + 18)[0] == 224:
            yield blob[at:]
        at = blob.find(b"\x7fELF", at + 4)


def _symbols(elf):
    """(name, type) of every symbol of an ELF image's symbol tables."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    size, n = struct.unpack_from("<HH", elf, 58)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * size) for i in range(n)]
    for s in sections:
        if s[1] in (2, 11):   # SHT_SYMTAB, SHT_DYNSYM
            names = sections[s[6]]
            for i in range(s[5] // 24):
                name, info = struct.unpack_from("<IB", elf, s[4] + 24 * i)
                start = names[4] + name
                yield elf[start:elf.index(b"\0", start)].decode(), info & 15


def test_every_device_function_is_a_kernel():
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    kernels, functions = set(), set()
    for elf in _code_objects(blob):
        for name, kind in _symbols(elf):
            if name.endswith(".kd"):
                kernels.add(name[:-3])
            elif kind == 2:   # STT_FUNC
                functions.add(name)
    assert len(kernels) > 100
    assert not functions - kernels, sorted(functions - kernels)
