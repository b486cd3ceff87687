"""Register use of the built kernels, as the compiler wrote it into the metadata of the library's gfx950 code objects."""
import re
import struct

import msgpack
import pytest

from turbodeberta_amd import _lib


def _sections(elf):
    at, size, count, names = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HHH", elf, 58)
    raw = [struct.unpack_from("<IIQQQQ", elf, at + i * size) for i in range(count)]
    return [(elf[raw[names][4] + s[0]:].split(b"\0", 1)[0], elf[s[4]:s[4] + s[5]]) for s in raw if s[1] != 8]


@pytest.fixture(scope="module")
def kernels():
    """Mangled name -> metadata of every kernel."""
    _lib.load()
    fat, found = dict(_sections(open(_lib.LIB_PATH, "rb").read()))[b".hip_fatbin"], {}
    for at in [m.start() for m in re.finditer(rb"\x7fELF", fat)]:
        note = dict(_sections(fat[at:])).get(b".note")
        if note:
            skip, size = struct.unpack_from("<II", note)
            skip = 12 + (skip + 3) // 4 * 4
            for k in msgpack.unpackb(note[skip:skip + size])["amdhsa.kernels"]:
                found[k[".name"]] = k
    return found


def test_persistent_kernel_keeps_its_arguments_out_of_the_key_steps(kernels):
    """The instances with tables once spilled whole blocks of arguments and reloaded them in every key step (84 to 126 scalar
    registers; the launches of long texts took 4 % longer).  What is left has to fit the lanes of one vector register."""
    table = {n: k for n, k in kernels.items() if re.search(r"attn_mfma_kernelIL.*Lb0EEEv15", n)}
    assert len(table) == 32
    spilled = {n: (k[".sgpr_spill_count"], k[".vgpr_spill_count"]) for n, k in table.items()}
    assert all(s <= 64 and v == 0 for s, v in spilled.values()), spilled
