"""Resources of the compiled kernels, from the metadata of the code objects in
libvlbm.so: the box-map step kernels keep a node's populations in registers. A
spill shows as scratch memory and costs them several percent of a step."""
import re
import struct

import msgpack
import pytest

from vlbm import _capi


def kernels():
    """(mangled name, scratch bytes a lane) of every kernel in the library."""
    data = open(_capi.LIB_PATH, "rb").read()
    out = {}
    for m in re.finditer(rb"\x7fELF\x02\x01", data):
        base = m.start()
        if struct.unpack_from("<H", data, base + 18)[0] != 224:          # EM_AMDGPU
            continue
        phoff = struct.unpack_from("<Q", data, base + 32)[0]
        phentsize, phnum = struct.unpack_from("<HH", data, base + 54)
        for k in range(phnum):
            ph = base + phoff + k * phentsize
            if struct.unpack_from("<I", data, ph)[0] != 4:               # PT_NOTE
                continue
            off, size = struct.unpack_from("<Q", data, ph + 8)[0], struct.unpack_from("<Q", data, ph + 32)[0]
            pos, end = base + off, base + off + size
            while pos + 12 <= end:
                namesz, descsz, kind = struct.unpack_from("<III", data, pos)
                desc = pos + 12 + (namesz + 3) // 4 * 4
                if kind == 32:                                           # NT_AMDGPU_METADATA
                    meta = msgpack.unpackb(data[desc:desc + descsz], strict_map_key=False)
                    for kern in meta["amdhsa.kernels"]:
                        out[kern[".name"]] = kern[".private_segment_fixed_size"]
                pos = desc + (descsz + 3) // 4 * 4
    return out


@pytest.mark.parametrize("q", [19, 27])
def test_box_map_population_steps_do_not_spill(q):
    step = {n: s for n, s in kernels().items() if re.match(rf"_ZN4vlbm6k_stepILi{q}E\w+?Li[012]ELb0ELb[01]ELb[01]ELi0ELi0E", n)}
    assert len(step) >= 24              # 4 storage types, 3 fluids, direct or not, with and without spheres
    assert not {n: s for n, s in step.items() if s}
