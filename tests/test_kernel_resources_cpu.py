"""Resources of the compiled kernels, from the metadata of the code objects in
libvlbm.so: the box-map step kernels keep a node's populations in registers (a
spill shows as scratch memory and costs them several percent of a step), and the
LDS box of the sphere spreading is allowed for the LDS that its kernel holds beside
it."""
import re
import struct
import subprocess
from pathlib import Path

import msgpack
import pytest

from vlbm import _capi


CSRC = Path(__file__).resolve().parent.parent / "viscoplastic-lbm_amd" / "csrc"


def kernels():
    """Metadata of every kernel in the library by mangled name."""
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
                        out[kern[".name"]] = kern
                pos = desc + (descsz + 3) // 4 * 4
    return out


@pytest.mark.parametrize("q", [19, 27])
def test_box_map_population_steps_do_not_spill(q):
    step = {n: k[".private_segment_fixed_size"] for n, k in kernels().items() if re.match(rf"_ZN4vlbm6k_stepILi{q}E\w+?Li[012]ELb0ELb[01]ELb[01]ELi0ELi0E", n)}
    assert len(step) >= 24              # 4 storage types, 3 fluids, direct or not, with and without spheres
    assert not {n: s for n, s in step.items() if s}


def test_half_precision_row_pull_runs_six_waves():
    """Box-map D3Q19 steps of 16-bit storage: 512 registers a SIMD lane hold six waves of up to 80."""
    step = {n: k[".vgpr_count"] for n, k in kernels().items()
            if re.match(r"_ZN4vlbm6k_stepILi19E(DF16_|NS_4bf16E)Li[012]ELb0ELb0ELb0ELi0ELi0E", n)}
    assert len(step) == 12
    assert not {n: v for n, v in step.items() if v > 80}


def test_spreading_box_leaves_room_for_the_rest_of_the_kernel(tmp_path):
    (beside,) = [k[".group_segment_fixed_size"] for n, k in kernels().items() if "k_ibm_spread_box" in n]
    (tmp_path / "edges.cpp").write_text("""
#include <cstdio>
#include <initializer_list>
#include "ibm.h"
int main() {
    for (size_t lds : {size_t(32) << 10, size_t(64) << 10, size_t(96) << 10, size_t(160) << 10})
        for (int r = 1; r <= 12; r++) std::printf("%zu %d\\n", lds, vlbm::ibm_lds_box_edge(r, lds));
}
""")
    subprocess.run(["g++", "-std=c++17", "-D__host__=", "-D__device__=", "-D__forceinline__=inline", "-I", str(CSRC),
                    str(tmp_path / "edges.cpp"), "-o", str(tmp_path / "edges")], check=True)
    rows = [tuple(map(int, l.split())) for l in subprocess.run([str(tmp_path / "edges")], capture_output=True, text=True,
                                                               check=True).stdout.splitlines()]
    assert (160 << 10, 22) in rows           # spheres of radius 8 keep their box
    for lds, edge in rows:
        assert edge == 0 or 12 * edge ** 3 + beside <= lds, (lds, edge)
