"""Registers of the built kernels, from the notes that the compiler leaves in each code object of the library (amdhsa.kernels)."""
import re
import struct

import pytest

from lightron_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """{mangled name: its notes} of every gfx950 kernel in the built library."""
    data, found = open(_lib.LIB_PATH, "rb").read(), {}
    for m in re.finditer(b"\x7fELF\x02\x01", data):
        elf = memoryview(data)[m.start():]
        if struct.unpack_from("<H", elf, 18)[0] != 224:   # EM_AMDGPU
            continue
        at, = struct.unpack_from("<Q", elf, 40)
        size, count = struct.unpack_from("<HH", elf, 58)
        for i in range(count):
            kind, offset, length = struct.unpack_from("<4xI16xQQ", elf, at + i * size)
            if kind != 7:   # SHT_NOTE
                continue
            name, desc, note = struct.unpack_from("<III", elf, offset)
            if note == 32:   # NT_AMDGPU_METADATA
                start = offset + 12 + (name + 3) // 4 * 4
                found.update((k[".name"], k) for k in msgpack.unpackb(bytes(elf[start:start + desc]))["amdhsa.kernels"])
    return found


@pytest.mark.parametrize("kernel,like", [
    ("fwd_bf16_pad_kernelILi128ELi1E", "fwd_bf16_kernelILi128ELi1E"), ("fwd_bf16_pad_kernelILi128ELi2E", "fwd_bf16_shares_kernelILi128ELi2E"),
    ("fwd_bf16_pad_kernelILi128ELi4E", "fwd_bf16_shares_kernelILi128ELi4E"), ("bwd_dq_pad_kernelILi128ELi1E", "bwd_dq_kernelILi128ELi1E"),
    ("bwd_dq_pad_kernelILi128ELi2E", "bwd_dq_shares_kernelILi128ELi2E"), ("bwd_dq_pad_kernelILi128ELi4E", "bwd_dq_shares_kernelILi128ELi4E"),
    ("bwd_dkdv_pad_kernelILi128E", "bwd_dkdv_kernelILi128ELi1E"), ("bwd_joint_pad_kernelILi128ELi1E", "bwd_joint_kernelILi128ELi1E"),
    ("bwd_joint_pad_kernelILi128ELi2E", "bwd_joint_kernelILi128ELi2E"), ("bwd_joint_delta_pad_kernelILi128E", "bwd_joint_delta_kernelILi128E"),
])
def test_a_padded_kernel_of_width_128_holds_one_body(kernel, like):
    """Three and four blocks of columns are kernels of their own: each keeps about the scalars of the kernel without padding (up to 21 more are
    spilled; 19 - 84 more, and twice as many as either body has, with both bodies in one kernel) and no more than one vector register is spilled."""
    all_kernels = _kernels()
    mine, plain = ([k for n, k in all_kernels.items() if "%d%s" % (len(x.split("I")[0]), x) in n] for x in (kernel, like))
    assert len(mine) == 2 and len(plain) == 1
    for k in mine:
        assert k[".sgpr_spill_count"] <= plain[0][".sgpr_spill_count"] + 24 and k[".vgpr_spill_count"] <= 1, k[".name"]
