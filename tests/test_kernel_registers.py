"""No kernel of the library keeps registers in scratch memory: the tiles' heights and
widths are chosen by times that a spill would change.  From the built library's own
kernel metadata, without a device."""
import os
import re
import subprocess

import jev

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def kernels(tmp_path):
    data = open(jev.lib()._name, "rb").read()
    for i, part in enumerate(data.split(b"\x7fELF")[2:]):  # the library itself, then its code objects
        obj = os.path.join(tmp_path, "%d.elf" % i)
        with open(obj, "wb") as f:
            f.write(b"\x7fELF" + part)
        notes = subprocess.run([READELF, "--notes", obj], capture_output=True, text=True).stdout
        # a kernel's fields come in alphabetical order: its name, then its scratch bytes
        yield from re.findall(r"\.name: +(_Z\w+)\n +\.private_segment_fixed_size: (\d+)", notes)


def test_no_kernel_spills(tmp_path):
    got = {name: int(size) for name, size in kernels(tmp_path)}
    assert sum("gemm_bd_kernel" in k for k in got) > 30 and sum("attn_tree_kernel" in k for k in got) == 9
    assert not {k: v for k, v in got.items() if v}
