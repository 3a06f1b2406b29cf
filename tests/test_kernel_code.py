"""Device code of the built library (llvm-objdump of the gfx950 objects).

The small-set kernels in FP32 arithmetic read an LDS slot per pair and lane:
in 16-byte (or 12-byte) reads, not word by word, which costs bank conflicts
that outweigh the pair's arithmetic; and they run about one wave per SIMD, so
they never raise the wave priority around v_rsq_f32 (common.h: rsq_f32).
"""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LDS_BYTES = {"ds_read_b128": 16, "ds_read_b96": 12, "ds_read_b64": 8,
             "ds_read2_b64": 16, "ds_read_b32": 4, "ds_read2_b32": 8}


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Mangled kernel name -> its instructions, of every device object."""
    from tupan_amd import _native
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    tmp = tmp_path_factory.mktemp("code")
    lib = str(tmp / "lib.so")
    shutil.copy(_native.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True,
                   stdout=subprocess.DEVNULL)
    out = {}
    for f in sorted(os.listdir(str(tmp))):
        if not f.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn",
                               str(tmp / f)], check=True, text=True,
                              stdout=subprocess.PIPE).stdout
        cur = None
        for line in text.splitlines():
            m = re.match(r"^[0-9a-f]+ <(_Z\w+)>:", line)
            if m:
                cur = out.setdefault(m.group(1), [])
            elif cur is not None and line.startswith("\t"):
                cur.append(line.split()[0])
    return out


def test_fp32_small_set_kernels_read_whole_slots(kernels):
    names = [k for k in kernels
             if "small_kernel" in k and re.search("Fast32|OpSplit", k)]
    assert len(names) >= 13, names
    for k in names:
        ins = kernels[k]
        assert "s_setprio" not in ins, k
        read = {x: LDS_BYTES[x] * ins.count(x) for x in LDS_BYTES}
        narrow = read["ds_read_b32"] + read["ds_read2_b32"]
        wide = read["ds_read_b128"] + read["ds_read_b96"]
        # at most a third of the slot word by word (PNAcc's last words)
        assert wide >= 16 and narrow * 2 <= wide, (k, read)
