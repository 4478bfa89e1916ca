"""Kernels whose work items are short keep their values in registers: what the built library says of its kernels' scratch memory."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from llmengine.ops import build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels_of(path, folder):
    """{kernel: (bytes of scratch a lane, vector registers spilled)} from the code objects' own notes."""
    readelf = next((p for p in (shutil.which("llvm-readelf"), "/opt/rocm/llvm/bin/llvm-readelf") if p and os.access(p, os.X_OK)), None)
    if readelf is None:
        pytest.skip("no llvm-readelf")
    with open(path, "rb") as f:
        data = f.read()
    found = {}
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count if count < 16 else 0):
            offset, size, name_len = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + name_len]
            p += 24 + name_len
            if b"gfx950" not in name or size == 0:
                continue
            obj = os.path.join(folder, "object")
            with open(obj, "wb") as f:
                f.write(data[at + offset:at + offset + size])
            notes = subprocess.run([readelf, "--notes", obj], stdout=subprocess.PIPE, text=True, check=True).stdout
            for kernel in re.split(r"\n  - \.a", notes)[1:]:
                symbol = re.search(r"\n    \.name: +(\S+)", kernel).group(1)
                found[symbol] = tuple(int(re.search(key + r": +(\d+)", kernel).group(1))
                                      for key in (r"\.private_segment_fixed_size", r"\.vgpr_spill_count"))
        at = data.find(MAGIC, at + 1)
    return found


def test_prompt_attention_keeps_its_items_in_registers(tmp_path):
    """A step of a prompt portion beside decoded tokens has items of 20 stretches of keys and fewer: trips to scratch memory in front of them
    are part of every layer's time."""
    library = build.built_library()
    if library is None:
        pytest.skip("no built library")
    found = {k: v for k, v in kernels_of(library, str(tmp_path)).items() if "attention_prefill_shared_kernel" in k}
    assert len(found) == 24                                # two head sizes, rows, cut or not, three groupings of heads
    assert all(v == (0, 0) for v in found.values()), found
