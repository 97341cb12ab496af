"""The kernels of a filter step keep their values in registers and LDS: private
(scratch) memory is device memory, and a kernel that stages a chunk's loads
there moves every value three times.  Read from the metadata of the code
objects in the built library."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from sdft_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _private_bytes():
    raw = open(build.lib_path(), "rb").read()
    out = {}
    p = raw.find(MAGIC)
    while p >= 0:
        q = p + 32
        for _ in range(struct.unpack_from("<Q", raw, p + 24)[0]):
            off, size, nid = struct.unpack_from("<QQQ", raw, q)
            if size and build.ARCH.encode() in raw[q + 24:q + 24 + nid]:
                with tempfile.NamedTemporaryFile(suffix=".co") as f:
                    f.write(raw[p + off:p + off + size])
                    f.flush()
                    notes = subprocess.run([READELF, "--notes", f.name], capture_output=True,
                                           text=True, check=True).stdout
                for k in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
                    name = re.search(r"\.name:\s+(\S+)", k).group(1)
                    out[name] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)",
                                              k).group(1))
            q += 24 + nid
        p = raw.find(MAGIC, p + 1)
    return out


@pytest.mark.skipif(not os.path.exists(READELF) or not os.path.exists(build.lib_path()),
                    reason="library not built, or no llvm-readelf")
def test_step_kernels_use_no_private_memory():
    sizes = _private_bytes()
    step = {k: v for k, v in sizes.items()
            if re.search(r"k_(contract|expand|wplane|kb_|nl_reduce|noise_plane)", k)}
    assert len(step) >= 100
    assert {k: v for k, v in step.items() if v} == {}
