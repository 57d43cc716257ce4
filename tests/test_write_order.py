"""The cache and index-key writers do not touch the values of a token they skip (padding slot, slot past the cache, another
rank's slot): in the compiled code every exit of a skipped token comes before the first vector load."""
import os
import re
import subprocess

import pytest

from arcagi2_flashnext_dots3_amd import build


def exits_before_first_load(body):
    """Conditional branches to an s_endpgm before the kernel's first vector memory load."""
    ends = [i for i, l in enumerate(body) if "s_endpgm" in l]
    labels = {m[1] for m in (re.match(r"(\.LBB\w+):", l) for e in ends for l in body[max(0, e - 3):e]) if m}
    first = next(i for i, l in enumerate(body) if re.match(r"\s*(global|buffer|flat)_load", l))
    return sum(1 for l in body[:first] if re.match(r"\s*s_cbranch", l) and l.split()[1] in labels)


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_values_are_loaded_after_the_slot_is_accepted(tmp_path):
    out = tmp_path / "write.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, "spmla_write.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    text = out.read_text().split("\n")
    # past the batch, outside the cache; past the batch, padding, another rank's, past the store
    for kernel, exits in (("cache_write_kernel", 2), ("key_write_kernel", 4)):
        at = next(i for i, l in enumerate(text) if re.match(rf"_ZN5spmla2wr\d+{kernel}\S+:", l))
        body = text[at:next(i for i in range(at, len(text)) if ".Lfunc_end" in text[i])]
        assert exits_before_first_load(body) >= exits, kernel
