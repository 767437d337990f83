"""What the compiler makes of a kernel's waits, from the assembly of this
package's own sources (hipcc cross-compiles without a GPU)."""

import os
import re
import subprocess

import pytest

from mtplx_amd import build


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_tiles_loop_keeps_loads_in_flight(tmp_path):
    """The main loop of qmm_tiles_kernel waits for all but the newest ring
    slot (vmcnt(5)) twice, and nowhere for everything in flight."""
    out = tmp_path / "tiles.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, "qmm_tiles.hip"), "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    start = re.search(r"^_ZN3mtp16qmm_tiles_kernel\w*:", text, flags=re.M).end()
    kernel = text[start:text.index("s_endpgm", start)]
    header = re.search(r"^(\.LBB\w+):.*Loop Header", kernel, flags=re.M)
    last = kernel.rindex("Loop: Header")   # the loop's last block that is labelled so, and what follows to its end
    loop = kernel[header.end():kernel.index("\n.LBB", last) if "\n.LBB" in kernel[last:] else len(kernel)]
    waits = re.findall(r"s_waitcnt vmcnt\((\d+)\)", loop)
    assert waits == ["5", "5"]
