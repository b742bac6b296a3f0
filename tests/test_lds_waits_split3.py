"""The hand-counted LDS waits of the float32-accuracy kernels (csrc/split3.hip) and
the waits that must retire their global->LDS loads before each barrier, on the
compiled gfx950 assembly (tests/lds_waits.py)."""
import os
import re
import shutil

import pytest

from tests import lds_waits
from tests.test_lds_waits import _asm

pytestmark = pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")),
                                reason="hipcc not available")


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    return _asm("split3.hip", tmp_path_factory)


@pytest.mark.parametrize("stem", ["fwd_s3", "bwd_dq_s3", "bwd_dkdv_s3"])
def test_reads_and_dma_are_waited_for(asm, stem):
    names = sorted(set(re.findall(rf"^(_ZN5mattn\w*\d{stem}\w+):", asm, re.M)))
    assert len(names) == 7, names  # float32 at D = 64, 128, 256; bfloat16 and float16 at 256, two output dtypes
    for name in names:
        body = lds_waits.kernel_body(asm, name)
        reads, problems = lds_waits.check(body)
        assert reads > 20, (name, reads)
        assert not problems, (name, problems[:5])
        if "bf16" in name:  # bfloat16 rows go to LDS directly
            loads, problems = lds_waits.check_dma(body)
            assert loads >= 8, (name, loads)
            assert not problems, (name, problems[:5])
