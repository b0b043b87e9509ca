"""The scan of test_isa_hazards.py over the kernel translation units that its list
does not name (the batch kernels of 8 waves, the reductions, the fixed-scratch
compress), and a check that the two lists together are all that the library is built from."""
import os

import pytest

from tests.test_isa_hazards import UNITS, B, _asm, sgpr_vmem_hazards

REST = [s for s in B.SOURCES if s.endswith(".hip") and s not in UNITS]


def test_lists_are_complete():
    assert {u for u in os.listdir(B.CSRC) if u.endswith(".hip")} == set(UNITS) | set(REST)


@pytest.mark.slow
def test_no_valu_sgpr_to_vmem_hazard_in_the_rest(tmp_path):
    if not os.path.exists(B.HIPCC):
        pytest.skip("hipcc not available")
    from concurrent.futures import ThreadPoolExecutor

    with ThreadPoolExecutor(max_workers=len(REST)) as ex:
        asms = list(ex.map(lambda u: _asm(u, tmp_path), REST))
    for unit, asm in zip(REST, asms):
        assert "global_store" in asm or "buffer_store" in asm, unit
        bad = sgpr_vmem_hazards(asm)
        assert not bad, (unit, bad[:5])
