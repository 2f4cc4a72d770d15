"""What the compiler made of attention for many tiles: no form has scratch memory, and the forms without a mask, whose loop takes two blocks of keys a turn, keep every scalar in a
register.  Read from the metadata of the built library."""
import os
import re

import pytest

from tests import test_kernel_resources as built


def test_forms_without_a_mask_spill_nothing():
    if not os.path.exists(built.LIB):
        pytest.skip("no built library")
    # (type, LDS row, head size, probabilities in parts, causal, mask)
    found = [(k, m.group(1)) for k in built._kernels() for m in [re.search(r"fa_fwd_kernelI\w+?Li\d+ELi\d+ELb\dELb\dELb(\d)E", k[".name"])] if m]
    assert {m for _, m in found} == {"0", "1"}
    assert [k[".name"] for k, _ in found if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]] == []
    assert [(k[".name"], k[".sgpr_spill_count"]) for k, masked in found if masked == "0" and k[".sgpr_spill_count"]] == []


@pytest.mark.parametrize("name", ["attend_project_kernel", "attend_project_layer_kernel", "finish_norm_kernel"])
def test_short_prompts_spill_no_vector(name):
    if not os.path.exists(built.LIB):
        pytest.skip("no built library")
    found = [k for k in built._kernels() if name in k[".name"]]
    assert found
    assert [k[".name"] for k in found if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]] == []
