"""The CG kernels' reads of a system's state, from the source: a kernel whose
first workgroup records a system's end (k1_test stores `done`) must not branch on
the wavefronts' own plain reads of `done`, which may differ within a workgroup; nor
a kernel that writes `left` on its own reads of that."""
import os
import re

CG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tbsla_amd", "csrc",
                  "cg.hip")


def kernels():
    parts = re.split(r"^__global__ .*?\b(k_cg_\w+)\(", open(CG).read(), flags=re.M)
    # a kernel's text ends with the brace in the first column
    return {name: text.split("\n}\n")[0] for name, text in zip(parts[1::2], parts[2::2])}


def test_kernels_that_make_the_test_share_one_flag():
    found = kernels()
    makes = {name for name, text in found.items() if "k1_test(" in text}
    assert {"k_cg_spmv_p", "k_cg_pnew", "k_cg_spmv_dia"} <= makes
    for name in makes:
        assert "sg.done" not in found[name], name
        assert "seg_finish(" in found[name], name


def test_left_is_not_read_where_it_is_written():
    found = kernels()
    reads = {name for name, text in found.items() if "sg.left" in text}
    writes = {name for name, text in found.items() if "S->left" in text}
    assert reads == {"k_cg_pnew"}
    assert writes == {"k_cg_update", "k_cg_update_gdia", "k_cg_vcheck"}
