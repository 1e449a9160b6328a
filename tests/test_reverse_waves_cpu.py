"""The waves of one workgroup of the reverse step run different instantiations of
the tile (an edge band beside an inner one). A workgroup barrier inside it would
be met at different places by the waves of one group, so there is none."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reverse_tile_has_no_workgroup_barrier():
    src = open(os.path.join(ROOT, "cardiax_amd", "csrc", "fk_adjoint.h")).read()
    code = re.sub(r"//[^\n]*", "", src)
    body = code[code.index("void adj_tile("):code.index("void adj_tile_any(")]
    assert "pair_sum16(" in body
    for name in ("lds_barrier", "__syncthreads", "s_barrier"):
        assert name not in body, name
