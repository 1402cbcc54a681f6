"""The tile loads carry M0 from one assembly statement to the next (llm_simple_amd/csrc/check_m0.py): in the library as built
nothing else uses it, and a use by the compiler would be seen.  No GPU needed."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("check_m0", os.path.join(ROOT, "llm_simple_amd", "csrc", "check_m0.py"))
check_m0 = importlib.util.module_from_spec(spec)
spec.loader.exec_module(check_m0)


def test_library_as_built():
    uses, foreign = check_m0.check(os.path.join(ROOT, "llm_simple_amd", "libllmhip.so"))
    assert uses > 100 and not foreign


OWN = ["s_add_u32 m0, s4, 0x1000", "s_nop 0", "buffer_load_dwordx4 v1, s[4:7], 0 offen lds",
       "buffer_load_dwordx4 v2, s[4:7], 0 offen offset:1024 lds"]


@pytest.mark.parametrize("at,planted,seen", [(0, [], 0), (2, ["s_mov_b32 m0, s9", "s_nop 0", "global_load_lds_dwordx4 v[2:3], off"], 0),
                                             (3, ["s_mov_b32 m0, s9"], 1), (3, ["s_mov_b32 m0, -1", "s_nop 0"], 1),
                                             (3, ["s_mov_b32 m0, s9", "s_nop 0", "ds_gws_init v0 gds"], 1),
                                             (3, ["s_add_i32 m0, s9, 4", "s_nop 0"], 1), (3, ["v_readlane_b32 s3, v4, m0"], 1),
                                             (4, ["s_add_u32 m0, s9, 4"], 1)])
def test_a_foreign_use_is_seen(at, planted, seen):
    code = OWN[:at] + planted + OWN[at:]
    listing = "\n".join(["0000000000001000 <_Z18matmul_tile_kernelv>:"] + ["\t%s    // 000000001000: 00" % t for t in code]
                        + ["0000000000002000 <_Z12other_kernelv>:", "\ts_mov_b32 m0, s3"])
    uses, foreign = check_m0.foreign_uses(listing)
    assert len(foreign) == seen and uses >= 1
