"""The wait states of the sources that issue instructions from inline assembly
(tests/wait_states.py), checked in the assembly their build makes of them."""
import subprocess

import pytest
import wait_states
from turboqwenfare_amd import build

SOURCES = ["tqf_grouped.hip", "tqf_stack.hip", "tqf_q6k.hip"]


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """The device assembly of SOURCES, by name (compiled side by side)."""
    out = tmp_path_factory.mktemp("asm")
    procs = {}
    for src in SOURCES:
        cmd = [build.hipcc_path(), *build.HIPCC_FLAGS, *build.EXTRA_FLAGS.get(src, []), "-w", "-S", "--cuda-device-only",
               str(build.CSRC / src), "-o", str(out / (src + ".s"))]
        procs[src] = subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    for src, p in procs.items():
        text, _ = p.communicate()
        assert p.returncode == 0, text.decode()
    return {src: (out / (src + ".s")).read_text() for src in SOURCES}


@pytest.mark.parametrize("src", SOURCES)
def test_no_use_comes_too_soon(assembly, src):
    assert wait_states.violations(assembly[src]) == []


# One function a rule, with the wait states it needs less one, then with them.
SHORT = {
    "sgpr": ["v_readfirstlane_b32 s4, v0", "buffer_load_dwordx4 v1, s[4:7], s8 offen lds"],
    "m0": ["s_mov_b32 m0, s3", "global_load_lds_dwordx4 v[2:3], off"],
    "dot": ["v_dot2_i32_i16 v4, v5, v6, 0", "v_add_u32_e32 v7, v4, v8"],
    "sdwa": ["v_mov_b32_sdwa v4, sext(v5) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0", "v_add_u32_e32 v7, v4, v8"],
}


@pytest.mark.parametrize("rule", SHORT)
def test_the_check_sees_each_rule(rule):
    first, second = SHORT[rule]
    need = wait_states.NEED[rule]

    def function(states, between=""):
        return "\n".join(["f:", first, between, *["s_waitcnt lgkmcnt(0)"] * states, second, "s_endpgm"])

    assert [v[1] for v in wait_states.violations(function(need - 1))] == [rule]
    assert wait_states.violations(function(need)) == []
    assert wait_states.violations(function(0, f"s_nop {need - 1}")) == []
    # over a branch the shortest path counts
    assert [v[1] for v in wait_states.violations(
        "\n".join(["f:", first, "s_cbranch_scc0 .LBB0_2", "s_nop 7", ".LBB0_2:", second, "s_endpgm"]))] == ([rule] if need > 1 else [])
