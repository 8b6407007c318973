"""The look over the assembly of a build for inline assembly that writes EXEC where some lanes may be off (rpeg_amd/exec_check.py):
short listings of the forms that branches and loops take.  CPU only."""

import pytest

from rpeg_amd.exec_check import exec_set_under_a_mask

MOVES = """	;;#ASMSTART
	s_mov_b64 exec, s[8:9]
	v_mov_b32 v1, v2
	s_mov_b64 exec, -1
	;;#ASMEND"""
OTHER = MOVES.replace("v1", "v3")

BRANCH = """	v_cmp_eq_u32_e64 s[2:3], 0, v0
	s_and_saveexec_b64 s[0:1], s[2:3]
	s_cbranch_execz .LBB0_2
	v_add_u32_e32 v1, 1, v1
{inside}
.LBB0_2:
{again}
	s_or_b64 exec, exec, s[0:1]
{behind}"""
BOTH_WAYS = """	s_and_saveexec_b64 s[0:1], vcc
	s_xor_b64 s[0:1], exec, s[0:1]
	s_cbranch_execz .LBB0_2
	v_add_u32_e32 v1, 1, v1
.LBB0_2:
	s_{back}_saveexec_b64 s[0:1], s[0:1]
	{flip}
	s_cbranch_execz .LBB0_4
	v_add_u32_e32 v1, 2, v1
{inside}
.LBB0_4:
	s_or_b64 exec, exec, s[0:1]
{behind}"""
LOOP = """	s_mov_b64 s[4:5], 0
.LBB0_1:
	v_cmp_eq_u32_e32 vcc, 0, v0
	s_and_saveexec_b64 s[6:7], s[2:3]
	v_add_u32_e32 v1, 1, v1
	s_or_b64 exec, exec, s[6:7]
{inside}
	s_or_b64 s[4:5], vcc, s[4:5]
	s_andn2_b64 exec, exec, s[4:5]
	s_cbranch_execnz .LBB0_1
	s_or_b64 exec, exec, s[4:5]
{behind}"""
SPILLED = """	s_mov_b64 s[0:1], exec
	s_and_b64 s[2:3], s[0:1], s[2:3]
	s_mov_b64 exec, s[2:3]
	v_writelane_b32 v9, s0, 4
	v_writelane_b32 v9, s1, 5
	s_mov_b64 s[0:1], 0
	v_readlane_b32 s6, v9, 4
	v_readlane_b32 s7, v9, {lane}
	s_or_b64 exec, exec, s[6:7]
{behind}"""


def found(text, *more):
    body = "k:                 ; @k\n; %bb.0:\n" + text + "\n\ts_endpgm\n"
    return exec_set_under_a_mask(body + "".join(more) + "\t.amdhsa_kernel k\n")


@pytest.mark.parametrize("text,wrong", [
    (MOVES, 0),
    (MOVES + "\n" + OTHER, 0),
    (BRANCH.format(inside="", again="", behind=MOVES), 0),
    (BRANCH.format(inside=MOVES, again="", behind=""), 1),
    (BRANCH.format(inside="", again=MOVES, behind=""), 1),                                   # ahead of what brings the lanes back
    (BRANCH.format(inside="\ts_mov_b64 s[0:1], 7", again="", behind=MOVES), 1),              # which a path has written meanwhile
    (BRANCH.format(inside="\tv_cmp_eq_u32_e64 s[0:1], 0, v1", again="", behind=MOVES), 1),
    (BRANCH.format(inside="\ts_branch .LBB0_9", again="", behind="") + "\n.LBB0_9:\n" + MOVES, 1),
    (BOTH_WAYS.format(back="andn2", flip="s_nop 0", inside="", behind=MOVES), 0),
    (BOTH_WAYS.format(back="andn2", flip="s_nop 0", inside=MOVES, behind=""), 1),
    (BOTH_WAYS.format(back="or", flip="s_xor_b64 exec, exec, s[0:1]", inside="", behind=MOVES), 0),
    (BOTH_WAYS.format(back="or", flip="s_xor_b64 exec, exec, s[0:1]", inside=MOVES, behind=""), 1),
    (LOOP.format(inside="", behind=MOVES), 0),
    (LOOP.format(inside=MOVES, behind=""), 1),                                               # from its second turn on
    (LOOP.format(inside="\ts_mov_b64 s[4:5], 0", behind=MOVES), 1),
    (SPILLED.format(lane=5, behind=MOVES), 0),
    (SPILLED.format(lane=4, behind=MOVES), 1),
    ("\tv_cmpx_eq_u32_e32 0, v0\n" + MOVES, 1),
    (MOVES.replace("\ts_mov_b64 exec, -1\n", ""), 1),                                       # leaves it as it is
    (BRANCH.format(inside=MOVES.replace("s_mov_b64 exec, s[8:9]", "s_nop 0").replace("s_mov_b64 exec, -1", "s_nop 0"), again="", behind=""), 0),
])
def test_where_lanes_may_be_off(text, wrong):
    assert found(text) == [("k", "s_mov_b64 exec, s[8:9]" if MOVES.splitlines()[1] in text else "v_mov_b32 v1, v2")] * wrong


CALL = """	s_getpc_b64 s[0:1]
	s_add_u32 s0, s0, f@rel32@lo+4
	s_addc_u32 s1, s1, f@rel32@hi+12
	s_swappc_b64 s[30:31], s[0:1]"""
FUNCTION = "f:\n" + MOVES + "\n\ts_setpc_b64 s[30:31]\n"


@pytest.mark.parametrize("text,wrong", [
    (CALL, 0),
    (CALL + "\n" + CALL + "\n" + MOVES, 0),
    (BRANCH.format(inside=CALL.replace("s[0:1]", "s[10:11]").replace("s0", "s10").replace("s1,", "s11,"), again="", behind=MOVES), 1),
    (CALL.replace("\ts_swappc_b64 s[30:31], s[0:1]", "\tv_mov_b32_e32 v0, s0"), 1),           # called from elsewhere
])
def test_a_function_is_entered_as_it_is_called(text, wrong):
    assert found(text, FUNCTION) == [("f", "s_mov_b64 exec, s[8:9]")] * wrong


def test_a_listing_without_kernels_is_refused():
    with pytest.raises(RuntimeError):
        exec_set_under_a_mask("k:\n\ts_endpgm\n")
