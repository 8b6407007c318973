"""The look over the assembly of a build (rpeg_amd/build.py): a 64-bit vector shift must not take its amount from the last
vector register of a kernel's allocation.  And over the inline assembly of the sources: what several instructions write may not share a
register with what they read.  CPU only."""

import re

import pytest

from rpeg_amd.build import HEADERS, SOURCES, shifts_by_last_register

LISTING = """
helper:                                 ; @helper
; %bb.0:
	s_waitcnt vmcnt(0) expcnt(0) lgkmcnt(0)
	{in_helper}
	s_setpc_b64 s[30:31]
leaf:
	s_setpc_b64 s[30:31]
k_one:                                  ; @k_one
	v_lshlrev_b64 v[2:3], 3, v[0:1]
	s_add_u32 s4, s4, leaf@rel32@lo+4
	{in_one}
	s_endpgm
k_two:
	s_getpc_b64 s[4:5]
	s_add_u32 s4, s4, {called}@rel32@lo+4
	s_addc_u32 s5, s5, {called}@rel32@hi+12
	v_lshl_add_u64 v[2:3], v[0:1], 2, v[62:63]
	s_endpgm
amdhsa.kernels:
  - .agpr_count:     0
    .name:           k_one
    .symbol:         k_one.kd
    .vgpr_count:     {n_one}
    .wavefront_size: 64
  - .agpr_count:     0
    .symbol:         'k_two.kd'
    .vgpr_count:     64
"""


@pytest.mark.parametrize("in_one,n_one,in_helper,called,want", [
    ("v_lshrrev_b64 v[4:5], v23, s[2:3]", 24, "s_nop 0", "leaf", ["k_one"]),
    ("v_ashrrev_i64 v[4:5], v23, v[6:7]", 24, "s_nop 0", "leaf", ["k_one"]),
    ("v_lshlrev_b64 v[4:5], v22, v[6:7]", 24, "s_nop 0", "leaf", []),          # another register
    ("v_lshlrev_b64 v[4:5], v23, v[6:7]", 26, "s_nop 0", "leaf", []),          # thirty-two allocated
    ("v_lshlrev_b64 v[4:5], v20, v[6:7]", 21, "s_nop 0", "leaf", []),          # twenty-four allocated
    ("v_lshlrev_b32 v4, v23, v6", 24, "s_nop 0", "leaf", []),
    ("s_nop 0", 24, "v_lshlrev_b64 v[4:5], v63, 1", "leaf", []),               # in a function that no such kernel calls
    ("s_nop 0", 24, "v_lshlrev_b64_e64 v[4:5], v63, 1", "helper", ["k_two"]),
])
def test_a_shift_by_the_last_register_is_found(in_one, n_one, in_helper, called, want):
    found = shifts_by_last_register(LISTING.format(in_one=in_one, n_one=n_one, in_helper=in_helper, called=called))
    assert [k for k, _, _ in found] == want and all("v_" in line for _, _, line in found)


def test_a_listing_without_kernels_is_refused():
    with pytest.raises(RuntimeError):
        shifts_by_last_register("k_one:\n\ts_endpgm\n")


def several_instructions(source):
    """(instructions, constraints of the outputs) of the inline assembly of a source that is more than one instruction."""
    for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", source):
        parts, depth, quoted, at = [""], 1, False, m.end()
        while depth:
            c = source[at]
            if c == '"' and source[at - 1] != "\\":
                quoted = not quoted
            if not quoted:
                depth += (c == "(") - (c == ")")
            if c == ":" and depth == 1 and not quoted:
                parts.append("")
            else:
                parts[-1] += c
            at += 1
        if "\\n" in parts[0] and len(parts) > 1:
            yield parts[0], re.findall(r'"([=+][^"]*)"', parts[1])


def test_outputs_of_several_instructions_share_no_register_with_inputs():
    """An operand that is written may be given the register of one that is read and has the same value, unless it is early-clobber:
    right only where nothing is read behind the first write."""
    seen = 0
    for path in SOURCES + HEADERS:
        with open(path) as f:
            for instructions, outputs in several_instructions(f.read()):
                seen += 1
                assert outputs and all("&" in x for x in outputs), (path, instructions, outputs)
    assert seen >= 15
    assert [x for _, x in several_instructions('asm("v_a %0, %1\\n\\tv_b %2" : "+v"(a), "=&v"(b[f(0)]) : "s"(m)); asm("v_c %0" : "=v"(d));')] == [["+v", "=&v"]]
