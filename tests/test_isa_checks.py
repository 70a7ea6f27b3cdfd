"""The two checks of xlstm_amd/isa_check.py: on small listings that show what they look for, and on the assembly the
compiler really makes of the kernels (no GPU needed: hipcc cross-compiles)."""
import os

from xlstm_amd import isa_check

HAZARD = """
_Z6kernelv:
	v_readlane_b32 s44, v83, 26
	v_mul_lo_u32 v62, v65, s0
	v_readlane_b32 s45, v83, 27
	;;#ASMSTART
	global_load_ubyte v68, v62, s[44:45]
	;;#ASMEND
	s_endpgm
"""

HAZARD_FIXED = HAZARD.replace("\tglobal_load_ubyte", "\ts_nop 4\n\tglobal_load_ubyte")

COPY_IN_FLIGHT = """
_Z6kernelv:
	;;#ASMSTART
	global_load_dwordx2 v[4:5], v60, s[2:3]
	;;#ASMEND
	v_mov_b64_e32 v[26:27], v[4:5]
	;;#ASMSTART
	s_waitcnt vmcnt(0)
	;;#ASMEND
	ds_write_b64 v67, v[26:27]
	s_endpgm
"""

COPY_AFTER_WAIT = """
_Z6kernelv:
	;;#ASMSTART
	global_load_dwordx2 v[4:5], v60, s[2:3]
	;;#ASMEND
	;;#ASMSTART
	global_load_dwordx2 v[6:7], v60, s[2:3]
	;;#ASMEND
	;;#ASMSTART
	s_waitcnt vmcnt(1)
	;;#ASMEND
	v_mov_b64_e32 v[26:27], v[4:5]
	s_endpgm
"""

TO_LDS = """
_Z6kernelv:
	;;#ASMSTART
	s_nop 4
	s_mov_b32 m0, s35
	s_nop 0
	buffer_load_dwordx4 v39, s[12:15], 0 offen lds
	;;#ASMEND
	v_mov_b32_e32 v39, 0
	s_endpgm
"""


def test_a_freshly_written_scalar_register_read_by_hand_issued_memory_instruction_is_found():
    assert len(isa_check.scalar_read_hazards(HAZARD)) == 2  # s44 (3 wait states behind) and s45 (1 behind)
    assert isa_check.scalar_read_hazards(HAZARD_FIXED) == []


def test_a_copy_of_a_register_with_a_hand_issued_load_in_flight_is_found():
    assert len(isa_check.inflight_register_uses(COPY_IN_FLIGHT)) == 1
    # vmcnt(1) with one younger load: the first load has landed, the second has not
    assert isa_check.inflight_register_uses(COPY_AFTER_WAIT) == []
    assert len(isa_check.inflight_register_uses(COPY_AFTER_WAIT.replace("v[26:27], v[4:5]", "v[26:27], v[6:7]"))) == 1
    # a load that goes straight to LDS has no destination register (v39 is its address)
    assert isa_check.inflight_register_uses(TO_LDS) == []


_LISTING = {}


def _compiled_listing(tmp_path):
    if "text" not in _LISTING:  # (one compilation for the tests of this file)
        _LISTING["text"] = isa_check.emit_assembly(os.path.join(tmp_path, "device.s"))
    return _LISTING["text"]


def test_the_kernels_as_compiled_have_neither(tmp_path):
    listing = _compiled_listing(tmp_path)
    assert listing.count("ASMSTART") > 50  # (the listing really is the kernels')
    assert isa_check.check(listing) == []


def test_the_backward_kernel_with_feeder_waves_keeps_its_registers_and_polls_with_scalar_offsets(tmp_path):
    """Two properties of slstm_bwd_split_kernel that its speed rests on and that only the assembly shows: the variants
    with feeder waves (twelve waves: 168 registers a lane) do not spill, and the polls of the exchange ring take their
    slot offset from a scalar register (with the offset in a vector register the compiler wraps every poll in a loop
    over the distinct values of the lanes)."""
    import re

    listing = _compiled_listing(tmp_path)
    meta = listing[listing.index("amdhsa.kernels:"):]
    seen = 0
    for entry in re.split(r"\n  - ", meta)[1:]:
        name = re.search(r"\.name:\s+(\S+)", entry)
        # (template arguments: bf16, S, feeder waves, gate deltas in bf16)
        if not name or not re.search(r"slstm_bwd_split_kernelILb[01]ELi\d+ELb1ELb[01]EEEvNS_14BwdSplitParamsE$", name.group(1)):
            continue
        seen += 1
        assert int(re.search(r"\.vgpr_count:\s*(\d+)", entry).group(1)) <= 168, name.group(1)
        assert int(re.search(r"\.private_segment_fixed_size:\s*(\d+)", entry).group(1)) == 0, name.group(1)
        body = listing[listing.index(name.group(1) + ":"):]
        body = body[: body.index(".end_amdhsa_kernel")].split("\n")
        polls = [i for i, line in enumerate(body) if "buffer_load_dwordx4" in line and "sc1" in line]
        assert polls, name.group(1)
        for i in polls:
            assert not any("v_readfirstlane" in line for line in body[max(0, i - 6): i]), (name.group(1), body[i - 6: i + 1])
    assert seen == 8  # bf16 at head dims 64, 128, 256 with the gate deltas in float32 and in bf16; float32 at 64, 128


def test_the_reverse_kernel_for_row_tiles_of_4_rows_publishes_behind_the_acknowledgement_of_what_it_rearmed(tmp_path):
    """The gradient waves of slstm_bwd_quad_kernel publish a step's deltas and re-arm the words of two steps ago with plain
    stores, and never load: without a wait between a re-arm and the next publication a peer that has seen the latter may poll
    re-armed words before they are there and take the deltas of four steps ago.  A publication is two stores of 8 bytes in
    one basic block; a wait for everything in flight has to stand in front of them in that block."""
    import re

    listing = _compiled_listing(tmp_path)
    kernels = re.findall(r"^(_Z\w*slstm_bwd_quad_kernelILi\d+ELi\d+ELb[01]E\w*):", listing, re.M)
    for name in kernels:
        body = listing[listing.index("\n" + name + ":"):]
        body = [line.strip() for line in body[: body.index(".end_amdhsa_kernel")].split("\n")]
        blocks, block = [], []
        for ins in body:
            if re.match(r"^\.LBB\w+:|^s_c?branch", ins):
                blocks.append(block)
                block = []
            elif _is_instruction(ins):
                block.append(ins)
        publications = [b for b in blocks if sum(i.startswith("global_store_dwordx2") for i in b) == 2]
        assert publications, name
        for b in publications:
            first = next(i for i, ins in enumerate(b) if ins.startswith("global_store_dwordx2"))
            assert any(re.match(r"s_waitcnt\b.*vmcnt\(0\)", ins) for ins in b[:first]), (name, b)
    assert len(kernels) == 12  # head dims 64, 128, 256; 32 and 64 units a workgroup; gate deltas in float32 and in bf16


def test_the_feeder_waves_of_that_kernel_wait_only_where_they_say_so(tmp_path):
    """The compiler sees one function, not roles: a load at the head of one role that it takes for pending where another role
    uses the register is waited for there, in the feeder waves' loop at the cost of a request's whole latency every step.
    In the loops that make requests every wait for memory is one written by hand (or that of a load in the loop itself)."""
    import re

    listing = _compiled_listing(tmp_path)
    kernels = re.findall(r"^(_Z\w*slstm_bwd_quad_kernelILi\d+ELi\d+ELb[01]E\w*):", listing, re.M)
    for name in kernels:
        body = listing[listing.index("\n" + name + ":"):]
        blocks, in_asm = [], False
        for line in body[: body.index(".end_amdhsa_kernel")].split("\n"):
            label = re.match(r"^\.L(BB\w+):(.*)", line)
            if label:
                blocks.append((label.group(1), label.group(2), []))
            elif line.lstrip().startswith("; ") and blocks and not blocks[-1][2]:  # (the loops around a block, over several lines)
                blocks[-1] = (blocks[-1][0], blocks[-1][1] + line, [])
            elif "ASMSTART" in line or "ASMEND" in line:
                in_asm = "ASMSTART" in line
            elif blocks and _is_instruction(line.strip()):
                blocks[-1][2].append((line.strip(), in_asm))
        loops = set()
        for label, where, code in blocks:
            if any(ins.startswith("buffer_load_ubyte") for ins, _ in code):
                loops.add(label if "Loop Header" in where else re.search(r"Header=(BB\w+)", where).group(1))
        assert len(loops) == 2, (name, loops)  # the requests in front of the first step, and those of the steps
        for label, where, code in blocks:
            if label in loops or any(re.search(r"(Header=|Parent Loop )%s\b" % loop, where) for loop in loops):
                for i, (ins, hand) in enumerate(code):
                    if ins.startswith("s_waitcnt") and "vmcnt" in ins and not hand:
                        assert i and re.match(r"(global|flat)_load", code[i - 1][0]), (name, label, ins)
    assert len(kernels) == 12


def _is_instruction(ins):
    return bool(ins) and not ins.startswith((";", ".")) and not ins.endswith(":")
