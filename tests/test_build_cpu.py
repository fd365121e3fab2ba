"""The build's resource check (flashmhf_amd/build.py): the hand-scheduled kernels must compile without private (scratch)
memory, the one known exception is named, and a compiler whose remarks can no longer be parsed must not pass silently."""
import os

import pytest

from flashmhf_amd import build


def _usage(extra=None, drop=None, scratch=None):
    names = []
    for dh in (64, 96, 128):
        names += [f"_ZN5mhffn16mhffn_fwd_kernelILi{dh}EEEvNS_7FwdArgsE", f"_ZN5mhffn21mhffn_bwd_dqdr_kernelILi{dh}EEEvNS_6DqArgsE"]
        names += [f"_ZN5mhffn23mhffn_bwd_dkdudv_kernelILi{dh}ELb{t}EEEvNS_6DwArgsE" for t in (0, 1)]
        for nt in (1, 2):
            for norm in (0, 1):
                names += [f"_ZN5mhffn21mhffn_gate_{d}_kernelILi{dh}ELi{nt}ELb{norm}EEEvNS_8GateArgsE" for d in ("fwd", "bwd")]
    u = {n: {"ScratchSize": "0", "VGPRs": "100"} for n in names if not (drop and drop in n)}
    for k, v in (scratch or {}).items():
        hit = [n for n in u if k in n]
        assert hit, k
        for n in hit:
            u[n]["ScratchSize"] = str(v)
    u.update(extra or {})
    return u


def test_clean_usage_passes_and_unrelated_kernels_may_spill():
    build.check_no_scratch(_usage(extra={"_ZN5mhffn12_GLOBAL__N_117dkdudv_f32_kernelENS0_7F32ArgsE": {"ScratchSize": "64"}}))


def test_a_spill_in_a_hand_scheduled_kernel_fails_the_build():
    for frag in ("mhffn_fwd_kernelILi128E", "mhffn_bwd_dqdr_kernelILi96E", "mhffn_bwd_dkdudv_kernelILi64ELb1E",
                 "mhffn_gate_bwd_kernelILi128ELi1ELb1E", "mhffn_gate_fwd_kernelILi96ELi2ELb0E"):
        with pytest.raises(RuntimeError, match="scratch"):
            build.check_no_scratch(_usage(scratch={frag: 8}))


def test_the_named_exception_is_the_only_one():
    build.check_no_scratch(_usage(scratch={"mhffn_gate_bwd_kernelILi128ELi2ELb1E": 452}))
    with pytest.raises(RuntimeError, match="scratch"):
        build.check_no_scratch(_usage(scratch={"mhffn_gate_bwd_kernelILi128ELi2ELb0E": 452}))


def test_missing_remarks_fail_instead_of_passing_vacuously():
    with pytest.raises(RuntimeError, match="expected resource-usage remarks"):
        build.check_no_scratch({})
    with pytest.raises(RuntimeError, match="mhffn_bwd_dkdudv_kernel"):
        build.check_no_scratch(_usage(drop="mhffn_bwd_dkdudv_kernelILi96ELb1E"))


def test_remark_parser_reads_hipcc_output():
    text = ("x.hip:1:1: remark: Function Name: _ZN5mhffn16mhffn_fwd_kernelILi128EEEvNS_7FwdArgsE [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     VGPRs: 239 [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     ScratchSize [bytes/lane]: 0 [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     Occupancy [waves/SIMD]: 1 [-Rpass-analysis=kernel-resource-usage]\n")
    u = build.parse_resource_usage(text)
    assert u == {"_ZN5mhffn16mhffn_fwd_kernelILi128EEEvNS_7FwdArgsE": {"VGPRs": "239", "ScratchSize": "0", "Occupancy": "1"}}


def test_the_committed_resource_listing_is_clean():
    """flashmhf_amd/_lib/resource_usage.txt is what the last build wrote: it must satisfy the same check."""
    path = os.path.join(build.LIBDIR, "resource_usage.txt")
    if not os.path.exists(path):
        pytest.skip("library not built")
    usage = {}
    for line in open(path):
        name, *fields = line.split("  ")
        usage[name] = dict(f.strip().split("=", 1) for f in fields if "=" in f)
    build.check_no_scratch(usage)


def _listing():
    path = os.path.join(build.LIBDIR, "resource_usage.txt")
    if not os.path.exists(path):
        pytest.skip("library not built")
    usage = {}
    for line in open(path):
        name, *fields = line.split("  ")
        usage[name] = dict(f.strip().split("=", 1) for f in fields if "=" in f)
    return usage


@pytest.mark.parametrize("frag,count", build.VARIANT_KERNELS)
def test_no_variant_and_no_float32_kernel_spills(frag, count):
    usage = _listing()
    build.check_variants(usage)
    found = [n for n in usage if frag in n]
    assert len(found) == count
    for n in found:
        with pytest.raises(RuntimeError, match="scratch"):
            build.check_variants({**usage, n: {**usage[n], "ScratchSize": "16"}})
        with pytest.raises(RuntimeError, match="scratch"):
            build.check_variants({k: v for k, v in usage.items() if k != n})


READ = """_Z6kernelv:
	ds_read_b32 v50, v50
	ds_read_b128 v[54:57], v186 offset:0x2000
	v_mov_b64_e32 v[60:61], v[62:63]
{}	;;#ASMSTART
	s_waitcnt lgkmcnt({})
	;;#ASMEND
	v_mov_b64_e32 v[52:53], v[50:51]
	v_add_f32_e32 v1, v2, v3
.Lfunc_end0:
	v_mov_b32_e32 v1, v54
"""


@pytest.mark.parametrize("between,left,found", [("", 0, False), ("", 1, False), ("", 2, True), ("\tv_mov_b64_e32 v[52:53], v[50:51]\n", 0, True),
                                                ("\tv_mov_b32_e32 v56, 0\n", 0, True), ("\ts_branch .LBB0_1\n", 2, False)])
def test_registers_of_reads_in_flight_are_found(between, left, found):
    got = build.reads_touched_in_flight(READ.format(between, left).splitlines())
    assert bool(got) is found and (not found or list(got) == ["_Z6kernelv"])


LOOP = """_Z6kernelv:
	ds_read_b32 v50, v1
	s_waitcnt lgkmcnt(0)
.LBB0_1:
	v_add_f32_e32 v2, v2, v{used}
	ds_read_b32 v50, v1
	{wait}
	s_cbranch_scc1 .LBB0_1
	s_waitcnt lgkmcnt(0)
	s_branch .LBB0_3
.LBB0_2:
	v_add_f32_e32 v2, v2, v50
	s_endpgm
.LBB0_3:
	ds_read_b32 v50, v1
	s_branch .LBB0_{target}
.LBB0_4:
	s_endpgm
.Lfunc_end0:
"""


@pytest.mark.parametrize("used,wait,target,found", [(50, "s_nop 0", 4, "v_add_f32_e32 v2, v2, v50"), (51, "s_nop 0", 4, "ds_read_b32 v50, v1"),
                                                    (50, "s_waitcnt lgkmcnt(0)", 4, None), (50, "s_waitcnt lgkmcnt(0)", 2, "v_add_f32_e32 v2, v2, v50")])
def test_reads_in_flight_are_followed_over_branches(used, wait, target, found):
    """Around a loop and through a jump, forwards and backwards in the text."""
    got = build.reads_touched_in_flight(LOOP.format(used=used, wait=wait, target=target).splitlines())
    assert got == ({} if found is None else {"_Z6kernelv": found})


def test_inline_assembly_leaves_m0_as_it_was():
    """The compiler keeps the LDS base of its own LDS-direct loads there, and takes no clobber of it."""
    import re
    found = 0
    for name in os.listdir(build.CSRC):
        for asm in re.findall(r'\basm\b[^"]*((?:"[^"]*"\s*)+)', open(os.path.join(build.CSRC, name)).read()):
            lines = [ln.strip(' "') for ln in re.sub(r'"\s*"', "", asm).strip().split("\\n\\t")]
            if any(ln.startswith("s_mov_b32 m0,") for ln in lines):
                found += 1
                assert lines[0] == "s_mov_b32 %0, m0" and lines[-1] == "s_mov_b32 m0, %0", (name, lines)
    assert found
