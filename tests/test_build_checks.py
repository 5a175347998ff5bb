"""The checks triton-mla_amd/build.py runs on every build, on planted inputs:
the resource-report parser and its scratch/LDS gate, and the scans for the
hazards of inline asm. (The real build runs them on the shipped code; here each
must catch what it is for.)"""

import os
import re
import subprocess
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-mla_amd"))
import asm_checks  # noqa: E402
import build  # noqa: E402

REMARKS = """\
remark: /x/mla_decode.hip:717:0: Function Name: _ZN4tmla18mla_partial_kernelILi0ELi512ELi64ELi1ELb1ELb1ELb0EEEvNS_11PartialArgsE [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     VGPRs: 256 [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     AGPRs: 130 [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     ScratchSize [bytes/lane]: 0 [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     Dynamic Stack: False [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     LDS Size [bytes/block]: 148544 [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0: Function Name: _ZN4tmla18mla_partial_kernelILi0ELi512ELi64ELi4ELb1ELb1ELb1EEEvNS_11PartialArgsE [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     ScratchSize [bytes/lane]: 12 [-Rpass-analysis=kernel-resource-usage]
remark: /x/mla_decode.hip:717:0:     LDS Size [bytes/block]: 160832 [-Rpass-analysis=kernel-resource-usage]
"""


def test_resource_report_parsed():
    usage = build.parse_resource_usage(REMARKS)
    assert len(usage) == 2
    k1 = next(k for k in usage if "ELi1ELb1ELb1ELb0E" in k)
    assert usage[k1] == {"VGPRs": 256, "AGPRs": 130, "ScratchSize": 0, "LDS Size": 148544}
    build.check_resources(usage)  # the fp8 ring's 12 bytes are within its allowance


@pytest.mark.parametrize("edit, why", [
    (("ScratchSize [bytes/lane]: 0", "ScratchSize [bytes/lane]: 4"), "scratch"),
    (("ScratchSize [bytes/lane]: 12", "ScratchSize [bytes/lane]: 16"), "scratch"),
    (("148544", "163844"), "LDS"),
])
def test_resource_gate_fails(edit, why):
    usage = build.parse_resource_usage(REMARKS.replace(*edit))
    with pytest.raises(RuntimeError, match=why):
        build.check_resources(usage)


def _asm(tmp_path, body):
    p = tmp_path / "k.s"
    p.write_text("_Zkernel:\n" + body)
    return str(p)


def test_mfma_hazard_scan(tmp_path):
    mfma = "\tv_mfma_f32_32x32x16_bf16 v[0:15], v[32:35], v[36:39], v[0:15]\n"
    filler = "".join(f"\tv_add_u32_e32 v{100 + i}, v{101 + i}, v{102 + i}\n" for i in range(17))
    early = "\tv_max_f32_e32 v40, v3, v40\n"
    # read one instruction after the MFMA: flagged
    assert len(build.mfma_result_hazards(_asm(tmp_path, mfma + early))) == 1
    # 17 independent instructions are still too few; 18 (or s_nop wait states) suffice
    assert len(build.mfma_result_hazards(_asm(tmp_path, mfma + filler + early))) == 1
    assert build.mfma_result_hazards(_asm(tmp_path, mfma + filler + "\ts_nop 0\n" + early)) == []
    assert build.mfma_result_hazards(_asm(tmp_path, mfma + "\ts_nop 7\n\ts_nop 7\n\ts_nop 1\n" + early)) == []
    # a register-allocator copy of the accumulator in flight: flagged
    assert len(build.mfma_result_hazards(_asm(tmp_path, mfma + "\tv_mov_b32_e32 v60, v7\n"))) == 1
    # back-to-back accumulation into the same registers: the hardware's case
    assert build.mfma_result_hazards(_asm(tmp_path, mfma + mfma)) == []
    # an MFMA that reads the in-flight result as an A/B operand: flagged
    bad_ab = "\tv_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[36:39], v[16:31]\n"
    assert len(build.mfma_result_hazards(_asm(tmp_path, mfma + bad_ab))) == 1
    # MFMAs into AGPRs are the compiler's own (it inserts their waits)
    agpr = "\tv_mfma_f32_32x32x16_bf16 a[0:15], v[32:35], v[36:39], a[0:15]\n"
    assert build.mfma_result_hazards(_asm(tmp_path, agpr + "\tv_mov_b32_e32 v60, v7\n")) == []


def _in_asm(body):
    return "\t;;#ASMSTART\n" + body + "\t;;#ASMEND\n"


def test_mfma_result_scan_follows_branches(tmp_path):
    mfma = "\tv_mfma_f32_32x32x16_bf16 v[0:15], v[32:35], v[36:39], v[0:15]\n"
    early = "\tv_max_f32_e32 v40, v3, v40\n"
    # one path to the read comes straight from the MFMA, the other waits
    body = ("\ts_cbranch_scc0 .LBB0_2\n.LBB0_1:\n" + mfma + "\ts_branch .LBB0_3\n.LBB0_2:\n\ts_nop 7\n.LBB0_3:\n" +
            early + "\ts_endpgm\n")
    assert len(build.mfma_result_hazards(_asm(tmp_path, body))) == 1
    # around a loop: the MFMA at the end of one turn, the read at the start of the next
    body = ".LBB0_1:\n" + early + mfma + "\ts_cbranch_scc1 .LBB0_1\n\ts_endpgm\n"
    assert len(build.mfma_result_hazards(_asm(tmp_path, body))) == 1
    # an AGPR result of an inline-asm MFMA is nobody else's to wait for
    agpr = "\tv_mfma_f32_32x32x16_bf16 a[0:15], v[32:35], v[36:39], a[0:15]\n"
    read = "\tv_accvgpr_read_b32 v60, a7\n"
    assert len(build.mfma_result_hazards(_asm(tmp_path, _in_asm(agpr) + read))) == 1
    assert build.mfma_result_hazards(_asm(tmp_path, agpr + read)) == []


def test_operand_scan(tmp_path):
    mfma = _in_asm("\tv_mfma_f32_32x32x16_bf16 v[2:17], v[222:225], v[22:25], v[2:17]\n")
    back = "\tv_accvgpr_read_b32 v24, a132\n"
    other = "\tv_add_u32_e32 v100, v101, v102\n"

    def hits(body):
        return len(build.operand_hazards(_asm(tmp_path, body + "\ts_endpgm\n")))

    # an operand brought back from an AGPR right before, or one instruction before
    assert hits(back + mfma) == 1 and hits(back + other + mfma) == 1
    assert hits(back + other + other + mfma) == 0 and hits(back + "\ts_nop 1\n" + mfma) == 0
    assert hits(back + "\ts_nop 0\n" + mfma) == 1
    # the accumulator is an operand too; reads of the registers and writes of others are not
    assert hits("\tv_mov_b32_e32 v5, 0\n" + mfma) == 1
    assert hits("\tv_add_u32_e32 v100, v24, v222\n" + mfma) == 0
    # the compiler's own MFMA, whose waits it inserts
    assert hits(back + mfma.replace("\t;;#ASMSTART\n", "")) == 0
    # before a branch, and in one of two predecessors
    assert hits(back + "\ts_cbranch_scc0 .LBB0_1\n" + other + ".LBB0_1:\n" + mfma) == 1
    # ... but not after a write in inline asm, which it does not see either
    own = mfma.replace("\t;;#ASMSTART\n", "")
    assert hits(_in_asm("\tv_accvgpr_read_b32 v24, a132\n") + own) == 1
    dpp = "\tv_add_u32_dpp v60, v61, v60 row_shr:1 row_mask:0xf bank_mask:0xf\n"
    swap = _in_asm("\tv_permlane16_swap_b32 v61, v62\n")
    assert hits(swap + dpp) == 1 and hits(swap + other + other + dpp) == 0
    assert hits("\tv_mov_b32_e32 v61, 0\n" + dpp) == 0
    # both registers of a swap are written
    assert hits("\tv_permlane32_swap_b32 v60, v223\n" + mfma) == 1


def test_inflight_load_scan(tmp_path):
    read = _in_asm("\tds_read_b128 v[54:57], v2 offset:0\n")
    more = _in_asm("\tds_read_b64_tr_b16 v[60:61], v3 offset:0\n")
    scalar = _in_asm("\ts_load_dword s30, s[98:99], 0x0\n")
    copy, scopy = "\tv_mov_b64_e32 v[70:71], v[56:57]\n", "\ts_mov_b32 s10, s30\n"

    def wait(n):
        return f"\ts_waitcnt lgkmcnt({n})\n"

    def hits(body):
        return len(build.inflight_touches(_asm(tmp_path, body + "\ts_endpgm\n")))

    # copied, overwritten (its value unused) or loaded again before it has arrived
    assert hits(read + copy) == 1 and hits(read + "\tv_mov_b32_e32 v55, 0\n") == 1 and hits(read + read) == 1
    assert hits(read + wait(0) + copy) == 0
    # a counted wait covers all but the newest reads and writes of LDS
    assert hits(read + more + wait(1) + copy) == 0 and hits(read + more + wait(2) + copy) == 1
    assert hits(read + "\tds_write_b32 v4, v5\n" + wait(1) + copy) == 0
    assert hits(more + read + wait(1) + copy) == 1
    # ... but a scalar load is covered by none but zero, and covers no LDS read
    assert hits(scalar + scopy) == 1 and hits(scalar + more + wait(1) + scopy) == 1
    assert hits(scalar + more + wait(0) + scopy) == 0 and hits(read + scalar + wait(1) + copy) == 1
    # a wait in one of two branches only, and around a loop
    branch = "\ts_cbranch_scc0 .LBB0_1\n" + wait(0) + ".LBB0_1:\n"
    assert hits(read + branch + copy) == 1 and hits(read + wait(0) + branch + copy) == 0
    assert hits(".LBB0_1:\n" + scopy + scalar + "\ts_cbranch_scc1 .LBB0_1\n") == 1
    # a wait for other counters; the compiler's own loads, which it waits for
    assert hits(read + "\ts_waitcnt vmcnt(0)\n" + copy) == 1
    assert hits("\tds_read_b128 v[54:57], v2\n" + copy) == 0


def test_inline_asm_mfmas_keep_their_distance(tmp_path):
    """Every inline-asm MFMA of the kernels starts with the two wait states an
    operand written by the vector ALU needs (but for the head-owner loop's,
    which the scan alone guards), and in compiled code they satisfy the scan."""
    csrc, bare = os.path.join(os.path.dirname(build.__file__), "csrc"), []
    for name in sorted(os.listdir(csrc)):
        with open(os.path.join(csrc, name)) as f:
            text = re.sub(r"//.*", "", f.read())
        for m in re.finditer(r"\basm(?: volatile)?\(\s*([^:]*v_mfma[^:]*):", text):
            if not m.group(1).startswith("TMLA_MFMA_GAP "):
                bare.append(re.findall(r"__forceinline__ \w+ (\w+)\(", text[:m.start()])[-1])
    assert sorted(bare) == ["own_mfma_acc", "own_mfma_acc", "own_mfma_first", "own_mfma_first"]

    probe = """
#include "cdna.h"
using namespace tmla;
__global__ void k(const i16x8* a, const i16x8* b, f32x16* o, short x) {
  f32x16 d = o[threadIdx.x];
  const i16x8 u = a[threadIdx.x] ^ (i16x8)x, v = b[threadIdx.x] ^ (i16x8)x;
  asm volatile(GAP "v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(u), "v"(v));
  asm volatile("s_nop 7\\n\\ts_nop 7\\n\\ts_nop 7" : "+v"(d));
  o[threadIdx.x] = d;
}
"""
    src = tmp_path / "probe.hip"
    src.write_text(probe)
    found = []
    for gap in ("", "TMLA_MFMA_GAP"):
        out = tmp_path / "probe.s"
        subprocess.run([build.hipcc()] + build.FLAGS + [f"-I{csrc}", f"-DGAP={gap}", "-S", "--cuda-device-only",
                                                        str(src), "-o", str(out)], check=True, capture_output=True)
        assert any(ins.asm and ins.op.startswith("v_mfma") for _, blocks in asm_checks.kernels(str(out))
                   for blk in blocks for ins in blk.ins)
        found.append(len(asm_checks.operand_hazards(str(out))))
    assert found[0] > 0 and found[1] == 0
