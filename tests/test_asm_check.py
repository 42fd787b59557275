"""The build-time checker of hand-issued LDS reads (csrc/check_asm_reads.py) on small pieces of
assembly text: it must accept the intended pattern and flag each way the pattern can break."""
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_spec = importlib.util.spec_from_file_location("check_asm_reads", os.path.join(ROOT, "bfuse-project_amd", "csrc", "check_asm_reads.py"))
chk = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(chk)

READ_A = "\t;;#ASMSTART\n\tds_read_b128 v[20:23], v14 offset:0\n\t;;#ASMEND\n"
READ_B = "\t;;#ASMSTART\n\tds_read_b64 v[24:25], v15 offset:0x800\n\t;;#ASMEND\n"
WAIT = "\t;;#ASMSTART\n\ts_waitcnt lgkmcnt({n})\n\t;;#ASMEND\n"


def _run(tmp_path, body):
    p = tmp_path / "k.s"
    p.write_text("kern:\n" + body + "\ts_endpgm\n")
    return chk.check(str(p))


def test_the_intended_pattern_is_accepted(tmp_path):
    body = (READ_A + READ_B + "\tv_mfma_f32_16x16x4_f32 a[0:3], v2, v3, a[0:3]\n" + WAIT.format(n=1) +
            "\tv_mfma_f32_16x16x32_bf16 a[4:7], v[20:23], v[30:33], a[4:7]\n" + WAIT.format(n=0) +
            "\tv_mov_b32_e32 v40, v24\n")
    findings, n = _run(tmp_path, body)
    assert n == 2 and findings == []


def test_a_copy_before_the_wait_is_flagged(tmp_path):
    findings, _ = _run(tmp_path, READ_A + "\tv_mov_b32_e32 v40, v21\n" + WAIT.format(n=0))
    assert len(findings) == 1 and "names v21" in findings[0]


def test_a_spill_or_an_overwrite_before_the_wait_is_flagged(tmp_path):
    findings, _ = _run(tmp_path, READ_A + "\tscratch_store_dword off, v22, off offset:8\n" + WAIT.format(n=0))
    assert len(findings) == 1
    findings, _ = _run(tmp_path, READ_A + "\tv_add_u32_e32 v20, v1, v2\n" + WAIT.format(n=0))
    assert len(findings) == 1 and "names v20" in findings[0]
    findings, _ = _run(tmp_path, READ_A + "\tv_accvgpr_write_b32 a3, v23\n" + WAIT.format(n=0))
    assert len(findings) == 1


def test_a_partial_wait_retires_only_the_older_reads(tmp_path):
    # lgkmcnt(1) after two reads: the first has landed, the second has not
    findings, _ = _run(tmp_path, READ_A + READ_B + WAIT.format(n=1) + "\tv_mov_b32_e32 v40, v20\n" + WAIT.format(n=0))
    assert findings == []
    findings, _ = _run(tmp_path, READ_A + READ_B + WAIT.format(n=1) + "\tv_mov_b32_e32 v40, v25\n" + WAIT.format(n=0))
    assert len(findings) == 1 and "names v25" in findings[0]


def test_a_scalar_load_in_flight_at_a_partial_wait_is_flagged(tmp_path):
    findings, _ = _run(tmp_path, "\ts_load_dwordx2 s[4:5], s[0:1], 0x10\n" + READ_A + READ_B + WAIT.format(n=1) + WAIT.format(n=0))
    assert len(findings) == 1 and "scalar-memory load" in findings[0]
    # a full wait between them makes it sound
    findings, _ = _run(tmp_path, "\ts_load_dwordx2 s[4:5], s[0:1], 0x10\n\ts_waitcnt lgkmcnt(0)\n" + READ_A + READ_B + WAIT.format(n=1) + WAIT.format(n=0))
    assert findings == []


def test_reads_never_waited_for_and_reads_across_a_backward_branch_are_flagged(tmp_path):
    findings, _ = _run(tmp_path, READ_A)
    assert len(findings) == 1 and "never waited for" in findings[0]
    findings, _ = _run(tmp_path, ".LBB0_1:\n" + READ_A + "\ts_cbranch_scc1 .LBB0_1\n" + WAIT.format(n=0))
    assert len(findings) == 1 and "backward branch" in findings[0]


def test_a_loop_may_carry_reads_round_its_branch_in_the_registers_it_was_entered_with(tmp_path):
    use_a = WAIT.format(n=0) + "\tv_mfma_f32_16x16x32_bf16 a[4:7], v[20:23], v[30:33], a[4:7]\n"
    # software pipelining: the first read of the next step is in flight at the loop head, each time
    findings, _ = _run(tmp_path, READ_A + ".LBB0_1:\n" + use_a + READ_A + "\ts_cbranch_scc1 .LBB0_1\n" + use_a)
    assert findings == []
    # the branch is taken with the read in other registers than the loop head expects
    findings, _ = _run(tmp_path, READ_A + ".LBB0_1:\n" + use_a + READ_B + "\ts_cbranch_scc1 .LBB0_1\n" + use_a)
    assert len(findings) == 1 and "backward branch" in findings[0]
    # ... or with nothing in flight where the loop head was entered with a read
    findings, _ = _run(tmp_path, READ_A + ".LBB0_1:\n" + use_a + "\ts_cbranch_scc1 .LBB0_1\n")
    assert len(findings) == 1 and "backward branch" in findings[0]


def test_the_compilers_own_reads_are_not_tracked_but_take_a_counter_slot(tmp_path):
    # a compiler-issued ds_read after the asm read is the youngest: lgkmcnt(1) retires the asm read
    body = READ_A + "\tds_read_b32 v50, v51\n" + "\ts_waitcnt lgkmcnt(1)\n" + "\tv_mov_b32_e32 v40, v20\n" + "\ts_waitcnt lgkmcnt(0)\n"
    findings, n = _run(tmp_path, body)
    assert n == 1 and findings == []


LDS_LOAD = "\tbuffer_load_dwordx4 v5, s[0:3], 0 offen lds\n"
LOAD = "\tbuffer_load_dwordx4 v[8:11], v6, s[4:7], 0 offen\n"
WRITE = "\tds_write_b128 v0, v[42:45]\n"
LANDED = "\t;;#ASMSTART\n\ts_waitcnt vmcnt({n}) ; loads into LDS have landed\n\t;;#ASMEND\n"


def _lds(tmp_path, body):
    p = tmp_path / "k.s"
    p.write_text("kern:\n" + body + "\ts_endpgm\n.Lfunc_end0:\n")
    return chk.check_lds_loads(str(p))


def test_a_write_to_lds_with_a_load_into_it_in_flight_is_flagged(tmp_path):
    # what was found: a loop of one stage, whose last loads into LDS nothing waits for before the partial sums go there
    findings, n = _lds(tmp_path, LDS_LOAD + LOAD * 2 + LANDED.format(n=2) + LDS_LOAD * 2 + "\ts_waitcnt vmcnt(4)\n" + WRITE + "\ts_waitcnt vmcnt(0)\n")
    assert n == 3 and len(findings) == 1 and "ds_write_b128" in findings[0]
    findings, _ = _lds(tmp_path, LDS_LOAD + LOAD * 2 + LANDED.format(n=2) + LDS_LOAD * 2 + LANDED.format(n=0) + WRITE)
    assert findings == []
    # the compiler's own wait for a register load behind it is as good
    findings, _ = _lds(tmp_path, LDS_LOAD + LOAD + "\ts_waitcnt vmcnt(1)\n" + WRITE)
    assert findings == []


def test_a_wait_that_counts_loads_that_are_not_there_is_flagged(tmp_path):
    findings, _ = _lds(tmp_path, LDS_LOAD + LOAD + LANDED.format(n=2))
    assert len(findings) == 1 and "landed" in findings[0]


def test_loads_into_lds_are_followed_round_loops_and_over_branches(tmp_path):
    findings, _ = _lds(tmp_path, LDS_LOAD + LOAD * 2 + ".LBB0_1:\n" + LANDED.format(n=2) + LDS_LOAD + LOAD * 2 + "\ts_cbranch_scc1 .LBB0_1\n" + LANDED.format(n=0) + WRITE)
    assert findings == []
    # one load fewer behind it in the loop than in front of it
    findings, _ = _lds(tmp_path, LDS_LOAD + LOAD * 2 + ".LBB0_1:\n" + LANDED.format(n=2) + LDS_LOAD + LOAD + "\ts_cbranch_scc1 .LBB0_1\n" + LANDED.format(n=0) + WRITE)
    assert len(findings) == 1 and "landed" in findings[0]
    # a branch past the wait
    findings, _ = _lds(tmp_path, LDS_LOAD + "\ts_cbranch_scc1 .LBB0_2\n" + LANDED.format(n=0) + ".LBB0_2:\n" + WRITE)
    assert len(findings) == 1 and "ds_write_b128" in findings[0]
    # another side's code, which no such load leads to
    findings, _ = _lds(tmp_path, "\ts_cbranch_scc1 .LBB0_2\n" + LDS_LOAD + "\ts_endpgm\n.LBB0_2:\n" + WRITE)
    assert findings == []


def test_loads_into_lds_from_asm_are_their_kernels_own_affair_and_count_as_others(tmp_path):
    by_hand = "\t;;#ASMSTART\n\ts_mov_b32 m0, s5\n\ts_nop 0\n\tbuffer_load_dword v5, s[0:3], s4 offen lds\n\t;;#ASMEND\n"
    assert _lds(tmp_path, by_hand + WRITE) == ([], 0)
    findings, n = _lds(tmp_path, LDS_LOAD + by_hand * 2 + LANDED.format(n=2) + WRITE)
    assert (findings, n) == ([], 1)
    findings, _ = _lds(tmp_path, LDS_LOAD + by_hand + LANDED.format(n=2) + WRITE)
    assert len(findings) == 2


@pytest.mark.parametrize("k1,k2,form", [
    # loads into LDS from asm on one side, and LDS writes on the other, which the graph reaches past waits and lanes that do not go there
    ("bgemm_f32_1024x208x64x208", "conv1x1s2p0_f32_1024x128x28x28_256", "hfuse"), ("conv7x7s2p3_f32_1024x3x224x224_64", "conv1x1s2p0_f32_1024x128x28x28_256", "bfuse"),
    # ... and by the compiler
    ("gemm_f32_1024x768x2304", "conv1x1s2p0_f32_1024x128x28x28_256", "bfuse")])
def test_kernels_fused_later_pass(k1, k2, form, tmp_path):
    from bfuse_project_amd import build_pairs
    (tmp_path / "pairs_0.hip").write_text(build_pairs.source_text([{"k1": k1, "k2": k2, "form": form, "name": ""}]))
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-w", "-I", build_pairs.CSRC, str(tmp_path / "pairs_0.hip"), "-o", str(tmp_path / "pairs_0.s")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    assert chk.check(str(tmp_path / "pairs_0.s"))[0] == []
    findings, n = chk.check_lds_loads(str(tmp_path / "pairs_0.s"))
    assert findings == [] and (n > 0) == k1.startswith("gemm")


def test_the_built_kernels_pass(tmp_path):
    import glob
    files = glob.glob(os.path.join(ROOT, "bfuse-project_amd", "csrc", "obj", "kernels_*-gfx950.s"))
    if not files:
        pytest.skip("device assembly not present (library not built in this tree)")
    total = loads = 0
    for f in files:
        findings, n = chk.check(f)
        more, m = chk.check_lds_loads(f)
        assert findings + more == [], (findings + more)[:3]
        total, loads = total + n, loads + m
    assert total > 1000          # the GEMMs' hand-issued reads were found and followed
    assert loads > 100           # ... and the loads into LDS
