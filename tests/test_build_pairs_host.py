"""build_pairs on the host: which fused kernels a suite lacks, the translation unit written for them, and the
registry's own spelling of the operator types (no GPU; the build step compiles the sample suite and the GPU tests run it,
here only the pairs of operators of more than 512 threads are compiled)."""
import os
import subprocess
from types import SimpleNamespace as NS

import pytest
import yaml

import bfuse_project_amd as bf
from bfuse_project_amd import build_pairs, configure

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _k(name, threads, barriers, kind=0):
    return NS(name=name, block=(threads, 1, 1), has_barriers=barriers, kind=kind)


def test_wanted_skips_what_the_registry_holds_and_writes_thread_fusion_only_where_it_fits():
    reg = {k.name: k for k in (_k("a", 256, True), _k("b", 64, False), _k("c", 256, True), _k("d", 896, False),
                               _k("a_b_fused_bfuse_c256", 256, True, kind=1))}
    lds = {"a": 70000, "b": 0, "c": 100000, "d": 0}.__getitem__
    got = build_pairs.wanted([("a", "b"), ("a", "c"), ("a", "d"), ("c", "b"), ("a", "b")], reg, "both", 256, lds)
    names = [k["name"] for k in got]
    assert names == ["a_b_fused_hfuse",                                   # block-fused a+b is already there
                     "a_c_fused_bfuse_c256",                              # both sides synchronise: no thread-level fusion
                     "a_d_fused_bfuse_c256",                              # 256 + 896 threads do not fit one workgroup
                     "c_b_fused_bfuse_c256", "c_b_fused_hfuse"]
    assert [k["name"] for k in build_pairs.wanted([("c", "b")], reg, "bfuse", 128, lds)] == ["c_b_fused_bfuse_c128"]
    assert [k["name"] for k in build_pairs.wanted([("c", "b")], reg, "bfuse", 256, lds, rt=True)] == ["c_b_fused_bfuse_c256", "c_b_fused_bfuse_rt"]
    # LDS: 100000 + 70000 bytes exceed a workgroup's 160 KB
    reg["e"] = _k("e", 64, False)
    assert [k["form"] for k in build_pairs.wanted([("c", "e")], reg, "both", 256, {"c": 100000, "e": 70000}.__getitem__)] == ["bfuse"]
    with pytest.raises(LookupError):
        build_pairs.wanted([("a", "zz")], reg)
    with pytest.raises(LookupError):
        build_pairs.wanted([("a", "a_b_fused_bfuse_c256")], reg)


def test_source_text_names_each_side_once_by_the_type_the_library_gives():
    todo = [{"k1": "a", "k2": "b", "form": "bfuse", "name": "a_b_fused_bfuse_c256"},
            {"k1": "a", "k2": "b", "form": "hfuse", "name": "a_b_fused_hfuse"},
            {"k1": "c", "k2": "b", "form": "bfuse", "name": "c_b_fused_bfuse_c256"},
            {"k1": "c", "k2": "b", "form": "rt", "name": "c_b_fused_bfuse_rt"}]
    text = build_pairs.source_text(todo, 256, {"a": "bfuse::A<1, 2>", "b": "bfuse::B<true>", "c": "bfuse::C<3>"}.__getitem__)
    lines = text.splitlines()
    assert lines.count("using Side0 = bfuse::A<1, 2>;   // a") == 1 and "using Side1 = bfuse::B<true>;   // b" in lines
    assert "BFUSE_BFUSE_KERNEL(a, Side0, b, Side1, _c256, bfuse::kChunked, 256, 1)" in lines
    assert "BFUSE_HFUSE_KERNEL(a, Side0, b, Side1)" in lines
    assert "BFUSE_BFUSE_KERNEL(c, Side2, b, Side1, _c256, bfuse::kChunked, 256, 1)" in lines
    assert "BFUSE_BFUSE_RT_KERNEL(c, Side2, b, Side1)" in lines
    assert [build_pairs._unit_kernel(l) for l in lines if l.startswith("BFUSE_")][-4:] == [k["name"] for k in todo]
    assert "BFUSE_MODULE_PROLOGUE()" in lines and '#include "fuse.h"' in lines
    for h in build_pairs.HEADERS:
        assert os.path.exists(os.path.join(build_pairs.CSRC, h))


def test_registry_spells_operator_types_and_their_lds():
    assert build_pairs.op_type("gemm_f32_512x768x2304") == "bfuse::GemmF32Dma<512, 2304, 768, 32, 144, 4>"
    assert build_pairs.op_type("conv3x3s1p1_f32_1024x448x8x8_384").startswith("bfuse::ConvF32Lds<448, 384, 8, 8, 3, 3, 1, 1,")
    assert build_pairs.op_type("conv1x1s1p0_f32_64x56x56_64") == "bfuse::SwapOperands<bfuse::GemmF32<64, 3136, 64, 16, 64, 1>>"
    assert build_pairs.op_lds("gemm_f32_512x768x2304") == 73728        # four waves x three stages of 6 KB
    assert build_pairs.op_lds("layernorm_512x768") >= 0
    with pytest.raises(LookupError):
        build_pairs.op_type("gemm_f32_512x768x2304_layernorm_512x768_fused_bfuse_r")    # a fused kernel has no operator type
    assert build_pairs.op_lds("no_such_kernel") == -1
    # every standalone kernel has a type that names a template of the library
    for k in bf.list_kernels():
        if k.kind == 0:
            assert build_pairs.op_type(k.name).startswith("bfuse::"), k.name


def test_sample_suite_lists_six_kernels_to_build(tmp_path):
    """The example the build step compiles: four pairs, none with a fused kernel in the library; both forms where
    thread-level fusion fits (the one-wave batched product beside a convolution), block fusion alone for the
    four-wave dense layer beside a four-wave convolution (both synchronise)."""
    out = tmp_path / "s"
    r = configure.configure(os.path.join(ROOT, "bfuse-project_amd", "examples", "batch_operators.yaml"), str(out))
    assert not r["missing"] and all(not v for v in r["fused"].values())
    b = build_pairs.build(str(out), compile_=False)
    assert sorted(k["form"] for k in b["kernels"]) == ["bfuse"] * 4 + ["hfuse"] * 2
    assert len(b["files"]) == 3 and all(os.path.exists(f) for f in b["files"])
    assert build_pairs.module_paths(str(out)) == []          # nothing compiled, nothing to load
    with pytest.raises(LookupError):
        build_pairs.build(str(out), only=["a+b"], compile_=False)
    with open(out / "config" / "modules.yaml", "w") as f:
        yaml.safe_dump(["hip/libbfuse_pairs.so"], f)
    assert build_pairs.module_paths(str(out)) == [os.path.join(str(out), "hip", "libbfuse_pairs.so")]


def test_units_written_for_another_tiling_of_an_operator_are_found(tmp_path):
    """A suite's translation units name each side by the operator type the library gave it when they were written;
    after a rebuild of the library with another tiling they are stale and must be written again."""
    d = tmp_path / "hip"
    d.mkdir()
    (d / "pairs_0.hip").write_text("using Side0 = bfuse::A<1>;   // a\nusing Side1 = bfuse::B<2>;   // b\nBFUSE_HFUSE_KERNEL(a, Side0, b, Side1)\n")
    (d / "pairs_1.hip").write_text("using Side0 = bfuse::A<1>;   // a\nBFUSE_HFUSE_KERNEL(a, Side0, a, Side0)\n")
    now = {"a": "bfuse::A<1>", "b": "bfuse::B<3>"}.__getitem__
    assert build_pairs.stale_units(str(d), now) == ["pairs_0.hip"]
    assert build_pairs.stale_units(str(d), {"a": "bfuse::A<1>", "b": "bfuse::B<2>"}.__getitem__) == []
    assert build_pairs.stale_units(str(tmp_path / "none")) == []


def test_kernels_that_spill_take_their_narrow_sides_and_are_left_out_only_then(tmp_path):
    d = tmp_path / "hip"
    d.mkdir()
    reg = {k.name: k for k in (_k("a", 640, True), _k("b", 256, False), _k("c", 768, True))}
    lines = ["using Side0 = bfuse::A<1, 2>;   // a", "BFUSE_BFUSE_KERNEL(a, Side0, b, Side1, _c256, bfuse::kChunked, 256, 1)", "BFUSE_BFUSE_RT_KERNEL(a, Side0, c, Side2)",
             "BFUSE_HFUSE_KERNEL(b, Side1, b, Side1)", "BFUSE_BFUSE_KERNEL(c, Side2, b, Side1, _c256, bfuse::kChunked, 256, 1)"]
    names = ["a_b_fused_bfuse_c256", "a_c_fused_bfuse_rt", "b_b_fused_hfuse"]
    (d / "pairs_0.hip").write_text("\n".join(lines) + "\n")
    (d / "pairs_0.res").write_text("".join(f"remark: Function Name: {n} [-R]\nremark:     ScratchSize [bytes/lane]: 8 [-R]\n" for n in names)
                                   + "remark: Function Name: c_b_fused_bfuse_c256 [-R]\nremark:     ScratchSize [bytes/lane]: 0 [-R]\n")
    assert build_pairs.narrow_spilling(str(d), reg) == names[:2]           # the third has no side of many waves
    got = (d / "pairs_0.hip").read_text().splitlines()
    assert got == [lines[0], "BFUSE_BFUSE_KERNEL(a, Narrow<Side0>, b, Side1, _c256, bfuse::kChunked, 256, 1)",
                   "BFUSE_BFUSE_RT_KERNEL(a, Narrow<Side0>, c, Narrow<Side2>)", lines[3], lines[4]]
    assert build_pairs.written(str(d)) == names + ["c_b_fused_bfuse_c256"]
    assert build_pairs.narrow_spilling(str(d), reg) == []                  # narrow already
    assert build_pairs.drop_spilling(str(d)) == names                      # spilled again: left out
    assert [l for l in (d / "pairs_0.hip").read_text().splitlines() if l.startswith("BFUSE_")] == [lines[4]]


def test_a_partner_short_of_registers_takes_its_slim_form_first(tmp_path):
    d = tmp_path / "hip"
    d.mkdir()
    reg = {k.name: k for k in (_k("a", 640, True), _k("b", 256, False), _k("c", 384, True))}
    lines = ["BFUSE_BFUSE_KERNEL(a, Side0, b, Side1, _c256, bfuse::kChunked, 256, 1)", "BFUSE_BFUSE_KERNEL(c, Side2, b, Side1, _c256, bfuse::kChunked, 256, 1)",
             "BFUSE_HFUSE_KERNEL(c, Side2, b, Side1)", "BFUSE_HFUSE_KERNEL(b, Side1, b, Side1)"]
    names = ["a_b_fused_bfuse_c256", "c_b_fused_bfuse_c256", "c_b_fused_hfuse", "b_b_fused_hfuse"]
    (d / "pairs_0.hip").write_text("\n".join(lines) + "\n")
    (d / "pairs_0.res").write_text("".join(f"remark: Function Name: {n} [-R]\nremark:     ScratchSize [bytes/lane]: 8 [-R]\n" for n in names))
    assert build_pairs.slim_spilling(str(d), reg) == [names[0], names[2]]           # nobody leaves the others less than 256
    want = ["BFUSE_BFUSE_KERNEL(a, Side0, b, Slim<Side1>, _c256, bfuse::kChunked, 256, 1)", lines[1], "BFUSE_HFUSE_KERNEL(c, Slim<Side2>, b, Slim<Side1>)", lines[3]]
    assert (d / "pairs_0.hip").read_text().splitlines() == want
    assert build_pairs.slim_spilling(str(d), reg) == []
    assert build_pairs.narrow_spilling(str(d), reg) == names[:1]                     # spilled again: 512 threads instead, and the partner as it was
    assert (d / "pairs_0.hip").read_text().splitlines()[0] == "BFUSE_BFUSE_KERNEL(a, Narrow<Side0>, b, Side1, _c256, bfuse::kChunked, 256, 1)"


def _suite_operators():
    out = set()
    for name in ("benchmark_batch1024", "inception_v3_batch1024", "interleave_scheduler_batch1024"):
        doc = configure.load_user_config(os.path.join(ROOT, "bfuse-project_amd", "examples", f"{name}.yaml"))
        out |= {k.name for k in configure.resolve(doc, {k.name: k for k in bf.list_kernels()}, None)[0].values()}
    return sorted(out)


def _compiled(k, src, tmp_path):
    (tmp_path / "pairs_0.hip").write_text(src)
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-device-only", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-Rpass-analysis=kernel-resource-usage", "-I", build_pairs.CSRC, "-c", str(tmp_path / "pairs_0.hip"), "-o", str(tmp_path / "pairs_0.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    assert f"Function Name: {k['name']}" in r.stderr
    return build_pairs.spilling_kernels(r.stderr)


@pytest.mark.parametrize("k1", ["conv3x3s1p1_f32_1024x32x147x147_64", "conv3x3s1p1_f32_1024x64x56x56_64"])
def test_patch_convolutions_fit_beside_ten_waves_in_their_slim_form(k1, tmp_path):
    """... whose own form of five (which the bf16 product does not have) they then do not need."""
    k = {"k1": k1, "k2": "gemm_bf16_512x4096x14336", "form": "bfuse", "name": f"{k1}_gemm_bf16_512x4096x14336_fused_bfuse_c256"}
    assert bf.operation.kernel_info(k["k2"]).block[0] > 512
    src = build_pairs.source_text([k]).replace("Side0, ", "Slim<Side0>, ") + "static_assert(Slim<Side0>::GRID.size() == Side0::GRID.size());\n"
    assert _compiled(k, src, tmp_path) == []


@pytest.mark.parametrize("form,k2", [("bfuse", "gemm_bf16_512x4096x14336"), ("hfuse", "conv1x1s1p0_f32_1024x768x17x17_160"), ("hfuse", "conv3x3s2p0_f32_1024x192x17x17_320")])
def test_rgb_layers_fit_beside_ten_waves_in_their_slim_form(form, k2, tmp_path):
    """Their own form takes 169 registers of the 168 that are left; with the products that have no form of fewer waves the pair would not be built."""
    k1 = "conv3x3s2p0_f32_1024x3x299x299_32"
    k = {"k1": k1, "k2": k2, "form": form, "name": f"{k1}_{k2}_fused_{'bfuse_c256' if form == 'bfuse' else 'hfuse'}"}
    src = build_pairs.source_text([k]).replace("Side0, ", "Slim<Side0>, ") + "static_assert(Slim<Side0>::GRID.size() == Side0::GRID.size() && sizeof(Slim<Side0>::Smem) == sizeof(Side0::Smem));\n"
    assert _compiled(k, src, tmp_path) == []


@pytest.mark.parametrize("i", range(4))
def test_no_block_fused_pair_of_the_batch_suites_is_left_out_for_registers(i, tmp_path):
    """A side of at most 512 threads is compiled for 256 registers a lane, as many as a fused workgroup of two such sides has.  The
    operators of more threads must have a form of fewer, and that must fit beside the partner that needs most."""
    reg = {k.name: k for k in bf.list_kernels()}
    wide = [n for n in _suite_operators() if reg[n].block[0] > 512]
    assert len(wide) == 4
    k = {"k1": wide[i], "k2": "bgemm_f32_1024x208x80x208", "form": "bfuse"}
    k["name"] = f"{k['k1']}_{k['k2']}_fused_bfuse_c256"
    src = build_pairs.source_text([k]).replace("Side0, ", "Narrow<Side0>, ") + "static_assert(Narrow<Side0>::THREADS <= 512 && Narrow<Side0>::GRID.size() == Side0::GRID.size());\n"
    (tmp_path / "pairs_0.hip").write_text(src)
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-device-only", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-Rpass-analysis=kernel-resource-usage", "-I", build_pairs.CSRC, "-c", str(tmp_path / "pairs_0.hip"), "-o", str(tmp_path / "pairs_0.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    assert f"Function Name: {k['name']}" in r.stderr and build_pairs.spilling_kernels(r.stderr) == []


@pytest.mark.parametrize("k1,k2", [
    # one wave without barriers beside operators that synchronise
    ("conv7x7s2p3_f32_1024x3x224x224_64", "bgemm_f32_1024x512x64x512"), ("conv7x7s2p3_f32_1024x3x224x224_64", "conv1x1s1p0_f32_1024x2048x8x8_320"),
    ("conv7x7s2p3_f32_1024x3x224x224_64", "conv3x3s2p0_f32_1024x192x17x17_320"), ("conv7x7s2p3_f32_1024x3x224x224_64", "gemm_f32_1024x768x2304"),
    # half a CU's LDS beside it
    ("conv3x3s1p0_f32_1024x128x28x28_256", "bgemm_f32_1024x208x64x208"), ("conv3x3s1p0_f32_1024x128x28x28_256", "bgemm_f32_1024x208x208x64"),
    ("conv3x3s1p0_f32_1024x128x28x28_256", "bgemm_f32_1024x208x80x208"), ("conv3x3s1p0_f32_1024x128x28x28_256", "bgemm_f32_1024x208x208x80"),
    ("conv3x3s1p0_f32_1024x128x28x28_256", "conv3x3s2p0_f32_1024x3x299x299_32")])
def test_operators_that_one_workgroup_can_hold(k1, k2):
    reg = {k.name: k for k in bf.list_kernels()}
    assert build_pairs.hfuse_possible(reg[k1], reg[k2], build_pairs.op_lds(k1), build_pairs.op_lds(k2))


def test_an_object_that_failed_a_check_is_not_there_for_the_next_make(tmp_path):
    """... which otherwise takes it for built and links a kernel that spills."""
    (tmp_path / "pairs_0.hip").write_text("""
#include <hip/hip_runtime.h>
extern "C" __global__ __launch_bounds__(1024) void spills(float* p)
{
    float v[160], s = 0.f;
    for (int i = 0; i < 160; ++i) v[i] = p[i * 1024 + threadIdx.x];
    for (int i = 0; i < 160; ++i) asm volatile("" : "+v"(v[i]));
    for (int i = 159; i >= 0; --i) s = s * 1.5f + v[i];
    p[threadIdx.x] = s;
}
""")
    for _ in range(2):
        r = subprocess.run(["make", "-C", build_pairs.CSRC, f"MODDIR={tmp_path}", str(tmp_path / "pairs_0.o")], capture_output=True, text=True)
        assert r.returncode != 0 and "spills registers" in r.stdout + r.stderr, r.stderr[-2000:]
        assert not (tmp_path / "pairs_0.o").exists() and build_pairs.spilling_kernels((tmp_path / "pairs_0.res").read_text()) == ["spills"]
