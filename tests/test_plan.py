"""The GEMM planner on the CPU (plan_check.cpp around runtime.cpp): operands that
a variant would not gather, split-K scratch, and which variants a size takes."""

import os
import shutil
import subprocess

import pytest

from conftest import ROOT

STORE, BIAS_N, BIAS_M, ELU_GRAD = range(4)


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cxx = shutil.which("g++")
    if not cxx or not os.path.isdir(f"{rocm}/include/hip"):
        pytest.skip("no g++ or HIP headers")
    exe = str(tmp_path_factory.mktemp("plan") / "plan_check")
    subprocess.run([cxx, "-w", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include", f"-I{ROOT}/include",
                    f"{ROOT}/tests/plan_check.cpp", "-o", exe, f"-L{rocm}/lib", f"-Wl,-rpath,{rocm}/lib", "-lamdhip64",
                    "-ldl"], check=True)

    def go(*lines):
        text = "\n".join(" ".join(str(int(x) if isinstance(x, bool) else x) for x in line) for line in lines) + "\n"
        return subprocess.run([exe], input=text, text=True, check=True, capture_output=True).stdout.splitlines()

    return go


def test_ungathered_operands_are_refused(ask):
    """A variant that would read B (or A) in order although the problem gathers
    it is refused; the gathers that the library uses are not."""
    refused = [(24576, 256, 128, True, False, ELU_GRAD, 128, 256, False, True),   # three-piece, K-contiguous A
               (24576, 256, 512, True, True, BIAS_N, 512, 512, False, True),      # three-piece forward
               (300, 256, 512, True, True, BIAS_N, 512, 512, False, True),        # strips of a short minibatch
               (4096, 512, 29, True, False, ELU_GRAD, 32, 512, False, True)]      # narrow K
    taken = [(24576, 512, 124, True, True, BIAS_N, 124, 124, True, False),        # a shuffled minibatch's forward
             (512, 124, 24576, False, False, STORE, 512, 124, False, True),       # and weight gradient
             (300, 512, 128, True, True, BIAS_N, 128, 128, True, False),
             (29, 128, 24576, False, False, STORE, 32, 128, False, True)]
    assert ask(*[("plan", *p) for p in refused]) == ["refused"] * len(refused)
    assert all(x != "refused" for x in ask(*[("plan", *p) for p in taken]))


@pytest.mark.parametrize("m,n", [(512, 123), (512, 124), (512, 128), (256, 512), (128, 256), (256, 288), (512, 64),
                                 (29, 128), (1, 128), (100, 33)])
def test_split_k_scratch_covers_every_shorter_batch(ask, m, n):
    """The scratch reserved for batches of up to K rows holds the partials of
    any K' <= K, whatever variant K' takes (a shortfall would refuse the call)."""
    for line in ask(*[("scratch", m, n, k) for k in (1, 40, 129, 384, 1000, 2400, 6145, 24577)]):
        have, need = map(int, line.split())
        assert have >= need


@pytest.mark.parametrize("rows", [3072, 4096, 4608, 5376, 6016, 24576])
@pytest.mark.parametrize("n,k", [(128, 128), (128, 64), (256, 128)])
def test_backward_of_a_layer_is_one_launch(ask, rows, n, k):
    """run_gemm_bwd merges a layer's weight and data gradients where both take
    the three-piece variants."""
    got = ask(("beside", rows, n, k, True, False, ELU_GRAD, k, n, False, False),
              ("beside", k, n, rows, False, False, STORE, k, n, False, False))
    assert [x.split()[0] for x in got] == ["zk_split_ak_bn_dg", "zk_split_am_bn"]


@pytest.mark.parametrize("m,n,k,want", [(256, 1000, 264, "zk_narrow_f22"), (256, 1500, 264, "zk_gemm_ak_bn_64x64x32_w22"),
                                        (512, 1000, 520, "zk_gemm_ak_bn_64x64x32_w22"), (512, 1000, 512, "zk_narrow_f22"),
                                        (512, 1000, 265, "zk_narrow_f22"), (512, 1500, 265, "zk_gemm_ak_bn_64x64x32_w22_s")])
def test_feature_major_layers_with_few_tiles(ask, m, n, k, want):
    """Where the K-splitting kernel measured faster than the 64 x 64 tiles: two
    tiles per CU, one where only the 64 x 64 tiles read A as float4 rows."""
    assert ask(("plan", m, n, k, True, False, BIAS_M, k, n, False, False))[0].split()[0] == want


@pytest.mark.parametrize("m,n,k,want", [(512, 8192, 64, False), (512, 10_000, 64, False), (256, 24_576, 64, True),
                                        (256, 24_576, 36, False), (512, 16_384, 36, True), (512, 10_000, 256, False),
                                        (512, 8192, 264, True), (512, 8193, 265, True), (512, 24_576, 128, True)])
def test_feature_major_layers_on_three_pieces(ask, m, n, k, want):
    """From 256 tiles of 128 x 128 on, with short reductions from 384 or 512, as
    measured against the fp32 tiles."""
    got = ask(("plan", m, n, k, True, False, BIAS_M, k, n, False, False))[0]
    assert got.startswith("zk_split_ak_bn") == want, got


@pytest.mark.parametrize("m,n,k,a,b,want", [(1500, 512, 256, 1, 0, "zk_gemm_ak_bn_64x64x32_w22 1"),
                                            (16_384, 64, 288, 1, 1, "zk_gemm_ak_bk_64x64x32_w22 1"),
                                            (128, 16_384, 256, 0, 0, "zk_gemm_am_bn_64x128x32_w24_x 1"),
                                            (512, 512, 384, 0, 0, "zk_split_am_bn 6"),
                                            (10_000, 512, 64, 1, 0, "zk_split_ak_bn 1"),
                                            (256, 512, 24_576, 1, 1, "zk_split_ak_bk 32"),
                                            (512, 24_576, 256, 0, 0, "zk_split_am_bn 1")])
def test_products_summed_apart(ask, m, n, k, a, b, want):
    """Products whose split-K partials take a launch of their own: few slices and
    fp32 tiles where that launch and the traffic cost more than they save. (The
    first three measured 10.2, 10.6 and 15.1 us, 15.4, 20.1 and 25.7 as a minibatch
    runs them.)"""
    assert ask(("apart", m, n, k, a, b, STORE, k if a else m, k if b else n, False, False)) == [want]


@pytest.mark.parametrize("how,m,n,k,ld,want", [("plan", 4096, 256, 512, 512, False), ("plan", 16_384, 128, 128, 128, False),
                                               ("plan", 10_000, 256, 512, 512, True), ("pair", 4096, 256, 512, 512, False),
                                               ("pair", 4608, 256, 512, 512, True), ("plan", 4096, 256, 123, 123, True),
                                               ("plan", 12_288, 512, 64, 64, True), ("pair", 2048, 512, 512, 512, False)])
def test_forwards_on_three_pieces(ask, how, m, n, k, ld, want):
    """By the tiles of the launch: 144 with float4-aligned rows, 64 without."""
    got = ask((how, m, n, k, True, True, BIAS_N, ld, ld, False, False))[0]
    assert got.startswith("zk_split_ak_bk") == want, got


@pytest.mark.parametrize("how,m,n,k,want", [
    ("plan", 1000, 512, 512, False), ("plan", 3000, 512, 256, False), ("plan", 4096, 128, 128, True),
    ("plan", 24_576, 512, 128, True), ("plan", 24_576, 512, 100, False), ("plan", 24_576, 192, 128, False),
    ("plan", 24_576, 64, 128, False), ("plan", 24_576, 384, 200, False), ("plan", 24_576, 192, 256, True),
    ("beside", 12_288, 100, 100, False), ("beside", 24_576, 100, 100, True), ("beside", 24_576, 64, 48, False)])
def test_data_gradients_on_three_pieces(ask, how, m, n, k, want):
    """Alone in their launch: whole column tiles and k-tiles from 4,096 rows on,
    others from K = 256 and 192 tiles; beside their weight gradient from 192."""
    got = ask((how, m, n, k, True, False, ELU_GRAD, (k + 3) // 4 * 4, n, False, False))[0]
    assert got.startswith("zk_split_ak_bn_dg") == want, got


def test_bench_counts_every_gemm_kernel(ask):
    """The layer GEMM time and FLOPs that bench.py reports cover every GEMM
    kernel of the table and the fixed kernels that contain one, and no other."""
    import bench

    names = ask(("names",))[0].split()
    fixed = {x for x in names[:names.index("zk_policy_pack") + 1] if x.startswith(("zk_split_bwd", "zk_head_fwd"))}
    table = set(names[names.index("zk_policy_pack") + 1:])
    assert {"zk_split_bwd", "zk_head_fwd"} <= fixed and {"zk_split_ak_bn_dg", "zk_narrow_f22"} <= table
    assert {x for x in names if bench.is_layer_gemm(x)} == fixed | table
