"""What build.py looks for in the generated code of the grouped GEMM kernels, on small listings."""

import importlib.util
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READ = ";;#ASMSTART\n\tds_read_b128 v[4:7], v1 offset:16\n\t;;#ASMEND\n"
LOAD = ";;#ASMSTART\n\tglobal_load_dword v9, v[10:11], off\n\t;;#ASMEND\n"
DMA = "\tbuffer_load_dwordx4 v2, s[0:3], 0 offen lds\n"
WAIT = "\ts_waitcnt lgkmcnt(0)\n"
MFMA = "\tv_mfma_f32_32x32x16_bf16 a[0:15], v[12:15], v[16:19], a[0:15]\n"
SPILL = "\tscratch_store_dword off, v2, off\n"


@pytest.fixture(scope="module")
def build():
    spec = importlib.util.spec_from_file_location("xma_build", os.path.join(ROOT, "accelerated-model-architectures_amd", "build.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def _check(build, tmp_path, body):
    listing = tmp_path / "kernel.s"
    listing.write_text("_Z6kernelv:  ; @kernel\n" + body + "\ts_endpgm\n.Lfunc_end0:\n")
    build._check_isa(str(listing), re.compile("kernel"))


@pytest.mark.parametrize("body", [
    READ + WAIT + "\tv_mov_b32_e32 v5, v2\n",
    READ + "\tv_mov_b32_e32 v8, v2\n",
    LOAD + "\ts_waitcnt vmcnt(0) lgkmcnt(0)\n\tv_add_u32_e32 v9, 1, v9\n",
    LOAD + DMA + DMA + "\ts_waitcnt vmcnt(2)\n\tv_add_u32_e32 v9, 1, v9\n",
    READ + "\ts_branch .LBB0_2\n.LBB0_1:\n\tv_mov_b32_e32 v5, v2\n\ts_endpgm\n.LBB0_2:\n" + WAIT,
    ".LBB0_1:\n" + WAIT + MFMA + READ + "\ts_cbranch_scc1 .LBB0_1\n" + WAIT,
    SPILL + ".LBB0_1:\n" + MFMA + "\ts_cbranch_scc1 .LBB0_1\n" + SPILL,
])
def test_sound_code_passes(build, tmp_path, body):
    _check(build, tmp_path, body)


@pytest.mark.parametrize("body", [
    READ + "\tv_mov_b32_e32 v5, v2\n" + WAIT,
    READ + "\tv_mov_b32_e32 v2, v7\n",
    READ + "\ts_waitcnt lgkmcnt(1)\n\tv_mov_b32_e32 v2, v7\n",
    READ + READ.replace("v[4:7], v1", "v[20:23], v4"),  # a read whose address is still on its way
    LOAD + WAIT + "\tv_add_u32_e32 v9, 1, v9\n",
    LOAD + DMA + "\ts_waitcnt vmcnt(2)\n\tv_add_u32_e32 v9, 1, v9\n",
    LOAD + DMA + "\ts_cbranch_scc1 .LBB0_1\n" + DMA + ".LBB0_1:\n\ts_waitcnt vmcnt(2)\n\tv_add_u32_e32 v9, 1, v9\n",  # one on one path
    READ + "\ts_branch .LBB0_2\n.LBB0_1:\n" + WAIT + "\ts_endpgm\n.LBB0_2:\n\tv_mov_b32_e32 v5, v2\n\ts_branch .LBB0_1\n",
    ".LBB0_1:\n\tv_accvgpr_read_b32 v6, a0\n" + WAIT + MFMA + READ + "\ts_cbranch_scc1 .LBB0_1\n" + WAIT,  # over the back edge
    ".LBB0_1:\n" + WAIT + MFMA + READ + "\ts_cbranch_scc1 .LBB0_1\n\tv_accvgpr_read_b32 v6, a0\n" + WAIT,  # behind the loop
])
def test_touched_in_flight_fails(build, tmp_path, body):
    with pytest.raises(RuntimeError, match="in flight"):
        _check(build, tmp_path, body)


def test_scratch_in_mfma_loop_fails(build, tmp_path):
    with pytest.raises(RuntimeError, match="scratch"):
        _check(build, tmp_path, ".LBB0_0:\n.LBB0_1:\n" + MFMA + SPILL + "\ts_cbranch_scc1 .LBB0_1\n\ts_cbranch_scc0 .LBB0_0\n")
