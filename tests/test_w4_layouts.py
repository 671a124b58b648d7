"""The 4-wave kernels with M-contiguous operands on the CPU: wait counts, the replay of addresses and data flow (tests/w4_emulator.py),
and compiled code that leaves the accumulators alone (what test_w4_generator, test_w4_emulator and test_w4_build check of the others)."""
import os
import re
import subprocess

import pytest

from test_w4_build import CSRC, HIPCC
from w4_emulator import Fail, load_generator, replay

KINDS = ["bf16_km", "bf16_mk", "bf16_mm"]


@pytest.mark.parametrize("kind", KINDS)
def test_wait_counts(kind):
    slack = load_generator().Gen(kind).check()
    assert slack and min(slack.values()) >= 0


@pytest.mark.parametrize("kind", KINDS)
def test_whole_and_ragged_tiles(kind):
    for ks in (4, 6, 8):
        assert replay(kind, 512, 768, ks, [(0, 0), (256, 0), (0, 256), (256, 512)]) > 0
    replay(kind, 600, 520, 4, [(0, 0), (512, 0), (256, 256), (0, 512), (512, 512), (256, 0)], pad=64)
    replay(kind, 512, 512, 8, [(0, 0), (256, 0), (0, 256)], c_bf16=False)


def test_replay_catches_a_wrong_copy_step_and_a_wrong_half(monkeypatch):
    import w4_emulator as E
    real = E.load_generator

    def patched(name, change):
        def load():
            g = real()
            method = getattr(g.Gen, name)
            setattr(g.Gen, name, lambda self, *a: [g.Op(change(o.text), o.vm) for o in method(self, *a)])
            return g
        return load
    for name, change in (("dma_advance", lambda t: t.replace("%[bstep]", "128")),
                         ("frag_read", lambda t: t.replace("offset:512", "offset:1024") if "_tr_" in t else t)):
        monkeypatch.setattr(E, "load_generator", patched(name, change))
        with pytest.raises(Fail):
            E.replay("bf16_mm", 512, 512, 8, [(0, 0), (256, 0)])


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_compiled_code_leaves_the_accumulators_alone(tmp_path):
    kinds = [t + k[4:] for t in ("bf16", "f16") for k in KINDS]
    subprocess.run(["make", "-C", CSRC, "-s"] + [f"w4_{p}_{k}.inc" for p in ("kloop", "clobbers") for k in kinds], check=True)
    out = tmp_path / "w4m.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-Wno-unused-command-line-argument", "-Wno-pass-failed", "-Wno-inline-asm", "-S", "--cuda-device-only",
                    os.path.join(CSRC, "gemm_inst_w4m.hip"), "-o", str(out)], cwd=CSRC, stderr=subprocess.DEVNULL, check=True)
    text = out.read_text()
    assert len(re.findall(r"^(_ZN2tb14gemm_kernel_w4\S+):", text, re.M)) == 6
    assert "v_accvgpr_write" not in text and "v_accvgpr_mov" not in text
    for line in text.splitlines():
        if "v_accvgpr_read" in line:
            assert re.search(r"v_accvgpr_read_b32 v\d+, a(\d+|\[\w+\])\s*$", line), line


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("ta,tb_", [("T", "T"), ("N", "N"), ("N", "T")])
def test_same_bits_as_the_eight_wave_kernel(ta, tb_, dtype, tb_option):
    """whole and ragged tiles, several per workgroup (a limited grid) and one, with and without a bias; both kernels add in the same order"""
    import torch
    import tritonblas_amd as tb
    from tritonblas_amd.matmul import persistent_matmul_lt
    dtype = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(1)
    for m, n, k, grid in [(256, 256, 256, 0), (512, 768, 384, 0), (520, 776, 640, 2), (1288, 1024, 256, 3), (768, 1536, 4096, 4)]:
        a, b = torch.randn((m, k), device="cuda", generator=gen).to(dtype), torch.randn((k, n), device="cuda", generator=gen).to(dtype)
        a, b = (a if ta == "T" else a.T.contiguous().T), (b if tb_ == "T" else b.T.contiguous().T)
        sel = tb.OrigamiMatmulSelector(m, n, k, dtype, dtype, dtype, a.device)
        sel._sel.block_m, sel._sel.block_n, sel._sel.block_k = 256, 256, 64
        bias = torch.randn(n, device="cuda", generator=gen).to(dtype)
        tb_option("grid", grid)
        out = []
        for waves in (0, 24):
            tb_option("waves", waves)
            for bv in (None, bias):
                c = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
                persistent_matmul_lt(a, b, c, sel, None, bias=bv)
                out.append(c)
        want = a.double() @ b.double()
        assert ((out[0].double() - want).norm() / want.norm()).item() <= torch.finfo(dtype).eps
        assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3]), (m, n, k)
