"""gemm_route (csrc/gemm.hip), the choice of a quantised long pass's kernel, on the host."""
import pytest
import torch

from swiftrwkv_amd import quant as Q
from tests.test_gpu_gemm_routes import SHAPES

FORMATS = [("sb6", 0), ("sb6", 1), ("sb6", 2), ("sym", 8), ("sym", 6)]


@pytest.mark.parametrize("fmt,M,OUT,IN,kernel", [
    # 65-128 rows of a large matrix: µs on ranges of K (128-row tiles) against the wave split's 64-row tiles
    (("sb6", 0), 98, 10240, 5888, "ranges"),      # 47, 54
    (("sym", 8), 98, 10240, 5888, "ranges"),      # 44, 66
    (("sym", 8), 128, 14336, 14336, "ranges"),    # 148, 224
    (("sym", 8), 87, 19200, 7680, "ranges"),      # 97, 122
    # short K, many rows: row-major weights against operand order
    (("sb6", 0), 4096, 3072, 768, "dense rows"),  # 31, 35
    (("sb6", 2), 8192, 3072, 256, "dense rows"),  # 32, 38
    (("sym", 8), 4177, 12288, 768, "dense rows"), # 108, 118
    # one stage or two of K: one range, no dequant, against the dense route
    (("sb6", 0), 512, 12288, 256, "ranges"),      # 15, 19
    # and where the other kernels stay the faster ones
    (("sb6", 0), 128, 3072, 768, "waves"),        # 13, 6
    (("sb6", 1), 128, 14336, 4096, "waves"),      # 67, 56
    (("sym", 6), 128, 4096, 4096, "waves"),       # 33, 20
    (("sb6", 0), 8192, 14336, 4096, "dense"),     # 805, 785
])
def test_fastest_kernel(fmt, M, OUT, IN, kernel):
    assert Q.rwkvq_gemm_route(*fmt, M, OUT, IN)[0] == kernel


@pytest.mark.parametrize("kind,bits", FORMATS)
def test_route_fits_its_workspace_and_its_inputs(kind, bits):
    """Whatever the workspace, the kernel's own need is within it; fp32 inputs take a kernel with fp16 inputs' sums."""
    for M in (1, 40, 65, 100, 128, 300, 1500, 4096, 20000):
        for OUT, IN in ((128, 256), (768, 768), (2304, 256), (4096, 4096), (10240, 5888), (14336, 4096), (16640, 768)):
            for out_per in {OUT, 128} | ({OUT // 3} if OUT % 384 == 0 else set()):
                for ws in (-1, 0, 16, 8 * M * OUT, OUT * IN * 2, Q.rwkvq_gemm_workspace(M, OUT, IN), None):
                    name, tm, tn, parts = Q.rwkvq_gemm_route(kind, bits, M, OUT, IN, out_per, workspace=ws)
                    have = Q.rwkvq_gemm_auto_workspace(kind, bits, M, OUT, IN, out_per) if ws is None else ws
                    need = OUT * IN * 2 if name.startswith("dense") else 4 * parts * M * OUT if name == "ranges" and parts > 1 else 0
                    assert need <= max(have, 0)
                    assert OUT % tn == 0 and (not name.startswith("dense") or out_per % tn == 0)
                    n32, tm32, tn32, parts32 = Q.rwkvq_gemm_route(kind, bits, M, OUT, IN, out_per, torch.float32, ws)
                    assert n32 == {"dense rows": "dense"}.get(name, name) and parts32 == parts
                    if ws == -1:
                        assert (name, parts) == ("ranges", 1)


def test_gpu_shapes_take_the_kernels_they_are_listed_for():
    """The GPU tests' shapes (tests/test_gpu_gemm_routes.py) reach every kernel and tile in every format."""
    listed = [(k, s) for k, v in SHAPES.items() if k for s in v]
    wrong = [(k, s, f, r) for k, s in listed for f in FORMATS
             if (r := Q.rwkvq_gemm_route(*f, *s[:3], s[1] // s[3])[:3]) != k]
    assert not wrong
    assert {k for k, _ in listed} == {("waves", m, n) for m, n in ((16, 16), (32, 16), (32, 32), (64, 16), (64, 32), (64, 64))} | {
        ("dense", m, n) for m, n in ((64, 64), (64, 128), (128, 128), (256, 256))} | {("dense rows", 256, 256),
                                                                                      ("ranges", 128, 128)}
