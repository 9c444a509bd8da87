"""The kernels a quantised long pass is routed to by its shape and format (csrc/gemm.hip, gemm_route): the K sum split
over a workgroup's waves or over ranges, and the dense routes over operand-ordered and row-major weights, on every tile.

Each shape: fp16 and fp32 inputs of equal values give equal bits; every output is the fp16 rounding of the exact
(float64) sum of the fp16 operands up to ½ fp16 ulp + 2^-16·Σ|x·w| (an fp32 sum's rounding), and bitwise the one-range
result where K is not split; an output with a row stride that rules out wide stores gets the same values and leaves its
other columns alone."""
import numpy as np
import pytest
import torch

from swiftrwkv_amd import _lib, quant as Q
from tests.test_gpu_prefill import check_f16_rounding

pytestmark = pytest.mark.gpu
DEV = "cuda"

# kernel and tile: (rows, OUT, IN, groups) with that route in all five formats (None: it differs between them); partial
# row blocks, one row, a single K step per wave, uneven steps per wave, more steps than one block of scale words
SHAPES = {
    ("waves", 16, 16): [(1, 256, 256, 1), (17, 128, 512, 1), (16, 768, 5376, 1), (31, 1536, 2304, 3)],
    ("waves", 32, 16): [(17, 2304, 256, 3), (257, 384, 768, 1), (128, 768, 768, 1), (96, 768, 3072, 1), (150, 1536, 512, 3),
                        (128, 1024, 5376, 1)],
    ("waves", 32, 32): [(31, 4608, 2048, 1), (129, 3072, 1024, 3), (129, 6144, 512, 1), (150, 3072, 5376, 1)],
    ("waves", 64, 16): [(33, 3072, 768, 1), (65, 2048, 1536, 1), (190, 3840, 5376, 3)],
    ("waves", 64, 32): [(257, 3840, 256, 3), (130, 2304, 2304, 1), (90, 4096, 2304, 1), (640, 640, 2304, 1)],
    ("waves", 64, 64): [(65, 8192, 512, 1), (129, 4608, 512, 3), (900, 1024, 512, 1), (127, 8192, 1792, 1)],
    ("dense", 64, 64): [(1030, 512, 2304, 1), (1100, 640, 3072, 1)],
    ("dense", 64, 128): [(700, 2304, 768, 3), (1030, 1024, 1280, 1), (3001, 640, 1536, 1)],
    ("dense", 128, 128): [(1001, 3072, 1024, 3), (257, 8192, 512, 1), (1300, 1920, 2048, 1)],
    ("dense", 256, 256): [(1999, 4608, 2816, 3), (4100, 2048, 2816, 1)],
    ("dense rows", 256, 256): [(1999, 4608, 512, 1), (1300, 6144, 256, 3)],
    ("ranges", 128, 128): [(400, 8192, 256, 1), (1001, 3840, 256, 3)],
    None: [(130, 1024, 4096, 1), (129, 2304, 768, 1), (257, 2304, 512, 1), (700, 768, 1024, 1), (1300, 512, 2048, 1),
           (1500, 2304, 256, 1)],
}


def matrix(fmt, OUT, IN, seed):
    """(loader buffers, the gemm of them, C entry, code bits, their fp16 weight) of a Gaussian matrix."""
    kind, bits = fmt.split(":")
    bits = int(bits)
    w = np.random.default_rng(seed).standard_normal((OUT, IN), dtype=np.float32) * np.float32(0.05)
    L = _lib.lib()
    if kind == "sb6":
        d = Q.encode_sb6(w, 4 + bits)
        qblk, qsqm, ddm, xb = Q.rwkvq_sb6_to_k3(d["codes_packed"], d["gw_qsqm"], d["gw_d"], d["gw_dm"], d.get("gw_qh"),
                                                d.get("gw_qh2"), (OUT, IN))
        assert xb == bits
        bufs = [torch.from_numpy(z).to(DEV) for z in (qblk, qsqm, ddm.view(np.float16))]
        return bufs, Q.rwkvq_sb6_gemm, L.rwkv_sb6_gemm, bits, Q.rwkvq_dequant_dense(*bufs, OUT, IN, 8, bits, torch.float16)
    d = Q.encode_sym(w, bits)
    codes = d["codes"].view(np.uint8) if bits == 8 else Q.rwkvq_sym_interleave(d["codes_packed"], d["gw_qh"], d["gw_qh2"],
                                                                               (OUT, IN))
    bufs = [torch.from_numpy(z).to(DEV) for z in (codes, d["gw_qs"].view(np.uint8), d["gw_d"])]
    return bufs, Q.rwkvq_sym_gemm, L.rwkv_sym_gemm, bits, Q.rwkvq_dequant_sym(*bufs, OUT, IN, bits, torch.float16)


@pytest.mark.parametrize("fmt", ["sb6:0", "sb6:1", "sb6:2", "sym:8", "sym:6"])
@pytest.mark.parametrize("kernel,M,OUT,IN,G", [(k, *s) for k, v in SHAPES.items() for s in v])
def test_quant_gemm_routes(fmt, kernel, M, OUT, IN, G):
    print(f"[case] gemm route {kernel} {fmt} M={M} {OUT}x{IN} G={G}", flush=True)
    bufs, gemm, entry, bits, w16 = matrix(fmt, OUT, IN, M + OUT)
    per = OUT // G
    route = Q.rwkvq_gemm_route(fmt[:3], bits, M, OUT, IN, per)
    assert kernel in (None, route[:3])
    gen = torch.Generator(device=DEV).manual_seed(M + IN)
    x = torch.randn((G, M, IN), generator=gen, device=DEV).half()
    dequants = f"{fmt[:3]}_dequant"
    n0 = _lib.counters()[dequants]
    y = gemm(x, *bufs, OUT, IN, bits, out_per=per)
    assert _lib.counters()[dequants] == n0 + route[0].startswith("dense")   # the kernel that the route names ran
    assert torch.equal(gemm(x.float(), *bufs, OUT, IN, bits, out_per=per), y)
    if route[3] == 1:
        assert torch.equal(gemm(x, *bufs, OUT, IN, bits, out_per=per, split=False), y)
    for g in range(G):
        xs, ws, got = x[g].double(), w16[g * per:(g + 1) * per].double(), y[:, g * per:(g + 1) * per]
        check_f16_rounding(got.cpu().numpy(), (xs @ ws.T).cpu().numpy(), (xs.abs() @ ws.abs().T).cpu().numpy())
    h = gemm(x, *bufs, OUT, IN, bits, out_per=per, epilogue="relu2_f16")
    assert torch.equal(h, (torch.relu(y) * torch.relu(y)).half())
    base = torch.randn((M, OUT + 3), generator=gen, device=DEV)
    out = base.clone()
    need = Q.rwkvq_gemm_workspace(M, OUT, IN)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    _lib.check(entry(x.data_ptr(), _lib.F16, M, IN, M * IN, *[b.data_ptr() for b in bufs], out.data_ptr(), OUT + 3, OUT,
                     IN, bits, per, 1, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out[:, :OUT], base[:, :OUT] + y)
    assert torch.equal(out[:, OUT:], base[:, OUT:])


@pytest.mark.parametrize("fmt", ["sb6:0", "sb6:1", "sb6:2", "sym:8", "sym:6"])
@pytest.mark.parametrize("M,OUT,IN,G,kernel,parts", [
    (65, 16640, 768, 1, "ranges", 3), (128, 16512, 1792, 3, "ranges", 3),
    (300, 12288, 256, 3, "ranges", 1),
    (700, 11008, 256, 1, "dense rows", 1), (2000, 4608, 512, 3, "dense rows", 1)])
def test_ranges_and_row_major_routes(fmt, M, OUT, IN, G, kernel, parts):
    """K ranges on 128-row tiles and the row-major dense route: each output as test_quant_gemm_routes has it, and bitwise
    the one-range result where K is not split."""
    print(f"[case] gemm route {kernel} {fmt} M={M} {OUT}x{IN} G={G}", flush=True)
    bufs, gemm, entry, bits, w16 = matrix(fmt, OUT, IN, M + OUT)
    per = OUT // G
    assert Q.rwkvq_gemm_route(fmt[:3], bits, M, OUT, IN, per)[::3] == (kernel, parts)
    gen = torch.Generator(device=DEV).manual_seed(M + IN)
    x = torch.randn((G, M, IN), generator=gen, device=DEV).half()
    y = gemm(x, *bufs, OUT, IN, bits, out_per=per)
    assert torch.equal(gemm(x.float(), *bufs, OUT, IN, bits, out_per=per), y)
    if parts == 1:
        assert torch.equal(gemm(x, *bufs, OUT, IN, bits, out_per=per, split=False), y)
    else:
        for g in range(G):
            xs, ws, got = x[g].double(), w16[g * per:(g + 1) * per].double(), y[:, g * per:(g + 1) * per]
            check_f16_rounding(got.cpu().numpy(), (xs @ ws.T).cpu().numpy(), (xs.abs() @ ws.abs().T).cpu().numpy())
    h = gemm(x, *bufs, OUT, IN, bits, out_per=per, epilogue="relu2_f16")
    assert torch.equal(h, (torch.relu(y) * torch.relu(y)).half())
    base = torch.randn((M, OUT), generator=gen, device=DEV)
    assert torch.equal(gemm(x, *bufs, OUT, IN, bits, out_per=per, epilogue="add", out=base.clone()), base + y)


@pytest.mark.parametrize("fmt,M,OUT,IN", [("sb6:0", 300, 12288, 256), ("sym:6", 300, 12288, 256), ("sb6:2", 1024, 4096, 512)])
def test_small_workspace_is_taken_where_one_range_fills_the_chip(fmt, M, OUT, IN):
    """160 or more 128 × 128 tiles, too few 256 × 256 ones for the dense kernel: any aligned workspace runs, by the
    kernels that fit in it; without one the _auto entry picks among those too."""
    print(f"[case] gemm small workspace {fmt} M={M} {OUT}x{IN}", flush=True)
    bufs, gemm, entry, bits, w16 = matrix(fmt, OUT, IN, M + OUT)
    x = torch.randn((M, IN), generator=torch.Generator(device=DEV).manual_seed(M), device=DEV).half()
    exact, mag = x.double() @ w16.double().T, x.double().abs() @ w16.double().abs().T
    ws = torch.zeros(64, dtype=torch.uint8, device=DEV)
    auto = getattr(_lib.lib(), f"rwkv_{fmt[:3]}_gemm_auto")
    got = []
    for f, p, n in ((entry, ws.data_ptr(), 16), (auto, ws.data_ptr(), 16), (auto, None, 0)):
        y = torch.empty((M, OUT), device=DEV)
        _lib.check(f(x.data_ptr(), _lib.F16, M, IN, M * IN, *[b.data_ptr() for b in bufs], y.data_ptr(), OUT, OUT, IN, bits,
                     OUT, 0, p, n, torch.cuda.current_stream().cuda_stream))
        got.append(y)
    check_f16_rounding(got[0].cpu().numpy(), exact.cpu().numpy(), mag.cpu().numpy())
    assert torch.equal(got[1], got[0]) and torch.equal(got[2], got[0])
    assert not ws.any()


@pytest.mark.parametrize("fmt,M,OUT,IN", [("sb6:0", 128, 3072, 768), ("sym:8", 700, 768, 768), ("sym:6", 33, 4096, 4096)])
def test_wave_split_takes_no_memory(fmt, M, OUT, IN):
    """A pass split over waves allocates its output and nothing else; its bits are those of a call with a workspace."""
    print(f"[case] gemm memory {fmt} M={M} {OUT}x{IN}", flush=True)
    bufs, gemm, entry, bits, _ = matrix(fmt, OUT, IN, M)
    assert Q.rwkvq_gemm_route(fmt[:3], bits, M, OUT, IN)[0] == "waves"
    assert Q.rwkvq_gemm_auto_workspace(fmt[:3], bits, M, OUT, IN) == 0
    x = torch.randn((M, IN), generator=torch.Generator(device=DEV).manual_seed(M), device=DEV).half()
    out = torch.empty((M, OUT), device=DEV)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    gemm(x, *bufs, OUT, IN, bits, out=out)
    assert torch.cuda.max_memory_allocated() == before
    need = Q.rwkvq_gemm_workspace(M, OUT, IN)
    ws, y = torch.empty(need, dtype=torch.uint8, device=DEV), torch.empty((M, OUT), device=DEV)
    _lib.check(entry(x.data_ptr(), _lib.F16, M, IN, M * IN, *[b.data_ptr() for b in bufs], y.data_ptr(), OUT, OUT, IN, bits,
                     OUT, 0, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(y, out)
