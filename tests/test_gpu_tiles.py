"""Block tiles of the GEMMs and the grouped MoE, and depths off the 128-byte stage.

Shapes pick each tile of the choosers (64x64 to 256x256) with ragged M and N
edges and K a multiple of 16 bytes only (last stages of 16, 64 and 112 bytes),
and the last-rows kernels with partial last stages.  Integer results are exact
against float64 products (sums below 2^53).
"""
import numpy as np
import pytest
import torch

from baracuda_amd import plans as P
from baracuda_amd.ffi import lib
from oracle.inputs import int8_uniform, moe_routing, rng
from tests import test_gpu_gemm as G
from tests import test_gpu_moe_wmma as W
from tests import test_gpu_sweep as S
from tests.gpu_util import FP8_FLOOR, dev, host_bits16, sync
from tests.test_gpu_decode import _gemv_check, _gemv_inputs, _gemv_run
from tests.test_gpu_moe import _block_routing, _run as _moe_run

pytestmark = pytest.mark.gpu

TILE_SHAPES = [(300, 1700, 208), (450, 2896, 1040), (1000, 2500, 1136), (1500, 5120, 336), (2300, 5008, 400),
               (3070, 4100, 336), (4000, 4100, 48), (513, 2064, 16)]
# one row (partial kilobyte), one / two / four / eight fragments, each column
# width, row blocks, whole tiles with last rows (test_dispatch_rules.py has the
# routes of the wider ones)
ROW_SHAPES = [(1, 4096, 4080), (1, 272, 48), (5, 512, 1040), (9, 12288, 304), (13, 6160, 1552), (24, 4096, 2752),
              (60, 12288, 304), (100, 272, 656), (120, 6144, 176), (200, 1024, 1072), (400, 1024, 208),
              (4160, 4096, 144),
              # 32 columns with four and eight fragments (test_dispatch_rules.py
              # has their routes), row blocks of deep K past 128 tiles
              (40, 6176, 304), (1856, 8224, 144), (1892, 8224, 144), (100, 14336, 8208), (160, 5120, 11280),
              (384, 2720, 9232), (200, 8192, 8208),
              # 48-, 96- and 112-column workgroups, the last one partly past N
              (20, 11008, 304), (12, 22016, 144), (30, 28656, 144), (12, 17920, 528), (20, 20464, 8720), (9, 43008, 272)]


def _acc(a, b):
    return (torch.from_numpy(a).double() @ torch.from_numpy(b).double().T).to(torch.int64).numpy()


@pytest.mark.parametrize("shape", TILE_SHAPES + ROW_SHAPES)
def test_int8_tiles_and_depth_tails(gpu, shape):
    m, n, k = shape
    print(f"case: int8 tiles {shape}", flush=True)
    g = rng(m + 3 * n + 7 * k)
    a, b, c = int8_uniform(g, (m, k)), int8_uniform(g, (n, k)), int8_uniform(g, (m, n))
    acc = _acc(a, b)
    ta, tb = dev(a), dev(b)
    d = torch.full((m, n), -7, dtype=torch.int32, device="cuda:0")
    P.IntGemmPlan.select(P.IntGemmDescriptor(m, n, k, output=P.ElementKind.I32)).run(ta, tb, d)
    sync()
    assert np.array_equal(d.cpu().numpy(), acc)
    accf = acc.astype(np.float32)
    # int8 out with C: f32 products and sum, round half to even, saturate
    alpha = np.float32(1.0 / (60.0 * np.sqrt(k)))
    d8 = torch.full((m, n), 99, dtype=torch.int8, device="cuda:0")
    P.IntGemmPlan.select(P.IntGemmDescriptor(m, n, k)).run(ta, tb, d8, c=dev(c), alpha=float(alpha), beta=0.5)
    sync()
    z = alpha * accf + np.float32(0.5) * c.astype(np.float32)
    assert np.array_equal(d8.cpu().numpy(), np.clip(np.rint(z), -128, 127).astype(np.int8))
    # W8A8: (sa * sw) * acc, bf16 / f32 / f64
    sa, sw = g.uniform(0.005, 0.02, m).astype(np.float32), g.uniform(0.001, 0.01, n).astype(np.float32)
    y = (sa[:, None] * sw[None, :]) * accf
    dw = torch.empty((m, n), dtype=torch.bfloat16, device="cuda:0")
    P.IntGemmPlan.select(P.IntGemmDescriptor(m, n, k, output=P.ElementKind.Bf16)).run(
        ta, tb, dw, scale_a=dev(sa), scale_b=dev(sw))
    out = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
    out64 = torch.empty((m, n), dtype=torch.float64, device="cuda:0")
    stream = torch.cuda.current_stream().cuda_stream
    tsa, tsw, tsa64, tsw64 = dev(sa), dev(sw), dev(sa.astype(np.float64)), dev(sw.astype(np.float64))
    assert lib().quantized_linear_w8a8_f32_gfx950_run(m, n, k, tb.data_ptr(), ta.data_ptr(), tsa.data_ptr(),
                                                      tsw.data_ptr(), out.data_ptr(), None, 0, stream) == 0
    assert lib().quantized_linear_w8a8_f64_gfx950_run(m, n, k, tb.data_ptr(), ta.data_ptr(), tsa64.data_ptr(),
                                                      tsw64.data_ptr(), out64.data_ptr(), None, 0, stream) == 0
    sync()
    assert np.array_equal(host_bits16(dw), host_bits16(torch.from_numpy(y).to(torch.bfloat16)))
    assert np.array_equal(out.cpu().numpy(), y)
    assert np.array_equal(out64.cpu().numpy(), y.astype(np.float64))


@pytest.mark.parametrize("shape", [(300, 1700, 208), (1500, 5120, 336), (2300, 5008, 400), (60, 12288, 304),
                                   (4160, 4096, 144)])
def test_int8_depth_tail_reads_stay_in_the_row(gpu, shape):
    """Rows wider than K: what lies past K in a row must not reach the sums."""
    m, n, k = shape
    g = rng(m + n + k)
    pa, pb = int8_uniform(g, (m, k + 112)), int8_uniform(g, (n, k + 64))
    print(f"case: int8 padded rows {shape}", flush=True)
    d = torch.empty((m, n), dtype=torch.int32, device="cuda:0")
    P.IntGemmPlan.select(P.IntGemmDescriptor(m, n, k, output=P.ElementKind.I32)).run(
        dev(pa)[:, :k], dev(pb)[:, :k], d)
    sync()
    assert np.array_equal(d.cpu().numpy(), _acc(np.ascontiguousarray(pa[:, :k]), np.ascontiguousarray(pb[:, :k])))


@pytest.mark.parametrize("shape", TILE_SHAPES + ROW_SHAPES)
def test_fp8_tiles_and_depth_tails(gpu, shape):
    """e4m3 RCR: f32 out within the FP8 tolerance, bf16 out its rounding; what
    lies past K in a row (NaN codes here) stays out."""
    m, n, k = shape
    print(f"case: fp8 tiles {shape}", flush=True)
    g = rng(m + 5 * n + 3 * k)

    def operand(rows, pad):
        x = torch.from_numpy(g.standard_normal((rows, k)).astype(np.float32) * 100)
        x = x.clamp(-448, 448).to(torch.float8_e4m3fn)      # past 464 torch casts to NaN
        t = torch.full((rows, k + pad), 0x7f, dtype=torch.uint8)
        t[:, :k] = x.view(torch.uint8)
        return x.double(), t.to("cuda:0")[:, :k]

    xa, ta = operand(m, 112)
    xb, tb = operand(n, 48)
    d = torch.zeros((m, n), dtype=torch.float32, device="cuda:0")
    P.Fp8GemmPlan.select(P.Fp8GemmDescriptor(m, n, k, output=P.ElementKind.F32)).run(ta, tb, d, alpha=0.5)
    db = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda:0")
    P.Fp8GemmPlan.select(P.Fp8GemmDescriptor(m, n, k, output=P.ElementKind.Bf16)).run(
        ta, tb, db, scale_a=0.5, scale_b=1.0)
    sync()
    got, exact = d.cpu().double(), 0.5 * (xa @ xb.T)
    bound = 1e-3 * exact.abs() + FP8_FLOOR * 0.5 * (xa.abs() @ xb.abs().T)
    assert bool(((got - exact).abs() <= bound).all())
    assert torch.equal(db.cpu(), d.cpu().to(torch.bfloat16))


@pytest.mark.parametrize("shape", [(300, 1696, 208), (900, 2064, 400), (13, 6160, 1552), (100, 272, 656),
                                   (200, 1024, 1072), (4160, 4096, 144)])
@pytest.mark.parametrize("fmt,layout", [("e4m3", P.LayoutSku.Rrr), ("e5m2", P.LayoutSku.Rcr)])
def test_fp8_out_depth_tails(gpu, shape, fmt, layout):
    S.test_fp8_out_with_c_sweep(gpu, shape, fmt, layout)


@pytest.mark.parametrize("shape", [(300, 520, 208), (700, 1000, 336), (900, 2064, 400), (2300, 5008, 400), (257, 262, 48),
                                   (13, 6160, 304), (1, 272, 48), (100, 272, 656), (200, 1024, 1072), (428, 1440, 2752)])
def test_rrr_and_u8_depth_tails(gpu, shape):
    """s8 RRR tiles (128x256 to 256x256) and last rows, u8 RCR / RRR on edge
    tiles and partial last stages."""
    S.test_int8_rrr_bias_relu_sweep(gpu, shape)
    S.test_u8_rcr_sweep(gpu, shape)
    S.test_u8_rrr_sweep(gpu, shape, False)


@pytest.mark.parametrize("shape", [(300, 520, 208), (900, 2072, 400), (1500, 3000, 336), (700, 4100, 1040), (13, 6160, 304),
                                   (100, 272, 656), (40, 8200, 144)])
@pytest.mark.parametrize("kind", ["s8", "u8", "e4m3", "e5m2"])
def test_rrr_padded_pitch(gpu, shape, kind):
    """B as the last columns of a wider tensor with more k-rows behind it: what
    surrounds the view (127, 255, NaN codes) stays out of the result, which is
    that of a dense copy on the same kernel, bit for bit."""
    m, n, k = shape
    print(f"case: rrr padded pitch {kind} {shape}", flush=True)
    g = torch.Generator()
    g.manual_seed(m + n + k)
    E = P.ElementKind
    el, fill, code = {"s8": (E.S8, 0x7f, torch.int8), "u8": (E.U8, 0xff, torch.uint8),
                      "e4m3": (E.Fp8E4M3, 0x7f, torch.float8_e4m3fn), "e5m2": (E.Fp8E5M2, 0x7e, torch.float8_e5m2)}[kind]
    lead = 48
    wide = torch.full((k + 128, lead + (n + 15) // 16 * 16), fill, dtype=torch.uint8)
    # finite FP8 codes below 2 in magnitude
    wide[:k, lead:lead + n] = torch.randint(0, 256, (k, n), dtype=torch.uint8, generator=g) & (0xff if kind[1] == "8" else 0xbf)
    wide = wide.to("cuda:0").view(code)
    a = torch.randint(0, 256, (m, k), dtype=torch.uint8, generator=g) & (0xff if kind[1] == "8" else 0xbf)
    a = a.to("cuda:0").view(code)
    if kind[1] == "8":
        plan = P.IntGemmPlan.select(P.IntGemmDescriptor(m, n, k, layout=P.LayoutSku.Rrr, element=el, output=el))
        alpha = 2e-4 if kind == "s8" else 1.0 / (128.0 * k)
    else:
        plan = P.Fp8GemmPlan.select(P.Fp8GemmDescriptor(m, n, k, layout=P.LayoutSku.Rrr, element=el, output=el))
        alpha = 0.25
    ldd = (n + 15) // 16 * 16

    def run(b):
        d = torch.zeros((m, ldd), dtype=torch.uint8, device="cuda:0").view(code)
        plan.run(a, b, d[:, :n], alpha=alpha)
        sync()
        return d.view(torch.uint8).cpu()

    view = wide[:k, lead:lead + n]
    dense = torch.zeros((k, ldd), dtype=torch.uint8, device="cuda:0").view(code)[:, :n]   # pitch a multiple of 16
    dense.view(torch.uint8).copy_(view.view(torch.uint8))
    got = run(view)
    assert torch.equal(got, run(dense))
    if kind[1] != "8":
        assert not bool(got.view(code).float().isnan().any())
        exact = alpha * (a.double().cpu() @ view.double().cpu())
        big = exact.abs() > 1.0
        err = (got.view(code)[:, :n].double() - exact).abs()
        step = 2.0 ** -3 if kind == "e4m3" else 2.0 ** -2      # spacing of the format, relative
        assert bool((err[big] <= step * exact.abs()[big]).all())
    else:
        exact = alpha * (a.double().cpu() @ view.double().cpu())
        lo, hi = (-128, 127) if kind == "s8" else (0, 255)
        assert bool(((got.view(code)[:, :n].double() - exact.clamp(lo, hi)).abs() <= 0.51).all())


# experts' row counts (ends of 64- and 128-row tiles, empty experts, more than
# 64 experts), N and K in bytes off 256 / 128
MOE_CASES = [([64, 1, 0, 129, 65, 300], 328, 208), ([3] * 70 + [0] * 30 + [200] * 3, 136, 80),
             ([700, 0, 641, 1200], 2312, 1040), ([2000, 1900, 1800, 2048], 2056, 272), ([90] * 16, 1408, 336),
             ([5, 0, 17, 1, 33], 360, 1040), ([1, 0, 1], 72, 48), ([20, 12], 1416, 3088)]


@pytest.mark.parametrize("case", MOE_CASES)
def test_moe_s8_tiles_and_depth_tails(gpu, case):
    counts, n, k = case
    print(f"case: moe s8 rows={counts[:8]} n={n} k={k}", flush=True)
    tokens, routing = _block_routing(counts, seed=n + k)
    _moe_run(tokens=tokens, E=len(counts), topk=1, n=n, k=k, seed=n, routing=routing)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("t", ["bf16", "f16"])
@pytest.mark.parametrize("shape", [(150, 8, 2, 328, 104), (40, 70, 3, 136, 264), (600, 4, 2, 264, 520), (12, 6, 2, 72, 136)])
def test_moe_float_tiles_and_depth_tails(gpu, shape, t, weighted):
    tokens, e, topk, n, k = shape
    print(f"case: moe {t} {shape} weighted={weighted}", flush=True)
    g = rng(tokens + e + n + k)
    sid, eid = moe_routing(tokens, e, topk, seed=tokens)[:2]
    rows = tokens * topk
    x = g.standard_normal((rows if weighted else tokens, k)).astype(np.float32)
    w = (g.standard_normal((e, n, k)) / np.sqrt(k)).astype(np.float32)
    tw = g.uniform(0.1, 1.0, rows).astype(np.float32) if weighted else None
    W._check(*W._run(t, x, w, sid, eid, topk, tw, rows), t)


@pytest.mark.parametrize("t", ["bf16", "f16"])
@pytest.mark.parametrize("counts,n,k", [([65, 1, 0, 130], 264, 136), ([33] * 12, 1408, 336), ([100, 300], 2312, 264)])
def test_moe_float_weights_of_padding_rows(gpu, counts, n, k, t):
    """Weighted pairs on tiles that end in padding rows: the weights are the
    first elements of the operand and the ids of a padding row have no weight."""
    print(f"case: moe {t} weighted, rows={counts[:4]} n={n} k={k}", flush=True)
    g = rng(n + k)
    rows = sum(counts)
    sid = g.permutation(rows).astype(np.int32)
    eid = np.repeat(np.arange(len(counts), dtype=np.int32), counts)
    x = g.standard_normal((rows, k)).astype(np.float32)
    w = (g.standard_normal((len(counts), n, k)) / np.sqrt(k)).astype(np.float32)
    W._check(*W._run(t, x, w, sid, eid, 1, g.uniform(0.1, 1.0, rows).astype(np.float32), rows), t)


@pytest.mark.parametrize("shape", [(1, 16), (5, 1040), (4097, 4672), (300, 3072), (130, 8176), (64, 11008), (7, 4080)])
def test_gemv_s8w_depth_tails(gpu, shape):
    print(f"case: gemv_s8w depth tail {shape}", flush=True)
    w, scale, xb = _gemv_inputs(*shape, seed=shape[0] + shape[1])
    _gemv_check(_gemv_run(w, scale, xb), w, scale, xb)


@pytest.mark.parametrize("dtype,n,k,batch", [(torch.bfloat16, 4096, 8199, 8), (torch.float32, 4100, 4099, 8)])
def test_gemv_dense_tall_slices(gpu, dtype, n, k, batch):
    """Split-K slices of several row groups, the last one short (f32 sums)."""
    print(f"case: gemv_dense {dtype} {batch}x{k}x{n}", flush=True)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(n + k)
    a = torch.empty((batch, k), dtype=dtype, device="cuda:0").normal_(generator=g)
    b = torch.empty((batch, k, n), dtype=dtype, device="cuda:0").normal_(0.0, k ** -0.5, generator=g)
    d = torch.empty((batch, n), dtype=dtype, device="cuda:0")
    plan = P.GemvDensePlan.select(P.GemvDenseDescriptor(n, k, batch), dtype)
    ws = torch.empty(plan.workspace_size(), dtype=torch.uint8, device="cuda:0")
    plan.run(a, b, d, lda=k, stride_a=k, ldb=n, stride_b=k * n, ldd=n, stride_d=n, workspace=ws)
    sync()
    for i in range(batch):
        x, w = a[i].double(), b[i].double()
        exact, mag = x @ w, x.abs() @ w.abs()
        # f32 sums of k products in chains of at most 128 + 64 + 16 additions, one output rounding
        bound = 208 * 2.0 ** -24 * mag + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * exact.abs()
        assert bool(((d[i].double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 8), (5, 512), (7, 520), (3, 2056), (256, 4096), (257, 4104), (2, 16384), (1, 16392), (300, 9000)])
def test_quantize_row_widths(gpu, dtype, shape):
    """Every chunk count and both workgroup sizes of the vector quantizer."""
    G.test_quantize_per_token_bit_exact(gpu, dtype, shape)
