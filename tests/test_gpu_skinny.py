"""The streaming kernel for few rows (skinny_kernel): equal to the oracle at
the edges of its tiles, and to the path it takes calls from in every form the
device entries accept (types, unaligned buffers, ragged sizes, the fused FFN,
the allocation-free entry). Bit for bit: the sums are exact integers and the
dequantization is the same sequence of single-rounding operations."""
import ctypes

import numpy as np
import pytest

from oracle import oracle
from open_rknpu2_lm_infer_amd import _ffi as F
from open_rknpu2_lm_infer_amd import device as D
from open_rknpu2_lm_infer_amd import npu
from tests import refdata as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    return D.DeviceContext(8)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# K: one unit; an odd count of W4 planes (640 + 64, 100 -> 128, 12000 -> 12032);
# the narrow window's last unit and the wide one's first; more units than the
# wide window holds (reloaded). N: one tile, ragged and padded columns, two
# column tiles per block (more than 4096 columns).
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("k,n", [(64, 16), (100, 100), (704, 768), (2560, 320), (2624, 1003), (12000, 64), (192, 4352)])
def test_skinny_matches_oracle(ctx, bits, k, n):
    codes, scales = R.weights(21, f"sk{bits}-{k}-{n}", bits, k, n)
    w = ctx.weights(bits, dev(codes), dev(scales))
    for rows in (2, 5, 8, 16, 17, 32, 33, 64, 65, 128, 129, 256):
        x = R.activations(21, f"sk-x{rows}-{k}", rows, k)
        for swiglu in (False, True)[:2 if n % 64 == 0 else 1]:
            want = oracle.linear_swiglu(codes, scales, x) if swiglu else oracle.linear(codes, scales, x)
            print(f"W{bits} K={k} N={n} rows={rows} swiglu={swiglu}", flush=True)
            y = torch.full(want.shape, float("nan"), device="cuda")
            with D.plan_switch("HM_SKINNY", 1):
                D.linear(ctx, w, dev(x), y, rows, swiglu=swiglu)
            torch.cuda.synchronize()
            assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [3, 8, 20, 70])
def test_skinny_equals_the_other_path_in_every_form(ctx, bits, rows):
    """Input and output types, bases off 16-byte alignment, K and N off every
    multiple: HM_SKINNY 1 against 0."""
    for k, n in ((512, 320), (333, 321)):
        codes, scales = R.weights(22, f"skf{bits}-{k}-{n}", bits, k, n)
        w = ctx.weights(bits, dev(codes), dev(scales))
        x = R.activations(22, f"skf-x{rows}-{k}", rows, k)
        for swiglu in (False, True)[:2 if n % 64 == 0 else 1]:
            width = n // 2 if swiglu else n
            for x_type in (torch.float16, torch.float32):
                for y_type in (torch.float16, torch.float32):
                    for off in (0, 1):
                        xb = torch.zeros(rows * k + off, dtype=x_type, device="cuda")
                        xin = xb[off:].view(rows, k)
                        xin.copy_(dev(x))
                        got = []
                        for skinny in (1, 0):
                            buf = torch.zeros(rows * width + off, dtype=y_type, device="cuda")
                            with D.plan_switch("HM_SKINNY", skinny):
                                D.linear(ctx, w, xin, buf[off:].view(rows, width), rows, swiglu=swiglu)
                            torch.cuda.synchronize()
                            got.append(buf.cpu())
                        assert torch.equal(got[0], got[1]), (k, n, swiglu, x_type, y_type, off)


@pytest.mark.parametrize("rows", [4, 8, 16, 40, 64, 130, 256])
@pytest.mark.parametrize("gu_bits,dn_bits", [(4, 4), (4, 8), (8, 8)])
def test_skinny_ffn_row_maxima(ctx, rows, gu_bits, dn_bits):
    """The middle's row maxima pass from the gate_up launch to the
    requantization as one partial per block (f = 2080: 130 blocks), whichever
    of the two launches runs on which kernel; three calls in a row."""
    h, f = 384, 2080
    gc, gs = R.weights(23, f"skg{gu_bits}", gu_bits, h, 2 * f)
    dc, ds = R.weights(23, f"skd{dn_bits}", dn_bits, f, h)
    gu, dn = ctx.weights(gu_bits, dev(gc), dev(gs)), ctx.weights(dn_bits, dev(dc), dev(ds))
    for rep, skinny in enumerate((1, -1, 0)):
        x = R.activations(23, f"skffn-x{rows}-{rep}", rows, h)
        y = torch.empty(rows, h, dtype=torch.float32, device="cuda")
        with D.plan_switch("HM_SKINNY", skinny):
            D.ffn(ctx, gu, dn, dev(x), y, rows)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), oracle.ffn(gc, gs, dc, ds, x)), skinny


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [8, 16, 100, 256])
def test_skinny_static_entry(ctx, bits, rows):
    """rk_npu_hip_linear_run_static (no workspace): the same result, plain
    and SwiGLU (which wants no row maxima there)."""
    k, n = 640, 512
    codes, scales = R.weights(24, f"sks{bits}", bits, k, n)
    w = ctx.weights(bits, dev(codes), dev(scales))
    x = R.activations(24, f"sks-x{rows}", rows, k)
    xd = dev(x)
    for epi, width, want in ((F.RK_NPU_HIP_PLAIN, n, oracle.linear(codes, scales, x)),
                             (F.RK_NPU_HIP_SWIGLU, n // 2, oracle.linear_swiglu(codes, scales, x))):
        y = torch.empty(rows, width, device="cuda")
        npu.check(F.lib().rk_npu_hip_linear_run_static(w.handle.raw, bits, ctypes.c_void_p(xd.data_ptr()),
                                                       F.RK_NPU_HIP_F32, ctypes.c_void_p(y.data_ptr()),
                                                       F.RK_NPU_HIP_F32, rows, epi, D.current_stream()), "static")
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("f", [1056, 2080])
@pytest.mark.parametrize("gu_bits,dn_bits", [(4, 4), (8, 8)])
def test_ffn_row_maxima_after_a_gemv_call(ctx, gu_bits, dn_bits, f):
    """One workspace pair for every row count, its gate_up width off 256
    (padding columns): after a call of a few much larger rows on the GEMV, which
    leaves its maxima in the same buffer, later calls requantize the middle by
    their own rows' maxima only."""
    h, most = 512, 64
    gc, gs = R.weights(25, f"skag{gu_bits}-{f}", gu_bits, h, 2 * f)
    dc, ds = R.weights(25, f"skad{dn_bits}-{f}", dn_bits, f, h)
    gu, dn = ctx.weights(gu_bits, dev(gc), dev(gs)), ctx.weights(dn_bits, dev(dc), dev(ds))
    gws, dws = ctx.workspace(gu_bits, most, h, 2 * f), ctx.workspace(dn_bits, most, f, h)
    for first in (1, 2, 4):
        for rows in (3, 8, 16, 64):
            for n, scale in ((first, 100.0), (rows, 1.0)):
                print(f"W{gu_bits}/W{dn_bits} f={f} {n} rows after {first}", flush=True)
                x = R.activations(25, f"ska-x{n}-{first}-{rows}", n, h) * np.float32(scale)
                y = torch.empty(n, h, dtype=torch.float32, device="cuda")
                D.ffn(ctx, gu, dn, dev(x), y, n, gws=gws, dws=dws)
                torch.cuda.synchronize()
                assert np.array_equal(y.cpu().numpy(), oracle.ffn(gc, gs, dc, ds, x))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [1, 2, 4, 8, 16])
def test_forced_gemm_is_the_tiled_one(ctx, bits, rows):
    """HM_FORCE_GEMM sends rows <= 8 to the tiled GEMM instead of the GEMV (more
    rows take what they take without it); HM_SKINNY=1 comes before it."""
    k, n = 512, 320
    codes, scales = R.weights(26, f"skfg{bits}", bits, k, n)
    w = ctx.weights(bits, dev(codes), dev(scales))
    x = R.activations(26, f"skfg-x{rows}", rows, k)
    ws = ctx.workspace(bits, 16, k, n)
    for skinny, kernel in ((-1, "gemm<" if rows <= 8 else "skinny<"), (1, "skinny<")):
        y = torch.empty(rows, n, device="cuda")
        with D.plan_switch("HM_FORCE_GEMM", 1), D.plan_switch("HM_SKINNY", skinny), D.KernelProfile(16) as p:
            D.linear(ctx, w, dev(x), y, rows, ws=ws)
            torch.cuda.synchronize()
        assert [s["name"].startswith(kernel) for s in p.stats if s["kind"] < 2] == [True], p.stats
        assert np.array_equal(y.cpu().numpy(), oracle.linear(codes, scales, x))


@pytest.mark.parametrize("k,n,bits,rows,swiglu,kernel", [
    # blocks of up to 16, 32, 64 and 256 rows at the last number a CU and past it
    (512, 24576, 4, 16, False, "skinny"), (512, 24832, 4, 16, False, "gemm"), (512, 8448, 8, 16, False, "gemm"),
    (1024, 16384, 8, 16, False, "skinny"), (512, 16384, 4, 32, False, "skinny"), (1024, 24576, 4, 32, False, "gemm"),
    (512, 8192, 8, 32, False, "skinny"), (512, 16384, 8, 32, False, "gemm"), (512, 8192, 4, 64, False, "skinny"),
    (512, 16384, 4, 64, False, "gemm"), (1536, 8448, 4, 64, False, "skinny"), (512, 8448, 8, 48, False, "gemm"),
    (512, 8192, 4, 128, False, "skinny"), (512, 16384, 4, 128, False, "gemm"), (512, 8192, 8, 128, False, "gemm"),
    (512, 2560, 8, 128, False, "skinny"), (512, 2560, 8, 256, False, "gemm"), (1536, 8192, 8, 128, False, "skinny"),
    (512, 8192, 8, 128, True, "skinny"), (512, 16384, 8, 128, True, "gemm"), (512, 16384, 4, 128, True, "skinny"),
    (512, 24576, 8, 64, True, "skinny"), (512, 32768, 8, 64, True, "gemm"), (512, 33024, 4, 20, True, "gemm"),
    # long K
    (8192, 512, 4, 64, False, "skinny"), (8192, 512, 8, 64, False, "gemm"), (8192, 512, 4, 65, False, "gemm"),
    # against the GEMV
    (3072, 2304, 4, 4, False, "gemv"), (3072, 2560, 4, 4, False, "skinny"), (2048, 512, 4, 3, False, "skinny"),
    (1536, 512, 8, 8, False, "gemv"), (2048, 512, 8, 8, False, "skinny"), (512, 512, 8, 5, True, "skinny"),
    (512, 8448, 8, 5, True, "gemv"), (2048, 512, 8, 4, False, "gemv"),
])
def test_dispatch_lines(ctx, k, n, bits, rows, swiglu, kernel):
    """Which kernel a call takes on either side of each line of the rule (256
    CUs), and that the other path gives the same bits there."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes lie at the lines of 256 CUs")
    g = torch.Generator(device="cuda").manual_seed(k + n)
    lo, hi = (-8, 8) if bits == 4 else (-127, 128)
    w = ctx.weights(bits, torch.randint(lo, hi, (k, n), generator=g, device="cuda", dtype=torch.int8),
                    torch.rand(n, generator=g, device="cuda") * 0.009 + 0.001)
    x = torch.randn(rows, k, generator=g, device="cuda")
    ws = ctx.workspace(bits, rows, k, n, cached=False)
    outs = []
    for skinny in (-1, 0 if kernel == "skinny" else 1):
        outs.append(torch.empty(rows, n // 2 if swiglu else n, device="cuda"))
        with D.plan_switch("HM_SKINNY", skinny), D.KernelProfile(16) as p:
            D.linear(ctx, w, x, outs[-1], rows, swiglu=swiglu, ws=ws)
            torch.cuda.synchronize()
        names = [s["name"] for s in p.stats if s["kind"] < 2]
        assert len(names) == 1 and names[0].startswith(kernel + "<") == (skinny == -1), (names, skinny)
    assert torch.equal(*outs)
