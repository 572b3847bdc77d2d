"""GEMM kernels on the GPU against float64 products, the oracle and the golden
fixtures (the reference's tests/test_matmul.py, plus the 1024^3 bf16 config)."""
import numpy as np
import pytest
import torch
from hypothesis import given, settings
from hypothesis import strategies as st

import oracle as O
from conftest import assert_within_bf16_ulps, load_golden, rel_err

pytestmark = pytest.mark.gpu


def _bf(t):
    return torch.from_numpy(np.asarray(t, np.float32)).to(torch.bfloat16).cuda()


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.parametrize("variant", ["naive", "blocked"])
@pytest.mark.parametrize("M,K,N", [(128, 128, 512), (256, 384, 1024), (200, 300, 130), (1, 7, 3)])
def test_matmul_fp32(rng, variant, M, K, N):
    from nkilab import ops

    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    assert rel_err(ops.matmul(a, b, variant=variant), a.astype(np.float64) @ b) < 1e-5


@pytest.mark.parametrize("variant", ["naive", "blocked"])
def test_matmul_bf16_accumulates_in_fp32(rng, variant):
    from nkilab import ops

    a = _bf(rng.standard_normal((256, 1024)))
    b = _bf(rng.standard_normal((1024, 1024)))
    ref = _np(a).astype(np.float64) @ _np(b)
    out = ops.matmul(a, b, variant=variant)
    assert out.dtype == torch.bfloat16
    assert rel_err(_np(out), ref) < 1e-2  # only the final bf16 rounding of C
    assert_within_bf16_ulps(_np(out), O.bf16_round(ref.astype(np.float32)), 1.0, 1e-3)


def test_matmul_1024_cubed_bf16_config():
    """M = N = K = 1024, A and B ~ N(0, 1) bf16 from seed 0: max relative error
    <= 3e-3 against the exact product (the bf16 rounding floor of this input is
    2.965e-3)."""
    from nkilab import ops, workloads

    a, b = (t.cuda() for t in workloads.matmul_inputs())
    out = _np(ops.matmul(a, b))
    exact = _np(a).astype(np.float64) @ _np(b).astype(np.float64)
    floor = rel_err(O.bf16_round(exact.astype(np.float32)), exact)
    err = rel_err(out, exact)
    assert err <= 3e-3, (err, floor)
    assert err <= floor * 1.01 + 1e-6, (err, floor)
    assert_within_bf16_ulps(out, O.bf16_round(exact.astype(np.float32)), 1.0, 1e-3)


def test_matmul_matches_golden_vectors():
    from nkilab import ops

    gd = load_golden("matmul")
    for tag, dt in (("f32", O.F32), ("f32b", O.F32), ("bf16", O.BF16)):
        to = (lambda x: torch.from_numpy(x).cuda()) if dt == O.F32 else _bf
        out = _np(ops.matmul(to(gd[f"{tag}_a"]), to(gd[f"{tag}_b"])))
        ref = gd[f"{tag}_c"]
        if dt == O.F32:
            assert rel_err(out, ref) < 1e-5
        else:
            assert_within_bf16_ulps(out, ref, 1.0, 1e-3)


@settings(max_examples=12, deadline=None)
@given(M=st.integers(1, 300), K=st.integers(1, 300), N=st.integers(1, 700))
def test_matmul_property_any_shape(M, K, N):
    from nkilab import ops

    r = np.random.default_rng(M * 1000003 + K * 1009 + N)
    a = r.uniform(-1, 1, (M, K)).astype(np.float32)
    b = r.uniform(-1, 1, (K, N)).astype(np.float32)
    out = ops.matmul(a, b)
    assert out.shape == (M, N)
    np.testing.assert_allclose(out, a.astype(np.float64) @ b, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_linear_layout_and_residual_epilogue(rng, dt):
    """C = A . W^T + R with W in nn.Linear [out, in] layout (the B^T kernel), and the
    bf16 -> fp32 output used for the decoder's residual stream."""
    from nkilab import ops

    M, K, N = 192, 320, 256
    a = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dt).cuda()
    w = torch.from_numpy(rng.standard_normal((N, K)).astype(np.float32)).to(dt).cuda()
    res = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).cuda()
    c = torch.empty((M, N), dtype=torch.float32, device="cuda")
    ops.linear_into(a, w, c, residual=res)
    ref = _np(a).astype(np.float64) @ _np(w).astype(np.float64).T + _np(res)
    assert rel_err(_np(c), ref) < 1e-5
    # the same product through gemm_into with b = w.t() (a column-major view)
    c2 = torch.empty((M, N), dtype=dt, device="cuda")
    ops.gemm_into(a, w.t(), c2)
    tol = 1e-5 if dt == torch.float32 else 1e-2
    assert rel_err(_np(c2), ref - _np(res)) < tol


def test_nonaligned_leading_dimensions(rng):
    from nkilab import ops

    base_a = torch.from_numpy(rng.standard_normal((100, 77)).astype(np.float32)).cuda()
    base_b = torch.from_numpy(rng.standard_normal((61, 90)).astype(np.float32)).cuda()
    a, b = base_a[:, :61], base_b[:, :45]  # lda 77, ldb 90, K 61: the general-stride kernel
    c = ops.matmul(a, b)
    ref = _np(a).astype(np.float64) @ _np(b)
    assert rel_err(_np(c), ref) < 1e-5


@pytest.mark.parametrize("M,K,N,out_dt,res", [(192, 320, 256, torch.bfloat16, False), (130, 64, 72, torch.bfloat16, True),
                                               (257, 128, 40, torch.float32, True), (1000, 256, 1536, torch.float32, True),
                                               (64, 96, 132, torch.float32, False)])
def test_staged_epilogue_matches_element_epilogue(rng, M, K, N, out_dt, res):
    """bf16 GEMMs whose outputs take the 16-byte staged epilogue (aligned rows)
    against the same product written into a view whose rows are not 16-byte
    aligned (the element epilogue): identical values, residual included."""
    from nkilab import ops

    a = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    w = torch.from_numpy(rng.standard_normal((N, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    r = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).to(out_dt).cuda() if res else None
    c = torch.empty((M, N), dtype=out_dt, device="cuda")
    ops.linear_into(a, w, c, residual=r)
    big = torch.empty((M, N + 1), dtype=out_dt, device="cuda")
    c_odd = big[:, 1:]  # data pointer off by one element, ld N + 1
    ops.linear_into(a, w, c_odd, residual=r)
    assert torch.equal(c, c_odd)
    ref = _np(a).astype(np.float64) @ _np(w).astype(np.float64).T + (_np(r) if res else 0)
    assert rel_err(_np(c), ref) < (1e-5 if out_dt == torch.float32 else 1e-2)


# Shapes the tile choice sends to 256x192, 256x256, 256x128 and 128x128 (in
# that order; rounds of 256 workgroups x measured cost per K-step), each with
# partial tiles at both edges of C; then long K-loops (hundreds of stage
# hand-overs) on 128x128, 256x128 and 64x128.
@pytest.mark.parametrize("M,K,N", [(2000, 136, 6104), (4000, 136, 4000), (2040, 136, 4088), (2000, 200, 2000),
                                   (2000, 5632, 2000), (2040, 2056, 4088), (1000, 3000, 1000)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_large_tile_gemms_with_ragged_edges(rng, M, K, N, layout):
    """bf16 GEMMs on the large tiles against a float64 product; the staged
    epilogue (aligned C) and the element epilogue (C one element off) agree
    exactly, residual included."""
    from nkilab import ops

    a = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    b = torch.from_numpy(rng.standard_normal((N, K) if layout == "nt" else (K, N)).astype(np.float32))
    b = b.to(torch.bfloat16).cuda()
    r = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).to(torch.bfloat16).cuda()
    run = (lambda c: ops.linear_into(a, b, c, residual=r)) if layout == "nt" else \
        (lambda c: ops.gemm_into(a, b, c, residual=r))
    c = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    run(c)
    big = torch.empty((M, N + 1), dtype=torch.bfloat16, device="cuda")
    run(big[:, 1:])
    assert torch.equal(c, big[:, 1:])
    bt = b.double().cpu() if layout == "nn" else b.double().cpu().t()
    ref = (a.double().cpu() @ bt + r.double().cpu()).numpy()
    assert rel_err(_np(c), ref) < 1e-2
    # one rounding of the fp32 sum: within one bf16 ulp of the exact value, plus
    # the fp32 accumulation error (~K * 2^-24 * |terms|) where C is near zero
    assert_within_bf16_ulps(_np(c), ref, 1, floor=2e-3)


@pytest.mark.parametrize("M,K,N", [(2048, 2048, 11264), (3000, 1024, 7000), (2000, 512, 11000)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float32])
def test_column_split_matches_column_slices(rng, M, K, N, layout, out_dt):
    """Shapes whose 256-row tiles leave a partial last round run as two
    launches over column ranges (2048 x 11264: 256 x 256 tiles over the first
    8192 columns, 256 x 128 over the rest).  Every column equals, bit for
    bit, what a GEMM over a slice of the columns computes, residual included,
    and is within one bf16 ulp of the float64 product."""
    from nkilab import ops

    a = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    b = torch.from_numpy(rng.standard_normal((N, K) if layout == "nt" else (K, N)).astype(np.float32))
    b = b.to(torch.bfloat16).cuda()
    r = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).to(out_dt).cuda()

    def run(bm, c, res):
        return ops.linear_into(a, bm, c, residual=res) if layout == "nt" else ops.gemm_into(a, bm, c, residual=res)

    c = torch.empty((M, N), dtype=out_dt, device="cuda")
    run(b, c, r)
    # slices of 2048 columns: their GEMMs take one-K-group tiles too, or the
    # element kernel for a [K, N] slice that is not 16-byte aligned, both
    # summing K in the same order (fewer columns would give the small
    # two-K-group tiles another sum order)
    for lo, hi in [(0, 2048), (N // 2 - 1088, N // 2 + 960), (N - 2048, N)]:
        bs = b[lo:hi] if layout == "nt" else b[:, lo:hi]
        cs = torch.empty((M, hi - lo), dtype=out_dt, device="cuda")
        run(bs, cs, r[:, lo:hi])
        assert torch.equal(c[:, lo:hi], cs), (lo, hi)
        bt = bs.double().cpu() if layout == "nn" else bs.double().cpu().t()
        ref = (a[:512].double().cpu() @ bt + r[:512, lo:hi].double().cpu()).numpy()  # first 512 rows
        if out_dt == torch.bfloat16:
            assert_within_bf16_ulps(_np(cs[:512]), ref, 1, floor=2e-3)
        else:
            assert rel_err(_np(cs[:512]), ref) < 1e-5


@pytest.mark.parametrize("M,K,N", [(2048, 2048, 5632), (300, 256, 96), (64, 128, 32), (1, 64, 64), (513, 384, 704)])
def test_gemm_swiglu_equals_gate_up_then_swiglu(rng, M, K, N):
    """The fused gate/up GEMM with SwiGLU in its epilogue is bit-identical to
    two bf16 linear layers followed by the SwiGLU kernel (model.py:88), and
    within bf16 tolerance of the float64 product."""
    from nkilab import ops

    h = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    wg = torch.from_numpy((0.05 * rng.standard_normal((N, K))).astype(np.float32)).to(torch.bfloat16).cuda()
    wu = torch.from_numpy((0.05 * rng.standard_normal((N, K))).astype(np.float32)).to(torch.bfloat16).cuda()
    fused = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    ops.gemm_swiglu_into(h, ops.pack_gate_up(wg, wu), fused)
    gate, up, act = (torch.empty((M, N), dtype=torch.bfloat16, device="cuda") for _ in range(3))
    ops.linear_into(h, wg, gate)
    ops.linear_into(h, wu, up)
    ops.swiglu_into(gate, up, act)
    assert torch.equal(fused, act)
    g64 = _np(h).astype(np.float64) @ _np(wg).astype(np.float64).T
    u64 = _np(h).astype(np.float64) @ _np(wu).astype(np.float64).T
    ref = g64 / (1 + np.exp(-g64)) * u64
    assert rel_err(_np(fused), ref) < 2e-2


@pytest.mark.parametrize("M,K,N,off", [
    (1, 4, 4, 0), (33, 36, 28, 4), (32, 64, 32, 0), (65, 132, 100, 8), (300, 256, 1024, 0),  # one round: 32x64, 64x64
    (1000, 96, 1028, 0), (700, 64, 4064, 4), (2049, 36, 2052, 0),                            # 64x64, 64x128, 128x128
    (33, 35, 28, 0), (33, 36, 27, 0), (33, 36, 28, 3)])                                      # the two-GEMM path
def test_gate_up_fp32(M, K, N, off):
    """The fp32 gate/up GEMM over two weights, every tile and the operands it
    leaves to two GEMMs, as views `off` elements into wider rows of NaN (so that
    anything read past K would show), against float64: silu has a slope of at
    most 1.1, and gate and up are within K roundings of 2^-24 of the sums of
    |a b|; 2^-20 covers the exponential, the division and the product."""
    from nkilab import ops

    g = torch.Generator(device="cuda").manual_seed(M * 31 + K * 7 + N)

    def operand(r, c):
        buf = torch.full((r, c + (12 if off else 0)), float("nan"), device="cuda")
        v = buf[:, off:off + c]
        v.copy_(torch.randn(r, c, generator=g, device="cuda"))
        return v

    a, wg, wu = operand(M, K), operand(N, K), operand(N, K)
    cb = torch.full((M, N + 8), 5.0, device="cuda")
    c = cb[:, 4:N + 4]
    ops.gate_up_into(a, wg, wu, c)
    gate, up = (a.double() @ w.double().t() for w in (wg, wu))
    eg, eu = ((K + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t()) for w in (wg, wu))
    silu = gate * torch.sigmoid(gate)
    bound = 1.1 * eg * (up.abs() + eu) + silu.abs() * eu + 2.0 ** -20 * (silu * up).abs() + 2.0 ** -126
    assert ((c.double() - silu * up).abs() <= bound).all()
    assert (cb[:, :4] == 5).all() and (cb[:, N + 4:] == 5).all()


@pytest.mark.parametrize("M,K,N", [(16, 1504, 2048), (16, 1508, 2048), (16, 4064, 2048), (200, 2048, 1024)])
def test_gate_up_fp32_around_the_k_split(M, K, N):
    """The last K taken by one GEMM whatever the tiles, the first whose two
    GEMMs split it, longer ones with and without a split."""
    test_gate_up_fp32(M, K, N, 0)


def test_gemm_swiglu_rejects_bad_shapes():
    from nkilab import ops

    h = torch.zeros((16, 64), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((2 * 48, 64), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError, match="multiple of 32"):
        ops.gemm_swiglu_into(h, w, torch.empty((16, 48), dtype=torch.bfloat16, device="cuda"))


@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_batched_gemm_on_large_tiles(rng, layout):
    """Three independent products in one launch (blockIdx.z over the batch,
    per-batch strides), a shape the tile choice sends to 256x128 and with
    partial tiles at both edges: each batch entry against its own float64
    product, residual included."""
    from nkilab import _lib
    from nkilab._tensors import stream_handle

    B, M, N, K = 3, 1500, 1600, 136
    a = torch.from_numpy(rng.standard_normal((B, M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    bsh = (B, N, K) if layout == "nt" else (B, K, N)
    b = torch.from_numpy(rng.standard_normal(bsh).astype(np.float32)).to(torch.bfloat16).cuda()
    r = torch.from_numpy(rng.standard_normal((B, M, N)).astype(np.float32)).to(torch.bfloat16).cuda()
    c = torch.empty((B, M, N), dtype=torch.bfloat16, device="cuda")
    ldb = K if layout == "nt" else N
    _lib.call("nkl_gemm", a.data_ptr(), b.data_ptr(), c.data_ptr(), r.data_ptr(), M, N, K, K, ldb, N, N,
              1 if layout == "nt" else 0, B, M * K, bsh[1] * bsh[2], M * N, M * N, 1, 1, 0, stream_handle())
    torch.cuda.synchronize()
    for i in range(B):
        bt = b[i].double().cpu() if layout == "nn" else b[i].double().cpu().t()
        ref = (a[i].double().cpu() @ bt + r[i].double().cpu()).numpy()
        assert_within_bf16_ulps(_np(c[i]), ref, 1, floor=2e-3)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,off", [
    (1, 1, 1, 0), (1, 7, 3, 1), (33, 5, 2, 0), (31, 63, 65, 3), (64, 64, 64, 1), (65, 129, 33, 0),  # K and N tails
    (300, 256, 1024, 0), (300, 1024, 256, 0), (1000, 1000, 1000, 0), (2000, 96, 1000, 0),           # fp32 tile choice
    (130, 515, 2050, 1), (2049, 71, 2051, 0), (8, 8021, 64, 0), (16, 4096, 260, 0), (9, 3333, 31, 5),  # K split
    (2945, 137, 2947, 0)])                                                                           # packed operands
def test_gemm_any_shape_and_alignment(dt, M, K, N, off):
    """Every staging path, tile choice, K split and operand copy, both layouts
    and a residual, as views `off` elements into wider rows of NaN (so that
    anything read past K or N would show), against float64: within K roundings
    of 2^-24 of the sum of |a b|, plus one rounding to the output type."""
    from nkilab import ops

    g = torch.Generator(device="cuda").manual_seed(M * 31 + K * 7 + N)

    def operand(r, c):
        buf = torch.full((r, c + (9 if off else 0)), float("nan"), dtype=dt, device="cuda")
        v = buf[:, off:off + c]
        v.copy_(torch.randn(r, c, generator=g, device="cuda"))
        return v

    u = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dt]
    for bt in (False, True):
        a, b, r = operand(M, K), operand(N, K) if bt else operand(K, N), operand(M, N)
        bd = b.double().t() if bt else b.double()
        ref, mag = a.double() @ bd, a.double().abs() @ bd.abs()
        run = ops.linear_into if bt else ops.gemm_into
        for res in (None, r):
            cb = torch.full((M, N + 3), 5.0, dtype=dt, device="cuda")
            c = cb[:, 1:N + 1]
            run(a, b, c, residual=res)
            want = ref if res is None else ref + res.double()
            bound = (K + 2) * 2.0 ** -24 * (mag + want.abs()) + u * want.abs() + 2.0 ** -24
            assert ((c.double() - want).abs() <= bound).all(), (bt, res is not None)
            assert (cb[:, 0] == 5).all() and (cb[:, N + 1:] == 5).all()
            again = torch.empty(M, N, dtype=dt, device="cuda")
            run(a, b, again, residual=res)
            assert torch.equal(again, c)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(1001, 77, 1301), (1537, 65, 1999)])  # 64x128; 128x128 in 16 bits, 64x128 in fp32
def test_gemm_unaligned_tiles(dt, M, K, N):
    test_gemm_any_shape_and_alignment(dt, M, K, N, 1)


@pytest.mark.parametrize("b_trans", [0, 1])
@pytest.mark.parametrize("dt,dt_out", [(0, 0), (1, 1), (1, 0), (2, 2), (2, 0)])
@pytest.mark.parametrize("M,N", [(40, 24), (300, 1024), (2048, 4096)])
def test_gemm_abi_with_no_k(b_trans, dt, dt_out, M, N):
    """K = 0 through the C entries: C is the residual, or zeros, on every tile."""
    from nkilab import _lib
    from nkilab._tensors import stream_handle

    t = {0: torch.float32, 1: torch.bfloat16, 2: torch.float16}
    a, b = (torch.full((r, 8), float("nan"), dtype=t[dt], device="cuda") for r in (M, N))
    b = b if b_trans else b.view(8, N)
    r = torch.randn((M, N), device="cuda").to(t[dt_out])
    for res in (None, r):
        c = torch.full((M, N + 8), 5.0, dtype=t[dt_out], device="cuda")
        args = (a.data_ptr(), b.data_ptr(), c.data_ptr(), None if res is None else res.data_ptr())
        _lib.call("nkl_gemm", *args, M, N, 0, 8, 8 if b_trans else N, N + 8, N, b_trans, 1, 0, 0, 0, 0, dt, dt_out, 0,
                  stream_handle())
        assert torch.equal(c[:, :N], torch.zeros_like(r) if res is None else r) and (c[:, N:] == 5).all()
        c.fill_(5)
        _lib.call("nkl_gemm_ws", *args, None, 0, M, N, 0, 8, 8 if b_trans else N, N + 8, N, b_trans, dt, dt_out,
                  stream_handle())
        assert torch.equal(c[:, :N], torch.zeros_like(r) if res is None else r) and (c[:, N:] == 5).all()


@pytest.mark.parametrize("M,K,N", [(1 << 20, 1024, 129), (130, 8192, 131073)])  # A, then B, of 2 GiB
def test_gemm_odd_columns_past_2_gib(M, K, N):
    """An operand of 2 GiB with N off a vector, with and without a residual:
    every element against fp32 products of row ranges, nothing written past the
    columns or the last row of C.  bf16 inputs are exact in fp32; both sides sum
    K products in fp32 (K 2^-24 of the sum of |a b| each) and C is rounded once
    to bf16."""
    from nkilab import ops

    free = torch.cuda.mem_get_info()[0]
    if free < 16 << 30:
        pytest.skip(f"needs 16 GiB of GPU memory, {free >> 30} free")
    g = torch.Generator(device="cuda").manual_seed(7)
    a, b = (torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(generator=g) for s in ((M, K), (K, N)))
    r = torch.empty((M, N), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    step = 1 << 17
    bf = b.float()
    for res in (None, r):
        cb = torch.full((M + 1, N + 3), 5.0, dtype=torch.bfloat16, device="cuda")
        ops.gemm_into(a, b, cb[:M, :N], residual=res)
        assert (cb[:, N:] == 5).all() and (cb[M] == 5).all()
        for m in range(0, M, step):
            want = a[m:m + step].float() @ bf
            if res is not None:
                want += res[m:m + step].float()
            mag = a[m:m + step].float().abs() @ bf.abs()
            bound = 2 * (K + 2) * 2.0 ** -24 * (mag + want.abs()) + 2.0 ** -8 * want.abs()
            assert ((cb[m:min(m + step, M), :N].float() - want).abs() <= bound).all(), (m, res is not None)


@pytest.mark.parametrize("K", [1, 13])  # nothing staged; staged through registers
@pytest.mark.parametrize("columns", [False, True])
def test_gemm_tiles_past_one_launch(K, columns):
    """One column (or row) of more elements than the 64x64 tiles of one launch
    hold (HIP's limit of 2^32 threads), with a residual: multiples of 1/8 below
    16, whose products and sums fp32 holds exactly, rounded once to bf16."""
    from nkilab import ops

    n = (1 << 30) + 65
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    if free < 64 << 30:
        pytest.skip(f"needs 64 GiB of GPU memory, {free >> 30} free")

    def eighths(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="cuda").random_(-127, 128).mul_(0.125)

    x, s, r = eighths(n, K), eighths(1, K), eighths(n)
    c = torch.full((n + 8,), 5.0, dtype=torch.bfloat16, device="cuda")
    shape = (1, n) if columns else (n, 1)
    ops.linear_into(*((s, x) if columns else (x, s)), c[:n].view(shape), residual=r.view(shape))
    step = 1 << 27
    for i in range(0, n, step):
        want = (x[i:i + step].float() * s.float()).sum(1) + r[i:i + step].float()
        assert torch.equal(c[i:min(i + step, n)], want.bfloat16()), i
    assert (c[n:] == 5).all()
    del x, c, r
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(2945, 137, 2947), (8, 8021, 64)])  # packed operands; K split
def test_gemm_without_memory_for_a_workspace(dt, M, K, N, monkeypatch):
    """A product whose workspace cannot be allocated is computed without one."""
    from nkilab import ops

    asked = []

    def none_left(nbytes, dev):
        asked.append(nbytes)
        raise torch.OutOfMemoryError("no memory left")

    monkeypatch.setattr(ops, "workspace", none_left)
    test_gemm_any_shape_and_alignment(dt, M, K, N, 0)
    assert asked or (dt == torch.float32 and N > 64)  # (fp32 operands are not packed)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [
    (1030, 1, 1301), (1030, 12, 1301), (1030, 13, 1300), (1030, 17, 1301), (1030, 20, 1301), (1030, 21, 1301),
    (1030, 8, 1301), (1030, 16, 1301), (2050, 24, 2049), (1030, 32, 1300), (1030, 33, 1301), (1030, 57, 1301),  # fp32
    (1030, 36, 1300), (2050, 36, 1300), (2050, 64, 1300), (2050, 384, 1300), (16500, 100, 60), (2050, 388, 1300),
    (65540, 70, 129), (65540, 70, 128)])                                             # 16 bits: packed, not packed
def test_gemm_short_k(dt, M, K, N):
    """Short K over more than a round of tiles: the unstaged kernel, one or two
    checked K-steps, two sums, and the K on both sides of each choice."""
    test_gemm_any_shape_and_alignment(dt, M, K, N, 0)


def test_gemm_workspace_is_for_the_shapes_that_use_it():
    """No workspace where one launch serves (the common aligned shapes); the K
    split and the packed operands ask for one, and refuse a smaller one."""
    from nkilab import _lib

    L = _lib.lib()
    a = torch.empty(1 << 24, dtype=torch.bfloat16, device="cuda")
    p = a.data_ptr()
    assert L.nkl_gemm_workspace_bytes(p, p, 1024, 1024, 1024, 1024, 1024, 0, 1, 1) == 0
    assert L.nkl_gemm_workspace_bytes(p, p, 1000, 1301, 777, 777, 1301, 0, 1, 1) == 0
    need = L.nkl_gemm_workspace_bytes(p, p, 8, 64, 8064, 8064, 64, 0, 1, 1)
    assert need >= 2 * 8 * 64 * 4
    assert L.nkl_gemm_workspace_bytes(p, p, 2945, 2947, 137, 137, 2947, 0, 1, 1) > 0
    assert L.nkl_gemm_ws(p, p, p, None, p, need - 1, 8, 64, 8064, 8064, 64, 64, 0, 0, 1, 1, None) == -4
