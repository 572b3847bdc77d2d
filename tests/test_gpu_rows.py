"""Row kernels on the GPU (softmax, RMSNorm, SwiGLU) against the oracle, torch and
the golden fixtures.  Tolerances follow the reference's tests
(tests/test_norm.py) for fp32; bf16 results must sit within one bf16 ulp of the
oracle's correctly rounded value."""
import numpy as np
import pytest
import torch

import oracle as O
from conftest import assert_within_bf16_ulps, load_golden, rel_err

pytestmark = pytest.mark.gpu


def _bf(t):
    return torch.from_numpy(np.asarray(t, np.float32)).to(torch.bfloat16).cuda()


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("R,D", [(128, 64), (1000, 2048), (5, 3), (3, 5000), (2, 20000)])
def test_softmax_matches_torch(rng, fused, R, D):
    from nkilab import ops

    x = (rng.standard_normal((R, D)) * 4).astype(np.float32)
    out = ops.softmax(x, fused=fused)
    assert out.dtype == np.float32 and out.shape == (R, D)
    ref = torch.softmax(torch.from_numpy(x), -1).numpy()
    np.testing.assert_allclose(out, ref, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(out, O.softmax_fused(x) if fused else O.softmax_unfused(x), rtol=1e-5, atol=1e-6)


def test_softmax_is_stable_for_large_logits(rng):
    from nkilab import ops

    x = (rng.standard_normal((256, 512)) * 1e4).astype(np.float32)
    out = ops.softmax(x)
    assert np.isfinite(out).all()
    np.testing.assert_allclose(out.sum(-1), 1.0, atol=1e-5)


@pytest.mark.parametrize("R,D,s", [(1, 1, 1.0), (400, 1023, 50.0), (37, 129, 0.1), (64, 777, 3.0)])
def test_softmax_rows_sum_to_one(R, D, s):
    from nkilab import ops

    x = (np.random.default_rng(R * 7 + D).standard_normal((R, D)) * s).astype(np.float32)
    out = ops.softmax(x)
    np.testing.assert_allclose(out.sum(-1), 1.0, atol=1e-5)
    assert (out >= 0).all()


@pytest.mark.parametrize("R,D", [(128, 256), (300, 1024), (7, 33)])
def test_rmsnorm_matches_torch(rng, R, D):
    from nkilab import ops

    x = rng.standard_normal((R, D)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, D).astype(np.float32)
    xt = torch.from_numpy(x)
    ref = (xt * torch.rsqrt(xt.pow(2).mean(-1, keepdim=True) + 1e-6) * torch.from_numpy(w)).numpy()
    assert rel_err(ops.rmsnorm(x, w), ref) < 1e-5


def test_rmsnorm_bf16(rng):
    from nkilab import ops

    x = _bf(rng.standard_normal((256, 512)))
    w = torch.ones(512, dtype=torch.bfloat16, device="cuda")
    xf = _np(x).astype(np.float64)
    ref = xf / np.sqrt((xf ** 2).mean(-1, keepdims=True) + 1e-6)
    out = ops.rmsnorm(x, w)
    assert out.dtype == torch.bfloat16 and out.is_cuda
    assert rel_err(_np(out), ref) < 1e-2


@pytest.mark.parametrize("R,D", [(64, 2048), (33, 520), (5, 77)])
def test_rmsnorm_bf16_activations_fp32_weight(rng, R, D):
    """bf16 x with an fp32 weight: the fp32 normalised row is multiplied by the
    fp32 weight and rounded once (norm.py:116), as the oracle does -- not by a
    weight first rounded to bf16."""
    from nkilab import ops

    x = _bf(rng.standard_normal((R, D)))
    w = torch.from_numpy(rng.uniform(0.5, 1.5, D).astype(np.float32)).cuda()
    out = ops.rmsnorm(x, w)
    assert out.dtype == torch.bfloat16
    ref = O.rmsnorm_fused(_np(x), w.cpu().numpy(), 1e-6, O.BF16)
    assert_within_bf16_ulps(_np(out), ref, 1.0, 1e-6)
    # rounding the weight to bf16 first gives a different result on some elements
    coarse = O.rmsnorm_fused(_np(x), O.bf16_round(w.cpu().numpy()), 1e-6, O.BF16)
    assert np.abs(ref - coarse).max() > 0


def test_swiglu_matches_torch(rng):
    from nkilab import ops

    g = rng.standard_normal((300, 1024)).astype(np.float32)
    u = rng.standard_normal((300, 1024)).astype(np.float32)
    ref = (torch.nn.functional.silu(torch.from_numpy(g)) * torch.from_numpy(u)).numpy()
    assert rel_err(ops.swiglu(g, u), ref) < 1e-5
    odd = rng.standard_normal(1001).astype(np.float32)  # not a multiple of the vector width
    np.testing.assert_allclose(ops.swiglu(odd, odd), O.swiglu_fused(odd, odd), rtol=1e-5, atol=1e-6)


def test_row_kernels_match_golden_vectors():
    from nkilab import ops

    gd = load_golden("rows")
    for tag, dt in (("f32", O.F32), ("f32b", O.F32), ("bf16", O.BF16), ("bf16r", O.BF16)):
        to = (lambda a: torch.from_numpy(a).cuda()) if dt == O.F32 else _bf
        x, w, g, u = (to(gd[f"{tag}_{k}"]) for k in ("x", "w", "g", "u"))
        got = {"softmax": ops.softmax(x), "softmax_unfused": ops.softmax(x, fused=False),
               "rmsnorm": ops.rmsnorm(x, w), "swiglu": ops.swiglu(g, u)}
        for k, v in got.items():
            ref = gd[f"{tag}_{k}"]
            if dt == O.F32:
                np.testing.assert_allclose(_np(v), ref, rtol=2e-5, atol=1e-6, err_msg=f"{tag}_{k}")
            else:
                assert_within_bf16_ulps(_np(v), ref, 1.0, 1e-6)


# --------------------------------------------- the 4096 x 2048 bf16 config --

@pytest.fixture(scope="module")
def rows_config():
    from nkilab import workloads

    x, w, gate, up = workloads.rows_inputs()
    return tuple(t.cuda() for t in (x, w, gate, up))


def test_softmax_config(rows_config):
    from nkilab import ops

    x = rows_config[0]
    out = _np(ops.softmax(x))
    xf = _np(x)
    assert np.abs(out - torch.softmax(torch.from_numpy(xf), -1).numpy()).max() <= 1e-2
    assert_within_bf16_ulps(out, O.softmax_fused(xf, O.BF16), 1.0, 1e-7)
    np.testing.assert_allclose(out.astype(np.float64).sum(-1), 1.0, atol=1e-2)


def test_rmsnorm_config(rows_config):
    from nkilab import ops

    x, w = rows_config[0], rows_config[1]
    out = _np(ops.rmsnorm(x, w, 1e-6))
    xf, wf = _np(x).astype(np.float64), _np(w).astype(np.float64)
    exact = xf / np.sqrt((xf ** 2).mean(-1, keepdims=True) + 1e-6) * wf
    assert rel_err(out, exact) < 1e-2
    assert_within_bf16_ulps(out, O.rmsnorm_fused(_np(x), _np(w), 1e-6, O.BF16), 1.0, 1e-6)


def test_swiglu_config(rows_config):
    from nkilab import ops

    g, u = rows_config[2], rows_config[3]
    out = _np(ops.swiglu(g, u))
    gf, uf = _np(g).astype(np.float64), _np(u).astype(np.float64)
    assert rel_err(out, gf / (1 + np.exp(-gf)) * uf) < 1e-2
    assert_within_bf16_ulps(out, O.swiglu_fused(_np(g), _np(u), O.BF16), 1.0, 1e-6)


def test_rmsnorm_fp32_input_to_bf16_output(rng):
    """The decoder's mixed path: an fp32 residual stream normalised into bf16."""
    from nkilab import ops

    x = torch.from_numpy(rng.standard_normal((64, 2048)).astype(np.float32)).cuda()
    w = torch.from_numpy(rng.uniform(0.5, 1.5, 2048).astype(np.float32)).cuda()
    y = torch.empty((64, 2048), dtype=torch.bfloat16, device="cuda")
    ops.rmsnorm_into(x, w, y, 1e-6)
    assert_within_bf16_ulps(_np(y), O.rmsnorm_fused(_np(x), _np(w), 1e-6, O.BF16), 1.0, 1e-6)


def test_strided_rows_and_async_tensors(rng):
    from nkilab import ops

    base = torch.from_numpy(rng.standard_normal((64, 300)).astype(np.float32)).cuda()
    x = base[:, :256]  # ld 300 > cols 256
    out = ops.softmax(x)
    assert out.is_cuda
    np.testing.assert_allclose(_np(out), torch.softmax(x.cpu(), -1).numpy(), rtol=1e-5, atol=1e-6)


# -------------------------------------------------- RoPE (not in the reference) --

@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
@pytest.mark.parametrize("H,S,d,pos0,base", [(2, 300, 128, 0, 10000.0), (4, 65, 64, 1000, 500000.0),
                                             (1, 7, 8, 5, 10000.0), (8, 2048, 128, 0, 10000.0)])
def test_rope_matches_oracle(rng, dt, H, S, d, pos0, base):
    """The RoPE kernel against the oracle (float64 angles).  fp32 outputs are
    within the fp32 angle error (relative 2e-7 of the angle, times the pair's
    norm); bf16 outputs within one bf16 step of the oracle's value plus that."""
    import torch

    import oracle as O
    from nkilab import ops

    x = rng.standard_normal((H, S, d)).astype(np.float32)
    tdt = getattr(torch, dt)
    xt = torch.from_numpy(x).to(tdt).cuda()
    out = ops.rope_into(xt, torch.empty_like(xt), base, pos0).float().cpu().numpy()
    ref = O.rope(xt.float().cpu().numpy(), pos0, base, O.F32)
    # fp32 angles: relative error ~2e-7 of (pos0 + s) rad, times the pair's norm
    angle_floor = 1e-5 + 4e-7 * (pos0 + S) * np.abs(x).max()
    if dt == "float32":
        assert np.abs(out - ref).max() <= angle_floor
    else:
        assert_within_bf16_ulps(out, ref, 1, floor=angle_floor)


def test_rope_in_place_on_strided_views(rng):
    """In place on the q columns of a packed [S, 3 d] qkv buffer (the decoder's
    layout), leaving the other columns untouched."""
    import torch

    import oracle as O
    from nkilab import ops

    S, H, hd = 200, 4, 64
    qkv = torch.from_numpy(rng.standard_normal((S, 3 * H * hd)).astype(np.float32)).cuda()
    before = qkv.clone()
    q = qkv[:, :H * hd].view(S, H, hd).transpose(0, 1)
    ops.rope_into(q, q, 10000.0)
    ref = O.rope(before[:, :H * hd].view(S, H, hd).transpose(0, 1).cpu().numpy(), 0, 10000.0)
    assert np.abs(q.cpu().numpy() - ref).max() < 1e-4
    assert torch.equal(qkv[:, H * hd:], before[:, H * hd:])


@pytest.mark.parametrize("nbytes", [16, 4096 * 2048 * 2, 16 * 1000 + 16 * 257, 16 * 1024 * 4 + 16])
def test_stream_copy_is_exact(nbytes):
    """The HBM-ceiling copy (measurement entry point): y == x byte for byte,
    including sizes that leave a partial last workgroup; bytes past the end
    stay untouched."""
    from nkilab import _lib
    from nkilab._tensors import stream_handle

    x = torch.randint(0, 256, (nbytes + 64,), dtype=torch.uint8, device="cuda")
    y = torch.full((nbytes + 64,), 7, dtype=torch.uint8, device="cuda")
    _lib.call("nkl_stream_copy", x.data_ptr(), y.data_ptr(), nbytes, stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(y[:nbytes], x[:nbytes])
    assert bool((y[nbytes:] == 7).all())


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("R,D", [(1, 1), (3, 7), (2049, 257), (5, 1025), (2048, 1024), (2049, 2048), (7, 4097),
                                 (1281, 4096), (3, 8191), (5, 16384), (2, 16389), (9, 31363), (2, 65536), (2, 70003)])
def test_row_kernels_at_every_plan(dt, R, D):
    """softmax and RMSNorm on rows held by 1, 4 and 16 wavefronts and by the
    looped kernels, contiguous and as views whose rows start off 16 bytes
    (another offset for x than for y), against float64.  fp32: 1e-5 relative
    (row sums of up to 7e4 positive terms in a tree: below 40 roundings of
    2^-24 and the exponential's 2^-22); bf16: one ulp of the exact value."""
    from nkilab import ops

    g = torch.Generator(device="cuda").manual_seed(R * 100003 + D)
    for off_x, off_y in ((0, 0), (3, 1)):
        xb = (torch.randn(R, D + 9, generator=g, device="cuda") * 3).to(dt)
        x = xb[:, off_x:off_x + D] if off_x else xb[:, :D].contiguous()
        yb = torch.full((R, D + 5), 7.0, dtype=dt, device="cuda")
        y = yb[:, off_y:off_y + D] if off_y else torch.empty(R, D, dtype=dt, device="cuda")
        ops.softmax_into(x, y)
        ref = torch.softmax(x.double(), -1)
        w = (torch.randn(D + 1, generator=g, device="cuda") * 0.1 + 1).to(dt)[off_y:off_y + D]
        n = torch.empty(R, D, dtype=dt, device="cuda")
        ops.rmsnorm_into(x, w, n)
        xd = x.double()
        nref = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
        if dt == torch.float32:
            assert ((y.double() - ref).abs() <= 1e-5 * ref).all()
            assert ((n.double() - nref).abs() <= 1e-5 * nref.abs()).all()
        else:
            assert_within_bf16_ulps(_np(y), ref.cpu().numpy())
            assert_within_bf16_ulps(_np(n), nref.cpu().numpy())
        if off_y:  # nothing outside the view is written
            assert (yb[:, :off_y] == 7).all() and (yb[:, off_y + D:] == 7).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D", [2, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129])
def test_short_unaligned_rows(dt, D):
    """Rows at the limits of the kernels that hold one element a lane (64; 32
    in fp32 softmax) or two (RMSNorm: 128 in bf16, 64 in fp32)."""
    test_row_kernels_at_every_plan(dt, 70, D)
    test_row_kernels_at_every_plan(dt, 1, D)


def test_softmax_of_infinite_and_masked_rows():
    """Masked entries (-inf, the type's lowest value) get probability 0, a row
    of them and a row with +inf or NaN is NaN, at every plan."""
    from nkilab import ops

    for D in (5, 1000, 5000, 20001, 70003):
        x = torch.randn(5, D, device="cuda")
        x[0, ::2] = -float("inf")
        x[1, 1:] = torch.finfo(torch.float32).min
        x[2] = -float("inf")
        x[3, D // 2] = float("inf")
        x[4, D - 1] = float("nan")
        y = ops.softmax(x)
        assert (y[0, ::2] == 0).all() and abs(y[0].double().sum().item() - 1) < 1e-5
        assert y[1, 0] == 1 and (y[1, 1:] == 0).all()
        assert torch.isnan(y[2]).all() and torch.isnan(y[3, D // 2]) and torch.isnan(y[4]).all()


def test_row_kernels_past_one_launch():
    """More rows than one launch of a workgroup per row takes (HIP's limit of
    2^32 threads, 16.8M rows of 256), in place: the rows on both sides of the
    second launch, and one column of every other."""
    from nkilab import ops

    R, D = (1 << 24) + 5, 4104
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    if free < (R * D * 2) + (8 << 30):
        pytest.skip(f"needs {(R * D * 2 >> 30) + 8} GiB of GPU memory, {free >> 30} free")
    rows = [0, 1, (1 << 24) - 2, (1 << 24) - 1, 1 << 24, R - 1]
    others = torch.ones(R, dtype=torch.bool, device="cuda")
    others[rows] = False
    x = torch.zeros(R, D, dtype=torch.bfloat16, device="cuda")
    special = torch.randn(len(rows), D, device="cuda").bfloat16()
    x[rows] = special
    ops.softmax_into(x, x)
    assert_within_bf16_ulps(_np(x[rows]), torch.softmax(special.double(), -1).cpu().numpy())
    assert (x[others, 7] == torch.tensor(1 / D).bfloat16().cuda()).all()
    x.fill_(2)
    x[rows] = special
    w = (torch.rand(D, device="cuda") + 0.5).bfloat16()
    ops.rmsnorm_into(x, w, x)
    s = special.double()
    ref = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    assert_within_bf16_ulps(_np(x[rows]), ref.cpu().numpy())
    assert (x[others, 7] == w[7]).all()
    del x
    torch.cuda.empty_cache()
