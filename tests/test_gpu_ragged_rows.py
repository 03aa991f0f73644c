"""Rows that are not whole aligned vectors (any width of at least one vector, any base address)
against the CPU oracle, through every operator that has a ragged form: one element past and before
whole vectors, the last vector the first of a wave's run of lanes (8 * 64 * k + 1 wide: in-place
operators turn the row there), the narrowest rows, and the widest that the registers hold; with few
rows, which mostly load one element at a time, and with many."""

import pytest
import torch

import oracle
import mcoplib_amd._C  # noqa: F401  (registers torch.ops._C.*)
from mcoplib_amd import op
from gpu_util import DEV, assert_codes, assert_exact, assert_scales, gen, randn, weight

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32
WIDTHS = [8, 9, 15, 127, 129, 511, 513, 519, 1025, 2047, 4097, 8193, 16385, 32761]
SHIFTED = [1024, 5120]  # whole vectors, from an address one element past alignment


def put(t, shift):
    """t on the GPU, its first element `shift` elements past an allocation's start."""
    d = torch.empty(t.numel() + shift, dtype=t.dtype, device=DEV)[shift:]
    return d.copy_(t.flatten().to(DEV)).view(t.shape)


def rows(H, T, dtype, shift):
    x, r, w = randn((T, H), H, dtype), randn((T, H), H + 1, dtype), weight(H, H + 2, dtype)
    return x, r, w, put(x, shift), put(r, shift), put(w, shift)


@pytest.mark.parametrize("T", [3, 300])
@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("H", WIDTHS + SHIFTED)
def test_norms_and_quantizers(H, dtype, T):
    if T * H > 3_000_000 or (dtype is F32 and H > 16385):
        T = 3
    shift = 1 if H in SHIFTED else 0
    eps = 1e-6
    x, r, w, xd, rd, wd = rows(H, T, dtype, shift)
    for qdt in (torch.int8, torch.float8_e4m3fn):
        for res in (r, None):
            q_ref, s_ref, r_ref = oracle.rms_norm_dynamic_per_token_quant(x, w, eps, qdt,
                                                                          residual=res)
            q = put(torch.full((T, H), 77, dtype=torch.int8).view(qdt), shift)
            s = torch.empty(T, 1, device=DEV)
            rr = None if res is None else put(r, shift)
            torch.ops._C.rms_norm_dynamic_per_token_quant(q, xd, wd, s, eps, None, rr)
            if res is not None:
                assert_exact(rr, r_ref, f"H2 {qdt} residual")
            assert_scales(s, s_ref, f"H2 {qdt} scales")
            assert_codes(q, q_ref, f"H2 {qdt} codes")
    x_ref, r_ref = oracle.fused_add_rms_norm(x, r, w, eps)
    xx, rr = put(x, shift), put(r, shift)
    torch.ops._C.fused_add_rms_norm(xx, rr, wd, eps)
    assert_exact(rr, r_ref, "H1 residual")
    assert_exact(xx, x_ref, "H1 output")
    out = torch.empty_like(xd)
    torch.ops._C.rms_norm(out, xd, wd, eps)
    assert_exact(out, oracle.vllm_rms_norm(x, w, eps), "vLLM norm")
    q_ref, s_ref, z_ref = oracle.dynamic_scaled_int8_quant(x, use_azp=True)
    q, s = torch.empty(T, H, dtype=torch.int8, device=DEV), torch.empty(T, 1, device=DEV)
    z = torch.empty(T, 1, dtype=torch.int32, device=DEV)
    torch.ops._C.dynamic_scaled_int8_quant(q, xd, s, z)
    assert_exact(z, z_ref, "azp")
    assert_codes(q, q_ref, "azp codes")
    q_ref, s_ref = oracle.dynamic_per_token_scaled_fp8_quant(x)
    q = torch.empty(T, H, dtype=torch.float8_e4m3fn, device=DEV)
    torch.ops._C.dynamic_per_token_scaled_fp8_quant(q, xd, s, None)
    assert_scales(s, s_ref, "fp8 scales")
    assert_codes(q, q_ref, "fp8 codes")


@pytest.mark.parametrize("T", [3, 300, 2100])
@pytest.mark.parametrize("H", WIDTHS)
def test_smooth_scale_and_padded(H, T):
    if T * H > 3_000_000:
        T = 3
    eps = 1e-6
    x, r, w, xd, rd, wd = rows(H, T, BF, 0)
    sm = 0.5 + torch.rand(H, generator=gen(H + 3))
    for qdt in (torch.int8, torch.float8_e4m3fn):
        q_ref, s_ref, ar_ref, an_ref = oracle.rms_norm_smooth_quant(x, w, sm, eps, qdt, r)
        q, s = torch.empty(T, H, dtype=qdt, device=DEV), torch.empty(T, device=DEV)
        ar, an = torch.empty_like(xd), torch.empty_like(xd)
        op.rms_norm_dynamic_per_token_quant(q, xd, wd, sm.to(DEV), s, eps, ar, an, rd)
        assert_exact(ar, ar_ref, "H4 after_res")
        assert_exact(an, an_ref, "H4 after_norm")
        assert_scales(s, s_ref, "H4 scales")
        assert_codes(q, q_ref, "H4 codes")
    q_ref, s_ref = oracle.scale_dynamic_quant(x, sm)
    q, s = op.scale_dynamic_quant(xd, sm.to(DEV), torch.int8)
    assert_scales(s, s_ref, "H5 scales")
    assert_codes(q, q_ref, "H5 codes")
    pad = (H + 4 + 1) // 2
    p = torch.full((T, 2 * pad), 77, dtype=torch.int8, device=DEV)
    rms, q = torch.empty_like(xd), torch.empty(T, H, dtype=torch.int8, device=DEV)
    s, rr = torch.empty(T, 1, device=DEV), rd.clone()
    op.fused_add_rms_norm_dynamic_per_token_quant_padding_output(p, rms, q, s, xd, rr, wd, pad,
                                                                 eps)
    p_ref, r_ref, rms_ref, q_ref, s_ref = oracle.add_rms_norm_quant_padded(x, r, w, pad, eps, 77)
    assert_exact(rr, r_ref, "padded residual")
    assert_exact(rms, rms_ref, "padded rms")
    assert_scales(s, s_ref, "padded scales")
    assert_codes(q, q_ref, "codes")
    assert_exact(p.view(torch.uint8), p_ref, "padded rows, the bytes between them untouched")


@pytest.mark.parametrize("H", [513, 1025, 1537, 2049, 4097, 5121, 8193, 5120, 7168, 7176, 50000])
def test_after_res_over_the_residual(H):
    """after_res given as the residual's (or the input's) own buffer: odd widths, where the last
    vector of a row would start a wave and overlaps the one before; whole vectors that leave lanes
    over (640, 896 and 897 of them), which load a copy of a vector that another wave
    stores; and the same in every slice of a split row (6250 vectors)."""
    T, eps = 2100 if H < 5000 else 300 if H < 10000 else 40, 1e-6
    x, r, w, xd, rd, wd = rows(H, T, BF, 0)
    sm = 0.5 + torch.rand(H, generator=gen(H + 3))
    ar, out, ref = torch.empty_like(xd), torch.empty_like(xd), torch.empty_like(xd)
    op.rms_norm(ref, xd, wd, eps, ar, rd, False)
    for own in ("residual", "input"):
        xx, rr = xd.clone(), rd.clone()
        over = rr if own == "residual" else xx
        op.rms_norm(out, xx, wd, eps, over, rr, False)
        assert_exact(over, (x.float() + r.float()).to(BF), f"norm after_res over the {own}")
        assert_exact(out, ref.cpu(), f"norm over the {own}")
    q_ref, s_ref, ar_ref, an_ref = oracle.rms_norm_smooth_quant(x, w, sm, eps, torch.int8, r)
    for own in ("residual", "input"):
        xx, rr, an = xd.clone(), rd.clone(), torch.empty_like(xd)
        over = rr if own == "residual" else xx
        q, s = torch.empty(T, H, dtype=torch.int8, device=DEV), torch.empty(T, device=DEV)
        op.rms_norm_dynamic_per_token_quant(q, xx, wd, sm.to(DEV), s, eps, over, an, rr)
        assert_exact(over, ar_ref, f"H4 after_res over the {own}")
        assert_exact(an, an_ref, f"H4 after_norm over the {own}")
        assert_scales(s, s_ref, f"H4 scales over the {own}")
        assert_codes(q, q_ref, f"H4 codes over the {own}")


# either side of each line between the element-wise and the ragged form: the narrowest rows, few
# rows, one vector a lane, the chip's SIMDs with a wave each, the element-wise form's widest row
@pytest.mark.parametrize("T,H", [(300, 31), (300, 33), (300, 63), (300, 66), (256, 511), (256, 513),
                                 (257, 513), (256, 2047), (256, 2049), (1000, 1023), (1025, 1023),
                                 (1024, 769), (256, 769), (1025, 769), (2048, 769), (2100, 769), (4, 4095),
                                 (4, 4097)])
@pytest.mark.parametrize("dtype", [BF, HF, F32])
def test_lines_between_the_forms(dtype, T, H):
    eps = 1e-6
    x, r, w, xd, rd, wd = rows(H, T, dtype, 0)
    sm = 0.5 + torch.rand(H, generator=gen(H + 3))
    x_ref, r_ref = oracle.fused_add_rms_norm(x, r, w, eps)
    xx, rr = xd.clone(), rd.clone()
    torch.ops._C.fused_add_rms_norm(xx, rr, wd, eps)
    assert_exact(rr, r_ref, "H1 residual")
    assert_exact(xx, x_ref, "H1 output")
    out, ar, an = torch.empty_like(xd), torch.empty_like(xd), torch.empty_like(xd)
    op.rms_norm(out, xd, wd, eps, ar, rd, False)
    out_ref, ar_ref = oracle.rms_norm(x, w, eps, r, False)
    assert_exact(ar, ar_ref, "norm after_res")
    assert_exact(out, out_ref, "norm")
    q_ref, s_ref, ar_ref, an_ref = oracle.rms_norm_smooth_quant(x, w, sm, eps, torch.int8, r)
    q, s = torch.empty(T, H, dtype=torch.int8, device=DEV), torch.empty(T, device=DEV)
    op.rms_norm_dynamic_per_token_quant(q, xd, wd, sm.to(DEV), s, eps, ar, an, rd)
    assert_exact(ar, ar_ref, "H4 after_res")
    assert_exact(an, an_ref, "H4 after_norm")
    assert_scales(s, s_ref, "H4 scales")
    assert_codes(q, q_ref, "H4 codes")
