"""The per-row scalars and row reductions against the CPU oracle where they can go wrong: every
number of waves a row can have (1 to 16, with one and two rows a workgroup), and rows whose sum of
squares, root or scale falls on either side of the short sequences' domains; and the sequences
themselves over every positive binary32 value."""

import pytest
import torch

import oracle
import mcoplib_amd._C  # noqa: F401  (registers torch.ops._C.*)
from mcoplib_amd import _lib, op
from gpu_util import DEV, assert_codes, assert_exact, assert_scales, randn, weight

pytestmark = pytest.mark.gpu


def _h2(x, r, w, eps, qdt, tag):
    q_ref, s_ref, r_ref = oracle.rms_norm_dynamic_per_token_quant(x, w, eps, qdt, residual=r)
    q = torch.empty(x.shape, dtype=qdt, device=DEV)
    s = torch.empty(x.shape[0], 1, device=DEV)
    rd = r.to(DEV)
    torch.ops._C.rms_norm_dynamic_per_token_quant(q, x.to(DEV), w.to(DEV), s, eps, None, rd)
    torch.cuda.synchronize()
    assert_exact(rd, r_ref, tag + " residual")
    assert_scales(s, s_ref, tag + " scales")
    assert_codes(q, q_ref, tag + " codes")


@pytest.mark.parametrize("waves", range(1, 17))
@pytest.mark.parametrize("T", [3, 300])
def test_waves_a_row(waves, T):
    """Two vectors a lane: `waves` waves a row; the last one partly filled at T = 300."""
    H = 1024 * waves - (8 if T > 256 else 0)
    x, r = randn((T, H), 1, torch.bfloat16), randn((T, H), 2, torch.bfloat16)
    w = weight(H, 3, torch.bfloat16)
    _h2(x, r, w, 1e-6, torch.int8, f"{T}x{H}")


# Binary exponents of the rows: sums of squares below 2^-60 and above 2^100 leave the short
# sequences, as do roots and scales outside [2^-100, 2^100].
@pytest.mark.parametrize("exponent", [-126, -70, -50, -36, -33, -31, -24, 0, 40, 44, 46, 60, 63])
@pytest.mark.parametrize("eps", [0.0, 1e-6])
@pytest.mark.parametrize("qdt", [torch.int8, torch.float8_e4m3fn])
def test_domains_of_the_short_sequences(exponent, eps, qdt):
    H = 1024
    x = torch.ldexp(randn((4, H), 4, torch.float32), torch.tensor(exponent)).bfloat16()
    r = torch.ldexp(randn((4, H), 5, torch.float32), torch.tensor(exponent)).bfloat16()
    w = weight(H, 6, torch.bfloat16)
    _h2(x, r, w, eps, qdt, f"2^{exponent}")
    sm = 0.5 + torch.rand(H, generator=torch.Generator().manual_seed(7))
    q_ref, s_ref, ar_ref, an_ref = oracle.rms_norm_smooth_quant(x, w, sm, eps, qdt, r)
    q, s = torch.empty(x.shape, dtype=qdt, device=DEV), torch.empty(4, device=DEV)
    ar, an = torch.empty_like(x, device=DEV), torch.empty_like(x, device=DEV)
    op.rms_norm_dynamic_per_token_quant(q, x.to(DEV), w.to(DEV), sm.to(DEV), s, eps, ar, an,
                                        r.to(DEV))
    torch.cuda.synchronize()
    assert_exact(an, an_ref, "H4 after_norm")
    assert_scales(s, s_ref, "H4 scales")
    assert_codes(q, q_ref, "H4 codes")


SCALARS = ("1/a", "a/127", "a/448", "127/a", "max(a/127, eps)", "max(a/448, 1/229376)", "1/rms")


# hidden 1 and eps 0: the root of every value; the others: the quotient by a row's width (powers of
# two, odd, the narrowest and widest) and its sum with the usual eps
@pytest.mark.parametrize("hidden,eps", [(1, 0.0), (1, 1e-6), (3, 0.0), (67, 1e-6), (128, 1e-6),
                                        (4096, 1e-5), (5120, 1e-6), (5137, 1e-6), (7168, 0.0),
                                        (65535, 1e-6), (131072, 1e-6), (4194303, 0.0)])
def test_short_sequences_over_every_positive_value(hidden, eps):
    bad = torch.zeros(len(SCALARS), dtype=torch.int64, device=DEV)
    _lib.check(_lib.lib.mcop_check_row_scalars(bad.data_ptr(), 0, 1 << 31, hidden, eps,
                                               _lib.stream_of(bad)))
    torch.cuda.synchronize()
    assert dict(zip(SCALARS, bad.tolist())) == dict.fromkeys(SCALARS, 0)
