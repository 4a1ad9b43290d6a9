"""AdaIN + Snake rows of T % 4 != 0 f32 (or T % 8 != 0 f16) elements: the row
kernel over interior 16-byte chunks with edges by element, at the edges of its
slot counts, with more rows than workgroups, rows on both sides of the
statistics switch (4 mean^2 > var), and sentinels around the output. The
reference is the float64 closed form at the bars of the parity tests."""
import numpy as np
import pytest
import torch

from nspeech_amd import abi, configs

from ._util import RTOL_F16, RTOL_F32, say

pytestmark = pytest.mark.gpu


def _closed_form(x, gam, bet, alp):
    x = x.double()
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt((x - m).square().mean(-1, keepdim=True) + 1e-5)
    y = y * (1.0 + gam.double()[:, :, None]) + bet.double()[:, :, None]
    al = alp.double()[None, :, None]
    return y + torch.sin(al * y).square() / (al + 1e-9)


def _run(B, C, T, dtype, rtol, seed):
    g = configs.rng(seed)
    x = torch.from_numpy(g.standard_normal((B, C, T), dtype=np.float32)).cuda()
    x[:, 1::3] += 3.0   # the centred pass
    x[:, 2::3] *= 0.01
    x = x.to(dtype)
    p = lambda s, lo: torch.from_numpy((g.standard_normal(s) * 0.1 + lo).astype(np.float32)).cuda()  # noqa: E731
    gam, bet, alp = p((B, C), 0.0), p((B, C), 0.0), p(C, 1.0)
    n, pad = B * C * T, 16
    buf = torch.full((n + 2 * pad,), -7.0, device="cuda", dtype=dtype)
    out = buf[pad:pad + n].view(B, C, T)
    abi.adain_snake(x, gam, bet, alp, out=out)
    assert bool((buf[:pad] == -7.0).all()) and bool((buf[pad + n:] == -7.0).all()), "wrote outside the output"
    for b in range(B):
        ref = _closed_form(x[b:b + 1], gam[b:b + 1], bet[b:b + 1], alp)
        worst = float(((out[b:b + 1].double() - ref).abs() / ref.abs().clamp_min(1.0)).max())
        assert worst <= rtol, f"batch {b}: {worst:.2e}"


@pytest.mark.parametrize("B,C,T", [
    (2, 3, 8191), (2, 3, 8193), (1, 5, 8195), (2, 3, 12289),                    # past the 256-lane kernels
    (1, 5, 4 * 512 * 10 + 3), (1, 5, 4 * 512 * 12 + 5), (1, 5, 4 * 512 * 16 + 5),   # a slot's edge
    (1, 5, 4 * 512 * 19 + 3), (1, 5, 4 * 512 * 19 + 5),                          # VGPR slots only / with LDS slots
    (1, 5, 4 * 512 * 21 + 1), (1, 5, 4 * 512 * 22 + 7),
    (1, 5, 4 * 512 * 57 + 1), (1, 5, 4 * 512 * 58 + 2), (1, 5, 4 * 512 * 58 + 3), (1, 5, 4 * 512 * 58 + 7),  # the end
    (6, 100, 40001), (5, 128, 19201), (2, 200, 9002),                            # several rows per workgroup
])
def test_f32_rows(B, C, T):
    say("adain ragged f32", B, C, T)
    _run(B, C, T, torch.float32, RTOL_F32, B + C + T)


@pytest.mark.parametrize("B,C,T", [(2, 3, 1), (2, 3, 15), (2, 5, 2049), (2, 5, 12001), (1, 128, 57601), (1, 6, 131071)])
def test_f16_rows(B, C, T):
    say("adain ragged f16", B, C, T)
    _run(B, C, T, torch.float16, RTOL_F16, B + C + T)
