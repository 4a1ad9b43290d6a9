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


def _closed_form(x, gam, bet, alp, eps=1e-5):
    x = x.double()
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt((x - m).square().mean(-1, keepdim=True) + eps)
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


# A length in every slot count of the row kernel's ragged form that its rule takes with few rows: 512 chunks of 16 bytes
# a slot, both ends of the slot count of one kernel (test_dispatch_routes.py checks that every such kernel is among them).
ROW_SLOTS = [5, 6, 7, 8, 9, 10] + list(range(13, 59))


def slot_lengths(slots):
    """The longest row of `slots` slots and the shortest of slots - 1 .. slots, neither a multiple of 4."""
    return 4 * (512 * slots + 2) - 3, 4 * (512 * (slots - 1) + 3) + 1


@pytest.mark.parametrize("slots", ROW_SLOTS)
def test_f32_every_slot_count(slots):
    for T in slot_lengths(slots):
        say("adain ragged f32 slots", slots, T)
        _run(1, 3, T, torch.float32, RTOL_F32, T)


@pytest.mark.parametrize("T", [500, 8197, 12000, 24000, 24001, 32771, 48001, 49152, 65000, 65536, 70001, 118784, 131073])
@pytest.mark.parametrize("shift_x,shift_out", [(1, 1), (1, 0), (0, 3)])
def test_f32_misaligned_views(T, shift_x, shift_out):
    """x or out 4 to 12 bytes past a 16-byte boundary: the one-row-per-workgroup kernels over their whole range of
    lengths, and the two-read kernel past it."""
    say("adain misaligned f32", T, shift_x, shift_out)
    g = configs.rng(T + 16 * shift_x + shift_out)
    B, C = 2, 3
    n = B * C * T
    xb = torch.from_numpy(g.standard_normal(n + 8, dtype=np.float32)).cuda()
    x = xb[shift_x:shift_x + n].view(B, C, T)
    x[:, 1] += 3.0  # the centred pass
    buf = torch.full((n + 32,), -7.0, device="cuda")
    out = buf[16 + shift_out:16 + shift_out + n].view(B, C, T)
    gam, bet = (torch.from_numpy((g.standard_normal((B, C)) * 0.1).astype(np.float32)).cuda() for _ in range(2))
    alp = torch.from_numpy(g.uniform(0.5, 1.5, C).astype(np.float32)).cuda()
    abi.adain_snake(x, gam, bet, alp, out=out)
    lo, hi = 16 + shift_out, 16 + shift_out + n
    assert bool((buf[:lo] == -7.0).all()) and bool((buf[hi:] == -7.0).all()), "wrote outside the output"
    ref = _closed_form(x, gam, bet, alp)
    assert float(((out.double() - ref).abs() / ref.abs().clamp_min(1.0)).max()) <= RTOL_F32


@pytest.mark.parametrize("T", [65543, 70001, 90002, 115201, 118790, 118797])
def test_f32_statistics_range(T):
    """Rows past the reach of the one-row-per-workgroup kernel keep statistics in f64: no overflow of the squares
    at an rms where f32 sums of them are infinite (T x^2 > 3.4e38), none of a large mean's, and a variance below
    the smallest normal f32 with eps = 0 (its f32 rounding, 2^-150 of 4e-40, moves 1 / sqrt(var) by 9e-7)."""
    say("adain ragged f32, range of the statistics", T)
    g = configs.rng(T)
    rows = [(1.0, 0.0, 1e-5), (1e17, 0.0, 1e-5), (1e15, 3e17, 1e-5), (2e-20, 0.0, 0.0)]
    for std, mean, eps in rows:
        x = torch.from_numpy((g.standard_normal((1, 3, T)) * std + mean).astype(np.float32)).cuda()
        gam, bet = (torch.from_numpy((g.standard_normal((1, 3)) * 0.1).astype(np.float32)).cuda() for _ in range(2))
        alp = torch.ones(3, device="cuda")
        ref = _closed_form(x, gam, bet, alp, eps)
        out = abi.adain_snake(x, gam, bet, alp, eps=eps)
        worst = float(((out.double() - ref).abs() / ref.abs().clamp_min(1.0)).max())
        assert worst <= RTOL_F32, f"std {std} mean {mean}: {worst:.2e}"
