"""The conv's record kernels by tile size and round: 128 x 128 tiles in one, two and more rounds over the chip, with
and without a last round on 64 x 64 tiles, and 128 x 64 tiles of several channel blocks. Every case compares the record
path with the one-launch kernels, which add the same products in the same order: outputs and the statistics handed
along (same 32-column blocks, same merge) must match bit for bit. The one-launch kernels are held to the oracle and
float64 in test_gpu_conv1d.py and test_gpu_conv_ragged_rows.py; that the shapes take the kernels named here is checked
without a GPU in test_dispatch_routes.py."""
import pytest
import torch

from nspeech_amd import abi

from ._util import say

# B, C_in, C_out, T, K, dilation, residual, kernels (128 x 128: pr, MT x 64 channels x 64 columns: psMT)
SHAPES = [
    (1, 128, 128, 128 * 200, 7, 1, False, "pr"),                  # one round, whole 32-column blocks
    (1, 128, 128, 128 * 255 + 5, 11, 5, True, "pr"),              # the widest window, ragged rows
    (2, 128, 128, 128 * 110 - 4, 11, 3, True, "pr"),              # T % 4 == 0, T % 32 != 0
    (1, 144, 128, 128 * 190 + 32, 7, 3, False, "pr"),             # a 16-channel second chunk
    (1, 128, 200, 128 * 100 + 1, 9, 1, True, "pr"),               # a partial second block
    (1, 144, 200, 128 * 70, 8, 3, True, "pr"),                    # odd (K - 1) dilation: 21
    (2, 96, 96, 128 * 120 + 3, 8, 1, False, "pr"),                # odd, a partial chunk and block
    (2, 256, 256, 128 * 45, 3, 5, True, "pr"),                    # K = 3, two chunks and blocks, whole blocks
    (1, 256, 256, 128 * 185 + 64, 5, 1, False, "pr"),             # K = 5, two rounds
    (4, 256, 256, 128 * 60 + 2, 4, 3, True, "pr"),                # K = 4, odd (K - 1) dilation
    (1, 512, 256, 128 * 220, 3, 1, True, "pr"),                   # four chunks
    (1, 128, 384, 128 * 190 + 7, 3, 1, False, "pr+ps1"),          # three blocks, K = 3, a rest on small tiles
    (3, 128, 128, 128 * 130, 7, 5, True, "pr"),                   # two rounds
    (4, 128, 128, 128 * 120 + 1, 11, 1, True, "pr"),              # two rounds, ragged
    (8, 128, 128, 128 * 75, 11, 5, True, "pr"),                   # three rounds, no rest below a quarter
    (5, 128, 128, 128 * 112 + 9, 11, 5, False, "pr+ps1"),         # a rest on small tiles, ragged
    (4, 128, 128, 57601, 11, 5, True, "pr+ps1"),                  # the generator's rows
    (2, 256, 256, 128 * 140 + 32, 11, 3, True, "pr+ps1"),         # two blocks, a rest, whole 32-column blocks
    (1, 256, 256, 128 * 40, 7, 1, True, "ps2"),                   # 128 x 64 tiles, two chunks and blocks
    (3, 256, 256, 2401, 11, 5, True, "ps2"),
    (1, 144, 200, 128 * 50 + 32, 8, 1, False, "ps2"),
    (1, 512, 512, 128 * 40, 3, 1, True, "ps2"),
    (2, 256, 256, 128 * 75, 7, 3, True, "ps1"),                   # 64 x 64 tiles in place of a short second round
    (1, 256, 256, 3200, 3, 1, True, "ps1"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("B,C_in,C_out,T,K,dil,res,kernels", SHAPES)
def test_record_tiles_match_one_launch(B, C_in, C_out, T, K, dil, res, kernels):
    say("conv record tiles", B, C_in, C_out, T, K, dil, res, kernels)
    g = torch.Generator(device="cuda").manual_seed(B + C_in + C_out + T + K + dil)
    n = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    pad = (K - 1) * dil // 2
    T_out = T + 2 * pad - dil * (K - 1)
    x, w, b = n(B, C_in, T) * 1.3 + 0.2, (n(C_out, C_in, K) * 0.05).half(), n(C_out).half()
    gam, bet, alp = n(B, C_in) * 0.1, n(B, C_in) * 0.1, n(C_in).abs() + 0.5
    r = n(B, C_out, T_out) if res else None
    wp = abi.conv1d_pack_f16(w)
    xs = torch.stack([x.mean(-1).flatten(), 1.0 / x.std(-1).flatten()], 1).contiguous()
    want = None
    for records in (False, True):
        for stats in (True, False):
            out = torch.full((B * C_out * T_out + 32,), -7.0, device="cuda")
            o, st = abi.adain_snake_conv1d_chain(x, gam, bet, alp, wp, b, r, x_stats=xs, want_stats=stats, padding=pad,
                                                 dilation=dil, records=records, out=out[16:-16].view(B, C_out, T_out))
            assert bool((out[:16] == -7.0).all()) and bool((out[-16:] == -7.0).all()), "wrote outside the output"
            if want is None:
                want, want_st = o, st
                assert bool(torch.isfinite(o).all()) and bool(torch.isfinite(st).all())
            assert torch.equal(o, want), f"records={records} stats={stats}: outputs differ"
            if stats:
                assert torch.equal(st, want_st), f"records={records}: statistics differ"
    if not res:
        f1 = abi.conv1d_f32io(x, w, b, padding=pad, dilation=dil, records=True)
        assert torch.equal(f1, abi.conv1d_f32io(x, w, b, padding=pad, dilation=dil, records=False))
