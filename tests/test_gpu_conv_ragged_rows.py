"""Conv rows that do not start on 16 bytes (T % 4 != 0, as the generator's last
stage gives with its reflection pad): the record kernels and the row statistics
on every remainder of T mod 4, at tile edges and ends.

The float64 conv of the float64 AdaIN + Snake is the reference. The bar is the
f32 accumulation bound: n = C_in K products, each with the input's own error of
at most 2e-6 |y|, summed in some order with n u relative to sum |w y| (u =
2^-24): (2e-6 + n u) sum |w y| + 2 u |out|. The output and the residual sit in
buffers with sentinels around them."""
import numpy as np
import pytest
import torch

from nspeech_amd import abi, configs

from ._util import say

pytestmark = pytest.mark.gpu


def _reference(x, gam, bet, alp, w, bias, res, pad, dil):
    """float64 output and sum |w y| of the fused stage."""
    x = x.double()
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt((x - m).square().mean(-1, keepdim=True) + 1e-5)
    y = y * (1.0 + gam.double()[:, :, None]) + bet.double()[:, :, None]
    al = alp.double()[None, :, None]
    y = y + torch.sin(al * y).square() / (al + 1e-9)
    T, K = x.shape[-1], w.shape[2]
    yp = torch.nn.functional.pad(y, (pad, pad))
    out = bias.double()[None, :, None].expand(x.shape[0], -1, T).clone()
    mag = torch.zeros_like(out)
    for k in range(K):
        s = yp[:, :, k * dil:k * dil + T].contiguous()
        for b in range(x.shape[0]):
            out[b] += w[:, :, k].double().contiguous() @ s[b]
            mag[b] += w[:, :, k].double().abs().contiguous() @ s[b].abs()
    if res is not None:
        out, mag = out + res.double(), mag + res.double().abs()
    return out, mag


@pytest.mark.parametrize("B,C_in,C_out,T,K,dil,res", [
    (1, 128, 128, 1, 7, 1, True),       # one column
    (2, 128, 128, 3, 11, 5, False),     # shorter than a quad
    (1, 128, 128, 129, 7, 1, True),     # one column past a 128-column tile
    (2, 128, 128, 130, 7, 3, True),
    (1, 128, 128, 127, 11, 5, True),    # one column short of a tile
    (2, 256, 256, 255, 7, 1, False),    # two channel chunks and blocks
    (1, 144, 200, 601, 9, 5, True),     # partial channel chunk and block
    (3, 64, 96, 1001, 8, 1, True),      # odd (K - 1) dilation
    (1, 128, 128, 19201, 11, 5, True),
    (2, 128, 128, 19203, 7, 5, True),
    (3, 128, 128, 128 * 257 - 63, 7, 1, True),   # three rounds of tiles and a rest of 3, a half tile at each row's end
    (2, 256, 256, 128 * 130 + 5, 7, 3, True),    # two channel blocks, a rest of 12 across the last batch
    (3, 128, 128, 128 * 171 + 32, 7, 1, False),  # a rest that starts inside the last batch, whole 32-column blocks
    (1, 64, 64, 601, 5, 2, True),       # K < 7: mostly without records
    (2, 128, 128, 1003, 3, 5, True),
    (1, 128, 128, 19201, 3, 1, False),
    (1, 256, 128, 333, 5, 3, True),
])
def test_fused_stage_ragged_rows(B, C_in, C_out, T, K, dil, res):
    say("conv ragged rows", B, C_in, C_out, T, K, dil, res)
    g = configs.rng(B * 7 + C_in + 3 * K + dil + T)
    t = lambda a, dt=np.float32: torch.from_numpy(np.ascontiguousarray(a.astype(dt))).cuda()  # noqa: E731
    x = t(g.standard_normal((B, C_in, T)) * 1.3 + 0.2)
    w = t(g.standard_normal((C_out, C_in, K)) * 0.05, np.float16)
    bias = t(g.standard_normal(C_out), np.float16)
    gam, bet, alp = t(g.standard_normal((B, C_in)) * 0.1), t(g.standard_normal((B, C_in)) * 0.1), t(g.uniform(0.5, 1.5, C_in))
    r = t(g.standard_normal((B, C_out, T))) if res else None
    pad = (K - 1) * dil // 2
    if 2 * pad != (K - 1) * dil:
        pad = None
    wp = abi.conv1d_pack_f16(w)
    n = B * C_out * T
    if pad is None:  # T_out != T: compare the two paths' plain conv instead of a reference of equal length
        pad = (K - 1) * dil // 2
        T_out = T + 2 * pad - dil * (K - 1)
        r = t(g.standard_normal((B, C_out, T_out))) if res else None
        o1, s1 = abi.conv1d_f16w_packed_stats(x, wp, bias, r, padding=pad, dilation=dil, records=True)
        o0 = abi.conv1d_f16w_packed(x, wp, bias, r, padding=pad, dilation=dil)
        assert torch.equal(o1, o0)
        return
    ref, mag = _reference(x, gam, bet, alp, w, bias, r, pad, dil)
    bar = (2e-6 + C_in * K * 2.0 ** -24) * mag + 2.0 ** -23 * ref.abs()
    outs = []
    for records in (True, False):
        for stats in (True, False):
            buf = torch.full((n + 32,), -7.0, device="cuda")
            out = buf[16:16 + n].view(B, C_out, T)
            o, st = abi.adain_snake_conv1d_chain(x, gam, bet, alp, wp, bias, r, want_stats=stats, padding=pad, dilation=dil,
                                                 out=out, records=records)
            assert bool((buf[:16] == -7.0).all()) and bool((buf[16 + n:] == -7.0).all()), "wrote outside the output"
            worst = float(((o.double() - ref).abs() / bar).max())
            assert worst <= 1.0, f"records={records} stats={stats}: {worst:.2f} of the bar"
            outs.append(o)
            if stats:
                d = o.double()
                mean, var = d.mean(-1), d.var(-1, unbiased=False)
                st = st.double().view(B, C_out, 2)
                spread = torch.sqrt(var + 1e-5)
                assert bool(((st[:, :, 0] - mean).abs() <= 1e-5 * torch.maximum(mean.abs(), spread)).all())
                assert bool(((st[:, :, 1] * spread - 1.0).abs() <= 1e-5).all())
    for o in outs[1:]:
        assert torch.equal(o, outs[0]), "paths differ"


def test_ragged_rows_from_misaligned_views():
    """Input, residual and output 4 bytes past a 16-byte boundary, T a multiple of 4 and not."""
    for T in (512, 517):
        g = configs.rng(T)
        B, C, K, dil, pad = 2, 128, 7, 1, 3
        n = B * C * T
        flat = lambda: torch.from_numpy(g.standard_normal(n + 8).astype(np.float32)).cuda()  # noqa: E731
        xb, rb, ob = flat(), flat(), flat()
        x, r, out = (v[1:1 + n].view(B, C, T) for v in (xb, rb, ob))
        w = torch.from_numpy((g.standard_normal((C, C, K)) * 0.05).astype(np.float16)).cuda()
        wp = abi.conv1d_pack_f16(w)
        want, _ = abi.conv1d_f16w_packed_stats(x.clone(), wp, None, r.clone(), padding=pad, dilation=dil)
        keep = ob.clone()
        got, _ = abi.conv1d_f16w_packed_stats(x, wp, None, r, padding=pad, dilation=dil, out=out)
        assert torch.equal(got, want)
        assert torch.equal(ob[:1], keep[:1]) and torch.equal(ob[1 + n:], keep[1 + n:])


@pytest.mark.parametrize("C,T,K,dil,pad,res", [
    (128, 1, 1, 1, 0, False), (16, 63, 1, 1, 5, True), (128, 200, 2, 1, 1, True), (96, 517, 3, 1, 1, True),
    (128, 64, 3, 32, 32, True),   # 64 columns shared between tiles (past this kernel's LDS: the streamed-weight kernel)
    (128, 3000, 3, 20, 19, False), (128, 3001, 2, 40, 21, False), (128, 130, 3, 18, 17, True),  # windows past 96 columns
    (128, 131, 3, 5, 70, True),   # padding wider than a tile
    (64, 1000, 2, 7, 0, False), (128, 40000, 3, 3, 3, True),
])
def test_resident_weight_kernel(C, T, K, dil, pad, res):
    """The K <= 3 kernel's padding, halo and run edges (several tiles per workgroup at T = 40000, B = 2)."""
    say("conv resident weights", C, T, K, dil, pad, res)
    g = configs.rng(C + T + K + pad)
    B, T_out = 2, T + 2 * pad - dil * (K - 1)
    x = torch.from_numpy(g.standard_normal((B, C, T)).astype(np.float32)).cuda()
    w = torch.from_numpy((g.standard_normal((C, C, K)) * 0.1).astype(np.float16)).cuda()
    b = torch.from_numpy(g.standard_normal(C).astype(np.float16)).cuda()
    r = torch.from_numpy(g.standard_normal((B, C, T_out)).astype(np.float32)).cuda() if res else None
    xp = torch.nn.functional.pad(x.double(), (pad, pad))
    ref = b.double()[None, :, None].expand(B, -1, T_out).clone()
    mag = torch.zeros_like(ref)
    for k in range(K):
        for i in range(B):
            s = xp[i, :, k * dil:k * dil + T_out].contiguous()
            ref[i] += w[:, :, k].double().contiguous() @ s
            mag[i] += w[:, :, k].double().abs().contiguous() @ s.abs()
    if res:
        ref, mag = ref + r.double(), mag + r.double().abs()
    # |y - hi - lo| <= 2^-22 |y|, C K products summed in f32
    bar = (2.0 ** -22 + C * K * 2.0 ** -24) * mag + 2.0 ** -23 * ref.abs() + 1e-30
    wp = abi.conv1d_pack_f16(w)
    o = abi.conv1d_f16w_packed(x, wp, b, r, padding=pad, dilation=dil)
    worst = float(((o.double() - ref).abs() / bar).max())
    assert worst <= 1.0, f"{worst:.2f} of the bar"
    o2, st = abi.conv1d_f16w_packed_stats(x, wp, b, r, padding=pad, dilation=dil)
    assert torch.equal(o, o2)
    d = o.double().view(B * C, T_out)
    spread = torch.sqrt(d.var(-1, unbiased=False) + 1e-5)
    assert bool(((st[:, 0].double() - d.mean(-1)).abs() <= 1e-5 * torch.maximum(d.mean(-1).abs(), spread)).all())
    assert bool(((st[:, 1].double() * spread - 1.0).abs() <= 1e-5).all())


@pytest.mark.parametrize("C_out,T,K", [(128, 31, 3), (128, 333, 7), (128, 2401, 3), (96, 2402, 11), (128, 19201, 7)])
def test_row_statistics_of_ragged_rows(C_out, T, K):
    """The statistics handed along, for outputs of |mean| up to 1000 std and up to 1e19 (the residual sets both):
    the mean within its f32 rounding and that of block means up to 2 std, 2^-24 |mean| + 2^-22 std; 1 / sqrt(var)
    within 10 u (u = 2^-24: nine roundings of a block's sum of squares, halved by the root, then those of the sum
    with eps, the root and the division)."""
    g = configs.rng(T + K)
    x = torch.from_numpy(g.standard_normal((2, 128, T)).astype(np.float32)).cuda()
    w = torch.from_numpy((g.standard_normal((C_out, 128, K)) / np.sqrt(128 * K)).astype(np.float16)).cuda()
    wp = abi.conv1d_pack_f16(w)
    n = torch.from_numpy(g.standard_normal((2, C_out, T)).astype(np.float32)).cuda()
    for std, mean in ((1.0, 0.0), (1.0, 3.0), (1.0, 30.0), (1.0, -1000.0), (1e17, 0.0), (1e19, 0.0), (1e15, 3e17)):
        say("conv statistics of ragged rows", C_out, T, K, std, mean)
        for records in (True, False):
            o, st = abi.conv1d_f16w_packed_stats(x, wp, None, n * std + mean, padding=(K - 1) // 2, records=records)
            d, st = o.double().view(2 * C_out, T), st.double()
            m, sd = d.mean(-1), torch.sqrt(d.var(-1, unbiased=False) + 1e-5)
            em = ((st[:, 0] - m).abs() / (2.0 ** -24 * m.abs() + 2.0 ** -22 * sd)).max()
            er = (st[:, 1] * sd - 1.0).abs().max() / (10 * 2.0 ** -24)
            assert em <= 1.0 and er <= 1.0, f"std {std} mean {mean} records={records}: {em:.2f}, {er:.2f} of the bars"


@pytest.mark.parametrize("C_in,C_out,T,K,dil,pad", [
    (128, 128, 1000, 3, 32, 31),    # 64 columns shared between tiles and one to align: past the pipelined kernels' window
    (144, 200, 513, 2, 64, 33), (64, 96, 301, 3, 31, 1), (16, 16, 70, 2, 63, 62), (256, 128, 400, 5, 16, 30),
    (64, 64, 1021, 3, 1, 1), (96, 96, 401, 5, 2, 4), (128, 128, 205, 5, 7, 14),  # ragged rows with few tiles: 9, 9, 12 pairs
    (32, 64, 333, 3, 10, 10), (32, 32, 2047, 7, 1, 3),
])
def test_fallback_kernel(C_in, C_out, T, K, dil, pad):
    """The kernel without a pipeline: windows of more than 128 columns, and ragged rows where it is the faster one; plain
    and fused, with and without a residual, and the statistics that a pass over its output takes."""
    say("conv fallback", C_in, C_out, T, K, dil, pad)
    g = configs.rng(C_in + C_out + T + K + pad)
    t = lambda a, dt=np.float32: torch.from_numpy(np.ascontiguousarray(a.astype(dt))).cuda()  # noqa: E731
    B, T_out = 2, T + 2 * pad - dil * (K - 1)
    x, w, b = t(g.standard_normal((B, C_in, T)) * 1.3 + 0.2), t(g.standard_normal((C_out, C_in, K)) * 0.05, np.float16), \
        t(g.standard_normal(C_out), np.float16)
    gam, bet, alp = t(g.standard_normal((B, C_in)) * 0.1), t(g.standard_normal((B, C_in)) * 0.1), t(g.uniform(0.5, 1.5, C_in))
    r = t(g.standard_normal((B, C_out, T_out)))
    wp = abi.conv1d_pack_f16(w)
    d = x.double()
    m = d.mean(-1, keepdim=True)
    y = (d - m) / torch.sqrt((d - m).square().mean(-1, keepdim=True) + 1e-5)
    y = y * (1.0 + gam.double()[:, :, None]) + bet.double()[:, :, None]
    y = y + torch.sin(alp.double()[None, :, None] * y).square() / (alp.double()[None, :, None] + 1e-9)
    for fused, src in ((False, d), (True, y)):
        sp = torch.nn.functional.pad(src, (pad, pad))
        ref = b.double()[None, :, None].expand(B, -1, T_out).clone()
        mag = torch.zeros_like(ref)
        for k in range(K):
            for i in range(B):
                s = sp[i, :, k * dil:k * dil + T_out].contiguous()
                ref[i] += w[:, :, k].double().contiguous() @ s
                mag[i] += w[:, :, k].double().abs().contiguous() @ s.abs()
        for res in (None, r):
            want = ref if res is None else ref + res.double()
            bar = (2e-6 + C_in * K * 2.0 ** -24) * mag + 2.0 ** -22 * want.abs() + 2.0 ** -24 * r.double().abs() + 1e-30
            for stats in (False, True):
                buf = torch.full((B * C_out * T_out + 32,), -7.0, device="cuda")
                out = buf[16:-16].view(B, C_out, T_out)
                if fused:
                    o, st = abi.adain_snake_conv1d_chain(x, gam, bet, alp, wp, b, res, want_stats=stats, padding=pad,
                                                         dilation=dil, records=False, out=out)
                elif stats:
                    o, st = abi.conv1d_f16w_packed_stats(x, wp, b, res, padding=pad, dilation=dil, records=False, out=out)
                else:
                    o = abi.conv1d_f16w_packed(x, wp, b, res, padding=pad, dilation=dil, out=out)
                assert bool((buf[:16] == -7.0).all()) and bool((buf[-16:] == -7.0).all()), "wrote outside the output"
                worst = float(((o.double() - want).abs() / bar).max())
                assert worst <= 1.0, f"fused={fused} residual={res is not None} stats={stats}: {worst:.2f} of the bar"
                if stats:
                    q = o.double().view(B * C_out, T_out)
                    sd = torch.sqrt(q.var(-1, unbiased=False) + 1e-5)
                    assert bool(((st[:, 0].double() - q.mean(-1)).abs() <= 2.0 ** -22 * (q.mean(-1).abs() + sd)).all())
                    assert bool(((st[:, 1].double() * sd - 1.0).abs() <= 10 * 2.0 ** -24).all())


@pytest.mark.parametrize("C,T,K,dil", [(128, 16389, 3, 1), (128, 16388, 2, 5), (256, 1029, 3, 3), (256, 1028, 5, 1)])
def test_one_launch_kernels_from_misaligned_views(C, T, K, dil):
    """x, residual and output 4, 8 and 12 bytes past a 16-byte boundary on the resident-weight (C = 128) and the
    streamed-weight kernel (C = 256): the results of aligned copies, bit for bit."""
    say("conv one-launch misaligned", C, T, K, dil)
    g = torch.Generator(device="cuda").manual_seed(C + T + K)
    B, pad = 2, (K - 1) * dil // 2
    T_out = T + 2 * pad - dil * (K - 1)
    flat = lambda n: torch.randn(n + 8, generator=g, device="cuda")  # noqa: E731
    xb, rb, ob = flat(B * C * T), flat(B * C * T_out), flat(B * C * T_out)
    x, r, out = xb[1:1 + B * C * T].view(B, C, T), rb[2:2 + B * C * T_out].view(B, C, T_out), \
        ob[3:3 + B * C * T_out].view(B, C, T_out)
    wp = abi.conv1d_pack_f16((torch.randn((C, C, K), generator=g, device="cuda") * 0.05).half())
    gam, bet = (torch.randn((B, C), generator=g, device="cuda") * 0.1 for _ in range(2))
    alp = torch.rand(C, generator=g, device="cuda") + 0.5
    kw = dict(padding=pad, dilation=dil, records=False)
    want, ws = abi.adain_snake_conv1d_chain(x.clone(), gam, bet, alp, wp, None, r.clone(), **kw)
    keep = ob.clone()
    got, gs = abi.adain_snake_conv1d_chain(x, gam, bet, alp, wp, None, r, out=out, **kw)
    assert torch.equal(got, want)
    assert torch.equal(ob[:3], keep[:3]) and torch.equal(ob[3 + B * C * T_out:], keep[3 + B * C * T_out:])
    assert bool(((gs - ws).abs() <= 2.0 ** -22 * ws.abs().clamp_min(1.0)).all())
