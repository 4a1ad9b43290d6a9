"""Which kernels a call launches, without a GPU: the built library is loaded over a recording HIP runtime
(tests/host/fake_hip.cpp) in a process of its own, its entry points are called with addresses that nothing reads,
and the launches (kernel, grid, block, LDS bytes, tile argument) are checked against what each kernel assumes."""
import json
import re
import subprocess
import sys
from pathlib import Path

import pytest

from .test_gpu_adain_ragged_rows import ROW_SLOTS, slot_lengths
from .test_gpu_conv_record_tiles import SHAPES as RECORD_TILE_SHAPES

ROOT = Path(__file__).resolve().parent.parent
LIB = ROOT / "nspeech_amd" / "lib" / "libnspeech_rocm.so"
CUS, LDS = 256, 163840
NSR_F32 = 0

_CHILD = """
import ctypes as C, json, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_hip_take_log.restype = C.c_char_p
req = json.load(sys.stdin)
fake.fake_hip_set(req["lds"], req["cus"], 1)
lib = C.CDLL(sys.argv[2])
conv = {"p": C.c_void_p, "l": C.c_int64, "i": C.c_int, "f": C.c_float}
out = []
for name, args in req["calls"]:
    st = getattr(lib, name)(*[conv[k](v) for k, v in args])
    log = fake.fake_hip_take_log().decode().split("\\n")[:-1]
    out.append([st, [[l.split()[0]] + [int(v) for v in l.split()[1:]] for l in log]])
json.dump(out, sys.stdout)
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    """routes(calls, lds, cus) -> [(status, [(kernel, gx, gy, gz, block, lds, n), ...])], one per call."""
    if not LIB.exists():
        pytest.fail(f"{LIB} is not built: run `python -m nspeech_amd.build`")
    so = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(ROOT / "tests" / "host" / "fake_hip.cpp"), "-o", str(so)], check=True, capture_output=True)

    def run(calls, lds=LDS, cus=CUS):
        p = subprocess.run([sys.executable, "-c", _CHILD, str(so), str(LIB)], capture_output=True, text=True, timeout=120,
                           input=json.dumps({"lds": lds, "cus": cus, "calls": calls}))
        assert p.returncode == 0, p.stderr
        return [(st, [tuple(x) for x in log]) for st, log in json.loads(p.stdout)]

    return run


def _adain(rows, T, off=0):
    p = [("p", 1 << 20)] * 3
    return ["nsr_adain_snake_f32", [("p", (1 << 32) + off), *p, ("i", NSR_F32), ("l", 0), ("l", 0), ("p", (1 << 33) + off),
                                    ("l", 1), ("l", rows), ("l", T), ("f", 1e-5), ("p", 0)]]


def _check_adain(rows, T, off, kernel, gx, block, lds, cus=CUS):
    """The launch covers every row and every 16-byte chunk, and masks the row end where the kernel does."""
    what = (rows, T, off, kernel, gx, block, lds)
    if kernel == "nsrk_adain_long":
        assert block == 1024 and lds == 0 and gx == min(rows, cus), what
        return
    aligned = T % 4 == 0 and off % 16 == 0
    most, least = (T // 4, T // 4) if aligned else (max((T + 6) // 4 - 2, 0), (T + 3) // 4 - 2)
    m = re.match(r"nsrk_adain_row(u?)_b(\d+)_v(\d+)_l(\d+)$", kernel)
    if m:  # persistent: workgroups walk the rows; only the last four slots are masked
        assert bool(m[1]) == (not aligned) and off % 16 == 0, what
        b, v, l = int(m[2]), int(m[3]), int(m[4])
        assert block == b and lds == 16 * b * l and 1 <= gx <= rows, what
        assert b * (v + l) >= most and b * (v + l - 4) <= least, what
        return
    m = re.match(r"nsrk_adain_res_b(\d+)_nv(\d+)_u$", kernel)
    assert m, what  # one row per workgroup, all of it in registers
    assert not aligned and block == int(m[1]) and lds == 0 and gx == rows and int(m[1]) * int(m[2]) >= most, what


ROWS = (1, 2, 127, 128, 129, 256, 257, 511, 512, 1024, 1025, 1280, 1281, 4000)


def _lengths():
    ts = {1, 2, 3, 4, 5, 7, 500, 8191, 8192, 8193, 8197, 8198, 8199, 200001}
    for chunks in range(512, 512 * 59 + 1, 512):  # both sides of every slot count
        ts |= {4 * chunks + d for d in range(-6, 12)}
    return sorted(ts)


def test_adain_launches_cover_every_row(routes):
    cases = [(r, T, off) for r in ROWS for T in _lengths() for off in (0, 4)]
    for (r, T, off), (st, log) in zip(cases, routes([_adain(*c) for c in cases])):
        assert st == 0 and len(log) == 1, (r, T, off, st, log)
        k, gx, gy, gz, block, lds, _ = log[0]
        assert (gy, gz) == (1, 1)
        _check_adain(r, T, off, k, gx, block, lds)


def test_adain_rows_without_room_for_lds_slots(routes):
    """On a device whose LDS does not hold the row kernel's slots, rows take the register or the two-read kernel."""
    cases = [(3000, T, 0) for T in (40001, 50002, 65537, 70001, 115203, 40000, 115200)]
    for (r, T, off), (st, log) in zip(cases, routes([_adain(*c) for c in cases], lds=100000)):
        assert st == 0 and len(log) == 1, (r, T, st, log)
        k, gx, _, _, block, lds, _ = log[0]
        assert "_l19" not in k and lds == 0, log
        _check_adain(r, T, off, k, gx, block, lds)


@pytest.mark.parametrize("rows,T,row_kernel", [
    (1024, 8193, False), (1024, 8201, True), (2048, 9001, True), (1024, 12001, True), (1280, 12001, False),
    (256, 14401, True), (512, 14401, False), (128, 19201, True), (1024, 19201, False), (128, 24001, False),
    (128, 28801, True), (400, 28801, False), (1024, 28801, True), (3000, 28801, True), (128, 48001, True),
    (256, 48001, False), (1024, 57601, True), (2048, 40001, False), (256, 70001, True), (3000, 115201, True)])
def test_adain_ragged_rows_take_the_faster_kernel(routes, rows, T, row_kernel):
    """Each side of the rule's lines (measured: see the rule), where the other kernel was slower or no faster."""
    (st, log), = routes([_adain(rows, T)])
    assert st == 0 and log[0][0].startswith("nsrk_adain_rowu_") == row_kernel, log


def _conv(mode, C_in, C_out, B, T, K, dil, records, res=False, off=0, pad=None):
    """mode "stats" / "fused": adain_snake_conv1d_chain with / without statistics out; "plain": conv1d_f32io."""
    pad = (K - 1) * dil // 2 if pad is None else pad
    T_out = T + 2 * pad - dil * (K - 1)
    x, out, r = [("p", (v << 40) + off) for v in (1, 2, 3)]
    big, ws = 1 << 46, ("p", 1 << 47)
    if mode == "plain":
        need = -(-2 * C_in * C_out * K // 256) * 256
        return ["nsr_conv1d_f32io", [x, ("p", 256), ("p", 0), out, ("l", B), ("l", C_in), ("l", C_out), ("l", T), ("l", K),
                                     ("l", 1), ("l", pad), ("l", dil), ws, ("l", big if records else need), ("p", 0)]]
    need = -(-8 * B * C_out * -(-T_out // 32) // 256) * 256 if mode == "stats" else 0
    a = [("p", 256)] * 3
    return ["nsr_adain_snake_conv1d_chain_f32",
            [x, ("p", 256), *a, ("i", NSR_F32), ("l", 0), ("l", 0), ("p", 256), ("p", 0), r if res else ("p", 0), out,
             ("p", 256 if mode == "stats" else 0), ("l", B), ("l", C_in), ("l", C_out), ("l", T), ("l", K), ("l", pad),
             ("l", dil), ("f", 1e-5), ws, ("l", big if records else need), ("p", 0)]]


def _family(log):
    names = [l[0] for l in log if l[0].startswith("nsrk_conv1d_") and l[0] != "nsrk_conv1d_pack"]
    kinds = {"records" if re.search(r"_p[rs]\d?_", n) else "one launch" if re.search(r"_(rw|pc)_", n) else "fallback"
             for n in names}
    assert len(kinds) == 1, log
    return kinds.pop()


@pytest.mark.parametrize("mode,C_in,C_out,B,T,K,dil,records,family", [
    # rows of T % 4 != 0, one dilation, where the kernels before or beside the choice were 10% slower or more
    ("plain", 16, 16, 4, 401, 3, 1, True, "fallback"), ("fused", 16, 16, 4, 2401, 2, 5, False, "fallback"),
    ("stats", 64, 64, 4, 1021, 3, 1, False, "fallback"), ("stats", 64, 64, 4, 16381, 3, 1, False, "one launch"),
    ("stats", 128, 128, 1, 1021, 3, 1, False, "fallback"), ("stats", 128, 128, 4, 4093, 3, 1, False, "one launch"),
    ("fused", 128, 128, 4, 4093, 3, 1, False, "fallback"), ("stats", 128, 128, 1, 19201, 3, 1, True, "one launch"),
    ("stats", 128, 128, 4, 1021, 5, 1, True, "fallback"), ("stats", 128, 128, 4, 8189, 5, 1, True, "one launch"),
    ("plain", 128, 128, 1, 1021, 3, 1, False, "one launch"), ("plain", 128, 128, 4, 1021, 5, 1, False, "fallback"),
    ("plain", 64, 64, 4, 16381, 5, 1, False, "fallback"), ("plain", 256, 256, 1, 401, 7, 1, False, "one launch"),
    ("plain", 512, 32, 4, 8189, 5, 1, False, "fallback"), ("stats", 256, 256, 4, 509, 2, 1, False, "one launch"),
    ("plain", 128, 128, 1, 2401, 7, 1, True, "records"), ("stats", 128, 128, 1, 19201, 7, 5, True, "records"),
    ("stats", 128, 128, 4, 57601, 11, 5, True, "records"), ("plain", 64, 64, 4, 8189, 7, 1, True, "fallback"),
    ("plain", 32, 32, 4, 8189, 7, 1, True, "fallback"), ("plain", 64, 64, 4, 1021, 7, 1, True, "records"),
    ("stats", 128, 128, 8, 401, 3, 5, True, "one launch"),
    # ragged inputs of an even K, outputs of whole vectors
    ("plain", 128, 128, 4, 1025, 2, 1, True, "fallback"), ("fused", 256, 256, 1, 1021, 2, 1, True, "fallback"),
    ("fused", 128, 128, 4, 16381, 2, 1, True, "one launch"), ("plain", 256, 256, 4, 4097, 2, 1, True, "fallback"),
    # K = 3 to 6 with several channel blocks: records where they win
    ("stats", 256, 256, 1, 3200, 3, 1, True, "records"), ("stats", 256, 256, 8, 9600, 3, 5, True, "records"),
    ("fused", 256, 256, 4, 2048, 3, 1, True, "one launch"), ("plain", 256, 256, 4, 2048, 3, 1, True, "one launch"),
    ("plain", 256, 128, 8, 9600, 3, 1, True, "one launch"), ("stats", 256, 128, 8, 9600, 3, 1, True, "one launch"),
    ("plain", 512, 32, 4, 3200, 3, 1, True, "one launch"), ("fused", 256, 128, 4, 5120, 3, 1, True, "records"),
    ("plain", 128, 256, 4, 4096, 3, 1, True, "one launch"), ("plain", 128, 256, 4, 512, 3, 1, True, "records"),
    ("stats", 128, 256, 8, 6400, 5, 1, True, "records"), ("stats", 128, 256, 4, 12288, 3, 1, True, "one launch"),
    ("stats", 128, 256, 4, 9600, 3, 1, True, "records"),
    ("fused", 256, 128, 8, 19200, 5, 1, True, "records"), ("fused", 256, 128, 4, 12288, 5, 1, True, "one launch"),
    ("plain", 512, 512, 4, 3200, 3, 1, True, "records"), ("plain", 256, 256, 4, 16384, 5, 1, True, "records"),
    # rows of whole vectors keep the kernels they had
    ("plain", 16, 16, 4, 400, 3, 1, True, "one launch"), ("plain", 32, 32, 4, 8188, 7, 1, True, "records"),
    ("stats", 128, 128, 8, 115200, 3, 5, True, "one launch"), ("stats", 256, 256, 1, 3200, 11, 3, True, "records")])
def test_conv_takes_the_faster_kernels(routes, mode, C_in, C_out, B, T, K, dil, records, family):
    (st, log), = routes([_conv(mode, C_in, C_out, B, T, K, dil, records)])
    assert st == 0 and _family(log) == family, log


@pytest.mark.parametrize("mode,C_in,C_out,B,T,K,dil,family", [
    ("fused", 128, 128, 4, 4093, 3, 1, "one launch"), ("stats", 128, 128, 1, 401, 3, 1, "one launch"),
    ("fused", 64, 64, 4, 8189, 7, 1, "one launch"), ("fused", 128, 128, 4, 1021, 5, 1, "fallback")])
def test_ragged_conv_with_a_residual(routes, mode, C_in, C_out, B, T, K, dil, family):
    (st, log), = routes([_conv(mode, C_in, C_out, B, T, K, dil, False, res=True)])
    assert st == 0 and _family(log) == family, log


@pytest.mark.parametrize("C,B,T,K,dil,kernels", [
    (128, 1, 128 * 64, 7, 1, ["ps1"]), (128, 1, 128 * 65, 7, 1, ["ps2"]), (128, 1, 128 * 179, 7, 1, ["ps2"]),
    (128, 1, 128 * 180, 7, 1, ["pr"]), (256, 1, 128 * 64, 7, 1, ["ps2"]), (256, 1, 128 * 65, 7, 1, ["pr"]),
    (256, 4, 2400, 11, 1, ["pr"]), (512, 1, 128 * 40, 7, 1, ["ps2"]), (128, 1, 128 * 320, 11, 5, ["ps1"]),
    (128, 1, 128 * 321, 11, 5, ["pr"]), (256, 1, 128 * 179, 7, 1, ["ps1"]), (128, 1, 128 * 576, 7, 1, ["pr", "ps1"]),
    (128, 1, 128 * 577, 7, 1, ["pr"]), (256, 1, 128 * 298, 7, 1, ["pr", "ps1"]), (256, 1, 128 * 299, 7, 1, ["pr"])])
def test_record_tiles(routes, C, B, T, K, dil, kernels):
    """64 x 64, 128 x 64 (ps1, ps2) or 128 x 128 tiles (pr), or the last, a third at most filled round on small ones."""
    (st, log), = routes([_conv("stats", C, C, B, T, K, dil, True)])
    assert st == 0
    assert _tiles(log).split("+") == kernels, log


def _tiles(log):
    return "+".join(l[0].split("_")[2] for l in log if l[0].startswith("nsrk_conv1d_p") and l[0] != "nsrk_conv1d_pack")


def test_record_tile_shapes_take_the_kernels_they_name(routes):
    for mode in ("stats", "fused"):
        calls = [_conv(mode, ci, co, B, T, K, dil, True, res) for B, ci, co, T, K, dil, res, _ in RECORD_TILE_SHAPES]
        one = [_conv(mode, ci, co, B, T, K, dil, False, res) for B, ci, co, T, K, dil, res, _ in RECORD_TILE_SHAPES]
        for shape, (st, log), (st1, log1) in zip(RECORD_TILE_SHAPES, routes(calls), routes(one)):
            assert st == 0 and _tiles(log) == shape[-1], (shape, log)
            assert st1 == 0 and _family(log1) == "one launch", (shape, log1)  # both emit the statistics


def _record_columns(log, B, T_out, C_out):
    """The 64-column tiles of the output that a record call's launches write, as (channel block of 64, batch, tile)."""
    n64, n128, seen = -(-T_out // 64), -(-T_out // 128), []
    for k, gx, gy, gz, block, lds, n in log:
        if k.startswith("nsrk_conv1d_pr_"):
            n_co = -(-C_out // 128)
            assert (gy, gz, block) == (1, 1, 512) and 1 <= gx <= CUS
            for tile in range(n):  # channel block fastest, then columns, then batch
                col, cb = divmod(tile, n_co)
                b, t = divmod(col, n128)
                seen += [(2 * cb + h, b, 2 * t + j) for h in (0, 1) for j in (0, 1) if 2 * t + j < n64]
        elif k.startswith("nsrk_conv1d_ps"):
            mt = int(k[len("nsrk_conv1d_ps")])
            cols = n64 * B - n
            assert (gy, gz, block) == (1, 1, 256) and gx == cols * -(-C_out // (64 * mt))
            for tile in range(gx):
                cb, ct = divmod(tile, cols)
                b, t = divmod(n + ct, n64)
                seen += [(mt * cb + m, b, t) for m in range(mt)]
    return seen


def test_record_launches_cover_the_output_once(routes):
    cases = []
    for C_out in (2, 64, 96, 128, 130, 200, 256, 384):
        for B in (1, 2, 3, 8):
            for T in (1, 63, 65, 128, 129, 400, 1001, 4096, 8224, 16384, 16449, 21920, 33000, 57601):
                for K, dil in ((7, 1), (11, 5)):
                    cases.append((("stats", 128, C_out, B, T, K, dil, True), B, T, C_out))
    for (c, B, T, C_out), (st, log) in zip(cases, routes([_conv(*c[0]) for c in cases])):
        assert st == 0, c
        if _family(log) != "records":
            continue
        blocks = range(2 * -(-C_out // 128))
        want = {(cb, b, t) for cb in blocks for b in range(B) for t in range(-(-T // 64))}
        seen = _record_columns(log, B, T, C_out)
        live = {(cb, b, t) for cb, b, t in want if 64 * cb < C_out}
        assert len(seen) == len(set(seen)), c
        assert live <= set(seen) <= want, c


def _listed(pattern):
    text = (ROOT / "nspeech_amd" / "csrc" / "runtime" / "nsr_kernels.def").read_text()
    return {k for k in re.findall(r"NSR_KERNEL\(\w+, (\w+)\)", text) if re.match(pattern, k)}


def test_every_ragged_row_kernel_is_run_by_a_test(routes):
    lengths = [T for s in ROW_SLOTS for T in slot_lengths(s)]
    seen = {log[0][0] for _, log in routes([_adain(3, T) for T in lengths])}
    assert _listed(r"nsrk_adain_rowu_") <= seen, sorted(_listed(r"nsrk_adain_rowu_") - seen)


def test_every_listed_adain_and_conv_kernel_is_reached(routes):
    """No kernel that nothing launches: rows of every slot count on both sides of 16-byte alignment, and convs over the
    shapes that the rules tell apart."""
    calls = [_adain(r, T, off) for r in (3, 300) for T in _lengths() for off in (0, 4)]
    for mode in ("stats", "fused", "plain"):
        for res in (False, True):
            for records in (False, True):
                for ci, co in ((16, 16), (128, 128), (256, 256)):
                    for K, dil in ((1, 1), (3, 1), (3, 5), (2, 40), (3, 32), (5, 1), (7, 5), (11, 5)):
                        for B, T in ((1, 401), (1, 3200), (1, 19200), (1, 19201), (4, 57600), (4, 57601)):
                            for pad in {(K - 1) * dil // 2, (K - 1) * dil // 2 + 1}:
                                calls.append(_conv(mode, ci, co, B, T, K, dil, records, res, pad=pad))
    # plain with a residual or statistics: nsr_conv1d_f16w_packed and its form with statistics
    for K, dil in ((1, 1), (3, 1), (2, 40), (7, 5), (11, 5)):
        for stats in (False, True):
            for res in (False, True):
                for T in (3200, 57600):
                    calls.append(_packed(128, 4, T, K, dil, stats, res))
    seen = {l[0] for st, log in routes(calls) for l in log}
    want = _listed(r"nsrk_(adain_row_b|adain_rowu|adain_res|adain_long|adain_stats|conv)")
    assert want <= seen, sorted(want - seen)


def _packed(C, B, T, K, dil, stats, res):
    pad = (K - 1) * dil // 2
    T_out = T + 2 * pad - dil * (K - 1)
    a = [("p", 1 << 40), ("p", 256), ("p", 0), ("p", 3 << 40 if res else 0), ("p", 2 << 40)]
    sh = [("l", B), ("l", C), ("l", C), ("l", T), ("l", K), ("l", pad), ("l", dil)]
    if not stats:
        return ["nsr_conv1d_f16w_packed", [*a, *sh, ("p", 0)]]
    need = -(-8 * B * C * -(-T_out // 32) // 256) * 256
    return ["nsr_conv1d_f16w_packed_stats", [*a, ("p", 256), *sh, ("f", 1e-5), ("p", 1 << 47),
                                             ("l", need), ("p", 0)]]
