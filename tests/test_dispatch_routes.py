"""Which kernels a call launches, without a GPU: the built library is loaded over a recording HIP runtime
(tests/host/fake_hip.cpp) in a process of its own, its entry points are called with addresses that nothing reads,
and the launches (kernel, grid, block, LDS bytes) are checked against what each kernel assumes."""
import json
import re
import subprocess
import sys
from pathlib import Path

import pytest

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
    """routes(calls, lds, cus) -> [(status, [(kernel, gx, gy, gz, block, lds), ...])], one per call."""
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
        k, gx, gy, gz, block, lds = log[0]
        assert (gy, gz) == (1, 1)
        _check_adain(r, T, off, k, gx, block, lds)


def test_adain_rows_without_room_for_lds_slots(routes):
    """On a device whose LDS does not hold the row kernel's slots, rows take the register or the two-read kernel."""
    cases = [(3000, T, 0) for T in (40001, 50002, 65537, 70001, 115203, 40000, 115200)]
    for (r, T, off), (st, log) in zip(cases, routes([_adain(*c) for c in cases], lds=100000)):
        assert st == 0 and len(log) == 1, (r, T, st, log)
        k, gx, _, _, block, lds = log[0]
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
