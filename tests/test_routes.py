"""Which kernel the dispatch chooses, call by call, asked of the library itself (tests/cpp/routes.cpp; no GPU needed)."""
import os
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    """routes(lines) -> one answer per line."""
    exe = tmp_path_factory.mktemp("routes") / "routes"
    lib = ROOT / "unholy_amd"
    r = subprocess.run([HIPCC, "-O1", "-std=c++20", "-I", str(ROOT / "include"), "-I", str(lib / "csrc"),
                        str(ROOT / "tests" / "cpp" / "routes.cpp"), "-L", str(lib), "-lunholy_amd",
                        f"-Wl,-rpath,{lib}", "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]

    def ask(lines):
        out = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True).stdout
        answers = out.split()
        assert len(answers) == len(lines)
        return answers

    return ask


DIRECT = {"kpart", "tiled", "rows"}  # operands go into LDS by direct 16-byte loads


def test_unaligned_operands_avoid_direct_loads(routes):
    """A direct 16-byte load needs a 16-byte aligned source; the GEMV, the row groups and the reference order read their
    operands with plain loads. Any operand off by 1 to 8 bytes takes those, aligned ones do not."""
    dense = [f"dense {m} {n} {k} {n} {f}" for m in (1, 8, 17, 64, 65, 200, 300, 1000) for n in (200, 4096)
             for k in (128, 4096, 8192) for f in (0, 1)]
    grouped = [f"grouped {m} {g} {r} {k}" for m in (1, 8, 9, 33, 100, 200, 400, 1200)
               for g, r, k in ((8, 1024, 4096), (3, 96, 640), (5, 48, 1152))]
    for off in ("8 0", "0 8", "4 4", "0 1"):
        lines = [f"{l} {off}" for l in dense + grouped]
        bad = [(l, a) for l, a in zip(lines, routes(lines)) if a in DIRECT]
        assert not bad, bad[:5]
    assert set(routes([f"{l} 0 0" for l in dense])) <= {"kpart", "tiled"}
    assert set(routes([f"{l} 0 16" for l in grouped])) <= DIRECT


def test_few_rows_never_change_the_order_of_sums(routes):
    """gemm_fp8_f32s of up to 16 rows equals gemm_fp8_f32s_x bit for bit, gemv_w8a8 of up to 32 every column range of
    gemv_w8a8_parts: at no shape may the plain entry points take the tiled GEMM, which adds in another order."""
    lines = [f"dense {m} {n} {k} {n} {f} 0 0" for f, ms in ((1, (1, 5, 16)), (0, (1, 8, 17, 32))) for m in ms
             for n in (128, 1024, 4096, 8192, 32768, 65536, 129280) for k in (128, 256, 512, 1024, 2048, 4096, 8192, 9216)]
    bad = [(l, a) for l, a in zip(lines, routes(lines)) if a not in ("kpart", "gemv")]
    assert not bad, bad[:5]
