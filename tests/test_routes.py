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


# One call with both kernels (gfx950, us, graph replays over weights that do not fit a cache): rows, N (G, R) x K, the
# K-part kernel's best form, the tiled GEMM. Each differs by more than a tenth.
MEASURED_DENSE = [
    (300, 4096, 4096, 0, 17.4, 26.6), (384, 4096, 4096, 0, 19.9, 27.7), (1000, 4096, 4096, 0, 52.6, 39.3),
    (2049, 4096, 4096, 0, 106.0, 83.2), (2176, 4096, 4096, 0, 108.9, 83.4), (2304, 4096, 4096, 0, 110.9, 83.5),
    (2560, 4096, 4096, 0, 129.1, 85.1), (300, 4096, 4096, 1, 18.0, 27.2), (384, 4096, 4096, 1, 21.4, 27.7),
    (2049, 4096, 4096, 1, 114.4, 96.7), (2304, 4096, 4096, 1, 121.1, 97.5), (512, 4096, 8192, 0, 46.7, 53.0),
    (1024, 4096, 8192, 0, 89.5, 73.5), (2176, 4096, 8192, 0, 186.5, 163.8), (2560, 4096, 8192, 0, 226.4, 165.7),
    (2304, 4096, 8192, 1, 210.9, 188.0), (64, 8192, 1024, 0, 6.0, 9.5), (300, 8192, 1024, 0, 15.7, 11.1),
    (768, 2048, 4096, 0, 19.5, 27.7), (2304, 2048, 4096, 1, 62.5, 51.1), (64, 32768, 1024, 1, 16.3, 13.4),
    (256, 5120, 5120, 0, 23.5, 33.0), (2100, 5120, 5120, 1, 173.7, 125.9), (1000, 1152, 4096, 0, 18.8, 24.2),
    (2000, 1152, 4096, 0, 37.8, 33.1)]
MEASURED_GROUPED = [
    (384, 8, 1024, 4096, 39.5, 66.5), (1024, 8, 1024, 4096, 95.0, 76.7), (2049, 8, 1024, 4096, 260.8, 183.3),
    (2304, 8, 1024, 4096, 276.0, 186.9), (768, 4, 1024, 4096, 37.9, 66.3), (2049, 4, 1024, 4096, 123.8, 89.2),
    (384, 32, 1024, 4096, 144.0, 108.3), (384, 8, 1024, 2048, 24.2, 32.0), (2304, 8, 1024, 2048, 157.6, 97.6),
    (64, 32, 1024, 4096, 42.8, 66.8),
    (256, 16, 512, 1024, 11.4, 17.7), (2100, 16, 512, 1024, 86.3, 54.0),
    (2100, 2, 2048, 4096, 120.8, 89.0), (2300, 7, 1152, 4096, 240.4, 194.9)]


def test_the_estimates_choose_the_measured_winner(routes):
    dense = [(f"dense {m} {n} {k} {n} {f} 0 0", kp, t) for m, n, k, f, kp, t in MEASURED_DENSE]
    grouped = [(f"grouped {m} {g} {r} {k} 0 0", kp, t) for m, g, r, k, kp, t in MEASURED_GROUPED]
    answers = routes([l for l, _, _ in dense + grouped])
    bad = [(l, a) for (l, kp, t), a in zip(dense + grouped, answers) if a != ("kpart" if kp < t else "tiled")]
    assert not bad, bad


# The K-part kernel's fastest tile (gfx950, us, M, N, K, fp32 scales): one-tile workgroups take longer with e8m0 scales.
MEASURED_FORMS = [
    (1, 8192, 1024, 0, "2x2"), (16, 8192, 1024, 0, "2x2"), (8, 7168, 2048, 0, "2x2"), (1, 8192, 1024, 1, "1x1"),
    (16, 32768, 1024, 0, "1x1"), (1, 4096, 4096, 0, "1x1"), (32, 4096, 4096, 1, "2x1"), (64, 4096, 4096, 0, "2x2"),
    (128, 4096, 4096, 0, "4x2"), (256, 4096, 4096, 1, "4x4"), (300, 4096, 4096, 0, "5x4"), (384, 4096, 4096, 1, "6x4"),
    (700, 2048, 4096, 0, "6x4"), (17, 2560, 640, 0, "2x1")]


def test_the_estimates_choose_the_measured_tile(routes):
    answers = routes([f"form {m} {n} {k} {n} {f} 0 0" for m, n, k, f, _ in MEASURED_FORMS])
    bad = [(c, a) for c, a in zip(MEASURED_FORMS, answers) if a != c[4]]
    assert not bad, bad


def test_operands_of_any_size_keep_the_fast_kernels(routes):
    """Weights and activations of 4 GiB and more go to the kernels that smaller ones go to."""
    dense = [(m, n, k, f) for m in (1, 16, 40, 200) for n, k in ((1 << 20, 8192), (524352, 8192)) for f in (0, 1)]
    assert set(routes([f"dense {m} {n} {k} {n} {f} 0 0" for m, n, k, f in dense])) <= {"kpart", "tiled"}
    assert routes(["grouped 20000 128 64 4096 0 0", "grouped 100 128 1008 65536 0 0"]) == ["kpart", "kpart"]


# The forward of one or two tokens in two launches and by the general path (gfx950, us): T, K, E, D, I.
MEASURED_TOKEN = [
    (1, 1, 256, 4096, 2048, 15.4, 24.5), (1, 6, 256, 4096, 2048, 25.0, 30.7), (1, 7, 256, 4096, 2048, 35.6, 32.3),
    (1, 8, 256, 4096, 2048, 37.3, 34.5), (2, 3, 256, 4096, 2048, 24.4, 30.1), (2, 4, 256, 4096, 2048, 34.6, 33.4),
    (2, 7, 256, 4096, 2048, 56.1, 45.6), (2, 8, 32, 4096, 2048, 57.3, 46.1), (2, 6, 64, 2048, 1024, 17.7, 22.7),
    (2, 7, 64, 2048, 1024, 25.4, 23.7), (1, 6, 16, 7168, 2048, 34.3, 42.2), (1, 7, 16, 7168, 2048, 51.9, 44.1),
    (2, 3, 16, 7168, 2048, 32.7, 42.2), (2, 6, 16, 7168, 2048, 61.2, 55.1), (1, 2, 8, 4096, 6144, 24.6, 35.8),
    (1, 5, 8, 4096, 6144, 54.1, 48.0), (2, 6, 8, 4096, 6144, 108.3, 64.3), (2, 8, 128, 1024, 512, 14.7, 19.6)]


def test_few_tokens_take_the_faster_path(routes):
    answers = routes([f"token {t} {k} {e} {d} {i}" for t, k, e, d, i, _, _ in MEASURED_TOKEN])
    bad = [(c, a) for c, a in zip(MEASURED_TOKEN, answers) if a != ("token" if c[5] < c[6] else "general")]
    assert not bad, bad


# The forward's w1 / w3 GEMV in workgroups of 4 and of 8 waves (gfx950, whole forward, us): T, K, E, D, I. An expert with
# more rows than a tile is several tiles (E = 8, T = 64); rows that do not fit a third of the LDS keep 8 waves.
MEASURED_SHAPE = [
    (1, 2, 4, 4096, 2048, 26.4, 30.1), (5, 4, 4, 4096, 2048, 35.4, 37.1), (8, 4, 4, 4096, 2048, 42.7, 40.4),
    (16, 4, 4, 4096, 2048, 57.1, 50.0), (24, 2, 4, 4096, 2048, 52.5, 47.2), (8, 4, 8, 2048, 1024, 25.5, 26.8),
    (16, 4, 8, 2048, 1024, 31.4, 30.1), (4, 6, 32, 4096, 2048, 61.6, 68.2), (5, 2, 32, 4096, 2048, 38.9, 37.4),
    (3, 6, 256, 4096, 2048, 63.7, 69.2), (4, 6, 256, 4096, 2048, 68.4, 71.5), (12, 2, 256, 4096, 2048, 69.6, 73.0),
    (2, 4, 16, 7168, 2048, 44.3, 48.9), (12, 4, 16, 7168, 2048, 100.4, 82.5), (16, 4, 8, 4096, 4096, 66.7, 60.8),
    (24, 2, 8, 4096, 4096, 63.7, 58.1), (16, 4, 8, 4096, 6144, 105.2, 95.3), (64, 8, 8, 4096, 6144, 339.7, 266.5)]


def test_the_gemv_workgroup_shape_is_the_measured_one(routes):
    answers = routes([f"shape {t} {k} {e} {d} {i}" for t, k, e, d, i, _, _ in MEASURED_SHAPE])
    bad = [(c, a) for c, a in zip(MEASURED_SHAPE, answers) if a != ("w4" if c[5] < c[6] else "w8")]
    assert not bad, bad


# The forward of up to 64 tokens by the GEMM on bf16 rows and by the GEMV (gfx950, us): T, K, E, D, I.
MEASURED_MOE = [
    (8, 6, 256, 4096, 2048, 114, 111), (9, 6, 256, 4096, 2048, 112.8, 118.6), (64, 6, 256, 4096, 2048, 337, 353),
    (9, 4, 32, 4096, 2048, 65.4, 70.4), (9, 4, 64, 2048, 1024, 35.0, 32.0), (16, 4, 64, 2048, 1024, 38.1, 40.9),
    (9, 6, 64, 2048, 1024, 39.6, 40.8), (9, 4, 8, 4096, 2048, 51.1, 42.6), (32, 4, 8, 4096, 2048, 65.5, 56.0),
    (64, 4, 8, 4096, 2048, 78.2, 87.3), (48, 8, 8, 4096, 2048, 75.2, 97.3), (64, 4, 4, 4096, 2048, 81.0, 59.7),
    (64, 8, 8, 2048, 1024, 54.9, 43.2), (12, 4, 24, 3072, 1536, 50.1, 41.6), (12, 4, 16, 7168, 2048, 77.1, 100.2),
    (9, 4, 128, 1024, 512, 24.8, 21.6), (20, 8, 128, 1024, 512, 35.3, 40.8), (9, 4, 256, 2048, 768, 35.1, 31.8),
    (10, 6, 256, 2048, 768, 42.9, 46.1)]


def test_the_forward_takes_the_faster_of_gemm_and_gemv(routes):
    answers = routes([f"moe {t} {k} {e} {d} {i}" for t, k, e, d, i, _, _ in MEASURED_MOE])
    bad = [(c, a) for c, a in zip(MEASURED_MOE, answers) if a != ("gemm" if c[5] < c[6] else "gemv")]
    assert not bad, bad


# A forward whose w2 launch (tiles, N, K) splits K over the waves of a workgroup, and does not (gfx950, whole forward, us).
MEASURED_SPLIT = [
    (1, 4096, 1024, 22.8, 23.8), (3, 4096, 1024, 27.5, 24.6), (1, 4096, 2048, 23.3, 25.6), (3, 4096, 2048, 29.9, 27.1),
    (6, 4096, 2048, 37.1, 30.2), (2, 7168, 2048, 39.1, 34.9), (6, 1024, 4096, 24.7, 26.1), (8, 1024, 4096, 26.8, 27.9),
    (4, 2048, 4096, 26.0, 27.9), (8, 2048, 4096, 39.2, 35.4), (2, 7168, 4096, 43.2, 40.1), (2, 4096, 6144, 31.9, 36.0),
    (3, 4096, 6144, 38.2, 40.9), (6, 4096, 6144, 66.2, 57.1), (6, 2048, 8192, 48.7, 50.2)]


def test_the_gemv_splits_k_where_measured(routes):
    answers = routes([f"split {t} {n} {k}" for t, n, k, _, _ in MEASURED_SPLIT])
    bad = [(c, a) for c, a in zip(MEASURED_SPLIT, answers) if a != ("split" if c[3] < c[4] else "whole")]
    assert not bad, bad


def test_every_kpart_form_has_a_gpu_test(routes):
    from tests.test_gpu_fp8 import MID_SIZES as dense
    from tests.test_gpu_grouped import MID_SIZES as grouped

    for f32 in (0, 1):
        route = routes([f"dense {m} {n} {k} {n + 8} {f32} 0 0" for m, n, k in dense])
        form = routes([f"form {m} {n} {k} {n + 8} {f32} 0 0" for m, n, k in dense])
        assert {f for f, r in zip(form, route) if r == "kpart"} == {"1x1", "2x1", "2x2", "4x2", "4x4", "5x4", "6x4"}
        assert set(route) == {"kpart", "tiled", "gemv", "skinny"}
    route = routes([f"grouped {m} {g} {r} {k} 0 0" for m, g, r, k in grouped])
    form = routes([f"gform {m} {g} {r} {k}" for m, g, r, k in grouped])
    assert {f for f, r in zip(form, route) if r == "kpart"} == {"1x1", "1x2", "2x2", "2x4", "4x4", "6x4", "8x4"}
    assert "tiled" in route
