"""GPU parity of the grouped fp8-weight GEMM ("mgk,grk->mgr", the reference's wo_a projection): the reference-order
entry bit-exact against the CPU oracle, the fast entries (GEMV, tiled MFMA GEMM, reference-order fallback for
untileable shapes) within the bf16 bar, and the GEMV's fused output quantization bit-exact."""
import numpy as np
import pytest

import oracle
from tests.helpers import from_bf16, max_rel, randn_bf16
from unholy_amd import call
from unholy_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu


def dev(a):
    return DeviceBuffer.from_array(np.ascontiguousarray(a))


def _case(rng, M, G, R, K):
    a = randn_bf16(rng, (M, G, K))
    w = rng.integers(0, 256, (G * R, K), dtype=np.uint8)
    w[(w & 0x7F) == 0x7F] = 0  # no NaN codes
    sw = rng.integers(118, 126, ((G * R + 127) // 128, K // 128), dtype=np.uint8)
    return a, w, sw


@pytest.mark.parametrize("M,G,R,K", [(3, 2, 256, 256), (1, 8, 1024, 512), (5, 3, 200, 384), (40, 2, 128, 128)])
def test_grouped_fp8w_reference_order_bit_exact(M, G, R, K):
    rng = np.random.default_rng(M * 31 + R)
    a, w, sw = _case(rng, M, G, R, K)
    ref16, _ = oracle.gemm_grouped_fp8w(a, w, sw, G, R)
    c = DeviceBuffer(M * G * R * 2)
    call("uh_gemm_grouped_fp8w", dev(a), dev(w), dev(sw), c, M, G, R, K, None)
    got = c.download((M, G, R), np.uint16)
    print(f"grouped fp8w ref order M={M} G={G} R={R} K={K}: bit-identical fraction {np.mean(got == ref16):.6f}")
    assert np.array_equal(got, ref16)


# The row-tile kernel (up to 8 rows of at least 256 workgroups, G R = 8,192: one to four 2,048-input chunks, ragged K), the
# K-part kernel (ragged K, row remainders, the DSV4 shape), the reference order (R = 200), the tiled GEMM in 256-column
# tiles (more than 256 workgroups: M = 400, G R = 16,896).
@pytest.mark.parametrize("M,G,R,K", [(1, 8, 1024, 4096), (16, 2, 512, 1024), (32, 3, 256, 640), (7, 2, 200, 256),
                                     (33, 2, 256, 512), (100, 2, 256, 512), (200, 3, 128, 384), (300, 2, 384, 1024),
                                     (257, 2, 256, 512), (200, 3, 512, 384), (65, 2, 200, 256), (64, 8, 1024, 4096),
                                     (17, 2, 128, 768), (160, 2, 192, 3072), (48, 3, 64, 1152), (95, 1, 64, 9216),
                                     (4, 3, 96, 640), (16, 1, 32, 8192), (9, 2, 160, 5120), (1, 2, 64, 128),
                                     (384, 1, 64, 256), (385, 1, 128, 384), (400, 2, 256, 512), (520, 2, 384, 1024),
                                     (400, 1, 16896, 128), (7, 8, 1024, 640), (8, 8, 1024, 6144), (2, 8, 1024, 8192)])
def test_grouped_fp8w_fast_path(M, G, R, K):
    rng = np.random.default_rng(M * 7 + G * R + K)
    a, w, sw = _case(rng, M, G, R, K)
    ref16, _ = oracle.gemm_grouped_fp8w(a, w, sw, G, R)
    ref64 = oracle.gemm_grouped_fp8w_f64(a, w, sw, G, R)
    c = DeviceBuffer(M * G * R * 2)
    call("uh_gemm_grouped_fp8w_wmma", dev(a), dev(w), dev(sw), c, M, G, R, K, None)
    got = from_bf16(c.download((M, G, R), np.uint16))
    mr = max_rel(got, from_bf16(ref16))
    print(f"grouped fp8w fast M={M} G={G} R={R} K={K}: max_rel {mr:.3e} vs f64 {max_rel(got, ref64):.3e} "
          f"bit-identical {np.mean(got == from_bf16(ref16)):.4f}")
    assert mr <= 1e-2
    assert max_rel(got, ref64) <= 1e-2


@pytest.mark.parametrize("M", [1, 8, 32])
def test_gemv_grouped_fp8w_fused_quant(M):
    """The GEMV entry with GemvQuant: its bf16 outputs as the fast path's, and q / qs exactly act_quant_fp8 (block 128)
    of those outputs; the counters are left zero."""
    G, R, K = 4, 256, 512
    rng = np.random.default_rng(M)
    a, w, sw = _case(rng, M, G, R, K)
    da, dw, dsw = dev(a), dev(w), dev(sw)
    c = DeviceBuffer(M * G * R * 2)
    q, qs = DeviceBuffer(M * G * R), DeviceBuffer(M * G * R // 128)
    counters = dev(np.zeros(G * R // 128, np.uint32))
    call("uh_gemv_grouped_fp8w", da, dw, dsw, c, M, G, R, K, q, qs, counters, None)
    c_fast = DeviceBuffer(M * G * R * 2)
    call("uh_gemm_grouped_fp8w_wmma", da, dw, dsw, c_fast, M, G, R, K, None)
    out = c.download((M, G * R), np.uint16)
    assert np.array_equal(out, c_fast.download((M, G * R), np.uint16))
    q_ref, qs_ref = oracle.act_quant_fp8(out)
    assert np.array_equal(q.download((M, G * R), np.uint8), q_ref)
    assert np.array_equal(qs.download((M, G * R // 128), np.uint8), qs_ref)
    assert not counters.download((G * R // 128,), np.uint32).any()


def test_grouped_fp8w_shape_errors():
    a, w, sw = _case(np.random.default_rng(0), 2, 2, 128, 256)
    da, dw, dsw = dev(a), dev(w), dev(sw)
    c = DeviceBuffer(2 * 2 * 128 * 2)
    with pytest.raises(Exception, match="K % 128"):
        call("uh_gemm_grouped_fp8w_wmma", da, dw, dsw, c, 2, 2, 128, 200, None)
    with pytest.raises(Exception, match="M > 32"):
        call("uh_gemv_grouped_fp8w", da, dw, dsw, c, 33, 2, 128, 256, None, None, None, None)
    call("uh_gemm_grouped_fp8w_wmma", da, dw, dsw, c, 0, 2, 128, 256, None)  # M = 0: nothing to do



# The K-part kernel's forms (1 x 1 .. 8 x 4 row x column blocks of 16, 128- and 64-input slots; test_routes.py checks that
# every one is here): row remainders, R a multiple of 16 or 32 only, one 128-block, uneven K parts, more than eight blocks
# a wave (K = 9,216); the tiled kernel with row tiles that do and do not divide over the XCDs.
MID_SIZES = [(9, 8, 512, 256), (16, 8, 1024, 128), (30, 8, 1024, 256), (61, 8, 1024, 384), (100, 8, 1024, 128),
             (180, 8, 1024, 128), (250, 8, 1024, 256), (23, 5, 48, 1152), (70, 3, 96, 640), (12, 2, 16, 9216),
             (600, 8, 1024, 256), (1030, 16, 512, 128), (1000, 8, 1024, 128), (1170, 4, 1024, 128), (100, 8, 1024, 384),
             (180, 8, 1024, 512), (250, 8, 1024, 640), (500, 4, 1024, 640), (1000, 4, 1024, 128)]


@pytest.mark.parametrize("M,G,R,K", MID_SIZES)
def test_grouped_fp8w_mid_sizes(M, G, R, K):
    rng = np.random.default_rng(M * 5 + G * R + K)
    a, w, sw = _case(rng, M, G, R, K)
    ref16, _ = oracle.gemm_grouped_fp8w(a, w, sw, G, R)
    c = dev(np.full((M * G * R + 64,), 0x7FC1, np.uint16))
    call("uh_gemm_grouped_fp8w_wmma", dev(a), dev(w), dev(sw), c, M, G, R, K, None)
    got = c.download((M * G * R + 64,), np.uint16)
    assert np.all(got[M * G * R:] == 0x7FC1)
    assert max_rel(from_bf16(got[:M * G * R].reshape(M, G, R)), from_bf16(ref16)) <= 1e-2


@pytest.mark.parametrize("M,G,R,K", [(1, 8, 1024, 256), (12, 2, 128, 384), (200, 2, 64, 256), (5, 2, 40, 128)])
def test_grouped_fp8w_unaligned_operands(M, G, R, K):
    """Activations or weights 8 bytes off a 16-byte address: the kernels with plain loads."""
    rng = np.random.default_rng(M + K)
    a, w, sw = _case(rng, M, G, R, K)
    ref = from_bf16(oracle.gemm_grouped_fp8w(a, w, sw, G, R)[0])
    c, dsw = DeviceBuffer(M * G * R * 2), dev(sw)
    for ao, wo in ((8, 0), (0, 8)):
        bufs = []
        for v, o in ((a, ao), (w, wo)):
            b = DeviceBuffer(v.nbytes + o)
            call("uh_memcpy_h2d", b.ptr + o, v.ctypes.data, v.nbytes)
            bufs.append((b, b.ptr + o))
        c.zero()
        call("uh_gemm_grouped_fp8w_wmma", bufs[0][1], bufs[1][1], dsw, c, M, G, R, K, None)
        assert max_rel(from_bf16(c.download((M, G, R), np.uint16)), ref) <= 1e-2
