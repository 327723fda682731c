"""The C-ABI library loads and exports every entry point of
include/trnblas_hip.h (no GPU needed: no compute call is made)."""

import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "trnblas_hip.h")


def _declared():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"\b(trnblas_hip_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_surface():
    names = _declared()
    for n in ("trnblas_hip_gemm", "trnblas_hip_syrk", "trnblas_hip_pair_energy",
              "trnblas_hip_ozaki_split", "trnblas_hip_ozaki_gemm", "trnblas_hip_mp2_energy"):
        assert n in names


def test_library_exports_every_declared_symbol():
    from trnblas_amd.hip import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built (run __graft_entry__.build())")
    lib = _lib.load()
    missing = [n for n in _declared() if getattr(lib, n, None) is None]
    assert not missing, missing
    assert set(_declared()) == set(_lib.SIGNATURES), "ctypes signatures out of sync with the header"
    assert lib.trnblas_hip_abi_version() == _lib.ABI_VERSION
    assert lib.trnblas_hip_last_error() == b""


def test_argument_errors_are_reported_without_a_gpu():
    # invalid arguments are rejected before any HIP call
    from trnblas_amd.hip import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built")
    lib = _lib.load()
    rc = lib.trnblas_hip_gemm(7, 0, 0, 4, 4, 4, 1.0, None, 4, 0, None, 4, 0, 0.0, None, 4, 0,
                              None, 4, 0, 1, None, 0, None)
    assert rc == _lib.E_ARG and b"dtype" in lib.trnblas_hip_last_error()
    rc = lib.trnblas_hip_pack_k(0, 4, 5, None, 5, 1, 0, None, 4, 20, 1, None)
    assert rc == _lib.E_ARG and b"bad sizes" in lib.trnblas_hip_last_error()  # kp < K
    rc = lib.trnblas_hip_pack_k(1, 4, 5, None, 5, 1, 0, None, 8, 20, 2, None)
    assert rc == _lib.E_ARG and b"batch stride" in lib.trnblas_hip_last_error()
    assert lib.trnblas_hip_pack_k(0, 0, 5, None, 5, 1, 0, None, 8, 0, 1, None) == 0  # R == 0: nothing to do
    rc = lib.trnblas_hip_ozaki_gemm(0, 13, 4, 4, 128, 128, None, 128, 0, None, 128, 0, None,
                                    None, None, 4, 1, None)
    assert rc == _lib.E_ARG and b"slices" in lib.trnblas_hip_last_error()
    assert lib.trnblas_hip_pair_energy_workspace(672, 4656) == (4656 * 28 + 4656) * 8
    # bf16x6: partials (256-byte aligned), then 3 bf16 pieces of every
    # (occupied, virtual) row, virtual rows in pairs, naux rounded up to 64,
    # per operand.
    part = -(-((4656 * 28 + 4656) * 8) // 256) * 256
    pieces = 96 * 672 * 3 * 2304 * 2
    assert lib.trnblas_hip_pair_energy_bf16x6_workspace(672, 2304, 4656, 96, 0) == part + pieces
    odd = -(-(5 * 8 * 3 * 64 * 2) // 256) * 256  # nvir 7 -> 4 row pairs, naux 33 -> 64
    assert lib.trnblas_hip_pair_energy_bf16x6_workspace(7, 33, 3, 5, 5) == 256 + 2 * odd
    # the implicit walk shares one set of pieces (nj == 0) and needs ni >= nocc
    rc = lib.trnblas_hip_pair_energy_bf16x6(7, 33, 16, 2, 231, 16, 0, 231, 33, 16, 16, 16, 3,
                                            6, None, None, None, None, 16, 16, 4096, None)
    assert rc == _lib.E_ARG and b"ni >= nocc" in lib.trnblas_hip_last_error()
    # fp16x3: 2 fp16 pieces per element, then one int32 exponent per
    # (occupied, padded virtual) row, per operand
    pieces2 = 96 * 672 * 2 * 2304 * 2
    exps = -(-(96 * 672 * 4) // 256) * 256
    assert lib.trnblas_hip_pair_energy_fp16x3_workspace(672, 2304, 4656, 96, 0) == part + pieces2 + exps
    odd2 = -(-(5 * 8 * 2 * 64 * 2) // 256) * 256
    exps2 = -(-(5 * 8 * 4) // 256) * 256
    assert lib.trnblas_hip_pair_energy_fp16x3_workspace(7, 33, 3, 5, 5) == 256 + 2 * odd2 + 2 * exps2
    rc = lib.trnblas_hip_pair_energy_fp16x3(7, 33, 16, 2, 231, 16, 0, 231, 33, 16, 16, 16, 3,
                                            6, None, None, None, None, 16, 16, 4096, None)
    assert rc == _lib.E_ARG and b"ni >= nocc" in lib.trnblas_hip_last_error()


def test_syrk_and_triangle_argument_errors_without_a_gpu():
    # the device-decided triangle rule needs its flags when beta != 0, and
    # the triangle check needs an aligned int32[2]; both are refused before
    # any HIP call (the chol_block size bound too)
    import ctypes

    from trnblas_amd.hip import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built")
    lib = _lib.load()
    fake = ctypes.c_void_p(4096)  # never dereferenced: the calls fail their argument checks
    rc = lib.trnblas_hip_syrk_flagged(0, 0, 0, 8, 8, 1.0, fake, 8, 0.5, fake, 8, fake, 8, None,
                                      None, 0, None)
    assert rc == _lib.E_ARG and b"flags" in lib.trnblas_hip_last_error()
    rc = lib.trnblas_hip_triangle_nonzero(0, 8, fake, 8, ctypes.c_void_p(4100), None)
    assert rc == _lib.E_ARG and b"aligned" in lib.trnblas_hip_last_error()
    rc = lib.trnblas_hip_chol_block(129, fake, 129, fake, 129, fake, 0, None)
    assert rc == _lib.E_ARG and b"nb" in lib.trnblas_hip_last_error()


def _plan(dtype, syrk, ta, tb, M, N, K, batch=1):
    from trnblas_amd.hip import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built")
    name = _lib.load().trnblas_hip_gemm_plan(dtype, syrk, ta, tb, M, N, K, M if ta else K, K if tb else N, batch)
    assert name is not None, _lib.load().trnblas_hip_last_error()
    return name.decode()


F32, BF16, F16 = 0, 1, 2


@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K,batch,direct", [
    (64, 64, 2048, 1, True), (64, 64, 65536, 1, False), (128, 128, 32768, 1, False), (256, 256, 16384, 1, False),
    (8, 32, 276928, 4, False), (63, 61, 2047, 1, True), (63, 61, 65537, 1, False), (3, 20, 110293, 1, False),
    (1, 1, 1 << 22, 1, False),
])  # fmt: skip
def test_16bit_gemm_of_few_tiles_and_long_k_is_split(M, N, K, batch, direct, ta, tb):
    # hgemm_direct_kernel runs a tile's whole K in one workgroup: products of few
    # tiles and long K belong on the stream-K kernels
    for dtype in (BF16, F16):
        assert (_plan(dtype, 0, ta, tb, M, N, K, batch) == "hgemm_direct_kernel") == direct


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("n,k,direct", [(64, 2048, True), (64, 8192, False), (56, 181568, False), (59, 2047, True),
                                        (59, 132806, False), (13, 74125, False)])  # fmt: skip
def test_16bit_syrk_of_few_tiles_and_long_k_is_split(n, k, direct, trans):
    assert (_plan(BF16, 1, trans, 0, n, n, k) == "hgemm_direct_kernel") == direct


def test_gemm_plan_refuses_what_the_launch_refuses():
    from trnblas_amd.hip import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("library not built")
    lib = _lib.load()
    assert lib.trnblas_hip_gemm_plan(0, 0, 0, 0, 4, 1 << 24, 4, 4, 1 << 24, 1) is None
    assert b"32-bit panel offsets" in lib.trnblas_hip_last_error()
    assert lib.trnblas_hip_gemm_plan(7, 0, 0, 0, 4, 4, 4, 4, 4, 1) is None
    assert lib.trnblas_hip_gemm_plan(0, 1, 0, 0, 4, 5, 4, 4, 5, 1) is None


def test_16bit_one_round_kernel_counts_half_tiles():
    # gemm_dma_kernel's 128 x 64 tiles do half the work where N is at most 64: with
    # many k-tiles they are faster than hgemm128_kernel's whole 128 x 128 ones
    for M, N, K, b in ((408, 8, 10264, 37), (1168, 24, 6592, 17)):
        assert _plan(BF16, 0, 1, 0, M, N, K, b) == "gemm_dma_kernel narrow"
    assert _plan(BF16, 0, 0, 0, 1784, 2032, 2048) == "hgemm128_kernel"


@pytest.mark.parametrize("M,N,K,batch", [(1200, 256, 4792, 1), (816, 368, 4344, 1), (40, 232, 5544, 18)])
def test_16bit_gemm_of_a_tile_per_cu_and_long_k(M, N, K, batch):
    assert _plan(BF16, 0, 1, 0, M, N, K, batch) != "hgemm_direct_kernel"


def test_fp32_gemm_of_few_tiles_and_long_k_is_split():
    # unaligned products have no stream-K kernel: K goes over as many workgroups as
    # the chip holds, and no workgroup walks tens of thousands of k alone
    for K, least in ((65537, 64), (300001, 128), (1000001, 256)):
        name = _plan(F32, 0, 0, 0, 63, 63, K)
        assert name.startswith("sgemm_tile_kernel<64, 64> in") and int(name.split()[-1]) >= least, name
    assert "direct" not in _plan(F32, 0, 0, 0, 549, 174, 41161, 10)
    # aligned, N <= 64: narrow tiles are half the work
    assert _plan(F32, 0, 0, 1, 66, 3, 33628, 10) == "gemm_dma_kernel narrow"


@pytest.mark.parametrize("M,N,K,ta,tb,kernel", [
    # the larger tiles of the LDS-DMA kernel, also where its last round is half full
    (6144, 6144, 6144, 0, 1, "gemm_dma_kernel"), (6144, 6144, 6144, 1, 1, "gemm_dma_kernel"),
    (5620, 5620, 5620, 0, 1, "gemm_dma_kernel"), (1968, 1968, 1968, 0, 1, "gemm_dma_kernel narrow"),
    # a little over one 32 x 32 tile per CU and a long K: its second round costs a whole one
    (864, 404, 4940, 1, 0, "gemm_dma_kernel narrow"), (532, 648, 6152, 0, 0, "gemm_dma_kernel narrow"),
])  # fmt: skip
def test_aligned_fp32_gemm_stays_on_the_lds_dma_kernel_where_it_is_faster(M, N, K, ta, tb, kernel):
    assert _plan(F32, 0, ta, tb, M, N, K) == kernel
