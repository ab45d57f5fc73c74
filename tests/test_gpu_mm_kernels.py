"""Every kernel that zs_retiled_mm picks (zs_retiled_mm_kernel), on shapes at the
edges of its tiles: ragged column blocks, rows that are no multiple of 128,
slices of unequal length.  The result is compared with the float64 product."""
import numpy as np
import pytest

import oracle as zo
import zipserv_asplos26_amd as zs
from zs_testutil import from_torch_bf16, to_torch_bf16, weights_bf16

WIDE, WIDE2 = "zs::rgemm_wide_kernel<%s, 2>", "zs::rgemm_wide2_kernel<%s, 2>"

# (kernel, M, K, N, split_k)
CASES = [("zs::rgemm_kernel<1, 1, 4, 4, 1>", 4160, 1088, 1, 2),
         ("zs::rgemm_kernel<1, 1, 4, 4, 2>", 4160, 512, 3, 2),
         ("zs::rgemm_kernel<1, 1, 4, 4, 4>", 4160, 512, 7, 2),
         ("zs::rgemm_kernel<1, 1, 8, 4, 0>", 64, 512, 9, 3),
         ("zs::rgemm_kernel<1, 1, 8, 4, 1>", 320, 2560, 1, 1),
         ("zs::rgemm_kernel<1, 1, 8, 4, 2>", 320, 1088, 4, 3),
         ("zs::rgemm_kernel<1, 1, 8, 4, 4>", 64, 4096, 6, 4),
         ("zs::rgemm_kernel<1, 1, 4, 4, 4>", 12288, 4096, 8, 1),
         ("zs::rgemm_kernel<1, 1, 8, 4, 0>", 4096, 4096, 9, 2),
         (WIDE % "1, 4, 4", 5120, 5120, 8, 2),
         ("zs::rgemm_kernel<2, 1, 4, 3, 0>", 4160, 512, 13, 2),
         ("zs::rgemm_kernel<2, 1, 8, 3, 0>", 1984, 512, 16, 4),
         (WIDE % "1, 4, 2", 4160, 512, 1, 4), (WIDE % "1, 4, 2", 8192, 1088, 9, 3),
         (WIDE % "1, 4, 4", 320, 1024, 45, 4), (WIDE % "1, 4, 4", 64, 64, 500, 1),
         (WIDE % "2, 4, 2", 1984, 512, 33, 3), (WIDE % "2, 4, 2", 1984, 64, 129, 1),
         (WIDE % "2, 4, 4", 320, 1088, 500, 2), (WIDE % "2, 4, 4", 4160, 1088, 17, 2),
         (WIDE % "3, 4, 4", 1984, 1088, 129, 2), (WIDE % "3, 4, 4", 4160, 1088, 100, 1),
         (WIDE % "4, 4, 2", 1984, 512, 65, 3), (WIDE % "4, 4, 2", 4160, 64, 113, 1),
         (WIDE % "4, 4, 4", 1984, 1088, 500, 1), (WIDE % "4, 4, 4", 1984, 2560, 100, 3),
         (WIDE % "8, 4, 2", 1984, 1088, 129, 4), (WIDE % "8, 4, 2", 12288, 64, 65, 1),
         (WIDE % "8, 4, 3", 1984, 6400, 129, 4), (WIDE2 % "2, 8", 12288, 64, 129, 1),
         (WIDE2 % "2, 8", 12288, 512, 17, 3), (WIDE2 % "4, 8", 14336, 512, 33, 4),
         (WIDE2 % "8, 8", 12288, 64, 200, 1), (WIDE2 % "8, 8", 6144, 512, 65, 4)]


def test_kernel_of_every_shape_is_named():
    lib = zs.lib()
    for M, K in ((64, 64), (320, 1024), (4096, 14336), (28672, 4096)):
        for N in (1, 16, 17, 500, 100000):
            for split_k in (1, 4):
                name = lib.zs_retiled_mm_kernel(M, N, K, split_k)
                refused = split_k > K // 64 or M * N * split_k > 2 * (2**31 - 1)
                assert (name is None) == refused, (M, K, N, split_k)
    # the last two: 2^32 outputs, records of a band past 2^32 bytes
    for bad in ((63, 1, 64, 1), (64, 0, 64, 1), (64, 1, 32, 1), (64, 1, 64, 0),
                (28672, 200000, 64, 1), (64, 1, 64 * 3050403, 1)):
        assert lib.zs_retiled_mm_kernel(*bad) is None
        # refused by the GEMM too, before any pointer is used
        assert lib.zs_retiled_mm(None, 16, 16, 16, 0, 16, 16, *bad[:2], bad[2], 16, bad[3]) < 0


def test_kernel_of_row_blocks_is_that_of_the_full_ones():
    # 2 * N * K past INT32_MAX: blocks of 8176 rows
    lib, K, full = zs.lib(), 131072, (2**31 - 1) // (2 * 131072) // 16 * 16
    assert full == 8176
    for N in (full + 100, 2 * full - 1, 3 * full):
        for split_k in (1, 4):
            assert lib.zs_retiled_mm_kernel(64, N, K, split_k) == \
                lib.zs_retiled_mm_kernel(64, full, K, split_k)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel,M,K,N,split_k", CASES)
def test_kernel_equals_the_float64_product(torch_cuda, kernel, M, K, N, split_k):
    torch = torch_cuda
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert zs.lib().zs_retiled_mm_kernel(M, N, K, split_k).decode() == kernel
    rng = np.random.default_rng(M + K + N + split_k)
    W = weights_bf16(rng, (M, K), outlier_frac=0.01)
    X = zo.f32_to_bf16(rng.standard_normal((N, K), dtype=np.float32))
    r, x = zs.compress_retiled(to_torch_bf16(W)), to_torch_bf16(X)
    y = zs.zipgemm(r, x, split_k=split_k)
    two = zs.zipgemm(r, x, split_k=split_k, fused=False)
    torch.cuda.synchronize()
    got = from_torch_bf16(y)
    np.testing.assert_array_equal(got, from_torch_bf16(two))
    w, v = zo.bf16_to_f32(W).astype(np.float64), zo.bf16_to_f32(X).astype(np.float64)
    step = ((K // 64 - 1) // split_k + 1) * 64
    parts = [v[:, k:k + step] @ w[:, k:k + step].T for k in range(0, K, step)]
    exact = sum(parts)
    # unit roundoff 2^-8 of the result and, split, of every partial sum (and
    # of the result again for what those move it), and the fp32 sums: K terms
    # of 2^-24 of sum |w x|
    eps = 2.0 ** -8
    fp32 = K * 2.0 ** -24 * (np.abs(v) @ np.abs(w).T)
    part = eps * sum(np.abs(p) for p in parts) + fp32 if split_k > 1 else fp32
    bound = eps * np.abs(exact) + (1 + eps) * part
    err = np.abs(zo.bf16_to_f32(got).astype(np.float64) - exact)
    assert np.all(err <= bound), float(np.max(err - bound))
