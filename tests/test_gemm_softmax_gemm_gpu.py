"""GPU parity: batched fused GEMM + softmax + GEMM ("attention", fp16) through the C ABI against the CPU
oracle -- ReferenceBatchedGemm with element_wise::Scale, the upper-triangle mask, ReferenceSoftmax over n
(reference_softmax.hpp:56-117) and a second ReferenceBatchedGemm, the chain upstream's
batched_gemm_scale_softmax_gemm example verifies with. The fused operator is absent from the reference
snapshot; the oracle chain is pinned bit for bit against those reference pieces in tests/test_oracle.py.
This row is TOLERANCE-ONLY, by construction: rtol = atol = 1e-2. The kernel rounds the unnormalised
probabilities exp(s - max) to fp16 (they are the A operand of the second MFMA GEMM) and divides the fp32
result by the row sum afterwards; the reference divides first and rounds the normalised probabilities. The two
round different numbers, so outputs differ by a few fp16 units in the last place of the probabilities (relative
2^-11 each, accumulated over n): a comparison at 1e-3 fails on a share of the elements for this reason alone,
and no reordering inside the kernel can make the row bit-exact without giving up the fused second GEMM.
What the mathematics fixes exactly is still checked exactly (uniform rows, one-hot rows, the masked first row)."""
import numpy as np
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi
from composable_kernel_amd.host_tensor import uniform_f16
from oracle import fast, lit

pytestmark = pytest.mark.gpu
RTOL = ATOL = 1e-2


def _close(out, ref):
    assert np.all(np.isfinite(out.astype(np.float32)))
    bad, max_err = lit.check_err_f16(out, ref, RTOL, ATOL)
    assert bad == 0, f"{bad} outside tolerance, max err {max_err}"


def _run(a_gmk, b0_gnk, b1_gno, scale=1.0, mask=False, instance=capi.INSTANCE_AUTO, pad=(0, 0, 0, 0), gap=0.0):
    """pad: extra elements per row of A, B0, B1, C (row strides larger than the extents), those of the operands filled with gap."""
    import torch
    import gpu_util
    G, M, K = a_gmk.shape
    N, O = b0_gnk.shape[1], b1_gno.shape[2]

    def padded(x, p):
        out = np.full(x.shape[:2] + (x.shape[2] + p,), gap, np.float16)
        out[..., :x.shape[2]] = x
        return out

    ha, hb0, hb1 = padded(a_gmk, pad[0]), padded(b0_gnk, pad[1]), padded(b1_gno, pad[2])
    da, db0, db1 = (torch.from_numpy(x.view(np.int16)).cuda() for x in (ha, hb0, hb1))
    dc = torch.full((G, M, O + pad[3]), 0x7E00, dtype=torch.int16, device="cuda")
    op = ck.DeviceBatchedGemmSoftmaxGemmF16(instance, MaskOutUpperTriangle=mask)
    arg = op.MakeArgumentPointer(da, db0, db1, dc, M, N, K, O, G, K + pad[0], K + pad[1], O + pad[2], O + pad[3],
                                 M * (K + pad[0]), N * (K + pad[1]), N * (O + pad[2]), M * (O + pad[3]),
                                 None, None, ck.Scale(scale))
    assert op.IsSupportedArgument(arg), capi.last_error()
    op.MakeInvokerPointer().Run(arg, ck.StreamConfig(gpu_util.stream()))
    torch.cuda.synchronize()
    out = dc.cpu().numpy().view(np.float16)
    if pad[3]:
        assert np.all(out[..., O:].view(np.uint16) == 0x7E00), "wrote outside the C rows"
    return out[..., :O]


SHAPES = [
    # G, M, N, K, O
    (3, 128, 128, 64, 64), (2, 200, 136, 64, 64), (2, 96, 512, 32, 64), (1, 130, 260, 128, 128),
    (2, 64, 72, 40, 24), (5, 16, 8, 8, 8), (1, 256, 300, 96, 128), (2, 40, 1, 16, 16), (1, 1, 257, 64, 64),
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("instance", [capi.INSTANCE_AUTO, 1, 2])
def test_gemm_softmax_gemm_shapes(shape, mask, instance):
    G, M, N, K, O = shape
    a = uniform_f16((G, M, K), -1, 1, 1900 + M)
    b0_gnk = uniform_f16((G, N, K), -1, 1, 1901 + N)
    b1 = uniform_f16((G, N, O), -1, 1, 1902 + O)
    scale = 1.0 / np.sqrt(K)
    out = _run(a, b0_gnk, b1, scale, mask, instance)
    _close(out, lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, scale, mask))


@pytest.mark.parametrize("G, M, N", [(1, 300, 300), (8, 260, 260), (65, 140, 140), (127, 129, 60), (128, 257, 257),
                                     (130, 130, 130), (200, 129, 200)])
def test_gemm_softmax_gemm_masked_slab_order(G, M, N):
    """The masked launch deals its slabs out over groups of 64 to 127 batches: batch counts at the groups' edges."""
    a, b0_gnk, b1 = (uniform_f16((G, x, 16), -1, 1, 1950 + i) for i, x in enumerate((M, N, N)))
    for instance in (capi.INSTANCE_AUTO, 1):
        _close(_run(a, b0_gnk, b1, 0.25, True, instance),
               lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, 0.25, True))


@pytest.mark.parametrize("N", [1, 31, 32, 33, 64, 65, 96, 97, 127, 129, 160, 225, 256])
@pytest.mark.parametrize("K", [32, 64, 128])
def test_gemm_softmax_gemm_edge_pairs(N, K):
    """Steps with masked columns multiply only the 32-column pairs that hold an unmasked one: N around the pairs' edges, rows
    above, on and below the diagonal of every wave."""
    a, b0_gnk, b1 = (uniform_f16((2, x, K), -1, 1, 1960 + i) for i, x in enumerate((161, N, N)))
    for mask in (False, True):
        ref = lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, 0.3, mask)
        for instance in (0, 1, 2):
            _close(_run(a, b0_gnk, b1, 0.3, mask, instance), ref)


@pytest.mark.parametrize("K, O", [(32, 32), (16, 64), (64, 64), (72, 40), (80, 80), (96, 96), (24, 104), (128, 32), (128, 128), (32, 128)])
def test_gemm_softmax_gemm_units(K, O):
    """The 32-row kernel walks N in units of 64 columns (32 with K past 96 or O past 96), the first, an even number in the middle and
    the last ones in code of their own: N around whole units, one to more than six of them, rows past the last wave's."""
    for N in (1, 63, 64, 65, 127, 129, 191, 193, 257, 320, 385):
        a, b0_gnk, b1 = (uniform_f16((2, x, y), -1, 1, 1970 + i) for i, (x, y) in enumerate(((133, K), (N, K), (N, O))))
        for mask in (False, True):
            _close(_run(a, b0_gnk, b1, 2.0 * K ** -0.5, mask, 0),
                   lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, 2.0 * K ** -0.5, mask))


@pytest.mark.parametrize("K, O", [(8, 8), (24, 104), (40, 24), (72, 40), (104, 72)])
def test_gemm_softmax_gemm_row_gaps_are_not_read(K, O):
    """K and O that leave chunks of a padded fragment row empty, NaNs between the rows of A, B0 and B1: units before, at and past the
    last one, whose rows and chunks that do not exist read as zeros."""
    for N in (64, 200, 257, 385):
        a, b0_gnk, b1 = (uniform_f16((2, x, y), -1, 1, 1980 + i) for i, (x, y) in enumerate(((133, K), (N, K), (N, O))))
        for mask in (False, True):
            ref = lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, K ** -0.5, mask)
            for instance in (0, 2):
                _close(_run(a, b0_gnk, b1, K ** -0.5, mask, instance, (8, 24, 16, 8), np.nan), ref)


@pytest.mark.parametrize("step", [0.01, 0.05, 0.2, 1.0])
def test_gemm_softmax_gemm_growing_scores(step):
    """The 32-row kernel rescales a unit after the maximum has risen, once the unit before has been added: scores that rise by step per
    column, so that every unit raises it, in one row of a wave or in all of them. Against float64, within four times the difference
    measured for scores that do not rise (2.5e-4 of the 2-norm; a probability is rounded to 2^-11 of itself)."""
    G, M, N, K, O = 1, 96, 640, 16, 64
    a = uniform_f16((G, M, K), -1, 1, 31)
    a[..., 0] = 0
    b0 = uniform_f16((G, N, K), -1, 1, 32)
    b0[0, :, 0] = (step * np.arange(N)).astype(np.float16)
    b1 = uniform_f16((G, N, O), -1, 1, 33)
    for rows in (slice(0, M), slice(37, 38)):
        x = a.copy()
        x[0, rows, 0] = 1
        for mask in (False, True):
            s = x[0].astype(np.float64) @ b0[0].astype(np.float64).T
            if mask:
                s = np.where(np.arange(N)[None, :] > np.arange(M)[:, None], -np.inf, s)
            p = np.exp(s - s.max(axis=1, keepdims=True))
            ref = (p / p.sum(axis=1, keepdims=True)) @ b1[0].astype(np.float64)
            out = _run(x, b0, b1, 1.0, mask, 0)[0].astype(np.float64)
            assert np.linalg.norm(out - ref) <= 1e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize("instance", [0, 2])
def test_gemm_softmax_gemm_nan_stays_in_its_row(instance):
    """A NaN in a row of A reaches that row of C only, and an infinity in a row of B1 that is masked for a whole wave reaches none of
    that wave's rows."""
    G, M, N, K, O = 1, 256, 256, 64, 64
    a, b0, b1 = (uniform_f16((G, x, 64), -1, 1, 41 + i) for i, x in enumerate((M, N, N)))
    clean = _run(a, b0, b1, 0.125, True, instance)
    for row in (0, 5, 21, 100, 255):
        x = a.copy()
        x[0, row, 3] = np.nan
        out = _run(x, b0, b1, 0.125, True, instance)
        assert np.all(np.isnan(out[0, row]))
        keep = np.arange(M) != row
        np.testing.assert_array_equal(out[0, keep].view(np.uint16), clean[0, keep].view(np.uint16))
    for n in (32, 96, 224):
        x = b1.copy()
        x[0, n] = np.inf
        out = _run(a, b0, x, 0.125, True, instance)
        np.testing.assert_array_equal(out[0, :n].view(np.uint16), clean[0, :n].view(np.uint16))


@pytest.mark.parametrize("G, M, N, K, mask, rows", [(2, 64, 1024, 64, False, 16), (2, 64, 1025, 64, False, 32), (129, 64, 960, 64, False, 16),
                                                    (129, 64, 961, 64, False, 32), (512, 128, 192, 64, True, 16), (513, 128, 192, 64, True, 32),
                                                    (304, 128, 513, 64, True, 16), (305, 128, 513, 64, True, 32), (352, 128, 640, 64, True, 16),
                                                    (353, 128, 640, 64, True, 32), (384, 128, 1023, 40, True, 16), (385, 128, 768, 64, True, 32),
                                                    (257, 128, 1024, 64, True, 32),
                                                    (256, 100, 192, 128, False, 16), (257, 100, 192, 128, False, 32), (512, 128, 192, 128, True, 16),
                                                    (513, 128, 192, 128, True, 32), (2, 64, 447, 32, False, 16), (2, 64, 448, 32, False, 32),
                                                    (2, 64, 192, 80, False, 32), (2, 128, 192, 96, True, 32)])
def test_gemm_softmax_gemm_auto_on_both_sides_of_its_rule(G, M, N, K, mask, rows):
    """AUTO takes 16-row waves for few slabs of a short N, 32-row waves otherwise: bit for bit the one, and not the other."""
    a, b0, b1 = (uniform_f16((G, x, K), -1, 1, 51 + i) for i, x in enumerate((M, N, N)))
    out = _run(a, b0, b1, K ** -0.5, mask)
    by_rows = {16: _run(a, b0, b1, K ** -0.5, mask, 2), 32: _run(a, b0, b1, K ** -0.5, mask, 0)}
    np.testing.assert_array_equal(out.view(np.uint16), by_rows[rows].view(np.uint16))
    assert np.any(out.view(np.uint16) != by_rows[48 - rows].view(np.uint16)), "both kernels give the same: this shape shows nothing"
    _close(out[:2], lit.batched_gemm_softmax_gemm_f16(a[:2], b0[:2].transpose(0, 2, 1), b1[:2], K ** -0.5, mask))


@pytest.mark.parametrize("instance", [0, 2])
def test_gemm_softmax_gemm_closed_forms(instance):
    """Zero scores: the uniform distribution, C = mean of B1's rows (exact: small integers over a power of
    two). Upper-triangle mask: row m averages rows 0..m, row 0 is B1[0] exactly. A dominant score selects
    one row of B1 exactly."""
    G, M, N, K, O = 2, 160, 256, 32, 64
    b1 = (np.arange(G * N * O).reshape(G, N, O) % 7).astype(np.float16)
    a0 = np.zeros((G, M, K), np.float16)
    b0 = uniform_f16((G, N, K), -1, 1, 71)
    out = _run(a0, b0, b1, instance=instance)
    np.testing.assert_array_equal(out, np.broadcast_to(b1.astype(np.float32).mean(axis=1, keepdims=True),
                                                       (G, M, O)).astype(np.float16))
    out = _run(a0, b0, b1, mask=True, instance=instance)
    np.testing.assert_array_equal(out[:, 0], b1[:, 0])
    for m in (1, 3, 7, 127, 159):        # m + 1 a power of two, or within fp16 rounding otherwise
        want = b1[:, :m + 1].astype(np.float64).mean(axis=1)
        assert np.abs(out[:, m].astype(np.float64) - want).max() <= 4e-3
    a = np.zeros((G, M, K), np.float16)
    a[:, np.arange(M), np.arange(M) % K] = 1
    b0h = np.zeros((G, N, K), np.float16)
    b0h[:, (np.arange(K) * 5) % N, np.arange(K)] = 40
    out = _run(a, b0h, b1, instance=instance)
    np.testing.assert_array_equal(out, b1[:, ((np.arange(M) % K) * 5) % N])


@pytest.mark.parametrize("instance", [0, 2])
def test_gemm_softmax_gemm_running_maximum_is_rescaled(instance):
    """The row maximum sits in the LAST 128-column step and the early steps hold large negative scores, and
    the other way round: the one-pass softmax must rescale what it accumulated."""
    G, M, N, K, O = 1, 64, 512, 16, 32
    a = np.zeros((G, M, K), np.float16)
    a[..., 0] = 1
    b1 = uniform_f16((G, N, O), -1, 1, 5)
    for ramp in (np.linspace(-30, 8, N), np.linspace(8, -30, N)):
        b0 = np.zeros((G, N, K), np.float16)
        b0[0, :, 0] = ramp.astype(np.float16)
        out = _run(a, b0, b1, instance=instance)
        _close(out, lit.batched_gemm_softmax_gemm_f16(a, b0.transpose(0, 2, 1), b1))
        # scores far apart (neighbours differ by 0.074 * 300): the result is the row of B1 at the maximum
        out = _run(a, b0, b1, scale=300.0, instance=instance)
        np.testing.assert_array_equal(out[0], np.broadcast_to(b1[0, int(np.argmax(b0[0, :, 0]))], (M, O)))


@pytest.mark.parametrize("instance", [0, 2])
def test_gemm_softmax_gemm_negative_scale(instance):
    """A negative scale turns the softmax towards the SMALLEST raw score (the kernel moves the sign into A)."""
    G, M, N, K, O = 2, 96, 300, 32, 32
    a = uniform_f16((G, M, K), -1, 1, 21)
    b0_gnk = uniform_f16((G, N, K), -1, 1, 22)
    b1 = uniform_f16((G, N, O), -1, 1, 23)
    for mask in (False, True):
        out = _run(a, b0_gnk, b1, -0.7, mask, instance)
        _close(out, lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, -0.7, mask))
        # same as a positive scale on the negated A
        np.testing.assert_array_equal(out.view(np.uint16), _run(-a, b0_gnk, b1, 0.7, mask, instance).view(np.uint16))


@pytest.mark.parametrize("instance", [0, 2])
def test_gemm_softmax_gemm_padded_strides_and_scale_zero(instance):
    G, M, N, K, O = 3, 72, 200, 64, 48
    a = uniform_f16((G, M, K), -1, 1, 11)
    b0_gnk = uniform_f16((G, N, K), -1, 1, 12)
    b1 = uniform_f16((G, N, O), -1, 1, 13)
    out = _run(a, b0_gnk, b1, 0.125, False, instance, pad=(8, 16, 24, 8))
    _close(out, lit.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, 0.125))
    # scale 0 makes the scores irrelevant: same result as A = 0
    np.testing.assert_array_equal(_run(a, b0_gnk, b1, 0.0, False, instance).view(np.uint16),
                                  _run(np.zeros_like(a), b0_gnk, b1, 1.0, False, instance).view(np.uint16))


@pytest.mark.parametrize("mask", [False, True])
def test_gemm_softmax_gemm_config5_shape(mask):
    """Benchmark configuration 5's shapes with the softmax in between: batch 64, 512 x 512 scores, K = O = 64."""
    G, M, N, K, O = 64, 512, 512, 64, 64
    a = uniform_f16((G, M, K), -1, 1, 1910)
    b0_gnk = uniform_f16((G, N, K), -1, 1, 1911)
    b1 = uniform_f16((G, N, O), -1, 1, 1912)
    out = _run(a, b0_gnk, b1, 0.125, mask)
    _close(out, fast.batched_gemm_softmax_gemm_f16(a, b0_gnk.transpose(0, 2, 1), b1, 0.125, mask))
    for g in (0, 63):
        _close(out[g:g + 1], lit.batched_gemm_softmax_gemm_f16(a[g:g + 1], b0_gnk[g:g + 1].transpose(0, 2, 1),
                                                               b1[g:g + 1], 0.125, mask))
    # rows of the output are convex combinations of B1's rows
    assert np.all(out.astype(np.float32).max(axis=1) <= b1.astype(np.float32).max(axis=1) + 1e-3)
    # batches are independent
    perm = np.random.default_rng(4).permutation(G)
    np.testing.assert_array_equal(_run(a[perm], b0_gnk[perm], b1[perm], 0.125, mask).view(np.uint16),
                                  out[perm].view(np.uint16))


def test_gemm_softmax_gemm_refused_arguments_and_empty_sum():
    import torch
    d = torch.zeros(1 << 16, dtype=torch.int16, device="cuda")
    op = ck.DeviceBatchedGemmSoftmaxGemmF16()
    # K above 128 is not built; a non-finite scale is invalid
    assert not op.IsSupportedArgument(op.MakeArgumentPointer(d, d, d, d, 64, 64, 256, 64, 1, 256, 256, 64, 64, 0, 0, 0, 0))
    assert not op.IsSupportedArgument(op.MakeArgumentPointer(d, d, d, d, 64, 64, 64, 64, 1, 64, 64, 64, 64, 0, 0, 0, 0,
                                                             None, None, ck.Scale(float("inf"))))
    with pytest.raises(TypeError):
        op.MakeArgumentPointer(d, d, d, d, 64, 64, 64, 64, 1, 64, 64, 64, 64, 0, 0, 0, 0, None, None, ck.AddRelu())
    assert capi.lib().ckx_num_instances(capi.OP_BATCHED_GEMM_SOFTMAX_GEMM) == 3
    assert b"SoftmaxGemm" in capi.lib().ckx_instance_name(capi.OP_BATCHED_GEMM_SOFTMAX_GEMM, 0)
    # N = 0: an empty sum, C = 0
    for instance in (0, 2):
        out = _run(np.ones((1, 16, 8), np.float16), np.zeros((1, 0, 8), np.float16), np.zeros((1, 0, 8), np.float16), instance=instance)
        np.testing.assert_array_equal(out, np.zeros((1, 16, 8), np.float16))


@pytest.mark.parametrize("G, M, N, K, O", [
    (2, 1, 576, 32, 32), (2, 133, 600, 16, 24), (1, 200, 641, 64, 64), (3, 64, 1026, 40, 24), (3, 65, 700, 40, 72), (1, 320, 673, 128, 128), (2, 64, 645, 24, 104),
    (1, 129, 999, 128, 32), (1, 66, 1536, 80, 80), (2, 70, 1570, 96, 72), (1, 1100, 1100, 64, 32),             # four shares of the columns
    (2, 133, 769, 80, 80), (1, 260, 801, 72, 96), (97, 65, 641, 64, 64), (97, 66, 577, 32, 32), (98, 70, 608, 128, 120), (99, 65, 800, 48, 104),
    (97, 128, 900, 104, 16), (1, 300, 1030, 96, 40),                                                           # two
    (193, 129, 640, 32, 32), (2, 100, 575, 32, 32), (2, 133, 639, 64, 64)])                                    # one (past the lines, and below)
def test_gemm_softmax_gemm_column_shares(G, M, N, K, O):
    """Launches of few workgroups deal the columns out to groups of waves and merge their sums: shares without columns (a causal slab's
    later ones, units that do not divide), rows past M, scores that rise so that the last share holds every maximum or fall so that the
    first does, NaNs between the rows. Against the oracle, and against the kernel with one share (instance 0): both round p to 2^-11 of
    itself, at different running maxima, and the result to 2^-11, so they differ by at most 2^-9 of the sum of p |B1| <= 1."""
    a, b0, b1 = (uniform_f16((G, x, y), -1, 1, 1990 + i) for i, (x, y) in enumerate(((M, K), (N, K), (N, O))))
    a[..., 0] = 1
    for mask in (False, True):
        for slope in (0, 8, -8):
            b0[..., 0] = (slope * np.arange(N) / N).astype(np.float16)
            out = _run(a, b0, b1, K ** -0.5, mask, pad=(8, 24, 16, 8), gap=np.nan)
            one = _run(a, b0, b1, K ** -0.5, mask, 0)
            assert np.max(np.abs(out.astype(np.float64) - one)) <= 2.0 ** -9
            _close(out[-1:], lit.batched_gemm_softmax_gemm_f16(a[-1:], b0[-1:].transpose(0, 2, 1), b1[-1:], K ** -0.5, mask))


@pytest.mark.parametrize("G, M, N, rows", [(48, 865, 865, 16), (52, 772, 772, 32), (44, 794, 794, 32), (24, 2083, 2083, 16), (24, 2499, 2499, 32), (28, 1909, 1909, 16),
                                           (31, 1970, 1970, 32), (45, 1066, 1066, 32), (32, 1588, 1588, 16), (40, 946, 946, 16), (64, 577, 577, 16), (64, 576, 576, 32),
                                           (8, 6472, 809, 32), (33, 1160, 893, 32), (16, 3101, 3101, 16)])
def test_causal_wide_heads_past_one_workgroup_a_cu(G, M, N, rows):
    """256 to 512 slabs: 16-row waves where the slabs that start second end before the longest chain, and the chains are long or the XCDs have whole
    batches, 32-row waves otherwise (csrc/gemm_gemm.hpp, rows_in_16s). Bit for bit the one kernel, and not the other."""
    a, b0, b1 = (uniform_f16((G, x, 128), -1, 1, 61 + i) for i, x in enumerate((M, N, N)))
    out = _run(a, b0, b1, 128 ** -0.5, True).view(np.uint16)
    by_rows = {16: _run(a, b0, b1, 128 ** -0.5, True, 2).view(np.uint16), 32: _run(a, b0, b1, 128 ** -0.5, True, 0).view(np.uint16)}
    assert np.array_equal(out, by_rows[rows]) and np.any(out != by_rows[48 - rows])
