"""Which GEMMs ask for a workspace for copies of their operands: K no whole number of 16-byte vectors, and work enough. Runs on the CPU."""
import pytest

import composable_kernel_amd as ck
from composable_kernel_amd import capi


@pytest.mark.parametrize("es, query", [(1, "ckx_gemm_i8_workspace_bytes"), (2, "ckx_gemm_f16_workspace_bytes"), (2, "ckx_gemm_bf16_workspace_bytes")])
def test_workspace_for_copies(es, query):
    need = getattr(capi.lib(), query)
    rows = 2049 + 2047
    assert need(2049, 2047, 2047, -1) == rows * 2048 * es                      # rows of whole 128-byte lines
    assert need(2049, 2047, 2049, -1) == rows * (2048 * es + 128)
    assert need(2049, 2047, 2048, -1) == 0 and need(64, 3001, 2049, -1) == 0    # whole vectors; little work
    assert need(3934, 139, 3815, -1) == 0                                      # more bytes to copy than the product repays
    generic = capi.lib().ckx_num_instances(capi.OP_GEMM_I8) - 1
    assert need(2049, 2047, 2047, generic) == 0                                # AUTO only
    split = need(600, 600, 16000, -1)
    assert split > 0 and need(600, 600, 15999, -1) == split + 1200 * 16000 * es # the copies come on top of the K runs' slices


@pytest.mark.parametrize("op, es", [(capi.OP_GEMM_I8, 1), (capi.OP_GEMM_F16, 2), (capi.OP_GEMM_BF16, 2)])
def test_plan_of_a_copied_product(op, es):
    """The query answers for the launch with copies: no instance index has it, and its K runs are those on the copies."""
    def plan(M, N, K, ws, **kw):
        return capi.gemm_plan(op, M, N, K, workspace_bytes=ws, **kw)
    generic = capi.lib().ckx_num_instances(op) - 1
    M, N, K = 2049, 2047, 2047
    copies = (M + N) * 2048 * es
    assert plan(M, N, K, copies) == (capi.INSTANCE_AUTO, 1)
    assert plan(M, N, K, copies - 1) == plan(M, N, K, 0) == (generic, 1)        # no room for both copies
    assert plan(M, N, K, 1 << 30, instance=generic) == (generic, 1)            # as asked for
    assert plan(M, N, K, 1 << 30, batch=2, sa=K, sb=K) == (generic, 1)          # batches are not copied
    assert plan(64, 3001, 2049, 1 << 30) == (generic, 1)                       # little work
    kn = dict(b_layout=capi.ROW_MAJOR)
    assert plan(2049, 2047, 1023, 1 << 30, **kn) == (generic, 1) and plan(2049, 2047, 2047, 1 << 30, **kn)[0] == capi.INSTANCE_AUTO
    # what is left of the workspace holds the K runs' slices, or not
    copies, room = 1200 * 16000 * es, 1 << 28
    runs = plan(600, 600, 16000, room)[1]
    assert runs > 1
    assert plan(600, 600, 15999, copies + room) == (capi.INSTANCE_AUTO, runs) and plan(600, 600, 15999, copies) == (capi.INSTANCE_AUTO, 1)
    assert capi.lib().ckx_instance_name(op, capi.INSTANCE_AUTO).endswith(b"<auto>")


@pytest.mark.parametrize("device_op, functor", [
    (ck.DeviceGemmInt8, None), (ck.DeviceGemmF16, None), (ck.DeviceGemmBF16, None), (ck.DeviceGemmMultipleDF16, ck.Bilinear(0.5, 2.0)),
    (ck.DeviceGemmMultipleDInt8, ck.ActivationMul2Clamp(ck.Relu()))])
def test_workspace_of_k_major_operands(device_op, functor):
    """The operators ask for room for copies where their layouts are copied, and for none where they are not."""
    def need(al, bl, M, N, K):
        op = device_op(ALayout=al, BLayout=bl)
        a, b = (M if al is ck.ColumnMajor else K), (N if bl is ck.RowMajor else K)
        if functor is None:
            return op.GetWorkSpaceSize(op.MakeArgumentPointer(0, 0, 0, M, N, K, a, b, N))
        return op.GetWorkSpaceSize(op.MakeArgumentPointer(0, 0, [0], 0, M, N, K, a, b, [0], N, None, None, functor))
    row, col = ck.RowMajor, ck.ColumnMajor
    es = 1 if "Int8" in device_op.__name__ else 2
    copies = lambda M, N, K: (M + N) * -(-K * es // 128) * 128
    assert need(row, col, 2049, 2047, 1023) == copies(2049, 2047, 1023)
    for al, bl in ((row, row), (col, col), (col, row)):
        assert need(al, bl, 2049, 2047, 1023) == 0                             # 8.6e9 operations
        assert need(al, bl, 2049, 2047, 2047) == copies(2049, 2047, 2047)      # 17e9


def test_lines_of_the_copies():
    """Both sides of what decides, each measured (csrc/ckx_api.hip, packing_pays): level or slower products stay without copies."""
    f16, i8 = capi.lib().ckx_gemm_f16_workspace_bytes, capi.lib().ckx_gemm_i8_workspace_bytes
    for M, N, K in ((3878, 661, 1053), (2030, 1381, 791), (2445, 1107, 1007), (2545, 869, 1005),    # short K, three tiles a CU
                    (305, 2995, 3385), (316, 3263, 2979), (970, 915, 2899),                        # one tile a CU
                    (251, 3973, 3783), (3943, 219, 3135), (4004, 285, 1969)):                      # thin
        assert f16(M, N, K, -1) == 0, (M, N, K)
    for M, N, K in ((2001, 1003, 1025), (1500, 901, 2001), (2428, 1503, 577), (838, 3089, 1289), (797, 903, 4069), (3001, 333, 3001), (1728, 3153, 493),
                    (1000, 1000, 8001)):
        assert f16(M, N, K, -1) >= (M + N) * (K + 1) * 2, (M, N, K)
    for M, N, K in ((1856, 729, 2111), (2107, 991, 1497), (2899, 593, 2019), (900, 1000, 6001)):
        assert i8(M, N, K, -1) >= (M + N) * (K + 1), (M, N, K)
