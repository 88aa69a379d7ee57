"""Which GEMMs ask for a workspace for copies of their operands: K no whole number of 16-byte vectors, and work enough. Runs on the CPU."""
import pytest

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
