"""Boxes and chunks of the windowed conv kernel (csrc/conv_window.hip), host code: every LDS address that the kernel forms lies in its buffers,
the boxes cover the output, and the line between it and the tile kernel."""
import random

import pytest

from conv_window_plan import SHAPES, choose, layer, plan


def _check(dtype, shape, a):
    bm, bn = SHAPES[shape]
    assert a.box == a.TO * a.TH * a.TW <= bm and a.TH <= a.Ho and a.TW <= a.Wo
    outer = a.Do if a.three_d else a.N
    assert a.tiles_o * a.TO >= outer and a.tiles_h * a.TH >= a.Ho and a.tiles_w * a.TW >= a.Wo and a.tiles_n * bn >= a.K
    assert a.tiles == a.tiles_o * a.tiles_h * a.tiles_w * a.tiles_n * (a.N if a.three_d else 1)
    # the window holds the box's pixels shifted by every tap
    z = a.taps // (a.Y * a.X)
    reach = ((z - 1) * a.dD if a.three_d else 0, (a.Y - 1) * a.dH, (a.X - 1) * a.dW)
    assert a.pitch == a.TW + reach[2] and a.Wh == a.TH + reach[1] and a.win_px == (a.TO + reach[0]) * a.Wh * a.pitch
    planes = (a.units + 1) // 2
    assert a.spp * 32 >= a.win_px and a.spp <= 4 * 12          # four window waves of twelve slots
    assert a.cu % 2 == 0 and a.wbuf == a.cu // 2 * a.spp * 1024
    assert (a.chunks - 1) * a.cu < a.units <= a.chunks * a.cu and (a.chunks - 1) * (a.cu // 2) < planes
    # K tiles: a chunk outlasts the K tile that it shares with the next one
    assert a.total == a.taps * a.units < 65536 and a.nk == -(-a.total // 8) >= 4
    assert a.chunks == 1 or a.taps * a.cu >= 16
    assert 2 <= a.issue <= 4
    stage = max(bn, 32) * 128
    assert 3 * stage + 2 * a.wbuf + -(-a.nk * 32 // 256) * 256 + (256 if dtype == "i8" else 0) <= 160 * 1024


@pytest.mark.parametrize("dtype", ["i8", "f16"])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_random_layers(dtype, shape):
    rng, taken = random.Random(shape), 0
    for _ in range(400):
        nd = rng.choice([2, 3])
        filt = [rng.choice([1, 2, 3, 3, 5]) for _ in range(nd)]
        dil = [rng.choice([1, 1, 2]) for _ in range(nd)]
        pads = [rng.randint(0, 3) for _ in range(nd)]
        hw = [max(rng.randint(1, 60), (filt[i] - 1) * dil[i] + 1) for i in range(nd)]
        a, _ = layer(dtype, hw, rng.randint(1, 64), 16 * rng.randint(1, 64), rng.randint(1, 300), filt, dil, pads)
        if plan(dtype, shape, a) >= 0:
            taken += 1
            _check(dtype, shape, a)
    assert taken > 100


def test_the_line():
    def at(tile_us, *l):
        return choose("f16", layer("f16", *l)[0], tile_us)
    few_channels = ((32, 32, 32), 16, 64, 64, (3, 3, 3), (1, 1, 1), (1, 1, 1))
    assert at(138.0, *few_channels) == 0 and at(90.0, *few_channels) == -1
    assert at(290.0, (43, 43, 43), 4, 176, 32, (3, 3, 3), (1, 1, 1), (1, 1, 1)) == 2
    assert at(1e9, (32, 32), 16, 64, 64, (1, 7), (1, 1), (0, 3)) == -1       # too few taps
    assert at(1e9, (32, 32), 16, 128, 64, (2, 4), (1, 1), (0, 1)) == -1 and at(1e9, (32, 32), 16, 128, 64, (1, 9), (1, 1), (0, 4)) >= 0
    assert at(1e9, (16, 16, 16), 4, 128, 64, (2, 2, 2), (1, 1, 1), (1, 1, 1)) == -1
    # one chunk of fourteen K tiles: the next window has little time to come in
    assert at(35.5, (18, 18, 18), 25, 32, 16, (3, 3, 3), (1, 1, 1), (1, 1, 1)) == -1 and at(39.0, (18, 18, 18), 25, 32, 16, (3, 3, 3), (1, 1, 1), (1, 1, 1)) == 2
    assert choose("i8", layer("i8", (35, 35, 35), 23, 64, 16, (3, 3, 3), (1, 1, 1), (1, 1, 1))[0], 162.3) == 2
    assert at(13.9, (8, 8), 1, 32, 32, (3, 3), (1, 1), (1, 1)) == -1          # small calls are not searched


def test_plan_query_of_a_windowed_layer():
    """No instance index makes that launch: the query answers with the automatic choice. By index, with a K split and for layers past the
    lines it answers with the tile instance."""
    from composable_kernel_amd import capi

    def query(N, C, K, hw, stride=1, op=capi.OP_CONV2D_FWD_F16, **kw):
        ho = (hw - 1) // stride + 1
        return capi.conv2d_fwd_plan(op, capi.Conv2dDesc(N, K, C, hw, hw, 3, 3, ho, ho, stride, stride, 1, 1, 1, 1, 1, 1), **kw)
    assert query(48, 88, 24, 57) == (capi.INSTANCE_AUTO, 1) and query(48, 88, 24, 57, instance=7) == (7, 1)
    assert query(32, 176, 24, 57, op=capi.OP_CONV2D_FWD_I8, instance=7) == (7, 1) and query(32, 176, 24, 57, op=capi.OP_CONV2D_FWD_I8) == (capi.INSTANCE_AUTO, 1)
    assert query(48, 88, 24, 57, stride=2)[0] >= 0 and query(1, 88, 24, 57)[0] >= 0
    capi.lib().ckx_set_forced_k_runs(2)
    try:
        inst, runs = query(48, 88, 24, 57, workspace_bytes=1 << 30)
        assert inst >= 0 and runs == 2
    finally:
        capi.lib().ckx_set_forced_k_runs(0)
