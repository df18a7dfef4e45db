"""Prefill past the bank with few experts per wave: 33 tokens and more of up to
1024 pairs take the streaming path with its one row-tile height, however many
pairs a wave's slots hold.  Host- and device-planned waves give the full
layer's bits (every path computes a pair's row alone), so no tolerance."""

import pytest
import torch

from oracle.bf16 import normal_bf16
from tests._util import to_dev_bf16
from tests.test_gpu_device_waves import _layer

pytestmark = pytest.mark.gpu


# pairs per slot past STREAM_MAX_PAIRS_PER_SLOT: of the whole layer over a
# host-planned wave's experts, and of one device-planned wave over the bank;
# the GEMV, streaming and MFMA paths' first and last token counts
@pytest.mark.parametrize("E,slots,T", [(64, 8, 100), (8, 2, 101), (8, 2, 32), (8, 2, 33), (8, 2, 128), (8, 2, 129)])
def test_waves_of_few_experts_equal_the_full_layer(E, slots, T):
    from vllm_moe_offload_amd import fused_moe

    H = 1024
    print(f"case waves E={E} slots={slots} T={T}", flush=True)
    layer, rt, rng = _layer({}, E=E, slots=slots)
    dx = to_dev_bf16(normal_bf16(rng, (T, H), 1.0))
    w, ids, _ = fused_moe.route(dx, layer.gate_weight, layer.router_spec)
    kw = dict(layer_id=layer.layer_id, hidden=dx, topk_weights=w, topk_ids=ids, num_logical_experts=E)
    full = fused_moe.run_full_layer(rt, **kw).clone()
    dev = fused_moe.run_device_waves(rt, **kw).clone()
    host, report = fused_moe.run_wave_prefill(rt, **kw)
    host = host.clone()
    torch.cuda.synchronize()
    assert len(report.waves) == E // slots
    assert torch.equal(dev.view(torch.int16), full.view(torch.int16))
    assert torch.equal(host.view(torch.int16), full.view(torch.int16))


# the first and last token counts of either path at the line of 2.1 pairs per
# expert of the layer (256 of them; a wave holds 64)
@pytest.mark.parametrize("T", [67, 68])
def test_waves_take_the_path_of_the_whole_layers_experts(T):
    from vllm_moe_offload_amd import fused_moe, native

    print(f"case waves at the line per expert T={T}", flush=True)
    layer, rt, rng = _layer({}, E=256, slots=64)
    dx = to_dev_bf16(normal_bf16(rng, (T, 1024), 1.0))
    w, ids, _ = fused_moe.route(dx, layer.gate_weight, layer.router_spec)
    kw = dict(layer_id=layer.layer_id, hidden=dx, topk_weights=w, topk_ids=ids, num_logical_experts=256)
    path = native.layer_path(T, 8, 1024, 256, 256)
    assert path == (native.LMOE_PATH_GEMV if T == 67 else native.LMOE_PATH_STREAM)
    want = fused_moe.run_full_layer(rt, path=path, **kw).clone()
    for out in (fused_moe.run_full_layer(rt, **kw), fused_moe.run_device_waves(rt, **kw),
                fused_moe.run_wave_prefill(rt, **kw)[0]):
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))


def test_waves_take_the_row_tiles_of_their_own_pairs(monkeypatch):
    """384 pairs of 3072 in a wave of 8 slots: 48 per slot, the 96-row tiles,
    by host- and device-planned waves alike; the bits are those of the 320-row
    tiles, which 384 per slot would take."""
    from vllm_moe_offload_amd import fused_moe, native

    T = 384
    print(f"case row tiles of waves T={T}", flush=True)
    layer, rt, rng = _layer({}, E=64, slots=8)
    dx = to_dev_bf16(normal_bf16(rng, (T, 1024), 1.0))
    w, ids, _ = fused_moe.route(dx, layer.gate_weight, layer.router_spec)
    kw = dict(layer_id=layer.layer_id, hidden=dx, topk_weights=w, topk_ids=ids, num_logical_experts=64)
    seen, permute, mlp = [], native.permute, native.grouped_mlp

    def outs():
        return [f.clone() for f in (fused_moe.run_device_waves(rt, **kw), fused_moe.run_wave_prefill(rt, **kw)[0])]

    monkeypatch.setattr(native, "permute", lambda *a, **k: (seen.append(k["block_m"]), permute(*a, **k))[1])
    got = outs()
    assert seen == [native.STREAM_BLOCK_M] * 16
    monkeypatch.setattr(native, "STREAM_MAX_PAIRS_PER_SLOT", 0)
    want = outs()
    assert set(seen[16:]) == {native.PART_BLOCK_M}
    monkeypatch.undo()
    # the kernel's form is chosen by the pass's pairs: none, and all of them
    for pairs in (0, T * 8):
        monkeypatch.setattr(native, "grouped_mlp", lambda *a, **k: mlp(*a, **{**k, "pass_pairs": pairs}))
        got += outs()
    for out in got:
        assert torch.equal(out.view(torch.int16), want[0].view(torch.int16))
    assert torch.equal(want[0], want[1])
