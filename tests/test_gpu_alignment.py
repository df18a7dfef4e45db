"""Hidden states (or gate-up weights) that start off a 16-byte boundary: the
layers that run in several passes take them at every token count of the GEMVs'
range, with the GEMVs' bits (the streaming kernel, which takes over from 33
tokens on, needs aligned operands), so no tolerance."""

import pytest
import torch

from oracle.bf16 import normal_bf16
from tests._util import to_dev_bf16, to_dev_i32
from tests.test_gpu_device_waves import _layer


def _offset(t, elems=1):
    """The same values, contiguous, `elems` elements past an aligned start."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    out = buf[elems: elems + t.numel()].view(t.shape)
    out.copy_(t)
    assert out.is_contiguous() and out.data_ptr() % 16 == 2 * elems
    return out


def _bits(t):
    return t.view(torch.int16)


def test_aligned_decides_the_path():
    from vllm_moe_offload_amd import native

    t = native.DECODE_GEMV_MAX_TOKENS + 1
    assert native.layer_path(t, 8, 1024, 256, aligned=False) == native.LMOE_PATH_GEMV
    assert native.layer_path(128, 8, 1024, 256, aligned=False) == native.LMOE_PATH_GEMV
    assert native.layer_path(129, 8, 1024, 256, aligned=False) == native.LMOE_PATH_MFMA
    x = torch.zeros(64, dtype=torch.bfloat16)
    base = x.data_ptr() // 2 % 8
    assert native.aligned16(x[(8 - base) % 8:]) and not native.aligned16(x[(8 - base) % 8:], x[(8 - base) % 8 + 1:])


@pytest.mark.gpu
@pytest.mark.parametrize("T,elems", [(33, 1), (64, 4), (128, 7)])
def test_waves_take_hidden_states_off_alignment(T, elems):
    from vllm_moe_offload_amd import fused_moe, native

    print(f"case waves off alignment T={T} elems={elems}", flush=True)
    layer, rt, rng = _layer({}, E=16, slots=4)
    dx = to_dev_bf16(normal_bf16(rng, (T, 1024), 1.0))
    w, ids, _ = fused_moe.route(dx, layer.gate_weight, layer.router_spec)
    kw = dict(layer_id=layer.layer_id, topk_weights=w, topk_ids=ids, num_logical_experts=16)
    ref = fused_moe.run_device_waves(rt, hidden=dx, path=native.LMOE_PATH_GEMV, **kw).clone()
    off = _offset(dx, elems)
    dev = fused_moe.run_device_waves(rt, hidden=off, **kw).clone()
    host = fused_moe.run_wave_prefill(rt, hidden=off, **kw)[0].clone()
    torch.cuda.synchronize()
    assert torch.equal(_bits(dev), _bits(ref)) and torch.equal(_bits(host), _bits(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("T,which", [(33, "hidden"), (64, "hidden"), (100, "hidden"), (64, "bank"), (64, "overflow")])
def test_overflow_layers_take_operands_off_alignment(T, which):
    from vllm_moe_offload_amd import fused_moe, native
    from vllm_moe_offload_amd.moe_offload.slot_mapping import PreparedSlotWeights

    print(f"case overflow off alignment T={T} {which}", flush=True)
    E, P, H, I, k = 24, 16, 1024, 256, 8
    g = torch.Generator(device="cuda").manual_seed(T)
    mk = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)
    dx, gate = mk(T, H), mk(E, H)
    bank, over = (mk(P, 2 * I, H), mk(P, H, I)), (mk(P, 2 * I, H), mk(P, H, I))
    table = to_dev_i32([e if e < P else -1 for e in range(E)])
    rest = to_dev_i32([e - P if e >= P else -1 for e in range(E)])
    x = _offset(dx) if which == "hidden" else dx
    b13 = _offset(bank[0]) if which == "bank" else bank[0]
    o13 = _offset(over[0]) if which == "overflow" else over[0]
    second = lambda w1: PreparedSlotWeights(w1=w1, w2=over[1], log2phy=rest, physical_expert_count=P, mapping=None)
    ws = fused_moe.get_workspace(T, k, P, H, I, "cuda", tag="alignment")
    out, w, ids = fused_moe.decode_layer(x, gate, fused_moe.RouterSpec(top_k=k), b13, bank[1], table, workspace=ws,
                                         overflow=second(o13))
    out = out.clone()
    again, _ = fused_moe._fused_experts_ws(x, w, ids, b13, bank[1], table, overflow=second(o13))
    again = again.clone()
    ref, _ = fused_moe._fused_experts_ws(dx, w, ids, *bank, table, overflow=second(over[0]),
                                         path=native.LMOE_PATH_GEMV)
    torch.cuda.synchronize()
    assert torch.equal(_bits(out), _bits(ref)) and torch.equal(_bits(again), _bits(ref))
