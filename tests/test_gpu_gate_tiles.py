"""The dense gate's tile rule: 64 x 64 tiles while they are at most one per CU
of 256, 64 x 128 tiles past that.  Every logit sums the same MFMA steps in the
same order, so a token's f32 logits are the same bits whichever tiles its
batch takes; tokens and experts at the tiles' edges included."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("H,E", [(64, 128), (192, 72), (320, 136), (2048, 8)])  # 1, 3, 5, 32 K steps of a 6-stage ring
def test_gate_bits_do_not_depend_on_the_tiles(H, E):
    from vllm_moe_offload_amd import native

    print(f"case gate tiles H={H} E={E}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(H + E)
    mk = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    T = 64 * 256 // ((E + 63) // 64) + 65  # past one 64 x 64 tile per CU
    x, wg = mk(T, H), mk(E, H)
    wide = torch.empty((T, E), dtype=torch.float32, device="cuda")
    native.router_gate(x, wg, wide)
    for t in (65, 127, 128, 129, 1000):
        narrow = torch.full((t + 1, E), -7.0, dtype=torch.float32, device="cuda")
        native.router_gate(x[:t].contiguous(), wg, narrow[:t])
        assert torch.equal(narrow[:t].view(torch.int32), wide[:t].view(torch.int32)), t
        assert (narrow[t] == -7.0).all()
    exact = x.double() @ wg.double().t()
    bound = 4.0 * H ** 0.5 * 2.0 ** -24 * (x.double().abs() @ wg.double().abs().t())
    assert ((wide.double() - exact).abs() <= bound + 1e-30).all()
