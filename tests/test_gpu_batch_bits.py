"""What a token's result depends on besides its own row and routing: the path
that its layer takes (native.layer_path), which a batch's size decides, and
nothing else of the batch.  Within a path the bits are the same whatever runs
beside the token; between the GEMVs and the streaming kernel, which add the
same products in another order, both are within the tolerance of bf16 outputs
(2e-2 x RMS of the result for any element) of each other.  The entries that
are the GEMVs by name (lmoe_fused_moe_decode, ..._noalloc) keep their bits at
every token count."""

import pytest
import torch

from tests._util import OUT_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,E,k", [
    (512, 256, 16, 4),     # the line at 32 tokens
    (2048, 768, 128, 8),   # the line at 2.75 pairs per expert: 44 tokens
])
def test_a_tokens_bits_depend_on_the_path_alone(H, I, E, k):
    from vllm_moe_offload_amd import fused_moe, native

    print(f"case batch bits H={H} I={I} E={E} k={k}", flush=True)
    T = native.FUSED_DECODE_MAX_PAIRS // k
    g = torch.Generator(device="cuda").manual_seed(H)
    mk = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)
    w13, w2 = mk(E, 2 * I, H), mk(E, H, I)
    x = torch.empty((T, H), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    score, ids = torch.rand((T, E), device="cuda", generator=g).topk(k, dim=1)
    ids, w = ids.to(torch.int32).contiguous(), torch.softmax(score, 1).to(torch.bfloat16)
    path = lambda t: native.layer_path(t, k, H, I, E)
    gemv = [t for t in range(1, T + 1) if path(t) == native.LMOE_PATH_GEMV]
    line = max(gemv)
    assert gemv == list(range(1, line + 1)) and all(path(t) == native.LMOE_PATH_STREAM for t in range(line + 1, T + 1))

    def run(t, **kw):
        return fused_moe.fused_experts(x[:t], w[:t].contiguous(), ids[:t].contiguous(), w13, w2, None, **kw).clone()

    many, few = run(T), run(line)
    bits = lambda t: t.view(torch.int16)
    for t in (line + 1, T - 1):
        assert torch.equal(bits(run(t)), bits(many[:t])), t
    for t in (1, 2, line - 1):
        assert torch.equal(bits(run(t)), bits(few[:t])), t
    ref = few.double()
    assert ((many[:line].double() - ref).abs().max() / ref.pow(2).mean().sqrt()).item() <= OUT_TOL
    # the GEMV entries past the line
    named = run(T, path=native.LMOE_PATH_GEMV)
    assert torch.equal(bits(named[:line]), bits(few))
    perm = native.Permutation.allocate(T * k, E, "cuda")
    native.permute(ids, perm)
    out = torch.empty_like(x)
    native.fused_moe_decode_noalloc(x, w, w13, w2, perm, out)
    assert torch.equal(bits(out), bits(named))
