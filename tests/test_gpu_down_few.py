"""The fused down + combine for a few pairs (one workgroup per CU): out and y
bit for bit those of the separate down GEMV and combine, which sum every
element in the same order, so no tolerance is needed; and the oracle's values
within 2e-2 x RMS (bf16 outputs)."""

import numpy as np
import pytest
import torch

from oracle import mlp as omlp
from oracle.bf16 import bf16_to_f32, f32_to_bf16
from tests._util import OUT_TOL, from_dev_bf16, normal_bf16, rel_max_err, to_dev_bf16, to_dev_i32


def _bits(t):
    return t.view(torch.int16)


@pytest.mark.gpu
@pytest.mark.parametrize("T,k,P,H,I,ids_of", [
    (2, 8, 16, 2048, 768, "spread"),     # 16 pairs: the last count without y
    (17, 1, 5, 2048, 768, "spread"),     # 17 pairs, fewer slots than waves
    (32, 8, 128, 2048, 768, "spread"),   # 256 pairs, the most it takes
    (43, 6, 40, 2048, 768, "spread"),    # 258 pairs: the separate kernels
    (64, 4, 3, 2048, 512, "hot"),        # every pair in one slot: 256 pairs of 64 steps
    (3, 2, 1, 1792, 320, "spread"),      # one slot; 224 blocks; a row's second chunk nearly empty
    (5, 7, 30, 2040, 960, "spread"),     # 255 blocks; a last chunk of 192 columns
    (9, 3, 9, 1784, 768, "spread"),      # 223 blocks: the separate kernels
    (4, 5, 64, 1024, 1024, "spread"),    # 4 columns per block, the widest I
    (11, 3, 8, 896, 768, "same"),        # 224 blocks of 4 columns; a token's pairs share a slot
    (6, 4, 12, 1000, 704, "unmapped"),   # 250 blocks of 4 columns; pairs with no slot
    (10, 4, 33, 2048, 1024, "unmapped"),
    (8, 4, 12, 1024, 256, "spread"),     # I too short: the separate kernels
])
def test_few_pairs_equal_separate_kernels(T, k, P, H, I, ids_of):
    from vllm_moe_offload_amd import native

    print(f"case down-few T={T} k={k} P={P} H={H} I={I} {ids_of}", flush=True)
    rng = np.random.default_rng(T * 1000 + k * 100 + H + I)
    E = P + (5 if ids_of == "unmapped" else 0)
    if ids_of == "hot":
        ids = np.full((T, k), P - 1, dtype=np.int32)
    elif ids_of == "same":
        ids = np.repeat(rng.integers(0, E, (T, 1)), k, axis=1).astype(np.int32)
    else:
        ids = rng.integers(0, E, (T, k)).astype(np.int32)
    l2p = np.full(E, -1, dtype=np.int32)
    l2p[:P] = rng.permutation(P)
    w13, w2 = normal_bf16(rng, (P, 2 * I, H), 0.02), normal_bf16(rng, (P, H, I), 0.02)
    wb = f32_to_bf16(rng.random((T, k)).astype(np.float32))
    x, add = normal_bf16(rng, (T, H), 1.0), normal_bf16(rng, (T, H), 1.0)
    d_x, d_w, d_add, d_w13, d_w2 = (to_dev_bf16(v) for v in (x, wb, add, w13, w2))

    def buffers():
        p = native.Permutation.allocate(T * k, P, "cuda")
        native.permute(to_dev_i32(ids), p, log2phy=to_dev_i32(l2p), skip_unmapped=True)
        return (p, torch.zeros((T * k, I), dtype=torch.bfloat16, device="cuda"),
                torch.full((T * k, H), -7.0, dtype=torch.bfloat16, device="cuda"),
                torch.empty((T, H), dtype=torch.bfloat16, device="cuda"))

    native.device_flags()  # earlier tests' flags
    p, act, y_ref, ref = buffers()
    native.gateup_silu(d_x, k, d_w13, p, act, path=native.LMOE_PATH_GEMV)
    native.down(act, d_w2, p, y_ref, path=native.LMOE_PATH_GEMV)
    native.combine(y_ref, d_w, ref, row_mask=p.row_idx, add=d_add)
    flags = native.device_flags()
    for with_y in (True, False):
        p, act, y, out = buffers()
        native.fused_moe_decode(d_x, d_w, d_w13, d_w2, p, act, out, add=d_add, y=y if with_y else None)
        assert native.device_flags() == flags, f"with_y={with_y}"
        assert torch.equal(_bits(out), _bits(ref)), f"with_y={with_y}"
        if with_y and T * k > 16:
            assert torch.equal(_bits(y), _bits(y_ref))
    if ids_of != "unmapped":
        want = bf16_to_f32(add) + omlp.moe_layer(x, ids, wb, l2p, w13, w2)
        assert rel_max_err(bf16_to_f32(from_dev_bf16(out)), want) <= OUT_TOL
