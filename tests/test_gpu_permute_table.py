"""The block permutations with a count table against the oracle, bit for bit, at
their edges: one pair past a wave's, a full block, one pair past it, partly
filled waves and chunks, slot counts at each lane width and one past the
largest (the form without a table), hot slots past 16 bits, unmapped and
invalid ids, and the keep-rows mode over several chunks."""

import numpy as np
import pytest
import torch

from oracle import permute as orc
from tests._util import to_dev_i32
from tests.test_gpu_permute import _check, _native


@pytest.mark.gpu
@pytest.mark.parametrize("N,P,ids_of", [
    (257, 64, "even"), (257, 1024, "even"), (321, 65, "bad"), (1024, 1, "even"), (1024, 128, "hot"),
    (1023, 256, "bad"), (600, 513, "even"), (1000, 1024, "hot"), (700, 1025, "hot"),
    (1025, 64, "even"), (2047, 129, "hot"), (4097, 300, "bad"), (3000, 1024, "even"), (2050, 1025, "bad"),
    (70000, 100, "one"),   # one slot of more than 65535 pairs
    (132000, 33, "hot"),   # 129 chunks: more than one per thread of a slot
])
def test_block_permutations_match_oracle(N, P, ids_of):
    native = _native()
    print(f"case permute table N={N} P={P} {ids_of}", flush=True)
    rng = np.random.default_rng(N * 7 + P)
    E = P + 9
    ids = rng.integers(0, E, N)
    if ids_of == "hot":  # a few heavy slots, ties among them
        ids = np.where(rng.random(N) < 0.6, rng.integers(0, min(E, 5), N), ids)
        ids[: N // 4] = np.arange(N // 4) % 4
    elif ids_of == "one":
        ids[: N - 50] = 3
    elif ids_of == "bad":
        ids[rng.integers(0, N, 20)] = -7
        ids[rng.integers(0, N, 20)] = E + 1
    ids = ids.astype(np.int32).reshape(N, 1)
    l2p = np.full(E, -1, dtype=np.int32)
    l2p[rng.permutation(E)[:P]] = rng.permutation(P)
    for skip in (False, True):
        perm = native.Permutation.allocate(N, P, "cuda")
        native.permute(to_dev_i32(ids), perm, log2phy=to_dev_i32(l2p), skip_unmapped=skip, block_m=96)
        _check(perm, orc.init_routing(ids, P, log2phy=l2p, block_m=96, skip_unmapped=skip), N)
    # a later pass's build: rows it does not place keep their row_idx
    other = torch.full((N,), 12345, dtype=torch.int32, device="cuda")
    perm = native.Permutation.allocate(N, P, "cuda")
    native.permute(to_dev_i32(ids), perm, log2phy=to_dev_i32(l2p), keep_rows=True, row_idx=other, block_m=96)
    ref = orc.init_routing(ids, P, log2phy=l2p, block_m=96, skip_unmapped=True).row_idx
    np.testing.assert_array_equal(other.cpu().numpy(), np.where(ref >= 0, ref, 12345))
