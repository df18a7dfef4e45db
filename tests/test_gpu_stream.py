"""The weight-streaming MFMA kernel (row tiles of 96 rows): bit for bit the
128-row tiles' act and y over the edges of its tiles, token groups, columns
and slot table; with partial sums (path STREAM) the oracle's values, each
token's bits whatever runs beside it, and the GEMVs' accuracy; the shared
launch of two passes; the rule that picks a layer's path.

Tolerance against the oracle: 2e-2 x RMS of y at most for any element (the
tier's bar for bf16 outputs); against the other MFMA kernels none, since every
element sums the same MFMA steps in the same order."""

import numpy as np
import pytest
import torch

from oracle import mlp as omlp
from oracle.bf16 import bf16_to_f32
from tests._util import OUT_TOL, from_dev_bf16, rel_max_err, to_dev_bf16, to_dev_i32


def _native():
    from vllm_moe_offload_amd import native

    return native


def _counts_ids(counts, T, rng):
    """[T, 1] ids giving slot s counts[s] tokens, in random order; -1 for the rest."""
    ids = np.full(T, -1, dtype=np.int32)
    ids[: sum(counts)] = np.repeat(np.arange(len(counts)), counts)
    return rng.permutation(ids).reshape(T, 1)


def _bank(P, H, I, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)
    return mk(P, 2 * I, H), mk(P, H, I)


def _run(native, d_x, k, w13, w2, d_ids, l2p, bm, n_slots, skip=False, path=None):
    n = d_ids.numel()
    perm = native.Permutation.allocate(n, n_slots, "cuda")
    native.permute(d_ids, perm, log2phy=l2p, skip_unmapped=skip, block_m=bm)
    act = torch.zeros((n, w13.shape[1] // 2), dtype=torch.bfloat16, device="cuda")
    y = torch.full((n, w13.shape[2]), -7.0, dtype=torch.bfloat16, device="cuda")
    native.grouped_mlp(d_x, k, w13, w2, perm, act, y, path=native.LMOE_PATH_MFMA if path is None else path)
    placed = int(perm.meta[native.META_PAIRS].item())
    return act[:placed].clone(), y


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,counts", [
    # token groups of 16: their edges, an empty slot, tiles of exactly 96 rows and of one more
    (512, 128, [1, 15, 16, 17, 0, 31, 32, 33, 48, 49, 63, 64, 65, 80, 95, 96, 97, 192, 193]),
    (64, 64, [3, 70, 100]),       # one K step in gate-up and in down, one block of columns
    (192, 192, [5, 20, 40]),      # three K steps, H and I no multiple of a block's columns
    (2048, 768, [7, 18, 36]),     # the Qwen3 expert shape
    (320, 1408, [2, 90, 9]),      # 22 K steps in down
    (7168, 256, [4, 33]),         # the DeepSeek-V3 row length
    (64, 64, [2] * 600 + [98, 0, 1]),  # past 256 and 512 slots, the wide form of the kernel in neither GEMM
    (64, 1088, [16, 17, 33, 48, 64, 65, 96, 97, 0, 150] * 6),  # 58 rows per slot, 540 blocks of 128 columns
    (1024, 1024, [97, 300, 5, 193, 96]),  # slots of several row tiles, column blocks a multiple of 8
    (192, 320, [1, 17, 66] * 101),     # 303 slots of 5 column blocks: the wide form
    (2112, 448, [5, 40, 97]),          # 33 K steps: the first past two phases in gate-up
])
def test_stream_tiles_equal_128_row_tiles_and_oracle(H, I, counts):
    native = _native()
    P, T = len(counts), sum(counts) + 3
    print(f"case stream H={H} I={I} P={P} T={T}", flush=True)
    rng = np.random.default_rng(H + I + P)
    ids = _counts_ids(counts, T, rng)
    l2p = rng.permutation(P).astype(np.int32)
    g = torch.Generator(device="cuda").manual_seed(T)
    d_x = torch.empty((T, H), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    w13, w2 = _bank(P, H, I, P + H)
    d_ids, d_l2p = to_dev_i32(ids), to_dev_i32(l2p)
    a64, y64 = _run(native, d_x, 1, w13, w2, d_ids, d_l2p, native.STREAM_BLOCK_M, P, skip=True)
    a128, y128 = _run(native, d_x, 1, w13, w2, d_ids, d_l2p, 128, P, skip=True)
    assert torch.equal(a64.view(torch.int16), a128.view(torch.int16))
    assert torch.equal(y64.view(torch.int16), y128.view(torch.int16))
    # partial sums: some tokens alone (other token groups, the narrow form)
    # have the bits they have among all, and match the oracle
    _, ys = _run(native, d_x, 1, w13, w2, d_ids, d_l2p, native.STREAM_BLOCK_M, P, skip=True,
                 path=native.LMOE_PATH_STREAM)
    assert torch.equal((ys == -7.0).all(dim=1).cpu(), torch.from_numpy(ids[:, 0] < 0))
    rows = rng.choice(T, size=min(T, 40), replace=False)
    rows = rows[ids[rows, 0] >= 0]
    sub = torch.from_numpy(rows).cuda()
    _, yr = _run(native, d_x[sub].contiguous(), 1, w13, w2, d_ids[sub].contiguous(), d_l2p, native.STREAM_BLOCK_M, P,
                 path=native.LMOE_PATH_STREAM)
    assert torch.equal(ys[sub].view(torch.int16), yr.view(torch.int16))
    used = np.unique(l2p[ids[rows, 0]])
    ref = omlp.grouped_mlp(from_dev_bf16(d_x)[rows],
                           np.searchsorted(used, l2p[ids[rows, 0]]).astype(np.int32).reshape(-1, 1), 1,
                           from_dev_bf16(w13[used.tolist()]), from_dev_bf16(w2[used.tolist()]))
    for y in (y64, ys):
        assert rel_max_err(bf16_to_f32(from_dev_bf16(y))[rows], ref) <= OUT_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("H,I", [(2048, 768), (7168, 512)])
def test_partial_sums_round_act_as_the_gemvs_do(H, I):
    """The share of act values that differ from what f64 sums give (at the
    same bf16 boundaries) marks the error of the f32 accumulation.  Path
    STREAM has no more of them than the GEMVs, up to the count's own spread:
    three standard deviations of a count of that mean."""
    native = _native()
    P, T = 8, 640
    rng = np.random.default_rng(H)
    ids = rng.integers(0, P, size=(T, 1)).astype(np.int32)
    g = torch.Generator(device="cuda").manual_seed(H)
    d_x = torch.empty((T, H), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    w13, w2 = _bank(P, H, I, H)
    order = np.argsort(ids[:, 0], kind="stable")
    gu = torch.stack([d_x[t].double() @ w13[int(ids[t, 0])].double().t() for t in order]).to(torch.bfloat16).double()
    ref = (gu[:, :I] * torch.sigmoid(gu[:, :I]) * gu[:, I:]).to(torch.bfloat16)
    flips = {}
    for name, path in (("gemv", native.LMOE_PATH_GEMV), ("stream", native.LMOE_PATH_STREAM)):
        act, _ = _run(native, d_x, 1, w13, w2, to_dev_i32(ids), None, native.STREAM_BLOCK_M, P, path=path)
        flips[name] = int((act != ref).sum().item())
    print(f"act off the f64 sums' value: {flips}", flush=True)
    assert flips["stream"] <= flips["gemv"] + 3 * (2 * flips["gemv"]) ** 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("T,k,E,Pa,Pb,H,I", [
    (64, 8, 128, 64, 64, 2048, 768),   # the batch of 64 past its 64-slot bank
    (150, 4, 40, 20, 16, 320, 192),    # guarded columns; some pairs in neither table
    (400, 1, 4, 2, 2, 512, 64),        # slots of more than one tile in both passes
])
def test_stream_two_passes_equal_passes_one_by_one(T, k, E, Pa, Pb, H, I):
    native = _native()
    print(f"case stream two passes T={T} k={k} H={H} I={I}", flush=True)
    rng = np.random.default_rng(T + H)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    used = rng.permutation(np.unique(ids))
    la, lb = np.full(E, -1, dtype=np.int32), np.full(E, -1, dtype=np.int32)
    na = min(Pa, used.size * 3 // 5)
    nb = min(Pb, used.size - na)
    la[used[:na]] = rng.permutation(Pa)[:na]
    lb[used[na:na + nb]] = rng.permutation(Pb)[:nb]
    g = torch.Generator(device="cuda").manual_seed(T)
    d_x = torch.empty((T, H), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    (a13, a2), (b13, b2) = _bank(Pa, H, I, 1), _bank(Pb, H, I, 2)
    d_ids = to_dev_i32(ids)
    pa, pb = (native.Permutation.allocate(T * k, p, "cuda") for p in (Pa, Pb))
    native.permute_two_tables(d_ids, pa, to_dev_i32(la), pb, to_dev_i32(lb), block_m=native.STREAM_BLOCK_M)
    act = torch.empty((T * k, I), dtype=torch.bfloat16, device="cuda")
    y1 = torch.full((T * k, H), -7.0, dtype=torch.bfloat16, device="cuda")
    placed = (la[ids.reshape(-1)] >= 0) | (lb[ids.reshape(-1)] >= 0)
    for path in (native.LMOE_PATH_STREAM, native.LMOE_PATH_MFMA):
        y1.fill_(-7.0)
        y2 = y1.clone()
        native.grouped_mlp(d_x, k, a13, a2, pa, act, y1, path=path)
        native.grouped_mlp(d_x, k, b13, b2, pb, act, y1, path=path)
        for _ in range(2):
            native.stream_mlp_two_passes(d_x, k, a13, a2, pa, b13, b2, pb, act, y2, path=path)
        assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
        assert (y2[torch.from_numpy(~placed).cuda()] == -7.0).all()


def test_layer_path_depends_on_the_layer_only():
    """Tokens, top-k and shape decide the path; H % 64 != 0 keeps the GEMVs
    over their whole range."""
    native = _native()
    n = native.DECODE_GEMV_MAX_TOKENS
    gemv, stream, mfma = native.LMOE_PATH_GEMV, native.LMOE_PATH_STREAM, native.LMOE_PATH_MFMA
    assert native.layer_path(1, 8, 2048, 768) == gemv and native.layer_path(n, 8, 2048, 768) == gemv
    assert native.layer_path(n + 1, 8, 2048, 768) == stream and native.layer_path(128, 8, 2048, 768) == stream
    assert native.layer_path(129, 8, 2048, 768) == mfma and native.layer_path(1, 8, 2048, 5632) == mfma
    assert native.layer_path(128, 8, 1000, 192) == gemv and native.layer_path(129, 8, 1000, 192) == mfma
    pick = lambda slots, pairs, h=2048: native.prefill_block_m(slots, h, 768, cu_count=256, n_pairs=pairs)
    most = 128 * native.STREAM_MAX_PAIRS_PER_SLOT
    assert pick(128, most) == native.STREAM_BLOCK_M and pick(128, most + 1) == native.PART_BLOCK_M
    assert pick(128, 512, h=1000) == native.MFMA_BLOCK_M


def test_few_pairs_per_expert_keep_the_gemvs():
    """Past the GEMVs' token count the line lies at a number of pairs per
    expert of the layer: where the streaming kernel is the faster one with
    every expert as likely.  Rows of other lengths have none."""
    native = _native()
    gemv, stream = native.LMOE_PATH_GEMV, native.LMOE_PATH_STREAM
    path = native.layer_path
    assert path(43, 8, 2048, 768, 128) == gemv and path(44, 8, 2048, 768, 128) == stream  # 344 and 352 pairs
    assert path(33, 4, 2048, 1408, 60) == stream  # 2.2 pairs per expert
    assert path(83, 4, 2048, 1408, 160) == gemv and path(84, 4, 2048, 1408, 160) == stream
    assert path(33, 9, 7168, 2048, 257) == stream and path(33, 8, 1536, 768, 128) == stream
    assert path(33, 1, 2048, 768, 1) == stream and path(32, 8, 2048, 768, 1) == gemv
    assert path(129, 8, 2048, 768, 1024) == native.LMOE_PATH_MFMA  # past 1024 pairs whatever the experts


def test_pass_pairs_choose_the_tiles_and_n_pairs_bound_the_offsets():
    native = _native()
    pick = lambda n, p=None, h=2048: native.prefill_block_m(64, h, 768, cu_count=256, n_pairs=n, pass_pairs=p)
    assert pick(9600) == native.PART_BLOCK_M and pick(9600, 4800) == native.STREAM_BLOCK_M
    assert pick(9600, 4801) == native.PART_BLOCK_M
    # a wave's kernels address rows of the whole layer's buffers
    assert pick(2**20 + 1, 4800) == native.MFMA_BLOCK_M
    import ctypes

    p = ctypes.c_void_p(4096)
    lib = native.load_library()
    args = (p, 64, 2048, 768, 8, p, p, 8, p, p, p, p, p, 512)
    assert lib.lmoe_grouped_mlp_pass(*args, -1, 96, native.LMOE_PATH_MFMA, p, p, None) == native.LMOE_ERR_ARG
    assert lib.lmoe_grouped_mlp_pass(*args[:13], 0, 0, 96, native.LMOE_PATH_MFMA, p, p, None) == 0


def test_stream_two_passes_refuse_shapes_on_the_host():
    native = _native()
    lib = native.load_library()
    import ctypes

    p = ctypes.c_void_p(4096)

    def call(H=2048, I=768, n=512, nb=8, x=p, path=native.LMOE_PATH_STREAM):
        return lib.lmoe_stream_mlp_two_passes(x, 64, H, I, 8, p, p, 8, p, p, p, p, p, p, nb, p, p, p, p, n, path, p, p, None)

    assert call(H=1000) == native.LMOE_ERR_SHAPE and call(I=100) == native.LMOE_ERR_SHAPE
    assert call(nb=0) == native.LMOE_ERR_ARG and call(x=None) == native.LMOE_ERR_ARG
    assert call(x=ctypes.c_void_p(4104)) == native.LMOE_ERR_SHAPE
    assert call(n=3_000_000) == native.LMOE_ERR_SHAPE  # 32-bit operand offsets
    assert call(path=native.LMOE_PATH_GEMV) == 1003  # LMOE_ERR_UNSUPPORTED
    assert call(n=0) == 0
