"""INT4 shapes outside the 128-multiples: group sizes 32 and 64, a group of
192, contraction lengths below 128 (one group = K, the reference's collapse at
moe_int4_kernel.py:61-64), and weight-row counts that are not multiples of 32
(the reference masks the N tail, moe_int4_kernel.py:206-207, 238-240).  Each
runs the rows kernels and is checked against the fp32
dequantise-then-matmul oracle; routing arrays bit-exact."""
import numpy as np
import pytest
import torch

from exq_amd import synth
from oracle import moe, quant, routing
from tests._helpers import assert_close_rel, banner, oracle_int4_layer

pytestmark = pytest.mark.gpu

TOL = 5e-3


def _bank(E, N, K, g, seed, device):
    from exq_amd.kernels import pack_experts_int4
    gen = torch.Generator(device="cpu").manual_seed(seed)
    w = (torch.randn(E, N, K, generator=gen) * 0.02).to(torch.float16).to(device)
    return pack_experts_int4(w, g)


@pytest.mark.parametrize("K,N,g", [(256, 96, 32), (256, 100, 64), (96, 40, 128), (384, 72, 192),
                                   (64, 17, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_moe_int4_forward_general_shapes(K, N, g, dtype, device):
    from exq_amd.kernels import moe_int4_forward
    banner(f"moe_int4_forward K={K} N={N} g={g} {dtype}")
    E, T, k = 6, 37, 2
    p, s = _bank(E, N, K, g, K + N, device)
    g_eff = min(g, K)
    assert s.shape == (E, N, K // g_eff)
    rng = np.random.default_rng(K * 7 + N)
    ids = np.stack([rng.choice(E, size=k, replace=False) for _ in range(T)]).astype(np.int64)
    x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float32)).to(dtype).to(device)
    out = moe_int4_forward(x, p, s, torch.from_numpy(ids).to(device), E)
    assert out.shape == (T * k, N) and out.dtype == dtype
    r_so, r_ends, _ = routing.sort_tokens_by_expert(ids, E)
    a = moe.gather_hidden(x.float().cpu().numpy(), r_so, k)
    ref = moe.grouped_gemm_sorted(a, quant.dequant_int4(p.cpu().numpy(), s.cpu().numpy()), r_ends)
    assert_close_rel(out, ref, TOL, f"moe_int4_forward K={K} N={N} g={g_eff} {dtype}")


@pytest.mark.parametrize("H,I,g", [(256, 192, 64), (96, 64, 32), (384, 192, 192), (160, 96, 32)])
@pytest.mark.parametrize("T", [1, 5, 80])
def test_fused_general_shapes(H, I, g, T, device):
    from exq_amd.kernels import fused_experts
    banner(f"fused H={H} I={I} g={g} T={T}")
    E, k = 8, 2
    p13, s13 = _bank(E, 2 * I, H, g, H + I, device)
    p2, s2 = _bank(E, H, I, g, H + I + 1, device)
    cfg = synth.MoeConfig("gen", 41, H, I, E, k, True)
    ids, w = synth.routing(cfg, T, 0)
    tid = torch.from_numpy(ids).to(device)
    tw = torch.from_numpy(w).to(device)
    x = torch.from_numpy(synth.hidden_np(T, H, 3)).to(torch.bfloat16).to(device)
    so = torch.empty(T * k, dtype=torch.int64, device=device)
    ends = torch.empty(E + 1, dtype=torch.int32, device=device)
    out = fused_experts(x, p13, s13, p2, s2, tw, tid, sort_order_out=so, expert_ends_out=ends)
    r_so, r_ends, _ = routing.sort_tokens_by_expert(ids, E)
    assert np.array_equal(so.cpu().numpy(), r_so)
    assert np.array_equal(ends.cpu().numpy(), r_ends)
    ref = oracle_int4_layer(x, p13, s13, p2, s2, ids, w)
    assert_close_rel(out, ref, TOL, f"fused general H={H} I={I} g={g} T={T}")
    # repeatable bit for bit, and fp16 activations
    assert torch.equal(fused_experts(x, p13, s13, p2, s2, tw, tid), out)
    out16 = fused_experts(x.to(torch.float16), p13, s13, p2, s2, tw, tid)
    assert out16.dtype == torch.float16
    assert_close_rel(out16, ref, TOL, f"fused general fp16 H={H} I={I} g={g} T={T}")


@pytest.mark.parametrize("H,I,g", [
    (2304, 224, 32),    # 72 groups a row: five 16-group scale windows; I not a multiple of 64
    (1120, 96, 32),     # K % 128 = 96: a short last chunk, windows that straddle chunks
    (1920, 480, 96),    # groups that straddle 128-k chunks
    (2176, 320, 64),    # 34 groups: a third window of two
    (512, 384, 128),    # standard shapes with few rows per expert take the same kernels
    (1024, 512, 256),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_kernel_edges(H, I, g, dtype, device):
    """Experts with 1, 31, 32, 33 and no rows and one with the rest (edges of the
    32-row token groups), above 64 tokens."""
    from exq_amd.kernels import fused_experts
    banner(f"rows kernel H={H} I={I} g={g} {dtype}")
    E, T, k = 9, 71, 2
    p13, s13 = _bank(E, 2 * I, H, g, H + 3 * I, device)
    p2, s2 = _bank(E, H, I, g, H + 3 * I + 1, device)
    counts = [1, 31, 32, 33, 0, 2, 16, 17]
    flat = np.concatenate([np.full(c, e) for e, c in enumerate(counts)])
    flat = np.concatenate([flat, np.full(T * k - flat.size, E - 1)])
    rng = np.random.default_rng(H + I)
    ids = rng.permutation(flat).reshape(T, k).astype(np.int64)
    w = rng.random((T, k)).astype(np.float32)
    x = torch.from_numpy(synth.hidden_np(T, H, 4)).to(dtype).to(device)
    out = fused_experts(x, p13, s13, p2, s2, torch.from_numpy(w).to(device),
                        torch.from_numpy(ids).to(device))
    ref = oracle_int4_layer(x, p13, s13, p2, s2, ids, w)
    assert_close_rel(out, ref, TOL, f"rows kernel H={H} I={I} g={g} {dtype}")


@pytest.mark.parametrize("K,N,g", [
    (32, 1, 32),        # one weight row of one scale group
    (160, 129, 32),     # K % 128 = 32: the last tile is one row whose last chunk is short
    (224, 257, 32),     # K % 128 = 96
    (640, 130, 32),     # 20 groups a row: two 16-group scale windows of two rows
    (544, 1, 32),       # 17 groups: the second window is one group
    (96, 129, 96),
    (1024, 129, 64),    # whole chunks, one row in the last tile
    (512, 1, 256),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_kernel_last_weight_row(K, N, g, dtype, device):
    """Tiles of one or two weight rows at the end of the packed weights and scales:
    chunks and scale windows past a row's end are past the resource too."""
    from exq_amd.kernels import moe_int4_forward
    banner(f"rows kernel K={K} N={N} g={g} {dtype}")
    E, T = 3, 41
    p, s = _bank(E, N, K, g, K + N, device)
    rng = np.random.default_rng(K + N)
    ids = rng.integers(0, E, (T, 1))
    x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float32)).to(dtype).to(device)
    out = moe_int4_forward(x, p, s, torch.from_numpy(ids).to(device), E)
    order = np.argsort(ids[:, 0], kind="stable")
    ends = np.searchsorted(ids[order, 0], np.arange(E + 1))
    ref = moe.grouped_gemm_sorted(x.float().cpu().numpy()[order],
                                  quant.dequant_int4(p.cpu().numpy(), s.cpu().numpy()), ends)
    assert_close_rel(out, ref, TOL, f"rows kernel K={K} N={N} g={g} {dtype}")


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8, 9, 12, 16, 17])
@pytest.mark.parametrize("H", [32, 96, 1056])
def test_combine_slot_batches(k, H, device):
    """Combine launch of the prefill and rows paths: slots in batches of 2, 4 or 8
    with a short last one, columns past a block's end, dropped ids (no weight),
    one token with none left."""
    from exq_amd.kernels import fused_experts
    banner(f"combine k={k} H={H}")
    E, T, I, g = 20, 11, 64, 32
    p13, s13 = _bank(E, 2 * I, H, g, H + k, device)
    p2, s2 = _bank(E, H, I, g, H + k + 1, device)
    rng = np.random.default_rng(100 * k + H)
    ids = np.stack([rng.choice(E, size=k, replace=False) for _ in range(T)]).astype(np.int64)
    ids[rng.random((T, k)) < 0.2] = -1
    ids[3] = -1
    w = rng.random((T, k)).astype(np.float32)
    x = torch.from_numpy(synth.hidden_np(T, H, 5)).to(torch.bfloat16).to(device)
    out = fused_experts(x, p13, s13, p2, s2, torch.from_numpy(w).to(device),
                        torch.from_numpy(ids).to(device))
    # the oracle's dropped slots: any expert, weight 0
    ref = oracle_int4_layer(x, p13, s13, p2, s2, np.maximum(ids, 0),
                            np.where(ids < 0, 0, w).astype(np.float32))
    assert_close_rel(out, ref, TOL, f"combine k={k} H={H}")
    assert not out[3].any()


@pytest.mark.parametrize("ids_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("w_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [3, 8, 9])
def test_combine_dropped_slots(k, w_dtype, ids_dtype, device):
    """Rows of dropped ids are neither fetched nor weighted: -1, E, (64-bit) an id
    whose low word is in range, each with a NaN or infinite weight."""
    from exq_amd.kernels import fused_experts
    banner(f"combine dropped k={k} {w_dtype} {ids_dtype}")
    E, T, H, I, g = 16, 33, 160, 64, 32
    p13, s13 = _bank(E, 2 * I, H, g, 900 + k, device)
    p2, s2 = _bank(E, H, I, g, 901 + k, device)
    rng = np.random.default_rng(k)
    good = np.stack([rng.choice(E, size=k, replace=False) for _ in range(T)]).astype(np.int64)
    w = torch.from_numpy(rng.random((T, k)).astype(np.float32)).to(w_dtype)
    drop = rng.random((T, k)) < 0.6
    bad = [-1, E] + ([2**32 + 3, -2**32 + 3] if ids_dtype == torch.int64 else [])
    ids = np.where(drop, rng.choice(np.array(bad), (T, k)), good)
    ref_w = np.where(drop, 0, w.float().numpy()).astype(np.float32)
    w[torch.from_numpy(drop)] = float("nan")
    w[0][torch.from_numpy(drop[0])] = float("inf")
    x = torch.from_numpy(synth.hidden_np(T, H, 6)).to(torch.bfloat16).to(device)
    out = fused_experts(x, p13, s13, p2, s2, w.to(device),
                        torch.from_numpy(ids).to(ids_dtype).to(device))
    ref = oracle_int4_layer(x, p13, s13, p2, s2, good, ref_w)
    assert_close_rel(out, ref, TOL, f"combine dropped k={k} {w_dtype} {ids_dtype}")


def test_general_shape_rejections(device):
    from exq_amd import _lib
    from exq_amd.kernels import MixedExpertBank, fused_experts, fused_experts_mixed, \
        moe_int4_forward
    E, T, k = 4, 3, 2
    ids = torch.tensor([[0, 1], [2, 3], [1, 0]], device=device)
    # group size 16 is below the reference's minimum of 32 (moe_int4_kernel.py:286-290)
    p, s = _bank(E, 64, 64, 16, 1, device)
    x = torch.randn(T, 64, device=device).to(torch.bfloat16)
    with pytest.raises(ValueError, match="group_size"):
        moe_int4_forward(x, p, s, ids, E)
    p13, s13 = _bank(E, 128, 64, 16, 2, device)
    p2, s2 = _bank(E, 64, 64, 16, 3, device)
    with pytest.raises(ValueError, match="group_size"):
        fused_experts(x, p13, s13, p2, s2, torch.ones(T, k, device=device), ids)
    # mixed-precision banks keep the 128-multiple shapes
    w13 = torch.randn(E, 2 * 96, 96, device=device) * 0.02
    w2 = torch.randn(E, 96, 96, device=device) * 0.02
    bank = MixedExpertBank.from_weights(w13, w2, [2, 1, 0, 2], group_size=32)
    xb = torch.randn(T, 96, device=device).to(torch.bfloat16)
    with pytest.raises(_lib.ExqError, match="mixed-precision banks need"):
        fused_experts_mixed(xb, bank, torch.ones(T, k, device=device), ids)
