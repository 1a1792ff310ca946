"""Gather, combine, SiLU-and-mul and the weight quantisers on the GPU vs the oracle."""
import numpy as np
import pytest
import torch

from oracle import moe, quant
from tests._helpers import banner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_gather_hidden_exact(dtype, device):
    from exq_amd.kernels.exq_dispatch import gather_hidden
    banner(f"gather {dtype}")
    rng = np.random.default_rng(0)
    T, k, H = 16, 8, 2048
    hidden = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(dtype)
    order = rng.permutation(T * k)
    out = torch.empty(T * k, H, dtype=dtype, device=device)
    gather_hidden(hidden.to(device), torch.from_numpy(order).to(device), out, k)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    ref = moe.gather_hidden(hidden.view(bits).numpy(), order, k)
    assert np.array_equal(out.cpu().view(bits).numpy(), ref)


@pytest.mark.parametrize("dtype,wdtype", [(torch.bfloat16, torch.float32),
                                          (torch.float16, torch.float16),
                                          (torch.float32, torch.bfloat16)])
def test_combine(dtype, wdtype, device):
    from exq_amd.kernels.exq_dispatch import combine
    banner(f"combine {dtype} {wdtype}")
    rng = np.random.default_rng(1)
    T, k, H = 13, 6, 384
    down = torch.from_numpy(rng.standard_normal((T * k, H)).astype(np.float32)).to(dtype)
    w = torch.from_numpy(rng.random((T, k)).astype(np.float32)).to(wdtype)
    order = rng.permutation(T * k)
    res = torch.empty(T, H, dtype=dtype, device=device)
    combine(down.to(device), torch.from_numpy(order).to(device), w.to(device), res)
    ref = moe.combine(down.float().numpy(), order, w.float().numpy())
    # fp32 accumulation then one rounding to the output dtype
    tol = {torch.float32: 1e-6, torch.float16: 1e-3, torch.bfloat16: 8e-3}[dtype]
    assert np.allclose(res.float().cpu().numpy(), ref, rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_silu_and_mul(dtype, device):
    from exq_amd.kernels.exq_dispatch import silu_and_mul
    banner(f"silu_and_mul {dtype}")
    rng = np.random.default_rng(2)
    x = torch.from_numpy((rng.standard_normal((37, 2 * 768)) * 4).astype(np.float32)).to(dtype)
    out = torch.empty(37, 768, dtype=dtype, device=device)
    silu_and_mul(x.to(device), out)
    ref = moe.silu_and_mul(x.float().numpy().astype(np.float64))
    tol = {torch.float32: 1e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[dtype]
    assert np.allclose(out.float().cpu().numpy(), ref, rtol=tol, atol=tol * 1e-2)


def _near_ties(rows, K, top, dtype, seed, group=None):
    """Weights whose quotient by their row's (or group's) scale is a half-way
    point, or up to three ulp from one."""
    rng = np.random.default_rng(seed)
    g = group or K
    s = rng.uniform(0.5, 2.0, (rows, K // g, 1)).astype(np.float32) * 0.01
    q = rng.integers(-top, top, (rows, K // g, g)).astype(np.float32) + 0.5
    w = (q * s).astype(np.float32)
    w = (w.view(np.int32) + rng.integers(-3, 4, w.shape, dtype=np.int32)).view(np.float32)
    w[..., 0] = top * s[..., 0]  # the maximum
    w = w.reshape(rows, K)
    return torch.from_numpy(w).to(dtype)


@pytest.mark.parametrize("K", [8, 1024, 1032, 2048, 4096, 4104, 16384, 16392, 130])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_quantize_int8_near_ties(K, dtype, device):
    """Row lengths at the edges of the per-wave and per-work-group kernels; every
    integer and scale equal to IEEE division and half-even rounding."""
    from exq_amd.kernels import quantize_int8_rows
    banner(f"quantize_int8 K={K} {dtype}")
    w = _near_ties(5, K, 127, dtype, K)
    q, s = quantize_int8_rows(w.to(device))
    rq, rs = quant.quantize_int8(w.float().numpy())
    assert np.array_equal(q.cpu().numpy(), rq)
    assert np.array_equal(s.cpu().numpy().reshape(-1), np.asarray(rs).reshape(-1))


@pytest.mark.parametrize("rows,K,g", [(1, 8, 8), (3, 128, 128), (33, 384, 128), (7, 512, 512),
                                      (9, 1024, 32), (5, 192, 64), (4, 288, 96)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_pack_int4_near_ties(rows, K, g, dtype, device):
    """Group sizes of 1 to 64 lanes (96: the serial kernel) and ragged last
    work-groups; every nibble and scale equal to IEEE division and half-even
    rounding."""
    from exq_amd.kernels import pack_int4_weights
    banner(f"pack_int4 rows={rows} K={K} g={g} {dtype}")
    w = _near_ties(rows, K, 7, dtype, K + g, g)
    p, s = pack_int4_weights(w.to(device), g)
    rp, rs = quant.pack_int4_weights(w.float().numpy(), g)
    assert np.array_equal(p.cpu().numpy(), rp) and np.array_equal(s.cpu().numpy(), rs)


@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (5, 9, 40), (3, 8, 33), (2, 17, 2056)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_combine_column_and_slot_edges(T, k, H, dtype, device):
    """Vector and one-column forms of the combine, slot counts around its batch
    of eight."""
    from exq_amd.kernels.exq_dispatch import combine
    banner(f"combine T={T} k={k} H={H} {dtype}")
    rng = np.random.default_rng(T + k + H)
    down = torch.from_numpy(rng.standard_normal((T * k, H)).astype(np.float32)).to(dtype)
    w = torch.from_numpy(rng.random((T, k)).astype(np.float32))
    order = rng.permutation(T * k)
    res = torch.empty(T, H, dtype=dtype, device=device)
    combine(down.to(device), torch.from_numpy(order).to(device), w.to(device), res)
    ref = moe.combine(down.float().numpy(), order, w.numpy())
    # fp32 sums of k products (k ulp), then one rounding to the output dtype
    tol = {torch.float32: 4e-6, torch.bfloat16: 8e-3}[dtype]
    assert np.allclose(res.float().cpu().numpy(), ref, rtol=tol, atol=tol)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8, 12, 16])
@pytest.mark.parametrize("H", [264, 257])
@pytest.mark.parametrize("w_dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_combine_slot_batches(k, H, w_dtype, device):
    """Slots in batches of 2, 4 and 8 with a short last one, in both column forms; a
    NaN row reaches its own token alone."""
    from exq_amd.kernels.exq_dispatch import combine
    banner(f"combine batches k={k} H={H} {w_dtype}")
    T = 13
    rng = np.random.default_rng(k * 1000 + H)
    down = torch.from_numpy(rng.standard_normal((T * k, H)).astype(np.float32))
    w = torch.from_numpy(rng.random((T, k)).astype(np.float32)).to(w_dtype)
    order = rng.permutation(T * k)
    res = torch.empty(T, H, dtype=torch.float32, device=device)
    ref = moe.combine(down.numpy(), order, w.float().numpy())
    down[0] = float("nan")
    combine(down.to(device), torch.from_numpy(order).to(device), w.to(device), res)
    got = res.cpu().numpy()
    own = order[0] // k
    keep = np.arange(T) != own
    # fp32 sums of k products of order 1: k ulp
    assert np.allclose(got[keep], ref[keep], rtol=k * 2.4e-7, atol=k * 2.4e-7)
    assert np.isnan(got[own]).all()


def test_combine_past_2_32_outputs(device):
    """More outputs than a launch has threads along one dimension."""
    from exq_amd.kernels import unsort_output
    T, N = (1 << 20) + 1, 4097
    banner(f"unsort_output T={T} N={N}")
    gen = torch.Generator(device=device).manual_seed(1)
    ids = torch.randint(0, 4, (T, 1), generator=gen, device=device)
    pos = torch.empty(T, dtype=torch.int64, device=device)
    pos[torch.argsort(ids[:, 0], stable=True)] = torch.arange(T, device=device)
    y = (torch.arange(T, device=device) % 251).to(torch.bfloat16)  # whole numbers: exact
    w = torch.full((T, 1), 0.5, device=device)
    out = unsort_output(y[:, None].expand(T, N).contiguous(), ids, w, 4)
    want = (pos % 251).to(torch.bfloat16) * 0.5
    assert all(bool((out[i:i + 65536] == want[i:i + 65536, None]).all())
               for i in range(0, T, 65536))


@pytest.mark.parametrize("rows,I", [(1, 8), (3, 12), (5, 1), (129, 2056)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_silu_and_mul_widths(rows, I, dtype, device):
    from exq_amd.kernels.exq_dispatch import silu_and_mul
    banner(f"silu_and_mul {rows} x {I} {dtype}")
    x = torch.from_numpy((np.random.default_rng(I).standard_normal((rows, 2 * I)) * 4)
                         .astype(np.float32)).to(dtype)
    out = torch.empty(rows, I, dtype=dtype, device=device)
    silu_and_mul(x.to(device), out)
    ref = moe.silu_and_mul(x.float().numpy().astype(np.float64))
    tol = {torch.float32: 1e-5, torch.bfloat16: 8e-3}[dtype]
    assert np.allclose(out.float().cpu().numpy(), ref, rtol=tol, atol=tol * 1e-2)
