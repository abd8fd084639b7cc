"""GPU parity of the float32 calls (split fp16 products, csrc/bsa_fwd_f32s.hip,
and the fp32 matrix-core kernel, csrc/bsa_fwd_f32.hip) against float64 closed
forms and the oracle.

The reference computes in the dtype it is given: DenseBackend hands
``dtype`` to SDPA (attention_backends/dense.py:34-47) and MatrixSparseBackend
computes in q's own dtype (sparse.py:700-708), which is how its float32
golden fixtures were written.  Either path accumulates in fp32 and holds its
operands and probabilities to an fp32 rounding or two, so the bar is fp32
rounding: outputs within 2e-5 of the float64 closed form (values of order
one), LSE within 2e-5, statistics within rtol 1e-5.
"""

import functools
import math

import numpy as np
import pytest
import torch

from oracle import attention as A
from oracle import sparse_path as S
from tests.golden.inputs import clustered_qkv, random_route

pytestmark = pytest.mark.gpu

OUT_ATOL = 2e-5
LSE_ATOL = 2e-5
MASS_RTOL = 1e-5


@pytest.fixture(scope="module")
def ops():
    from dit_sparse_atten_amd import ops as module
    return module


def _qkv(batch, q_tokens, kv_tokens, heads, head_dim, seed):
    generator = torch.Generator().manual_seed(seed)
    q = torch.randn(batch, q_tokens, heads, head_dim, generator=generator)
    k = torch.randn(batch, kv_tokens, heads, head_dim, generator=generator)
    v = torch.randn(batch, kv_tokens, heads, head_dim, generator=generator)
    return q, k, v


def _check(out, lse, want_out, want_lse):
    out = out.double().cpu().numpy()
    assert np.isfinite(out).all()
    np.testing.assert_allclose(out, want_out, atol=OUT_ATOL, rtol=0)
    if lse is not None:
        np.testing.assert_allclose(lse.double().cpu().numpy(), want_lse, atol=LSE_ATOL, rtol=0)


@pytest.mark.parametrize("batch,q_tokens,kv_tokens,heads,head_dim,causal", [
    (1, 1000, 1000, 3, 128, False),
    (2, 333, 333, 2, 64, True),
    (1, 256, 256, 2, 8, False),
    (2, 200, 517, 2, 128, False),   # cross-attention (unequal lengths)
])
def test_fp32_dense_matches_float64(ops, cuda_device, batch, q_tokens, kv_tokens, heads,
                                    head_dim, causal):
    q, k, v = _qkv(batch, q_tokens, kv_tokens, heads, head_dim, seed=q_tokens + head_dim)
    out, lse = ops.bsa_fwd(*(x.to(cuda_device) for x in (q, k, v)), return_lse=True,
                           causal=causal)
    torch.cuda.synchronize()
    assert out.dtype == torch.float32
    want_out, want_lse = A.block_sparse_attention(q.numpy(), k.numpy(), v.numpy(), None, 128,
                                                  causal=causal)
    _check(out, lse, want_out, want_lse)


@pytest.mark.parametrize("tokens,block", [(1024, 128), (1000, 64), (720, 72), (1000, 100),
                                          (512, 16), (40, 1)])
def test_fp32_routed_matches_float64(ops, cuda_device, tokens, block):
    """Routed calls of whole and partial blocks of 1..128 tokens, rows with
    empty routes included, against the float64 closed form."""
    heads = 2
    q, k, v = _qkv(1, tokens, tokens, heads, 128, seed=tokens + block)
    blocks = math.ceil(tokens / block)
    route = random_route(heads, blocks, seed=block, keep=0.5).numpy()
    route[0, 0] = False  # one empty row
    csr = ops.route_to_csr(torch.from_numpy(route).to(cuda_device), block_size=block)
    out, lse = ops.bsa_fwd(*(x.to(cuda_device) for x in (q, k, v)), csr, return_lse=True,
                           block_size=block)
    torch.cuda.synchronize()
    want_out, want_lse = A.block_sparse_attention(q.numpy(), k.numpy(), v.numpy(), route, block)
    _check(out, lse, want_out, want_lse)
    assert (out[0, :block, 0] == 0).all()


@pytest.mark.parametrize("tokens,heads,block,routed", [
    (33, 8, 128, False), (97, 8, 128, False), (130, 8, 64, True), (4096, 16, 64, True),
    (1100, 8, 100, True)])
def test_fp32_split_heads_against_fp32_products(ops, cuda_device, monkeypatch, tokens, heads,
                                                block, routed):
    """Heads of very different magnitudes in one call, with the workspace (split
    fp16 products) and without (fp32 products): each head by its own scales, and
    heads with non-finite or extreme elements on the fp32 kernel, bit for bit.
    2-wave workgroups with one stage (1,024 of them) and with two, 4-wave ones,
    sub-tiles of 1, 2, 4 and 32 keys, and (1,100 tokens: 88 workgroups, 11 key
    blocks) every query block in two key ranges.  33 tokens: every head on the
    fp32 kernel (few keys)."""
    q, k, v = (x.to(cuda_device) for x in _qkv(1, tokens, tokens, heads, 128, seed=tokens))
    q[:, :, 1] *= 2.0 ** 20
    k[:, :, 1] *= 2.0 ** -20
    v[:, :, 1] *= 2.0 ** -30
    v[:, :, 2] *= 2.0 ** 30
    q[:, :, 2] = 0
    q[:, :, 3] *= 1e-30              # extreme: fp32 products
    v[0, tokens // 2, 4, 5] = float("inf")
    k[0, tokens - 1, 5, 0] = float("nan")
    q[0, 0, 6, 0] = float("-inf")
    k[0, 3, 7] *= 2.0 ** 20          # one token far above the others
    csr = None
    if routed:
        blocks = math.ceil(tokens / block)
        route = random_route(heads, blocks, seed=block, keep=0.5)
        csr = ops.route_to_csr(route.to(cuda_device), block_size=block)
    got, got_lse = ops.bsa_fwd(q, k, v, csr, return_lse=True, block_size=block)
    monkeypatch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
    want, want_lse = ops.bsa_fwd(q, k, v, csr, return_lse=True, block_size=block)
    torch.cuda.synchronize()
    for head, scale in enumerate((1.0, 2.0 ** -30, 2.0 ** 30)):
        # Two fp32 results, each within OUT_ATOL of float64 at |v| of order one.
        torch.testing.assert_close(got[:, :, head] / scale, want[:, :, head] / scale,
                                   atol=2 * OUT_ATOL, rtol=0)
        torch.testing.assert_close(got_lse[:, head], want_lse[:, head], atol=2 * LSE_ATOL, rtol=0)
    # Two different kernels ran, or with few keys the same one.
    assert torch.equal(got[:, :, 0], want[:, :, 0]) == (tokens == 33)
    for head in range(3, 8):
        assert torch.equal(got[:, :, head].view(torch.int32), want[:, :, head].view(torch.int32))
        assert torch.equal(got_lse[:, head].view(torch.int32),
                           want_lse[:, head].view(torch.int32))


@pytest.mark.parametrize("q_tokens,kv_tokens,split", [
    (64, 64, False), (16500, 64, False), (96, 96, False), (16384, 96, False), (16500, 65, True),
    (16500, 96, True), (97, 97, True)])
def test_fp32_few_keys_keep_one_launch(ops, cuda_device, monkeypatch, q_tokens, kv_tokens, split):
    """Up to 64 keys, and up to 96 with at most 256 query blocks, a float32 call
    runs the fp32 kernel alone (2 heads: 16,384 queries are 256 blocks)."""
    q, k, v = (x.to(cuda_device) for x in _qkv(1, q_tokens, kv_tokens, 2, 128, seed=kv_tokens))
    got = ops.bsa_fwd(q, k, v)
    monkeypatch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
    want = ops.bsa_fwd(q, k, v)
    assert torch.equal(got, want) != split
    torch.testing.assert_close(got, want, atol=2 * OUT_ATOL, rtol=0)


@pytest.mark.parametrize("tokens,routed", [(1024, False), (6000, False), (6016, True)])
def test_fp32_split_error_is_no_larger(ops, cuda_device, monkeypatch, tokens, routed):
    """Relative error of O against float64 (torch, on the device): the split
    products' is at most that of the fp32 products."""
    q, k, v = (x.to(cuda_device) for x in _qkv(1, tokens, tokens, 2, 128, seed=tokens))
    route = torch.ones(2, -(-tokens // 128), -(-tokens // 128), dtype=torch.bool)
    if routed:
        route = random_route(2, route.shape[1], seed=3, keep=0.5)
    csr = ops.route_to_csr(route.to(cuda_device)) if routed else None
    keep = route.to(cuda_device).repeat_interleave(128, 1).repeat_interleave(128, 2)
    s = (q[0].double().transpose(0, 1) @ k[0].double().permute(1, 2, 0).contiguous()) * 128 ** -0.5
    s.masked_fill_(~keep[:, :tokens, :tokens], -math.inf)
    exact = (torch.softmax(s, dim=-1) @ v[0].double().transpose(0, 1).contiguous()).transpose(0, 1)
    errors = []
    for workspace in (True, False):
        if not workspace:
            monkeypatch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
        out = ops.bsa_fwd(q, k, v, csr)[0].double()
        errors.append(((out - exact).norm() / exact.norm()).item())
    assert errors[0] <= errors[1] <= 1e-5, errors


def _dense_float64(q, k, v):
    """O [T, H, D] in float64 (torch, on the device)."""
    s = (q[0].double().transpose(0, 1) @ k[0].double().permute(1, 2, 0).contiguous())
    p = torch.softmax(s * q.shape[-1] ** -0.5, dim=-1)
    return (p @ v[0].double().transpose(0, 1).contiguous()).transpose(0, 1)


def _sink(q, k, strength):
    """Token 7 of head 1 takes a row's attention e^(8 strength / sqrt(128)) times
    over any other."""
    q[:, :, 1, 0] = 8
    k[:, :, 1, 0] = 0
    k[:, 7, 1, 0] = strength


def _spread_inputs(kind, power, q, k, v):
    """Gives head 1 dims or tokens of very different magnitudes; returns the
    first output dim to compare."""
    if kind == "v_dim":
        v[:, :, 1, 0] *= 2.0 ** power
        return 1
    if kind == "qk_dim":
        k[:, :, 1, 0] *= 2.0 ** power
        q[:, :, 1, 0] *= 2.0 ** -power
    elif kind == "k_dim":
        k[:, :, 1, 0] *= 2.0 ** power
    elif kind == "q":
        q[:, :, 1] *= 2.0 ** power
    elif kind == "v_tokens":  # in every range of tokens, and given no attention
        q[:, :, 1, 0] = 8
        k[:, :, 1, 0] = 0
        k[:, ::8, 1, 0] = -40
        v[:, ::8, 1] *= 2.0 ** power
    elif kind == "v_tokens_dims":  # even tokens large in dim 0, odd ones in the others
        q[:, :, 1, 0] = 8
        k[:, :, 1, 0] = 0
        k[:, 1::2, 1, 0] = -40
        v[:, ::2, 1, 0] *= 2.0 ** power
        v[:, 1::2, 1, 1:] *= 2.0 ** power
        return 8
    elif kind == "sink":
        _sink(q, k, 26)
        v[:, 7, 1] *= 2.0 ** power
    elif kind == "sink_zero":
        _sink(q, k, 26)
        v[:, 7, 1] = 0
    elif kind == "sink_one_dim":
        _sink(q, k, 30)
        v[:, 7, 1, 1:] *= 2.0 ** power
        return 8
    elif kind == "zero_dims":  # 64 dims used of 128: exact zeros, which cost nothing
        for x in (q, k, v):
            x[:, :, 1, 64:] = 0
    return 0


@pytest.mark.parametrize("kind,power,split", [
    ("v_dim", 6, True), ("v_dim", 18, False), ("v_dim", 24, False), ("v_dim", 38, False),
    ("qk_dim", 6, True), ("qk_dim", 20, False), ("qk_dim", 24, False),
    ("k_dim", 6, True), ("k_dim", 16, False), ("q", 5, True), ("q", 11, False),
    ("v_tokens", 6, True), ("v_tokens", 28, False), ("v_tokens_dims", 24, False),
    ("sink", -6, True), ("sink", -14, False), ("sink_zero", 0, False),
    ("sink_one_dim", -30, False), ("zero_dims", 0, True)])
@pytest.mark.parametrize("tokens", [256, 1100])
def test_fp32_split_error_on_spread_inputs(ops, cuda_device, monkeypatch, tokens, kind, power,
                                           split):
    """Finite heads whose dims or tokens differ widely: the error of O against
    float64 is at most that of the fp32 products, over the dims that are not the
    large ones.  ``split``: whether the head runs on the split products (the
    other head always does)."""
    q, k, v = (x.to(cuda_device) for x in _qkv(1, tokens, tokens, 2, 128, seed=tokens))
    first = _spread_inputs(kind, power, q, k, v)
    exact = _dense_float64(q, k, v)[:, 1, first:]
    got = ops.bsa_fwd(q, k, v)[0]
    monkeypatch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
    want = ops.bsa_fwd(q, k, v)[0]
    assert not torch.equal(got[:, 0], want[:, 0])
    assert torch.equal(got[:, 1], want[:, 1]) != split
    errors = [((x[:, 1, first:].double() - exact).norm() / exact.norm()).item()
              for x in (got, want)]
    assert errors[0] <= errors[1], errors


@pytest.mark.parametrize("tokens,head_dim,causal,routed,split", [
    (160, 8, False, False, False), (256, 8, False, False, True), (600, 8, True, False, False),
    (1024, 32, False, True, False), (256, 64, False, True, True), (256, 64, True, False, True)])
def test_fp32_split_error_of_short_rows(ops, cuda_device, monkeypatch, tokens, head_dim, causal,
                                        routed, split):
    """Head dims below 64 keep the fp32 products unless every row attends 256
    keys: with fewer their error is the smaller one."""
    q, k, v = (x.to(cuda_device) for x in _qkv(1, tokens, tokens, 2, head_dim, seed=tokens))
    csr = None
    if routed:
        csr = ops.route_to_csr(random_route(2, tokens // 32, seed=3, keep=0.5).to(cuda_device),
                               block_size=32)
    call = functools.partial(ops.bsa_fwd, q, k, v, csr, causal=causal,
                             block_size=32 if routed else 128)
    got = call()
    monkeypatch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
    assert torch.equal(got, call()) != split


def _tile_inputs(grid, tile, heads, seed):
    case = S.SparsePathCase(grid, tile=tile)
    tokens = grid[0] * grid[1] * grid[2]
    perm = torch.as_tensor(case.permutation, dtype=torch.long)
    q, k, v = clustered_qkv(tokens, heads, 128, group=case.tile, seed=seed, permutation=perm)
    return case, q[:, perm].contiguous(), k[:, perm].contiguous(), v[:, perm].contiguous()


def _oracle(case, q, k, v, route):
    qf, kf, vf = (x.numpy() for x in (q, k, v))
    tokens, heads = qf.shape[1:3]
    tiles = tokens // case.tile
    stats = S.empty_stats(heads, tiles)
    offsets = S.spatial_offsets(case.tile_shape, tiles)
    scale = 128 ** -0.5
    if route is None:
        _, _, out = S.dense_route(qf, kf, vf, case.tile, 256, 0.95, 0.625, scale, stats, offsets)
    else:
        out = np.empty_like(qf)
        for start in range(0, tokens, case.tile * 4):
            end = min(start + case.tile * 4, tokens)
            out[:, start:end] = S.sparse_chunk(qf, kf, vf, route, case.tile, start, end, scale,
                                               stats, offsets)
    return stats, out


@pytest.mark.parametrize("routed", [True, False])
@pytest.mark.parametrize("grid,tile", [((4, 16, 16), 64), ((2, 18, 32), 64), ((2, 15, 26), 64),
                                       ((2, 22, 22), 121), ((2, 12, 12), 36)])
def test_fp32_tile_step_matches_oracle(ops, cuda_device, routed, grid, tile):
    """dsa_bsa_fwd_tile_stats in float32 (8 x 8, 9 x 8, 5 x 13, 11 x 11 and
    6 x 6 tiles, routed and dense) against the oracle's sparse_chunk /
    _dense_route restatement in float32: output, mass at rtol 1e-5, the fp16
    mass and centroids at fp16 rounding."""
    case, q, k, v = _tile_inputs(grid, tile, 2, seed=sum(grid) + tile)
    tokens = q.shape[1]
    tiles = tokens // case.tile
    route = None
    csr = None
    if routed:
        route = random_route(2, tiles, seed=tile, keep=0.55).numpy()
        route[..., 0] = True
        csr = ops.route_to_csr(torch.from_numpy(route).to(cuda_device), block_size=case.tile)
    out, _, got = ops.bsa_fwd_tile_stats(*(x.to(cuda_device) for x in (q, k, v)), csr,
                                         case.tile_shape, deterministic=True)
    torch.cuda.synchronize()
    stats, want_out = _oracle(case, q, k, v, route)
    np.testing.assert_allclose(out.double().cpu().numpy(), want_out, atol=OUT_ATOL, rtol=0)
    mass = stats["mass"] / np.float32(tokens)
    np.testing.assert_allclose(got["mass"].cpu().numpy(), mass, rtol=MASS_RTOL, atol=1e-9)
    np.testing.assert_allclose(got["mass_f16"].float().cpu().numpy(), mass, rtol=1e-3, atol=1e-7)
    den = np.maximum(stats["mass"], np.float32(1e-12))
    for name in ("q_y", "q_x", "k_y", "k_x"):
        np.testing.assert_allclose(got[f"centroid_{name}"].float().cpu().numpy(),
                                   stats[name] / den, atol=1e-3, err_msg=name)
    if routed:
        assert (got["mass"].cpu().numpy()[~route] == 0).all()


def test_fp32_statistics_take_one_scratch(ops, cuda_device):
    """The workspace of a float32 call with statistics holds the row statistics
    and the split products' scratch, not the 16-bit kernels' beside them: 2,048
    tokens x 2 heads in 8 x 8 tiles, peak memory of the call."""
    tokens, heads, tiles = 2048, 2, 32
    q, k, v = (x.to(cuda_device) for x in _qkv(1, tokens, tokens, heads, 128, seed=1))
    for call, rows in ((lambda: ops.bsa_fwd_tile_stats(q, k, v, None, (8, 8)),
                        8 * tiles * tiles * 64),
                       (lambda: ops.bsa_fwd_block_mass(q, k, v), 4 * 16 * 16 * 128)):
        call()
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        outputs = call()  # noqa: F841 (held while the peak is read)
        peak = torch.cuda.max_memory_allocated() - before
        split = heads * (5 * 64 * 4 + 2 * tokens * 512) + 1024 * (128 * 128 + 256) * 4
        out = 4 * tokens * heads * 129 + heads * tiles * tiles * 14
        assert peak <= split + heads * rows + out + (4 << 20), peak


def test_fp32_block_mass_matches_float64(ops, cuda_device):
    """The exact 128-token block mass of a float32 dense call (the flex
    backend's exact bootstrap) against the float64 closed form."""
    q, k, v = _qkv(1, 640, 640, 2, 128, seed=5)
    out, lse, mass = ops.bsa_fwd_block_mass(*(x.to(cuda_device) for x in (q, k, v)))
    torch.cuda.synchronize()
    want_out, want_lse = A.block_sparse_attention(q.numpy(), k.numpy(), v.numpy(), None, 128)
    _check(out, lse, want_out, want_lse)
    qd, kd = q.double().numpy()[0], k.double().numpy()[0]
    blocks = 5
    want = np.zeros((2, blocks, blocks))
    for h in range(2):
        p = np.exp(qd[:, h] @ kd[:, h].T * 128 ** -0.5 - want_lse[0, h][:, None])
        want[h] = p.reshape(blocks, 128, blocks, 128).sum((1, 3))
    np.testing.assert_allclose(mass.double().cpu().numpy(), want, rtol=MASS_RTOL, atol=1e-9)


def test_fp32_through_the_dense_and_flex_backends(cuda_device):
    """DenseBackend with dtype=float32, and FlexReuseBackend's float32 calls
    (exact bootstrap on the fp32 block mass, then a routed step), against the
    float64 closed form of the route each step used."""
    from dit_sparse_atten_amd.attention_backends import context
    from dit_sparse_atten_amd.attention_backends.dense import DenseBackend
    from dit_sparse_atten_amd.attention_backends.flex import FlexReuseBackend, FlexReuseConfig
    q, k, v = _qkv(1, 1024, 1024, 2, 128, seed=9)
    qd, kd, vd = (x.to(cuda_device) for x in (q, k, v))
    dense = DenseBackend()(qd, kd, vd, dtype=torch.float32)
    want, _ = A.block_sparse_attention(q.numpy(), k.numpy(), v.numpy(), None, 128)
    np.testing.assert_allclose(dense.double().cpu().numpy(), want, atol=OUT_ATOL, rtol=0)

    backend = FlexReuseBackend(FlexReuseConfig(keep=0.5))
    context.reset_runtime_state()
    try:
        context.set_routing_context(attention_id=1, step=0, branch=0, grid=None)
        out0 = backend(qd, kd, vd, dtype=torch.float32)
        state = next(iter(backend.state.values()))
        route = state["route"].clone()
        context.set_routing_context(step=1)
        out1 = backend(qd, kd, vd, dtype=torch.float32)
        torch.cuda.synchronize()
    finally:
        context.reset_runtime_state()
    assert out0.dtype == torch.float32 and out1.dtype == torch.float32
    np.testing.assert_allclose(out0.double().cpu().numpy(), want, atol=OUT_ATOL, rtol=0)
    routed, _ = A.block_sparse_attention(q.numpy(), k.numpy(), v.numpy(),
                                         route.cpu().numpy(), 128)
    np.testing.assert_allclose(out1.double().cpu().numpy(), routed, atol=OUT_ATOL, rtol=0)
    assert not route.cpu().numpy().all()


def test_fp32_batched_routes_and_strided_views(ops, cuda_device):
    """Two batch items with their own routes (route_batches 2), read through
    the transposed views of BHSD storage the Diffusers processor passes, with
    a partial last block, against the float64 closed form."""
    batch, heads, tokens, block = 2, 3, 700, 128
    generator = torch.Generator().manual_seed(12)
    bhsd = [torch.randn(batch, heads, tokens, 64, generator=generator) for _ in range(3)]
    q, k, v = (x.to(cuda_device).transpose(1, 2) for x in bhsd)
    assert not q.is_contiguous()
    blocks = math.ceil(tokens / block)
    route = np.stack([random_route(heads, blocks, seed=20 + b, keep=0.6).numpy()
                      for b in range(batch)])
    csr = ops.route_to_csr(torch.from_numpy(route).to(cuda_device), block_size=block)
    out, lse = ops.bsa_fwd(q, k, v, csr, return_lse=True, block_size=block)
    torch.cuda.synchronize()
    want, want_lse = A.block_sparse_attention(*(x.transpose(1, 2).numpy() for x in bhsd),
                                              route, block)
    _check(out, lse, want, want_lse)
