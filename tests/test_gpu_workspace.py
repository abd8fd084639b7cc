"""Calls whose workspace the device has no memory for take the way that needs
less: the same results as that way gives by itself."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dit_sparse_atten_amd import ops as module
    return module


@pytest.fixture
def short_of_memory(ops, monkeypatch):
    """Workspaces above the given bytes do not fit; returns the sizes asked for."""
    empty, asked = torch.empty, []

    def limit(most):
        def allocate(*size, dtype=None, **kwargs):
            if dtype is torch.uint8:
                asked.append(size[0])
                if size[0] > most:
                    raise torch.OutOfMemoryError("no memory for this workspace")
            return empty(*size, dtype=dtype, **kwargs)

        monkeypatch.setattr(ops.torch, "empty", allocate)
        return asked

    return limit


def _qkv(tokens, heads, device, dtype):
    generator = torch.Generator(device=device).manual_seed(tokens)
    return [torch.randn(1, tokens, heads, 128, device=device, generator=generator).to(dtype)
            for _ in range(3)]


def test_float32_attention_without_room_for_the_split(ops, cuda_device, monkeypatch,
                                                      short_of_memory):
    q, k, v = _qkv(1100, 2, cuda_device, torch.float32)
    asked = short_of_memory(1 << 20)
    got = ops.bsa_fwd(q, k, v)
    assert len(asked) == 1
    monkeypatch.undo()
    monkeypatch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
    assert torch.equal(got, ops.bsa_fwd(q, k, v))


def test_no_float32_workspace_where_the_split_is_not_taken(ops, cuda_device, short_of_memory):
    """Head dims below 64 with a route or a causal mask, and few keys."""
    generator = torch.Generator(device=cuda_device).manual_seed(0)
    q, k, v = (torch.randn(1, 512, 2, 32, device=cuda_device, generator=generator)
               for _ in range(3))
    csr = ops.route_to_csr(torch.ones(2, 4, 4, dtype=torch.bool, device=cuda_device))
    asked = short_of_memory(1 << 40)
    ops.bsa_fwd(q, k, v, csr)
    ops.bsa_fwd(q, k, v, causal=True)
    ops.bsa_fwd(q, k[:, :64], v[:, :64])
    assert not asked
    ops.bsa_fwd(q, k, v)
    assert len(asked) == 1


def test_sampled_mass_without_room_for_its_sums(ops, cuda_device, monkeypatch, short_of_memory):
    q, k, _ = _qkv(13312, 40, cuda_device, torch.bfloat16)
    want = ops.sampled_block_mass(q, k, 128, 32)
    full = 1040 * 128 * 512
    asked = short_of_memory(0)
    got = ops.sampled_block_mass(q, k, 128, 32)
    assert asked == [full, full // 2]
    # Two scans: another order of the same fp32 sums (one exp2 per score each).
    torch.testing.assert_close(got, want, rtol=2.5e-4, atol=1e-9)


def test_partial_block_mass_without_room_for_its_row_sums(ops, cuda_device, monkeypatch,
                                                          short_of_memory):
    q, k, v = _qkv(4097, 3, cuda_device, torch.bfloat16)
    want_out, want_lse = ops.bsa_fwd(q, k, v, return_lse=True)
    want = ops.block_mass(q, k, want_lse)
    attention = ops._lib.load().dsa_bsa_workspace_bytes(1, 3, 4097, 128)
    asked = short_of_memory(attention)
    out, lse, mass = ops.bsa_fwd_block_mass(q, k, v)
    assert len(asked) == 2 and asked[1] == attention
    assert torch.equal(out, want_out) and torch.equal(lse, want_lse) and torch.equal(mass, want)


def test_float32_statistics_without_room_for_the_split(ops, cuda_device, monkeypatch,
                                                       short_of_memory):
    q, k, v = _qkv(2048, 2, cuda_device, torch.float32)
    lib = ops._lib.load()
    calls = (("dsa_bsa_fwd_tile_stats", lambda: ops.bsa_fwd_tile_stats(q, k, v, None, (8, 8)),
              lib.dsa_bsa_fwd_tile_stats_workspace_bytes(2, 2048, 128, 8, 8, 2 * 32 * 32)),
             ("dsa_bsa_fwd_block_mass", lambda: ops.bsa_fwd_block_mass(q, k, v),
              lib.dsa_bsa_fwd_block_mass_workspace_bytes(2, 2048, 128)))
    for name, call, own in calls:
        with monkeypatch.context() as patch:
            patch.setattr(ops, "_f32_workspace_bytes", lambda *args: 0)
            want = call()[0]
        asked = short_of_memory(own)
        got = call()[0]
        monkeypatch.undo()
        assert len(asked) == 2 and asked[1] == own, name
        asked.clear()
        assert torch.equal(got, want), name


def test_a_workspace_it_cannot_do_without(ops, cuda_device, monkeypatch, short_of_memory):
    q, k, v = _qkv(4096, 2, cuda_device, torch.bfloat16)
    short_of_memory(1 << 20)
    with pytest.raises(torch.OutOfMemoryError):
        ops.bsa_fwd_tile_stats(q, k, v, None, (8, 8))
