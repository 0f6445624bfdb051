"""GPU parity of extend (chunked prefill) attention through the C ABI:
each sequence's newest tokens attend causally over the whole cache,
against the oracle (bf16 row-relative 2e-2, f32 max-abs 1e-5), plus the
identities the oracle tests pin (the chunk's last query equals decode
attention) and the error paths. Three paths: bf16 and f32 MFMA row tiles
(head_dim 64/128/256) and per-token decode segments (head_dim 32)."""
from __future__ import annotations

import numpy as np
import pytest

from mitten_amd import BackendError, DeviceIndexError, DeviceKvPool, PoolDesc
from mitten_amd import device_pool as dp
from mitten_amd import workloads as wl
from oracle import oracle as orc
from tests.helpers import assert_attention_close, bits, normal, odesc, to_device, to_host, widen

pytestmark = pytest.mark.gpu

SHAPES = {
    # name: (Hq, Hkv, D): query heads per KV head G = 7, 8, 7, 4, 16, 1, 4, 16
    "qwen7b": (28, 4, 128),
    "gemma2b": (8, 1, 256),
    "qwen0.5b": (14, 2, 64),
    "llama8b": (32, 8, 128),
    "g16": (64, 4, 128),
    "mha": (4, 4, 64),
    "d256-g4": (16, 4, 256),
    "d256-g16": (16, 1, 256),
}
# Shapes beside the engine's bf16 ones: f32, head_dim 32, large groups.
SEGMENT_SHAPES = {
    # name: (Hq, Hkv, D, dtype)
    "qwen0.5b-f32": (14, 2, 64, "f32"),   # the reference's CPU-runnable configuration
    "d32-f32": (8, 4, 32, "f32"),
    "d128-f32": (28, 4, 128, "f32"),
    "g32-bf16": (64, 2, 128, "bf16"),     # 32 query heads per KV head
    "d32-bf16": (8, 2, 32, "bf16"),
}


def _i32(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()


def _case(shape, ctx, nq, seed, zero_sink=False, layer=1, dtype="bf16"):
    """shape: a SHAPES name or an (Hq, Hkv, D) tuple."""
    Hq, Hkv, D = SHAPES[shape] if isinstance(shape, str) else shape
    rng = wl.SplitMix64(seed)
    batch = wl.decode_batch_from_contexts([c - 1 for c in ctx], rng, extra_blocks=2)
    desc = PoolDesc(2, Hkv, Hq, D, batch.num_blocks, dtype)
    host = normal(seed + 1, desc.shape, dtype)
    q_indptr = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    q = normal(seed + 2, (int(q_indptr[-1]), Hq, D), dtype)
    with DeviceKvPool(desc) as pool:
        pool.write(host)
        o = pool.extend_attention(layer, to_device(q), _i32(q_indptr), _i32(batch.block_indptr),
                                  _i32(batch.block_ids), _i32(batch.ctx_lens), max(nq), max(ctx),
                                  zero_sink=zero_sink)
        pool.check()
        got = to_host(o)
        dec = None
        if not zero_sink:  # the last query of each chunk is a decode query over the whole context
            last = q_indptr[1:] - 1
            dec = to_host(pool.decode_attention(layer, to_device(q[last]), _i32(batch.block_indptr),
                                                _i32(batch.block_ids), _i32(batch.ctx_lens), max(ctx)))
    ref = orc.extend_attention(odesc(desc), host, layer, widen(q), q_indptr, batch.block_indptr,
                               batch.block_ids, batch.ctx_lens, zero_sink=zero_sink)
    return got, ref, dec, q_indptr


CTX = [1, 16, 17, 40, 200, 530, 97]
NQ = [1, 16, 5, 40, 33, 512, 1]  # whole prompts, chunks after a prefix, a single token


@pytest.mark.parametrize("shape", list(SHAPES))
def test_extend_attention_matches_oracle(shape):
    got, ref, dec, q_indptr = _case(shape, CTX, NQ, 90)
    assert_attention_close(got, ref, "bf16")
    last = q_indptr[1:] - 1
    assert_attention_close(dec, ref[last], "bf16")


def test_extend_attention_zero_sink():
    got, ref, _, _ = _case("qwen7b", [1, 20, 300], [1, 20, 64], 91, zero_sink=True)
    assert_attention_close(got, ref, "bf16")


@pytest.mark.parametrize("shape", ["qwen7b", "qwen0.5b", "mha"])
def test_extend_short_chunks(shape):
    """Chunks of at most 16 tokens (workgroups that compute few rows) after
    prefixes of assorted lengths."""
    got, ref, dec, q_indptr = _case(shape, [16, 300, 1000, 47, 8], [16, 1, 9, 16, 3], 97)
    assert_attention_close(got, ref, "bf16")
    assert_attention_close(dec, ref[q_indptr[1:] - 1], "bf16")


def test_extend_long_context_chunk():
    """A 512-token chunk at the end of an 8k context (the pool-pressure
    configuration's chunked prefill)."""
    got, ref, _, _ = _case("qwen7b", [8192, 700], [512, 64], 92)
    assert_attention_close(got, ref, "bf16")


def test_extend_key_range_past_the_staged_ids():
    """A workgroup whose key range holds more blocks than the kernel stages
    in LDS for its unmasked steps (1,024 ids) takes the generic step
    throughout: one 16-token chunk at the end of a 16,900-token context
    (1,057 blocks), beside 255 short prompts so that the launch fills the
    device and the long range is not split."""
    ctx = [16900] + [16] * 255
    nq = [16] * 256
    got, ref, dec, q_indptr = _case("qwen7b", ctx, nq, 98)
    assert_attention_close(got, ref, "bf16")
    assert_attention_close(dec, ref[q_indptr[1:] - 1], "bf16")


def test_extend_errors_are_reported():
    Hq, Hkv, D = SHAPES["qwen7b"]
    desc = PoolDesc(1, Hkv, Hq, D, 10, "bf16")
    with DeviceKvPool(desc) as pool:
        pool.write(normal(93, desc.shape, "bf16"))
        q = to_device(normal(94, (4, Hq, D), "bf16"))
        qi = _i32([0, 2, 4])
        # block id outside the pool
        pool.extend_attention(0, q, qi, _i32([0, 2, 4]), _i32([1, 2, 3, 10]), _i32([20, 30]), 2, 30)
        with pytest.raises(DeviceIndexError) as ei:
            pool.check()
        assert ei.value.bits & dp.DEVERR_BLOCK
        # table too short for the context
        pool.extend_attention(0, q, qi, _i32([0, 1, 3]), _i32([1, 2, 3]), _i32([20, 30]), 2, 30)
        with pytest.raises(DeviceIndexError) as ei:
            pool.check()
        assert ei.value.bits & dp.DEVERR_TABLE
        # context beyond max_ctx_len
        pool.extend_attention(0, q, qi, _i32([0, 2, 4]), _i32([1, 2, 3, 4]), _i32([20, 30]), 2, 25)
        with pytest.raises(DeviceIndexError) as ei:
            pool.check()
        assert ei.value.bits & dp.DEVERR_CTX
        with pytest.raises(BackendError):  # max_q_len > max_ctx_len
            pool.extend_attention(0, q, qi, _i32([0, 2, 4]), _i32([1, 2, 3, 4]), _i32([20, 30]), 40, 30)
    f32 = PoolDesc(1, 2, 14, 64, 4, "f32")
    with DeviceKvPool(f32) as pool:
        import torch

        q = torch.zeros((2, 14, 64), dtype=torch.bfloat16, device="cuda")
        with pytest.raises(BackendError):  # q must be in the pool dtype
            pool.extend_attention(0, q, _i32([0, 2]), _i32([0, 1]), _i32([0]), _i32([2]), 2, 2)


def test_extend_split_key_ranges_with_empty_splits():
    """Few sequences over long contexts split each key range (f32 partials,
    then a merge); short contexts in the same launch leave some splits with
    no blocks, which must merge as empty partials."""
    got, ref, dec, q_indptr = _case("qwen7b", [3000, 1, 17, 6000, 40], [16, 1, 3, 12, 40], 98)
    assert_attention_close(got, ref, "bf16")
    assert_attention_close(dec, ref[q_indptr[1:] - 1], "bf16")


def test_extend_split_rejects_chunk_past_max_q_len():
    """With split key ranges chunks past num_seqs * max_q_len tokens are
    reported (their partial rows would lie past the workspace), not written."""
    Hq, Hkv, D = SHAPES["qwen7b"]
    rng = wl.SplitMix64(99)
    batch = wl.decode_batch_from_contexts([2000 - 1], rng, extra_blocks=2)
    desc = PoolDesc(1, Hkv, Hq, D, batch.num_blocks, "bf16")
    with DeviceKvPool(desc) as pool:
        pool.write(normal(99, desc.shape, "bf16"))
        q = to_device(normal(100, (20, Hq, D), "bf16"))
        pool.extend_attention(0, q, _i32([0, 20]), _i32(batch.block_indptr), _i32(batch.block_ids),
                              _i32(batch.ctx_lens), 16, 2000)
        with pytest.raises(DeviceIndexError) as ei:
            pool.check()
        assert ei.value.bits & dp.DEVERR_CTX


@pytest.mark.parametrize("name", list(SEGMENT_SHAPES))
def test_extend_segment_path_matches_oracle(name):
    """f32 row tiles, a group above 16 on the bf16 tiles, and head_dim 32 on
    per-token segments: f32 within max-abs 1e-5, bf16 within row-relative 2e-2."""
    Hq, Hkv, D, dt = SEGMENT_SHAPES[name]
    ctx, nq = [1, 17, 40, 300, 97], [1, 17, 25, 64, 1]
    got, ref, dec, q_indptr = _case((Hq, Hkv, D), ctx, nq, 95, dtype=dt)
    assert_attention_close(got, ref, dt)
    assert_attention_close(dec, ref[q_indptr[1:] - 1], dt)
    got, ref, _, _ = _case((Hq, Hkv, D), [50, 33], [20, 33], 96, zero_sink=True, dtype=dt)
    assert_attention_close(got, ref, dt)


@pytest.mark.parametrize("shape", [(14, 2, 64), (3, 1, 64), (40, 1, 64), (2, 2, 128), (5, 1, 256)])
def test_extend_f32_row_tiles(shape):
    """f32 row tiles at their edges: groups that do and do not divide a tile,
    a single row, contexts ending at, before and after a block's last slot,
    chunks after a prefix, and stale slots past the context holding NaN."""
    Hq, Hkv, D = shape
    ctx, nq = [1, 16, 17, 80, 129, 47, 300], [1, 16, 2, 5, 129, 33, 64]
    batch = wl.decode_batch_from_contexts([c - 1 for c in ctx], wl.SplitMix64(101), extra_blocks=2)
    desc = PoolDesc(1, Hkv, Hq, D, batch.num_blocks, "f32")
    host = normal(102, desc.shape, "f32")
    stale = host.copy()
    for b, c in enumerate(ctx):
        if c % 16:
            stale[:, :, batch.block_ids[batch.block_indptr[b] + c // 16], c % 16:] = np.nan
    q_indptr = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    q = normal(103, (int(q_indptr[-1]), Hq, D), "f32")
    args = (to_device(q), _i32(q_indptr), _i32(batch.block_indptr), _i32(batch.block_ids), _i32(batch.ctx_lens))
    with DeviceKvPool(desc) as pool:
        pool.write(stale)
        got = to_host(pool.extend_attention(0, *args, max(nq), max(ctx)))
        pool.check()
        # a rejected block id: its keys are skipped and the call reports it
        bad = batch.block_ids.copy()
        bad[batch.block_indptr[6]] = desc.num_blocks
        pool.extend_attention(0, args[0], args[1], args[2], _i32(bad), args[4], max(nq), max(ctx))
        with pytest.raises(DeviceIndexError) as ei:
            pool.check()
        assert ei.value.bits & dp.DEVERR_BLOCK
    ref = orc.extend_attention(odesc(desc), host, 0, q, q_indptr, batch.block_indptr, batch.block_ids, batch.ctx_lens)
    assert_attention_close(got, ref, "f32")


@pytest.mark.parametrize("shape", [(6, 2, 64), (5, 1, 128), (40, 2, 128), (1, 1, 64), (6, 2, 256)])
@pytest.mark.parametrize("chunks", [
    # (contexts, new tokens): ragged whole prompts (tiles dealt over all
    # sequences) with and without a multiple of 8 (KV head, sequence) pairs,
    # one row, and chunks whose last wave or tile is nearly empty
    ([1, 16, 17, 80, 129, 47, 300, 333], [1, 16, 17, 80, 129, 47, 300, 333]),
    ([257, 3, 40], [257, 3, 40]),
    ([500], [1]),
    ([700, 90, 400], [52, 4, 13]),
])
def test_extend_row_tiles(shape, chunks):
    """bf16 row tiles (row = position * group + head) for groups that do not
    divide a wave's 16 rows, at the edges of waves, tiles and workgroups."""
    ctx, nq = chunks
    got, ref, _, _ = _case(shape, ctx, nq, 104)
    assert_attention_close(got, ref, "bf16")


@pytest.mark.parametrize("shape", [(28, 4, 128, "bf16"), (64, 2, 128, "bf16"), (8, 1, 256, "bf16"), (6, 2, 64, "bf16"),
                                   (14, 2, 64, "f32"), (5, 1, 256, "f32")])
@pytest.mark.parametrize("chunks", [
    # (contexts, new tokens, max_q_len): key ranges in one piece (fewer than
    # 512 keys), one chunk just past a tile and one of many rounds; and key
    # ranges that are cut, the chunks' tokens within num_seqs * max_q_len
    ([200, 150, 30], [70, 150, 5], 16),
    ([90, 255], [2, 255], 1),
    ([2000, 900, 1500], [20, 3, 1], 16),
])
@pytest.mark.parametrize("first", [0, 7])
def test_extend_chunk_longer_than_max_q_len(shape, chunks, first):
    """Every token of q_indptr is computed, whatever max_q_len said of the
    chunks and wherever q_indptr starts, and rows outside it are left alone."""
    Hq, Hkv, D, dt = shape
    ctx, nq, max_q = chunks
    batch = wl.decode_batch_from_contexts([c - 1 for c in ctx], wl.SplitMix64(105), extra_blocks=2)
    desc = PoolDesc(1, Hkv, Hq, D, batch.num_blocks, dt)
    host = normal(106, desc.shape, dt)
    q_indptr = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    total = int(q_indptr[-1])
    q = normal(107, (first + total + 3, Hq, D), dt)
    with DeviceKvPool(desc) as pool:
        pool.write(host)
        out = to_device(np.zeros_like(q))
        pool.extend_attention(0, to_device(q), _i32(q_indptr + first), _i32(batch.block_indptr),
                              _i32(batch.block_ids), _i32(batch.ctx_lens), max_q, max(ctx), out=out)
        pool.check()
        got = to_host(out)
        # a chunk that starts before row 0 is reported, not read
        pool.extend_attention(0, to_device(q), _i32(q_indptr - 2), _i32(batch.block_indptr), _i32(batch.block_ids),
                              _i32(batch.ctx_lens), max_q, max(ctx), out=out)
        with pytest.raises(DeviceIndexError) as ei:
            pool.check()
        assert ei.value.bits & dp.DEVERR_CTX
    ref = orc.extend_attention(odesc(desc), host, 0, widen(q[first:first + total]), q_indptr, batch.block_indptr,
                               batch.block_ids, batch.ctx_lens)
    assert_attention_close(got[first:first + total], ref, dt)
    assert not np.any(got[:first]) and not np.any(got[first + total:])


@pytest.mark.parametrize("shape", [(28, 4, 128, "bf16"), (64, 2, 128, "bf16"), (8, 1, 256, "bf16"), (3, 3, 64, "bf16"),
                                   (14, 2, 64, "f32"), (2, 1, 128, "f32"), (5, 1, 256, "f32")])
@pytest.mark.parametrize("chunks", [
    ([70, 33, 200], [70, 20, 190]),   # whole prompts and chunks, key ranges in one piece
    ([2000, 600, 900], [20, 3, 40]),  # bf16: key ranges that are cut
])
def test_extend_hidden_values_that_are_not_finite(shape, chunks):
    """An Inf or NaN in a token's V row reaches the queries from that token on,
    in its dims alone: a query before it has weight 0 there, not 0 * Inf."""
    Hq, Hkv, D, dt = shape
    ctx, nq = chunks
    batch = wl.decode_batch_from_contexts([c - 1 for c in ctx], wl.SplitMix64(108), extra_blocks=2)
    desc = PoolDesc(1, Hkv, Hq, D, batch.num_blocks, dt)
    host = normal(109, desc.shape, dt)
    inf, nan = (np.inf, np.nan) if dt == "f32" else (0x7F80, 0x7FC1)
    ninf = -np.inf if dt == "f32" else 0xFF80

    def v_row(b, pos):
        return host[0, 1, batch.block_ids[batch.block_indptr[b] + pos // 16], pos % 16]

    v_row(0, ctx[0] - 5)[:, 3] = inf
    v_row(0, ctx[0] - 2)[:, 3] = ninf          # Inf - Inf from here on
    v_row(0, ctx[0] - 9)[Hkv - 1, D - 1] = nan
    v_row(1, ctx[1] - nq[1] + 1)[0, 8:17] = ninf
    v_row(2, ctx[2] - 1)[:] = nan              # the last query alone
    v_row(2, ctx[2] - nq[2])[0, 0] = inf       # every query of the chunk
    q_indptr = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    q = normal(110, (int(q_indptr[-1]), Hq, D), dt)
    with DeviceKvPool(desc) as pool:
        pool.write(host)
        got = widen(to_host(pool.extend_attention(0, to_device(q), _i32(q_indptr), _i32(batch.block_indptr),
                                                  _i32(batch.block_ids), _i32(batch.ctx_lens), max(nq), max(ctx))))
        pool.check()
    ref = orc.extend_attention(odesc(desc), host, 0, widen(q), q_indptr, batch.block_indptr, batch.block_ids,
                               batch.ctx_lens)
    odd = ~np.isfinite(ref)
    assert odd.any() and not odd.all()
    np.testing.assert_array_equal(got[odd], ref[odd])
    assert np.isfinite(got[~odd]).all()
    got, ref = np.where(odd, 0, got).astype(np.float32), np.where(odd, 0, ref).astype(np.float32)
    assert_attention_close(got if dt == "f32" else orc.f32_to_bf16(got), ref, dt)


def test_extend_captured_before_the_workspace_has_room():
    """A call whose key ranges would be split, captured on a pool whose
    workspace was never grown: unsplit, and every replay equals the oracle, with
    the split call of the same sizes (which grows the workspace) in between."""
    import torch

    Hq, Hkv, D = SHAPES["qwen7b"]
    ctx, nq = [2000, 700], [16, 5]
    batch = wl.decode_batch_from_contexts([c - 1 for c in ctx], wl.SplitMix64(111), extra_blocks=2)
    desc = PoolDesc(1, Hkv, Hq, D, batch.num_blocks, "bf16")
    host = normal(112, desc.shape, "bf16")
    q_indptr = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    q = normal(113, (int(q_indptr[-1]), Hq, D), "bf16")
    ref = orc.extend_attention(odesc(desc), host, 0, widen(q), q_indptr, batch.block_indptr, batch.block_ids,
                               batch.ctx_lens)
    with DeviceKvPool(desc) as pool:
        pool.write(host)
        args = (to_device(q), _i32(q_indptr), _i32(batch.block_indptr), _i32(batch.block_ids), _i32(batch.ctx_lens),
                max(nq), max(ctx))
        out, eager = torch.empty_like(args[0]), torch.empty_like(args[0])
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            pool.extend_attention(0, *args, out=out)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert_attention_close(to_host(out), ref, "bf16")
            pool.extend_attention(0, *args, out=eager)
            assert_attention_close(to_host(eager), ref, "bf16")
        pool.check()


@pytest.mark.parametrize("shape", [(28, 4, 128, "bf16"), (12, 1, 64, "bf16"), (40, 2, 256, "bf16"), (18, 1, 32, "bf16"),
                                   (14, 2, 64, "f32"), (4, 4, 128, "f32"), (9, 1, 256, "f32"), (20, 2, 32, "f32")])
def test_extend_segments(shape):
    """Per-token decode segments, which the C ABI's FORCE_VALU flag selects at
    every head_dim (head_dim 32 has no other path), with groups of more than
    one chunk of 8 query heads."""
    Hq, Hkv, D, dt = shape
    ctx, nq = [1, 17, 40, 300, 97], [1, 17, 25, 64, 1]
    batch = wl.decode_batch_from_contexts([c - 1 for c in ctx], wl.SplitMix64(114), extra_blocks=2)
    desc = PoolDesc(1, Hkv, Hq, D, batch.num_blocks, dt)
    host = normal(115, desc.shape, dt)
    q_indptr = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    q = normal(116, (int(q_indptr[-1]), Hq, D), dt)
    with DeviceKvPool(desc) as pool:
        pool.write(host)
        qd = to_device(q)
        out = to_device(np.zeros_like(q))
        meta = [_i32(a) for a in (q_indptr, batch.block_indptr, batch.block_ids, batch.ctx_lens)]
        dp._raise(pool._lib.mkv_extend_attention(
            pool._h, 0, dp._dptr(qd), dp._dptr(out), *[dp._dptr(t) for t in meta], len(ctx), max(nq), max(ctx),
            float(np.float32(D ** -0.5)), dp.ATTN_FORCE_VALU, dp._stream_handle(None)))
        pool.check()
        got = to_host(out)
    ref = orc.extend_attention(odesc(desc), host, 0, widen(q), q_indptr, batch.block_indptr, batch.block_ids,
                               batch.ctx_lens)
    assert_attention_close(got, ref, dt)


@pytest.mark.parametrize("shape,num_seqs,chunk", [
    # the waves per workgroup and key-range splits that a device of 256 CUs
    # takes where the other tests' sizes take four waves
    ((14, 2, 64), 64, (48, 48)),    # 8 waves, unsplit
    ((16, 1, 64), 100, (5, 1000)),  # 8 waves, split
    ((8, 8, 128), 100, (20, 20)),   # 8 waves, unsplit
    ((16, 1, 128), 100, (5, 2500)), # 8 waves, split
    ((8, 4, 128), 48, (48, 48)),    # 16 waves, unsplit
    ((16, 1, 128), 48, (5, 1000)),  # 16 waves, split
])
def test_extend_row_tiles_in_wide_batches(shape, num_seqs, chunk):
    """Batches that fill the device: one chunk of the given new tokens and
    context among chunks of one to five tokens."""
    nq = [1 + b % min(5, chunk[0]) for b in range(num_seqs)]
    ctx = [n + 7 * b % 40 for b, n in enumerate(nq)]
    nq[num_seqs // 2], ctx[num_seqs // 2] = chunk
    got, ref, dec, q_indptr = _case(shape, ctx, nq, 117)
    assert_attention_close(got, ref, "bf16")
    assert_attention_close(dec, ref[q_indptr[1:] - 1], "bf16")
