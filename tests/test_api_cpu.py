"""Reference-API surface that needs no kernel: the baseline caches' legacy
converters, HeteroCache.clear_temp_kv_cache, and the refusals of
inputs that the prefill attention and the column sums do not take (CPU only)."""
import json
import os

import pytest
import torch

from heterocache_amd import kv_cluster, llama_model, ops, utils
from heterocache_amd.cache_utils import (BaseKVCache, CompressionCacheConfig, HeteroCache, HeteroCacheConfig,
                                         SnapKVCache)

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def _kv(seed, L):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(1, 4, L, 8, generator=g), torch.randn(1, 4, L, 8, generator=g)


def test_legacy_round_trip_keeps_the_pairs():
    """to_legacy_cache returns the per-layer pairs (heterocache/cache_utils.py:213-217);
    from_legacy_cache restores them unchanged, with layer 0's length as the
    token count (the pairs are already compressed: no second compression)."""
    pairs = tuple(_kv(s, 7 + s) for s in range(3))
    cache = SnapKVCache.from_legacy_cache(pairs, CompressionCacheConfig())
    assert isinstance(cache, SnapKVCache)
    assert cache.get_seq_length() == 7
    legacy = cache.to_legacy_cache()
    assert len(legacy) == 3
    for (k, v), (k2, v2) in zip(pairs, legacy):
        assert k2 is k and v2 is v
    base = BaseKVCache.from_legacy_cache(legacy)
    assert base.to_legacy_cache() == legacy
    assert BaseKVCache.from_legacy_cache(()).get_seq_length() == 0


def test_temp_cache_cleared_and_counted_back():
    """The baseline caches' temporary KV (update_global_past_kv=False) is
    appended behind the global cache and clear_temp_kv_cache takes its
    tokens back off the count (heterocache/cache_utils.py:178-233)."""
    cache = BaseKVCache.from_legacy_cache((_kv(0, 5),))
    cache._seen_tokens = 5
    k, v = _kv(1, 2)
    q = torch.zeros(1, 4, 2, 8)
    kk, vv = cache.update(k, v, 0, {"query_states": q, "num_key_value_groups": 1, "update_global_past_kv": False})
    assert kk.shape[2] == 7 and torch.equal(kk[:, :, 5:], k)
    assert cache.get_seq_length() == 7
    cache.clear_temp_kv_cache()
    assert cache.get_seq_length() == 5 and cache.temp_key_cache == []


def test_heterocache_clear_temp_kv_cache_is_a_no_op_when_empty():
    """heterocache/cache_utils.py:1192-1196 on a cache that never filled its
    temporary caches: the token count stays, the caches stay empty."""
    raw = json.load(open(os.path.join(GOLDEN, "head_analysis_llama-3.1-8b-instruct.json")))
    data = utils.augment_head_data(raw, [utils.head_permutation(r) for r in raw["classification_matrix"]])
    cache = HeteroCache(HeteroCacheConfig(data))
    cache._seen_tokens = 11
    cache.clear_temp_kv_cache()
    assert cache.get_seq_length() == 11
    assert cache.temp_key_cache == {} and cache.temp_value_cache == {}


def test_prefill_attention_refuses_padding_and_host_tensors():
    """No second code path: a padded mask, or tensors off the ROCm device,
    raise instead of falling back to another attention."""
    B, H, L, D = 2, 2, 6, 128
    q = torch.zeros(B, H, L, D)
    causal = torch.full((L, L), float("-inf")).triu(1)
    padded = causal.expand(B, 1, L, L).clone()
    padded[1, :, :, :2] = float("-inf")  # left padding of the second row
    with pytest.raises(NotImplementedError, match="padding"):
        llama_model.prefill_attention(q, q, q, padded, 1.0)
    with pytest.raises(NotImplementedError, match="ROCm device"):
        llama_model.prefill_attention(q, q, q, causal.expand(B, 1, L, L), 1.0)
    with pytest.raises(NotImplementedError, match="ROCm device"):
        llama_model.prefill_attention(q, q, q, None, 1.0)


@pytest.mark.parametrize("q,k", [
    ((1, 8, 40, 128), (1, 2, 40, 128)),    # GQA keys, not repeated per query head
    ((2, 4, 40, 128), (1, 4, 40, 128)),    # a batch too few
    ((1, 4, 40, 128), (1, 4, 39, 128)),    # a token too few
    ((1, 4, 40, 128), (1, 5, 40, 128)),
    ((1, 4, 40, 64), (1, 4, 40, 64)),      # head_dim
    ((1, 4, 40, 128), (1, 4, 40, 64)),
    ((4, 40, 128), (4, 40, 128))])
def test_column_sums_refuse_shapes_they_would_read_past(q, k):
    """Keys that do not cover the queries' batches, heads and tokens, or rows
    of another head_dim, are refused before any device work."""
    q, k = torch.zeros(q), torch.zeros(k)
    with pytest.raises(ValueError, match=r"must be \[B, H, L, 128\]|must hold the batches and heads"):
        ops.attn_column_sums(q, k, 0.1)
    if q.dim() == 4 and k.shape[1] <= q.shape[1]:
        with pytest.raises(ValueError, match=r"must be \[B, H, L, 128\]|must hold the batches and heads"):
            kv_cluster.H2OKVCluster().heavy_hitter_scores(k, q)
