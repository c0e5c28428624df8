"""ops.attn_column_sums (the heavy-hitter sums of H2O) vs the float64 oracle,
at the edges of its 64-row sets, 128- and 256-column blocks and row splits.

Tolerance: the inputs are exact in float32, logits reach |x| <= 64 and round
to 2^-18 in each of the few operations on them (product sums, scaling,
log-sum-exp), so a probability is off by under 64 * 2^-18 / 2 = 1.3e-4 at the
very worst and a sum of them by less; 1e-4 of the largest sum bounds it.
"""
import math

import numpy as np
import pytest
import torch

from heterocache_amd import kv_cluster, ops
from oracle import hc_oracle as O
from tests.gpu_util import as_np

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128)


def _check(q, k):
    got = as_np(ops.attn_column_sums(q, k, SCALE)).reshape(q.shape[:3])
    ref = O.h2o_scores(as_np(q), as_np(k))
    assert np.max(np.abs(got - ref)) < 1e-4 * max(1.0, float(ref.max()))
    assert np.allclose(got.sum(-1), q.shape[2], rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("L", [1, 15, 63, 64, 65, 127, 129, 255, 256, 257, 1100])
def test_sizes(dev, dtype, L):
    print(f"column sums L={L} {dtype}", flush=True)
    g = torch.Generator().manual_seed(L)
    q = torch.randn(2, L, 3, 128, generator=g).to(dtype).to(dev).transpose(1, 2)  # token-major rows
    k = torch.randn(2, 3, L, 128, generator=g)
    k[..., :4] *= 4
    _check(q, k.to(dtype).to(dev))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_growing_maxima(dev, dtype):
    """Keys whose logits grow along the prompt, so the row reference moves
    often, and one row whose largest logit comes last."""
    L = 700
    g = torch.Generator().manual_seed(3)
    q = torch.randn(1, 2, L, 128, generator=g)
    k = 0.1 * torch.randn(1, 2, L, 128, generator=g)
    k += torch.linspace(0.0, 4.0, L)[:, None] * q[:, :, 5:6] / 12
    q[:, :, 7] = 5 * k[:, :, -1] / k[:, :, -1].norm(dim=-1, keepdim=True)
    _check(q.to(dtype).to(dev), k.to(dtype).to(dev))


def test_layouts_that_are_copied(dev):
    """A base off 16 bytes and a token stride off 16 bytes (queries)."""
    L = 200
    g = torch.Generator().manual_seed(4)
    flat = torch.randn(1 + 2 * L * 128, generator=g).half().to(dev)
    k = flat[1:].view(1, 2, L, 128)
    q = torch.randn(1, 2, L, 131, generator=g).half().to(dev)[..., :128]
    _check(q, k)
    with pytest.raises(ValueError):
        ops.attn_column_sums(q, q, SCALE)  # keys: token stride not a multiple of 8


def test_longer_and_wider_keys(dev):
    """Keys of more tokens than the queries count up to the queries' length;
    the cluster takes the first heads of keys that have more of them."""
    L = 100
    g = torch.Generator().manual_seed(7)
    q = torch.randn(2, 3, L, 128, generator=g).half().to(dev)
    k = torch.randn(3, 5, L + 30, 128, generator=g).half().to(dev)
    want = ops.attn_column_sums(q, k[:2, :3, :L].contiguous(), SCALE)
    assert torch.equal(ops.attn_column_sums(q, k[:2, :3], SCALE), want)
    assert torch.equal(kv_cluster.H2OKVCluster().heavy_hitter_scores(k, q), want)


def test_token_stride_past_32_bit_offsets(dev):
    """64 token strides of 2^31 bytes or more: copied first."""
    g = torch.Generator().manual_seed(8)
    flat = torch.zeros(2 * (1 << 24) + 128, dtype=torch.float16, device=dev)
    k = flat.as_strided((1, 1, 3, 128), (0, 0, 1 << 24, 1))
    k.copy_(torch.randn(1, 1, 3, 128, generator=g))
    q = torch.randn(1, 1, 3, 128, generator=g).half().to(dev)
    _check(q, k)
    assert torch.equal(ops.attn_column_sums(k, q, SCALE), ops.attn_column_sums(k.contiguous(), q, SCALE))


def test_copies_run_on_the_given_stream(dev):
    """Keys off 16 bytes, written on the call's stream behind a queue of other
    work: the copy that aligns them waits for them."""
    L = 200
    g = torch.Generator().manual_seed(9)
    flat = torch.zeros(1 + 2 * L * 128, dtype=torch.float16, device=dev)
    k = flat[1:].view(1, 2, L, 128)
    src = torch.randn(1, 2, L, 128, generator=g).half().to(dev)
    q = torch.randn(1, 2, L, 128, generator=g).half().to(dev)
    big = torch.randn(4096, 4096, device=dev)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for _ in range(20):
            big = big @ big * 1e-4
        k.copy_(src)
    got = ops.attn_column_sums(q, k, SCALE, stream=s)
    s.synchronize()
    assert torch.equal(got, ops.attn_column_sums(q, src, SCALE))


def test_infinite_and_nan_rows(dev):
    """A NaN query makes its softmax NaN, and so every sum of its head; a key
    that all queries of a head score -inf takes no probability."""
    L = 150
    g = torch.Generator().manual_seed(5)
    q = torch.rand(1, 2, L, 128, generator=g).half() + 0.1
    k = torch.randn(1, 2, L, 128, generator=g).half()
    k[0, 1, 40, 3] = -math.inf
    q[0, 0, 70, 0] = math.nan
    got = as_np(ops.attn_column_sums(q.to(dev), k.to(dev), SCALE))
    assert np.isnan(got[0]).all()
    ref = O.h2o_scores(as_np(q), as_np(k))[0, 1]
    assert got[1, 40] == 0 and np.allclose(got[1], ref, atol=1e-4)


def test_replayed_graph(dev):
    L = 500
    g = torch.Generator().manual_seed(6)
    q, k = (torch.randn(1, 4, L, 128, generator=g).half().to(dev) for _ in range(2))
    out = torch.empty((4, L), dtype=torch.float32, device=dev)
    ops.attn_column_sums(q, k, SCALE, out=out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.attn_column_sums(q, k, SCALE, out=out)
    for i in range(4):
        q.copy_(torch.randn(q.shape, generator=g))
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.attn_column_sums(q, k, SCALE))
