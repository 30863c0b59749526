"""The C entries that the Python package does not call itself (GPU): the
summary with the cache write and no pages, and the anchors' mask of dense
(anchors, heads, group, dim) queries, against the entries it does call."""

import pytest
import torch

from refinekv import RefineKVConfig, build_summary, select_blocks_union

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
FIELDS = ("counts", "key_mean", "value_mean", "ellipsoid", "value_norm", "max_value_norm")


@pytest.fixture(scope="module")
def hip():
    if not torch.cuda.is_available():
        pytest.skip("no GPU in this environment")
    from refinekv import _hip

    _hip.lib()
    return _hip


def bits(t):
    return t.contiguous().view(torch.uint8)


@pytest.mark.parametrize("dtype,dim,block,length", [
    (torch.bfloat16, 128, 32, 32 * 5 + 1), (torch.float16, 64, 16, 16 * 9),
    (torch.float32, 256, 64, 64 * 2 + 17), (torch.bfloat16, 256, 16, 16 * 7 + 15),
])
def test_summary_store(hip, dtype, dim, block, length):
    gen = torch.Generator(device=DEV).manual_seed(length)
    keys, values = (torch.randn(3, length, dim, generator=gen, device=DEV).to(dtype)
                    for _ in range(2))
    want = build_summary(keys, values, RefineKVConfig(backend="hip", block_size=block))
    got = [torch.empty_like(getattr(want, name)) for name in FIELDS]
    rows = torch.full((2, 3, length + 70, dim), -7.0, device=DEV, dtype=dtype)
    cache = [rows[0, :, :length], rows[1, :, :length]]
    args = [x for t in (keys, values) for x in (hip._ptr(t), t.stride(0), t.stride(1))]
    args += [hip.DTYPE_CODES[dtype], 3, length, dim, block]
    args += [x for t in cache for x in (hip._ptr(t), t.stride(0), t.stride(1))]
    rc = hip.lib().rkv_summary_store(*args, *(hip._ptr(t) for t in got), hip._stream(DEV))
    hip._check(rc, "rkv_summary_store")
    for name, field in zip(FIELDS, got):
        assert torch.equal(bits(field), bits(getattr(want, name))), name
    assert torch.equal(bits(cache[0]), bits(keys)) and torch.equal(bits(cache[1]), bits(values))
    assert (rows[:, :, length:] == -7.0).all()


@pytest.mark.parametrize("heads,group,dim,block,length,anchors", [
    (2, 4, 128, 32, 3000, 6), (3, 1, 64, 16, 1100, 1), (1, 7, 256, 64, 700, 9),
])
def test_select_anchors(hip, heads, group, dim, block, length, anchors):
    gen = torch.Generator(device=DEV).manual_seed(length)
    rand = lambda *s: torch.randn(s, generator=gen, device=DEV).bfloat16()  # noqa: E731
    queries = rand(anchors, heads, group, dim)
    cfg = RefineKVConfig(backend="hip", block_size=block)
    summary = build_summary(rand(heads, length, dim), rand(heads, length, dim), cfg)
    blocks = summary.num_blocks
    # an eps that about half of the blocks pass for some anchor
    risk = torch.empty(anchors, heads, group, blocks, device=DEV)
    for a in range(anchors):
        hip.select(queries[a].unsqueeze(2), summary, cfg, risk_out=risk[a])
    eps = float(risk.amax((0, 2)).median())
    cfg = RefineKVConfig(backend="hip", block_size=block, eps=eps)
    scratch = torch.empty(hip.workspace_bytes(heads * anchors, group, dim, blocks), device=DEV,
                          dtype=torch.uint8)
    mask = torch.empty(heads, blocks, device=DEV, dtype=torch.bool)
    rc = hip.lib().rkv_select_anchors(
        hip._ptr(queries), *hip._summary_args(summary), heads, group, dim, blocks, block, length,
        cfg.eps, hip.REDUCTION_CODES[cfg.gqa_reduction], anchors, hip._ptr(mask),
        hip._ptr(scratch), scratch.numel(), hip._stream(DEV))
    hip._check(rc, "rkv_select_anchors")
    want = select_blocks_union(queries.permute(1, 2, 0, 3), summary, cfg, workspace={})
    assert torch.equal(mask, want)
    assert bool(want.any()) and not bool(want.all())
