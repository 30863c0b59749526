"""The batched anchor selection against one select_blocks per anchor (GPU):
row counts at the edges of its four-row steps and of its cuts of a head's
rows, queries in several memory orders, every reduction, and queries and
summaries with values that are not finite."""

import pytest
import torch

from refinekv import RefineKVConfig, build_summary, select_blocks, select_blocks_union, testing

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")

# heads, group, dim, block, prompt, anchors
CASES = [
    (2, 1, 128, 32, 2048, 1),
    (2, 3, 64, 32, 2050, 3),       # 9 rows: a last step of one row
    (3, 7, 128, 64, 4096 + 5, 33),  # anchors that straddle the four-row steps
    (8, 4, 128, 32, 9000, 64),     # several cuts of a head's rows
    (1, 16, 32, 16, 1000, 20),
    (2, 5, 96, 16, 1040, 17),
    (2, 2, 160, 32, 700, 6),       # two words per thread
    (2, 3, 256, 64, 999, 9),
    (40, 4, 64, 16, 2100, 2),      # many heads of few tiles
    (2100, 1, 32, 16, 100, 9),     # more (tile, head) cells than resident workgroups
    (1, 4, 128, 16, 70000, 5),     # 69 tiles
]


def inputs(heads, group, dim, block, prompt, anchors):
    inp = testing.decode_inputs(heads=heads, group=group, dim=dim, prompt=prompt, suffix=0,
                                block=block, spike_fraction=0.05, anchors=anchors, seed=dim + anchors)
    return (inp["prompt_keys"].bfloat16().to(DEV), inp["prompt_values"].bfloat16().to(DEV),
            inp["anchor_queries"].bfloat16().to(DEV))


def union(queries, summary, cfg):
    masks = [select_blocks(queries[:, :, a:a + 1], summary, cfg, workspace={})
             for a in range(queries.shape[2])]
    return torch.stack(masks).any(0)


@pytest.mark.parametrize("heads,group,dim,block,prompt,anchors", CASES)
@pytest.mark.parametrize("reduction", ["any", "max", "mean"])
def test_union_equals_select_per_anchor(heads, group, dim, block, prompt, anchors, reduction):
    keys, values, queries = inputs(heads, group, dim, block, prompt, anchors)
    ws = {}
    for eps in (0.05, 0.0, 1e6):
        cfg = RefineKVConfig(backend="hip", block_size=block, eps=eps, gqa_reduction=reduction)
        summary = build_summary(keys, values, cfg)
        want = union(queries, summary, cfg)
        orders = {
            "(H, G, A, D)": queries,
            "(A, H, G, D)": queries.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3),
            "(A, D) rows apart": torch.cat([queries, queries[..., :8]], -1)[..., :dim],
            "odd rows": torch.cat([queries, queries[..., :1]], -1)[..., :dim],
        }
        for name, q in orders.items():
            assert torch.equal(q, queries)
            got = select_blocks_union(q, summary, cfg, workspace=ws)
            assert torch.equal(got, want), (name, eps)


@pytest.mark.parametrize("heads,group,anchors", [(8, 4, 1), (4, 1, 20), (1, 3, 5), (1, 1, 1)])
def test_axes_of_length_one_may_have_any_stride(heads, group, anchors):
    """The stride of a length-one axis says nothing: is_contiguous() ignores
    it, and views carry odd values there."""
    keys, values, queries = inputs(heads, group, 64, 32, 1000, anchors)
    cfg = RefineKVConfig(backend="hip", eps=0.05)
    summary = build_summary(keys, values, cfg)
    shape = queries.shape
    strides = [1 if n == 1 else s for n, s in zip(shape, queries.stride())]
    view = queries.as_strided(shape, strides)
    assert view.is_contiguous() and torch.equal(view, queries)
    assert torch.equal(select_blocks_union(view, summary, cfg, workspace={}),
                       union(queries, summary, cfg))
    # a column of a wider tensor
    wide = torch.cat([queries, queries[..., :1]], -1)[..., :64]
    assert torch.equal(select_blocks_union(wide, summary, cfg, workspace={}),
                       union(queries, summary, cfg))


@pytest.mark.parametrize("reduction", ["any", "max", "mean"])
@pytest.mark.parametrize("what", ["inf query", "nan query", "zero query", "nan block", "huge"])
def test_union_with_values_that_are_not_finite(what, reduction):
    keys, values, queries = inputs(2, 4, 128, 32, 3000, 6)
    if what == "inf query":
        queries[0, 2, 3, 5] = float("inf")
    elif what == "nan query":
        queries[1, 0, 5] = float("nan")
    elif what == "zero query":
        queries[:, :, 2:] = 0
    elif what == "nan block":
        keys[1, 70, 3] = float("nan")
    else:
        queries *= 1e19
        keys *= 1e19
    cfg = RefineKVConfig(backend="hip", eps=0.02, gqa_reduction=reduction)
    summary = build_summary(keys, values, cfg)
    assert torch.equal(select_blocks_union(queries, summary, cfg, workspace={}),
                       union(queries, summary, cfg))
