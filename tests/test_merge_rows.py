"""The merge of a row's partials and the attention of tiles by the three
kernels (GPU), at the partial counts where the merge's stripes, batches and
forms change: one partial, one past a batch of the 32-column form (64), its
last count and the first of the 8-column form (128, 129), one past that
form's batch (512) and a ragged last tile.

Bar: every element within 2^-8 of itself (bf16's rounding is 2^-9) plus
1e-4: the weights reach the matrix cores as two bf16 halves (2^-17 of values
below 6) and fp32 sums add less.  eps 0 expands every block, so the result is
attention over all tokens; an eps above any risk expands none, so it is
attention over the block means with log counts.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    if not torch.cuda.is_available():
        pytest.skip("no GPU in this environment")
    from refinekv import _hip

    _hip.lib()
    return _hip


def _check(got, want):
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2 ** -8 + 1e-4).all()), f"max-abs {float(err.max()):.3e}"


@pytest.mark.parametrize("heads,group,dim,blocks,last,suffix", [
    (2, 4, 128, 1, 16, 3), (2, 4, 128, 65, 5, 1), (1, 3, 96, 64 * 64 + 1, 16, 70),
    (2, 4, 128, 128 * 64, 16, 33), (1, 4, 64, 128 * 64 + 7, 9, 1), (1, 2, 32, 512 * 64 + 1, 3, 5),
    (1, 8, 128, 129 * 64, 3, 200), (1, 16, 64, 130, 16, 17), (1, 5, 160, 131, 2, 40),
    (1, 8, 256, 129, 16, 9),
])
@pytest.mark.parametrize("expand", [True, False])
def test_three_kernels_match_attention(hip, heads, group, dim, blocks, last, suffix, expand):
    from refinekv import RefineKVConfig, build_summary, sparse_attention

    gen = torch.Generator("cuda").manual_seed(blocks * 31 + dim)
    tokens = 16 * (blocks - 1) + last
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    query = rand(heads, group, 1, dim)
    keys, values = rand(heads, tokens + suffix, dim), rand(heads, tokens + suffix, dim)
    config = RefineKVConfig(backend="hip", block_size=16, eps=0.0 if expand else 1e30)
    hip.set_decode_path("split")
    try:
        summary = build_summary(keys[:, :tokens], values[:, :tokens], config)
        result = sparse_attention(query, summary, keys[:, tokens:], values[:, tokens:], config,
                                  return_selected=True)
    finally:
        hip.set_decode_path("step")
    assert bool(result.selected.all()) if expand else not bool(result.selected.any())
    scale = dim ** -0.5
    for h in range(heads):
        q = query[h, :, 0].double()
        k, v = keys[h].double(), values[h].double()
        logits = q @ k.T.contiguous() * scale
        if not expand:
            mean = summary.key_mean[h].double()
            z = q @ mean.T.contiguous() * scale + summary.counts.double().log()
            logits = torch.cat([z, logits[:, tokens:]], -1)
            v = torch.cat([summary.value_mean[h].double(), v[tokens:]])
        _check(result.output.view(heads, group, dim)[h], logits.softmax(-1) @ v)


@pytest.mark.parametrize("tokens", [1, 17, 4096, 40000])
def test_dense_splits_match_attention(hip, tokens):
    gen = torch.Generator("cuda").manual_seed(tokens)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    query, keys, values = rand(1, 4, 96), rand(1, tokens, 96), rand(1, tokens, 96)
    out = hip.dense_decode(query, keys, values, length=tokens, workspace={})
    logits = query[0].double() @ keys[0].double().T.contiguous() / math.sqrt(96)
    _check(out.view(4, 96), logits.softmax(-1) @ values[0].double())


@pytest.mark.parametrize("path", ["split", "step"])
@pytest.mark.parametrize("what", ["suffix key", "query", "every suffix key"])
@pytest.mark.parametrize("dim", [128, 256])
def test_nan_reaches_the_output(hip, path, what, dim):
    """A row whose logits hold a NaN comes out NaN, as softmax gives it (its
    partial is not an empty one), and no row of another head; with three
    kernels no other row at all."""
    from refinekv import RefineKVConfig, build_summary, sparse_attention

    gen = torch.Generator("cuda").manual_seed(dim)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    heads, group, tokens, suffix = 2, 3, 1000, 33
    query = rand(heads, group, 1, dim)
    keys, values = rand(heads, tokens + suffix, dim), rand(heads, tokens + suffix, dim)
    nan = torch.zeros(heads, group, dtype=torch.bool, device="cuda")
    config = RefineKVConfig(backend="hip", eps=0.05)
    summary = build_summary(keys[:, :tokens], values[:, :tokens], config)
    if what == "query":
        query[1, 2, 0, 5] = float("nan")
        nan[1, 2] = True
    else:
        keys[1, tokens + 20 if what == "suffix key" else slice(tokens, None), 7] = float("nan")
        nan[1] = True
    hip.set_decode_path(path)
    try:
        out = sparse_attention(query, summary, keys[:, tokens:], values[:, tokens:],
                               config).output
    finally:
        hip.set_decode_path("step")
    got = out.isnan().view(heads, group, dim)
    assert bool(got[nan].all()) and not bool(got[0].any())
    if path == "split":
        assert not bool(got[~nan].any())


@pytest.mark.parametrize("what", ["key", "query", "every key"])
def test_nan_reaches_the_dense_output(hip, what):
    gen = torch.Generator("cuda").manual_seed(1)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    query, keys, values = rand(2, 4, 64), rand(2, 5000, 64), rand(2, 5000, 64)
    nan = torch.zeros(2, 4, dtype=torch.bool, device="cuda")
    if what == "query":
        query[1, 3, 9] = float("nan")
        nan[1, 3] = True
    else:
        keys[0, 4321 if what == "key" else slice(None), 0] = float("nan")
        nan[0] = True
    out = hip.dense_decode(query, keys, values, workspace={})
    assert torch.equal(out.isnan(), nan[..., None].expand(-1, -1, 64))
