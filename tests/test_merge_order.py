"""The merge's fixed order (GPU): the bf16 outputs of the dense decode and of
the three-kernel decode equal, bit for bit, an fp32 fold of the partials that
the call left in its workspace -- stripe k takes partials k, k + K, ... one
after another, the stripes follow in order -- at the partial counts where its
stripes, batches and forms (K 8 up to 128 partials, 32 above) change.  The
values' sign turns halfway, so the partials cancel and sums in another order
give other bf16 values in most elements.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
NEG = float("-inf")


@pytest.fixture(scope="module")
def hip():
    if not torch.cuda.is_available():
        pytest.skip("no GPU in this environment")
    from refinekv import _hip

    _hip.lib()
    return _hip


def _fma(a, b, c):
    return (a.double() * b.double() + c.double()).float()


def _merge_one(hip, part, state):
    """(m, l (R), acc (R, D)) merged into (mx, den, num)."""
    m, l, acc = part
    mx, den, num = state
    live, up = l > 0, (l > 0) & (m > mx)
    w = hip.math_probe("exp_hw", torch.where(up, mx - m, m - mx))

    def one(x, s, w, up, live):
        return torch.where(live, torch.where(up, s * w + x, _fma(x, w, s)), s)

    return (torch.where(up, m, mx), one(l, den, w, up, live),
            one(acc, num, w[:, None], up[:, None], live[:, None]))


def _empty(rows, dim):
    return (torch.full((rows,), NEG, device="cuda"), torch.zeros(rows, device="cuda"),
            torch.zeros(rows, dim, device="cuda"))


def _merged(hip, ml, acc):
    """ml (R, P, 2), acc (R, P, D) -> bf16 (R, D)."""
    rows, parts, dim = acc.shape
    stripes = 8 if parts <= 128 else 32
    total = _empty(rows, dim)
    for k in range(min(stripes, parts)):
        state = _empty(rows, dim)
        for i in range(k, parts, stripes):
            state = _merge_one(hip, (ml[:, i, 0], ml[:, i, 1], acc[:, i]), state)
        total = _merge_one(hip, (state[0], state[1], state[2]), total)
    _, den, num = total
    return (num.double() / den.clamp_min(1e-30)[:, None].double()).float().bfloat16()


def _inputs(heads, group, tokens, dim):
    gen = torch.Generator("cuda").manual_seed(tokens + dim)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    values = rand(heads, tokens, dim) + 8
    values[:, tokens // 2:] -= 16
    return (rand(heads, group, dim).bfloat16(), rand(heads, tokens, dim).bfloat16(),
            values.bfloat16())


@pytest.mark.parametrize("heads,group,dim,tokens", [
    (8, 4, 128, 65573), (1, 16, 32, 40000), (2, 3, 96, 1000), (1, 1, 64, 17),
])
def test_dense_outputs_are_the_ordered_fold(hip, heads, group, dim, tokens):
    query, keys, values = _inputs(heads, group, tokens, dim)
    workspace = {}
    out = hip.dense_decode(query, keys, values, workspace=workspace)
    splits, _ = hip.dense_plan(heads, group, dim, tokens)
    rows = heads * group
    raw = workspace["hip_dense_scratch"]
    first = rows * splits * 8
    acc_at = -(-first // 256) * 256
    ml = raw[:first].view(torch.float32).view(rows, splits, 2)
    acc = raw[acc_at:acc_at + rows * splits * dim * 4].view(torch.float32)
    assert torch.equal(out.view(rows, dim), _merged(hip, ml, acc.view(rows, splits, dim)))


@pytest.mark.parametrize("heads,group,dim,tiles", [
    (2, 4, 128, 1), (1, 4, 64, 64), (1, 3, 96, 128), (1, 4, 128, 129), (1, 2, 32, 513),
    (1, 2, 256, 5),
])
def test_three_kernel_outputs_are_the_ordered_fold(hip, heads, group, dim, tiles):
    from refinekv import RefineKVConfig, build_summary, sparse_attention

    blocks = tiles * 64 - 3
    query, keys, values = _inputs(heads, group, blocks * 16 + 9, dim)
    tokens = blocks * 16
    config = RefineKVConfig(backend="hip", block_size=16, eps=0.05)
    workspace = {}
    hip.set_decode_path("split")
    try:
        summary = build_summary(keys[:, :tokens], values[:, :tokens], config)
        out = sparse_attention(query.unsqueeze(2), summary, keys[:, tokens:], values[:, tokens:],
                               config, workspace=workspace).output
    finally:
        hip.set_decode_path("step")
    at = hip.workspace_layout(heads, group, dim, blocks)
    assert at["n_tiles"] == tiles
    rows, stride = heads * group, at["tile_stride"]
    raw = workspace["hip_scratch"]
    ml = raw[at["part_ml"]:][:rows * stride * 8].view(torch.float32).view(rows, stride, 2)
    acc = raw[at["part_acc"]:][:rows * stride * dim * 4].view(torch.float32)
    want = _merged(hip, ml[:, :tiles], acc.view(rows, stride, dim)[:, :tiles])
    assert torch.equal(out.view(rows, dim), want)
