"""Pages and cache rows written by the summary kernels (GPU): bit copies of
the prompt, zeros up to the whole block, nothing outside, and the summary's
own fields unchanged."""

import pytest
import torch

from refinekv import RefineKVConfig, build_summary
from refinekv.summary import _pages, store_and_build_summary

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
FIELDS = ("counts", "key_mean", "value_mean", "ellipsoid", "value_norm", "max_value_norm")

# dtype, dim, block, length: each kernel form (split blocks, one staged wave,
# the stream, the two-pass form) with a last block of one row, of all but one,
# of a whole number of 16-row chunks, and whole
CASES = [
    (torch.bfloat16, 128, 32, 32 * 9 + 1),
    (torch.bfloat16, 128, 64, 64 * 5 - 1),
    (torch.bfloat16, 96, 64, 64 * 3 + 16),
    (torch.float16, 64, 16, 16 * 21 + 7),
    (torch.bfloat16, 256, 16, 16 * 40 + 15),
    (torch.bfloat16, 256, 64, 64 * 4 + 33),
    (torch.float32, 128, 32, 32 * 3 + 17),
    (torch.float32, 256, 64, 64 * 2 + 1),
    (torch.bfloat16, 32, 16, 5),
    (torch.bfloat16, 128, 32, 32 * 6),
    # whole blocks that go out through registers: with dense keys and strided
    # values only the values' pages are written
    (torch.float32, 128, 32, 32 * 3),
    (torch.float32, 256, 64, 64 * 2),
    (torch.bfloat16, 256, 16, 16 * 9),
]


def bits(t):
    return t.contiguous().view(torch.uint8)


def prompt(dtype, dim, length, heads=3):
    gen = torch.Generator(device=DEV).manual_seed(dim * 7 + length)
    # the projection's layout: token stride heads * dim
    return [torch.randn(length, heads, dim, generator=gen, device=DEV).to(dtype).transpose(0, 1)
            for _ in range(2)]


@pytest.mark.parametrize("dtype,dim,block,length", CASES)
@pytest.mark.parametrize("layout", ["dense", "strided", "values strided"])
def test_build_summary_pages(dtype, dim, block, length, layout):
    keys, values = prompt(dtype, dim, length)
    if layout != "strided":
        keys = keys.contiguous()
    if layout == "dense":
        values = values.contiguous()
    cfg = RefineKVConfig(backend="hip", block_size=block)
    got = build_summary(keys, values, cfg)
    ref = build_summary(_pages(keys, block).flatten(1, 2)[:, :length], values.contiguous(), cfg)
    assert torch.equal(bits(got.keys), bits(_pages(keys, block)))
    assert torch.equal(bits(got.values), bits(_pages(values, block)))
    # whole blocks of dense rows stay views of the prompt
    assert (got.keys.data_ptr() == keys.data_ptr()) == (length % block == 0
                                                        and layout != "strided")
    for name in FIELDS:
        assert torch.equal(bits(getattr(got, name)), bits(getattr(ref, name))), name


@pytest.mark.parametrize("dtype,dim,block,length", CASES)
@pytest.mark.parametrize("extra", [0, 8, 4], ids=["dense", "16-byte rows", "odd rows"])
def test_store_pages_and_cache(dtype, dim, block, length, extra):
    """extra: elements between cache rows, so rows that are dense, on 16-byte
    boundaries but apart, and (2-byte types) on no 16-byte boundary."""
    keys, values = prompt(dtype, dim, length)
    rows = torch.full((2, 3, length + 70, dim + extra), -7.0, device=DEV, dtype=dtype)
    cache_k, cache_v = (rows[i, :, :length, :dim] for i in range(2))
    cfg = RefineKVConfig(backend="hip", block_size=block)
    got = store_and_build_summary(keys, values, cache_k, cache_v, cfg)
    for cache, source, pages in ((cache_k, keys, got.keys), (cache_v, values, got.values)):
        assert torch.equal(bits(cache), bits(source))
        assert torch.equal(bits(pages), bits(_pages(source, block)))
        assert (pages.data_ptr() == cache.data_ptr()) == (length % block == 0 and not extra)
    assert (rows[:, :, length:] == -7.0).all() and (rows[..., dim:] == -7.0).all()
    ref = build_summary(keys.contiguous(), values.contiguous(), cfg)
    for name in FIELDS:
        assert torch.equal(bits(getattr(got, name)), bits(getattr(ref, name))), name
