"""Products of 257 to 512 rows by few columns, whose parts of K the consumer adds: over tiles dealt evenly to the chip."""
import pytest
import torch


def _choice(rows, out_features, in_features):
    from ginfer_amd.parts.linear import linear_choice
    return linear_choice(rows, out_features, in_features, False, False, True, False, True)


def test_which_products_of_few_columns_are_dealt_evenly():
    from ginfer_amd.kernels.tuning import TUNING as T
    N, most = T.spread_parts_few_columns, T.spread_parts_few_columns_most_rows
    assert _choice(257, 1536, 1536)[0] == _choice(most, 1536, 1536)[0] == _choice(385, 896, 4864)[0] == "tiles"
    assert _choice(most + 1, 1536, 1536)[0] == "library"
    assert _choice(320, N, 2048)[0] == "tiles" and _choice(320, N + 16, 2048) == ("library", 1)       # a short K of more columns
    K = T.spread_parts_few_columns_weights // N
    assert _choice(400, N, K - 64)[0] == "tiles" and _choice(400, N, K)[0] == "library" and _choice(384, N, K)[0] == "tiles"


@pytest.mark.gpu
# the fewest and the most rows, around a row tile's edge; few columns, a number that makes no whole groups, the most; K with and without a
# rest of 64 behind its slabs of 128
@pytest.mark.parametrize("rows", [257, 320, 383, 385, 449, 512])
@pytest.mark.parametrize("out_features, in_features", [(16, 1024), (784, 1152), (1536, 1536), (1792, 1856), (2048, 2048), (896, 4864)])
def test_sums_of_products_of_few_columns(rows, out_features, in_features):
    """A chain of in_features 32-bit sums, in parts: the first order of its bound."""
    from ginfer_amd.parts.linear import linear
    g = torch.Generator().manual_seed(rows)
    a, w = (torch.randn(s, generator=g).bfloat16().cuda() for s in ((rows, in_features), (out_features, in_features)))
    plan = _choice(rows, out_features, in_features)
    got = linear(a, w, None, parts_ok=True)
    assert plan[0] == "tiles" and got.shape == (plan[2], rows, out_features) and got.dtype == torch.float32
    want = a.double() @ w.double().t()
    bound = (in_features + 8) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t()) * 1.01
    assert bool(((got.double().sum(dim=0) - want).abs() <= bound).all())
