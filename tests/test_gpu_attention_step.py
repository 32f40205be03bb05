"""Single tokens and rows of prompt portions in one launch (attn_step_kernel of csrc/attention_mfma.hip) against the attention in 32-bit."""
import math

import pytest
import torch

from test_gpu_kernels import _paged_case, _Step, close, rnd

pytestmark = pytest.mark.gpu

# one of either; fewer workgroups of tokens than of tiles and the other way round, neither a multiple of eight; contexts around a tile of
# every wavefront (256 keys of eight), one far beyond
STEPS = [[(1, 1), (2, 2)], [(1, 33), (150, 150), (1, 700)], [(1, n) for n in (1, 31, 32, 33, 159, 160, 161, 255, 256, 257, 289, 1500)] + [(3, 40), (17, 100)]]


@pytest.mark.parametrize("wide", [False, True])
# workgroups of 8, 5 to 7 and again 8 wavefronts; with the prompts' operands through LDS (fill 1) and straight from memory
@pytest.mark.parametrize("nh,nkv,hd", [(12, 2, 128), (28, 4, 128), (4, 1, 128), (5, 1, 64), (6, 1, 256), (12, 2, 48), (40, 2, 64), (3, 3, 80)])
@pytest.mark.parametrize("fill", [1, 256])
@pytest.mark.parametrize("keys, window", [(1024, None), (1 << 20, None), (0, None), (0, 70)])     # the most in one split
@pytest.mark.parametrize("seqs", STEPS)
def test_tokens_beside_prompts(nh, nkv, hd, fill, keys, window, wide, seqs, monkeypatch):
    from ginfer_amd.kernels import ops
    monkeypatch.setattr(ops.TUNING, "prefill_wide_tiles_from", 0 if wide else 1 << 30)
    monkeypatch.setattr(ops.TUNING, "prefill_fill_workgroups", fill)
    monkeypatch.setattr(ops.TUNING, "decode_beside_unsplit_keys", keys)
    if not keys:
        monkeypatch.setattr(ops.TUNING, "decode_target_workgroups", 1 << 20)
        monkeypatch.setattr(ops.TUNING, "decode_min_split_keys", 32)
    a, ref, _ = _paged_case(seqs, nh, nkv, hd, 16, torch.bfloat16, seed=hd + nh, window=window)
    out = ops.paged_attention_mfma(a["q"], a["k_pages"], a["v_pages"], a["block_table"], _Step(seqs, a), nh, nkv, hd, 1.0 / math.sqrt(hd), window=window)
    close(out, ref, 2e-2)


@pytest.mark.parametrize("keys", [1 << 20, 0])
def test_tokens_beside_prompts_with_sinks_and_gates_as_apart(keys, monkeypatch):
    """As the two launches give it: weights rounded to bfloat16 against other running maxima, 2^-9 of each on either side, so 2^-8 of the
    attention over the values' magnitudes, and the results' own roundings and denominators, 2^-7 of the result."""
    from ginfer_amd.kernels import ops
    seqs = STEPS[2]
    a, _, _ = _paged_case(seqs, 12, 2, 128, 16, torch.bfloat16, seed=5)
    T = a["q"].shape[0]
    more = dict(sinks=rnd((12,), torch.float32, 8), gate=rnd((T, 12), torch.float32, 9), gate_scale=2.0)
    monkeypatch.setattr(ops.TUNING, "decode_beside_unsplit_keys", keys)

    def run(order, v_pages):
        at, rows, tables = 0, [], []
        for e, (n, kv) in enumerate(seqs):
            if e in order:
                rows += range(at, at + n)
                tables.append(e)
            at += n
        idx = torch.tensor(rows, device="cuda")
        part = {k: a[k][idx] for k in ("q", "positions")}
        part["token_entry"] = torch.tensor([i for i, e in enumerate(tables) for _ in range(seqs[e][0])], dtype=torch.int32, device="cuda")
        out = ops.paged_attention_mfma(part["q"], a["k_pages"], v_pages, a["block_table"][tables].contiguous(), _Step([seqs[e] for e in tables], part),
                                       12, 2, 128, 128 ** -0.5, sinks=more["sinks"], gate=more["gate"][idx].contiguous(), gate_scale=2.0)
        return idx, out.float()
    _, both = run(range(len(seqs)), a["v_pages"])
    for kind in (0, 1):
        entries = [e for e, (n, _) in enumerate(seqs) if (n > 1) == bool(kind)]
        idx, apart = run(entries, a["v_pages"])
        assert bool(((both[idx] - apart).abs() <= 2.0 ** -8 * 1.01 * run(entries, a["v_pages"].abs())[1] + 2.0 ** -7 * apart.abs()).all())
