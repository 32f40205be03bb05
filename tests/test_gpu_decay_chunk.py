"""The recurrences with a decay in chunks of 64 tokens (csrc/decay_chunk.hip) against the recurrence token by token in 64 bits."""
import numpy as np
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


class _Step:
    def __init__(self, lens, starts):
        self.cu_tokens = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device="cuda")
        self.q_start = torch.tensor(starts, dtype=torch.int32, device="cuda")
        self.host_q_len, self.host_q_start, self.extra = list(lens), list(starts), {}
        self.max_q_len, self.max_kv_len = max(lens), max(a + b for a, b in zip(lens, starts))


def _recurrence(q, k, v, a, S):
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = S * a[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
        out[t] = (S * q[t][:, :, None]).sum(dim=1)
    return out, S


# whole chunks and parts of one, one token behind a chunk, entries too short for chunks between them, an entry that goes on
@pytest.mark.parametrize("lens, starts", [([64], [0]), ([65], [3]), ([1, 130, 5, 63, 64, 200], [0, 0, 9, 0, 70, 1]), ([127, 48], [0, 0])])
# every row of state there, some missing; columns: whole blocks of 32, odd ones, more than a workgroup's 128
@pytest.mark.parametrize("heads, dim, vdim", [(3, 64, 128), (2, 128, 64), (2, 37, 33), (1, 100, 161), (2, 5, 7)])
@pytest.mark.parametrize("kind", ["channel", "steep", "head", "rotated", "silu", "hgrn2"])
def test_chunks_against_the_recurrence(kind, heads, dim, vdim, lens, starts, monkeypatch):
    """Steep: decays down to 0, of which a logarithm or a quotient would make nothing.  32-bit sums of up to 64 + dim terms and chains of
    carried states: 2e-6 of the result is four times what is seen."""
    from ginfer_amd.kernels import ops
    for name in ("decay_chunk_from_few_rows", "decay_chunk_from", "decay_chunk_from_many_rows"):
        monkeypatch.setattr(ops.TUNING, name, 1)
    monkeypatch.setattr(ops.TUNING, "decay_chunk_few_rows_entries", 10 ** 6)
    monkeypatch.setattr(ops.TUNING, "decay_chunk_least", 48)
    g = torch.Generator().manual_seed(dim * 7 + len(lens))
    E, T, k0, v0 = len(lens), sum(lens), heads * dim, 2 * heads * dim
    proj = torch.randn((T, v0 + heads * vdim + (0 if kind == "hgrn2" else 3)), generator=g)
    q, k = (proj[:, i * k0:(i + 1) * k0].double().view(T, heads, dim) for i in (0, 1))
    v = proj[:, v0:v0 + heads * vdim].double().view(T, heads, vdim)
    state = torch.randn((E + 2, heads, dim, vdim), generator=g)
    slots = torch.randperm(E + 2, generator=g)[:E]
    step, kw, pos = _Step(lens, starts), {}, torch.cat([torch.arange(s, s + n) for n, s in zip(lens, starts)])
    hd = torch.linspace(0.8, 1.0, heads)
    a = hd.double()[None, :, None].expand(T, heads, dim)
    if kind in ("channel", "steep"):
        decay = torch.sigmoid(torch.randn((T, k0), generator=g) * 2) ** (1 / 16 if kind == "channel" else 30)
        if kind == "steep":
            decay[::5] = 0
        kw, a, q = dict(decay=decay.cuda(), q_scale=dim ** -0.5), decay.double().view(T, heads, dim), q * float(np.float32(dim ** -0.5))
    elif kind == "head":
        kw, k = dict(head_decay=hd.cuda(), k_scale=0.25), k * 0.25
    elif kind == "rotated":
        half = max(1, dim // 4)
        if 2 * half > dim:
            pytest.skip("no pair to turn")
        angles = torch.arange(step.max_kv_len)[:, None].double() * torch.linspace(1.0, 0.01, half).double()
        cos, sin = torch.cos(angles).float(), torch.sin(angles).float()
        kw = dict(head_decay=hd.cuda(), cos=cos.cuda().contiguous(), sin=sin.cuda().contiguous())

        def turned(x):
            c, s = cos.double()[pos][:, None], sin.double()[pos][:, None]
            lo, hi = x[..., :half], x[..., half:2 * half]
            return torch.cat([lo * c - hi * s, hi * c + lo * s, x[..., 2 * half:]], dim=-1)
        q, k = turned(q), turned(k)
    elif kind == "silu":
        kw, (q, k, v) = dict(head_decay=hd.cuda(), silu_inputs=True), (torch.nn.functional.silu(z) for z in (q, k, v))
    else:
        bias, lower = torch.randn(k0, generator=g) * 0.2, torch.rand(k0, generator=g)
        a = (lower.double() + (1 - lower.double()) * torch.sigmoid(proj[:, k0:v0].double() + bias.double())).view(T, heads, dim)
        q, k = torch.nn.functional.silu(q), 1 - a
    want, final, at = [], state.clone().double(), 0
    for e, (n, s) in enumerate(zip(lens, starts)):
        rows = slice(at, at + n)
        S = state[slots[e]].double() if s else torch.zeros((heads, dim, vdim), dtype=torch.float64)
        o, final[slots[e]] = _recurrence(q[rows], k[rows], v[rows], a[rows], S)
        want.append(o)
        at += n
    dev = state.cuda()
    if kind == "hgrn2":
        got = ops.hgrn2_scan(proj.cuda(), bias.cuda(), lower.cuda(), dev, slots.cuda(), step, heads, dim, vdim, chunked=True)
    else:
        got = ops.decay_scan(proj.cuda(), 0, k0, v0, dev, slots.cuda(), step, heads, dim, vdim, chunked=True, **kw)
    assert H.rel_err(got.cpu(), torch.cat(want)) < 2e-6
    assert H.rel_err(dev.cpu(), final) < 2e-6
    untouched = [i for i in range(E + 2) if i not in slots.tolist()]
    assert torch.equal(dev.cpu()[untouched], state[untouched])


def test_which_entries_go_in_chunks():
    from ginfer_amd.kernels import ops
    T = ops.TUNING
    assert ops.decay_in_chunks([T.decay_chunk_from], 64) == T.decay_chunk_least and ops.decay_in_chunks([T.decay_chunk_from - 1], 64) is None
    assert ops.decay_in_chunks([4096], ops.DECAY_CHUNK_MAX_DIM + 1) is None and ops.decay_in_chunks([], 64) is None
    assert ops.decay_in_chunks([700] * 7, 32) is None and ops.decay_in_chunks([700] * 7, 64) is not None

    def split(lens, chunked=True, extra=None, dim=64, vdim=128):
        step = _Step(lens, [0] * len(lens))
        step.extra = extra or {}
        return ops._decay_split(step, sum(lens), len(lens), 12, dim, vdim, chunked)
    assert split([2048]) == (None, 0, T.decay_chunk_least)                 # nothing to walk
    assert split([2048, 1, 1]) == (1, T.decay_chunk_least - 1, T.decay_chunk_least)
    for walked in (split([2048], chunked=False), split([2048], extra={"static_plan": {}}), split([100, 1]), split([2048], vdim=65537)):
        assert walked[1:] == (ops._ALL, None)
