"""How a step is laid into the padded sizes of a recorded step (host arrays only: no GPU)."""
import numpy as np
import pytest

from ginfer_amd.engine.runner import ModelRunner, pad_step, single_records
from ginfer_amd.kernels import ops


def host_arrays(q_len, q_start, page=8, want_last=True):
    """What ModelRunner._host_arrays makes for entries of these lengths, one cache group, pages numbered from 1."""
    q_len, q_start = np.asarray(q_len, dtype=np.int64), np.asarray(q_start, dtype=np.int64)
    E, T = len(q_len), int(q_len.sum())
    cu = np.zeros(E + 1, dtype=np.int32)
    np.cumsum(q_len, out=cu[1:])
    ent = np.repeat(np.arange(E, dtype=np.int32), q_len)
    pos = (np.arange(T) - np.repeat(cu[:-1], q_len) + np.repeat(q_start, q_len)).astype(np.int32)
    width = int(-(-(q_start + q_len).max() // page))
    table = np.full((E, width), -1, dtype=np.int32)
    nxt = 1
    for e in range(E):
        for b in range(-(-int(q_start[e] + q_len[e]) // page)):
            table[e, b] = nxt
            nxt += 1
    slots = table[ent, pos // page].astype(np.int64) * page + pos % page
    rows = np.asarray([int(cu[e + 1]) - 1 for e in range(E)] if want_last else [], dtype=np.int32)
    return dict(E=E, T=T, ids=np.arange(1, T + 1, dtype=np.int32), pos=pos, ent=ent, cu=cu, q_start=q_start.astype(np.int32),
                q_len=q_len, rows=rows, width=width, tables=[table], slot_maps=[slots],
                state_slots=np.arange(E, dtype=np.int64), max_kv=int((q_start + q_len).max()),
                decode_info=ModelRunner._decode_info(cu, q_len, q_start, ent, T == E))


@pytest.mark.parametrize("q_len,q_start", [([1, 5, 1, 20], [30, 0, 7, 16]), ([40], [0]), ([1, 1, 2], [3, 9, 0]), ([17, 33, 1], [0, 16, 99])])
def test_a_step_laid_into_padded_sizes(q_len, q_start):
    host = host_arrays(q_len, q_start)
    T, E = host["T"], host["E"]
    t_pad, e_pad, width = 64, 8, 16
    p = pad_step(host, t_pad, e_pad, width, pad_slot=99)
    dummy = e_pad
    # sizes
    assert p["T"] == t_pad and p["E"] == e_pad + 1 and p["width"] == width
    assert all(len(p[k]) == t_pad for k in ("ids", "pos", "ent")) and len(p["slot_maps"][0]) == t_pad
    assert len(p["cu"]) == e_pad + 2 and len(p["q_start"]) == e_pad + 1 and len(p["rows"]) == e_pad
    assert p["tables"][0].shape == (e_pad + 1, width) and p["decode_info"].shape == (e_pad, 4)
    assert p["tiles"].shape == (t_pad // ops.PLAN_TILE_ROWS + e_pad, 4)
    # the step's own part is untouched
    for k in ("ids", "pos", "ent"):
        assert np.array_equal(p[k][:T], host[k])
    assert np.array_equal(p["slot_maps"][0][:T], host["slot_maps"][0]) and np.array_equal(p["rows"][:E], host["rows"])
    assert np.array_equal(p["tables"][0][:E, :host["width"]], host["tables"][0])
    # the padding: tokens of the extra entry at position 0, which write nothing and read page 0 only
    assert (p["ent"][T:] == dummy).all() and (p["pos"][T:] == 0).all() and (p["slot_maps"][0][T:] == -1).all()
    assert p["tables"][0][dummy, 0] == 0 and (p["tables"][0][dummy, 1:] == -1).all() and (p["tables"][0][E:dummy] == -1).all()
    # entries: cu is monotone, the empty entries own nothing, the extra entry owns the padding rows
    assert (np.diff(p["cu"]) >= 0).all() and p["cu"][E] == T and p["cu"][dummy] == T and p["cu"][dummy + 1] == t_pad
    assert int(p["q_len"].sum()) == t_pad and p["q_len"][dummy] == t_pad - T and (p["q_len"][E:dummy] == 0).all()
    # the plan: every own row is covered exactly once by a record of a single token or by a tile; what fills the plan
    # points at the first padding row
    covered = np.zeros(t_pad, dtype=int)
    singles = sum(1 for n in q_len if n == 1)
    for i, (row, pos, entry, _) in enumerate(p["decode_info"]):
        if i < singles:
            assert entry < E and host["q_len"][entry] == 1 and pos == host["q_start"][entry] and row == host["cu"][entry]
            covered[row] += 1
        else:
            assert (row, pos, entry) == (T, 0, dummy)
    for entry, row0, rows, pos0 in p["tiles"]:
        if entry == dummy:
            assert (row0, rows, pos0) == (T, 1, 0)
            continue
        assert 1 <= rows <= ops.PLAN_TILE_ROWS and host["cu"][entry] <= row0 and row0 + rows <= host["cu"][entry + 1]
        assert pos0 == host["q_start"][entry] + row0 - host["cu"][entry]
        covered[row0:row0 + rows] += 1
    assert (covered[:T] == 1).all() and (covered[T:] == 0).all()


def test_rows_go_to_records_and_tiles():
    rows, pos, entries, tiles = ops.plan_rows([1, 20, 1, 3], [5, 0, 8, 40], 16)
    assert rows == [0, 21] and pos == [5, 8] and entries == [0, 2]
    assert sorted(tiles) == [(1, 1, 16, 0), (1, 17, 4, 16), (3, 22, 3, 40)]
    assert tiles[0] == (3, 22, 3, 40)            # the tile with the most keys comes first


def test_a_step_of_portions_alone_gets_no_records_of_single_tokens():
    host = host_arrays([40, 7], [0, 16])
    assert len(host["decode_info"]) == 0
    p = pad_step(host, 64, 8, 16, pad_slot=99, n_single=0)
    assert p["decode_info"].shape == (0, 4)
    full = pad_step(host, 64, 8, 16, pad_slot=99)
    assert all(np.array_equal(p[k], full[k]) for k in ("ids", "pos", "ent", "cu", "q_len", "rows", "tiles", "state_slots"))


def test_padding_of_one_row_has_a_record_of_its_own():
    """An entry of one token is left out by kernels for portions: the row behind 63 tokens of portions is covered by the
    records of single tokens, longer paddings by the portions' own way."""
    assert single_records(62, 64, 8, 0) == 0 and single_records(100, 128, 16, 0) == 0
    assert single_records(63, 64, 8, 0) == 8 and single_records(127, 128, 16, 0) == 16
    assert single_records(40, 64, 8, 1) == 8 and single_records(63, 64, 8, 3) == 8
    host = host_arrays([40, 23], [0, 16])
    p = pad_step(host, 64, 8, 16, pad_slot=99, n_single=single_records(63, 64, 8, 0))
    assert p["decode_info"].shape == (8, 4) and (p["decode_info"][:, 0] == 63).all() and p["q_len"][8] == 1


def test_rows_of_recorded_steps():
    from ginfer_amd.engine.runner import padded_rows
    assert [padded_rows(n) for n in (1, 64, 65, 128, 129, 256, 257, 384, 385, 512, 513, 1025)] == [64, 64, 128, 128, 256, 256, 384, 384, 512, 512, 1024, 2048]


def test_heads_side_by_side_do_not_follow_the_padding():
    """12 heads in 2 groups beside 64 entries: three heads to a workgroup in steps of 384 and 512 rows alike, two in one of 256; a step
    that is launched as it is keeps its own number."""
    from types import SimpleNamespace
    from ginfer_amd.engine.runner import ModelRunner
    from ginfer_amd.kernels import ops
    recorded, plain = SimpleNamespace(extra={"static_plan": {}}), SimpleNamespace(extra={})
    heads = lambda rows, step: ops._shared_heads(ModelRunner._padded_tiles(rows, 64), 6, 2, ops._prefill_fill(recorded, 128), ops._prefill_prefer(step))
    assert [heads(rows, recorded) for rows in (256, 384, 512)] == [2, 3, 3] and heads(384, plain) == 2


def test_one_length_of_splits_for_contexts_far_apart():
    """The longest context of the single tokens, not of the step, while their mean is below 0.8 of it; 0: each token's own."""
    host = host_arrays([1, 40, 1, 1], [300, 1000, 16, 700])
    assert host["decode_info"].tolist() == [[0, 300, 0, 701], [41, 16, 2, 701], [42, 700, 3, 701]]
    p = pad_step(host, 64, 8, 160, pad_slot=99)
    assert p["decode_info"][:3].tolist() == host["decode_info"].tolist() and host_arrays([40], [0])["decode_info"].shape == (0, 4)
    assert ops.single_tokens_length([99, 59]) == 0 and ops.single_tokens_length([99, 58]) == 100 and ops.single_tokens_length([7]) == 0
    assert host_arrays([1, 1], [99, 59])["decode_info"].tolist() == [[0, 99, 0, 0], [1, 59, 1, 0]]


def test_rows_that_a_step_is_laid_into():
    """Multiples of 64, where the next of the sizes by which steps are recorded is no larger than what a model's steps may have."""
    from ginfer_amd.engine.runner import recorded_rows
    assert [recorded_rows(n, 512) for n in (1, 64, 65, 129, 193, 257, 321, 385, 449, 512, 513)] == [64, 64, 128, 192, 256, 320, 384, 448, 512, 512, None]
    assert [recorded_rows(n, 214) for n in (65, 128, 129, 192)] == [128, 128, None, None]
    assert [recorded_rows(n, 500) for n in (257, 384, 385)] == [320, 384, None] and recorded_rows(513, 1024) == 1024 and recorded_rows(1, 50) is None
