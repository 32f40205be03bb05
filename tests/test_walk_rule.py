"""Which way the recurrences with a decay walk a step: by the sizes of its entries alone."""
import types

from ginfer_amd.kernels import ops


def test_one_token_an_entry_takes_tiles_of_one():
    for entries in (1, 8, 16, 64, 256):
        for heads, dim, vdim in ((12, 64, 128), (28, 128, 128), (8, 256, 256), (16, 32, 64)):
            assert ops.decay_walk_way(entries, entries, 1, heads, dim, vdim) == 1
            assert ops.decay_walk_way(entries, entries, 0, heads, dim, vdim) == 1      # a recorded step of single tokens


def test_narrow_workgroups_while_the_long_entries_leave_the_chip_room():
    way = lambda lens, heads, dim, vdim, turned=False: ops.decay_walk_way(sum(lens), len(lens), max(lens), heads, dim, vdim, turned)
    # a prompt alone, short or long
    assert way([2048], 12, 64, 128) == 8 and way([64], 12, 64, 128) == 8 and way([300], 8, 256, 256) == 8
    # the mean says nothing about the longest: a portion beside decoding requests
    assert way([500] + [1] * 32, 12, 64, 128) == 8 and way([2000] + [1] * 48, 12, 64, 128) == 8
    # ... unless the states beside it cost more than its chain gains
    assert way([500] + [1] * 32, 8, 256, 256) == 16 and way([157, 101] + [1] * 32, 12, 64, 128) == 16
    # enough long entries to fill the chip: operands read once for 16 columns
    assert way([918] * 5, 12, 64, 128) == 16 and way([918] * 5, 28, 128, 128) == 16 and way([100] * 8, 12, 64, 128) == 16
    assert way([300] * 4, 12, 64, 128) == 8 and way([300] * 4, 12, 64, 128, True) == 16 and way([300] * 4, 12, 32, 128, True) == 8
    assert way([2000] + [1] * 32, 8, 256, 256) == 16 and way([157, 101] + [1] * 32, 16, 32, 64) == 16
    assert way([300] * 2, 12, 64, 128) == 8 and way([300] * 2, 8, 256, 256) == 16 and way([2048], 28, 128, 128) == 16
    # the grid's third dimension
    assert way([2048], 1, 1, 8 * 65535) == 16


def test_a_recorded_step_goes_by_the_mean_and_others_by_the_longest():
    step = lambda lens, extra: types.SimpleNamespace(host_q_len=lens, extra=extra)
    lens = [500] + [1] * 32
    assert ops._walk_of(step(lens, {}), 532, 33, 12, 64, 128) == 8
    assert ops._walk_of(step(lens, None), 532, 33, 12, 64, 128) == 8
    assert ops._walk_of(step(lens, {"static_plan": {}}), 532, 33, 12, 64, 128) == 16
    assert ops._walk_of(types.SimpleNamespace(), 532, 33, 12, 64, 128) == 16
