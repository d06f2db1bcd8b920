"""What the kernels' host side decides.  The argument types that Python gives the kernel libraries
(tests that call one kernel) come from the declarations in tinyinfer_kernels.h: pointers are passed as
plain ints, which ctypes would cut to 32 bits for a function without declared types.  And the number of
runs the decode attention cuts a context into."""
import ctypes
import os
import re

import pytest

import tinyinfer_amd  # noqa: F401
from tinyinfer_amd.csrc import build
from tinyinfer_amd.ops import kernels


def header_text():
    with open(os.path.join(build.HERE, "tinyinfer_kernels.h")) as f:
        return f.read()


def test_every_kernel_the_host_library_calls_is_declared():
    """ops.cpp resolves kernels by name (`KERNEL("lib", ti_fn)`) with the type of the header's declaration:
    a name the header does not declare would not compile.  Here: every such name is in the header, and the
    library it is looked up in is one the build knows."""
    declared = kernels.header_signatures(header_text())
    with open(os.path.join(os.path.dirname(build.HERE), "ops", "ops.cpp")) as f:
        used = re.findall(r'KERNEL\("(\w+)",\s*(ti_\w+)\)', f.read())
    assert len(used) > 15, "the pattern of this test is out of date"
    for lib, fn in used:
        assert fn in declared, fn
        assert lib in build.SOURCES, lib


def test_declarations_are_read_as_written():
    sig = kernels.header_signatures(header_text())
    restype, args = sig["ti_rmsnorm"]
    # int ti_rmsnorm(int out_dtype, const float* x, const float* w, const int* rows, void* out, int n_rows, int H,
    #                float eps, hipStream_t stream)
    assert restype is ctypes.c_int
    assert args == [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int,
                    ctypes.c_int, ctypes.c_float, ctypes.c_void_p]
    restype, args = sig["ti_gemm_bf16"]
    assert args[6] is ctypes.c_long and args[-1] is ctypes.c_void_p and len(args) == 9
    with open(os.path.join(build.HERE, "tinyinfer_kernels_tuning.h")) as f:
        tuning = kernels.header_signatures(f.read())
    assert tuning["ti_tuning_set"] == (ctypes.c_int, [ctypes.c_void_p, ctypes.c_long]) and tuning["ti_tuning_reset"] == (None, [])
    assert sig["ti_fill_random"][1][6] is ctypes.c_ulong
    # what the call sites pass for such arguments is accepted
    assert ctypes.c_void_p.from_param(None) is None
    ctypes.c_void_p.from_param(ctypes.byref(ctypes.c_int(0)))
    ctypes.c_void_p.from_param(1 << 45)
    ctypes.c_long.from_param(ctypes.c_long(5))
    ctypes.c_float.from_param(ctypes.c_float(1.0))


def test_a_declaration_with_an_unknown_type_is_refused():
    import pytest
    with pytest.raises(kernels.KernelError):
        kernels.header_signatures("int ti_x(double y);")


def test_context_splits_of_the_decode_kernel(monkeypatch):
    """The number of runs the decode attention cuts the context into: bounded by the context the
    launch is sized for, chosen for the typical one, and never just beyond a whole round of the
    compute units when fewer runs fill one round (12 rows x 8 kv heads: 2 runs, not 3)."""
    from tinyinfer_amd.ops import kernels as a
    monkeypatch.setattr(a, "compute_units", lambda: 256)
    assert a.decode_splits(8, 8, 16, 4096, 2112) == 4          # 256 workgroups
    assert a.decode_splits(12, 8, 16, 4096, 2112) == 2         # 192, not 288
    assert a.decode_splits(24, 8, 16, 4096, 2112) == 1         # 192 in one round, and no merge
    assert a.decode_splits(64, 8, 16, 4096, 2112) == 1
    assert a.decode_splits(1, 8, 16, 4096, 2112) == 16         # bounded: 16 blocks of 16 keys a run at least
    assert a.decode_splits(1, 8, 16, 100, 100) == 1            # a short context is not split
    assert a.decode_splits(1, 1, 64, 10 ** 6, 10 ** 6) <= a.MAX_SPLITS
    # half the bytes per token (head size 64): a run is worth its prologue only if twice as long
    assert a.decode_splits(12, 8, 16, 4096, 2112, head_dim=64) <= a.decode_splits(12, 8, 16, 4096, 2112)
    for rows in range(1, 70):
        for context in (300, 2000, 9000, 40000):
            s = a.decode_splits(rows, 8, 16, context)
            assert 1 <= s <= max(1, min(-(-context // 16) // a.MIN_BLOCKS_PER_SPLIT, a.MAX_SPLITS))


@pytest.mark.parametrize("heads,tiles,paired,light", [
    (16, 1, 0, 0), (16, 16, 0, 0), (16, 17, 0, 0), (16, 19, 0, 0), (16, 20, 0, 1), (16, 21, 0, 1), (16, 30, 0, 1), (16, 31, 1, 1), (16, 32, 1, 1), (16, 33, 0, 0),
    (16, 48, 0, 0), (16, 51, 0, 0), (16, 52, 0, 1), (16, 62, 0, 1), (16, 63, 1, 1), (16, 64, 1, 1), (16, 65, 0, 0), (16, 96, 1, 1), (16, 112, 0, 0), (16, 128, 1, 1),
    (32, 15, 0, 1), (32, 16, 1, 1), (32, 17, 0, 0), (3, 162, 0, 1), (3, 163, 1, 1), (3, 170, 1, 1), (3, 171, 0, 0), (1, 319, 0, 0), (1, 320, 0, 1), (0, 0, 0, 0),
    (64, 1 << 20, 1, 1)])
def test_two_tiles_a_workgroup_where_they_are_an_even_number_of_rounds(heads, tiles, paired, light):
    """On 256 units, in the last tenth of an even round; light tiles (up to 256 keys, by their context or their window) from its first quarter on.  The keys
    of as many tiles are never cut into runs."""
    from tinyinfer_amd import native
    said = ctypes.c_int()
    for context, window, want in ((2048, 0, paired), (257, 0, paired), (40000, 0, paired), (40000, 256, paired), (256, 0, light), (64, 0, light), (40000, 128, light)):
        runs = native.lib().ti_portion_launch(tiles, heads, context, window, 256, ctypes.byref(said))
        assert bool(said.value) == want, (context, window)
        assert runs == 1 or (not want and 2 * tiles * heads <= 256)


@pytest.mark.parametrize("portions,tokens,start,kv_heads,together", [
    (12, 64, 500, 4, True), (12, 64, 500, 2, True), (32, 64, 1500, 4, True), (8, 500, 0, 4, True), (5, 130, 700, 4, True), (12, 64, 500, 3, True),
    (12, 64, 500, 8, False), (12, 64, 500, 16, False), (12, 100, 0, 4, False), (6, 200, 0, 4, False), (3, 500, 0, 4, False), (1, 2048, 0, 4, False),
    (1, 64, 100000, 4, False), (2, 1000, 0, 4, False), (2, 512, 8000, 4, True), (0, 0, 0, 4, False)])
def test_which_tiles_have_their_heads_on_one_die(portions, tokens, start, kv_heads, together):
    """Several portions of up to eight tiles each, whose keys and values are more than 4 MiB, under kv heads that eight does not divide."""
    from tinyinfer_amd import native
    tiles = portions * -(-tokens // 64)
    assert native.lib().ti_heads_together(portions, portions * (tokens + start), tiles, kv_heads, 128) == together


def test_what_the_rows_of_a_draw_ask_for_packs_from_any_iterable():
    """Requests and counters as lists, tuples, views and iterators give the same bytes, numbers beyond their type's range what ctypes
    makes of them."""
    from tinyinfer_amd.sampling import Sampler, SamplingParams
    params = [SamplingParams(0.5, 7, 0.9, -3), SamplingParams()]
    want = [bytes(a) for a in Sampler._arguments(2, params, [11, 5], [0, 2])]
    live = {11: "a", 5: "b"}
    for requests, counters in (((11, 5), (0, 2)), (live.keys(), iter([0, 2])), (iter([11, 5]), (c for c in (0, 2)))):
        assert [bytes(a) for a in Sampler._arguments(2, params, requests, counters)] == want
    assert bytes(Sampler._arguments(2, params, iter([11 + (1 << 64), 5]), [0, 2])[4]) == want[4]


def test_records_of_a_draw_say_what_the_lists_say():
    """A record's fields are the lists' elements; parameters and numbers that a record cannot hold go by the lists (None)."""
    import copy
    import dataclasses
    import pickle
    import struct

    import numpy as np
    from tinyinfer_amd.sampling import Sampler, SamplingParams

    class Lists:                                      # parameters of a caller's own
        temperature, top_k, top_p, seed = 0.5, 7, 0.9, 1
    params = [SamplingParams(0.5, 7, 0.9, -3), SamplingParams(1, 0, 1, 1 << 63), dataclasses.replace(SamplingParams(0.5, 7), top_k=9),
              pickle.loads(pickle.dumps(SamplingParams(0.25, 3, 0.5, 4))), copy.copy(SamplingParams(1e39))]
    n = len(params)
    records, requests, counters = Sampler._records(n, params, (1, 2, 3, 4, 5), (0,) * n)
    lists = Sampler._arguments(n, params, (1, 2, 3, 4, 5), (0,) * n)
    fields = list(struct.iter_unpack("@fif4xQ", records))
    assert len(records) == 24 * n
    for i, kind in enumerate("fifQ"):
        assert struct.pack(f"{n}{kind}", *[f[i] for f in fields]) == lists[i]
    assert (requests, counters) == lists[4:]
    for odd in (Lists(), SamplingParams(0.5, 1 << 40), SamplingParams(0.5, 2.0), SamplingParams(np.float32(0.5))):
        assert Sampler._records(2, [odd, params[0]], (1, 2), (0, 0)) is None
    assert Sampler._records(2, params[:2], (1 << 64, 2), (0, 0)) is None
    assert Sampler._records(2, params[:2], (1,), (0, 0)) is None
    assert SamplingParams(0.5, 7) == SamplingParams(0.5, 7) and repr(SamplingParams()).count("record") == 0


def test_parameters_of_a_draw_hold_what_they_were_given():
    """Drawn with or not, a SamplingParams' attributes are its four, in vars, in a pickle and in a copy; parameters of a caller's own class, whose
    numbers may change between draws, go by the lists whether or not it derives from SamplingParams."""
    import copy
    import pickle

    from tinyinfer_amd.sampling import Sampler, SamplingParams
    p = SamplingParams(0.5, 7, 0.9, -3)
    given = {"temperature": 0.5, "top_k": 7, "top_p": 0.9, "seed": -3}
    fresh = pickle.dumps(p)
    for _ in range(2):
        assert vars(p) == given and SamplingParams(**vars(p)) == p and pickle.dumps(p) == fresh
        first = Sampler._records(1, [p], (1,), (0,))
        again = Sampler._records(2, [pickle.loads(fresh), copy.copy(p)], (1, 1), (0, 0))
        assert again[0] == 2 * first[0] and len(first[0]) == 24

    class Cooling(SamplingParams):
        calls = 0

        @property
        def top_p(self):
            Cooling.calls += 1
            return 1.0 / Cooling.calls

        @top_p.setter
        def top_p(self, value):
            pass

    class Named(SamplingParams):
        _record = b"not a record"
    for own in (Cooling, Named):
        assert Sampler._records(1, [own.__new__(own)], (1,), (0,)) is None
    bad = SamplingParams(0.5, 1 << 40)                    # cut to 32 bits by the lists, at every call
    for _ in range(2):
        assert Sampler._records(2, [p, bad], (1, 2), (0, 0)) is None
    assert Sampler._records(1, [p], (1,), (0,)) == first


@pytest.mark.parametrize("heads,rows,context,tokens,behind,one", [
    # whole portions: enough units left, or short rows; then long rows beside portions on most units or all, which took up to 12 % longer in one launch
    (16, 2, 2000, 512, 0, True), (16, 2, 2000, 768, 0, True), (16, 2, 12000, 768, 4000, True), (16, 4, 500, 1024, 8000, True),
    (16, 6, 12000, 576, 8000, True), (16, 16, 4000, 576, 8000, True), (16, 64, 4000, 1024, 4000, True), (32, 2, 2000, 384, 0, True),
    (16, 2, 2000, 1024, 4000, False), (16, 2, 12000, 768, 0, False), (16, 2, 12000, 1024, 0, False), (16, 4, 4000, 832, 0, False),
    (16, 1, 4000, 1024, 8000, False), (16, 6, 12000, 640, 0, False), (32, 2, 2000, 512, 1500, False), (32, 2, 12000, 512, 6000, False),
    # portions whose keys want runs
    (16, 48, 2048, 16, 4000, True), (16, 2, 2048, 64, 1000, True), (16, 8, 2048, 16, 2500, False), (16, 32, 2048, 16, 2500, False),
    (16, 2, 2048, 16, 8000, False), (16, 8, 2048, 512, 8000, False)])
def test_portions_and_rows_share_a_launch_where_that_was_measured_to_be_faster(heads, rows, context, tokens, behind, one):
    """Steps of 8 heads for keys on 256 compute units, each timed with one attention launch and with two: the rule takes the faster."""
    from tinyinfer_amd import native
    blocks = context // 16 + 1
    assert native.lib().ti_portions_with_rows(-(-tokens // 64), behind + tokens, behind + min(tokens, 64), rows, blocks, rows * blocks, 16384,
                                              heads, 8, 0, 256, 128) == one


@pytest.mark.parametrize("rows,context,cut", [(33, 300, False), (33, 2000, True), (33, 5000, True), (36, 3000, True), (40, 5000, True), (44, 3000, True),
                                              (48, 300, False), (48, 3000, True), (52, 3000, False), (64, 3000, False), (66, 300, False),
                                              (66, 3000, True), (72, 3000, True), (96, 3000, False)])
def test_rows_on_more_than_a_round_of_the_units_are_cut_where_whole_ones_leave_units_idle(rows, context, cut):
    """Rows of one length, 8 heads for keys on 256 units: a fifth of the two workgroups a unit idle and long contexts; the others stay whole."""
    from tinyinfer_amd import native
    used = native.lib().ti_decode_runs(rows, context // 16 + 1, 8192, 16, 8, 256, 128)
    assert used > rows if cut else used == rows
