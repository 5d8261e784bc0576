"""CPU-side checks of the product package: its packer against the oracle's bytes, the C-ABI
library's exports and host-side validation, and the nn.Module plumbing.  No kernel runs here."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

from oracle import cbk_ref as R
from cobalt_amd import _lib, format as F
from cobalt_amd.linear import CobaltLinear, patch_model
from helpers import FIXED_CASES, case_id, kw_of, make_raw, oracle_pack, product_pack

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("case", FIXED_CASES, ids=case_id)
def test_product_packer_matches_oracle_bytes(case):
    K, N = 12, 640
    raw = make_raw(case, K, N, seed=7)
    raw["zero"][0, 0] = -3        # one off-grid group, exercises the zero repair
    raw["zero"][5, 1] = 99 if case[1] < 8 else 300
    pk = oracle_pack(case, raw)
    pm = product_pack(case, raw)
    assert np.array_equal(pm.array("data").numpy(), pk["data"])
    assert np.array_equal(pm.array("scale").numpy(), pk["scale"].reshape(-1))
    assert np.array_equal(pm.array("zero").numpy(), pk["zero"].reshape(-1))
    assert pm.n_zero_fixed == pk["n_zero_fixed"] == 2 and pm.n_survivors == pk["n_survivors"]
    assert pm.data_bytes == K * R.row_stride(case[0], N, *case[1:]) and pm.stream_bytes() == R.stream_bytes(pk)
    assert abs(pm.bpw() - R.bpw(pk, K, N)) < 1e-12
    assert all(o % 256 == 0 for o in pm.offs.values())


@pytest.mark.parametrize("case", FIXED_CASES, ids=case_id)
def test_synth_packed_is_valid(case):
    layout, bits, group, keep = case
    K, N = 8, 384
    pm = F.synth_packed(K, N, layout, bits, group, keep or None, seed=3)
    pk = dict(data=pm.array("data").numpy(), scale=pm.array("scale").numpy().reshape(K, -1),
              zero=pm.array("zero").numpy().reshape(K, -1), row_off=None)
    q, kp = R.unpack_codes(pk, K, N, layout, **kw_of(case))
    if keep:
        assert (kp.reshape(K, N // 32, 32).sum(-1) == keep).all()
    assert q.max() <= (1 << bits) - 1
    # padding bits of the stream are zero, so re-packing the decoded codes reproduces the bytes
    pk2 = R.pack_matrix(R.pack_bits(kp), q, pk["scale"], pk["zero"], layout, fix_zero=False, **kw_of(case))
    assert np.array_equal(pk2["data"], pk["data"])


@pytest.mark.parametrize("layout", [F.SPARSE4, F.SPARSE4X, F.SPARSE4E], ids=lambda l: F.LAYOUT_NAME[l])
def test_synth_packed_survivor_streams_are_valid(layout):
    """The synthetic rows have the structure the oracle's reader checks (stored group offsets equal
    the bitmap's prefix sums, rows padded to 16 bytes) and, random padding nibbles aside, are the
    bytes the oracle's packer makes from the decoded codes."""
    K, N = 9, 640
    pm = F.synth_packed(K, N, layout, seed=5)
    pm.validate(deep=True)
    ro = pm.array("row_off").numpy().view(np.uint32)
    pk = dict(data=pm.array("data").numpy(), scale=pm.array("scale").numpy().reshape(K, -1),
              zero=pm.array("zero").numpy().reshape(K, -1), row_off=ro)
    q, kp = R.unpack_codes(pk, K, N, layout)
    assert int(kp.sum()) == pm.n_survivors and q.max() <= 15 and (q[~kp] == 0).all()
    pk2 = R.pack_matrix(R.pack_bits(kp), q, pk["scale"], pk["zero"], layout, fix_zero=False)
    assert np.array_equal(pk2["row_off"], ro) and pk2["data"].size == pk["data"].size
    q2, kp2 = R.unpack_codes(pk2, K, N, layout)
    assert np.array_equal(q2, q) and np.array_equal(kp2, kp)


def test_stream_helpers_roundtrip():
    g = torch.Generator().manual_seed(0)
    for bits in (2, 3, 4, 6, 8):
        for n in (8, 40, 92, 250):
            c = torch.randint(0, 1 << bits, (5, n), generator=g, dtype=torch.int32)
            s = F.pack_stream(c, bits)
            assert s.shape[1] == (n * bits + 7) // 8
            assert torch.equal(F.unpack_stream(s, n, bits), c)
            assert np.array_equal(s.numpy(), R._pack_stream(c.numpy(), bits))


# ------------------------------------------------------------------ C ABI
def test_group_offsets_turn_sparse4_rows_into_the_oracles_sparse4x_bytes():
    """ops.with_group_offsets: the SPARSE4 image of a matrix plus the offset tables is, byte for
    byte, the SPARSE4X image the packer writes for the same matrix (pack_cobalt.py:201-250);
    groups with no, one and all survivors, a row count off the 16-row grid."""
    from cobalt_amd import ops
    from helpers import packed_from_oracle
    K, N = 37, 1024
    raw = R.synth_raw_matrix(K, N, 0.5, 4, seed=21)
    rng = np.random.default_rng(3)
    keep = R.unpack_bits(raw["mask"], N)
    keep[3, :256] = False
    keep[4, 128:384] = True
    keep[5] = False
    keep[5, 700] = True
    raw["q"] = (rng.integers(0, 16, (K, N), dtype=np.uint8) * keep).astype(np.uint8)
    raw["mask"] = R.pack_bits(keep)
    p4 = R.pack_matrix(raw["mask"], raw["q"], raw["scale"], raw["zero"], R.SPARSE4)
    px = R.pack_matrix(raw["mask"], raw["q"], raw["scale"], raw["zero"], R.SPARSE4X)
    pm4 = packed_from_oracle((F.SPARSE4, 4, 128, 0), p4, raw["col_scale"], K, N, "cpu")
    pmx = ops.with_group_offsets(pm4)
    assert pmx.layout == F.SPARSE4X and pmx.validate(deep=True) is pmx
    assert np.array_equal(pmx.array("row_off").numpy().view(np.uint32), px["row_off"])
    assert np.array_equal(pmx.array("data").numpy(), px["data"])
    assert np.array_equal(pmx.array("scale").numpy().view(np.uint16), np.asarray(px["scale"]).view(np.uint16).reshape(-1))
    assert np.array_equal(pmx.array("zero").numpy(), np.asarray(px["zero"]).reshape(-1))
    assert torch.equal(pmx.array("col_scale"), pm4.array("col_scale"))
    with pytest.raises(ValueError):
        ops.with_group_offsets(pmx)


def test_library_exports_every_declared_symbol():
    hdr = open(os.path.join(ROOT, "include", "cbk.h")).read()
    names = set(re.findall(r"\b(cbk_[a-z_]+)\s*\(", hdr))
    assert {"cbk_gemv", "cbk_gemm", "cbk_linear", "cbk_dequant", "cbk_workspace_bytes"} <= names
    L = ctypes.CDLL(_lib.LIB_PATH)
    for n in names:
        assert hasattr(L, n), n
    assert set(_lib.SIGNATURES) == names
    assert _lib.lib().cbk_abi_version() == 1


def test_bench_helper_library_loads():
    """libcbk_bench.so (the measured-ceiling probes of bench.py) is built beside the C-ABI library
    and exports its two entry points; nothing is launched here."""
    path = os.path.join(ROOT, "cobalt_amd", "libcbk_bench.so")
    if not os.path.exists(path):
        pytest.skip("libcbk_bench.so is not built (python -m cobalt_amd.build)")
    L = ctypes.CDLL(path)
    assert hasattr(L, "cbk_bench_mfma_f16") and hasattr(L, "cbk_bench_read")


def test_descriptor_validation_and_strides():
    L = _lib.lib()
    for case in FIXED_CASES:
        layout, bits, group, keep = case
        for N in (128, 4096, 5376, 14336, 21504):
            d = F.CbkDesc(K=16, N=N, layout=layout, bits=bits, group=group, keep=keep)
            assert L.cbk_row_stride(ctypes.byref(d)) == R.row_stride(layout, N, bits, group, keep or None)
    d = F.CbkDesc(K=16, N=4096, layout=F.BLK1632_4)
    o = F.CbkDesc()
    assert L.cbk_desc_check(ctypes.byref(d), ctypes.byref(o)) == 0 and (o.bits, o.group, o.keep) == (4, 128, 16)
    assert L.cbk_stream_bytes(ctypes.byref(d), 0) == 16 * 4096 * 3 // 8 + 16 * 32 * 3
    bad = [F.CbkDesc(K=16, N=4096, layout=11), F.CbkDesc(K=16, N=4096, layout=F.BLKC, bits=5, group=128, keep=16),
           F.CbkDesc(K=16, N=4096, layout=F.BLKC, bits=4, group=32, keep=16),
           F.CbkDesc(K=16, N=4096, layout=F.BLKC, bits=4, group=64, keep=33),
           F.CbkDesc(K=16, N=4096, layout=F.BF16)]
    for b in bad:
        assert L.cbk_desc_check(ctypes.byref(b), ctypes.byref(o)) == -2
    assert L.cbk_desc_check(ctypes.byref(F.CbkDesc(K=16, N=4000, layout=F.DENSE4)), ctypes.byref(o)) == -3
    assert L.cbk_desc_check(ctypes.byref(F.CbkDesc(K=0, N=4096, layout=F.DENSE4)), ctypes.byref(o)) == -3
    assert L.cbk_desc_check(None, ctypes.byref(o)) == -1


def test_workspace_sizes_of_the_decode_path():
    """cbk_workspace_bytes at decode sizes (host arithmetic only, nothing is launched): two to eight
    activation rows of a long row (8192 columns and more, digits beyond LDS) leave room for the
    part sums of the column-split kernel, K * M * parts * 4 bytes with 14 parts at 21504 columns;
    the figure is a multiple of 256, grows with M, and a batch asks for the sum of its matrices."""
    L = _lib.lib()
    flags = F.zero_flags(15, 4)
    long_row = F.CbkDesc(K=5376, N=21504, layout=F.BLK1632_4, flags=flags)
    short_row = F.CbkDesc(K=21504, N=5376, layout=F.BLK1632_4, flags=flags)
    last = 0
    for M in (2, 4, 8):
        need = L.cbk_workspace_bytes(ctypes.byref(long_row), M)
        assert need >= 5376 * M * 14 * 4 and need % 256 == 0 and need >= last
        last = need
    descs = (F.CbkDesc * 2)(long_row, short_row)
    assert L.cbk_gemv_batch_workspace_bytes(2, descs, 8) == \
        L.cbk_workspace_bytes(ctypes.byref(long_row), 8) + L.cbk_workspace_bytes(ctypes.byref(short_row), 8)


def test_entry_points_reject_bad_arguments_before_any_launch():
    L = _lib.lib()
    d = F.CbkDesc(K=16, N=256, layout=F.BLK1632_4)
    # NULL device arrays
    assert L.cbk_gemv(ctypes.byref(d), None, 1, 1, 256, None, 0, 16, None, None, 0, None) == -1
    assert L.cbk_dequant(ctypes.byref(d), 0, 16, 1, None, 0, 256, None) == -1
    d.data, d.scale, d.zero = 0x1000, 0x2000, 0x3000           # never dereferenced: checks fail first
    assert L.cbk_gemv(ctypes.byref(d), None, 1, 1, 256, None, 0, 16, None, None, 0, None) == -1
    assert L.cbk_gemv(ctypes.byref(d), 0x4000, 0, 1, 256, 0x5000, 0, 16, None, None, 0, None) == -5
    assert L.cbk_gemv(ctypes.byref(d), 0x4000, 1, 17, 256, 0x5000, 0, 16, None, None, 0, None) == -3
    assert L.cbk_gemv(ctypes.byref(d), 0x4000, 1, 1, 128, 0x5000, 0, 16, None, None, 0, None) == -3
    assert L.cbk_gemv(ctypes.byref(d), 0x4004, 1, 1, 256, 0x5000, 0, 16, None, None, 0, None) == -4
    assert L.cbk_gemm(ctypes.byref(d), 0x4000, 2, 300, 260, 0x5000, 2, 16, None, None, 0, None) == -4
    assert L.cbk_dequant(ctypes.byref(d), 8, 16, 1, 0x5000, 0, 256, None) == -3
    d.data = 0x1004
    assert L.cbk_gemv(ctypes.byref(d), 0x4000, 1, 1, 256, 0x5000, 0, 16, None, None, 0, None) == -4
    d.data, d.cs_rows = 0x1000, 1
    assert L.cbk_gemv(ctypes.byref(d), 0x4000, 1, 1, 256, 0x5000, 0, 16, None, None, 0, None) == -1
    assert b"aligned" in L.cbk_strerror(-4)
    # the packing and the static-scratch entry points check before they launch, too
    d = F.CbkDesc(K=16, N=256, layout=F.BLK1632_4)
    assert L.cbk_pack(ctypes.byref(d), None, 0x4000, 0x5000, 0x6000, 1, 1, None, None) == -1      # no destination arrays
    d.data, d.scale, d.zero = 0x1000, 0x2000, 0x3000
    assert L.cbk_pack(ctypes.byref(d), None, None, 0x5000, 0x6000, 1, 1, None, None) == -1
    assert L.cbk_pack(ctypes.byref(d), None, 0x4000, 0x5000, 0x6000, 0, 1, None, None) == -5      # zero points are fp16 or uint8
    assert L.cbk_pack(ctypes.byref(d), None, 0x4004, 0x5000, 0x6000, 1, 1, None, None) == -4
    assert L.cbk_pack(ctypes.byref(d), 0x7001, 0x4000, 0x5000, 0x6000, 3, 1, None, None) == -4
    ds = F.CbkDesc(K=16, N=256, layout=F.SPARSE4, data=0x1000, scale=0x2000, zero=0x3000, row_off=0x8000)
    assert L.cbk_pack(ctypes.byref(ds), None, 0x4000, 0x5000, 0x6000, 1, 1, None, None) == -8     # variable-length layouts are not produced
    big = F.CbkDesc(K=256, N=21504, layout=F.BLK1632_4, data=0x1000, scale=0x2000, zero=0x3000)
    assert L.cbk_gemm_static(ctypes.byref(big), 0x4000, 2, 4096, 21504, 0x5000, 2, 256, None, None) == -6


@pytest.mark.skipif(torch.cuda.is_available(), reason="addresses that are none: only where no launch can follow")
def test_prefill_results_do_not_depend_on_the_workspace():
    """A prefill call has one plan: a byte less than cbk_workspace_bytes is refused, whatever a plan with fewer
    parts would need.  cbk_gemm_static, which promises cbk_gemm's results, takes the calls it always took
    (its answer here is the HIP error of a machine without a GPU) and refuses the others."""
    L = _lib.lib()
    fmts = ((F.BLK1632_4, 0, 0, 0), (F.BLKC, 2, 64, 16), (F.BLKC, 3, 64, 10), (F.DENSE4, 0, 0, 0), (F.DENSE8, 0, 0, 0), (F.DENSEB, 2, 64, 0))

    def desc(fmt, K, N, cs, splits=(0, 0)):
        return F.CbkDesc(K=K, N=N, layout=fmt[0], bits=fmt[1], group=fmt[2], keep=fmt[3], data=0x1000, scale=0x2000, zero=0x3000,
                         col_scale=0x4000, cs_rows=cs, cs_split0=splits[0], cs_split1=splits[1],
                         flags=F.FLAG_ZERO_LE_128 | F.FLAG_ZERO_ON_GRID)

    for fmt in fmts:
        for K, N in ((256, 14336), (1024, 4096), (4096, 4096), (14336, 4096)):
            for cs, splits in ((1, (0, 0)), (2, (0, 0)), (3, (K // 2, K // 4)), (3, (K // 2 - 48, K // 4 + 16))):
                for M in (17, 64, 130, 333, 600, 2048):
                    d = desc(fmt, K, N, cs, splits)
                    need = L.cbk_workspace_bytes(ctypes.byref(d), M)
                    for fn in (L.cbk_gemm, L.cbk_linear):
                        assert fn(ctypes.byref(d), 0x8000, 1, M, N, 0x9000, 1, K, None, 0x10000, need - 1, None) == -6, (fmt, K, N, cs, M)
    b64_2, b64_3, d8 = fmts[1], fmts[2], fmts[4]
    for fmt, K, N, M, cs, takes in ((b64_2, 1430, 7040, 405, 2, True), (b64_3, 2602, 4864, 540, 2, True), (d8, 1459, 11264, 486, 1, True),
                                    (fmts[0], 84, 6016, 577, 2, True), (fmts[0], 21504, 5376, 1024, 1, True),
                                    (fmts[0], 256, 5376, 1792, 1, False), (d8, 4096, 14336, 1024, 1, False)):
        d = desc(fmt, K, N, cs)
        assert (L.cbk_gemm_static(ctypes.byref(d), 0x8000, 1, M, N, 0x9000, 1, K, None, None) == -6) == (not takes), (fmt, K, N, M)
        assert (L.cbk_workspace_bytes(ctypes.byref(d), M) <= 16 << 20) == takes
    # the tile kernel's split of these does not fit, whatever the plan that the call then runs on takes
    for fmt, K, N, M in ((b64_2, 44547, 13184, 320), (fmts[5], 45932, 9600, 270)):
        assert L.cbk_gemm_static(ctypes.byref(desc(fmt, K, N, 1)), 0x8000, 1, M, N, 0x9000, 1, K, None, None) == -6, (fmt, K, N, M)


def _sizes_only(K, N, case, cs_rows=1):
    """A matrix for questions about sizes: no memory behind its arrays."""
    return _lib.native().Matrix(torch.empty(0, dtype=torch.uint8), dict.fromkeys(("data", "scale", "zero", "col_scale"), 0), (0, 0),
                                (K, N, *case[:3], case[3] or 0, cs_rows, F.FLAG_ZERO_LE_128 | F.FLAG_ZERO_ON_GRID))


@pytest.mark.parametrize("K,N,cs_rows,M,plan,tail", [
    (5376, 21504, 1, 3485, (2, 4, 4), (3, 1)), (5376, 21504, 1, 3600, (2, 4, 3), (4, 1)), (21504, 5376, 1, 816, (1, 3, 1), (20, 2)),
    (21504, 5376, 1, 864, (1, 3, 1), (20, 2)), (14336, 4096, 1, 1200, (1, 3, 1), (5, 1)), (44224, 2176, 1, 289, (1, 2, 1), (45, 1)),
    (38323, 256, 1, 294, (2, 2, 1), (22, 1)), (36612, 768, 2, 278, (2, 2, 1), (16, 1)), (21504, 5376, 1, 1024, (2, 4, 1), (20, 2)),
    (43008, 5376, 2, 2048, (2, 4, 1), (8, 1)), (34516, 256, 2, 519, (2, 4, 1), (0, 0)), (21716, 256, 2, 519, (2, 4, 1), (2, 1))])
def test_the_last_round_of_smaller_tiles_does_not_choose_the_plan(K, N, cs_rows, M, plan, tail):
    """Kernel, token tile and split of a call (1: rows kernel, 2: tile kernel) go by whole rounds.  `tail`, the row tiles
    and the 64-token units of the second launch that a call on unsplit 256-token tiles ends with, takes no part: counted
    as a share of a round, it moved the calls of the first eight cases to that plan, where most run slower, some
    with weights rounded to a half that were not.  Gate/up row tiles (cs_rows 2) count in pairs, as they are launched."""
    h = _sizes_only(K, N, (F.BLK1632_4, 4, 128, 16), cs_rows)
    assert _lib.native().gemm_plan(h, M, -1) == plan
    assert _lib.native().gemm_last_round(h, M, 2, 4, 1) == tail
    for other in ((2, 2, 1), (2, 4, 2), (1, 3, 1)):
        assert _lib.native().gemm_last_round(h, M, *other) == (0, 0)


@pytest.mark.parametrize("shapes,M,main,slots,split", [
    # main kernel: one row on both sides of five quarters of a step per wavefront and of the room in LDS
    ([(24, 9728)], 1, 0, 32, -1), ([(24, 10240)], 1, 1, 32, -1), ([(24, 29440)], 1, 1, 8, -1), ([(24, 31232)], 1, 0, 16, -1),
    # several rows: the wide table beside as many slots, or beside eight that hold six rounds of parts; not for fewer
    ([(65536, 2944)], 8, 1, 16, -1), ([(65536, 3584)], 8, 0, 16, -1), ([(32768, 3072)], 8, 0, 16, -1), ([(28672, 7168)], 4, 0, 16, -1),
    ([(21504, 5376)], 4, 1, 16, -1), ([(8192, 28672)], 1, 1, 8, -1),
    # split kernel: both sides of half a step; one choice for matrices that have room for it and one that has none
    ([(2976, 5376)], 8, -1, 0, 0), ([(2992, 5376)], 8, -1, 0, 1), ([(2992, 5376), (40, 65024)], 8, -1, 0, 0)])
def test_which_selector_table_a_decode_call_takes(shapes, M, main, slots, split):
    h = [_sizes_only(K, N, (F.BLK1632_4, 4, 128, 16)) for K, N in shapes]
    assert _lib.native().decode_choice(h, M) == (main, slots, split)


def test_selector_table_of_one_dword_blocks_and_of_dense_layouts():
    choice = lambda case, K: _lib.native().decode_choice([_sizes_only(K, 5376, case)], 8)[2]
    assert [choice((F.BLKC, 2, 64, keep), 1024) for keep in (10, 16, 23)] == [0, 1, 0]
    assert choice((F.BLKC, 2, 64, 10), 8192) == 1 and choice((F.DENSEB, 2, 64, None), 8192) == 0


@pytest.mark.parametrize("shapes,M,split", [
    # both ends of the heights that have the lower limit, and of the limit; eight rows of 3072 columns take 72 KB
    ([(8176, 4096)], 6, False), ([(8192, 4096)], 6, True), ([(32752, 4096)], 6, True), ([(32768, 4096)], 6, False),
    ([(14336, 3840)], 6, False), ([(14336, 3968)], 6, True), ([(14336, 4096)], 4, False), ([(14336, 3072)], 8, True),
    # matrices of unequal height go by the tiles of the launch, all one way; one that is not long enough keeps the others
    ([(8192, 4096), (1024, 4096), (1024, 4096)], 6, True), ([(6144, 4096), (1024, 4096), (1008, 4096)], 6, False),
    ([(6144, 4096), (1024, 4096), (1024, 4096)], 6, True), ([(8192, 5120), (1024, 5120), (1024, 5120)], 5, True),
    ([(14336, 4096), (14336, 4096)], 6, True), ([(16384, 4096), (16384, 4096)], 6, False), ([(14336, 4096), (1024, 2048)], 6, False)])
def test_a_launch_is_split_by_columns_as_a_whole(shapes, M, split):
    h = [_sizes_only(K, N, (F.BLK1632_4, 4, 128, 16)) for K, N in shapes]
    main, _, other = _lib.native().decode_choice(h, M)
    assert (main < 0, other >= 0) == (split, split)
    d = (type(F.synth_packed(16, 128, F.BLK1632_4, seed=1).desc()) * len(shapes))()
    for i, (K, N) in enumerate(shapes):
        d[i] = F.synth_packed(16, N, F.BLK1632_4, seed=1).desc()
        d[i].K = K
    parts = sum(K * 2 * M * 4 for K, _ in shapes)                   # two parts of a row at least
    assert not split or _lib.lib().cbk_gemv_batch_workspace_bytes(len(shapes), d, M) >= parts


@pytest.mark.parametrize("K,N,case,M,slabs", [
    # slots of six parts (four of them) and of two (eight) beside the longest rows, and what leaves room for fewer
    (21504, 5376, (F.BLK1632_4, 4, 128, 16), 8, 1), (21504, 5376, (F.BLKC, 4, 64, 10), 8, 2),
    (262144, 5376, (F.BLKC, 4, 64, 10), 8, 1), (262144, 5632, (F.BLK1632_4, 4, 128, 16), 8, 1), (262144, 5760, (F.BLK1632_4, 4, 128, 16), 8, 2),
    (262144, 5632, (F.DENSEB, 3, 128, None), 8, 1), (262144, 6400, (F.BLK1632_4, 4, 128, 16), 7, 1), (65552, 8832, (F.DENSEB, 8, 64, None), 4, 1)])
def test_rows_are_staged_whole_beside_a_slot_part_for_every_wavefront(K, N, case, M, slabs):
    """Without a workspace a row whose digits do not fit in LDS is staged slab by slab.  It fits where the reduction slots
    beside it hold a part for each of sixteen wavefronts: with fewer they wait for each other."""
    assert _lib.native().decode_slabs([_sizes_only(K, N, case)], M) == slabs


@pytest.mark.parametrize("case,K,N,M,split", [
    ((F.BLKC, 4, 64, 10), 65552, 5120, 8, True), ((F.BLKC, 4, 64, 10), 65552, 4992, 8, False), ((F.BLK1632_4, 4, 128, 16), 262144, 5888, 8, True),
    ((F.BLK1632_4, 4, 128, 16), 65552, 4096, 8, False), ((F.DENSEB, 3, 128, None), 262144, 5632, 8, True),
    # dense 4-bit: where whole rows do not fit; 8-bit at five rows and more: always
    ((F.DENSE4, 4, 128, None), 262144, 5632, 8, False), ((F.DENSE4, 4, 128, None), 262144, 5760, 8, True),
    ((F.DENSEB, 8, 64, None), 65552, 8832, 4, True), ((F.DENSEB, 8, 64, None), 65552, 4352, 8, True),
    ((F.DENSEB, 8, 64, None), 65552, 4352, 4, False), ((F.DENSEB, 8, 64, None), 65552, 512, 5, True)])
def test_which_tall_matrices_are_split_by_columns(case, K, N, M, split):
    """More than 4096 tiles: above 120 KB of digits, unless the main kernel is at the memory's rate; the workspace goes with it."""
    assert (_lib.native().decode_choice([_sizes_only(K, N, case)], M)[0] < 0) == split
    d = F.synth_packed(16, N, *case, seed=1).desc()
    d.K = K
    assert (_lib.lib().cbk_workspace_bytes(ctypes.byref(d), M) >= K * M * 4) == split


def test_ops_refuse_to_run_without_gpu_tensors():
    from cobalt_amd import ops
    pm = F.synth_packed(16, 256, F.BLK1632_4, seed=1)
    with pytest.raises(_lib.CbkError):
        ops.linear(pm, torch.zeros(1, 256, dtype=torch.float16))
    with pytest.raises(_lib.CbkError):
        ops.dequant(pm)


# ------------------------------------------------------------------ module plumbing
class _FakeSQL(torch.nn.Module):
    """Same buffers as the reference's SparseQuantLinear (benchmark_suite.py:1178-1198)."""

    def __init__(self, W_q, scales, zeros, mask, scale2, bias, meta):
        super().__init__()
        for n, v in dict(W_q=W_q, scales=scales, zeros=zeros, mask=mask, scale2=scale2).items():
            self.register_buffer(n, v)
        self.bias = torch.nn.Parameter(bias) if bias is not None else None
        self.meta = meta


def _fake_sql(K, N, bits, group, block, seed):
    raw = R.synth_raw_matrix(K, N, 0.5, bits, seed=seed, block=block, group=group)
    keep = torch.from_numpy(R.unpack_bits(raw["mask"], N))
    m = _FakeSQL(torch.from_numpy(raw["q"]).half(), torch.from_numpy(raw["scale"]).reshape(K, -1, 1),
                 torch.from_numpy(raw["zero"]).reshape(K, -1, 1), keep.half(),
                 torch.from_numpy(raw["col_scale"]).reshape(1, N), torch.randn(K).half(),
                 {"nbits": bits, "group_size": group})
    return m, raw


def test_from_sparse_quant_linear_layout_choice_and_bytes():
    m, raw = _fake_sql(16, 256, 4, 128, 32, 1)
    cl = CobaltLinear.from_sparse_quant_linear(m)
    p = cl.packed()
    assert (p.layout, p.bits, p.group, p.keep) == (F.BLK1632_4, 4, 128, 16)
    pk = R.pack_matrix(raw["mask"], raw["q"], raw["scale"], raw["zero"], R.BLK1632_4)
    assert np.array_equal(p.array("data").numpy(), pk["data"])
    assert np.array_equal(p.array("col_scale").numpy(), raw["col_scale"])
    m2, _ = _fake_sql(16, 256, 3, 64, 0, 2)               # unconstrained mask -> dense stream
    p2 = CobaltLinear.from_sparse_quant_linear(m2).packed()
    assert (p2.layout, p2.bits, p2.group) == (F.DENSEB, 3, 64)
    m3, _ = _fake_sql(16, 256, 2, 64, 32, 3)
    p3 = CobaltLinear.from_sparse_quant_linear(m3).packed()
    assert (p3.layout, p3.bits, p3.group, p3.keep) == (F.BLKC, 2, 64, 16)
    assert cl.bias is not None and cl.in_features == 256 and cl.out_features == 16
    assert "BLK1632_4" in repr(cl)
    with pytest.raises(ValueError):
        cl.set_forward_backend("pytorch")


def test_state_dict_roundtrip_and_patch_model():
    m, _ = _fake_sql(16, 256, 4, 128, 32, 4)
    cl = CobaltLinear.from_sparse_quant_linear(m)
    sd = cl.state_dict()
    assert set(sd) == {"blob", "cbk_meta", "bias"}
    cl2 = CobaltLinear(F.synth_packed(16, 256, F.BLK1632_4, seed=9), bias=torch.zeros(16).half())
    cl2.load_state_dict(sd)
    assert torch.equal(cl2.blob, cl.blob) and cl2.packed().offs == cl.packed().offs

    net = torch.nn.Sequential(torch.nn.Linear(256, 16), torch.nn.ReLU())
    net.add_module("inner", torch.nn.Sequential(torch.nn.Linear(256, 16)))
    done = patch_model(net, lambda name, mod: cl if isinstance(mod, torch.nn.Linear) and name == "inner.0" else None)
    assert done == ["inner.0"] and net.inner[0] is cl
    done = patch_model(net, {"0": cl2})
    assert done == ["0"] and net[0] is cl2
    with pytest.raises(TypeError):
        F.dtype_code(torch.float64)


def test_packed_matrix_validate_refuses_descriptions_that_do_not_fit_the_image():
    """A description from a state dict or a manifest is outside input: offsets past the image,
    misaligned arrays, a byte count that is not rows x stride, row ranges beyond K, parameters the
    layout does not take and row offsets that are not increasing multiples of 16 all raise."""
    import dataclasses
    pm = F.synth_packed(48, 256, F.BLK1632_4, seed=1)
    assert pm.validate() is pm and pm.to_tiled().validate().tiled
    for change in (dict(offs={**pm.offs, "scale": pm.blob.numel()}), dict(offs={**pm.offs, "data": 8}),
                   dict(offs={k: v for k, v in pm.offs.items() if k != "zero"}), dict(data_bytes=pm.data_bytes - 96),
                   dict(K=pm.K + 1), dict(cs_rows=4), dict(cs_rows=3, cs_splits=(40, 16)), dict(bits=3), dict(keep=8),
                   dict(layout=4), dict(N=192), dict(blob=pm.blob[:-256])):
        with pytest.raises(ValueError):
            dataclasses.replace(pm, **change).validate()
    import os
    z = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "sparse_stream.npz"))
    sp = F.from_arrays(z["c0_SPARSE4X_data"], z["c0_SPARSE4X_scale"], z["c0_SPARSE4X_zero"], None, 5, 256, F.SPARSE4X,
                       row_off=z["c0_SPARSE4X_row_off"].astype(np.int32))
    assert sp.validate(deep=True) is sp
    ro = sp.array("row_off").clone()
    ro[3] += 8
    broken = sp.clone()
    broken.array("row_off")[:] = ro
    with pytest.raises(ValueError):
        broken.validate(deep=True)
    cl = CobaltLinear(pm)
    meta = cl.cbk_meta.clone()
    meta[12] = pm.blob.numel()                                         # off_scale past the image
    with pytest.raises(ValueError):
        CobaltLinear.from_state(pm.blob, meta)
