"""Every instantiation of the two prefill kernels by name: code configuration x token tile x column-scale vectors
(plain, gate/up, q|k|v) x split of the column range x byte order, for activations of both signs and of one.
Against float64 on the dequantised weights, held to the error of operands of 11 bits in exact sums (2 % for
float32 sums and the draw); every call twice, bit for bit."""
import ctypes

import pytest
import torch

from cobalt_amd import _lib, format as F, ops
from helpers import TOKENS, acts, case_id, column_parts, gemm_as, gemm_plan, last_round

pytestmark = pytest.mark.gpu
DEV = "cuda"
CASES = [(F.BLK1632_6, 6, 128, 16), (F.DENSEB, 8, 64, 0), (F.DENSE8, 8, 128, 0)] + [
    (F.BLKC if k else F.DENSEB, b, g, k) for b in (2, 3, 4) for k in (0, 10, 16, 23) for g in (64, 128)]
# (kernel, splits of the column range): 13 groups of 128 columns are 28 stages of the tile kernel
SPLITS = {"rows": (1, 2, 3), "tile": (1, 2)}


def _matrix(case, vectors, N, seed):
    mk = lambda k, s: F.synth_packed(k, N, case[0], case[1], case[2], case[3] or None, seed=seed + s, device=DEV)
    if vectors == 1:
        return mk(267, 0)                                             # two row tiles of 128, ragged
    if vectors == 2:
        return F.fuse_rows([mk(131, 0), mk(131, 1)], interleave=True)
    return F.fuse_rows([mk(256, 0), mk(256, 1), mk(57, 2)])           # ranges on the row tiles of both kernels


def _vectors_of_rows(pm):
    k = torch.arange(pm.K, device=DEV)
    return k * 0 if pm.cs_rows == 1 else k % 2 if pm.cs_rows == 2 else (k >= pm.cs_splits[0]).long() + (k >= sum(pm.cs_splits)).long()


@pytest.mark.parametrize("vectors", [1, 2, 3], ids=["plain", "gate_up", "qkv"])
@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_every_instantiation(case, vectors):
    N = 1664
    rows = _matrix(case, vectors, N, seed=vectors)
    W = ops.dequant(rows, torch.float32).double()
    Wh = ops.dequant(rows, torch.float32, with_col_scale=False).half().double()
    cs = rows.array("col_scale").view(rows.cs_rows, N).float()
    vec = _vectors_of_rows(rows)
    x257 = acts(257, N, torch.float16, seed=case[1]).to(DEV)
    ran = set()
    for one_sign in (False, True):
        x = x257.abs() if one_sign else x257
        ref = x.double() @ W.t()
        each = torch.stack([(x.float() * c).half().double() @ Wh.t() for c in cs])       # [vectors, 257, K]
        rounded = each.gather(0, vec.view(1, 1, -1).expand(1, *ref.shape))[0]
        for pm in (rows, rows.to_tiled()):
            for kernel, tiles in TOKENS.items():
                for tokens in tiles:
                    M = tokens + 1                                      # a whole tile and one token
                    bound = float((rounded[:M] - ref[:M]).norm() / ref[:M].norm())
                    for s in SPLITS[kernel]:
                        if kernel == "tile" and s > 1 and (vectors == 2 or case[1] == 8):
                            with pytest.raises(_lib.CbkError):             # gate/up and 8-bit codes are not split there
                                gemm_as(pm, x[:M], kernel, tokens, s)
                            continue
                        y = gemm_as(pm, x[:M], kernel, tokens, s, out_dtype=torch.float32)
                        err = float((y.double() - ref[:M]).norm() / ref[:M].norm())
                        assert err <= 1.02 * bound, (kernel, tokens, s, pm is rows, one_sign, err, bound)
                        assert torch.equal(y, gemm_as(pm, x[:M], kernel, tokens, s, out_dtype=torch.float32)), (kernel, tokens, s)
                        ran.add((kernel, tokens, s))
    assert len(ran) == 9 + (3 if vectors == 2 or case[1] == 8 else 6)


@pytest.mark.parametrize("case", [c for c in CASES if c[3]], ids=case_id)
def test_runs_of_kept_columns(case):
    """Mask bytes with all eight columns kept beside bytes with none: in the tile kernel the eighth survivor's place
    holds the zero point unless the byte is full.  Zero points on the grid's ends and at 128.  Bound as above."""
    N, keep = 1664, case[3]
    pm = _matrix(case, 1, N, seed=5)
    turn = (torch.arange(pm.K, device=DEV)[:, None] + torch.arange(N // 32, device=DEV)) % 32
    run = ((((1 << keep) - 1) << turn) | (((1 << keep) - 1) >> (32 - turn))) & 0xFFFFFFFF    # a run that starts at column `turn`
    mask = pm.array("data")[: pm.data_bytes].view(pm.K, -1)[:, : N // 8]
    mask[:] = ((run[..., None] >> torch.arange(0, 32, 8, device=DEV)) & 255).to(torch.uint8).view(pm.K, N // 8)
    zero = pm.array("zero")
    zero[:] = torch.tensor([0, 2 ** case[1] - 1, 128], dtype=torch.uint8, device=DEV)[torch.arange(zero.numel(), device=DEV) % 3].view(zero.shape)
    pm.flags = F.FLAG_ZERO_LE_128
    W = ops.dequant(pm, torch.float32).double()
    kept = F.unpack_mask(mask, N)
    assert bool((W[~kept] == 0).all()) and int(kept.sum()) == pm.K * N * keep // 32
    Wh = ops.dequant(pm, torch.float32, with_col_scale=False).half().double()
    x = acts(257, N, torch.float16, seed=case[1]).to(DEV)
    ref = x.double() @ W.t()
    bound = float(((x.float() * pm.array("col_scale").view(-1, N).float()).half().double() @ Wh.t() - ref).norm() / ref.norm())
    for tokens in TOKENS["tile"]:
        y = gemm_as(pm.to_tiled(), x, "tile", tokens, out_dtype=torch.float32)
        assert float((y.double() - ref).norm() / ref.norm()) <= 1.02 * bound, tokens


@pytest.mark.parametrize("vectors", [1, 2, 3], ids=["plain", "gate_up", "qkv"])
@pytest.mark.parametrize("rows,tail", [(7423, {1: (1, 64), 2: (2, 64), 3: (1, 64)}), (7700, {1: (3, 64), 2: (4, 64), 3: (3, 64)}),
                                       (10300, {1: (13, 128), 2: (14, 128), 3: (13, 128)}), (14800, {1: (2, 64), 2: (2, 64), 3: (2, 64)}),
                                       (12800, {1: (0, 0), 2: (0, 0), 3: (0, 0)})],
                         ids=["64 tokens", "64 tokens, ragged", "128 tokens", "third round", "none"])
def test_last_round_in_smaller_tiles(rows, tail, vectors):
    """More than 256 tiles of 256 tokens: the row tiles past the last whole round run as smaller tiles in a launch of
    their own if that fits one round (`tail`).  Bit for bit what slices of 700 tokens, at most 174 tiles, give."""
    N, M = 256, 2100                                                    # nine token tiles, 29 / 31 / 41 / 58 / 50 row tiles
    mk = lambda k, s: F.synth_packed(k, N, F.BLKC, 4, 128, 16, seed=s, device=DEV)
    if vectors == 1:
        pm = mk(rows, 0)
    elif vectors == 2:
        pm = F.fuse_rows([mk(rows // 2, 0), mk(rows // 2, 1)], interleave=True)
    else:
        pm = F.fuse_rows([mk(rows // 512 * 256, 0), mk(256, 1), mk(rows - rows // 512 * 256 - 256, 2)])
    pm = pm.to_tiled()
    x = acts(M, N, torch.float16, seed=7).to(DEV)
    assert last_round(pm, M, "tile", 256) == tail[vectors] and last_round(pm, 700, "tile", 256) == (0, 0)
    for act in (None, "silu") if vectors == 2 else (None,):
        y = gemm_as(pm, x, "tile", 256, act=act)
        assert torch.equal(y, torch.cat([gemm_as(pm, x[i:i + 700], "tile", 256, act=act) for i in range(0, M, 700)])), act


@pytest.mark.parametrize("act", ["gelu_tanh", "silu"])
@pytest.mark.parametrize("case", [c for c in CASES if c[2:] in ((128, 16), (64, 10), (128, 0))], ids=case_id)
def test_gated_call_on_every_tile(case, act):
    """act(gate) * up where the column parts meet (rows kernel, also over workgroups: the reduction kernel) and
    from the two halves the tile kernel leaves.  float32 results, the float64 product of the dequantised weights;
    gate and up carry 3e-4 each, the activations have slopes up to 1.1."""
    N = 1664
    pm = _matrix(case, 2, N, seed=9).to_tiled()
    W = ops.dequant(pm, torch.float32).double()
    x = acts(257, N, torch.float16, seed=3).to(DEV)
    bias = acts(1, pm.K, torch.float32, seed=4)[0].to(DEV)
    t = x.double() @ W.t() + bias.double()
    g, u = t[:, 0::2], t[:, 1::2]
    ref = (torch.nn.functional.gelu(g, approximate="tanh") if act == "gelu_tanh" else torch.nn.functional.silu(g)) * u
    for kernel, tiles in TOKENS.items():
        for tokens in tiles:
            M = tokens + 1
            for s in (1, 2, 3) if kernel == "rows" else (1,):
                y = gemm_as(pm, x[:M], kernel, tokens, s, bias=bias, out_dtype=torch.float32, act=act)
                assert y.shape == (M, pm.K // 2)
                assert float((y.double() - ref[:M]).norm() / ref[:M].norm()) < 1e-3, (kernel, tokens, s)
                assert torch.equal(y, gemm_as(pm, x[:M], kernel, tokens, s, bias=bias, out_dtype=torch.float32, act=act))
                yh = gemm_as(pm, x[:M], kernel, tokens, s, bias=bias.bfloat16(), out_dtype=torch.bfloat16, act=act)
                assert float((yh.double() - ref[:M]).norm() / ref[:M].norm()) < (4e-3 if M <= 128 or kernel == "rows" else 8e-3)


def test_a_plain_call_is_the_call_its_plan_names():
    """What `ops.gemm` and `ops.linear_act` return is the named kernel's result, over sizes that meet both
    kernels, every token tile and splits."""
    seen = set()
    for case, K, N, vectors in (((F.BLK1632_4, 4, 128, 16), 640, 14336, 1), ((F.BLK1632_4, 4, 128, 16), 14336, 4096, 1),
                                ((F.BLKC, 2, 64, 16), 3072, 4096, 3), ((F.DENSE8, 8, 128, 0), 1024, 5376, 1),
                                ((F.BLK1632_6, 6, 128, 16), 4096, 4096, 1), ((F.BLKC, 3, 128, 10), 6400, 2048, 2)):
        mk = lambda k, s: F.synth_packed(k, N, case[0], case[1], case[2], case[3] or None, seed=s, device=DEV)
        pm = (mk(K, 1) if vectors == 1 else F.fuse_rows([mk(K, 1), mk(K, 2)], interleave=True) if vectors == 2
              else F.fuse_rows([mk(K // 2, 1), mk(K // 4, 2), mk(K // 4, 3)])).to_tiled()
        for M in (9, 40, 64, 90, 128, 200, 333, 500, 1100):
            x = acts(M, N, torch.float16, seed=M).to(DEV)
            plan = gemm_plan(pm, M)
            assert torch.equal(ops.gemm(pm, x), gemm_as(pm, x, *plan)), (case, M, plan)
            seen.add(plan[:2] + (plan[2] > 1,))
            if vectors == 2:
                plan = gemm_plan(pm, M, "silu")
                assert torch.equal(ops.linear_act(pm, x, "silu"), gemm_as(pm, x, *plan, act="silu")), (case, M, plan)
    kinds = {k[:2] for k in seen}
    assert {("rows", 32), ("rows", 64), ("rows", 96), ("tile", 256)} <= kinds and {k[2] for k in seen} == {False, True}, sorted(seen)


@pytest.mark.parametrize("tokens", [64, 128, 256])
@pytest.mark.parametrize("row_tiles,token_tiles,parts,N,runs", [(9, 16, 3, 1536, 2), (10, 16, 3, 1664, 2), (12, 16, 4, 2048, 2),
                                                                (11, 13, 3, 1664, 2), (13, 13, 3, 1664, 2), (13, 15, 4, 4096, 4)])
def test_columns_in_two_unequal_parts(row_tiles, token_tiles, parts, N, runs, tokens):
    """144, 160, 192, 143 and 169 tiles (the last two no multiple of the XCDs) whose plan is three or four parts run as a long and a
    short one, 195 tiles as four equal ones (the last
    tiles ragged on both sides, a padded last chunk of columns).  Operands are rounded to 2^-12 twice: 3e-4, as everywhere on this
    kernel; against the unsplit call only the order of float32 sums differs."""
    K, M = 256 * row_tiles - 7, token_tiles * tokens - 5
    pm = F.synth_packed(K, N, F.BLK1632_4, 4, 128, 16, seed=row_tiles, device=DEV).to_tiled()
    ran, first, rest = column_parts(pm, M, tokens, parts)
    assert ran == runs and ((first > rest) if runs == 2 else (first == rest)), (ran, first, rest)
    x = acts(M, N, torch.float16, seed=tokens).to(DEV)
    y = gemm_as(pm, x, "tile", tokens, parts, out_dtype=torch.float32).double()
    ref = x.double() @ ops.dequant(pm, torch.float32).double().t()
    assert float((y - ref).norm() / ref.norm()) < 5e-4
    one = gemm_as(pm, x, "tile", tokens, out_dtype=torch.float32).double()
    assert float((y - one).norm() / one.norm()) < 1e-5
    assert torch.equal(y, gemm_as(pm, x, "tile", tokens, parts, out_dtype=torch.float32).double())
    bias = acts(1, K, torch.float32, seed=4)[0].to(DEV)
    assert torch.equal(gemm_as(pm, x, "tile", tokens, parts, bias=bias, out_dtype=torch.float32), y.float() + bias)


@pytest.mark.parametrize("tokens", [64, 128, 256])
@pytest.mark.parametrize("K", [256, 260, 262, 263, 129])
def test_rows_of_y_that_start_anywhere(K, tokens):
    """Heights that are multiples of 8, 4, 2 and 1: whole 16-byte pieces, dwords of two outputs, single elements.  Every
    output of a 16-bit call is the float32 call's rounded once."""
    M = tokens + 37
    pm = F.synth_packed(K, 512, F.BLK1632_4, 4, 128, 16, seed=K, device=DEV).to_tiled()
    x = acts(M, 512, torch.float16, seed=tokens).to(DEV)
    y = gemm_as(pm, x, "tile", tokens, out_dtype=torch.float32)
    ref = x.double() @ ops.dequant(pm, torch.float32).double().t()
    assert float((y.double() - ref).norm() / ref.norm()) < 5e-4
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(gemm_as(pm, x, "tile", tokens, out_dtype=dt), y.to(dt)), dt


@pytest.mark.parametrize("half", [256, 260, 262, 263])
def test_halves_that_start_anywhere(half):
    """A gate/up call on the tile kernel leaves its up outputs `half` elements behind its gate outputs.  Each half is the
    plain product of its matrix, bit for bit; the activation of those, rounded once (float32: an exponential and two divisions)."""
    N, M = 512, 293
    rounded = {torch.float16: 1.01 * 2 ** -11, torch.bfloat16: 1.01 * 2 ** -8, torch.float32: 4e-6}   # significands of 11 and 8 bits
    parts = [F.synth_packed(half, N, F.BLK1632_4, 4, 128, 16, seed=half + s, device=DEV) for s in (0, 1)]
    pm = F.fuse_rows(parts, interleave=True).to_tiled()
    x = acts(M, N, torch.float16, seed=half).to(DEV)
    for tokens in TOKENS["tile"]:
        for dt in (torch.float16, torch.bfloat16, torch.float32):
            g, u = (gemm_as(p.to_tiled(), x, "tile", tokens, out_dtype=dt) for p in parts)
            both = torch.stack((g, u), -1).view(M, 2 * half)
            assert torch.equal(gemm_as(pm, x, "tile", tokens, out_dtype=dt), both), (tokens, dt)
            ref = torch.nn.functional.silu(g.double()) * u.double()
            err = (gemm_as(pm, x, "tile", tokens, out_dtype=dt, act="silu").double() - ref).abs()
            assert bool((err <= rounded[dt] * ref.abs() + 1e-7).all()), (tokens, dt)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("at,pitch", [(0, 0), (1, 0), (2, 8), (8, 0), (8, 8), (0, (1 << 22) - 8200), (0, (1 << 22) - 8192)],
                         ids=["as it is", "one element on", "two", "a piece", "a piece and wider", "32-bit offsets end", "and past it"])
def test_y_that_starts_anywhere(dtype, at, pitch):
    """y from any element on, rows any distance apart: the same outputs, and nothing else written.  8192 outputs of 520 tokens
    at strides below and from 4 M elements, where a tile's offsets no longer fit 32 bits."""
    K, N, M = 8192, 512, 520
    pm = F.synth_packed(K, N, F.BLK1632_4, 4, 128, 16, seed=3, device=DEV).to_tiled()
    assert gemm_plan(pm, M)[0] == "tile"
    x = acts(M, N, torch.float16, seed=3).to(DEV)
    ref = ops.gemm(pm, x, out_dtype=dtype)
    ld = K + pitch
    y = torch.full((M * ld + 16,), 7.0, dtype=dtype, device=DEV)
    d, L = pm.desc(), _lib.lib()
    ws = torch.empty(L.cbk_workspace_bytes(ctypes.byref(d), M), dtype=torch.uint8, device=DEV)
    _lib.check(L.cbk_gemm(ctypes.byref(d), x.data_ptr(), F.dtype_code(x.dtype), M, N, y.data_ptr() + at * y.element_size(), F.dtype_code(dtype), ld,
                          None, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "cbk_gemm")
    rows = y[at:at + M * ld].view(M, ld)
    assert torch.equal(rows[:, :K], ref)
    assert bool((rows[:, K:] == 7).all()) and bool((y[:at] == 7).all()) and bool((y[at + M * ld:] == 7).all())
