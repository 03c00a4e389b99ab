"""Each HIP kernel alone against its plain torch reference (tests/ref_ops.py), at sizes other than the engine's."""
import math

import pytest
import torch

from . import ref_ops
from .tiny import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"f32": torch.float32, "bf16": torch.bfloat16}


@pytest.fixture(scope="module")
def ops():
    from trapetum_amd import kernels
    return kernels.load(torch.device(DEV))


def randn(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def tol(dtype):
    return 2e-6 if dtype == torch.float32 else 6e-3


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("m,d,v", [(1, 64, 17), (5, 88, 331), (33, 2304, 1000)])
def test_embed_rows(ops, dt, m, d, v):
    table = randn(v, d, dtype=DT[dt])
    tok = torch.randint(0, v, (m,), dtype=torch.int32, device=DEV)
    got = ops.embed_rows(tok, table, math.sqrt(d))
    assert torch.equal(got.cpu(), ref_ops.embed_rows(tok.cpu(), table.cpu(), math.sqrt(d)))


@pytest.mark.parametrize("din,dout", [("f32", "f32"), ("f32", "bf16"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("m,d", [(1, 16), (3, 88), (7, 2304), (2, 5000)])
def test_rms_norm(ops, din, dout, m, d):
    x = randn(m, d, dtype=DT[din], seed=1, scale=3.0)
    gain = 1.0 + randn(d, seed=2, scale=0.3)
    got = ops.rms_norm(x, gain, 1e-5, DT[dout])
    ref = ref_ops.rms_norm(x.cpu(), gain.cpu(), 1e-5, DT[dout])
    assert rel_l2(got, ref) < tol(DT[dout])


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("post,nxt", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("m,d", [(1, 64), (5, 88), (4, 3584),
                                 # many rows: four elements per lane, one width for each of its forms and their edges
                                 (130, 88), (200, 1000), (150, 2304), (140, 3072), (129, 4608), (130, 8192), (131, 8200), (130, 90),
                                 # few rows of many chunks: a chunk a lane, every form and its edges
                                 (8, 1028), (3, 2304), (64, 2560), (5, 2564), (2, 4096), (7, 4608), (9, 5120), (4, 5124), (6, 8192)])
def test_add_rms_norm(ops, dt, post, nxt, m, d):
    stream = randn(m, d, seed=3, scale=2.0)
    rows = randn(m, d, dtype=DT[dt], seed=4, scale=5.0)
    gp = (1.0 + randn(d, seed=5, scale=0.2)) if post else None
    gn = (1.0 + randn(d, seed=6, scale=0.2)) if nxt else None
    ref_stream = stream.cpu().clone()
    ref = ref_ops.add_rms_norm(ref_stream, rows.cpu(), gp.cpu() if post else None, 1e-6, gn.cpu() if nxt else None, 1e-4, DT[dt])
    got = ops.add_rms_norm(stream, rows, gp, 1e-6, gn, 1e-4, DT[dt])
    assert rel_l2(stream, ref_stream) < 2e-6
    if nxt:
        assert rel_l2(got, ref) < tol(DT[dt])
    else:
        assert got is None


@pytest.mark.parametrize("m,n,k", [(8, 2304, 2048), (3, 600, 9216), (64, 2304, 4096), (700, 2304, 2048), (300, 520, 4104),
                                   (2048, 2304, 4096), (1, 2304, 9216), (2, 601, 14336),
                                   (5, 2304, 9216), (8, 77, 1544), (4, 4608, 4096), (7, 1000, 20000)])
def test_deferred_product_into_add_rms_norm(ops, m, n, k):
    """A product left in K slices and added by add_rms_norm equals the product, then the norm."""
    from trapetum_amd.kernels.ops import SplitRows
    x, w = randn(m, k, dtype=torch.bfloat16, seed=70), randn(n, k, dtype=torch.bfloat16, seed=71, scale=0.05)
    rows = ops.linear(x, w, torch.bfloat16, defer=True)
    assert isinstance(rows, SplitRows) and rows.shape == (m, n) and rows.slices.shape[0] > 1
    ref_rows = x.cpu().double() @ w.cpu().double().T
    assert rel_l2(ops.rows(rows, torch.float32), ref_rows) < 1e-5
    stream = randn(m, n, seed=72)
    gp, gn = 1.0 + randn(n, seed=73, scale=0.2), 1.0 + randn(n, seed=74, scale=0.2)
    ref_stream = stream.cpu().clone()
    ref = ref_ops.add_rms_norm(ref_stream, ref_rows.float(), gp.cpu(), 1e-6, gn.cpu(), 1e-6, torch.float32)
    got = ops.add_rms_norm(stream, rows, gp, 1e-6, gn, 1e-6, torch.bfloat16)
    assert rel_l2(stream, ref_stream) < 1e-5 and rel_l2(got, ref) < 6e-3


# shapes that the tiles of 128 rows and the kernels of few rows would cut in slices, and of which the faster plan makes one
@pytest.mark.parametrize("m,n,k", [(1145, 2304, 2048), (1280, 2304, 2048), (2048, 2304, 2048), (2049, 2048, 2048), (1500, 4096, 2304), (1000, 4608, 2304),
                                   (2500, 1536, 2304), (8, 9216, 2304), (16, 12288, 2304), (64, 9216, 2304), (512, 9216, 2304)])
def test_deferred_product_of_one_slice_keeps_its_sums(ops, m, n, k):
    """What the consumer of a deferred product adds up is float32 whether the plan makes one slice of it or several."""
    x, w = randn(m, k, dtype=torch.bfloat16, seed=76), randn(n, k, dtype=torch.bfloat16, seed=77, scale=0.05)
    rows = ops.linear(x, w, torch.bfloat16, defer=True)
    ref = x.cpu().double() @ w.cpu().double().T
    assert rows.dtype == torch.float32 and rel_l2(ops.rows(rows, torch.float32), ref) < 1e-5


# small matrices at few rows: both sides of where the kernel that streams W takes over from the 8-row kernel (and, at two rows, from
# the multiply-adds, algo 4, where those cut K)
@pytest.mark.parametrize("m,n,k,algo", [(2, 128, 1024, 5), (2, 1024, 2560, 5), (2, 1024, 2624, 4), (2, 1000, 20032, 4), (2, 1025, 7744, 4), (2, 1025, 7808, 16),
                                        (3, 1024, 9216, 5), (3, 1024, 9280, 16), (8, 2048, 2048, 5), (8, 2049, 2048, 16), (5, 4096, 1024, 5), (9, 1024, 2304, 16)])
def test_deferred_product_of_a_small_matrix(ops, m, n, k, algo):
    """Few blocks of 64 rows of W are slower there than a wave for every 2 or 8 of them; the sums stay float32 slices."""
    x, w = randn(m, k, dtype=torch.bfloat16, seed=78), randn(n, k, dtype=torch.bfloat16, seed=79, scale=0.05)
    got = ops.linear(x, w, torch.bfloat16, defer=True)
    ops.force_linear = algo
    try:
        own = ops.linear(x, w, torch.bfloat16, defer=True)
    finally:
        ops.force_linear = 0
    assert got.dtype == torch.float32 and got.slices.shape == own.slices.shape and torch.equal(got.slices, own.slices)
    assert rel_l2(ops.rows(got, torch.float32), x.cpu().double() @ w.cpu().double().T) < 1e-5


def test_rows_wider_than_the_fused_kernel_takes_are_added_first(ops):
    """A product in K slices whose rows are wider than `add_rms_norm` keeps in registers (8192): the slices are added by
    a kernel of their own, in slice order, and the result is what the fused path gives for narrower rows."""
    m, d = 5, 8192 + 8
    slices = randn(3, m, d, seed=70)
    stream = randn(m, d, seed=71)
    gp, gn = randn(d, seed=72).abs() + 0.5, randn(d, seed=73).abs() + 0.5
    ref_stream = stream.cpu().clone()
    ref = ref_ops.add_rms_norm(ref_stream, slices.cpu().sum(0), gp.cpu(), 1e-5, gn.cpu(), 1e-6, torch.bfloat16)
    from trapetum_amd.kernels.ops import SplitRows
    got = ops.add_rms_norm(stream, SplitRows(slices), gp, 1e-5, gn, 1e-6, torch.bfloat16)
    assert rel_l2(stream, ref_stream) < 3e-3 and rel_l2(got, ref) < 6e-3
    summed = ops.rows(SplitRows(slices), torch.float32)
    assert torch.equal(summed.cpu(), (slices[0] + slices[1] + slices[2]).cpu())
    # a product may leave its slices to the consumer only without an epilogue
    x, w = randn(8, 64, dtype=torch.bfloat16, seed=74), randn(128, 64, dtype=torch.bfloat16, seed=75)
    y = torch.empty(8, 128, dtype=torch.float32, device=DEV)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=DEV)
    rc = ops.lib.tp_linear(x.data_ptr(), w.data_ptr(), y.data_ptr(), 1, 0, 8, 128, 64, 1, 30.0, 0, 0, 0.0, 0.0, ws.data_ptr(), 1 << 20, 1, 0, None)
    assert rc != 0 and b"epilogue" in ops.lib.tp_last_error()


def test_gather_rows(ops):
    x = randn(9, 88)
    rows = torch.tensor([8, 0, 3, 3], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.gather_rows(x, rows).cpu(), x.cpu()[[8, 0, 3, 3]])


# ---- matrix products: every kernel, ragged edges -------------------------------------------------------
LINEAR_SHAPES = [(1, 16, 8), (3, 100, 72), (17, 331, 88), (64, 130, 2304), (5, 2304, 2048), (8, 1000, 9216),
                 (65, 200, 136), (300, 257, 520)]


LINEAR_SHAPES += [(65, 100, 64), (300, 257, 576), (1000, 520, 192), (513, 2304, 2048)]
# grids of more than a thousand tiles, which the tiled kernel walks in another order (per XCD, in panels): tile counts
# that are no multiple of 8 and a last panel that is not whole
LINEAR_SHAPES += [(300, 44177, 64), (40, 70001, 72)]


# one and two rows, for the kernel that takes no more: widths of one to ten chunks a lane, an odd number of rows of W
LINEAR_SHAPES += [(1, 77, 8), (2, 301, 1000), (2, 130, 1536), (1, 257, 3584), (2, 99, 4608), (1, 64, 5120)]


# three to eight rows, for the kernel of blocks of 8 rows of W: an N that is no multiple of 8 or 16, a K that ends inside a
# step of 64, inside a wave's quarter and in a second round of loads, every number of rows of X
LINEAR_SHAPES += [(3, 77, 8), (8, 1001, 2304), (7, 130, 2312), (6, 250, 5000), (4, 4099, 600), (5, 9, 9216)]


# nine to 64 rows: every number of 16-row groups of X, an N and a K that end inside a tile and inside a k step, K slices
# whose number a whole number of k steps makes smaller than was asked for
LINEAR_SHAPES += [(9, 77, 64), (33, 1001, 2304), (48, 130, 2312), (64, 250, 5000), (20, 4099, 600), (50, 9, 9216), (16, 64, 72)]


@pytest.mark.parametrize("algo", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11])
@pytest.mark.parametrize("m,n,k", LINEAR_SHAPES)
def test_linear_bf16(ops, algo, m, n, k):
    if algo in (8, 9) and k % 64:
        pytest.skip("the loop that loads straight into LDS takes whole k steps of 64")
    if algo == 2 and m > 64:
        pytest.skip("the skinny kernel takes at most 64 rows")
    if algo == 4 and (m > 2 or k > 5120):
        pytest.skip("the multiply-add kernel takes at most 2 rows and, unsliced, a K of 5120")
    if algo == 5 and m > 8:
        pytest.skip("the kernel of 8-row blocks takes at most 8 rows")
    x, w = randn(m, k, dtype=torch.bfloat16, seed=7), randn(n, k, dtype=torch.bfloat16, seed=8, scale=0.05)
    ops.force_linear = algo
    try:
        got_b = ops.linear(x, w, torch.bfloat16)
        got_f = ops.linear(x, w, torch.float32)
        got_c = ops.linear(x, w, torch.float32, softcap=3.0)
        got_d = ops.rows(ops.linear(x, w, torch.bfloat16, defer=True), torch.float32)      # K slices, where the kernel makes them
    finally:
        ops.force_linear = 0
    ref = x.cpu().double() @ w.cpu().double().T
    assert rel_l2(got_f, ref) < 1e-5
    assert rel_l2(got_b, ref) < 4e-3
    assert rel_l2(got_c, 3.0 * torch.tanh(ref / 3.0)) < 1e-5
    assert rel_l2(got_d, ref) < 4e-3


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("counts,H,KV", [([1, 5, 300, 1], 8, 4), ([290, 1, 2], 4, 2), ([1, 33, 1, 700, 1, 1, 40], 4, 1), ([1, 500], 16, 16)])
def test_attention_of_uneven_sequences(ops, counts, H, KV, shape):
    """Where a step's sequences differ much in length, its blocks go round the chip in another order: every sequence's rows
    are what they are alone, bit for bit (a choice by size may give the short ones other blocks: to rounding)."""
    hd, M = 256, sum(counts)
    q = randn(M, H * hd, dtype=torch.bfloat16, seed=61)
    k, v = randn(M, KV * hd, dtype=torch.bfloat16, seed=62), randn(M, KV * hd, dtype=torch.bfloat16, seed=63)

    def attend(q, k, v, counts, shape):
        cu = torch.tensor([sum(counts[:i]) for i in range(len(counts) + 1)], dtype=torch.int32, device=DEV)
        return ops.attention_prefill(q, k, v, H, KV, hd, cu, max(counts), hd ** -0.5, 30.0, 0, torch.bfloat16, shape=shape)
    got, at = attend(q, k, v, counts, shape), 0
    for n in counts:
        own = attend(q[at:at + n], k[at:at + n], v[at:at + n], [n], shape)
        if shape:
            assert torch.equal(got[at:at + n], own)
        else:
            assert rel_l2(got[at:at + n], own) < 4e-3
        at += n


# portions of long prompts beside single tokens over a paged cache, without and with a ring: one long sequence of four (a
# sequence's streams cover half of the XCDs, all of them, twice that), among three, sixteen and nine, two among six, and steps whose
# plain order already spreads them; the blocks are turned in each of the shapes
@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("counts,held,H,KV,hd", [([1, 1, 1, 700], (150, 611, 48, 900), 8, 4, 256), ([1, 1, 600, 1], (150, 611, 700, 48), 16, 8, 256),
                                                 ([1, 530, 1, 1], (30, 100, 70, 333), 32, 16, 128), ([520, 1, 1], (640, 1, 77), 16, 8, 64),
                                                 ([1] * 15 + [580], tuple(range(20, 36)), 8, 4, 128), ([1] * 8 + [640], (50,) * 9, 8, 1, 192),
                                                 ([300, 1, 1, 350, 1, 1], (500, 9, 8, 130, 6, 5), 4, 2, 64)])
@pytest.mark.parametrize("window,rows_cap", [(0, 0), (190, 256)])
def test_attention_of_uneven_portions_over_a_cache(ops, counts, held, H, KV, hd, shape, window, rows_cap):
    """Every sequence's rows are what they are alone, bit for bit (a choice of the shape by size may give others: to rounding)."""
    n, page = len(counts), 64
    new_len = torch.tensor([a + b for a, b in zip(counts, held)], dtype=torch.int32, device=DEV)
    width = rows_cap // page if rows_cap else -(-int(new_len.max()) // page)
    table = torch.randperm(n * width, generator=torch.Generator().manual_seed(5)).to(torch.int32).view(n, width).to(DEV)
    pools = [randn(n * width, KV, page, hd, dtype=torch.bfloat16, seed=64 + i) for i in range(2)]
    q, k, v = (randn(sum(counts), heads * hd, dtype=torch.bfloat16, seed=66 + i) for i, heads in enumerate((H, KV, KV)))

    def attend(first, last):
        a, b = sum(counts[:first]), sum(counts[:last])
        cu = torch.tensor([sum(counts[first:i]) for i in range(first, last + 1)], dtype=torch.int32, device=DEV)
        return ops.attention_prefill(q[a:b], k[a:b], v[a:b], H, KV, hd, cu, max(counts[first:last]), hd ** -0.5, 30.0, window, torch.bfloat16, shape=shape,
                                     cached=(new_len[first:last], table[first:last], *pools, rows_cap))
    got, at = attend(0, n), 0
    for i, c in enumerate(counts):
        own = attend(i, i + 1)
        if shape:
            assert torch.equal(got[at:at + c], own), i
        else:
            assert rel_l2(got[at:at + c], own) < 4e-3, i
        at += c


# one long sequence first, last and between short ones, so that only the blocks that hold a query are launched: two sequences and as many
# as are packed, more blocks of a sequence than lanes look at once (64, and a cache of many times that before them), a last block of
# one row, a sequence without rows, windows; without a cache and over one; then several long ones, whose blocks come late positions first:
# with as many positions in the cache and with very different ones, and one long one of more blocks than run at once
@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("counts,held,H,KV,hd,window", [([1, 1, 1, 2113], (150, 611, 48, 700), 4, 2, 64, 0), ([2600, 3], (0, 0), 4, 2, 64, 0), ([1] * 11 + [641] + [1] * 12, (77,) * 24, 4, 2, 64, 0),
                                                        ([33, 0, 1500, 7, 64], (0, 0, 0, 0, 0), 2, 2, 256, 0), ([1, 700, 1, 1], (3000, 5000, 40, 3), 4, 1, 256, 400),
                                                        ([5, 1025, 5, 5, 5], (4, 4000, 300, 20, 1), 8, 4, 128, 0),
                                                        ([900, 3, 1100, 5, 1, 0, 4, 6, 33], (0,) * 9, 4, 2, 256, 0), ([700, 3, 650, 64, 1, 2, 4, 6], (5000, 1, 20, 333, 0, 64, 3, 900), 4, 1, 256, 0),
                                                        ([600] + [1] * 21 + [577, 40], (0,) * 12 + (70,) * 12, 2, 1, 192, 100), ([3] * 9 + [2600], (0,) * 10, 32, 16, 256, 0)])
def test_attention_launches_the_blocks_that_hold_queries(ops, counts, held, H, KV, hd, window, shape):
    """Every sequence's rows are what they are alone, bit for bit (a choice of the shape by size may give others: to rounding)."""
    n, page = len(counts), 64
    new_len = torch.tensor([a + b for a, b in zip(counts, held)], dtype=torch.int32, device=DEV)
    width = -(-int(new_len.max()) // page)
    table = torch.randperm(n * width, generator=torch.Generator().manual_seed(6)).to(torch.int32).view(n, width).to(DEV)
    pools = [randn(n * width, KV, page, hd, dtype=torch.bfloat16, seed=70 + i) for i in range(2)]
    q, k, v = (randn(sum(counts), heads * hd, dtype=torch.bfloat16, seed=72 + i) for i, heads in enumerate((H, KV, KV)))

    def attend(first, last):
        a, b = sum(counts[:first]), sum(counts[:last])
        cu = torch.tensor([sum(counts[first:i]) for i in range(first, last + 1)], dtype=torch.int32, device=DEV)
        return ops.attention_prefill(q[a:b], k[a:b], v[a:b], H, KV, hd, cu, max(counts[first:last]), hd ** -0.5, 30.0, window, torch.bfloat16, shape=shape,
                                     cached=(new_len[first:last], table[first:last], *pools, 0) if any(held) else None)
    got, at = attend(0, n), 0
    for i, c in enumerate(counts):
        if c:
            own = attend(i, i + 1)
            if shape:
                assert torch.equal(got[at:at + c], own), i
            else:
                assert rel_l2(got[at:at + c], own) < 4e-3, i      # two shapes' sums, rounded to bfloat16, as above
        at += c


# the kernel that streams up to 64 rows through LDS: each of its blocks (32, 64 and 128 rows of W, up to 16, 32 and 64 of X), one
# k step and fewer than it asks for ahead, an N that ends inside a block and is no multiple of 4 (outputs element by element),
# K slices of which the last is shorter; it is what is chosen from two rows on where the consumer adds the slices of a large matrix
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (2, 77, 128), (3, 2304, 2048), (16, 1001, 320), (17, 8200, 64), (32, 4099, 640),
                                   (33, 130, 1088), (64, 250, 4672), (48, 18432, 64), (9, 18432, 704), (64, 16500, 192), (40, 33000, 512),
                                   (33, 24609, 192), (64, 24610, 64), (40, 32701, 512), (50, 57344, 128)])
def test_linear_up_to_64_rows(ops, m, n, k):
    x, w = randn(m, k, dtype=torch.bfloat16, seed=7), randn(n, k, dtype=torch.bfloat16, seed=8, scale=0.05)
    into = torch.full((m * n + 1,), 7.0, dtype=torch.bfloat16, device=DEV)
    half = n // 2 // 16 * 16
    ops.force_linear = 16
    try:
        got_b = ops.linear(x, w, torch.bfloat16)
        got_f = ops.linear(x, w, torch.float32, softcap=3.0)
        deferred = ops.linear(x, w, torch.bfloat16, defer=True)
        got_d = ops.rows(deferred, torch.float32)
        got_s = ops.linear_act(x, w, torch.float32, "silu", columns=n // 2 or 1)
        ops.linear(x, w, torch.bfloat16, out=into[1:].view(m, n))                         # two bytes beyond an aligned address
        got_g = ops.gated_linear(x, ops.pack_gate_up(w[:half - 3], w[half:2 * half - 3]), half - 3, "silu", torch.bfloat16) if half else None
        with pytest.raises(Exception, match="does not take"):
            ops.linear(x[:, :k - 8].contiguous(), w[:, :k - 8].contiguous(), torch.bfloat16)
    finally:
        ops.force_linear = 0
    if m > 1 and not isinstance(deferred, torch.Tensor):
        assert torch.equal(ops.rows(ops.linear(x, w, torch.bfloat16, defer=True), torch.float32), got_d)
    ref = x.cpu().double() @ w.cpu().double().T
    assert rel_l2(got_b, ref) < 4e-3 and rel_l2(got_d, ref) < 4e-3
    assert rel_l2(got_f, 3.0 * torch.tanh(ref / 3.0)) < 1e-5
    cols = n // 2 or 1
    assert rel_l2(got_s, torch.cat([torch.nn.functional.silu(ref[:, :cols]), ref[:, cols:]], 1)) < 1e-5
    assert torch.equal(into[1:].view(m, n), got_b) and float(into[0]) == 7.0
    if half:
        assert rel_l2(got_g, torch.nn.functional.silu(ref[:, :half - 3]) * ref[:, half:2 * half - 3]) < 4e-3


def test_linear_up_to_64_rows_takes_blocks_of_each_height(ops):
    """The shapes above reach the blocks of 32, 64 and 128 rows of W, the tallest in every form that their test calls."""
    from trapetum_amd.kernels.ops import EPI_GATED, EPI_NONE, EPI_SILU, EPI_SOFTCAP
    rows = ops.lib.tp_linear_stream_rows
    assert rows(64, 16500, 192, EPI_NONE, 0) == 32 and rows(40, 33000, 512, EPI_NONE, 0) == 64 and rows(64, 250, 4672, EPI_NONE, 1) == 64
    for m, n, k in ((33, 24609, 192), (64, 24610, 64), (40, 32701, 512), (50, 57344, 128)):
        assert all(rows(m, n, k, epilogue, 0) == 128 for epilogue in (EPI_NONE, EPI_SOFTCAP, EPI_SILU)) and rows(m, n, k, EPI_NONE, 1) == 128
        assert rows(m, n // 2 // 16 * 32, k, EPI_GATED, 0) == 128
    assert rows(32, 32701, 512, EPI_NONE, 0) == 64 and rows(65, 32701, 512, EPI_NONE, 0) == 0


# blocks of 96 rows of W: the fewest and the most of them, a last one of one row or of rows that no unit has, as many k steps as the ring
# holds and one more, rows of X in each of its two heights
@pytest.mark.parametrize("m,n,k", [(2, 16450, 256), (32, 20449, 320), (33, 16417, 256), (64, 24576, 704), (9, 18432, 1088), (50, 16418, 640)])
def test_linear_blocks_of_96_rows(ops, m, n, k):
    from trapetum_amd.kernels.ops import EPI_GATED, EPI_NONE
    half = n // 2 // 16 * 16
    assert ops.lib.tp_linear_stream_rows(m, n, k, EPI_NONE, 0) == 96 and ops.lib.tp_linear_stream_rows(m, 2 * half, k, EPI_GATED, 0) == 96
    assert ops.lib.tp_linear_stream_rows(m, n, 192, EPI_NONE, 0) == 32
    test_linear_up_to_64_rows(ops, m, n, k)


# the tiles of 8 waves (12: 256 x 256, 13: 256 x 192, 14: 192 x 256, 15: 256 x 128): one k step, two, three and a long odd number
# of them, a tile and one row more or less, an N that is no multiple of 8 or 4 (outputs element by element), a last K slice
# that is shorter, more tiles than CUs
@pytest.mark.parametrize("algo", [12, 13, 14, 15])
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (255, 257, 64), (257, 190, 128), (192, 384, 192), (193, 129, 320), (300, 1001, 1088),
                                   (513, 2304, 2048), (1000, 250, 4672), (2100, 9000, 192)])
def test_linear_wide_tiles(ops, algo, m, n, k):
    x, w = randn(m, k, dtype=torch.bfloat16, seed=7), randn(n, k, dtype=torch.bfloat16, seed=8, scale=0.05)
    into = torch.full((m * n + 1,), 7.0, dtype=torch.bfloat16, device=DEV)
    half = n // 2 // 16 * 16
    ops.force_linear = algo
    try:
        got_b = ops.linear(x, w, torch.bfloat16)
        got_f = ops.linear(x, w, torch.float32, softcap=3.0)
        got_d = ops.rows(ops.linear(x, w, torch.bfloat16, defer=True), torch.float32)
        got_s = ops.linear_act(x, w, torch.float32, "silu", columns=n // 2 or 1)
        ops.linear(x, w, torch.bfloat16, out=into[1:].view(m, n))                         # two bytes beyond an aligned address
        got_g = ops.gated_linear(x, ops.pack_gate_up(w[:half - 3], w[half:2 * half - 3]), half - 3, "silu", torch.bfloat16) if half else None
    finally:
        ops.force_linear = 0
    ref = x.cpu().double() @ w.cpu().double().T
    assert rel_l2(got_b, ref) < 4e-3 and rel_l2(got_d, ref) < 4e-3
    assert rel_l2(got_f, 3.0 * torch.tanh(ref / 3.0)) < 1e-5
    split = n // 2 or 1
    assert rel_l2(got_s, torch.cat([torch.nn.functional.silu(ref[:, :split]), ref[:, split:]], 1)) < 1e-5
    assert torch.equal(into[1:].view(m, n), got_b) and float(into[0]) == 7.0
    if half:
        assert rel_l2(got_g, torch.nn.functional.silu(ref[:, :half - 3]) * ref[:, half:2 * half - 3]) < 4e-3


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("m,n,k", [(1, 16, 8), (8, 2304, 2048), (70, 331, 88), (300, 77, 136)])
def test_linear_with_a_bias(ops, dt, m, n, k):
    """x @ w^T + bias, the bias added by a kernel of its own after whichever product kernel the shape takes."""
    x, w = randn(m, k, dtype=DT[dt], seed=17), randn(n, k, dtype=DT[dt], seed=18, scale=0.05)
    bias = randn(n, seed=19)
    got = ops.linear(x, w, DT[dt], bias=bias)
    ref = x.cpu().double() @ w.cpu().double().T + bias.cpu().double()
    assert got.shape == (m, n) and rel_l2(got, ref) < (2e-6 if dt == "f32" else 4e-3)
    assert rel_l2(ops.linear(x, w, DT[dt], defer=True, bias=bias), ref) < (2e-6 if dt == "f32" else 4e-3)   # never left in slices
    with pytest.raises(Exception, match="bias"):
        ops.linear(x, w, DT[dt], softcap=30.0, bias=bias)
    with pytest.raises(Exception, match="bias"):
        ops.linear(x, w, DT[dt], bias=bias[:-1].contiguous())


@pytest.mark.parametrize("m,n,k", [(1, 16, 8), (3, 100, 71), (70, 331, 88), (5, 700, 2304)])
def test_linear_f32(ops, m, n, k):
    x, w = randn(m, k, seed=9), randn(n, k, seed=10, scale=0.05)
    got = ops.linear(x, w, torch.float32)
    ref = x.cpu().double() @ w.cpu().double().T
    assert rel_l2(got, ref) < 2e-6
    # the sum's order per element does not depend on the other rows: a row alone gives the same bits
    alone = ops.linear(x[m - 1:m].contiguous(), w, torch.float32)
    assert torch.equal(alone[0], got[m - 1])


# one launch: a matrix alone and as many as it takes, matrices of one row, of less than a block and of less than all of its last, with and
# without a bias, both output types, one and two groups of 8 rows a block, a K of one round, of two and of four, the last of them short;
# beside it, what goes product after product (9 rows, a single product whose K is beyond one round, a K beyond all, K no multiple of 8, more matrices)
@pytest.mark.parametrize("m,k,ns", [(1, 8, (1,)), (4, 2304, (2304, 2304, 2304, 2304, 144)), (8, 256, (7, 8, 9, 33, 1, 16, 15, 500)), (3, 1160, (2056, 2048, 20)),
                                    (5, 776, (4097,)), (9, 256, (40, 8)), (2, 2560, (24, 40)), (4, 20, (9, 3)), (8, 64, (8,) * 9),
                                    (1, 2312, (2312, 20)), (8, 4104, (2056, 2048, 9)), (7, 9216, (33, 16)), (3, 9224, (24, 8)), (4, 2568, (40,))])
def test_linear_group(ops, m, k, ns):
    parts = []
    for i, n in enumerate(ns):
        x, w = randn(m, k, dtype=torch.bfloat16, seed=20 + i), randn(n, k, dtype=torch.bfloat16, seed=40 + i, scale=0.05)
        parts.append((x, w, torch.float32 if i % 3 == 1 else torch.bfloat16, randn(n, seed=60 + i) if i % 2 else None))
    for got, (x, w, dtype, bias) in zip(ops.linear_group(parts), parts):
        ref = x.cpu().double() @ w.cpu().double().T + (bias.cpu().double() if bias is not None else 0.0)
        assert got.dtype == dtype and rel_l2(got, ref) < (1e-5 if dtype == torch.float32 else 4e-3)
    turned = range(0, len(ns), 2)                        # through tanh: the bits of the rounded products' own tanh
    for i, (got, plain) in enumerate(zip(ops.linear_group(parts, tanh=turned), ops.linear_group(parts))):
        assert torch.equal(got, ops.unary_(plain, "tanh") if i in turned else plain)
    with pytest.raises(Exception, match="linear_group"):
        ops.linear_group(parts + [(parts[0][0], parts[0][1][:, :-1].contiguous(), torch.bfloat16, None)])
    if m <= 8 and k % 8 == 0 and k <= 2304:
        with pytest.raises(Exception, match="bias"):
            ops.linear_group([(parts[0][0], parts[0][1], torch.bfloat16, torch.zeros(ns[0] + 1, device=DEV))])


# few rows (up to 32) and many, a row tile and one more or less, parts of K that end inside a block of 16 or are empty, a K of one
# piece, K slices for the consumer, two tiles of W a block (from 16384 rows of W on), operands off their 16 bytes
@pytest.mark.parametrize("m,n,k", [(1, 16, 4), (16, 17, 260), (17, 2304, 2048), (32, 33, 2300), (33, 129, 36), (64, 500, 1028), (309, 250, 4100),
                                   (5, 16400, 68), (20, 16390, 84), (70, 200, 71)])
def test_linear_f32_is_one_order(ops, m, n, k):
    x, w = randn(m, k, seed=9), randn(n, k, seed=10, scale=0.05)
    half = n // 2 // 16 * 16
    ref = x.cpu().double() @ w.cpu().double().T
    got = ops.linear(x, w, torch.float32)
    assert rel_l2(got, ref) < 2e-6
    assert rel_l2(ops.linear(x, w, torch.float32, softcap=3.0), 3.0 * torch.tanh(ref / 3.0)) < 2e-6
    # the bits of an element are those of its row alone, of the product left in slices, and of a view that starts anywhere
    row = m // 2
    assert torch.equal(ops.linear(x[row:row + 1].contiguous(), w, torch.float32)[0], got[row])
    assert torch.equal(ops.rows(ops.linear(x, w, torch.float32, defer=True), torch.float32), got)
    off = torch.empty(m * k + 1, device=DEV)[1:].view(m, k)
    off.copy_(x)
    assert torch.equal(ops.linear(off, w, torch.float32), got)
    if half > 3:
        packed = ops.pack_gate_up(w[:half - 3], w[half:2 * half - 3])
        gated = ops.gated_linear(x, packed, half - 3, "silu", torch.float32, limit=2.0, up_shift=0.5)
        g, u = ref[:, :half - 3].clamp(max=2.0), ref[:, half:2 * half - 3].clamp(-2.0, 2.0)
        assert rel_l2(gated, torch.nn.functional.silu(g) * (u + 0.5)) < 5e-6
        assert torch.equal(ops.gated_linear(x[row:row + 1].contiguous(), packed, half - 3, "silu", torch.float32, limit=2.0, up_shift=0.5)[0], gated[row])
        assert torch.equal(ops.gated_linear(off, packed, half - 3, "silu", torch.float32, limit=2.0, up_shift=0.5), gated)


@pytest.mark.parametrize("m,n,k", [(1, 16, 4), (17, 33, 260), (33, 129, 36), (70, 200, 2304), (309, 250, 1028)])
def test_linear_f32_bits_do_not_depend_on_where_operands_lie(ops, m, n, k):
    def off(t, by):
        room = torch.empty(t.numel() + by, device=DEV)[by:].view(t.shape)
        return room.copy_(t)
    x, w = randn(m, k, seed=11), randn(n, k, seed=12, scale=0.05)
    got = ops.linear(x, w, torch.float32)
    half = n // 2 // 16 * 16
    for i, j in ((1, 0), (0, 2), (3, 1)):
        assert torch.equal(ops.linear(off(x, i), off(w, j), torch.float32), got)
        assert torch.equal(ops.rows(ops.linear(off(x, i), off(w, j), torch.float32, defer=True), torch.float32), got)
        if half:
            packed = ops.pack_gate_up(w[:half], w[half:2 * half])
            assert torch.equal(ops.gated_linear(off(x, i), off(packed, j), half, "silu", torch.float32), ops.gated_linear(x, packed, half, "silu", torch.float32))


# up to 32 rows on 16 bytes: rings that wrap and rings with fewer steps than places, a step that ends in the next part, empty waves,
# W's last tile and a gated tile's second half, slices for the consumer, two tiles of W a block; the order is that of operands off 16
# bytes, whose kernel holds no ring
@pytest.mark.parametrize("m,n,k", [(1, 7, 4), (3, 96, 9216), (4, 2304, 2048), (15, 100, 1028), (16, 64, 3620), (17, 48, 2304), (31, 16402, 260), (32, 130, 1500),
                                   (2, 8208, 1100)])
def test_linear_f32_ring(ops, m, n, k):
    def off(t):
        return torch.empty(t.numel() + 1, device=DEV)[1:].view(t.shape).copy_(t)
    x, w = randn(m, k, seed=13), randn(n, k, seed=14, scale=0.05)
    got = ops.linear(x, w, torch.float32)
    assert rel_l2(got, x.cpu().double() @ w.cpu().double().T) < 2e-6
    assert torch.equal(ops.linear(off(x), w, torch.float32), got)
    assert torch.equal(ops.rows(ops.linear(x, w, torch.float32, defer=True), torch.float32), got)
    half = n // 2 // 16 * 16
    if half:
        packed = ops.pack_gate_up(w[:half - 5], w[half:2 * half - 5])
        gated = ops.gated_linear(x, packed, half - 5, "gelu_tanh", torch.float32)
        assert torch.equal(ops.gated_linear(off(x), packed, half - 5, "gelu_tanh", torch.float32), gated)


def test_linear_f32_off_16_bytes_takes_more_rows_than_a_launch(ops):
    m, n, k = 65535 * 32 + 21, 5, 4
    x, w = torch.empty(m * k + 1, device=DEV)[1:].view(m, k).normal_(), randn(n, k, seed=12)
    got = ops.linear(x, w, torch.float32)
    some = [0, 31, 65535 * 32 - 1, 65535 * 32, m - 1]
    assert torch.equal(got, ops.linear(x.clone(), w, torch.float32))
    assert rel_l2(got[some], x[some].cpu().double() @ w.cpu().double().T) < 2e-6


@pytest.mark.parametrize("algo", [1, 2, 3, 4, 5, 6, 8, 10, 11])
@pytest.mark.parametrize("dt", ["bf16", "f32"])
@pytest.mark.parametrize("m,inter,k", [(1, 16, 16), (4, 200, 88), (40, 320, 96), (9, 1000, 2304), (150, 72, 136),
                                       (150, 72, 128), (700, 1000, 320), (130, 36010, 64), (2, 1000, 2304), (1, 75, 4608),
                                       (8, 9216, 2304), (3, 41, 2504), (7, 8, 520), (64, 9216, 2304), (33, 1000, 200),
                                       (17, 41, 2504), (48, 8, 520)])
def test_gated_linear(ops, algo, dt, m, inter, k):
    if dt == "f32" and algo != 1:
        pytest.skip("float32 runs on the plain kernel only")
    if algo == 4 and m > 2:
        pytest.skip("the multiply-add kernel takes at most 2 rows")
    if algo == 5 and m > 8:
        pytest.skip("the kernel of 8-row blocks takes at most 8 rows")
    if algo == 2 and m > 64:
        pytest.skip("the skinny kernel takes at most 64 rows")
    if algo in (8, 9) and k % 64:
        pytest.skip("the loop that loads straight into LDS takes whole k steps of 64")
    wg, wu = randn(inter, k, dtype=DT[dt], seed=11, scale=0.2), randn(inter, k, dtype=DT[dt], seed=12, scale=0.2)
    x = randn(m, k, dtype=DT[dt], seed=13)
    packed = ops.pack_gate_up(wg, wu)
    assert torch.equal(packed.cpu(), ref_ops.pack_gate_up(wg.cpu(), wu.cpu()))
    ops.force_linear = algo
    try:
        got = ops.gated_linear(x, packed, inter, "gelu_tanh", DT[dt])
        silu = ops.gated_linear(x, packed, inter, "silu", DT[dt])
        relu = ops.gated_linear(x, packed, inter, "relu", DT[dt])
        with pytest.raises(Exception, match="no kernel"):
            ops.gated_linear(x, packed, inter, "softsign", DT[dt])
    finally:
        ops.force_linear = 0
    g, u = x.cpu().double() @ wg.cpu().double().T, x.cpu().double() @ wu.cpu().double().T
    ref = torch.nn.functional.gelu(g, approximate="tanh") * u
    assert rel_l2(got, ref) < (5e-6 if dt == "f32" else 4e-3)
    assert rel_l2(silu, torch.nn.functional.silu(g) * u) < (5e-6 if dt == "f32" else 4e-3)      # the other activations offered
    assert rel_l2(relu, torch.relu(g) * u) < (5e-6 if dt == "f32" else 4e-3)


@pytest.mark.parametrize("algo,m", [(2, 8), (3, 8), (3, 200), (5, 8), (5, 3)])
def test_gated_linear_at_the_ends_of_the_activation(ops, algo, m):
    """Gate values far out on both sides (the activation is the identity on one, zero on the other): no overflow of the
    exponential shows in the result."""
    k, inter = 64, 96
    wg, wu = randn(inter, k, dtype=torch.bfloat16, seed=14), randn(inter, k, dtype=torch.bfloat16, seed=15, scale=0.2)
    x = randn(m, k, dtype=torch.bfloat16, seed=16)
    x[::2] *= 1.0e4
    x[1::4] *= 1.0e15
    ops.force_linear = algo
    try:
        got = ops.gated_linear(x, ops.pack_gate_up(wg, wu), inter, "gelu_tanh", torch.float32)
    finally:
        ops.force_linear = 0
    g, u = x.cpu().double() @ wg.cpu().double().T, x.cpu().double() @ wu.cpu().double().T
    ref = torch.nn.functional.gelu(g, approximate="tanh") * u
    assert torch.isfinite(got).all()
    assert rel_l2(got, ref) < 1e-5


# ---- RoPE + cache write, attention over pages --------------------------------------------------------------
def build_cache_case(dt, H, KV, hd, lens, page, rows_cap, n_pages, seed):
    """Random q/k/v rows for sequences of the given lengths, pushed through rope_kv_write of the reference."""
    m = sum(lens)
    q = randn(m, H * hd, dtype=dt, seed=seed)
    k = randn(m, KV * hd, dtype=dt, seed=seed + 1)
    v = randn(m, KV * hd, dtype=dt, seed=seed + 2)
    row_seq = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32)
    row_pos = torch.cat([torch.arange(n) for n in lens]).to(torch.int32)
    new_len = torch.tensor(lens, dtype=torch.int32)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    perm = torch.randperm(n_pages, generator=torch.Generator().manual_seed(seed)).tolist()
    width = max(-(-(min(n, rows_cap) if rows_cap else n) // page) for n in lens)
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    for i, n in enumerate(lens):
        need = -(-(min(n, rows_cap) if rows_cap else n) // page)
        for j in range(need):
            table[i, j] = perm.pop()
    inv_freq = (1.0 / (10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd)))
    return dict(q=q, k=k, v=v, row_seq=row_seq, row_pos=row_pos, new_len=new_len, cu=cu, table=table, inv_freq=inv_freq)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd,lens,page,rows_cap", [
    (4, 2, 16, (5, 11, 17), 16, 0), (6, 1, 32, (1, 9, 23, 40), 16, 16), (3, 3, 48, (70, 3), 64, 64),
    (8, 4, 256, (130,), 64, 0), (2, 2, 80, (33, 50), 16, 32), (4, 2, 64, (200, 90), 16, 0), (5, 1, 32, (300,), 16, 64),
    (2, 2, 80, (150, 140), 16, 0), (8, 4, 256, (300, 77), 64, 128)])
def test_rope_kv_write(ops, dt, H, KV, hd, lens, page, rows_cap):
    c = build_cache_case(DT[dt], H, KV, hd, lens, page, rows_cap, 24, 20)
    rot = hd if hd != 80 else 48                            # one head size with a rotation over part of the head
    c["inv_freq"] = c["inv_freq"][:rot // 2].contiguous()
    pools_ref = [torch.zeros(24, KV, page, hd, dtype=DT[dt]) for _ in range(2)]
    pools = [p.to(DEV) for p in pools_ref]
    q_ref, k_ref = c["q"].cpu().clone(), c["k"].cpu().clone()
    ref_ops.rope_kv_write(q_ref, k_ref, c["v"].cpu(), H, KV, hd, c["inv_freq"], rot, c["row_seq"], c["row_pos"],
                          c["new_len"], c["table"], pools_ref[0], pools_ref[1], rows_cap)
    ops.rope_kv_write(c["q"], c["k"], c["v"], H, KV, hd, c["inv_freq"].to(DEV), rot, c["row_seq"].to(DEV),
                      c["row_pos"].to(DEV), c["new_len"].to(DEV), c["table"].to(DEV), pools[0], pools[1], rows_cap)
    t = 3e-6 if dt == "f32" else 6e-3
    assert rel_l2(c["q"], q_ref) < t and rel_l2(c["k"], k_ref) < t
    assert rel_l2(pools[0], pools_ref[0]) < t
    assert torch.equal(pools[1].cpu(), pools_ref[1])
    # rows that no sequence owns stay untouched
    assert torch.equal((pools[0].cpu() != 0).any(dim=-1), (pools_ref[0] != 0).any(dim=-1))


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd,lens,page,rows_cap,rot", [
    (4, 2, 16, (5, 11, 17), 16, 0, 16), (2, 2, 80, (33, 50), 16, 32, 48), (8, 4, 256, (300, 77), 64, 128, 256),
    (3, 1, 64, (290,), 16, 0, 32)])
def test_rope_kv_write_turning_neighbours(ops, dt, H, KV, hd, lens, page, rows_cap, rot):
    """The other pairing: elements 2d and 2d + 1 turn together by the angle of pair d; few rows and many, a rotation over
    part of the head, a ring."""
    c = build_cache_case(DT[dt], H, KV, hd, lens, page, rows_cap, 24, 21)
    inv_freq = (1.0 / (10000.0 ** (torch.arange(0, rot, 2, dtype=torch.float32) / rot)))
    pools_ref = [torch.zeros(24, KV, page, hd, dtype=DT[dt]) for _ in range(2)]
    pools = [p.to(DEV) for p in pools_ref]
    q_ref, k_ref = c["q"].cpu().clone(), c["k"].cpu().clone()
    halves = c["q"].cpu().clone()
    ref_ops.rope_kv_write(q_ref, k_ref, c["v"].cpu(), H, KV, hd, inv_freq, rot, c["row_seq"], c["row_pos"],
                          c["new_len"], c["table"], pools_ref[0], pools_ref[1], rows_cap, pairing="neighbours")
    ref_ops.rope_kv_write(halves, None, None, H, KV, hd, inv_freq, rot, c["row_seq"], c["row_pos"], c["new_len"], c["table"],
                          None, None, rows_cap)
    assert rel_l2(halves, q_ref) > 0.1                       # the two pairings are not the same rotation
    ops.rope_kv_write(c["q"], c["k"], c["v"], H, KV, hd, inv_freq.to(DEV), rot, c["row_seq"].to(DEV),
                      c["row_pos"].to(DEV), c["new_len"].to(DEV), c["table"].to(DEV), pools[0], pools[1], rows_cap,
                      pairing="neighbours")
    t = 3e-6 if dt == "f32" else 6e-3
    assert rel_l2(c["q"], q_ref) < t and rel_l2(c["k"], k_ref) < t
    assert rel_l2(pools[0], pools_ref[0]) < t
    assert torch.equal(pools[1].cpu(), pools_ref[1])
    with pytest.raises(Exception, match="pairing"):
        ops.rope_kv_write(c["q"], c["k"], c["v"], H, KV, hd, inv_freq.to(DEV), rot, c["row_seq"].to(DEV),
                          c["row_pos"].to(DEV), c["new_len"].to(DEV), c["table"].to(DEV), pools[0], pools[1], rows_cap,
                          pairing="thirds")


ATTN_CASES = [
    # H, KV, hd, lens, page, window, rows_cap, cap
    (4, 2, 16, (5, 11, 17), 16, 8, 16, 50.0),
    (6, 1, 32, (1, 9, 23, 40), 16, 16, 16, 20.0),
    (3, 3, 48, (70, 3), 16, 5, 16, 8.0),
    (8, 4, 256, (130, 64), 64, 0, 0, 50.0),
    (8, 4, 256, (200,), 64, 100, 128, 0.0),
    (2, 2, 80, (33, 50), 16, 0, 0, 0.0),
    (16, 2, 128, (300, 17, 129), 64, 0, 0, 30.0),
    (32, 1, 64, (90,), 16, 0, 0, 0.0),
]


@pytest.mark.parametrize("kernel", ["plain", 0, 1, 2, 3])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd,lens,page,window,rows_cap,cap", ATTN_CASES)
def test_attention_prefill(ops, kernel, dt, H, KV, hd, lens, page, window, rows_cap, cap):
    """kernel: the plain one, or the matrix-core kernel with its block shape (0: its own choice)."""
    plain = kernel == "plain"
    if dt == "f32" and not plain:
        pytest.skip("float32 runs on the plain kernel only")
    c = build_cache_case(DT[dt], H, KV, hd, lens, page, rows_cap, 24, 30)
    scale = 1.0 / math.sqrt(hd * 0.7)
    ref = ref_ops.attention_prefill(c["q"].cpu(), c["k"].cpu(), c["v"].cpu(), H, KV, hd, c["cu"], max(lens), scale,
                                    cap, window, torch.float32)
    ops.force_plain_attention = plain
    try:
        got = ops.attention_prefill(c["q"], c["k"], c["v"], H, KV, hd, c["cu"].to(DEV), max(lens), scale, cap, window,
                                    DT[dt], row_seq=c["row_seq"].to(DEV), row_pos=c["row_pos"].to(DEV),
                                    shape=0 if plain else kernel)
    finally:
        ops.force_plain_attention = False
    assert rel_l2(got, ref) < (3e-6 if dt == "f32" else 8e-3)


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("H,KV,hd,lens,window,cap", [(64, 8, 16, (450, 130, 64), 100, 30.0), (8, 4, 256, (3300,), 0, 50.0),
                                                    (8, 4, 256, (1000, 77), 300, 0.0), (12, 4, 128, (700, 1), 0, 30.0),
                                                    (6, 2, 80, (333,), 64, 0.0), (4, 4, 48, (97, 300), 0, 20.0)])
def test_attention_prefill_many_tiles(ops, shape, H, KV, hd, lens, window, cap):
    """Steps of many and of few query tiles in every block shape of the kernel (column groups that are heads of a kv
    head or further positions; one, two or four groups of keys), against dense masked attention per sequence and
    head."""
    m, g, scale = sum(lens), H // KV, 1.0 / math.sqrt(hd * 0.7)
    q, k, v = (randn(m, n * hd, dtype=torch.bfloat16, seed=40 + i) for i, n in enumerate((H, KV, KV)))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    ref = torch.zeros(m, H, hd)
    for i, n in enumerate(lens):
        rows = slice(int(cu[i]), int(cu[i + 1]))
        qs, ks, vs = (t.cpu().float()[rows].reshape(n, -1, hd) for t in (q, k, v))
        pos = torch.arange(n)
        hidden = (pos[None, :] > pos[:, None]) | ((pos[:, None] - pos[None, :] >= window) if window else False)
        for h in range(H):
            s = qs[:, h] @ ks[:, h // g].T * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            ref[rows, h] = torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1) @ vs[:, h // g]
    got = ops.attention_prefill(q, k, v, H, KV, hd, cu.to(DEV), max(lens), scale, cap, window, torch.bfloat16, shape=shape)
    assert rel_l2(got.reshape(m, H, hd), ref) < 8e-3


EXTEND_CASES = [
    # H, KV, hd, lens, starts (what the cache already holds), page, window, rows_cap, cap
    (4, 2, 16, (25, 11, 17), (20, 0, 16), 16, 8, 16, 50.0),
    (6, 1, 32, (50, 9, 23, 40), (17, 8, 0, 1), 16, 16, 16, 20.0),         # a ring without a row to spare
    (3, 3, 48, (70, 3), (64, 2), 16, 5, 16, 8.0),
    (8, 4, 256, (330, 64), (130, 63), 64, 0, 0, 50.0),
    (8, 4, 256, (700,), (451,), 64, 128, 128, 0.0),                       # the portion is longer than the ring
    (2, 2, 80, (33, 50), (0, 31), 16, 0, 0, 0.0),
    (16, 2, 128, (1300, 17, 129), (1234, 0, 128), 64, 512, 512, 30.0),
    (32, 1, 64, (90,), (89,), 16, 0, 0, 0.0),
    # portions of hundreds of rows, which the rotation and cache write take 16 bytes at a time
    (8, 4, 256, (700, 300), (300, 20), 64, 0, 0, 50.0),
    (4, 2, 64, (600,), (200,), 16, 128, 128, 30.0),
]


@pytest.mark.parametrize("kernel", ["plain", 0, 1, 2, 3])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd,lens,starts,page,window,rows_cap,cap", EXTEND_CASES)
def test_attention_over_cached_positions_and_the_steps_rows(ops, kernel, dt, H, KV, hd, lens, starts, page, window, rows_cap, cap):
    """A step that continues sequences by several tokens: the queries attend over the cached positions, read in place
    through the page table (a ring's rows too), and over the step's own rows, which are cached only afterwards.
    Against whole-sequence attention of the reference; afterwards the cache holds what a whole-sequence step would
    have left.  kernel: the plain one, or the matrix-core kernel with its block shape (0: its own choice)."""
    plain = kernel == "plain"
    if dt == "f32" and not plain:
        pytest.skip("float32 runs on the plain kernel only")
    n_pages = 64
    c = build_cache_case(DT[dt], H, KV, hd, lens, page, rows_cap, n_pages, 50)
    scale = 1.0 / math.sqrt(hd * 0.9)
    q_ref, k_ref = c["q"].cpu().clone(), c["k"].cpu().clone()
    pools_ref = [torch.zeros(n_pages, KV, page, hd, dtype=DT[dt]) for _ in range(2)]
    ref_ops.rope_kv_write(q_ref, k_ref, c["v"].cpu(), H, KV, hd, c["inv_freq"], hd, c["row_seq"], c["row_pos"],
                          c["new_len"], c["table"], pools_ref[0], pools_ref[1], rows_cap)
    ref = ref_ops.attention_prefill(q_ref, k_ref, c["v"].cpu(), H, KV, hd, c["cu"], max(lens), scale, cap, window, torch.float32)
    # what earlier steps left: positions below `starts`, written as one step per sequence set
    pools = [torch.full((n_pages, KV, page, hd), 7.0, dtype=DT[dt], device=DEV) for _ in range(2)]
    first = torch.cat([torch.arange(int(c["cu"][i]), int(c["cu"][i]) + s) for i, s in enumerate(starts)]).long()
    if first.numel():
        ops.rope_kv_write(c["q"][first.to(DEV)].contiguous(), c["k"][first.to(DEV)].contiguous(), c["v"][first.to(DEV)].contiguous(),
                          H, KV, hd, c["inv_freq"].to(DEV), hd, c["row_seq"][first].to(DEV), c["row_pos"][first].to(DEV),
                          torch.tensor(starts, dtype=torch.int32, device=DEV), c["table"].to(DEV), pools[0], pools[1], rows_cap)
    # the step: positions starts[i] .. lens[i] - 1 of every sequence
    counts = [n - s for n, s in zip(lens, starts)]
    rows = torch.cat([torch.arange(int(c["cu"][i]) + s, int(c["cu"][i + 1])) for i, s in enumerate(starts)]).long()
    q, k, v = (c[name][rows.to(DEV)].contiguous() for name in ("q", "k", "v"))
    cu = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=DEV)
    row_seq, row_pos, new_len, table = (c[name].to(DEV) for name in ("row_seq", "row_pos", "new_len", "table"))
    row_seq, row_pos = row_seq[rows.to(DEV)].contiguous(), row_pos[rows.to(DEV)].contiguous()
    ops.force_plain_attention = plain
    try:
        ops.rope_kv_write(q, k, v, H, KV, hd, c["inv_freq"].to(DEV), hd, row_seq, row_pos, new_len, table, pools[0], pools[1],
                          rows_cap, write=False)
        before = [p.clone() for p in pools]
        got = ops.attention_prefill(q, k, v, H, KV, hd, cu, max(counts), scale, cap, window, DT[dt],
                                    row_seq=row_seq, row_pos=row_pos, cached=(new_len, table, pools[0], pools[1], rows_cap),
                                    shape=0 if plain else kernel)
        assert all(torch.equal(a, b) for a, b in zip(before, pools))       # neither the rotation nor the attention cached anything
        ops.kv_write(k, v, KV, hd, row_seq, row_pos, new_len, table, pools[0], pools[1], rows_cap)
    finally:
        ops.force_plain_attention = False
    assert rel_l2(got, ref[rows]) < (3e-6 if dt == "f32" else 8e-3)
    worst = max(rel_l2(got[i], ref[rows][i]) for i in range(0, len(rows), max(1, len(rows) // 50)))
    assert worst < (1e-5 if dt == "f32" else 3e-2)
    # the cache afterwards: every row a whole-sequence step writes holds the same values
    written = (pools_ref[0] != 0).any(dim=-1)
    t = 3e-6 if dt == "f32" else 6e-3
    assert rel_l2(pools[0].cpu()[written], pools_ref[0][written]) < t
    assert torch.equal(pools[1].cpu()[written], pools_ref[1][written])
    assert bool((pools[0].cpu()[~written] == 7.0).all())


@pytest.mark.parametrize("plain", [True, False])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd,lens,page,window,rows_cap,cap", ATTN_CASES)
def test_attention_decode(ops, plain, dt, H, KV, hd, lens, page, window, rows_cap, cap):
    if dt == "f32" and not plain:
        pytest.skip("float32 runs on the plain kernel only")
    n_pages = 24
    c = build_cache_case(DT[dt], H, KV, hd, lens, page, rows_cap, n_pages, 40)
    pools_ref = [torch.zeros(n_pages, KV, page, hd, dtype=DT[dt]) for _ in range(2)]
    # stale rows of an earlier occupant must not leak: fill the pools with large values first
    for p in pools_ref:
        p.fill_(7.0)
    ref_ops.rope_kv_write(c["q"].cpu().clone(), c["k"].cpu().clone(), c["v"].cpu(), H, KV, hd, None, 0, c["row_seq"],
                          c["row_pos"], c["new_len"], c["table"], pools_ref[0], pools_ref[1], rows_cap)
    qlast = torch.stack([c["q"].cpu()[int(c["cu"][i + 1]) - 1] for i in range(len(lens))]).contiguous()
    scale = 1.0 / math.sqrt(hd * 1.3)
    ref = ref_ops.attention_decode(qlast, H, KV, hd, c["new_len"], c["table"], pools_ref[0], pools_ref[1], rows_cap, scale,
                                   cap, window, torch.float32)
    ops.force_plain_attention = plain
    try:
        got = ops.attention_decode(qlast.to(DEV), H, KV, hd, c["new_len"].to(DEV), c["table"].to(DEV),
                                   pools_ref[0].to(DEV), pools_ref[1].to(DEV), rows_cap, scale, cap, window, DT[dt],
                                   max_keys=max(lens))
        if not plain:
            for splits in (1, 2, 5):
                again = ops.attention_decode(qlast.to(DEV), H, KV, hd, c["new_len"].to(DEV), c["table"].to(DEV),
                                             pools_ref[0].to(DEV), pools_ref[1].to(DEV), rows_cap, scale, cap, window,
                                             DT[dt], max_keys=max(lens), splits=splits)
                assert rel_l2(again, ref) < 8e-3, splits
    finally:
        ops.force_plain_attention = False
    assert rel_l2(got, ref) < (3e-6 if dt == "f32" else 8e-3)


CHUNK_CASES = [
    # H, KV, hd, lens, page, chunk, window, rows_cap, cap
    (4, 2, 16, (5, 41, 17), 16, 20, 0, 0, 0.0),             # chunks that end inside a tile of keys
    (6, 3, 64, (130, 64, 65), 64, 64, 0, 64, 0.0),          # a ring of one chunk
    (8, 2, 128, (300, 99), 16, 100, 30, 0, 25.0),           # a window inside the chunk, capped scores
    (2, 2, 48, (70,), 16, 1, 0, 16, 0.0),                   # a chunk of one position: the query's own key and the sink
    (3, 1, 80, (33, 200), 16, 1000, 0, 0, 0.0),             # a chunk longer than every sequence
    (16, 4, 256, (257, 31), 64, 96, 0, 0, 0.0),
]


_chunk_refs = {}


def chunk_case(dt, case):
    """The inputs of a case and what the slow functions make of them, computed once for all kernels."""
    if (dt, case) not in _chunk_refs:
        H, KV, hd, lens, page, chunk, window, rows_cap, cap = case
        n_pages = 32
        c = build_cache_case(DT[dt], H, KV, hd, lens, page, rows_cap, n_pages, 50)
        scale = 1.0 / math.sqrt(hd * 0.6)
        temp = (0.5 + torch.rand(H, generator=torch.Generator().manual_seed(5))).float()
        sink = randn(H, seed=6).cpu().float() * 2.0
        more = dict(chunk=chunk, head_scale=temp, sink=sink)
        ref = ref_ops.attention_prefill(c["q"].cpu(), c["k"].cpu(), c["v"].cpu(), H, KV, hd, c["cu"], max(lens), scale,
                                        cap, window, torch.float32, **more)
        pools = [torch.full((n_pages, KV, page, hd), 7.0, dtype=DT[dt]) for _ in range(2)]
        ref_ops.rope_kv_write(c["q"].cpu().clone(), c["k"].cpu().clone(), c["v"].cpu(), H, KV, hd, None, 0, c["row_seq"],
                              c["row_pos"], c["new_len"], c["table"], pools[0], pools[1], rows_cap)
        qlast = torch.stack([c["q"].cpu()[int(c["cu"][i + 1]) - 1] for i in range(len(lens))]).contiguous()
        ref_one = ref_ops.attention_decode(qlast, H, KV, hd, c["new_len"], c["table"], pools[0], pools[1], rows_cap, scale,
                                           cap, window, torch.float32, **more)
        bare = ref_ops.attention_decode(qlast, H, KV, hd, c["new_len"], c["table"], pools[0], pools[1], rows_cap, scale,
                                        cap, window, torch.float32, chunk=chunk, head_scale=temp)
        assert rel_l2(bare, ref_one) > 0.01                 # the sink is no small matter in these cases
        _chunk_refs[(dt, case)] = (c, scale, temp, sink, ref, pools, qlast, ref_one)
    return _chunk_refs[(dt, case)]


@pytest.mark.parametrize("kernel", ["plain", 0, 1, 2, 3])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("case", CHUNK_CASES)
def test_attention_in_chunks_with_temperatures_and_sinks(ops, kernel, dt, case):
    """Keys of the query's own chunk only, a factor per head on the scores, a score without key that joins the sum: in
    the plain kernels and the matrix-core kernels, many queries and one, the keys of one query in slices too."""
    plain = kernel == "plain"
    if dt == "f32" and not plain:
        pytest.skip("float32 runs on the plain kernel only")
    H, KV, hd, lens, page, chunk, window, rows_cap, cap = case
    c, scale, temp, sink, ref, pools, qlast, ref_one = chunk_case(dt, case)
    dev = dict(chunk=chunk, head_scale=temp.to(DEV), sink=sink.to(DEV))
    tol = 3e-6 if dt == "f32" else 8e-3
    ops.force_plain_attention = plain
    try:
        got = ops.attention_prefill(c["q"], c["k"], c["v"], H, KV, hd, c["cu"].to(DEV), max(lens), scale, cap, window,
                                    DT[dt], row_seq=c["row_seq"].to(DEV), row_pos=c["row_pos"].to(DEV),
                                    shape=0 if plain else kernel, **dev)
        assert rel_l2(got, ref) < tol
        if kernel in ("plain", 0):
            for splits in (None,) if plain else (None, 1, 2, 5):
                one = ops.attention_decode(qlast.to(DEV), H, KV, hd, c["new_len"].to(DEV), c["table"].to(DEV),
                                           pools[0].to(DEV), pools[1].to(DEV), rows_cap, scale, cap, window, DT[dt],
                                           max_keys=max(lens), splits=splits, **dev)
                assert rel_l2(one, ref_one) < tol, splits
    finally:
        ops.force_plain_attention = False


@pytest.mark.parametrize("splits", [None, 1, 3])
@pytest.mark.parametrize("slices", [0, 1, 3])
@pytest.mark.parametrize("H,KV,hd,lens,page,window,rows_cap,cap", ATTN_CASES)
def test_attention_decode_step(ops, splits, slices, H, KV, hd, lens, page, window, rows_cap, cap):
    """Rotation, cache write and attention of a decode step in one launch, against the three reference parts.  The
    cache holds every earlier position; the step's projections come as bf16 rows (slices 0) or as float32 K slices."""
    from trapetum_amd.kernels.ops import SplitRows
    n_pages, n = 24, len(lens)
    c = build_cache_case(torch.bfloat16, H, KV, hd, lens, page, rows_cap, n_pages, 70)
    rot = hd if hd != 80 else 48                            # one case with a rotation over part of the head
    inv_freq = c["inv_freq"][:rot // 2].contiguous()
    pools_ref = [torch.full((n_pages, KV, page, hd), 7.0, dtype=torch.bfloat16) for _ in range(2)]
    earlier = c["row_pos"] < (c["new_len"][c["row_seq"].long()] - 1)          # all rows but each sequence's last
    keep = earlier.nonzero().flatten()
    ref_ops.rope_kv_write(c["q"].cpu()[keep].clone(), c["k"].cpu()[keep].clone(), c["v"].cpu()[keep], H, KV, hd, inv_freq, rot,
                          c["row_seq"][keep], c["row_pos"][keep], c["new_len"] - 1, c["table"], pools_ref[0], pools_ref[1], rows_cap)
    pools = [p.to(DEV) for p in pools_ref]
    last = torch.tensor([int(c["cu"][i + 1]) - 1 for i in range(n)])
    qkv = torch.cat([c["q"].cpu()[last], c["k"].cpu()[last], c["v"].cpu()[last]], dim=1).float()
    if slices:
        parts = torch.randn(slices, *qkv.shape, generator=torch.Generator().manual_seed(71))
        parts[0] += qkv - parts.sum(0)
        given, summed = SplitRows(parts.contiguous().to(DEV)), parts[0].clone()
        for sl in range(1, slices):
            summed += parts[sl]
    else:
        given, summed = qkv.to(torch.bfloat16).to(DEV), qkv.to(torch.bfloat16).float()
    scale = 1.0 / math.sqrt(hd * 1.3)
    ref = ref_ops.attention_decode_step(summed, H, KV, hd, inv_freq, rot, c["new_len"], c["table"], pools_ref[0], pools_ref[1],
                                        rows_cap, scale, cap, window, torch.float32)
    if not ops.fuses_decode_step(torch.bfloat16, H, KV, hd, pools[0]):
        assert H // KV > 16
        pytest.skip("more than 16 query heads per kv head run on the separate kernels")
    got = ops.attention_decode_step(given, H, KV, hd, inv_freq.to(DEV), rot, c["new_len"].to(DEV), c["table"].to(DEV),
                                    pools[0], pools[1], rows_cap, scale, cap, window, torch.bfloat16, max_keys=max(lens),
                                    splits=splits)
    assert rel_l2(got, ref) < 8e-3
    assert rel_l2(pools[0], pools_ref[0]) < 6e-3 and rel_l2(pools[1], pools_ref[1]) < 6e-3
    assert torch.equal((pools[0].cpu() != 7.0).any(dim=-1), (pools_ref[0] != 7.0).any(dim=-1))      # no other row touched
    # queries only, on a cache that another run filled: the pools stay as they are
    before = [p.clone() for p in pools]
    got_q = ops.attention_decode_step(given.slices[..., :H * hd].contiguous() if slices else given[:, :H * hd].contiguous(),
                                      H, KV, hd, inv_freq.to(DEV), rot, c["new_len"].to(DEV), c["table"].to(DEV),
                                      pools[0], pools[1], rows_cap, scale, cap, window, torch.bfloat16, max_keys=max(lens),
                                      write_kv=False, splits=splits) if not slices else None
    if got_q is not None:
        assert rel_l2(got_q, ref) < 8e-3
        assert torch.equal(before[0], pools[0]) and torch.equal(before[1], pools[1])


# launches of many rows that see few keys, which a wave a row works on: prompts that end inside a group of keys, at one and after
# the eighth, decode steps, a window over a long prompt, chunks; and rows that see more keys than the caller's bound says
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd", [(8, 2, 48), (8, 8, 100), (8, 4, 256), (8, 2, 300), (8, 4, 520)])
def test_plain_attention_of_many_rows_with_few_keys(ops, dt, H, KV, hd):
    lens = ([1, 2, 3, 4, 5, 8, 9, 31, 32, 33] * 40)[:400 if hd > 256 else 120]
    M, seqs = sum(lens), len(lens)
    q, k, v = (randn(M, heads * hd, dtype=DT[dt], seed=84 + i) for i, heads in enumerate((H, KV, KV)))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    seq = torch.repeat_interleave(torch.arange(seqs, dtype=torch.int32), torch.tensor(lens))
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens])
    bias, sink, temp = randn(H, 12, seed=87), randn(H, seed=88), (0.5 + torch.rand(H)).to(DEV)

    def run(a, b, cu, seq, pos, most, **more):
        return ops.attention_prefill(q[a:b], k[a:b], v[a:b], H, KV, hd, cu.to(DEV), most, hd ** -0.5, 20.0, more.pop("window", 0), DT[dt],
                                     row_seq=seq.to(DEV), row_pos=pos.to(DEV), **more)
    ops.force_plain_attention = True
    try:
        for more in ({}, dict(window=5), dict(window=6, keep=2, sink=sink), dict(chunk=7, head_scale=temp),
                     dict(by_position=ops.ByPosition(temperature=(0.3, 4), bias=bias))):
            got = run(0, M, cu, seq, pos, 33, **more)
            for s in range(0, seqs, 13 if seqs > 13 else 1):      # a sequence alone: few rows, which blocks work on
                a, b = int(cu[s]), int(cu[s + 1])
                own = run(a, b, torch.tensor([0, b - a], dtype=torch.int32), torch.zeros(b - a, dtype=torch.int32), pos[a:b], 1000, **more)
                assert torch.equal(got[a:b], own), (s, more)
        one, whole = torch.tensor([0, M], dtype=torch.int32), (torch.zeros(M, dtype=torch.int32), torch.arange(M, dtype=torch.int32))
        assert torch.equal(run(0, M, one, *whole, 1), run(0, M, one, *whole, 10 ** 6))      # a bound that is too small costs time alone
        few = run(0, M, one, *whole, 10 ** 6, window=40)
        for r in range(0, M, 97):
            a = max(0, r - 39)
            own = ops.attention_prefill(q[a:r + 1], k[a:r + 1], v[a:r + 1], H, KV, hd, torch.tensor([0, r + 1 - a], dtype=torch.int32, device=DEV), 1000,
                                        hd ** -0.5, 20.0, 40, DT[dt], row_seq=torch.zeros(r + 1 - a, dtype=torch.int32, device=DEV),
                                        row_pos=torch.arange(r + 1 - a, dtype=torch.int32, device=DEV))[-1]
            assert torch.equal(few[r], own), r
        n, page = 300, 16
        pools = [randn(n, KV, page, hd, dtype=DT[dt], seed=90 + i) for i in range(2)]
        held, table = torch.arange(n, dtype=torch.int32, device=DEV) % page + 1, torch.arange(n, dtype=torch.int32, device=DEV).view(n, 1)
        step = lambda a, b, most: ops.attention_decode(q[a:b], H, KV, hd, held[a:b], table[a:b], *pools, 0, hd ** -0.5, 20.0, 0, DT[dt], max_keys=most)
        together = step(0, n, page if hd <= 256 else 4)
        assert all(torch.equal(together[r:r + 1], step(r, r + 1, 1000)) for r in range(0, n, 7))
    finally:
        ops.force_plain_attention = False


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,KV,hd", [(2, 1, 64), (2, 2, 300), (1, 1, 520)])
def test_plain_attention_with_hidden_groups_and_infinite_values(ops, dt, H, KV, hd):
    """A bias of minus infinity hides whole groups of keys, a wave's first ones among them; a value of infinity at the query's
    own position comes out as infinity in its element and nowhere else."""
    n, reach = 131, 140
    q, k = randn(n, H * hd, dtype=DT[dt], seed=80), randn(n, KV * hd, dtype=DT[dt], seed=81)
    v = randn(n, KV * hd, dtype=DT[dt], seed=82)
    bias = randn(H, reach + 1, seed=83).float()
    bias[:, 60:87] = bias[:, 30:34] = bias[:, 97:127] = -math.inf
    cu = torch.tensor([0, n], dtype=torch.int32)
    args = (H, KV, hd, cu, n, hd ** -0.5, 20.0, 0)
    more = dict(row_seq=torch.zeros(n, dtype=torch.int32), row_pos=torch.arange(n, dtype=torch.int32))
    ref = ref_ops.attention_prefill(q.cpu(), k.cpu(), v.cpu(), *args, torch.float32, **more, by_position=ref_ops.ByPosition(bias=bias.cpu()))
    dev = dict((name, t.to(DEV)) for name, t in more.items())
    ops.force_plain_attention = True
    try:
        run = lambda v: ops.attention_prefill(q, k, v, H, KV, hd, cu.to(DEV), *args[4:], DT[dt], **dev, by_position=ops.ByPosition(bias=bias))
        got = run(v)
        v[100, 3] = math.inf
        last = run(v)[100].float()
    finally:
        ops.force_plain_attention = False
    assert rel_l2(got, ref) < (3e-6 if dt == "f32" else 8e-3)
    of_head = [h * hd + 3 for h in range(H) if h // (H // KV) == 0]
    assert all(float(last[c]) == math.inf for c in of_head)
    rest = [c for c in range(H * hd) if c not in of_head]
    assert torch.equal(last[rest], got[100].float()[rest])


@pytest.mark.parametrize("H,KV,hd,n,long,others", [(8, 4, 256, 64, 5000, 37), (4, 2, 64, 96, 2500, 70), (16, 16, 128, 17, 3001, 5), (8, 4, 256, 64, 120, 90)])
def test_attention_decode_of_one_long_sequence_among_short_ones(ops, H, KV, hd, n, long, others):
    """The slices are counted for the longest sequence: every sequence's result is that of its own keys."""
    page, lens = 64, [others - i % 3 for i in range(n)]
    lens[n // 3] = long
    pages = [-(-x // page) for x in lens]
    pools = [randn(sum(pages), KV, page, hd, dtype=torch.bfloat16, seed=94 + i) for i in range(2)]
    table = torch.zeros(n, max(pages), dtype=torch.int32)
    for i, c in enumerate(pages):
        table[i, :c] = torch.arange(sum(pages[:i]), sum(pages[:i]) + c)
    q, held = randn(n, H * hd, dtype=torch.bfloat16, seed=96), torch.tensor(lens, dtype=torch.int32)
    got = ops.attention_decode(q, H, KV, hd, held.to(DEV), table.to(DEV), *pools, 0, hd ** -0.5, 30.0, 0, torch.bfloat16, max_keys=long)
    some = [0, n // 3, n - 1]
    ref = ref_ops.attention_decode(q.cpu()[some], H, KV, hd, held[some], table[some], *[p.cpu() for p in pools], 0, hd ** -0.5, 30.0, 0, torch.float32)
    assert (ops.decode_splits(n, KV, hd, long) > 1) == (long > 128)
    assert all(rel_l2(got[s], ref[i]) < 8e-3 for i, s in enumerate(some))
    alone = ops.attention_decode(q[:1], H, KV, hd, held[:1].to(DEV), table[:1].to(DEV), *pools, 0, hd ** -0.5, 30.0, 0, torch.bfloat16, max_keys=lens[0])
    assert rel_l2(got[:1], alone) < 8e-3


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("H,KV,hd", [(8, 4, 256), (3, 3, 64), (8, 2, 96), (16, 2, 240), (2, 2, 16)])
def test_attention_decode_of_few_keys_in_one_launch(ops, H, KV, hd, fused):
    """Up to WHOLE_KEYS keys a block has them all: at and beside a tile's, a page's, a round's and the launch's last key, behind a
    window, in a ring; fused, the new token's row of the cache holds NaN until the launch writes it.  bfloat16 probabilities are not
    rounded, so the result is off by the rounding of queries, keys and outputs: 2^-8 each at most, 2^-8 (1 + 1 / sqrt(hd)) in norm."""
    lens, page = (1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 177, 191, 192), 64
    n, width = len(lens), (H + 2 * KV) * hd
    inv_freq = (10000.0 ** (-torch.arange(hd // 2).float() / (hd // 2))).contiguous()
    for window, rows_cap in ((0, 0), (100, 0), (100, 128)):
        per = 2 if rows_cap else 3
        table = torch.randperm(n * per, generator=torch.Generator().manual_seed(7)).to(torch.int32).view(n, per)
        pools = [randn(n * per, KV, page, hd, dtype=torch.bfloat16, seed=30 + i).cpu() for i in range(2)]
        held = torch.tensor(lens, dtype=torch.int32)
        rows = randn(n, width, dtype=torch.bfloat16, seed=33).cpu()
        if fused:
            ref = ref_ops.attention_decode_step(rows.float(), H, KV, hd, inv_freq, hd, held, table, pools[0].clone(), pools[1].clone(), rows_cap,
                                                hd ** -0.5, 30.0, window, torch.float32)
            for i, l in enumerate(lens):
                r = (l - 1) % rows_cap if rows_cap else l - 1
                for p in pools:
                    p[int(table[i, r // page]), :, r % page] = math.nan
        else:
            ref = ref_ops.attention_decode(rows[:, :H * hd].contiguous(), H, KV, hd, held, table, pools[0], pools[1], rows_cap, hd ** -0.5, 30.0, window, torch.float32)
        dev = [p.to(DEV) for p in pools]
        common = (held.to(DEV), table.to(DEV), *dev, rows_cap, hd ** -0.5, 30.0, window, torch.bfloat16)
        assert ops._decode_slices(None, n, KV, H, hd, max(lens)) == 0
        if fused:
            got = ops.attention_decode_step(rows.to(DEV), H, KV, hd, inv_freq.to(DEV), hd, *common, max_keys=max(lens))
            assert all(bool(torch.isfinite(p.float()).all()) for p in dev)
        else:
            got = ops.attention_decode(rows[:, :H * hd].contiguous().to(DEV), H, KV, hd, *common, max_keys=max(lens))
        assert rel_l2(got, ref) < 2 ** -8 * (1 + hd ** -0.5) + 2e-3, (window, rows_cap)


def test_attention_far_key_stands_out(ops):
    """One key among hundreds carries the answer: its score is made to dominate, so a kernel that drops
    or misplaces it (a chunk boundary, a page boundary) returns another value row."""
    H, KV, hd, n, page = 4, 2, 64, 700, 64
    for target in (0, 63, 64, 333, 699):
        c = build_cache_case(torch.bfloat16, H, KV, hd, (n,), page, 0, 16, 50 + target)
        k = c["k"].cpu().float().reshape(n, KV, hd) * 0.05
        q = torch.zeros(1, H, hd)
        q[0, :, :] = k[target, :, :].repeat_interleave(H // KV, dim=0) * 4000.0
        pools = [torch.zeros(16, KV, page, hd, dtype=torch.bfloat16) for _ in range(2)]
        kb = k.reshape(n, KV * hd).to(torch.bfloat16)
        ref_ops.rope_kv_write(torch.zeros(n, H * hd, dtype=torch.bfloat16), kb, c["v"].cpu(), H, KV, hd, None, 0,
                              c["row_seq"], c["row_pos"], c["new_len"], c["table"], pools[0], pools[1], 0)
        qb = q.reshape(1, H * hd).to(torch.bfloat16)
        for plain in (True, False):
            ops.force_plain_attention = plain
            try:
                got = ops.attention_decode(qb.to(DEV), H, KV, hd, c["new_len"].to(DEV), c["table"].to(DEV),
                                           pools[0].to(DEV), pools[1].to(DEV), 0, 1.0, 0.0, 0, torch.bfloat16, max_keys=n,
                                           splits=None if plain else 1 + target % 7)
            finally:
                ops.force_plain_attention = False
            want = c["v"].cpu().float().reshape(n, KV, hd)[target].repeat_interleave(H // KV, dim=0).reshape(1, H * hd)
            assert rel_l2(got, want) < 2e-2, (target, plain)


@pytest.mark.parametrize("window,rows_cap,lens", [(4096, 4096, (5000, 4100, 4096, 9000)), (0, 0, (5000, 8191, 63, 64)),
                                                  (1000, 1024, (1000, 1001, 3333, 2048))])
def test_attention_decode_long_contexts(ops, window, rows_cap, lens):
    """Thousands of keys at the 2B head size: rings that have wrapped once and twice, a window shorter than its ring,
    lengths at and beside a page's end, pages scattered over the pool, and every way of cutting the keys into slices."""
    H, KV, hd, page, scale, cap = 8, 4, 256, 64, 1 / 16.0, 50.0
    g = torch.Generator().manual_seed(5)
    n = len(lens)
    per = [-(-(min(l, rows_cap) if rows_cap else l) // page) for l in lens]
    n_pages = sum(per) + 3
    kp, vp = (torch.zeros(n_pages, KV, page, hd, dtype=torch.bfloat16) for _ in range(2))
    free = torch.randperm(n_pages, generator=g).tolist()
    table = torch.full((n, max(per)), -1, dtype=torch.int32)
    q = (torch.randn(n, H, hd, generator=g) * 0.5).to(torch.bfloat16)
    ref = torch.zeros(n, H, hd)
    for i, l in enumerate(lens):
        table[i, :per[i]] = torch.tensor([free.pop() for _ in range(per[i])], dtype=torch.int32)
        k = (torch.randn(l, KV, hd, generator=g) * 0.5).to(torch.bfloat16)
        v = torch.randn(l, KV, hd, generator=g).to(torch.bfloat16)
        kept = torch.arange(max(0, l - rows_cap) if rows_cap else 0, l)            # what the ring still holds
        rows = kept % rows_cap if rows_cap else kept
        pages = table[i].long()[rows // page]
        kp[pages, :, rows % page] = k[kept]
        vp[pages, :, rows % page] = v[kept]
        lo = max(0, l - window) if window else 0
        scores = torch.einsum("tgd,gqd->gqt", k[lo:].float(), q[i].float().reshape(KV, H // KV, hd)) * scale
        weights = torch.softmax(cap * torch.tanh(scores / cap), dim=-1)
        ref[i] = torch.einsum("gqt,tgd->gqd", weights, v[lo:].float()).reshape(H, hd)
    for splits in (None, 1, 7, 33, 128):
        got = ops.attention_decode(q.reshape(n, H * hd).to(DEV), H, KV, hd, torch.tensor(lens, dtype=torch.int32, device=DEV),
                                   table.to(DEV), kp.to(DEV), vp.to(DEV), rows_cap, scale, cap, window, torch.bfloat16,
                                   max_keys=max(lens), splits=splits)
        assert rel_l2(got.reshape(n, H, hd), ref) < 8e-3, splits


def test_argmax_ties_and_nan(ops):
    z = torch.full((3, 7001), -1.0)
    z[0, 100] = z[0, 7000] = 5.0               # tie: the smaller index wins (runtime/src/bin/opt_check.rs:37-65)
    z[1, 7000] = 2.0
    z[2, 0] = float("nan")
    z[2, 5] = 0.5
    assert ops.argmax(z.to(DEV)).tolist() == [100, 7000, 5]
    big = randn(5, 256000, seed=60)
    assert ops.argmax(big).tolist() == big.cpu().argmax(dim=-1).tolist()


# ---- token choice ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("vocab,temperature,top_k,top_p", [(256, 0.7, 256, 0.95), (7001, 1.0, 40, 1.0), (7001, 0.3, 1000, 0.5),
                                                           (256000, 0.9, 256, 0.95), (513, 1.5, 1, 1.0), (513, 0.8, 600, 0.99), (513, 0.8, 0, 1.0),
                                                           (50001, 1.2, 0, 1.0)])
def test_sample_follows_the_plain_sampler(ops, vocab, temperature, top_k, top_p):
    """Sort by logit (ties: smaller id), keep top_k, softmax at the temperature, shortest prefix reaching top_p, walk
    with u (runtime/src/bin/serve.rs:41-72).  Ties and a dominant token are planted; where the uniform number falls
    within float32 rounding of a boundary of the walk either neighbour is right."""
    rows = 6
    z = randn(rows, vocab, seed=80, scale=3.0).cpu()
    z[1, 5] = z[1, 77] = z[1].max() + 1.0                    # a tie at the top
    z[2, vocab - 1] = z[2].max() + 30.0                      # one token takes all the mass
    u = torch.tensor([0.0, 0.5, 0.999, 0.25, 0.75, 0.9999], dtype=torch.float32)
    with pytest.raises(Exception, match="top_k"):            # the kernel sorts at most 1024 candidates and says so
        ops.sample(z.to(DEV), temperature, 2000, top_p, u.to(DEV))
    with pytest.raises(Exception, match="nucleus"):          # the whole vocabulary (top_k 0) goes without a nucleus
        ops.sample(z.to(DEV), temperature, 0, 0.9, u.to(DEV))
    got = ops.sample(z.to(DEV), temperature, top_k, top_p, u.to(DEV)).cpu().tolist()
    for b in range(rows):
        choices = set()
        for du in (-2e-6, 0.0, 2e-6):
            ub = min(max(float(u[b]) + du, 0.0), 0.9999999)
            choices.add(int(ref_ops.sample(z[b:b + 1], temperature, top_k, top_p, torch.tensor([ub]))[0]))
        assert got[b] in choices, (b, got[b], choices)
    assert got[2] == vocab - 1


@pytest.mark.parametrize("vocab", [32768, 50001])
@pytest.mark.parametrize("top_k", [1, 300, 1024])
def test_sample_in_turn_on_one_workspace(ops, vocab, top_k):
    """What the candidate filter leaves behind is ready for the next call: rows with few candidates, with more than are sorted
    at once, with more than a block or the list holds (the whole row is read then), one after the other."""
    flat = torch.zeros(3, vocab)                             # every logit in one bin
    flat[:, 7] = 5.0
    crowd = randn(3, vocab, seed=91, scale=0.01).cpu()       # thousands of logits in the bins of the largest
    steep = randn(3, vocab, seed=92, scale=4.0).cpu()
    u = torch.tensor([0.1, 0.6, 0.95], dtype=torch.float32)
    for z in (steep, flat, steep, crowd, flat, steep):
        got = ops.sample(z.to(DEV), 0.9, top_k, 0.97, u.to(DEV)).cpu().tolist()
        for b in range(3):
            near = {int(ref_ops.sample(z[b:b + 1], 0.9, top_k, 0.97, torch.tensor([min(max(float(u[b]) + du, 0.0), 0.9999999)]))[0])
                    for du in (-2e-6, 0.0, 2e-6)}            # float32 rounding at a boundary of the walk
            assert got[b] in near, (b, got[b], near)


def could_be_drawn(z, temperature, top_k, top_p, u, token, off=1e-5):
    """Whether `token` is the draw from one row, or its neighbour where u or top_p lies within `off` of a boundary of the cumulative sums
    (the kernel's, in float32, are chains of at most 40 + 16 + 64 additions: 120 2^-24 = 7e-6, and the exponentials' last places)."""
    z = z.double()
    order = torch.sort(z, descending=True, stable=True).indices[:top_k] if top_k else torch.arange(len(z))
    cum = torch.softmax(z[order] / temperature, 0).cumsum(0)
    at = int((order == token).nonzero()[0]) if bool((order == token).any()) else None
    for p in (top_p - off, top_p + off):
        keep = min(int((cum < p).sum()), len(cum) - 1) if top_k else len(cum) - 1
        r = u * float(cum[keep])
        if at is not None and at <= keep and (float(cum[at - 1]) if at else 0.0) - off <= r < float(cum[at]) + off:
            return True
        if at == 0 and r >= float(cum[keep]) - off:          # rounding left the walk without a hit: the first candidate
            return True
    return False


# numbers that come with the launch and numbers on the device; candidates of one wave, of two, of all sixteen, of more than the block
# sorts at once (few different logits: a bin of many, and ties that the smaller id wins), the whole vocabulary
@pytest.mark.parametrize("rows", [1, 5, 64])
@pytest.mark.parametrize("vocab,top_k,levels", [(300, 40, 0), (40000, 1, 0), (40000, 100, 0), (256000, 256, 0), (33000, 1024, 0), (50000, 700, 37), (40000, 0, 0), (90, 90, 5)])
def test_sample_takes_its_numbers_from_host_and_device(ops, rows, vocab, top_k, levels):
    z = randn(rows, vocab, seed=80, scale=2.0)
    if levels:
        z = torch.round(z * (levels / 12.0)) * (12.0 / levels)
    top_p = 0.9 if top_k else 1.0
    u = torch.rand(rows, generator=torch.Generator().manual_seed(81))
    device = ops.sample(z, 0.8, top_k, top_p, u.to(DEV))
    assert torch.equal(ops.sample(z, 0.8, top_k, top_p, u.tolist()), device)
    zc = z.cpu()
    for i in range(rows):
        assert could_be_drawn(zc[i], 0.8, top_k, top_p, float(u[i]), int(device[i])), i
    with pytest.raises(Exception, match="uniform"):
        ops.sample(z, 0.8, top_k, top_p, u.tolist() + [0.5])
    with pytest.raises(Exception, match="at most"):
        ops.sample(z[:1].expand(65, -1).contiguous(), 0.8, top_k, top_p, [0.5] * 65)


def test_recent_push(ops):
    """A row's id goes to the place its cursor names, the cursor moves on and wraps at the ring's end."""
    ring = torch.full((3, 5), -1, dtype=torch.int32, device=DEV)
    cursor = torch.tensor([0, 4, 2], dtype=torch.int32, device=DEV)
    ops.recent_push(torch.tensor([7, 8, 9], dtype=torch.int32, device=DEV), ring, cursor)
    ops.recent_push(torch.tensor([1, 2, 3], dtype=torch.int32, device=DEV), ring, cursor)
    assert ring.cpu().tolist() == [[7, 1, -1, -1, -1], [2, -1, -1, -1, 8], [-1, -1, 9, 3, -1]]
    assert cursor.cpu().tolist() == [2, 1, 4]


@pytest.mark.parametrize("vocab,window", [(256, 8), (256000, 128)])
def test_repetition_penalty(ops, vocab, window):
    """Each distinct recent token once: z / penalty if z > 0 else z * penalty (runtime/src/bin/serve.rs:1330-1340)."""
    z = randn(3, vocab, seed=81, scale=2.0)
    recent = torch.full((3, window), -1, dtype=torch.int32)
    recent[0, :4] = torch.tensor([3, 3, 9, vocab - 1])       # a token twice in the window is penalised once
    recent[1, :] = torch.arange(window) * 2 % vocab
    ref = z.cpu().clone()
    ref_ops.apply_repetition_penalty(ref, recent, 1.3)
    ops.apply_repetition_penalty(z, recent.to(DEV), 1.3)
    assert torch.allclose(z.cpu(), ref, rtol=1e-6, atol=0)
    untouched = z.cpu().clone()
    ops.apply_repetition_penalty(z, recent.to(DEV), 1.0)     # 1.0 switches it off
    assert torch.equal(z.cpu(), untouched)


@pytest.mark.parametrize("kind", ["capped", "narrow", "levels", "nan", "masked", "sorted", "lowest"])
def test_sample_by_groups_is_the_sampler_alone(ops, kind):
    """Sampling over the groups' largest keys against the same call without a workspace, which reads whole rows by one block each: the
    same tokens, at the smallest row that is cut into groups, groups of 2 to 128, either number of them, and lists that overflow."""
    for rows, vocab in ((2, 8192), (3, 8195), (1, 20480), (3, 32000), (2, 100001), (2, 262144), (1, 262145), (1, 300001)):
        z = torch.randn(rows, vocab, generator=torch.Generator().manual_seed(vocab)) * 2.0
        if kind == "capped": z = 30.0 * torch.tanh(z / 30.0)
        if kind == "narrow": z = z * 0.05 + 100.0
        if kind == "levels": z = torch.round(z * 2.0) / 2.0
        if kind == "nan": z[:, ::7], z[:, 5], z[-1, 11] = math.nan, -math.inf, math.inf
        if kind == "masked": z[:, vocab // 3:] = -math.inf
        if kind == "sorted": z = torch.sort(z, dim=1, descending=True).values.contiguous()
        if kind == "lowest": z[:, 40:] = torch.finfo(torch.float32).min
        z, u = z.to(DEV), torch.rand(rows, generator=torch.Generator().manual_seed(3)).to(DEV)
        for top_k, top_p in ((0, 1.0), (1, 0.9), (256, 0.95), (512, 1.0), (513, 0.95), (1024, 1.0)):
            alone = torch.empty(rows, dtype=torch.int32, device=DEV)
            assert ops.lib.tp_sample(z.data_ptr(), rows, vocab, 0.8, top_k, top_p, u.data_ptr(), alone.data_ptr(), None, ops._stream()) == 0
            assert torch.equal(ops.sample(z, 0.8, top_k, top_p, u), alone), (rows, vocab, top_k)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("M", [1, 5, 40, 300])
@pytest.mark.parametrize("hd,rot,turn,rows_cap", [(128, 64, 128, 0), (64, 64, 32, 0), (96, 16, 48, 128), (24, 24, 6, 0)])
def test_values_turned_with_queries_and_keys(ops, hd, rot, turn, rows_cap, M, dt):
    """Values that turn in the launch that turns queries and keys: the bits of a launch of their own before it, in the step's rows and in
    the cache, at few rows (a block a head), some (several heads a block) and many (a block a row), with and without the write."""
    H, KV, page = 6, 2, 64
    rows = randn(M, (H + 2 * KV) * hd, dtype=DT[dt], seed=11)
    freq, v_freq = ((100.0 ** (-torch.arange(n // 2).float() / (n // 2))).contiguous().to(DEV) for n in (rot, turn))
    cut = M // 3
    row_seq = torch.tensor([0] * cut + [1] * (M - cut), dtype=torch.int32, device=DEV)
    row_pos = torch.tensor(list(range(7, 7 + cut)) + list(range(M - cut)), dtype=torch.int32, device=DEV)
    new_len = torch.tensor([7 + cut, M - cut], dtype=torch.int32, device=DEV)
    pages = -(-(rows_cap or 310) // page)
    table = torch.arange(2 * pages, dtype=torch.int32, device=DEV).view(2, pages)
    for write in (True, False):
        got = []
        for together in (True, False):
            t = rows.clone()
            q, k, v = t[:, :H * hd], t[:, H * hd:(H + KV) * hd], t[:, (H + KV) * hd:]
            pools = [torch.full((2 * pages, KV, page, hd), 7.0, dtype=DT[dt], device=DEV) for _ in range(2)]
            if not together:
                ops.rope_kv_write(v, None, None, KV, 0, hd, v_freq, turn, row_seq, row_pos, new_len, None, None, None, 0, write=False)
            ops.rope_kv_write(q, k, v, H, KV, hd, freq, rot, row_seq, row_pos, new_len, table, *pools, rows_cap, write=write,
                              **(dict(value_freq=v_freq) if together else {}))
            got.append([t] + pools)
        assert all(torch.equal(a, b) for a, b in zip(*got)), write
        assert bool((got[0][2] != 7.0).any()) == write
    with pytest.raises(Exception, match="values that turn"):
        ops.rope_kv_write(q, None, None, H, 0, hd, freq, rot, row_seq, row_pos, new_len, None, None, None, 0, write=False, value_freq=v_freq)
