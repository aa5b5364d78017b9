"""Each HIP kernel alone against a plain float32 torch formula of the same
operation, at sizes other than the engine tests use."""
import math

import pytest
import torch

import plain_llama
from host_launches import TILES

pytestmark = pytest.mark.gpu

DT = [torch.float32, torch.bfloat16]
IDS = ["fp32", "bf16"]


def tol(dtype):
    return dict(atol=2e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)


@pytest.fixture(scope="module")
def ops(gpu_device):
    from pytriton_llama_amd import ops
    return ops


@pytest.mark.parametrize("dtype", DT, ids=IDS)
def test_embedding(ops, dtype):
    table = torch.randn(301, 72, device="cuda").to(dtype)
    ids = torch.tensor([0, 300, 5, 5, 17], dtype=torch.int32, device="cuda")
    assert torch.equal(ops.embedding(table, ids), table[ids.long()])


def test_stage_step(ops):
    """The tables of a replayed step go from pinned host memory to the device buffer by a
    kernel; tokens that are still on the device take their places among them."""
    host = torch.arange(1000, 1000 + 777, dtype=torch.int32).pin_memory()
    dev = torch.zeros(777, dtype=torch.int32, device="cuda")
    ops.stage_step(dev, host)
    assert torch.equal(dev.cpu(), host)
    tokens = torch.tensor([7, 8, 9, 10], dtype=torch.int32, device="cuda")
    host[:] = torch.arange(777, dtype=torch.int32)
    ops.stage_step(dev, host, tokens, 300, 3)
    want = host.clone()
    want[300:303] = torch.tensor([7, 8, 9], dtype=torch.int32)
    assert torch.equal(dev.cpu(), want)
    with pytest.raises(ops.KernelError):
        ops.stage_step(dev, torch.zeros(777, dtype=torch.int32))          # not pinned
    with pytest.raises(ops.KernelError):
        ops.stage_step(dev, host, tokens, 775, 4)                         # past the end


@pytest.mark.parametrize("dtype", DT, ids=IDS)
@pytest.mark.parametrize("shape", [(5, 72), (3, 2048), (2, 5000), (1, 16),
                                   (513, 328), (515, 2048), (600, 3072), (517, 4096)])
def test_add_rmsnorm(ops, dtype, shape):
    torch.manual_seed(0)
    x = torch.randn(shape, device="cuda").to(dtype)
    r = torch.randn(shape, device="cuda").to(dtype)
    w = (1 + 0.1 * torch.randn(shape[1], device="cuda")).float()
    eps = 1e-3
    want_y, want_r = plain_llama.add_rms_norm(x.float().cpu(), r.float().cpu(), w.cpu(), eps)
    res = r.clone()
    y = ops.add_rmsnorm(x, res, w, eps)
    torch.testing.assert_close(y.float().cpu(), want_y, **tol(dtype))
    torch.testing.assert_close(res.float().cpu(), want_r.to(dtype).float(), atol=0, rtol=0)
    # without a residual: the input stays what it is
    x2 = x.clone()
    y2 = ops.add_rmsnorm(x2, None, w, eps)
    torch.testing.assert_close(y2.float().cpu(), plain_llama.rms_norm(x.float().cpu(), w.cpu(), eps),
                               **tol(dtype))
    assert torch.equal(x2, x)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
def test_silu_mul(ops, dtype):
    torch.manual_seed(1)
    gu = (3 * torch.randn(7, 2 * 200, device="cuda")).to(dtype)
    want = plain_llama.silu(gu[:, :200].float()) * gu[:, 200:].float()
    torch.testing.assert_close(ops.silu_mul(gu).float(), want, **tol(dtype))
    z = torch.zeros(1, 8, device="cuda", dtype=dtype)
    assert torch.all(ops.silu_mul(z) == 0)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
@pytest.mark.parametrize("mnk", [(1, 300, 72), (7, 65, 130), (130, 257, 96), (64, 64, 16), (3, 1000, 2050)])
def test_gemm_nt(ops, dtype, mnk):
    M, N, K = mnk
    torch.manual_seed(2)
    x = torch.randn(M, K, device="cuda").to(dtype)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(dtype)
    want = (x.double() @ w.double().T).float()
    y = ops.gemm_nt(x, w)
    torch.testing.assert_close(y.float(), want, **tol(dtype))
    if dtype == torch.bfloat16:
        y32 = ops.gemm_nt(x, w, torch.float32)
        torch.testing.assert_close(y32, want, atol=1e-4, rtol=1e-4)
    # strided rows of x (a slice of a wider buffer)
    wide = torch.randn(M, K + 24, device="cuda").to(dtype)
    ys = ops.gemm_nt(wide[:, 8:8 + K], w)
    torch.testing.assert_close(ys.float(), (wide[:, 8:8 + K].double() @ w.double().T).float(),
                               **tol(dtype))


@pytest.mark.parametrize("mnk", [
    # few rows: one piece of K, a row and a column past a tile, several waves with a short last one, 8-row tiles
    # with one and with two tiles of x, 16-row tiles
    (1, 9, 516), (8, 2049, 2052), (9, 70, 1028), (16, 2048, 4100), (16, 3073, 516), (12, 5000, 512),
    # many rows: one and just over one tile, K short of and past a step, cuts along K with a short last one
    (1, 8, 4), (12, 300, 508), (17, 16, 512), (64, 64, 32), (65, 129, 36), (129, 66, 2052), (33, 515, 8196), (700, 1000, 96), (1030, 2100, 260)])
def test_gemm_f32_matrix_cores(ops, mnk):
    """The float32 products on the matrix cores, and the vector kernel on the same operands shifted by one
    float (rows that are not aligned), element by element within the bound of a float32 sum of K products
    in any order: (K + 1) 2^-24 sum |x w|."""
    M, N, K = mnk
    torch.manual_seed(9)
    wide = torch.randn(M, K + 8, device="cuda")
    w = torch.randn(N, K, device="cuda")
    for x in (wide[:, 4:4 + K], wide[:, 4:4 + K].contiguous(), wide[:, 3:3 + K]):
        want = x.double() @ w.double().T
        bound = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        out = torch.full((M, N + 3), 7.0, device="cuda")
        y = ops.gemm_nt(x, w, out=out[:, :N])
        assert ((y.double() - want).abs() <= bound).all()
        assert (out[:, N:] == 7.0).all()
    # what is not finite stays in its row of x and its row of w
    x = wide[:, 4:4 + K].contiguous()
    x[M - 1, K - 1] = float("inf")
    w[N - 1, 0] = float("nan")
    y = ops.gemm_nt(x, w)
    assert torch.isnan(y[:, N - 1]).all() and torch.isfinite(y[:M - 1, :N - 1]).all()
    assert (~torch.isfinite(y[M - 1])).all()


# rows of x kept in registers: several tiles a workgroup, the longest sums that are kept (16 waves), a wave with
# fewer columns than the others and one without any, 16-row tiles; just too long to be kept
@pytest.mark.parametrize("mnk", [(3, 17001, 516), (8, 40, 8192), (5, 2100, 2564), (11, 9001, 4096), (16, 2731, 1028),
                                 (5, 70, 8196), (9, 2800, 4100)])
def test_gemm_f32_rows_kept(ops, mnk):
    test_gemm_f32_matrix_cores(ops, mnk)


@pytest.mark.parametrize("nk", [
    # one chunk of K and a part of one, chunks of 128, 256, 512 and 1,024 columns with a short last one, few and many
    # tiles of W, columns past a tile, odd N
    (16, 64), (37, 128), (70, 388), (2048, 512), (3073, 2052), (9001, 4096), (66, 4100), (2100, 8192), (40, 12292),
    (515, 16388), (2048, 2048)])
def test_gemm_f32_same_bits_alone_and_in_a_batch(ops, nk):
    """A row's float32 results are the same bits whatever the number of rows beside it: every kernel and plan
    adds the products in one order."""
    N, K = nk
    torch.manual_seed(4)
    x, w = torch.randn(700, K, device="cuda"), torch.randn(N, K, device="cuda")
    want = ops.gemm_nt(x, w)
    for M in (1, 2, 8, 9, 16, 17, 33, 64, 65, 129, 300, 483):
        for first in (0, 700 - M):
            assert torch.equal(ops.gemm_nt(x[first:first + M], w), want[first:first + M]), (M, first)


@pytest.mark.parametrize("mnk", [
    # many rows: an odd and an even number of blocks of 32 columns, one block, cuts along K with a short last one, N of no
    # whole 16-byte piece, more tiles than the compute units hold at a time
    (64, 64, 32), (65, 130, 96), (127, 127, 4128), (128, 128, 2080), (129, 257, 64), (300, 66, 8224), (20, 2051, 544),
    (515, 9001, 160), (1500, 4100, 128)])
def test_gemm_f32_streamed_tiles(ops, mnk):
    """Within the bound of test_gemm_f32_matrix_cores, and what is infinite or too large for the bfloat16 parts as the
    float32 sums have it, with the plan's choice of tiles for so many rows and with few rows."""
    test_gemm_f32_matrix_cores(ops, mnk)
    M, N, K = mnk
    torch.manual_seed(47)
    x, w = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda")
    x[M - 1, K // 2] = float("-inf")
    x[0, 0] = 3.4e38                       # rounds to infinity in bfloat16
    w[:, 0] *= 1e-3
    want = x.double() @ w.double().T
    for rows in {1, min(9, M - 1), M - 1}:
        y = ops.gemm_nt(x[M - rows:], w)
        assert torch.equal(y[-1].double(), want[-1])                 # all infinite
        y = ops.gemm_nt(x[:rows], w).double()
        bound = (K + 1) * 2.0 ** -24 * (x[:rows].double().abs() @ w.double().abs().T)
        assert ((y - want[:rows]).abs() <= bound).all()


F32_TILES = [(128, 128), (64, 128), (64, 64), (64, 64)]      # rows of x and of W; the last one splits x itself


def _f32_tiles(ops, x, w, tile, splits, out=None):
    """x @ w.T by a tile of csrc/gemm_f32.hip's, the spans of K in ``splits`` parts; None where there is no such plan."""
    import ctypes
    (M, K), N = x.shape, w.shape[0]
    lib = ops.library.load("gemm_f32")
    lib.ptl_gemm_f32_tiles_workspace.restype = ctypes.c_long
    floats = lib.ptl_gemm_f32_tiles_workspace(M, N, K, tile, splits)
    if floats < 0:
        return None
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    work = torch.full((max(floats, 4),), float("nan"), device="cuda")
    y = torch.empty((M, N), device="cuda") if out is None else out
    code = lib.ptl_gemm_f32_tiles(ptr(y), ptr(x), ptr(w), M, N, K, ctypes.c_long(x.stride(0)), ctypes.c_long(y.stride(0)), tile, splits,
                                  ptr(work), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert code == 0
    return y


@pytest.mark.parametrize("tile", range(4), ids=["128x128", "64x128", "64x64", "64x64_splits_x"])
@pytest.mark.parametrize("K", [32, 96, 1312, 2048, 4128, 2052])
def test_every_f32_tile(ops, tile, K):
    """Each tile by its index, whole and with K cut, with rows and columns one below, at and one above a tile's and more tiles than
    the chip holds: the bits of the kernels for few rows (which test_gemm_f32_matrix_cores and test_f32_low_parts compare with
    64 bits), where operands are infinite or NaN too, and nothing past the rows' ends."""
    bm, bn = F32_TILES[tile]
    torch.manual_seed(K)
    wide = 2 * ops.compute_units("cuda") * bn + 8 if K == 96 else 0
    for M, N in ((17, bn), (bm - 1, bn + 1), (bm, bn - 1), (bm + 1, 2 * bn + 4), (2 * bm, 5)) + (((bm + 3, wide),) if wide else ()):
        x, w = torch.randn(M, K + 4, device="cuda")[:, :K], torch.randn(N, K, device="cuda")
        for odd in (False, True):
            if odd:
                x = x.contiguous()
                _odd_operands(x, w)
            want = torch.cat([ops.gemm_nt(x[m:m + 8], w) for m in range(0, M, 8)])
            for splits in (1, 2, 5):
                out = torch.full((M, N + 3), 7.0, device="cuda")
                if _f32_tiles(ops, x, w, tile, splits, out[:, :N]) is None:
                    assert splits > 1 or (tile < 3 and K % 32)
                    continue
                _same(out[:, :N].contiguous(), want)
                assert (out[:, N:] == 7.0).all()
    assert _f32_tiles(ops, torch.zeros(17, 64, device="cuda"), torch.zeros(8, 64, device="cuda"), 4, 1) is None


def _low_parts(rows, K, seed):
    """Positive numbers (1 + m + l) 2^e whose three bfloat16 parts are 2^e, m 2^e and l 2^e with m in [2^-9, 2^-8), l in [2^-18,
    2^-17): what a sum misses without one of the parts adds up, it does not cancel."""
    g = torch.Generator().manual_seed(seed)
    m = torch.randint(128, 256, (rows, K), generator=g).double() * 2.0 ** -16
    l = torch.randint(32, 64, (rows, K), generator=g).double() * 2.0 ** -23
    v = (1 + m + l) * 2.0 ** torch.randint(-2, 3, (rows, K), generator=g).double()
    assert torch.equal(v.float().double(), v)
    return v.float().cuda()


def _f32_sum_bound(K, width):
    """What a sum of K positive products is off by, in 2^-24 of it: 2 sqrt(n) for n additions that round (six standard deviations of
    independent roundings of partial sums that grow evenly), those of the blocks of a span and those of the spans; 2 for the
    products that are left out, 12 for the six matrix instructions of a block, should they truncate. Without h l or l h it
    would be off by 90 and more, without m m by 64 and more."""
    return 2 * math.sqrt(min(K, width) / 32) + 2 * math.sqrt(math.ceil(K / width)) + 14


def _span_width(K):
    width = 128 if K <= 1024 else 256
    while -(-K // width) > 16:
        width *= 2
    return width


@pytest.mark.parametrize("K", [512, 1024, 2048, 2052, 8192])
def test_f32_low_parts(ops, K):
    """All parts of the operands count in every kernel, over the whole of K: a bound that does not grow with K as the worst case
    of test_gemm_f32_matrix_cores does."""
    bound = _f32_sum_bound(K, _span_width(K)) * 2.0 ** -24
    for M, N in ((4, 70), (8, 5000), (4, 17001), (12, 70), (12, 9001), (70, 140), (300, 2100)):
        x, w = _low_parts(M, K, 1), _low_parts(N, K, 2)
        want = x.double() @ w.double().T
        forms = {"plan": ops.gemm_nt(x, w)}
        if M > 16:
            forms.update({(t, s): _f32_tiles(ops, x, w, t, s) for t in range(4) for s in (1, 3)})
        for form, y in forms.items():
            if y is not None:
                off = float(((y.double() - want).abs() / want).max())
                assert off <= bound, f"{M} x {N}, {form}: {off * 2 ** 24:.1f} of {bound * 2 ** 24:.1f}"


@pytest.mark.parametrize("sizes", [(70, 1024, 512, 3, 1), (130, 1028, 1028, 4, 2)], ids=["whole_blocks", "part_of_a_block"])
def test_moe_f32_low_parts(ops, sizes):
    """The same of the routed experts: the first product's error counts twice in relu(u)^2, the second's once."""
    T, K, I, E, top = sizes
    x = _low_parts(T, K, 3)
    up, down = _low_parts(E * I, K, 4).view(E, I, K) / 1024, _low_parts(E * K, I, 5).view(E, K, I) / 1024
    r = ops.moe_route(torch.randn(T, E, device="cuda"), E, top)
    got = ops.moe_experts(x, r, up, down, ops.ACT_RELU2, 0.0, False)
    idx, wgt = r.idx.view(T, top).long().cpu(), r.wgt.view(T, top).double()
    want = torch.zeros(T, K, dtype=torch.float64, device="cuda")
    for e in range(E):
        h = (x.double() @ up[e].double().T) ** 2 @ down[e].double().T
        for c in range(top):
            rows = (idx[:, c] == e).nonzero()[:, 0].cuda()
            want[rows] += wgt[rows, c:c + 1] * h[rows]
    off = float(((got.double() - want).abs() / want).max()) * 2 ** 24
    bound = 2 * _f32_sum_bound(K, K) + _f32_sum_bound(I, I) + 8      # (8: the square, the weights and the sum over experts)
    assert off <= bound, f"{off:.1f} of {bound:.1f}"


@pytest.mark.parametrize("mn", [(4, 100), (4, 17000), (12, 5000), (70, 300)])
def test_gemm_f32_small_numbers(ops, mn):
    """Powers of two change nothing for numbers from 2^-110 on, times numbers around one. Below, the parts that are too small for
    bfloat16 are lost, less than 2^-126 of a number each, and products that small in the matrix cores."""
    M, N = mn
    K = 2048
    x, w = _low_parts(M, K, 6), _low_parts(N, K, 7)
    y = ops.gemm_nt(x, w)
    assert torch.equal(ops.gemm_nt(x * 2.0 ** -108, w), y * 2.0 ** -108)      # (the smallest of x are 2^-2)
    for power in (-112, -118, -124):
        small = x.double() * 2.0 ** power
        got = ops.gemm_nt(small.float(), w).double()
        rounded = small.float().double()
        want = rounded @ w.double().T
        lost = 2.0 ** -125 * (w.double().sum(1) + K)
        assert ((got - want).abs() <= lost[None] + (K + 1) * 2.0 ** -24 * want.abs()).all(), power


def _gpu_us(fn, times=5):
    """The fastest of some calls, in us."""
    fn()
    best = math.inf
    for _ in range(times):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        fn()
        b.record()
        b.synchronize()
        best = min(best, 1e3 * a.elapsed_time(b))
    return best


@pytest.mark.parametrize("mnk", [(4, 16384, 2048), (8, 2048, 8192), (16, 3072, 2048), (64, 2048, 2048), (300, 4096, 1024),
                                 (260, 2500, 1028)])
def test_gemm_f32_with_a_nan_is_not_slow(ops, mnk):
    """A NaN in one row of x makes every result of the row one; the product takes about as long as without it (four times
    as long is allowed here; sums made again by single lanes took twenty to fifty times)."""
    M, N, K = mnk
    torch.manual_seed(51)
    x, w = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda")
    out = torch.empty(M, N, device="cuda")
    without = _gpu_us(lambda: ops.gemm_nt(x, w, out=out))
    want = out.clone()
    x[M // 2, K // 2] = float("nan")
    assert _gpu_us(lambda: ops.gemm_nt(x, w, out=out)) < 4 * without + 20
    assert out[M // 2].isnan().all()
    keep = [m for m in range(M) if m != M // 2]
    assert torch.equal(out[keep], want[keep])


def _odd_operands(x, w):
    """Puts in x and w what the bfloat16 parts do not take: an infinity, a number that rounds to infinity, a NaN in a row of
    either, each with rows of the other kind."""
    M, K = x.shape
    w[:, 0] *= 1e-3                                          # (3.4e38 times up to 5e-3: within float32)
    x[:, 2] *= 1e-3
    x[0, 0] = 3.4e38
    if M > 1:
        x[1, K // 2] = float("-inf")
    if M > 2:
        x[2, K - 1] = float("nan")
    w[1, K - 1] = float("inf")
    w[2, 1] = float("nan")
    w[3, 2] = 3.4e38


def _same(got, want):
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))


@pytest.mark.parametrize("nk", [(16, 4), (70, 388), (3073, 2052), (2048, 2048), (2100, 8192), (515, 12292), (9001, 1024)])
def test_gemm_f32_what_is_not_finite(ops, nk):
    """Infinities, NaN and numbers that round to infinity give what sums of float32 products give, within the bound of
    test_gemm_f32_matrix_cores where that is finite, and the same bits whatever the number of rows."""
    N, K = nk
    torch.manual_seed(52)
    x, w = torch.randn(700, K, device="cuda"), torch.randn(N, K, device="cuda")
    _odd_operands(x, w)
    got = ops.gemm_nt(x, w)
    want = x.double() @ w.double().T
    finite = want.abs() < 3e38
    assert (finite | want.isnan() | want.isinf()).all()
    _same(torch.where(finite, 0.0, got.double()), torch.where(finite, 0.0, want))
    bound = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert (((got.double() - want).abs() <= bound) | ~finite).all()
    for M in (1, 3, 8, 9, 16, 17, 64, 130, 300):
        _same(ops.gemm_nt(x[:M], w), got[:M])


@pytest.mark.parametrize("K", [64, 2048, 4100, 8192])
def test_f32_pairs_of_what_is_not_finite(ops, K):
    """The forms of few rows that finish pairs of sums (gate-up, q | k | v): the bits of the kernels that they stand for."""
    torch.manual_seed(53)
    for M in (1, 3, 8):
        x, w = torch.randn(M, K, device="cuda"), torch.randn(2 * 4100, K, device="cuda")
        _odd_operands(x, w)
        w[4100] = w[1].flip(0)                               # (the other half of a pair)
        for act in (ops.GLU_SILU, ops.GLU_GELU_TANH):
            _same(ops.gate_up_f32(x, w, act), ops.silu_mul(ops.gemm_nt(x, w), act))
        Hq, Hkv, D, P = 6, 2, 16, 4
        w = w[:(Hq + 2 * Hkv) * D].contiguous()
        w[(Hq + Hkv) * D + 1, 0] = float("inf")
        pos, slots = (torch.arange(M, dtype=torch.int32, device="cuda") for _ in range(2))
        inv = (10000.0 ** (-torch.arange(0, D, 2).float() / D)).cuda()
        caches = [torch.zeros((3, Hkv, P, D), device="cuda") for _ in range(4)]
        q = ops.qkv_rope_store_f32(x, w, pos, inv, slots, caches[0], caches[1], Hq, Hkv, D, P)
        y = ops.gemm_nt(x, w).view(M, Hq + 2 * Hkv, D)
        ops.rope_store(y[:, :Hq], y[:, Hq:Hq + Hkv], y[:, Hq + Hkv:], pos, inv, slots, caches[2], caches[3], P)
        _same(q, y[:, :Hq])
        _same(caches[0], caches[2])
        _same(caches[1], caches[3])


@pytest.mark.parametrize("width", [4, 252, 260, 4096, 4100, 12292, 16384, 16388, 2050])
def test_add_rmsnorm_f32_widths(ops, width):
    """Every number of pieces a thread, a last piece alone in its wave, rows beyond the kernel with registers; and rows of
    any alignment."""
    torch.manual_seed(48)
    x, r = torch.randn(3, width, device="cuda"), torch.randn(3, width, device="cuda")
    w = 1 + 0.1 * torch.randn(width, device="cuda")
    odd = torch.empty(3 * width + 1, device="cuda")[1:].view(3, width)
    for a in (x, odd.copy_(x)):
        res = r.clone()
        y = ops.add_rmsnorm(a, res, w, 1e-5)
        s = a.double() + r.double()
        want = s / torch.sqrt((s * s).mean(-1, keepdim=True) + 1e-5) * w.double()
        assert torch.equal(res, a + r)
        torch.testing.assert_close(y.double(), want, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("sizes", [(1, 36, 8, 3, 2), (70, 132, 66, 2, 1), (200, 64, 130, 5, 2), (9, 30, 20, 4, 2)],
                         ids=["one_row", "65_rows_an_expert", "edges", "unaligned"])
@pytest.mark.parametrize("gated", [True, False])
def test_moe_f32_matrix_cores(ops, sizes, gated):
    """The routed experts in float32, within the bound that the sums of both products give: an element of the
    first is off by (K + 2) 2^-24 sum |x w|, which the activation passes on with its slope, and the second adds
    (I + 2) 2^-24 of its own sum."""
    T, K, I, E, top = sizes
    torch.manual_seed(K)
    x = torch.randn(T, K, device="cuda")
    gu = torch.randn(E, (2 if gated else 1) * I, K, device="cuda") / math.sqrt(K)
    down = torch.randn(E, K, I, device="cuda") / math.sqrt(I)
    r = ops.moe_route(torch.randn(T, E, device="cuda"), E, top)
    got = ops.moe_experts(x, r, gu, down, 0 if gated else ops.ACT_RELU2, 0.0, False)
    u = 2.0 ** -24
    idx, wgt = r.idx.view(T, top).long(), r.wgt.view(T, top).double()
    want, bound = torch.zeros(T, K, dtype=torch.float64, device="cuda"), torch.zeros(T, K, dtype=torch.float64, device="cuda")
    for c in range(top):
        w1, w2 = gu.double()[idx[:, c]], down.double()[idx[:, c]]
        p = torch.bmm(w1, x.double()[:, :, None].contiguous())[:, :, 0]
        e = (K + 2) * u * torch.bmm(w1.abs(), x.double().abs()[:, :, None].contiguous())[:, :, 0]
        if gated:
            g, v = p[:, :I], p[:, I:]
            h = g * torch.sigmoid(g) * v
            e = 1.1 * e[:, :I] * v.abs() + g.abs() * e[:, I:] + 8 * u * h.abs()
        else:
            h = p.clamp(min=0) ** 2
            e = 2 * p.abs() * e + 4 * u * h
        want += wgt[:, c:c + 1] * torch.bmm(w2, h[:, :, None].contiguous())[:, :, 0]
        bound += wgt[:, c:c + 1] * torch.bmm(w2.abs(), (e + (I + 8) * u * h.abs())[:, :, None].contiguous())[:, :, 0]
    assert ((got.double() - want).abs() <= bound * 1.01).all()


@pytest.mark.parametrize("gated", [True, False])
def test_moe_f32_what_is_not_finite(ops, gated):
    """Routed experts with infinities, NaN and numbers that round to infinity in bfloat16: what the vector kernel (operands
    that are not 16-byte aligned) gives, in both products; and a NaN in one row costs little time."""
    T, K, I, E, top = 70, 1024, 512, 8, 2
    torch.manual_seed(54)
    G = 2 if gated else 1
    x = torch.randn(T, K, device="cuda")
    gu = torch.randn(E, G * I, K, device="cuda") / math.sqrt(K)
    down = torch.randn(E, K, I, device="cuda") / math.sqrt(I)
    r = ops.moe_route(torch.randn(T, E, device="cuda"), E, top)
    act = 0 if gated else ops.ACT_RELU2
    without = _gpu_us(lambda: ops.moe_experts(x, r, gu, down, act, 0.0, False))
    x[5, K // 2] = float("nan")
    assert _gpu_us(lambda: ops.moe_experts(x, r, gu, down, act, 0.0, False)) < 4 * without + 20
    x[0, 0] = 3.4e38
    gu[:, :, 0] *= 1e-32                                      # (sums of some 1e5, whose square is far from float32's end)
    x[1, 7] = float("inf")
    gu[0, 1, 3], gu[1, G * I - 2, 4] = float("-inf"), float("nan")
    gu[2, 0] *= 1e-3                                          # (a result below 1, times 3.4e38)
    down[2, 3, 0] = 3.4e38
    down[3, 1, 5], down[3, 2, 6] = float("inf"), float("nan")

    def unaligned(t):
        return torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape).copy_(t)

    got = ops.moe_experts(x, r, gu, down, act, 0.0, False)
    want = ops.moe_experts(unaligned(x), r, unaligned(gu), unaligned(down), act, 0.0, False)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got.isinf() & (got > 0), want.isinf() & (want > 0))
    finite = got.isfinite()
    assert 0.3 < finite.float().mean() < 1
    # sums of the same products in another order, in either product: a part of 2 (K + I) 2^-24 of a row's largest result at most
    scale = want.where(finite, 0.0).abs().amax(1, keepdim=True)
    assert (((got - want).abs() <= 2 * (K + I) * 2.0 ** -24 * scale) | ~finite).all()


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32], ids=["to_bf16", "to_fp32"])
@pytest.mark.parametrize("mnk", [(1, 300, 72), (7, 65, 136), (16, 3072, 2048), (17, 100, 200),
                                 (33, 16, 8192), (64, 1000, 64), (8, 2048, 8192), (5, 130, 2056),
                                 # a W wide enough for the streaming form: tiles past the end, K with a
                                 # partial last batch, one row and sixteen
                                 (1, 16384, 256), (8, 20003, 328), (16, 17000, 2048), (3, 40001, 72),
                                 # every way of packing the loads of x: 1, 2, 4, 8 rows a block, and none
                                 (2, 520, 264), (4, 136, 1032), (6, 264, 520), (9, 72, 296), (2, 4112, 2048)])
def test_gemm_skinny(ops, out_dtype, mnk):
    M, N, K = mnk
    torch.manual_seed(7)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    want = (x.double() @ w.double().T).float()
    y = ops.gemm_skinny(x, w, out_dtype)
    assert y.dtype == out_dtype
    t = dict(atol=1e-4, rtol=1e-4) if out_dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(y.float(), want, **t)
    # rows of x as a slice of a wider buffer
    wide = torch.randn(M, K + 24, device="cuda").to(torch.bfloat16)
    xs = wide[:, 8:8 + K]
    torch.testing.assert_close(ops.gemm_skinny(xs, w, out_dtype).float(),
                               (xs.double() @ w.double().T).float(), **t)
    with pytest.raises(ops.KernelError):
        ops.gemm_skinny(torch.zeros(65, K, device="cuda", dtype=torch.bfloat16), w)
    with pytest.raises(ops.KernelError):
        ops.gemm_skinny(x[:, :K - 4], w[:, :K - 4].contiguous())


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32], ids=["to_bf16", "to_fp32"])
@pytest.mark.parametrize("mnk", [(1, 300, 72), (17, 100, 200), (64, 3072, 2048), (300, 130, 136),
                                 (512, 2048, 2048), (777, 1000, 328), (2048, 352, 176)])
def test_gemm_library(ops, out_dtype, mnk):
    """The library product called directly: against a float64 product, also for rows of x that
    are a slice of a wider buffer; the second call takes the kept plan, the third times the
    library's proposals for the shape and the fourth runs the fastest of them."""
    M, N, K = mnk
    torch.manual_seed(9)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    want = (x.double() @ w.double().T).float()
    t = dict(atol=1e-4, rtol=1e-4) if out_dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    for call in range(4):
        if call == 2:
            with ops.timed_library_products():
                y = ops.gemm_library(x, w, out_dtype)
        else:
            y = ops.gemm_library(x, w, out_dtype)
        assert y.dtype == out_dtype and y.shape == (M, N)
        torch.testing.assert_close(y.float(), want, **t)
    wide = torch.randn(M, K + 24, device="cuda").to(torch.bfloat16)
    xs = wide[:, 8:8 + K]
    torch.testing.assert_close(ops.gemm_library(xs, w, out_dtype).float(),
                               (xs.double() @ w.double().T).float(), **t)
    assert not ops.gemm_library_fits(wide[:, 1:1 + K], w)            # rows not 16-byte aligned
    assert not ops.gemm_library_fits(x.float(), w)
    with pytest.raises(ops.KernelError):
        ops.gemm_library(x.float(), w)


def test_gemm_library_runs_the_first_proposal_unless_asked_for_the_timed_one(ops):
    """A shape for which the timing keeps another proposal than the library's first on this
    GPU (64 rows, depth 8,192): calls outside ``timed_library_products`` give the same bits
    before and after the timing, the timed choice agrees with them within the rounding of
    bfloat16 (proposals add in different orders), and the choice can be asked for."""
    M, N, K = 64, 2048, 8192
    torch.manual_seed(11)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    before = ops.gemm_library(x, w)
    with ops.timed_library_products():
        timed = ops.gemm_library(x, w)
        again = ops.gemm_library(x, w)
    after = ops.gemm_library(x, w)
    assert torch.equal(before, after)
    assert torch.equal(timed, again)
    choice = ops.library_product_choice(M, N, K, K)
    assert choice >= 0
    assert ops.library_product_choice(M + 1, N, K, K) == -1               # never timed
    want = (x.double() @ w.double().T).float()
    ulp = 2.0 ** -7 * want.abs() + 1e-3 * float(want.abs().max())
    assert bool(((timed.float() - before.float()).abs() <= ulp).all())
    torch.testing.assert_close(timed.float(), want, atol=2e-2, rtol=2e-2)
    with ops.timed_library_products(False):                               # a switch passed on as off
        assert torch.equal(ops.gemm_library(x, w), before)


def test_gemm_library_times_nothing_while_a_graph_is_recorded(ops):
    """Timing switched on while a HIP graph is recorded: nothing waits for the stream there (the
    recording would fail), every replay gives the product, and the call after the recording,
    which does time the proposals, gives it too."""
    M, N, K = 48, 264, 520
    torch.manual_seed(10)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    want = (x.double() @ w.double().T).float()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.gemm_library(x, w)                                   # plan, handle and workspace
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), ops.timed_library_products():
        ys = [ops.gemm_library(x, w) for _ in range(3)]
    for _ in range(3):
        for y in ys:
            y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for y in ys:
            torch.testing.assert_close(y.float(), want, atol=2e-2, rtol=2e-2)
    with ops.timed_library_products():
        torch.testing.assert_close(ops.gemm_library(x, w).float(), want, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(ops.gemm_library(x, w).float(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("mik", [(1, 176, 64), (8, 8192, 2048), (16, 320, 136), (5, 48, 2056)])
def test_gate_up_silu(ops, mik):
    M, I, K = mik
    torch.manual_seed(8)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * I, K, device="cuda") / math.sqrt(K) * 2).to(torch.bfloat16)
    got = ops.gate_up_silu(x, w)
    want = ops.silu_mul(ops.gemm_nt(x, w))              # the unfused kernels
    torch.testing.assert_close(got.float(), want.float(), atol=2e-2, rtol=2e-2)
    gu = (x.double() @ w.double().T).float()
    plain = plain_llama.silu(gu[:, :I]) * gu[:, I:]
    torch.testing.assert_close(got.float(), plain, atol=3e-2, rtol=3e-2)
    with pytest.raises(ops.KernelError):
        ops.gate_up_silu(torch.zeros(17, K, device="cuda", dtype=torch.bfloat16), w)


@pytest.mark.parametrize("dims", [(4, 2, 64, 16, 72), (3, 1, 32, 4, 128), (8, 8, 128, 16, 2048), (6, 3, 96, 5, 200)])
def test_qkv_rope_store(ops, dims):
    Hq, Hkv, D, P, K = dims
    M = 7
    torch.manual_seed(9)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    positions = torch.tensor([0, 1, 5, 77, 1000, 4095, 100000], dtype=torch.int32, device="cuda")
    inv_freq = plain_llama.rope_inv_freq_default(500000.0, D).cuda()
    pages = 5
    slots = torch.randperm(pages * P)[:M].to(torch.int32).cuda()
    slots[3] = -1                                           # this row's keys are not stored
    kc = torch.zeros(pages, Hkv, P, D, device="cuda", dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    q = ops.qkv_rope_store(x, w, positions, inv_freq, slots, kc, vc, Hq, Hkv, D, P)
    # the unfused kernels on the same inputs
    qkv = ops.gemm_nt(x, w)
    q2 = qkv[:, :Hq * D].view(M, Hq, D)
    k2 = qkv[:, Hq * D:(Hq + Hkv) * D].view(M, Hkv, D)
    v2 = qkv[:, (Hq + Hkv) * D:].view(M, Hkv, D)
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    ops.rope_store(q2, k2, v2, positions, inv_freq, slots, kc2, vc2, P)
    torch.testing.assert_close(q.float(), q2.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(kc.float(), kc2.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(vc.float(), vc2.float(), atol=2e-2, rtol=2e-2)
    assert torch.all(kc.view(pages, Hkv, P, D)[:, :, :, :].sum() != 0)
    # and the plain formulas
    full = (x.double() @ w.double().T).float().cpu()
    cos, sin = plain_llama.rope_cos_sin(inv_freq.cpu(), positions.cpu())
    want_q = plain_llama.apply_rope(full[:, :Hq * D].view(M, Hq, D), cos, sin)
    torch.testing.assert_close(q.float().cpu(), want_q, atol=3e-2, rtol=3e-2)
    # without rotation and without a store
    q3 = ops.qkv_rope_store(x, w, positions, None, None, None, None, Hq, Hkv, D, P)
    torch.testing.assert_close(q3.float().cpu(), full[:, :Hq * D].view(M, Hq, D), atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("mnk", [(1, 64, 176), (8, 2048, 2048), (16, 136, 320), (5, 4096, 72), (3, 2056, 48)])
def test_gemm_skinny_add_norm_and_row_scale(ops, mnk):
    """Product + residual sum + norm weight in one kernel, the rsqrt factor left as partial sums:
    the residual it leaves, and its output once the factor is applied, are those of the product
    followed by add_rmsnorm, and of the plain formulas."""
    M, N, K = mnk
    torch.manual_seed(12)
    eps = 1e-5
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    res = torch.randn(M, N, device="cuda").to(torch.bfloat16)
    nw = (1.0 + 0.2 * torch.randn(N, device="cuda")).float()
    res_fused = res.clone()
    y, scale = ops.gemm_skinny_add_norm(x, w, res_fused, nw, eps)
    assert scale.partials.shape[0] == M and scale.size == N
    got = ops.row_scale(y, scale)
    # the separate kernels
    res_sep = res.clone()
    want = ops.add_rmsnorm(ops.gemm_skinny(x, w), res_sep, nw, eps)
    assert torch.equal(res_fused, res_sep)                       # same roundings, same sums
    torch.testing.assert_close(got.float(), want.float(), atol=3e-2, rtol=2e-2)
    # the sums of squares against the residual itself
    ss = scale.partials.sum(dim=1)
    torch.testing.assert_close(ss, (res_fused.float() ** 2).sum(dim=1), rtol=2e-2, atol=1e-3)
    # the plain formulas
    h = (x.double() @ w.double().T).float().cpu() + res.float().cpu()
    plain, _ = plain_llama.add_rms_norm(h, None, nw.cpu(), eps)
    torch.testing.assert_close(got.float().cpu(), plain, atol=5e-2, rtol=3e-2)
    with pytest.raises(ops.KernelError):
        ops.gemm_skinny_add_norm(torch.zeros(17, K, device="cuda", dtype=torch.bfloat16), w,
                                 torch.zeros(17, N, device="cuda", dtype=torch.bfloat16), nw, eps)
    with pytest.raises(ops.KernelError):
        ops.row_scale(y, ops.RowScale(scale.partials, N + 8, eps))


def test_fused_products_apply_a_row_scale(ops):
    """gate_up_silu and qkv_rope_store with rows that still lack their factor give what they
    give for the rows with the factor applied."""
    torch.manual_seed(13)
    M, H, I, Hq, Hkv, D, P = 6, 328, 176, 4, 2, 32, 8
    eps = 1e-6
    v = torch.randn(M, H, device="cuda").to(torch.bfloat16)
    partials = torch.rand(M, 41, device="cuda") * 30                 # any positive sums do
    scale = ops.RowScale(partials, H, eps)
    f = torch.rsqrt(partials.sum(dim=1) / H + eps)
    xs = (v.float() * f[:, None])                                     # the finished rows, float32
    wg = (torch.randn(2 * I, H, device="cuda") / math.sqrt(H)).to(torch.bfloat16)
    got = ops.gate_up_silu(v, wg, scale)
    gu = xs.double() @ wg.double().T
    want = (plain_llama.silu(gu[:, :I]) * gu[:, I:]).float()
    torch.testing.assert_close(got.float(), want, atol=3e-2, rtol=3e-2)
    wq = (torch.randn((Hq + 2 * Hkv) * D, H, device="cuda") / math.sqrt(H)).to(torch.bfloat16)
    positions = torch.tensor([0, 3, 9, 100, 2000, 7], dtype=torch.int32, device="cuda")
    inv_freq = plain_llama.rope_inv_freq_default(10000.0, D).cuda()
    slots = torch.arange(M, dtype=torch.int32, device="cuda")
    kc = torch.zeros(2, Hkv, P, D, device="cuda", dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    q = ops.qkv_rope_store(v, wq, positions, inv_freq, slots, kc, vc, Hq, Hkv, D, P, scale)
    full = (xs.double() @ wq.double().T).float().cpu()
    cos, sin = plain_llama.rope_cos_sin(inv_freq.cpu(), positions.cpu())
    want_q = plain_llama.apply_rope(full[:, :Hq * D].view(M, Hq, D), cos, sin)
    torch.testing.assert_close(q.float().cpu(), want_q, atol=3e-2, rtol=3e-2)
    want_k = plain_llama.apply_rope(full[:, Hq * D:(Hq + Hkv) * D].view(M, Hkv, D), cos, sin)
    got_k = kc.view(2 * 1, Hkv, P, D).permute(0, 2, 1, 3).reshape(2 * P, Hkv, D)[:M]
    torch.testing.assert_close(got_k.float().cpu(), want_k, atol=3e-2, rtol=3e-2)
    want_v = full[:, (Hq + Hkv) * D:].view(M, Hkv, D)
    got_v = vc.permute(0, 2, 1, 3).reshape(2 * P, Hkv, D)[:M]
    torch.testing.assert_close(got_v.float().cpu(), want_v, atol=3e-2, rtol=3e-2)
    # the factor really is used: without it the result differs
    q_plain = ops.qkv_rope_store(v, wq, positions, inv_freq, None, None, None, Hq, Hkv, D, P)
    assert (q_plain.float() - q.float()).abs().max() > 0.1


def test_qkv_rope_store_with_a_large_row_scale(ops):
    """Rows whose pending factor is large (a residual stream that is nearly zero: one partial
    sum of 1e-3 .. 30 over 6,184 columns gives factors of 14 to 930) make q and k values of
    some hundreds. The kernel rounds the scaled projection to bfloat16 before it rotates, as
    the separate kernels store it between product and rotation, so an element of the result
    carries the rounding of both elements of its pair: the bound is half a bfloat16 ulp (at most
    2^-8 of the value) of x1 and of x2 from before the rotation plus half an ulp of the result,
    not a share of the element itself, which the rotation can make small. Every element must
    lie within that bound."""
    torch.manual_seed(249)
    M, K, D, Hq, Hkv, P = 13, 6184, 128, 7, 1, 5
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    partials = torch.logspace(-3, math.log10(30.0), M, device="cuda").view(M, 1).contiguous()
    scale = ops.RowScale(partials, K, 1e-6)
    f = torch.rsqrt(partials.sum(dim=1).double() / K + 1e-6)
    assert float(f.max()) > 900 and float(f.min()) < 20
    positions = torch.tensor([5000, 0, 0, 5000, 77, 77, 0, 77, 5000, 1, 77, 1, 100000],
                             dtype=torch.int32, device="cuda")
    inv_freq = plain_llama.rope_inv_freq_default(500000.0, D).cuda()
    npage = -(-M // P) + 1
    slots = torch.randperm(npage * P)[:M].to(torch.int32).cuda()
    kc = torch.zeros(npage, Hkv, P, D, device="cuda", dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    q = ops.qkv_rope_store(x, w, positions, inv_freq, slots, kc, vc, Hq, Hkv, D, P, scale)
    full = ((x.double() * f[:, None]) @ w.double().T).cpu()
    cos, sin = plain_llama.rope_cos_sin(inv_freq.cpu(), positions.cpu())

    def check(got, projected, what, rotated=True):
        want = plain_llama.apply_rope(projected, cos.double(), sin.double()) if rotated else projected
        a = projected.abs()
        pair = a + torch.cat((a[..., D // 2:], a[..., :D // 2]), dim=-1) if rotated else a
        bound = 2.0 ** -8 * (pair + want.abs() if rotated else pair) + 1e-5 * a.amax(dim=(-2, -1), keepdim=True)
        over = (got.double() - want).abs() - bound
        assert float(over.max()) <= 0, f"{what}: {float(over.max()):.3g} beyond the rounding bound"
        assert float(want.abs().max()) > 300          # the case is about large values

    check(q.cpu(), full[:, :Hq * D].view(M, Hq, D), "q")
    rows = slots.long().cpu()
    got_k = kc.permute(0, 2, 1, 3).reshape(npage * P, Hkv, D).cpu()[rows]
    got_v = vc.permute(0, 2, 1, 3).reshape(npage * P, Hkv, D).cpu()[rows]
    check(got_k, full[:, Hq * D:(Hq + Hkv) * D].view(M, Hkv, D), "k")
    check(got_v, full[:, (Hq + Hkv) * D:].view(M, Hkv, D), "v", rotated=False)


@pytest.mark.parametrize("dims", [(8, 2048, 2048, 8192, 32, 8, 64, 16), (1, 2048, 2048, 8192, 32, 8, 64, 16),
                                  (16, 160, 224, 224, 3, 1, 32, 8), (5, 3072, 3072, 1024, 24, 8, 128, 16),
                                  (3, 64, 64, 160, 8, 2, 32, 4), (13, 4128, 96, 64, 2, 2, 96, 16),
                                  (7, 1000, 96, 48, 5, 5, 32, 2)])
def test_decode_kernels_read_the_blocked_copy_of_a_weight(ops, dims):
    """The decode kernels with the second, blocked copy of their weights (tiles of 16 rows x 32
    columns, each in one piece) give bit for bit what they give with the row-major matrix: the
    same sums in the same order, only fetched from other addresses. Widths that are no multiple
    of 16 rows (padding), 8- and 16-row tiles, one to sixteen rows of x."""
    M, H, Kin, I, Hq, Hkv, D, P = dims
    g = torch.Generator().manual_seed(M * 7 + H)
    rnd = lambda *s: torch.randn(*s, generator=g)
    dev = "cuda"
    x = rnd(M, Kin).to(torch.bfloat16).to(dev)
    wo = (rnd(H, Kin) / math.sqrt(Kin)).to(torch.bfloat16).to(dev)
    wgu = (rnd(2 * I, H) / math.sqrt(H)).to(torch.bfloat16).to(dev)
    wq = (rnd((Hq + 2 * Hkv) * D, H) / math.sqrt(H)).to(torch.bfloat16).to(dev)
    nw = (1 + 0.1 * rnd(H)).to(dev)
    res = rnd(M, H).to(torch.bfloat16).to(dev)
    bo, bgu, bq = ops.blocked_weight(wo), ops.blocked_weight(wgu), ops.blocked_weight(wq)
    assert bo.shape == (-(-H // 16), Kin // 32, 16, 32)
    # the layout itself: tile t, column block b holds rows 16 t .. 16 t + 15, columns 32 b .. 32 b + 31
    t, b = bo.shape[0] - 1, bo.shape[1] - 1
    rows = wo[16 * t:16 * t + 16, 32 * b:32 * b + 32]
    assert torch.equal(bo[t, b, :rows.shape[0]], rows) and bool((bo[t, b, rows.shape[0]:] == 0).all())
    for out_dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(ops.gemm_skinny(x, wo, out_dtype), ops.gemm_skinny(x, wo, out_dtype, blocked=bo))
    r1, r2 = res.clone(), res.clone()
    y1, s1 = ops.gemm_skinny_add_norm(x, wo, r1, nw, 1e-5)
    y2, s2 = ops.gemm_skinny_add_norm(x, wo, r2, nw, 1e-5, blocked=bo)
    assert torch.equal(y1, y2) and torch.equal(r1, r2) and torch.equal(s1.partials, s2.partials)
    assert torch.equal(ops.gate_up_silu(y1, wgu, s1), ops.gate_up_silu(y1, wgu, s1, blocked=bgu))
    assert torch.equal(ops.gate_up_silu(y1, wgu), ops.gate_up_silu(y1, wgu, blocked=bgu))
    positions = torch.randint(0, 3000, (M,), generator=g).to(torch.int32).to(dev)
    inv_freq = plain_llama.rope_inv_freq_default(10000.0, D).to(dev)
    slots = (torch.randperm(2 * P, generator=g)[:M]).to(torch.int32).to(dev) if M <= 2 * P else None
    outs = []
    for blocked in (None, bq):
        kc = torch.zeros(2, Hkv, P, D, device=dev, dtype=torch.bfloat16)
        vc = torch.zeros_like(kc)
        q = ops.qkv_rope_store(y1, wq, positions, inv_freq, slots, kc if slots is not None else None,
                               vc if slots is not None else None, Hq, Hkv, D, P, s1, blocked=blocked)
        outs.append((q, kc, vc))
    for a, b2 in zip(*outs):
        assert torch.equal(a, b2)
    # a copy that belongs to another matrix is refused, more rows than the kernels take fall back
    with pytest.raises(ops.KernelError):
        ops.gemm_skinny(x, wo, blocked=torch.zeros((bo.shape[0] + 1, *bo.shape[1:]), dtype=torch.bfloat16, device=dev))
    x20 = rnd(20, Kin).to(torch.bfloat16).to(dev)
    assert torch.equal(ops.gemm_skinny(x20, wo), ops.gemm_skinny(x20, wo, blocked=bo))
    assert ops.blocked_weight(rnd(8, 40).to(torch.bfloat16).to(dev)) is None       # K no multiple of 32


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32], ids=["to_bf16", "to_fp32"])
@pytest.mark.parametrize("mnk", [(17, 64, 32), (24, 1000, 96), (33, 2048, 2080), (64, 130, 4096), (100, 3000, 160),
                                 (128, 16400, 512), (5, 70, 64), (9, 200, 96), (16, 2048, 2048), (12, 70000, 64),
                                 (40, 66000, 96), (48, 3072, 2048), (37, 100, 4128)])
def test_gemm_rows(ops, out_dtype, mnk):
    """The product for some tens of rows (x through LDS, the blocked copy of W streamed): widths
    that are no multiple of a workgroup's 64 rows or of a tile's 16, depths that are no multiple
    of a chunk, one to eight tiles of x, one and two tiles of W a wave (two from 1,024 workgroups
    on), against a float64 product; and as partial sums over slices of K, whose sum is the
    product."""
    M, N, K = mnk
    torch.manual_seed(21)
    wide = torch.randn(M, K + 8, device="cuda").to(torch.bfloat16)
    x = wide[:, :K]                                               # rows of a wider buffer
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    b = ops.blocked_weight(w)
    want = (x.double() @ w.double().T).float()
    t = dict(atol=1e-4, rtol=1e-4) if out_dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    y = ops.gemm_rows(x, w, b, out_dtype) if M >= ops.ROWS_MIN else None
    if M >= ops.ROWS_MIN:
        assert y.dtype == out_dtype and y.shape == (M, N)
        torch.testing.assert_close(y.float(), want, **t)
        for splits in (2, 3, 8):
            parts = ops.gemm_rows(x, w, b, torch.float32, splits=splits)
            assert parts.shape == (splits, M, N)
            torch.testing.assert_close(parts.sum(dim=0), want, atol=1e-4, rtol=1e-4)
        with pytest.raises(ops.KernelError):
            ops.gemm_rows(x, w, b, torch.bfloat16, splits=2)      # partial sums are float32
        with pytest.raises(ops.KernelError):
            ops.gemm_rows(x, w, torch.zeros_like(b)[1:], out_dtype)   # a copy of another matrix
    else:
        with pytest.raises(ops.KernelError):
            ops.gemm_rows(x, w, b, out_dtype)                      # fewer rows than ROWS_MIN: the other kernels


@pytest.mark.parametrize("mnk", [(17, 64, 96), (40, 2048, 2048), (64, 2056, 320), (128, 4096, 8192), (9, 2048, 2048),
                                 (16, 264, 96), (48, 2048, 8192), (35, 72, 64)])
def test_gemm_rows_add_rmsnorm(ops, mnk):
    """Partial sums over slices of K, then one kernel that adds them up, adds the residual and
    normalises whole rows: the residual it leaves and its output are those of the product
    followed by add_rmsnorm, and of the plain formulas."""
    M, N, K = mnk
    torch.manual_seed(22)
    eps = 1e-5
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    b = ops.blocked_weight(w)
    res = torch.randn(M, N, device="cuda").to(torch.bfloat16)
    nw = (1.0 + 0.2 * torch.randn(N, device="cuda")).float()
    r1, r2 = res.clone(), res.clone()
    partials = ops.gemm_rows(x, w, b, torch.float32, splits=ops.gemm_rows_splits(M, N, K))
    got = ops.sum_add_rmsnorm(partials, r1, nw, eps)
    want = ops.add_rmsnorm(ops.gemm_nt(x, w), r2, nw, eps)               # the separate kernels
    torch.testing.assert_close(r1.float(), r2.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(got.float(), want.float(), atol=3e-2, rtol=2e-2)
    h = (x.double() @ w.double().T).float().cpu() + res.float().cpu()
    plain, plain_res = plain_llama.add_rms_norm(h, None, nw.cpu(), eps)
    torch.testing.assert_close(got.float().cpu(), plain, atol=5e-2, rtol=3e-2)
    torch.testing.assert_close(r1.float().cpu(), plain_res, atol=3e-2, rtol=2e-2)
    # a float32 product of one piece is a partial sum of one slice
    r3 = res.clone()
    one = ops.sum_add_rmsnorm(ops.gemm_rows(x, w, b, torch.float32), r3, nw, eps)
    torch.testing.assert_close(one.float(), got.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("smn", [(1, 3, 8), (3, 2, 512), (4, 5, 520), (8, 64, 2056), (5, 20, 3072), (2, 7, 4096), (4, 3, 4104),
                                 (4, 64, 5120), (9, 2, 8184), (1, 300, 8192)])
def test_sum_add_rmsnorm(ops, smn):
    """Widths around the pieces a thread and the threads a row: the float64 result of the same rounded sums."""
    S, M, N = smn
    torch.manual_seed(28)
    p, res = torch.randn(S, M, N, device="cuda"), torch.randn(M, N, device="cuda").to(torch.bfloat16)
    nw, eps = torch.randn(N, device="cuda"), 1e-5
    total = p[0].clone()
    for s in range(1, S):
        total += p[s]                                              # float32, in the order of the slices
    h = total.to(torch.bfloat16).double() + res.double()
    want = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + eps) * nw.double()
    got = ops.sum_add_rmsnorm(p, res, nw, eps)
    assert torch.equal(res, h.float().to(torch.bfloat16))
    # one rounding to bfloat16 (2^-9 of the value) and the float32 statistics
    torch.testing.assert_close(got.double(), want, atol=1e-5, rtol=2 ** -8)


@pytest.mark.parametrize("mnk", [(1, 8, 64), (65, 2048, 8192), (80, 72, 128), (97, 4096, 2048), (129, 264, 4096),
                                 (200, 2048, 2048), (285, 2048, 8192), (401, 3072, 3072), (532, 4096, 1536),
                                 (700, 1032, 576), (1024, 2048, 8192), (1088, 3072, 2048)])
def test_gemm_tile_add_rmsnorm(ops, mnk):
    """Products of some hundred rows as partial sums over slices of K, in the tiles the plan takes for them (six of the
    twelve; test_every_tile runs all): rows of x and of W that are no multiple of a tile, one chunk of K, depths with and
    without slices; against a float64 product
    (float32 sums of up to 8,192 exact products: 1e-4), and with the norm behind them against the separate kernels."""
    M, N, K = mnk
    torch.manual_seed(41)
    x = torch.randn(M, K + 16, device="cuda").to(torch.bfloat16)[:, :K]          # rows of a wider buffer
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    parts = ops.gemm_tile_sums(x, w)
    assert parts.shape[1:] == (M, N) and K % (64 * parts.shape[0]) == 0
    torch.testing.assert_close(parts.sum(dim=0), (x.double() @ w.double().T).float(), atol=1e-4, rtol=1e-4)
    res = torch.randn(M, N, device="cuda").to(torch.bfloat16)
    nw = (1.0 + 0.2 * torch.randn(N, device="cuda")).float()
    r1, r2 = res.clone(), res.clone()
    got = ops.gemm_tile_add_rmsnorm(x, w, r1, nw, 1e-5)
    want = ops.add_rmsnorm(ops.gemm_nt(x, w), r2, nw, 1e-5)
    torch.testing.assert_close(r1.float(), r2.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(got.float(), want.float(), atol=3e-2, rtol=2e-2)
    with pytest.raises(ops.KernelError):
        ops.gemm_tile_sums(x[:, :K - 32], w[:, :K - 32].contiguous())            # K no multiple of a chunk
    with pytest.raises(ops.KernelError):
        ops.gemm_tile_sums(x, w[:, 1:])


@pytest.mark.parametrize("rows", [20, 64, 70, 300])
@pytest.mark.parametrize("shift", [(4, 0), (0, 1), (4, 1), (0, 0)], ids=["residual", "weight", "both", "aligned"])
def test_a_norm_behind_a_product_with_rows_that_are_not_aligned(ops, rows, shift):
    """A residual that begins 8 bytes into a buffer (an embedding's own), a norm weight 4 bytes into one (a checkpoint held
    as one flat buffer): kernels that read 16 bytes at a time leave them to the others."""
    from pytriton_llama_amd.parts.base import PendingProduct
    from pytriton_llama_amd.parts.norm import RMSNorm
    N, K = 512, 1024
    torch.manual_seed(46)
    x = torch.randn(rows, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    res = torch.randn(rows * N + 8, device="cuda").to(torch.bfloat16)[shift[0]:shift[0] + rows * N].view(rows, N)
    norm = RMSNorm(N, 1e-5)
    norm.weight = (1.0 + 0.2 * torch.randn(N + 4, device="cuda"))[shift[1]:shift[1] + N]
    h = (x.double() @ w.double().T).to(torch.bfloat16).double() + res.double()
    want = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5) * norm.weight.double()
    got, out = norm.forward(PendingProduct(x, w, ops.blocked_weight(w)), res)
    torch.testing.assert_close(got.double(), want, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(out.double(), h, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("mik", [(1, 4, 64), (65, 8192, 2048), (81, 36, 192), (130, 2048, 2048), (200, 8192, 2048),
                                 (285, 8192, 3072), (400, 1000, 512), (532, 8192, 2048), (576, 14336, 1024)])
def test_gate_up_tile(ops, mik, act):
    """Gate and up rows in one tile, the one the plan takes for these rows (five of the twelve come up; test_every_tile
    runs all): columns that are no multiple of a tile, the three activations; against float64 with the two products rounded to bfloat16 (a product on
    the edge of a rounding may fall to the other side: 2^-8 of it, and the same once more for the result's rounding)."""
    M, I, K = mik
    torch.manual_seed(42)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * I, K, device="cuda") / math.sqrt(K) * 2).to(torch.bfloat16)
    code = {"silu": ops.GLU_SILU, "gelu_tanh": ops.GLU_GELU_TANH, "clamped": ops.GLU_CLAMPED}[act]
    got = ops.gate_up_tile(x, w, code, 1.5)
    g, u = (x.double() @ w.double().T).to(torch.bfloat16).double().chunk(2, dim=1)
    if act == "silu":
        want = g * torch.sigmoid(g) * u
    elif act == "gelu_tanh":
        want = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3))) * u
    else:
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    torch.testing.assert_close(got.double(), want, atol=2e-2, rtol=2e-2)
    # the activation itself: the hardware's exponential and reciprocal are far below the result's rounding
    assert (got.double() - want).norm() <= 3e-3 * want.norm()


@pytest.mark.parametrize("sums", [True, False], ids=["sums", "gate_up"])
@pytest.mark.parametrize("tile", range(len(TILES)), ids=["x".join(map(str, t[:2])) for t in TILES])
def test_every_tile(ops, tile, sums):
    """Each tile by its index: one chunk of K with a remainder of rows and columns, slices of one chunk, more tiles than the
    chip holds (with slices, for the sums). Small whole numbers, so every product is exact in whatever order it is added
    up and is compared for equality; the activation is SiLU of two exact products (float32, rounded)."""
    import ctypes
    rows, cols, places = TILES[tile]
    cols = cols if sums else cols // 2
    lib = ops.library.load("gemm_tile")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    g = torch.Generator(device="cuda").manual_seed(tile)
    wide = -(-(places * ops.compute_units("cuda") + 1) // (4 * (4 if sums else 1)))      # tiles along W for more than all places
    for M, N, K, splits in ((rows + 3, cols - 4, 64, 1), (2 * rows - 5, 2 * cols + 12, 192, 3 if sums else 1),
                            (3 * rows + 1, (wide - 1) * cols + 4, 512, 4 if sums else 1)):
        x = torch.randint(-3, 4, (M, K), generator=g, device="cuda").to(torch.bfloat16)
        w = torch.randint(-3, 4, (N if sums else 2 * N, K), generator=g, device="cuda").to(torch.bfloat16)
        if not sums:
            x, w = x / 8, w / 8                              # (gates of some units: neither 0 nor 1 after the sigmoid)
        want = x.double() @ w.double().T
        y = torch.full((splits, M, N), float("nan"), device="cuda", dtype=torch.float32 if sums else torch.bfloat16)
        code = lib.ptl_tile_product(ptr(y), ptr(x), ptr(w), M, N, K, ctypes.c_long(K), int(sums), tile, splits, 0,
                                    ctypes.c_float(0.0), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert code == 0
        if sums:
            at = [slice(s * (K // splits), (s + 1) * (K // splits)) for s in range(splits)]
            want = torch.stack([x[:, a].double() @ w[:, a].double().T for a in at])
            assert torch.equal(y.double(), want), f"{M} x {N} x {K}"
        else:
            gate, up = want.to(torch.bfloat16).float().chunk(2, dim=1)
            assert N % 8                            # (silu_mul: the kernel with expf and a division)
            assert torch.equal(y[0], ops.silu_mul(want.to(torch.bfloat16))), f"{M} x {N} x {K}"
            exact = gate.double() * torch.sigmoid(gate.double()) * up.double()
            torch.testing.assert_close(y[0].double(), exact, atol=1e-30, rtol=2 ** -8)


def test_gate_up_tile_has_the_activation_of_the_kernels_beside_it(ops):
    """Every finite bfloat16 gate (columns of x that W picks out, so the products are exact): SiLU has the bits of the
    kernel for up to 64 rows, so a feed-forward's result does not get less exact with the 65th row; with ``hw_silu`` the bits
    of the separate activation kernel, which takes over from 577 rows on."""
    gates = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    gates = gates[gates.isfinite()]
    x = torch.zeros(gates.numel(), 64, dtype=torch.bfloat16)
    x[:, 0], x[:, 1] = gates, 1.25
    w = torch.zeros(128, 64, dtype=torch.bfloat16)
    w[:64, 0], w[64:, 1] = 1.0, 1.0
    x, w = x.cuda(), w.cuda()
    blocked = ops.blocked_weight(w)
    few = torch.cat([ops.gate_up_silu(part, w, blocked=blocked) for part in x.split(60)])
    assert torch.equal(ops.gate_up_tile(x, w), few)
    for I in (64, 60):                          # rows of whole 16-byte pieces, and others: silu_mul has a kernel for either
        dense = torch.cat([x[:, :1].expand(-1, I), x[:, 1:2].expand(-1, I)], dim=1).contiguous()
        assert torch.equal(ops.gate_up_tile(x, w[64 - I:64 + I], hw_silu=True), ops.silu_mul(dense))


@pytest.mark.parametrize("mik", [(1, 4, 4), (3, 36, 100), (8, 8192, 2048), (4, 1000, 1028), (5, 512, 8192), (2, 20, 516),
                                 (7, 2816, 1024)])
def test_gate_up_f32(ops, mik):
    """Pairs of gate and up rows finished in the float32 product of few rows: the bits of the product and the
    activation by themselves, for every number of columns a wave holds."""
    M, I, K = mik
    torch.manual_seed(43)
    x = torch.randn(M, K + 4, device="cuda")[:, :K]
    w = torch.randn(2 * I, K, device="cuda") / math.sqrt(K)
    for act in (ops.GLU_SILU, ops.GLU_GELU_TANH):
        assert torch.equal(ops.gate_up_f32(x, w, act), ops.silu_mul(ops.gemm_nt(x, w), act))
    assert not ops.gate_up_f32_fits(torch.zeros(9, K, device="cuda"), w)
    with pytest.raises(ops.KernelError):
        ops.gate_up_f32(x, w[:-2])


@pytest.mark.parametrize("mik", [(700, 8192, 2048), (17, 4096, 64), (128, 20, 96), (129, 68, 64), (301, 2816, 1024),
                                 (1030, 1028, 1024), (64, 12000, 32)])
def test_gate_up_f32_tiles(ops, mik):
    """A prompt's gate-up product with its activation, in either tile and where a tile has columns past the end: the bits of
    the product and the activation by themselves, also of what is not finite."""
    M, I, K = mik
    torch.manual_seed(49)
    x = torch.randn(M, K + 4, device="cuda")[:, :K]
    w = torch.randn(2 * I, K, device="cuda") / math.sqrt(K)
    x[M - 1, K - 1] = float("inf")
    w[I - 1, 0] = 3.4e38
    for act in (ops.GLU_SILU, ops.GLU_GELU_TANH):
        got, want = ops.gate_up_f32_tiles(x, w, act), ops.silu_mul(ops.gemm_nt(x, w), act)
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    assert not ops.gate_up_f32_tiles_fits(x[:16], w) and not ops.gate_up_f32_tiles_fits(x[:, :K - 4], w[:, :K - 4].contiguous())


@pytest.mark.parametrize("rotated", [True, False])
@pytest.mark.parametrize("case", [(1, 2, 1, 8, 64), (4, 32, 8, 64, 2048), (8, 3, 3, 128, 516), (5, 5, 1, 40, 4100),
                                  (3, 8, 2, 16, 8192)])
def test_qkv_rope_store_f32(ops, case, rotated):
    """The float32 q | k | v projection of few rows with rotation and cache write: the bits of the three kernels it
    stands for, in q and in the pages; rows without a slot write nothing."""
    M, Hq, Hkv, D, K = case
    torch.manual_seed(44)
    P, pages = 4, 6
    x = torch.randn(M, K, device="cuda")
    w = torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") / math.sqrt(K)
    pos = torch.randint(0, 9000, (M,), dtype=torch.int32, device="cuda")
    inv = (10000.0 ** (-torch.arange(0, D, 2).float() / D)).cuda() if rotated else None
    slots = torch.randperm(P * pages)[:M].to(torch.int32)
    slots[M // 2] = -1
    slots = slots.cuda()
    caches = [torch.full((pages, Hkv, P, D), 7.0, device="cuda") for _ in range(4)]
    q = ops.qkv_rope_store_f32(x, w, pos, inv, slots, caches[0], caches[1], Hq, Hkv, D, P)
    y = ops.gemm_nt(x, w).view(M, Hq + 2 * Hkv, D)
    ops.rope_store(y[:, :Hq], y[:, Hq:Hq + Hkv], y[:, Hq + Hkv:], pos, inv, slots, caches[2], caches[3], P)
    assert torch.equal(q, y[:, :Hq])
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])
    assert torch.equal(ops.qkv_rope_store_f32(x, w, pos, inv, None, None, None, Hq, Hkv, D, P), q)
    with pytest.raises(ops.KernelError):
        ops.qkv_rope_store_f32(x, w, pos[:0], inv, slots, caches[0], caches[1], Hq, Hkv, D, P)


@pytest.mark.parametrize("mik", [(17, 64, 64), (33, 8192, 2048), (64, 352, 160), (128, 1024, 4096), (9, 64, 64),
                                 (16, 8192, 2048), (13, 352, 160), (44, 2048, 512), (48, 96, 64)])
def test_gate_up_silu_for_tens_of_rows(ops, mik):
    M, I, K = mik
    torch.manual_seed(23)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * I, K, device="cuda") / math.sqrt(K) * 2).to(torch.bfloat16)
    got = ops.gate_up_silu(x, w, None, ops.blocked_weight(w))
    gu = (x.double() @ w.double().T).float()
    plain = plain_llama.silu(gu[:, :I]) * gu[:, I:]
    torch.testing.assert_close(got.float(), plain, atol=3e-2, rtol=3e-2)
    if M > 16:
        with pytest.raises(ops.KernelError):
            ops.gate_up_silu(x, w)                                       # no blocked copy: not this many rows
    else:                                                                # the kernel for at most 16 rows
        torch.testing.assert_close(ops.gate_up_silu(x, w).float(), plain, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("dims", [(4, 2, 64, 16, 96, 20), (3, 1, 32, 4, 128, 33), (32, 8, 128, 16, 4096, 64),
                                  (6, 3, 96, 8, 224, 128), (32, 8, 64, 16, 2048, 9), (5, 5, 32, 2, 160, 16),
                                  (8, 2, 64, 16, 512, 48), (3, 3, 96, 4, 96, 37)])
def test_qkv_rope_store_for_tens_of_rows(ops, dims):
    """Partial sums of the projection, then one kernel that adds them up, rotates q and k and
    writes k and v into their pages, against the plain formulas; rows whose slot is -1 store
    nothing."""
    Hq, Hkv, D, P, K, M = dims
    torch.manual_seed(24)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    positions = torch.randint(0, 100000, (M,), device="cuda").to(torch.int32)
    positions[0] = 0
    inv_freq = plain_llama.rope_inv_freq_default(500000.0, D).cuda()
    pages = -(-M // P) + 2
    slots = torch.randperm(pages * P, device="cuda")[:M].to(torch.int32)
    slots[3] = -1
    kc = torch.zeros(pages, Hkv, P, D, device="cuda", dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    q = ops.qkv_rope_store(x, w, positions, inv_freq, slots, kc, vc, Hq, Hkv, D, P, None, ops.blocked_weight(w))
    full = (x.double() @ w.double().T).float().cpu()
    cos, sin = plain_llama.rope_cos_sin(inv_freq.cpu(), positions.cpu())
    want_q = plain_llama.apply_rope(full[:, :Hq * D].view(M, Hq, D), cos, sin)
    torch.testing.assert_close(q.float().cpu(), want_q, atol=3e-2, rtol=3e-2)
    want_k = plain_llama.apply_rope(full[:, Hq * D:(Hq + Hkv) * D].view(M, Hkv, D), cos, sin)
    want_v = full[:, (Hq + Hkv) * D:].view(M, Hkv, D)
    flat_k = kc.permute(0, 2, 1, 3).reshape(pages * P, Hkv, D).float().cpu()
    flat_v = vc.permute(0, 2, 1, 3).reshape(pages * P, Hkv, D).float().cpu()
    stored = torch.zeros(pages * P, dtype=torch.bool)
    for m in range(M):
        sl = int(slots[m])
        if sl < 0:
            continue
        stored[sl] = True
        torch.testing.assert_close(flat_k[sl], want_k[m], atol=3e-2, rtol=3e-2)
        torch.testing.assert_close(flat_v[sl], want_v[m], atol=3e-2, rtol=3e-2)
    assert bool((flat_k[~stored] == 0).all()) and bool((flat_v[~stored] == 0).all())
    assert int(stored.sum()) == M - 1


def _rope_reference(x, positions, inv_freq):
    cos, sin = plain_llama.rope_cos_sin(inv_freq, positions)
    return plain_llama.apply_rope(x, cos, sin)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
@pytest.mark.parametrize("dims", [(5, 2, 48, 4), (3, 1, 128, 16), (4, 4, 8, 2)])
def test_rope_store(ops, dtype, dims):
    Hq, Hkv, D, P = dims
    T = 9
    torch.manual_seed(3)
    width = (Hq + 2 * Hkv) * D
    qkv = torch.randn(T, width, device="cuda").to(dtype)
    orig = qkv.clone()
    q = qkv[:, :Hq * D].view(T, Hq, D)
    k = qkv[:, Hq * D:(Hq + Hkv) * D].view(T, Hkv, D)
    v = qkv[:, (Hq + Hkv) * D:].view(T, Hkv, D)
    positions = torch.tensor([0, 1, 2, 77, 1000, 4095, 8191, 100000, 5], dtype=torch.int32, device="cuda")
    inv_freq = plain_llama.rope_inv_freq_default(500000.0, D)
    pages = 7
    kc = torch.zeros(pages, Hkv, P, D, device="cuda", dtype=dtype)
    vc = torch.zeros_like(kc)
    slots = torch.randperm(pages * P)[:T].to(torch.int32).cuda()
    ops.rope_store(q, k, v, positions, inv_freq.cuda(), slots, kc, vc, P)
    o = orig.float().cpu()
    want_q = _rope_reference(o[:, :Hq * D].view(T, Hq, D), positions.cpu(), inv_freq)
    want_k = _rope_reference(o[:, Hq * D:(Hq + Hkv) * D].view(T, Hkv, D), positions.cpu(), inv_freq)
    torch.testing.assert_close(q.float().cpu(), want_q, **tol(dtype))
    # k in the projection buffer is untouched, the cache holds the rotated k and v
    assert torch.equal(k, orig[:, Hq * D:(Hq + Hkv) * D].view(T, Hkv, D))
    for t in range(T):
        page, off = int(slots[t]) // P, int(slots[t]) % P
        torch.testing.assert_close(kc[page, :, off].float().cpu(), want_k[t], **tol(dtype))
        assert torch.equal(vc[page, :, off], v[t])
    # untouched slots stay zero
    mask = torch.ones(pages * P, dtype=torch.bool)
    mask[slots.long().cpu()] = False
    assert torch.all(kc.permute(0, 2, 1, 3).reshape(pages * P, -1)[mask.cuda()] == 0)


def _paged_setup(seq_lens, q_lens, Hkv, D, P, dtype, seed, shuffle=True):
    """Random keys/values laid into shuffled pages; returns tensors and the dense copies."""
    g = torch.Generator().manual_seed(seed)
    n = len(seq_lens)
    pages_per = [-(-s // P) for s in seq_lens]
    total = sum(pages_per) + 3
    perm = torch.randperm(total, generator=g).tolist() if shuffle else list(range(total))
    kc = torch.randn(total, Hkv, P, D, generator=g).to(dtype)    # garbage everywhere first
    vc = torch.randn(total, Hkv, P, D, generator=g).to(dtype)
    maxp = max(pages_per)
    bt = torch.full((n, maxp), -1, dtype=torch.int32)
    dense_k, dense_v = [], []
    it = iter(perm)
    for i, s in enumerate(seq_lens):
        k = torch.randn(s, Hkv, D, generator=g).to(dtype)
        v = torch.randn(s, Hkv, D, generator=g).to(dtype)
        dense_k.append(k.float())
        dense_v.append(v.float())
        for j in range(pages_per[i]):
            pg = next(it)
            bt[i, j] = pg
            lo, hi = j * P, min(s, (j + 1) * P)
            kc[pg, :, :hi - lo] = k[lo:hi].transpose(0, 1)
            vc[pg, :, :hi - lo] = v[lo:hi].transpose(0, 1)
    return kc, vc, bt, dense_k, dense_v


def _attention_case(ops, dtype, seq_lens, q_lens, Hq, Hkv, D, P, window=0, seed=0, boost=None,
                    kernel="generic", splits=1, unroll=0, groups=0, longest=0):
    kc, vc, bt, dk, dv = _paged_setup(seq_lens, q_lens, Hkv, D, P, dtype, seed)
    g = torch.Generator().manual_seed(seed + 100)
    T = sum(q_lens)
    q = torch.randn(T, Hq, D, generator=g).to(dtype)
    if boost is not None:
        boost(q, dk, kc, bt)
    q_start = [0]
    for ql in q_lens:
        q_start.append(q_start[-1] + ql)
    rows = {"mfma": 64, "mfma128": 128}.get(kernel, 16)
    work_seq, work_qoff = [], []
    for s, ql in enumerate(q_lens):
        for off in range(0, ql, rows):
            work_seq.append(s)
            work_qoff.append(off)
    dev = "cuda"
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    out = torch.zeros(T, Hq, D, dtype=dtype, device=dev)
    scale = 1.0 / math.sqrt(D)
    # q as the engine has it: a slice of a wider projection buffer
    wide = torch.zeros(T, Hq * D + 64, dtype=dtype, device=dev)
    wide[:, :Hq * D] = q.to(dev).view(T, Hq * D)
    qd = wide[:, :Hq * D].view(T, Hq, D)
    if kernel == "generic":
        ops.attention_generic(out, qd, kc.to(dev), vc.to(dev), i32(q_start), i32(seq_lens),
                              bt.to(dev), i32(work_seq), i32(work_qoff), scale, window)
    elif kernel in ("mfma", "mfma128"):
        ops.attention_prefill_mfma(out, qd, kc.to(dev), vc.to(dev), i32(q_start), i32(seq_lens),
                                   bt.to(dev), i32(work_seq), i32(work_qoff), scale, window, rows,
                                   groups, longest=longest)
    else:
        assert all(ql == 1 for ql in q_lens)
        ops.attention_decode(out, qd, kc.to(dev), vc.to(dev), i32(q_start), i32(seq_lens),
                             bt.to(dev), len(q_lens), scale, window, splits,
                             matrix_cores=(kernel == "decode_mfma"), unroll=unroll)
    # plain: full causal attention over the sequence, rows of the portion kept
    for i, (s, ql) in enumerate(zip(seq_lens, q_lens)):
        full_q = torch.zeros(s, Hq, D)
        full_q[s - ql:] = q[q_start[i]:q_start[i + 1]].float()
        want = plain_llama.causal_attention(full_q, dk[i], dv[i], scale,
                                            window if window else None)[s - ql:]
        got = out[q_start[i]:q_start[i + 1]].float().cpu()
        torch.testing.assert_close(got, want, **tol(dtype), msg=lambda m: f"sequence {i}: {m}")


@pytest.mark.parametrize("dtype", DT, ids=IDS)
@pytest.mark.parametrize("case", [
    dict(seq_lens=[40], q_lens=[40], Hq=4, Hkv=4, D=64, P=16),            # whole prompt, MHA
    dict(seq_lens=[37, 5, 130], q_lens=[1, 1, 1], Hq=8, Hkv=2, D=48, P=4),  # decode, GQA
    dict(seq_lens=[100, 64, 33], q_lens=[30, 1, 33], Hq=6, Hkv=1, D=128, P=8),  # mixed, MQA
    dict(seq_lens=[70], q_lens=[19], Hq=2, Hkv=1, D=256, P=5),            # big heads, odd page size
    dict(seq_lens=[50, 21], q_lens=[17, 2], Hq=4, Hkv=2, D=8, P=3),       # tiny heads
])
def test_attention_generic(ops, dtype, case):
    _attention_case(ops, dtype, **case)


@pytest.mark.parametrize("V", [1, 4095, 4096, 4097, 3 * 4096 + 5])
def test_token_logprob_at_the_edges_of_chunks(ops, V):
    """Against 64 bits: the sum of V exponentials is off by (V / 256 + 16) 2^-24 of itself (a thread's share and
    the tree) and two roundings of each, the logarithm and the two differences by a few ulps of |x - max|."""
    torch.manual_seed(V)
    x = 3 * torch.randn(3, V + 2, device="cuda")[:, :V]
    if V > 4096:
        x[1, :4096] = float("-inf")                  # a chunk without mass
    t = torch.tensor([0, V - 1, V], dtype=torch.int32, device="cuda")
    got = ops.token_logprob(x, t)
    want = torch.log_softmax(x[:2].double(), -1).gather(1, t[:2, None].long())[:, 0]
    assert float((got[:2].double() - want).abs().max()) <= (V / 256 + 24) * 2.0 ** -24 + 4 * 2.0 ** -24 * 30
    assert got[2] == float("-inf")                   # a token outside the row
    x[0, 0] = float("nan")
    assert torch.isnan(ops.token_logprob(x, t)[0])


@pytest.mark.parametrize("V", [1023, 1025, 32000, 32768, 32769])
def test_token_logprob_of_short_rows(ops, V):
    """Rows of up to 32,768 logits take one launch and allocate their result alone; on both sides of the line the
    bound of the test above, a thread's share being V / 1024 or V / 256 exponentials."""
    test_token_logprob_at_the_edges_of_chunks(ops, V)
    x, t = torch.randn(2, V, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    out = ops.token_logprob(x, t)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == (1 if V <= 32768 else 2)
    assert out.shape == (2,)


@pytest.mark.parametrize("case", [
    # one and two heads a workgroup, tiles of 32, 64 and 128 columns with and without columns beyond the head,
    # blocks of one row, keys one past and short of a tile
    dict(seq_lens=[65, 33, 1], q_lens=[65, 1, 1], Hq=3, Hkv=1, D=64, P=16),
    dict(seq_lens=[130, 31], q_lens=[17, 31], Hq=4, Hkv=4, D=20, P=3),
    dict(seq_lens=[97, 64], q_lens=[97, 64], Hq=6, Hkv=3, D=128, P=16),
    dict(seq_lens=[700, 333], q_lens=[650, 333], Hq=16, Hkv=2, D=64, P=16, window=100),
    dict(seq_lens=[1200], q_lens=[1100], Hq=32, Hkv=8, D=32, P=8),
    dict(seq_lens=[1100], q_lens=[1100], Hq=32, Hkv=8, D=100, P=16),
    dict(seq_lens=[700], q_lens=[500], Hq=64, Hkv=32, D=64, P=16),
])
def test_attention_f32_matrix_cores(ops, case):
    _attention_case(ops, torch.float32, **case)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
@pytest.mark.parametrize("splits", [1, 3, 8])
@pytest.mark.parametrize("case", [
    dict(seq_lens=[37, 5, 130, 1], Hq=8, Hkv=2, D=48, P=4),         # 3 lanes of 4 per key
    dict(seq_lens=[300, 64, 65], Hq=4, Hkv=4, D=64, P=16),          # MHA
    dict(seq_lens=[100, 257], Hq=16, Hkv=2, D=16, P=8),             # 8 heads a kv head: two groups
    dict(seq_lens=[90, 33], Hq=3, Hkv=1, D=128, P=16),              # 3 heads of a tile of 4
    dict(seq_lens=[70], Hq=2, Hkv=1, D=256, P=5),                   # widest head, odd page size
    dict(seq_lens=[50, 200], Hq=6, Hkv=3, D=80, P=16),              # 5 lanes of 8 per key
])
def test_attention_decode(ops, dtype, splits, case):
    _attention_case(ops, dtype, q_lens=[1] * len(case["seq_lens"]), kernel="decode", splits=splits,
                    **case)


@pytest.mark.parametrize("splits", [1, 2, 5])
@pytest.mark.parametrize("case", [
    dict(seq_lens=[300, 64, 65, 1], Hq=4, Hkv=4, D=64, P=16),
    dict(seq_lens=[100, 257], Hq=32, Hkv=2, D=32, P=8),             # 16 heads a kv head
    dict(seq_lens=[90, 33, 700], Hq=3, Hkv=1, D=128, P=16),
    dict(seq_lens=[70, 130], Hq=8, Hkv=2, D=96, P=4),
    dict(seq_lens=[500, 3, 129], Hq=4, Hkv=1, D=64, P=64),          # a page longer than a turn
])
@pytest.mark.parametrize("unroll", [1, 2])
def test_attention_decode_mfma(ops, splits, case, unroll):
    _attention_case(ops, torch.bfloat16, q_lens=[1] * len(case["seq_lens"]), kernel="decode_mfma",
                    splits=splits, unroll=unroll, **case)


@pytest.mark.parametrize("unroll", [1, 2])
@pytest.mark.parametrize("case", [
    # contexts that differ much: workgroups by length, or, beyond 64 sequences, as they come; wide and narrow heads, a
    # window
    dict(seq_lens=[3000] + [17 * i + 5 for i in range(19)], Hq=8, Hkv=2, D=64, P=16, splits=4),
    dict(seq_lens=[7] * 5 + [2500, 1, 1900, 33], Hq=6, Hkv=3, D=128, P=16, splits=3),
    dict(seq_lens=[40 + 3 * i for i in range(69)] + [4100], Hq=4, Hkv=1, D=32, P=8, splits=2),
    dict(seq_lens=[1] * 64 + [3500], Hq=2, Hkv=2, D=96, P=16, splits=2),
    dict(seq_lens=[4000] + [300] * 9, Hq=4, Hkv=2, D=64, P=16, window=3000, splits=2),
    # and the longest on both sides of 512 keys a split
    dict(seq_lens=[1024] + [5] * 15, Hq=4, Hkv=1, D=64, P=16, splits=2),
    dict(seq_lens=[1025] + [5] * 15, Hq=4, Hkv=1, D=64, P=16, splits=2),
])
def test_attention_decode_mfma_shares(ops, case, unroll):
    _attention_case(ops, torch.bfloat16, q_lens=[1] * len(case["seq_lens"]), kernel="decode_mfma", unroll=unroll,
                    **case)


@pytest.mark.parametrize("Hq,Hkv,D", [(4, 1, 32), (3, 1, 64), (2, 2, 96), (5, 2, 128)])
@pytest.mark.parametrize("tile", range(-1, 14))
def test_qkv_rope_store_tile(ops, tile, Hq, Hkv, D):
    """Every tile, rows and heads that do not fill it, rows that are stored nowhere: what the product (float32, rounded once) and
    rope_store give, a bfloat16 rounding apart where the product's last bit differs by the order of its sum."""
    P, pages, K = 8, 40, 192
    torch.manual_seed(100 * D + tile)
    for M in (1, 37, 150):
        x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
        w = (torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") * K ** -0.5).to(torch.bfloat16)
        pos = torch.randint(0, 100000, (M,), device="cuda").int()
        inv = (500000.0 ** (-torch.arange(0, D, 2, device="cuda").double() / D)).float()
        slots = torch.randperm(P * pages, device="cuda")[:M].int()
        slots[M // 2] = -1
        caches = [torch.zeros(pages, Hkv, P, D, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
        for table in (ops.rope_table(pos, inv), None):
            q = ops.qkv_rope_store_tile(x, w, table, slots, *caches[:2], Hq, Hkv, D, P, tile=tile)
            y = (x.float() @ w.float().T).to(torch.bfloat16)
            parts = [t.view(M, -1, D) for t in y.split([Hq * D, Hkv * D, Hkv * D], 1)]
            ops.rope_store(*parts, pos, inv if table is not None else None, slots, *caches[2:], P)
            for got, want in ((q, parts[0]), (caches[0], caches[2]), (caches[1], caches[3])):
                torch.testing.assert_close(got.float(), want.float(), **tol(torch.bfloat16))
        none = ops.qkv_rope_store_tile(x, w, None, None, None, None, Hq, Hkv, D, P, tile=tile)
        assert torch.equal(none, q)


@pytest.mark.parametrize("n,rows,half", [(1, 1, 16), (3, 40, 32), (16, 277, 64), (65, 9, 16), (130, 3, 144)])
def test_rope_tables(ops, n, rows, half):
    """Cosines and sines for many arrays of frequencies, more than a launch takes among them: arrays of other bits (in the last
    number, or a sign of zero) have tables of their own, equal ones share that of their launch's first."""
    pos = torch.randint(0, 5000, (rows,), device="cuda").int()
    base = (10000.0 ** (-torch.arange(half, device="cuda").double() / half)).float()
    base[0] = 0.0
    other, signed = base.clone(), base.clone()
    other[-1] *= 0.5
    signed[0] = -0.0
    freqs = [{2: other, 5: signed, 64: other, 66: other}.get(i, base.clone()) for i in range(n)]
    made = ops.rope_tables(pos, freqs)
    at = [(a - made.tables.data_ptr()) // (8 * rows * half) for a in made.at.tolist()]
    bits = lambda f: f.view(torch.int32).tolist()
    first = [i // ops.ROPE_TABLES * ops.ROPE_TABLES for i in range(n)]
    assert at == [first[i] if bits(freqs[i]) == bits(freqs[first[i]]) else i for i in range(n)]
    for i in range(n):
        angle = (pos[:, None].float() * freqs[i]).double()
        torch.testing.assert_close(made.tables[at[i]].double(), torch.stack([angle.cos(), angle.sin()], 2), atol=3e-7, rtol=0)


@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("M", [37, 150])
def test_qkv_rope_store_tile_copies_what_is_not_turned(ops, value, turned, M):
    """An infinity or a NaN in one column of a value (and, without a rotation, of q and k) stays in that column: the other of the
    pair keeps its number, as a stored product does."""
    P, pages, K, Hq, Hkv, D = 8, 40, 192, 3, 2, 64
    torch.manual_seed(M)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") * K ** -0.5).to(torch.bfloat16)
    for head, col in ((Hq + Hkv, 5), (Hq + 2 * Hkv - 1, 40)) + (() if turned else ((1, 40), (Hq, 5), (Hq + 1, 63))):
        w[head * D + col, 7] = value
    pos = torch.arange(M, device="cuda").int()
    inv = (500000.0 ** (-torch.arange(0, D, 2, device="cuda").double() / D)).float()
    slots = torch.randperm(P * pages, device="cuda")[:M].int()
    caches = [torch.zeros(pages, Hkv, P, D, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    q = ops.qkv_rope_store_tile(x, w, ops.rope_table(pos, inv) if turned else None, slots, *caches[:2], Hq, Hkv, D, P)
    parts = [t.view(M, -1, D) for t in (x.float() @ w.float().T).to(torch.bfloat16).split([Hq * D, Hkv * D, Hkv * D], 1)]
    ops.rope_store(*parts, pos, inv if turned else None, slots, *caches[2:], P)
    for got, want in ((q, parts[0]), (caches[0], caches[2]), (caches[1], caches[3])):
        torch.testing.assert_close(got.float(), want.float(), equal_nan=True, **tol(torch.bfloat16))
    assert int((~torch.isfinite(caches[1].float())).sum()) == 2 * M


@pytest.mark.parametrize("n", [12, 80])
def test_attention_decode_mfma_shares_beside_empty_rows(ops, n):
    """Rows without keys (padding of a recorded step) between sequences of very different lengths: zeros
    there, and the other rows as without them."""
    D, P = 64, 16
    torch.manual_seed(n)
    real = [(3 * i, 3000 if i == 1 else 20 + i) for i in range(n // 3)]
    pages = 200
    kc, vc = (torch.randn(pages, 2, P, D, device="cuda").to(torch.bfloat16) for _ in range(2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    ctx = [0] * n
    for r, c in real:
        ctx[r] = c
    q = torch.randn(n, 8, D, device="cuda").to(torch.bfloat16)
    bt = torch.arange(pages, dtype=torch.int32, device="cuda").repeat(n, 1)

    def run(rows):
        out = torch.full((len(rows), 8, D), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_decode(out, q[rows].contiguous(), kc, vc, i32(list(range(len(rows) + 1))), i32([ctx[r] for r in rows]),
                             bt[rows].contiguous(), len(rows), 0.125, num_splits=2, matrix_cores=True)
        return out.float()
    out = run(list(range(n)))
    for r, c in real:
        torch.testing.assert_close(out[r], run([r])[0], atol=2e-2, rtol=2e-2)
    assert all(bool((out[r] == 0).all()) for r in range(n) if ctx[r] == 0)


def _masked_attention(q, k, v, pos, scale, window=0, keep_first=0, chunk=0, sink=None, gate=None, softcap=0.0):
    """One query [Hq, D] at position pos on keys [pos + 1, Hkv, D] under the masks, in float64."""
    Hq, G = q.shape[0], q.shape[0] // k.shape[1]
    s = torch.einsum("hd,khd->hk", q.double(), k.double().repeat_interleave(G, 1)) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    at = torch.arange(pos + 1)
    first = max(0, pos + 1 - window) if window else pos // chunk * chunk if chunk else 0
    s[:, ~((at >= first) | (at < keep_first))] = -math.inf
    if sink is not None:
        s = torch.cat([s, sink.double()[:, None]], 1)
    p = torch.softmax(s, 1)[:, :pos + 1]
    o = torch.einsum("hk,khd->hd", p, v.double().repeat_interleave(G, 1))
    return o if gate is None else o * torch.sigmoid(gate.double())[:, None]


@pytest.mark.parametrize("masks", ["none", "sink_gate", "softcap", "kept", "kept_softcap_sink_gate", "chunk_sink"])
@pytest.mark.parametrize("n,splits,Hq,Hkv,D", [(9, 2, 4, 2, 64), (33, 4, 3, 1, 128), (64, 2, 8, 8, 32), (65, 3, 4, 2, 96)])
def test_attention_decode_mfma_ragged_batch_gives_what_each_gives_alone(ops, n, splits, Hq, Hkv, D, masks):
    """Workgroups in the order of very different lengths (up to 64 sequences), rows without keys among them, under
    every mask: the bits of each sequence alone, and the plain result at the tolerance of the other cases."""
    P, pages = 16, 300
    g = torch.Generator().manual_seed(n)
    ctx = [3 * i * i % 700 + 1 for i in range(n)]
    ctx[n // 2], ctx[1], ctx[n - 1], ctx[3] = 512 * splits + 300, 512 * splits + 7, 1000, 0
    kc, vc = (torch.randn(pages, Hkv, P, D, generator=g).to(torch.bfloat16) for _ in range(2))
    bt = torch.stack([torch.randperm(pages, generator=g) for _ in range(n)]).to(torch.int32)
    q = torch.randn(n, Hq, D, generator=g).to(torch.bfloat16)
    sink, gate = torch.randn(Hq, generator=g), torch.randn(n, Hq, generator=g)
    kw = {}
    if "kept" in masks:
        kw.update(window=512 * splits + 100, keep_first=21)
    if "chunk" in masks:
        kw.update(chunk=512 * splits + 200)
    if "softcap" in masks:
        kw.update(softcap=2.0)
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    kd, vd, scale = kc.cuda(), vc.cuda(), D ** -0.5

    def run(rows):
        out = torch.full((len(rows), Hq, D), 9.0, dtype=torch.bfloat16, device="cuda")
        more = dict(kw, **({"sink": sink.cuda()} if "sink" in masks else {}),
                    **({"gate": gate[rows].cuda()} if "gate" in masks else {}))
        ops.attention_decode(out, q[rows].cuda(), kd, vd, dev(list(range(len(rows) + 1))), dev([ctx[r] for r in rows]),
                             bt[rows].cuda(), len(rows), scale, num_splits=splits, matrix_cores=True, **more)
        return out
    out = run(list(range(n)))
    for r in range(n):
        assert torch.equal(out[r], run([r])[0]), f"sequence {r}"
    assert bool((out[3] == 0).all())
    for r in (0, 1, n // 2, n - 1):
        c = ctx[r]
        rows = [t[bt[r].long()].transpose(1, 2).reshape(pages * P, Hkv, D)[:c] for t in (kc, vc)]
        want = _masked_attention(q[r], *rows, c - 1, scale, sink=sink if "sink" in masks else None,
                                 gate=gate[r] if "gate" in masks else None, **kw)
        torch.testing.assert_close(out[r].float().cpu(), want.float(), **tol(torch.bfloat16))


@pytest.mark.parametrize("n,Hkv,D", [(33, 8, 64), (64, 8, 64), (64, 5, 128), (56, 8, 96)])
@pytest.mark.parametrize("longest", [1024, 1025, 3000])
def test_attention_decode_mfma_one_split_in_order(ops, n, Hkv, D, longest):
    """More workgroups than compute units and one split: the order by length (from 1,025 keys on) covers every pair, a
    turn that the kv heads do not fill and a short last turn among them; the bits are those of each sequence alone."""
    P, pages, Hq = 16, 200, 2 * Hkv
    g = torch.Generator().manual_seed(n)
    ctx = [7 * i * i % 400 + 1 for i in range(n)]
    ctx[n // 3], ctx[2], ctx[n - 1], ctx[5] = longest, longest - 1, longest // 2, 0
    kc, vc = (torch.randn(pages, Hkv, P, D, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    bt = torch.stack([torch.randperm(pages, generator=g) for _ in range(n)]).to(torch.int32).cuda()
    q = torch.randn(n, Hq, D, generator=g).to(torch.bfloat16).cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")

    def run(rows):
        out = torch.full((len(rows), Hq, D), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_decode(out, q[rows], kc, vc, i32(list(range(len(rows) + 1))), i32([ctx[r] for r in rows]),
                             bt[rows], len(rows), D ** -0.5, num_splits=1, matrix_cores=True)
        return out
    out = run(list(range(n)))
    assert bool((out[5] == 0).all())
    for r in range(n):
        assert torch.equal(out[r], run([r])[0]), f"sequence {r}"


@pytest.mark.parametrize("dtype,D,Hq,Hkv", [(torch.bfloat16, 64, 8, 2), (torch.bfloat16, 128, 3, 3), (torch.float32, 64, 8, 2)])
@pytest.mark.parametrize("n", [1, 9, 64, 65])
def test_attention_decode_parts_meet_in_the_last_workgroup(ops, n, dtype, D, Hq, Hkv):
    """Sequences of no, one and up to 16 parts (of 128 keys at least): the plain result, the same bits from every launch over one
    set of tickets, which are zero again each time."""
    P, pages = 16, 135
    edges = [3000, 0, 128, 129, 2047, 2048, 2049, 2150, 1]
    g = torch.Generator().manual_seed(n)
    ctx = [edges[i] if i < len(edges) else 1 + 97 * i % 700 for i in range(n)]
    ctx = [min(c, pages * P) for c in ctx]
    kc, vc = (torch.randn(pages, Hkv, P, D, generator=g).to(dtype) for _ in range(2))
    bt = torch.stack([torch.randperm(pages, generator=g) for _ in range(n)]).to(torch.int32)
    q = torch.randn(n, Hq, D, generator=g).to(dtype)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tickets = torch.zeros(ops.TICKET * n * Hkv, dtype=torch.int32, device="cuda")
    mfma = dtype == torch.bfloat16
    outs = []
    for _ in range(3):
        out = torch.full((n, Hq, D), 9.0, dtype=dtype, device="cuda")
        ops.attention_decode(out, q.cuda(), kc.cuda(), vc.cuda(), i32(list(range(n + 1))), i32(ctx), bt.cuda(), n, D ** -0.5,
                             num_splits=1 if mfma else 16, matrix_cores=mfma, tickets=tickets, piece=128 if mfma else 0)
        assert int(tickets.abs().max()) == 0
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    for r in range(n):
        if not ctx[r]:
            assert bool((outs[0][r] == 0).all())
            continue
        rows = [t[bt[r].long()].transpose(1, 2).reshape(pages * P, Hkv, D)[:ctx[r]] for t in (kc, vc)]
        want = _masked_attention(q[r], *rows, ctx[r] - 1, D ** -0.5)
        torch.testing.assert_close(outs[0][r].float().cpu(), want.float(), **tol(dtype))


@pytest.mark.parametrize("D", [16, 32, 48, 64, 80, 128])
@pytest.mark.parametrize("heads", [3, 4, 8, 16])
def test_attention_decode_float32_form_by_head_size(ops, D, heads):
    """float32 decode attention takes the matrix-core form for sizes 32 to 64, for larger ones from 8 and for
    smaller ones from 4 heads a kv head on; the others give the bits of the vector form, which rows of odd stride
    always take."""
    n, Hq, Hkv, P, ctx = 3, 2 * heads, 2, 16, [5, 300, 70]
    torch.manual_seed(D)
    kc, vc = (torch.randn(60, Hkv, P, D, device="cuda") for _ in range(2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    bt = torch.randperm(60)[:57].reshape(3, 19).to(dtype=torch.int32, device="cuda")
    q = torch.randn(n, Hq, D, device="cuda")
    outs = []
    for stride in (Hq * D, Hq * D + 1):
        out = torch.empty(n, stride, device="cuda")[:, :Hq * D].unflatten(1, (Hq, D))
        ops.attention_decode(out, q, kc, vc, i32([0, 1, 2, 3]), i32(ctx), bt, n, D ** -0.5, num_splits=2)
        outs.append(out)
    torch.testing.assert_close(outs[0], outs[1], atol=1e-5, rtol=1e-5)
    assert torch.equal(outs[0], outs[1]) == (heads < (8 if D > 64 else 4 if D < 32 else 1))


def test_attention_decode_mfma_refuses_odd_page_size(ops):
    """A page size that is no power of two is for the general kernel; the fast one says so."""
    assert not ops.attention_decode_mfma_fits(torch.bfloat16, 8, 2, 96, 5)
    assert ops.attention_decode_mfma_fits(torch.bfloat16, 8, 2, 96, 4)
    with pytest.raises(ops.KernelError, match="power of two"):
        _attention_case(ops, torch.bfloat16, seq_lens=[70, 130], q_lens=[1, 1], Hq=8, Hkv=2, D=96,
                        P=5, kernel="decode_mfma")


def test_attention_decode_mfma_window(ops):
    _attention_case(ops, torch.bfloat16, seq_lens=[90, 40, 7], q_lens=[1, 1, 1], Hq=4, Hkv=2, D=32,
                    P=8, window=20, kernel="decode_mfma", splits=2)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
def test_attention_decode_window(ops, dtype):
    _attention_case(ops, dtype, seq_lens=[90, 40, 7], q_lens=[1, 1, 1], Hq=4, Hkv=2, D=32, P=8,
                    window=20, kernel="decode", splits=2)


@pytest.mark.parametrize("case", [
    dict(seq_lens=[40], q_lens=[40], Hq=4, Hkv=4, D=64, P=16),
    dict(seq_lens=[200, 64, 33], q_lens=[130, 2, 33], Hq=6, Hkv=1, D=128, P=8),
    dict(seq_lens=[150], q_lens=[70], Hq=2, Hkv=1, D=32, P=32),
    dict(seq_lens=[129, 300], q_lens=[129, 65], Hq=4, Hkv=2, D=96, P=16),
    dict(seq_lens=[450], q_lens=[333], Hq=2, Hkv=1, D=64, P=128),      # a page longer than a tile
    dict(seq_lens=[1, 2, 64, 65], q_lens=[1, 2, 64, 65], Hq=2, Hkv=2, D=64, P=4),
])
@pytest.mark.parametrize("kernel", ["mfma", "mfma128"])
def test_attention_prefill_mfma(ops, case, kernel):
    _attention_case(ops, torch.bfloat16, kernel=kernel, **case)


@pytest.mark.parametrize("kernel", ["mfma", "mfma128"])
def test_attention_prefill_mfma_window(ops, kernel):
    _attention_case(ops, torch.bfloat16, seq_lens=[300, 90], q_lens=[150, 25], Hq=4, Hkv=2, D=64,
                    P=8, window=70, kernel=kernel)


@pytest.mark.parametrize("masks", [dict(), dict(window=70), dict(chunk=96)], ids=["all", "window", "chunk"])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("rows", [64, 128])
def test_attention_prefill_mfma_page_numbers_of_a_wave(ops, D, masks, rows):
    """Pages of 16 rows and more have their numbers read once for the rows of a load instruction: the bits that pages of 8 rows
    give, whose numbers every lane reads, at portions that begin and end inside pages, with pages left of a window given back."""
    torch.manual_seed(D)
    q_lens, lens, Hq, Hkv = [1, 65, 130, 200], [77, 300, 130, 513], 6, 2
    first = [0] * 4
    if "window" in masks:
        first = [max(0, n - q - masks["window"] + 1) for q, n in zip(q_lens, lens)]
    if "chunk" in masks:
        first = [(n - q) // masks["chunk"] * masks["chunk"] for q, n in zip(q_lens, lens)]
    keys = [torch.randn(2, n, Hkv, D).to(torch.bfloat16) for n in lens]
    q = torch.randn(sum(q_lens), Hq, D, device="cuda").to(torch.bfloat16)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    from pytriton_llama_amd.engine.batch import work_items
    lists = [i32(t.tolist()) for t in work_items(q_lens, lens, 0, rows)]
    outs = []
    for P in (8, 16, 32, 128):
        pages = [-(-n // P) for n in lens]
        table = torch.full((4, max(pages)), -1, dtype=torch.int32)
        pool = torch.full((2, sum(pages), Hkv, P, D), float("nan"), dtype=torch.bfloat16)
        order, at = torch.randperm(sum(pages)), 0
        for i, n in enumerate(lens):
            for p in range(pages[i]):
                page, take = int(order[at]), keys[i][:, p * P:(p + 1) * P]
                pool[:, page, :, :take.shape[1]] = take.transpose(1, 2)
                table[i, p] = page if (p + 1) * P > first[i] else -1
                at += 1
        out = torch.zeros_like(q)
        ops.attention_prefill_mfma(out, q, pool[0].cuda(), pool[1].cuda(), i32([0, 1, 66, 196, 396]), i32(lens), table.cuda(),
                                   *lists, D ** -0.5, block_rows=rows, **masks)
        outs.append(out)
    assert bool(torch.isfinite(outs[0].float()).all())
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("rows", [64, 128])
def test_attention_prefill_mfma_portion_without_keys(ops, D, rows):
    """A portion whose context says that there are no keys: zeros, and nothing is read in front of the table; the one beside it as
    by itself. Pages whose numbers are read once for a load instruction's rows and pages whose numbers every lane reads."""
    torch.manual_seed(D)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    q = torch.randn(45, 4, D, device="cuda").to(torch.bfloat16)
    for P in (8, 16):
        k, v = (torch.randn(5 * 16 // P, 2, P, D, device="cuda").to(torch.bfloat16) for _ in range(2))
        table = torch.full((2, 80 // P), -1, dtype=torch.int32)
        table[1] = torch.arange(80 // P)
        outs = []
        for ctx, work in ((0, [0, 1]), (0, [1])):
            out = torch.full((45, 4, D), 9.0, dtype=torch.bfloat16, device="cuda")
            ops.attention_prefill_mfma(out, q, k, v, i32([0, 5, 45]), i32([ctx, 75]), table.cuda(), i32(work), i32([0] * len(work)),
                                       D ** -0.5, block_rows=rows)
            outs.append(out)
        assert bool((outs[0][:5] == 0).all()) and torch.equal(outs[0][5:], outs[1][5:])


def test_attention_prefill_mfma_refuses_odd_page_size(ops):
    """A page size that is no power of two is for the general kernel; the fast one says so."""
    assert not ops.attention_prefill_mfma_fits(torch.bfloat16, 1, 32, 5)
    assert ops.attention_prefill_mfma_fits(torch.bfloat16, 1, 32, 8)
    with pytest.raises(ops.KernelError, match="power of two"):
        _attention_case(ops, torch.bfloat16, seq_lens=[150], q_lens=[70], Hq=2, Hkv=1, D=32, P=5,
                        kernel="mfma")


@pytest.mark.parametrize("groups", [1, 2, 3, 5])
@pytest.mark.parametrize("kernel", ["mfma", "mfma128"])
def test_attention_prefill_mfma_workgroups_share_the_blocks(ops, kernel, groups):
    """Fewer workgroups a head than query blocks: each walks several blocks (of different
    sequences, with and without a prefix in the cache), forwards and backwards over the
    list, and reuses its LDS buffers from one block to the next."""
    _attention_case(ops, torch.bfloat16, seq_lens=[520, 90, 300], q_lens=[390, 90, 129], Hq=4, Hkv=2,
                    D=64, P=16, kernel=kernel, groups=groups)
    _attention_case(ops, torch.bfloat16, seq_lens=[333], q_lens=[333], Hq=2, Hkv=1, D=128, P=8,
                    window=100, kernel=kernel, groups=groups)


@pytest.mark.parametrize("Hq", [2, 264], ids=["two_sides", "one_side"])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("window", [0, 70])
def test_attention_prefill_mfma_sides(ops, D, Hq, window):
    """Few workgroups: two groups of waves share the key tiles of a block (one to six of them, with
    and without a masked last one, shared list and a workgroup a block); many: one group. Tolerance as
    for the other cases: the sums differ in order only, in float32."""
    case = dict(seq_lens=[1, 64, 65, 129, 200, 321], q_lens=[1, 64, 65, 66, 70, 65], Hq=Hq, Hkv=1, D=D, P=16)
    for groups in (0, 3):
        _attention_case(ops, torch.bfloat16, kernel="mfma", window=window, groups=groups, **case)


@pytest.mark.parametrize("Hq,D,lens,q_lens,longest", [
    (64, 64, [520, 90], [390, 25], 0),
    (65, 64, [520, 90], [390, 25], 0),
    (65, 64, [520], [250], 0),
    (33, 32, [700], [512], 512),
    (33, 32, [700], [511], 511),
    (40, 128, [700], [450], 450),
    (40, 96, [700, 64], [450, 64], 450),
    (40, 128, [700, 64, 64], [321, 64, 64], 321)])
def test_attention_prefill_mfma_sides_up_to_two_workgroups_a_unit(ops, Hq, D, lens, q_lens, longest):
    """Both sides of the lines between one group of waves and two where there are one to two workgroups a compute unit (which
    of them it is on 256 units: test_host_launches.py)."""
    _attention_case(ops, torch.bfloat16, seq_lens=lens, q_lens=q_lens, Hq=Hq, Hkv=1, D=D, P=16, kernel="mfma", longest=longest)


@pytest.mark.parametrize("rows,groups", [(300, 0), (300, 2), (257, 0)])
@pytest.mark.parametrize("masks", ["kept", "kept_sink_gate", "softcap_sink_gate", "chunk_sink"])
def test_attention_prefill_mfma_sides_with_masks(ops, masks, rows, groups):
    """Two groups of waves on blocks of four and more key tiles whose walk is two stretches (kept first keys and a
    window), with sinks and gates, and under capped scores and chunks."""
    Hq, Hkv, D, P, total = 2, 1, 64, 16, 900
    kc, vc, bt, dk, dv = _paged_setup([total], [rows], Hkv, D, P, torch.bfloat16, 5)
    g = torch.Generator().manual_seed(rows)
    q = torch.randn(rows, Hq, D, generator=g).to(torch.bfloat16)
    sink, gate = torch.randn(Hq, generator=g), torch.randn(rows, Hq, generator=g)
    kw = {}
    if "kept" in masks:
        kw.update(window=310, keep_first=70)
    if "chunk" in masks:
        kw.update(chunk=400)
    if "softcap" in masks:
        kw.update(softcap=2.0)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    off = list(range(0, rows, 64))[::-1]
    out = torch.zeros(rows, Hq, D, dtype=torch.bfloat16, device="cuda")
    ops.attention_prefill_mfma(out, q.cuda(), kc.cuda(), vc.cuda(), i32([0, rows]), i32([total]), bt.cuda(),
                               i32([0] * len(off)), i32(off), D ** -0.5, groups=groups,
                               **kw, **({"sink": sink.cuda()} if "sink" in masks else {}),
                               **({"gate": gate.cuda()} if "gate" in masks else {}))
    for r in (0, 1, 63, 64, 100, 200, rows - 1):
        pos = total - rows + r
        want = _masked_attention(q[r], dk[0][:pos + 1], dv[0][:pos + 1], pos, D ** -0.5, sink=sink if "sink" in masks else None,
                                 gate=gate[r] if "gate" in masks else None, **kw)
        torch.testing.assert_close(out[r].float().cpu(), want.float(), **tol(torch.bfloat16))


@pytest.mark.parametrize("n_dec", [0, 2])
def test_short_portion_beside_decoding_requests_takes_two_sides(ops, n_dec):
    """PagedAttention: a portion of 70 rows behind a prefix of 900, alone (the bits of one group of waves) and beside
    decoding requests (of two); both near the plain result."""
    from types import SimpleNamespace

    from pytriton_llama_amd.parts import attention as part
    D, P, rows, total = 64, 16, 70, 970
    att = part.PagedAttention(128, 2, 1, D)
    lens, q_lens = [40] * n_dec + [total], [1] * n_dec + [rows]
    kc, vc, bt, dk, dv = _paged_setup(lens, q_lens, 1, D, P, torch.bfloat16, 3)
    torch.manual_seed(0)
    q = torch.randn(n_dec + rows, 2, D).to(torch.bfloat16)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    q_start = [0]
    for n in q_lens:
        q_start.append(q_start[-1] + n)
    off = [64, 0]
    lists = (i32([n_dec] * 2), i32(off))
    ctx = SimpleNamespace(num_decode_seqs=n_dec, num_seqs=n_dec + 1, q_start=i32(q_start), ctx_len=i32(lens), q_lens=q_lens,
                          ctx_lens=lens, work={part.PORTIONS_64: lists, part.PORTIONS_128: lists})
    out = torch.zeros(n_dec + rows, 2, D, dtype=torch.bfloat16, device="cuda")
    att.attend(out, q.cuda(), SimpleNamespace(k=kc.cuda(), v=vc.cuda(), page_size=P), ctx, SimpleNamespace(block_table=bt.cuda()))
    sides = []
    for longest in (rows, 0):
        o = torch.zeros_like(out)
        ops.attention_prefill_mfma(o, q.cuda(), kc.cuda(), vc.cuda(), i32(q_start), i32(lens), bt.cuda(), *lists, D ** -0.5,
                                   longest=longest)
        sides.append(o[n_dec:])
    assert not torch.equal(*sides)
    assert torch.equal(out[n_dec:], sides[1 if n_dec else 0])
    for r in (0, 69):
        pos = total - rows + r
        want = _masked_attention(q[n_dec + r], dk[-1][:pos + 1], dv[-1][:pos + 1], pos, D ** -0.5)
        torch.testing.assert_close(out[n_dec + r].float().cpu(), want.float(), **tol(torch.bfloat16))


@pytest.mark.parametrize("D", [64, 128])
def test_attention_prefill_mfma_short_portions_keep_one_side(ops, D):
    """Portions of up to 256 rows give the bits of one group of waves (which a launch of many heads always takes),
    longer ones those of two; nothing known: two."""
    P, total = 16, 400
    for rows in (60, 256, 257):
        kc, vc, bt, _, _ = _paged_setup([total], [rows], 1, D, P, torch.bfloat16, 3)
        torch.manual_seed(rows)
        q = torch.randn(rows, 1, D, device="cuda").to(torch.bfloat16)
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
        off = list(range(0, rows, 64))[::-1]

        def run(heads, **kw):
            out = torch.zeros(rows, heads, D, dtype=torch.bfloat16, device="cuda")
            ops.attention_prefill_mfma(out, q.expand(rows, heads, D).contiguous(), kc.cuda(), vc.cuda(), i32([0, rows]),
                                       i32([total]), bt.cuda(), i32([0] * len(off)), i32(off), D ** -0.5, **kw)
            return out[:, 0]
        one = run(264)
        assert torch.equal(run(2, longest=rows), one) == (rows <= 256)
        assert not torch.equal(run(2), one)
        torch.testing.assert_close(run(2).float(), one.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("D,Hkv,G,P", [(64, 8, 4, 16), (64, 1, 2, 64), (128, 2, 3, 16), (128, 8, 16, 32)])
@pytest.mark.parametrize("masks", [dict(), dict(window=70), dict(chunk=96)], ids=["all", "window", "chunk"])
@pytest.mark.parametrize("contexts", [[1], [40, 0, 700, 129, 0], [17, 1100, 0, 256, 33, 512, 90, 1, 300], [31 + 7 * i for i in range(65)]],
                         ids=["one", "five", "listed", "many"])
def test_attention_of_a_step_in_one_launch(ops, D, Hkv, G, P, masks, contexts):
    """The bits of the decode kernel and of one group of waves for the portions (which portions of few rows always take), with
    rows without keys, an empty work item, shared blocks, sinks and gates, twice over the same tickets, and in a replayed graph."""
    torch.manual_seed(D + len(contexts))
    n, q_lens, lens = len(contexts), [70, 200], [130, 460]
    Hq, rows, seqs = Hkv * G, [1] * n + q_lens, contexts + lens
    T, pages = sum(rows), [-(-k // P) for k in seqs]
    order, at = torch.randperm(sum(pages) + 1).tolist(), 0
    table = torch.full((len(seqs), max(pages)), -1, dtype=torch.int32)
    for i, k in enumerate(pages):
        table[i, :k] = torch.tensor(order[at:at + k], dtype=torch.int32)
        at += k
    k, v = (torch.randn(sum(pages) + 1, Hkv, P, D, device="cuda").to(torch.bfloat16) for _ in range(2))
    q = torch.randn(T, Hq, D, device="cuda").to(torch.bfloat16)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    start = i32([0] + torch.tensor(rows).cumsum(0).tolist())
    from pytriton_llama_amd.engine.batch import work_items
    ws, wo = (t.tolist() for t in work_items(rows, seqs, n, 64))
    ws, wo = i32(ws + [n + 1]), i32(wo + [256])
    extras = dict(masks, sink=torch.randn(Hq, device="cuda"), gate=torch.randn(T, Hq, device="cuda"))
    tables = (start, i32(seqs), table.cuda())
    tickets = torch.zeros(ops.TICKET * n * Hkv, dtype=torch.int32, device="cuda")
    for splits, groups in ((1, 0), (3, 2)):
        apart = torch.zeros_like(q)
        ops.attention_decode(apart, q, k, v, *tables, n, D ** -0.5, num_splits=splits, matrix_cores=True, **extras)
        ops.attention_prefill_mfma(apart, q, k, v, *tables, ws, wo, D ** -0.5, groups=groups, longest=1, **extras)

        def step(out):
            ops.attention_step(out, q, k, v, *tables, n, ws, wo, D ** -0.5, num_splits=splits, groups=groups, tickets=tickets,
                               **extras)
            return out
        for _ in range(2):
            assert torch.equal(step(torch.zeros_like(q)), apart)
        assert not bool(tickets.any())
        out, graph = torch.zeros_like(q), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step(out)
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            assert torch.equal(out, apart)


@pytest.mark.parametrize("D,Hkv,G", [(64, 2, 4), (128, 3, 2)])
@pytest.mark.parametrize("where,value", [("key", math.nan), ("key", math.inf), ("value", math.nan), ("query", math.nan)])
def test_attention_gives_nans_for_scores_that_are_no_numbers(ops, D, Hkv, G, where, value):
    """Decode attention with one part a sequence and with several, and both kinds of rows in one launch: NaNs where the plain
    attention has them, the other heads' and sequences' numbers as it has them, zeros for a row without keys."""
    torch.manual_seed(D)
    P, Hq, contexts, rows = 16, Hkv * G, [300, 0, 5, 700], [1, 1, 1, 1, 40]
    lens, n = contexts + [90], 4
    pages = [-(-c // P) for c in lens]
    table, at = torch.full((5, max(pages)), -1, dtype=torch.int32), 0
    for i, k in enumerate(pages):
        table[i, :k] = torch.arange(at, at + k)
        at += k
    k, v = (torch.randn(at, Hkv, P, D).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(sum(rows), Hq, D).abs().to(torch.bfloat16)          # (an infinite key then is an infinite score)
    for seq, key in ((0, 10), (3, 650), (4, 20)):
        page, off = int(table[seq, key // P]), key % P
        if where == "query":
            q[seq, 1, 3] = value
        else:
            (k if where == "key" else v)[page, 0, off, 3] = value
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    starts = [0, 1, 2, 3, 4, 44]
    want = torch.zeros(44, Hq, D, dtype=torch.float64)
    for seq, c in enumerate(lens):
        keys, values = (t[table[seq, :pages[seq]].long()].transpose(1, 2).reshape(-1, Hkv, D)[:c] for t in (k, v))
        for i in range(rows[seq] if c else 0):
            pos = c - rows[seq] + i
            want[starts[seq] + i] = _masked_attention(q[starts[seq] + i], keys[:pos + 1], values[:pos + 1], pos, D ** -0.5)
    assert 0 < int(want[:4].isnan().sum()) < want[:4].numel() // 2
    tables, dev = (i32(starts), i32(lens), table.cuda()), (q.cuda(), k.cuda(), v.cuda())
    for splits, piece in ((1, 1 << 20), (1, 128), (4, 0)):
        out = torch.full((44, Hq, D), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_decode(out, *dev, *tables, n, D ** -0.5, num_splits=splits, matrix_cores=True, piece=piece)
        torch.testing.assert_close(out[:n].double().cpu(), want[:n], equal_nan=True, **tol(torch.bfloat16))
    for splits in (1, 4):
        out = torch.full((44, Hq, D), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_step(out, *dev, *tables, n, i32([4]), i32([0]), D ** -0.5, num_splits=splits)
        torch.testing.assert_close(out.double().cpu(), want, equal_nan=True, **tol(torch.bfloat16))


def test_attention_of_a_step_refuses(ops):
    """What one of the two kernels does not take, and steps without one kind of rows."""
    bf = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")

    def call(D=64, Hq=2, P=16, dtype=torch.bfloat16, n_seq=1, work=1, rows=3):
        q, kv = bf(rows, Hq, D).to(dtype), bf(2, 1, P, D).to(dtype)
        ops.attention_step(torch.empty_like(q), q, kv, kv, i32([0, 1, rows]), i32([1, 2]), i32([[0], [1]]), n_seq, i32([1] * work),
                           i32([0] * work), 0.1)
    call()
    for wrong in (dict(D=32), dict(D=96), dict(P=8), dict(P=24), dict(Hq=17), dict(dtype=torch.float32), dict(n_seq=0),
                  dict(n_seq=2), dict(work=0)):
        with pytest.raises(ops.KernelError, match="attention_step"):
            call(**wrong)


@pytest.mark.parametrize("D,n_dec,rows,one", [(64, 2, 70, False), (64, 3, 70, True), (128, 7, 70, False), (128, 8, 70, True),
                                              (96, 8, 70, False), (64, 8, 64 * 257, False), (128, 8, 64 * 129, False)])
def test_which_steps_take_one_launch(ops, D, n_dec, rows, one):
    """Two heads on 256 compute units: up to two workgroups a unit at head size 64, one above; from three and eight decoding
    requests on."""
    from types import SimpleNamespace

    from pytriton_llama_amd.parts import attention as part
    if ops.compute_units(torch.device("cuda", 0)) != 256:
        pytest.skip("the sizes are for 256 compute units")
    ctx = SimpleNamespace(num_seqs=n_dec + 1, work={part.PORTIONS_64: (torch.zeros(-(-rows // 64)), None)})
    q = torch.zeros(1, 2, D, dtype=torch.bfloat16, device="cuda")
    assert part.PagedAttention(128, 2, 1, D)._one_launch(n_dec, q, ctx, 16) == one


def test_attention_prefill_mfma_plan(ops):
    """128-row blocks once there are 1.25 t of them (t: workgroups a head can have resident);
    a workgroup a block up to 2 t blocks, t workgroups beyond; never more workgroups than blocks."""
    dev = torch.device("cuda", 0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    t = max(1, 3 * cus // 32)
    plan = lambda n64, n128: ops.attention_prefill_mfma_plan(dev, 32, 64, n64, n128)
    assert plan(3, 2) == (64, 3)
    assert plan(2 * t, t) == (64, 2 * t)
    assert plan(2 * t + 2, t + 1) == (64, t)
    n128 = -(-5 * t // 4)
    assert plan(2 * n128, n128) == (128, n128)
    assert plan(2 * n128 - 2, n128 - 1)[0] == 64
    assert plan(8 * t, 4 * t) == (128, t)
    assert ops.attention_prefill_mfma_plan(dev, 4 * cus, 128, 1, 1) == (64, 1)
    # head sizes above 64: 128-row blocks from 0.5 t blocks on when a context has 4,096 keys
    t128 = max(1, 2 * cus // 32)
    wide = lambda n128, keys: ops.attention_prefill_mfma_plan(dev, 32, 128, 2 * n128, n128, keys)
    half = -(-t128 // 2)
    assert wide(half, 4096) == (128, half) and wide(half, 4095)[0] == 64 and wide(half, 0)[0] == 64
    if half > 1:
        assert wide(half - 1, 16384)[0] == 64
    assert plan(2 * half, half) == ops.attention_prefill_mfma_plan(dev, 32, 64, 2 * half, half, 16384)


def test_attention_prefill_mfma_long(ops):
    """Many key tiles, a prefix in the cache, rows that end inside a block."""
    _attention_case(ops, torch.bfloat16, seq_lens=[1100, 700], q_lens=[777, 300], Hq=4, Hkv=1, D=64,
                    P=16, kernel="mfma128")


def _hot_keys(dk, kc, bt, P, seq, places, value=2.0):
    """Key ``places[h]`` of kv head h of sequence ``seq`` becomes ``value`` in every element, in
    the pages and in the dense copy: a query of the same direction then reads that key alone."""
    D = kc.shape[-1]
    for h, pos in enumerate(places):
        kc[int(bt[seq, pos // P]), h, pos % P] = value
        dk[seq][pos, h] = torch.full((D,), value)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("keys", [8200, 16400])
def test_attention_decode_long_contexts(ops, D, keys):
    """Eight decoded rows over up to 8,200 and 16,400 keys with 32 heads on 8 kv heads, cut into
    the splits the attention part plans for such a step. In every group of four heads, two
    queries point at one key each (the first key, the last, both sides of a page's and of a
    split's edge, ...), so that a tile that is dropped or read twice changes the whole row, and
    two are random with scores spread over about three, so that the sums over all tiles count."""
    from types import SimpleNamespace

    from pytriton_llama_amd.parts.attention import PagedAttention
    Hq, Hkv, P = 32, 8, 16
    G = Hq // Hkv
    seq_lens = [keys, keys - 7, keys - 16, keys // 2 + 1, keys - 1, 4100, keys, keys - 33]
    n = len(seq_lens)
    part = PagedAttention(hidden_size=Hq * D, num_heads=Hq, num_kv_heads=Hkv, head_dim=D)
    splits = part.decode_splits(SimpleNamespace(ctx_lens=seq_lens), n, True, torch.device("cuda", 0))
    assert splits >= 4, "the case is meant to run with several splits"
    kc, vc, bt, dk, dv = _paged_setup(seq_lens, [1] * n, Hkv, D, P, torch.bfloat16, seed=keys + D)
    g = torch.Generator().manual_seed(5)
    q = (3.0 * torch.randn(n, Hq, D, generator=g)).to(torch.bfloat16)
    per_split = -(-seq_lens[0] // splits)
    special = [0, 1, P - 1, P, 127, 128, per_split - 1, per_split, 2 * per_split + 1, 4095, 4096]
    for i, s in enumerate(seq_lens):
        places = [(special[(i * Hkv + h) % len(special)] if (i + h) % 3 else s - 1 - h) % s
                  for h in range(Hkv)]
        _hot_keys(dk, kc, bt, P, i, places)
        q[i, 0::G] = 2.0
        q[i, 1::G] = 2.0
    dev = "cuda"
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    out = torch.zeros(n, Hq, D, dtype=torch.bfloat16, device=dev)
    scale = 1.0 / math.sqrt(D)
    ops.attention_decode(out, q.to(dev), kc.to(dev), vc.to(dev), i32(list(range(n + 1))),
                         i32(seq_lens), bt.to(dev), n, scale, 0, splits, matrix_cores=True)
    for i, s in enumerate(seq_lens):
        want = plain_llama.causal_attention(q[i:i + 1].float(), dk[i], dv[i], scale,
                                            query_positions=[s - 1])[0]
        got = out[i].float().cpu()
        # the rows that point at one key return its value
        assert float(want[0::G].abs().max()) > 0.5
        err = float((got - want).abs().max()) / float(want.abs().max())
        assert err < 2e-2, f"sequence {i} ({s} keys, {splits} splits): error {err:.3g} of the largest value"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("prefix,rows", [(14336, 2048), (8192, 8192)])
def test_attention_prefill_mfma_long_prefix(ops, D, prefix, rows):
    """A portion of 2,048 rows behind 14,336 keys in the cache (one workgroup a block by the
    plan for 32 heads: 64-row blocks at head size 64, 128-row blocks at head size 128, where
    the long prefix decides) and one of 8,192 rows behind 8,192 (128-row blocks, the list shared
    by fewer workgroups than blocks), with the block size and workgroups that the plan gives
    and the work list the engine builds. Compared for the first, a middle and the last 128 rows;
    one query head a group points at one far key, the others are random with wide scores."""
    from pytriton_llama_amd.engine.batch import work_items
    Hq, Hkv, P = 32, 8, 16
    G = Hq // Hkv
    total = prefix + rows
    kc, vc, bt, dk, dv = _paged_setup([total], [rows], Hkv, D, P, torch.bfloat16, seed=prefix + D)
    g = torch.Generator().manual_seed(6)
    q = (3.0 * torch.randn(rows, Hq, D, generator=g)).to(torch.bfloat16)
    q[:, 0::G] = 2.0
    _hot_keys(dk, kc, bt, P, 0, [0, 15, 16, 4095, 8192, prefix - 1, prefix, prefix + 5])
    n64, n128 = -(-rows // 64), -(-rows // 128)
    block_rows, groups = ops.attention_prefill_mfma_plan(torch.device("cuda", 0), Hq, D, n64, n128, total)
    if rows == 8192:
        assert block_rows == 128 and groups < n128, "the case is meant to share the list"
    elif torch.cuda.get_device_properties(0).multi_processor_count <= 256:
        # few blocks, all of them long: 128 rows a block at head size 128, 64 at head size 64
        assert block_rows == (128 if D > 64 else 64) and groups == (n128 if D > 64 else n64)
    ws, wo = work_items([rows], [total], 0, block_rows)
    dev = "cuda"
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    out = torch.zeros(rows, Hq, D, dtype=torch.bfloat16, device=dev)
    scale = 1.0 / math.sqrt(D)
    ops.attention_prefill_mfma(out, q.to(dev), kc.to(dev), vc.to(dev), i32([0, rows]), i32([total]),
                               bt.to(dev), torch.from_numpy(ws).to(dev), torch.from_numpy(wo).to(dev),
                               scale, 0, block_rows, groups)
    out = out.float().cpu()
    for lo in (0, (rows // 2 // 128) * 128 - 64, rows - 128):
        sel = list(range(lo, lo + 128))
        want = plain_llama.causal_attention(q[sel].float(), dk[0], dv[0], scale,
                                            query_positions=[prefix + r for r in sel])
        err = float((out[sel] - want).abs().max()) / float(want.abs().max())
        assert err < 2e-2, f"rows {lo}..{lo + 127} behind {prefix} keys: error {err:.3g} of the largest value"


@pytest.mark.parametrize("kernel", ["decode", "decode_mfma", "mfma", "mfma128"])
def test_attention_far_key_stands_out_fast_kernels(ops, kernel):
    def boost(q, dk, kc, bt):
        direction = torch.ones(64) * 2.0
        q[-1, :, :] = direction.to(q.dtype)
        page = int(bt[0, 0])
        kc[page, :, 3] = direction.to(kc.dtype)
        dk[0][3] = direction
    ql = 2 if kernel.startswith("mfma") else 1
    _attention_case(ops, torch.bfloat16, seq_lens=[700], q_lens=[ql], Hq=2, Hkv=1, D=64, P=16,
                    boost=boost, kernel=kernel, splits=4)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
def test_attention_window(ops, dtype):
    _attention_case(ops, dtype, seq_lens=[90, 40], q_lens=[25, 1], Hq=4, Hkv=2, D=32, P=8, window=20)


@pytest.mark.parametrize("dtype", DT, ids=IDS)
def test_attention_far_key_stands_out(ops, dtype):
    """One early key is made to dominate the last query's scores, so a kernel
    that drops or misplaces a far page fails."""
    def boost(q, dk, kc, bt):
        # key 3 of sequence 0 (first page) aligned with the last query, head 0
        direction = torch.ones(32) * 3.0
        q[-1, :, :] = direction.to(q.dtype)
        page = int(bt[0, 0])
        kc[page, :, 3] = direction.to(kc.dtype)
        dk[0][3] = direction
    _attention_case(ops, dtype, seq_lens=[300], q_lens=[1], Hq=2, Hkv=1, D=32, P=16, boost=boost)


def test_attention_page_placement_does_not_matter(ops):
    """The same keys in differently permuted pages give the same output bit for bit."""
    outs = []
    for shuffle_seed in (0, 1):
        kc, vc, bt, dk, dv = _paged_setup([75], [75], 2, 32, 8, torch.float32, seed=4, shuffle=True)
        if shuffle_seed:
            perm = torch.randperm(kc.shape[0], generator=torch.Generator().manual_seed(99))
            inv = torch.empty_like(perm)
            inv[perm] = torch.arange(len(perm))
            kc, vc = kc[perm], vc[perm]
            bt = torch.where(bt >= 0, inv[bt.clamp(min=0).long()].to(torch.int32), bt)
        q = torch.randn(75, 4, 32, generator=torch.Generator().manual_seed(8))
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
        out = torch.zeros(75, 4, 32, device="cuda")
        ops.attention_generic(out, q.cuda(), kc.cuda(), vc.cuda(), i32([0, 75]), i32([75]),
                              bt.cuda(), i32([0, 0, 0, 0, 0]), i32([0, 16, 32, 48, 64]),
                              1 / math.sqrt(32), 0)
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("V", [1003, 4096, 8193, 128256])
def test_argmax(ops, V):
    torch.manual_seed(5)
    logits = torch.randn(6, V, device="cuda")
    logits[2, 7] = logits[2, V - 100] = 50.0       # a tie goes to the lowest id, across chunks too
    logits[3, 401] = logits[3, 402] = 70.0         # ... and inside one 16-byte load
    logits[4, V - 1] = 60.0
    logits[1, 0] = logits[5, 9] = float("nan")     # a NaN is never the choice
    got = ops.argmax(logits).cpu()
    want = torch.argmax(torch.nan_to_num(logits.cpu(), nan=-float("inf")), dim=-1)
    want[2], want[3] = 7, 401
    assert got.tolist() == want.tolist()
    # the kernel can leave the choices in pinned host memory as well
    host = torch.full((8,), -1, dtype=torch.int32).pin_memory()
    again = ops.argmax(logits, host_out=host)
    torch.cuda.synchronize()
    assert again.cpu().tolist() == want.tolist() and host.tolist() == want.tolist() + [-1, -1]


def test_sample_top_p_distribution(ops):
    """The kernel's nucleus equals the plain rule's, and the draw follows it."""
    torch.manual_seed(6)
    R, V = 5, 777
    logits = (3 * torch.randn(R, V)).cuda()
    temperature = torch.tensor([0.8, 1.0, 0.5, 2.0, 0.7]).cuda()
    top_p = torch.tensor([0.9, 1.0, 0.3, 0.95, 1e-6]).cuda()
    u = torch.tensor([0.0, 0.5, 0.999, 0.25, 0.7]).cuda()
    tok, probs = ops.sample_top_p(logits, temperature, top_p, u, return_probs=True)
    for r in range(R):
        want = plain_llama.top_p_probs(logits[r].cpu(), float(temperature[r]), float(top_p[r]))
        torch.testing.assert_close(probs[r].cpu().double(), want, atol=1e-5, rtol=1e-4)
        # inverse CDF in vocabulary order
        cdf = torch.cumsum(want, 0)
        expect = int(torch.searchsorted(cdf, torch.tensor(float(u[r]), dtype=torch.double), right=True))
        got = int(tok[r])
        assert want[got] > 0
        assert abs(float(cdf[got]) - float(cdf[min(expect, V - 1)])) < 1e-4 or got == expect
    # top_p -> 0 is greedy
    assert int(tok[4]) == int(torch.argmax(logits[4]))


def test_sample_top_p_frequencies(ops):
    """Many draws with different uniforms reproduce the probabilities."""
    logits = torch.tensor([[2.0, 1.0, 0.0, -1.0, 0.5, -30.0]]).cuda().repeat(4000, 1)
    t = torch.full((4000,), 1.0).cuda()
    p = torch.full((4000,), 0.9).cuda()
    u = torch.rand(4000, generator=torch.Generator().manual_seed(1)).cuda()
    tok = ops.sample_top_p(logits, t, p, u).cpu()
    want = plain_llama.top_p_probs(logits[0].cpu(), 1.0, 0.9)
    freq = torch.bincount(tok.long(), minlength=6).double() / 4000
    assert torch.all((freq - want).abs() < 0.03), (freq, want)
    assert freq[want == 0].sum() == 0


@pytest.mark.parametrize("V", [16384, 20000, 128256])
def test_sample_top_p_one_and_many_workgroups_a_row_agree(ops, V):
    """The one-kernel and the many-workgroup samplers follow the same rule: the same nucleus
    (up to a token at its edge, where float32 sums taken in another order meet top_p) and the
    same draw, for peaked, ordinary and flat rows, top_p from almost 0 to 1, -inf and NaN
    logits, and u at both ends."""
    g = torch.Generator().manual_seed(V)
    R = 12
    logits = torch.randn(R, V, generator=g)
    scale = torch.tensor([8.0, 4.0, 2.0, 1.0, 0.3, 0.02, 3.0, 3.0, 3.0, 3.0, 3.0, 1e-3]).view(R, 1)
    logits = logits * scale
    logits[6, ::3] = float("-inf")
    logits[7, 5] = float("nan")
    logits[8, V - 1] = 30.0                                  # the last token holds the mass
    t = torch.tensor([0.6, 1.0, 0.8, 1.5, 1.0, 1.0, 0.7, 0.7, 0.7, 0.7, 0.7, 1.0])
    p = torch.tensor([0.9, 0.9, 0.5, 0.95, 0.9, 0.9, 0.9, 0.9, 0.9, 1.0, 1e-6, 0.37])
    u = torch.tensor([0.0, 0.3, 0.999999, 0.5, 0.77, 0.123, 0.9, 0.2, 0.5, 0.6, 0.4, 0.999])
    args = [a.cuda() for a in (logits, t, p, u)]
    tok1, pr1 = ops.sample_top_p(*args, return_probs=True, wide=False)
    tokw, prw = ops.sample_top_p(*args, return_probs=True, wide=True)
    tokw2 = ops.sample_top_p(*args, wide=True)
    assert tokw.tolist() == tokw2.tolist()                    # the same call, the same tokens
    for r in range(R):
        a, b = pr1[r].double().cpu(), prw[r].double().cpu()
        assert abs(float(b.sum()) - 1) < 1e-4
        assert float((a - b).abs().sum()) < 2e-3, r
        # the draw: same token, or a neighbour in the cumulative distribution
        ca = torch.cumsum(b, 0)
        assert int(tokw[r]) == int(tok1[r]) or abs(float(ca[int(tokw[r])] - ca[int(tok1[r])])) < 1e-3, r
        assert b[int(tokw[r])] > 0
    assert int(tokw[8]) == V - 1 and int(tokw[10]) == int(torch.argmax(logits[10]))
    for r in (0, 2, 4):                                       # against the plain rule
        want = plain_llama.top_p_probs(torch.nan_to_num(logits[r], nan=float("-inf")), float(t[r]), float(p[r]))
        assert float((prw[r].double().cpu() - want).abs().sum()) < 1e-3


def test_sampler_at_vocabulary_size(ops):
    """A request draws the same tokens alone, with others and beside a greedy one, with and without a seed of its own, with
    tokens on their way or in its list, and on the host too."""
    from pytriton_llama_amd.engine.request import Request, SamplingParams
    from pytriton_llama_amd.sampling import Sampler
    V, R = 32000, 7
    logits = (2 * torch.randn(R + 1, V, generator=torch.Generator().manual_seed(60))).cuda()
    params = [SamplingParams(temperature=0.7 + 0.1 * i, top_p=(0.9, 1.0, 0.95)[i % 3], seed=(None, 5, 6)[i % 3]) for i in range(R)]
    requests = [Request(("chat é", i), [1, 2], p, output=[3] * (i % 4)) for i, p in enumerate(params)]
    greedy = Request("greedy", [1], SamplingParams(temperature=0.0))
    sampler = Sampler(seed=8)
    for ahead in (0, 2):
        host = torch.full((R + 1,), -1, dtype=torch.int32).pin_memory()
        together = sampler.sample_device(logits[:R], requests, ahead, host).tolist()
        assert host.tolist() == together + [-1]                 # (tolist has waited for the stream)
        assert together == [int(sampler.sample_device(logits[i:i + 1], [r], ahead)) for i, r in enumerate(requests)]
        beside = sampler.sample_device(logits, requests + [greedy], ahead, host).tolist()
        assert host.tolist() == beside
        assert beside == together + [int(logits[R].argmax())]
        later = [Request(r.id, r.prompt, r.params, output=r.output + [4] * ahead) for r in requests]
        assert sampler.sample_device(logits[:R], later).tolist() == together
    assert len({tuple(sampler.sample_device(logits[:R], requests, a).tolist()) for a in range(4)}) == 4


@pytest.mark.parametrize("rows,V", [(1, 16384), (70, 20001), (64, 32000), (3, 128256)])
def test_sample_rows(ops, rows, V):
    """Tokens from parameters in the launch and numbers made of texts: those of ``sample_top_p`` with the same numbers, and, where
    a row's candidates alone decide (peaked rows), where they are too many (flat ones, equal logits) and where all tokens
    are kept, a token of the nucleus that the other kernels find, at the same place of its cumulative distribution."""
    from pytriton_llama_amd.sampling.sampler import uniform_for, uniform_text
    g = torch.Generator().manual_seed(V)
    logits = torch.randn(rows, V + 3, generator=g)
    kinds = [4.0, 0.02, 2.0, 0.7, 30.0, 1.0]
    for r in range(rows):
        logits[r] *= kinds[r % 6]
        if r % 6 == 5:
            logits[r] = logits[r].round()                     # many equal logits
    logits = logits.cuda()[:, :V]                             # rows of any alignment
    params = [(0.6 + 0.1 * (r % 5), (0.9, 0.95, 0.5, 1.0, 0.999999)[r % 5], 0.0) for r in range(rows)]
    texts = [uniform_text(9, ("chat é", r), 7) for r in range(rows)]
    got = ops.sample_rows(logits, [v for p in params for v in p], texts)
    t, p = (torch.tensor([q[i] for q in params]).cuda() for i in (0, 1))
    u = torch.tensor([uniform_for(9, ("chat é", r), 7) for r in range(rows)]).cuda()
    assert torch.equal(got, ops.sample_top_p(logits, t, p, u))
    tok, probs = ops.sample_top_p(logits, t, p, u, return_probs=True)
    for r in range(rows):
        cdf = torch.cumsum(probs[r].double(), 0)
        assert probs[r, int(got[r])] > 0
        assert int(got[r]) == int(tok[r]) or abs(float(cdf[int(got[r])] - cdf[int(tok[r])])) < 1e-4, r
    with pytest.raises(ops.KernelError):
        ops.sample_rows(logits, [0.6, 0.9, 0.0] * rows, texts[1:])


@pytest.mark.parametrize("temperature,share", [(1e-4, 3e-3), (1e-3, 3e-4), (1e-5, 3e-2)])
def test_sample_edge_at_low_temperature(ops, temperature, share):
    """Two tokens with 0.7 and 0.3 of the mass and top_p a ``share`` of 0.7 above and below it: the second one belongs to the nucleus
    above only, whatever the largest logit is (largest logit over temperature times log2(e): off by up to 2^-25 of itself where it is
    rounded, 1 % of the mass at 25 and 1e-4)."""
    R, V = 64, 16384
    gap = temperature * math.log(0.7 / 0.3)
    logits = torch.randn(R, V, generator=torch.Generator().manual_seed(50)) - 50.0        # (few candidates in every chunk)
    logits[:, 100] = torch.linspace(20.0, 31.0, R)
    logits[:, 9000] = logits[:, 100] - gap                    # (in another chunk)
    d = (logits[:, 100].double() - logits[:, 9000].double()) / temperature
    first = 1.0 / (1.0 + torch.exp(-d))                       # of the logits as float32 has them
    t = torch.full((R,), temperature).cuda()
    u = torch.full((R,), 0.9999).cuda()
    for sign, token in ((-1, 100), (1, 9000)):
        p = (first * (1 + sign * share)).float().cuda()
        assert ops.sample_top_p(logits.cuda(), t, p, u).tolist() == [token] * R, sign


@pytest.mark.parametrize("wide", [False, True], ids=["one_workgroup", "many_workgroups"])
def test_sample_top_p_nearly_flat_row_and_signed_zeros(ops, wide):
    """A nearly flat row with a top_p that admits two tokens keeps exactly those two (the most
    likely token is always kept, its neighbours only by the rule); +0 and -0 are one logit."""
    V = 20000
    g = torch.Generator().manual_seed(4)
    flat = torch.randn(V, generator=g) * 1e-3
    top = torch.topk(flat, 3).indices.tolist()
    zeros = torch.zeros(V)
    zeros[::2] = -0.0
    zeros[[11, 500]] = torch.tensor([1.0, 0.5])
    logits = torch.stack([flat, zeros]).cuda()
    t = torch.ones(2).cuda()
    # row 0: every token has about 1/V of the mass; the mass before the third token is ~2/V
    # row 1: tokens 11 and 500 hold e + sqrt(e) of e + sqrt(e) + V - 2; 0.01 lets in the zeros' first
    p = torch.tensor([1.5 / V, 0.01]).cuda()
    u = torch.tensor([0.99, 0.5]).cuda()
    tok, probs = ops.sample_top_p(logits, t, p, u, return_probs=True, wide=wide)
    kept0 = torch.nonzero(probs[0]).flatten().tolist()
    assert sorted(kept0) == sorted(top[:2]) and int(tok[0]) in kept0
    want = plain_llama.top_p_probs(zeros, 1.0, 0.01)
    got = probs[1].double().cpu()
    # all zeros, whatever their sign, are kept together (the plain sort would split them)
    rest = got[torch.arange(V)[(torch.arange(V) != 11) & (torch.arange(V) != 500)]]
    assert float(rest.min()) == float(rest.max()) and got[11] > got[500] > rest[0] >= 0
    assert bool((got > 0).all()) == bool(rest[0] > 0) and want[11] > 0


def test_kernels_refuse_cpu_tensors(ops):
    with pytest.raises(ops.KernelError):
        ops.silu_mul(torch.zeros(2, 4))
    with pytest.raises(ops.KernelError):
        ops.add_rmsnorm(torch.zeros(2, 64), None, torch.ones(64), 1e-5)
    with pytest.raises(ops.KernelError):        # a weight of the wrong length
        ops.add_rmsnorm(torch.zeros(2, 64, device="cuda"), None, torch.ones(63, device="cuda"), 1e-5)


def test_sample_top_p_large_vocabulary_and_ties(ops):
    """At vocabulary size, with a peaked and a flat row, and a row of many equal
    logits (more tokens in one histogram bin than the kernel gathers)."""
    torch.manual_seed(11)
    V = 128256
    logits = torch.randn(4, V)
    logits[0] *= 4.0                                   # peaked
    logits[1] *= 0.05                                  # nearly flat
    logits[2] = 0.0                                    # all equal but a few
    logits[2, [5, 77, 99999]] = torch.tensor([3.0, 2.0, 1.0])
    logits[3, 1234] = 40.0                             # one token holds all the mass
    t = torch.tensor([0.8, 1.0, 1.0, 0.6])
    p = torch.tensor([0.9, 0.5, 0.5, 0.9])
    u = torch.tensor([0.3, 0.9, 0.999999, 0.5])
    tok, probs = ops.sample_top_p(logits.cuda(), t.cuda(), p.cuda(), u.cuda(), return_probs=True)
    for r in (0, 1, 3):
        want = plain_llama.top_p_probs(logits[r], float(t[r]), float(p[r]))
        got = probs[r].cpu().double()
        # the nucleus may differ by a token or two at its edge where the float32 running
        # mass meets top_p; the mass that changes hands is tiny
        assert float((got - want).abs().sum()) < 1e-3
        assert want[int(tok[r])] > 0
    assert int(tok[3]) == 1234
    # equal logits are kept or dropped together: the three larger ones first, then all or none
    got2 = probs[2].cpu()
    assert got2[5] > got2[77] > got2[99999] > 0
    rest = got2[torch.arange(V)[(torch.arange(V) != 5) & (torch.arange(V) != 77) & (torch.arange(V) != 99999)]]
    assert float(rest.min()) == float(rest.max())
    assert abs(float(got2.sum()) - 1) < 1e-4
