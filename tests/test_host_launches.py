"""The launchers of the kernel libraries, called without a GPU (host_launches.py)."""
import pytest

from host_launches import TILES, run

P = ("p", 1 << 20)                     # an aligned address that nothing reads
NO = ("p", 0)


def i(*values):
    return [("i", v) for v in values]


GATE_UP = ("ptl_tile_gate_up", [P, P, P, *i(285, 8192, 2048), ("l", 2048), ("i", 0), ("f", 0.0), ("i", 0), NO])
ROWS = ("ptl_rows_gate_up_silu", [P, P, P, *i(64, 8192, 2048), ("l", 2048), ("i", 0), ("f", 0.0), NO])
EXTRAS = [*i(0, 0, 0), NO, NO, ("l", 0), ("f", 0.0), ("f", 0.1)]


def generic(head_dim, dtype):
    return ("ptl_attention_generic", [P, ("l", 4 * head_dim), P, ("l", 4 * head_dim), P, P, P, P, P, *i(4), P, P,
                                      *i(8, 4, 2, head_dim, 16), *EXTRAS, ("i", dtype), NO])


SCAN = ("ptl_linear_scan", [*i(0), P, P, ("l", 512), P, ("l", 512), P, ("l", 512), ("f", 1.0), P, ("l", 8), P, P, P, NO,
                            ("l", 0), NO, NO, ("l", 0), ("i", 0), ("l", 0), ("i", 0), P, ("l", 1 << 20), P, *i(2, 128), P,
                            P, *i(1, 4, 1, 256, 64), NO])


@pytest.mark.parametrize("library,entry,args", [("gemm_tile", *GATE_UP), ("gemm_rows", *ROWS),
                                                ("attention", *generic(576, 1)), ("attention", *generic(112, 0)),
                                                ("linear_scan", *SCAN)])
def test_lds_beyond_64_kb_is_asked_for_on_every_device(tmp_path, library, entry, args):
    """Kernels with more dynamic LDS than one gets unasked, launched on three devices of one process in turn."""
    devices = (0, 0, 1, 2, 0)
    took = run(tmp_path, library, [(d, entry, args) for d in devices])
    assert [t["code"] for t in took] == [0] * len(devices)
    for d, t in zip(devices, took):
        assert t["launches"] and all(k["device"] == d for k in t["launches"])
        assert max(k["lds"] for k in t["launches"]) > 64 * 1024


def test_a_larger_size_is_asked_for_after_a_smaller_one(tmp_path):
    """One kernel whose LDS follows the head size: 300, 640, then 300 again, on two devices."""
    took = run(tmp_path, "attention", [(d, *generic(h, 1)) for d in (0, 1) for h in (300, 640, 300, 576)])
    assert [t["code"] for t in took] == [0] * 8
    assert len({t["launches"][0]["kernel"] for t in took}) == 1


def tile_of(launch):
    """(rows of x, rows of W) of a launched tile product, from the kernel's template arguments."""
    inner = launch["kernel"].split("gemm_tile_kernelI")[1]
    return tuple(int(v) for v in inner.split("Li")[1:3] for v in [v.rstrip("E")])


def product(M, N, K, sums, tile, splits):
    return ("ptl_tile_product", [P, P, P, *i(M, N, K), ("l", K), *i(sums, tile, splits, 0), ("f", 0.0), NO])


@pytest.mark.parametrize("sums", [1, 0])
def test_every_tile_of_the_tile_products(tmp_path, sums):
    """An index launches its own tile, with no more workgroups than tiles or than the chip holds; refused: an index that
    is none, slices that are no whole chunks, slices of a gate-up product."""
    bad = [product(100, 512, 512, sums, len(TILES), 1), product(100, 512, 512, sums, -1, 1),
           product(100, 512, 512, sums, 0, 0), product(100, 512, 512, sums, 0, 3 if sums else 2)]
    good = [product(M, N, 512, sums, t, 4 if sums else 1) for t in range(len(TILES)) for M, N in ((65, 132), (1000, 16384))]
    took = run(tmp_path, "gemm_tile", [(0, *c) for c in [("ptl_tile_shapes", [])] + bad + good])
    assert took[0]["code"] == len(TILES)
    assert all(t == {"code": -1, "launches": []} for t in took[1:5])
    for n, t in enumerate(took[5:]):
        rows, cols, places = TILES[n // 2]
        M, N = ((65, 132), (1000, 16384))[n % 2]
        tiles = -(-M // rows) * -(-N // (cols if sums else cols // 2)) * (4 if sums else 1)
        assert t["code"] == 0 and len(t["launches"]) == 1 and tile_of(t["launches"][0]) == (rows, cols)
        assert t["launches"][0]["grid"] == [min(tiles, 256 * places), 1, 1]


def test_products_of_every_number_of_rows_launch_a_tile(tmp_path):
    """Gate-up over the rows it takes at the 1B, 3B and 8B widths: which tiles come up, so that a refit of the plan's times
    that no longer uses one, or uses it elsewhere, shows here."""
    calls = [("ptl_tile_gate_up", [P, P, P, *i(M, I, K), ("l", K), ("i", 0), ("f", 0.0), ("i", 1), NO])
             for I, K, most in ((8192, 2048, 576), (8192, 3072, 576), (14336, 4096, 160)) for M in range(65, most + 1, 7)]
    took = run(tmp_path, "gemm_tile", [(0, *c) for c in calls])
    assert all(t["code"] == 0 and len(t["launches"]) == 1 for t in took)
    used = {tile_of(t["launches"][0]) for t in took}
    assert used <= {t[:2] for t in TILES} and len(used) >= 6, used


@pytest.mark.parametrize("M,N,K,parts", [(300, 200, 96, False), (17, 64, 32, False), (300, 512, 512, False), (128, 1024, 1024, False),
                                         (130, 16384, 128, False), (300, 200, 100, False), (130, 4096, 512, True),
                                         (64, 7000, 1024, True), (700, 16384, 128, True), (17, 2048, 2048, True), (300, 200, 1056, True)])
def test_small_f32_products_have_no_kernel_that_splits_x(tmp_path, M, N, K, parts):
    """Small products of more than 16 rows of float32 are one kernel, and the sum of the spans' where K is cut; others have the
    parts of x made first. Both want the workspace they say."""
    took = run(tmp_path, "gemm_f32", [(0, "ptl_gemm_f32_workspace", i(M, N, K)),
                                      (0, "ptl_gemm_f32", [P, P, P, *i(M, N, K), ("l", K), ("l", N), P, NO]),
                                      (0, "ptl_gemm_f32", [P, P, P, *i(M, N, K), ("l", K), ("l", N), NO, NO])])
    kernels = [k["kernel"] for k in took[1]["launches"]]
    assert took[1]["code"] == 0
    assert any("split_rows_kernel" in k for k in kernels) == parts
    assert any("gemm_f32_stream_kernel" in k for k in kernels) == parts and any("gemm_f32_tile_kernel" in k for k in kernels) != parts
    wants = took[0]["code"] != 0
    assert wants == (parts or any("gemm_f32_sum_kernel" in k for k in kernels))
    assert took[2] == ({"code": -1, "launches": []} if wants else took[1])


@pytest.mark.parametrize("splits,acc,ml,tickets,matrix_cores", [(4, 0, 0, 1, True), (4, 8, 8, 1, True), (4, 4, 0, 1, False),
                                                                (4, 0, 4, 1, False), (4, 0, 0, 0, False), (1, 4, 4, 0, True)])
def test_float32_decode_attention_by_its_workspaces(tmp_path, splits, acc, ml, tickets, matrix_cores):
    """The last workgroup of a sequence reads the parts eight bytes at a time: workspaces that do not lie so, like a call
    without tickets, go to the general kernel and its merge."""
    at = lambda off: ("p", (1 << 20) + off)
    took = run(tmp_path, "attention", [(0, "ptl_attention_decode", [
        P, ("l", 512), P, ("l", 512), P, P, P, P, P, *i(64), at(acc), at(ml), P if tickets else NO, *i(3, 8, 2, 64, 16), *EXTRAS,
        *i(splits, 0), NO])])[0]
    names = [k["kernel"] for k in took["launches"]]
    assert took["code"] == 0 and any("attn_f32_kernel" in n for n in names) == matrix_cores
    assert [any(part in n for n in names) for part in ("attn_decode_kernel", "attn_decode_merge_kernel")] == [not matrix_cores] * 2


@pytest.mark.parametrize("rows,kv_heads,head_dim,splits", [(1, 8, 64, 32), (8, 8, 128, 8), (16, 8, 64, 4), (32, 8, 64, 3), (32, 8, 128, 2),
                                                           (48, 8, 128, 2), (64, 8, 64, 1), (64, 8, 128, 1), (65, 8, 64, 1),
                                                           (256, 8, 64, 1), (200, 32, 128, 1)])
def test_decode_attention_is_not_launched_for_the_longest_table(tmp_path, rows, kv_heads, head_dim, splits):
    """However long the contexts that a block table can hold: no more workgroups than four a compute unit, or than the splits
    ask for; a table of short contexts has no parts beyond them; a piece of the caller's own is taken as it is."""
    pairs = rows * kv_heads
    keys = [128, 8192, 32768, 131072, 1 << 20]
    parts = [t["code"] for t in run(tmp_path, "attention", [
        (0, "ptl_attention_decode_mfma_parts", [*i(head_dim, splits), ("l", k), ("l", pairs), ("i", piece)])
        for piece in (0, 128) for k in keys])]
    assert parts[0] == splits and parts == sorted(parts[:5]) + parts[5:]
    # a batch that fills the chip is not cut up to 8,192 keys, nor one whose requests have many parts
    assert splits > 1 or parts[1] == 1
    assert splits < 5 or parts[:5] == [splits] * 5
    assert all(m == splits or m * pairs <= 4 * 256 for m in parts[:5]) and parts[4] <= max(splits, 16)
    assert parts[5:] == [max(splits, m) for m in (1, 16, 16, 16, 16)]
    took = run(tmp_path, "attention", [(0, "ptl_attention_decode_mfma", [
        P, ("l", 4096), P, ("l", 4096), P, P, P, P, P, *i(8192), P, P, *i(most, rows, 2 * kv_heads, kv_heads, head_dim, 16), *EXTRAS,
        *i(splits, 0, 0), NO]) for most in parts[:5]])
    for most, t in zip(parts, took):
        assert t["code"] == 0 and len(t["launches"]) == 1
        # (a list of parts is in whole turns of eight and of the units)
        assert rows * kv_heads * most <= t["launches"][0]["grid"][0] < pairs * most + 8 * kv_heads + 256


@pytest.mark.parametrize("heads,head_dim,blocks,longest,two", [
    (64, 64, 8, 0, True),              # 512 workgroups on 256 units
    (65, 64, 8, 0, False),
    (65, 64, 4, 0, False),             # four blocks: as likely short portions
    (64, 64, 4, 0, True),              # ... which find a unit each
    (64, 64, 4, 256, False),           # ... and are known to be short
    (33, 32, 8, 512, True),
    (33, 32, 8, 511, False),
    (40, 128, 8, 450, True),           # a prompt by itself
    (40, 96, 9, 450, True),            # ... with one more (empty, in a recorded step) block
    (40, 128, 8, 321, False),          # with two more
    (65, 128, 8, 450, False)])
def test_prompt_attention_with_one_group_of_waves_or_two(tmp_path, heads, head_dim, blocks, longest, two):
    """Both sides of the lines, for the entry of one head size and for the general one."""
    step = [P, P, P, P, P, *i(40), P, P]
    masks = [*EXTRAS, NO]
    took = run(tmp_path, "attention_prefill", [
        (0, "ptl_attention_prefill_mfma", [P, ("l", heads * head_dim), P, ("l", heads * head_dim), *step,
                                           *i(blocks, blocks, 64, longest, heads, 1, head_dim, 16), *masks]),
        (0, "ptl_attention_prefill_mfma_kv", [P, ("l", heads * head_dim), *i(0), P, ("l", heads * head_dim), *step,
                                              *i(blocks, blocks, longest, heads, 1, 1, head_dim, head_dim, 16), *masks])])
    for t in took:
        assert t["code"] == 0 and len(t["launches"]) == 1 and t["launches"][0]["threads"] == (512 if two else 256)
        assert t["launches"][0]["grid"][0] * t["launches"][0]["grid"][1] == heads * blocks
