"""The launchers of the kernel libraries, called without a GPU (host_launches.py)."""
import pytest

from host_launches import run

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
