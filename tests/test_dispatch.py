"""Which kernels a call launches (csrc/abi.hip, csrc/echain.hip), on the CPU: the library's
host side over a HIP runtime that records launches."""
from __future__ import annotations

import pytest

import dispatch as D


def _grid(result):
    st, events, msg = result
    assert st == 0, msg
    (launch,) = [e for e in events if e[0] == "launch"]
    return launch


# The K splits of engine calls of nine rows and more are part of their results' definition
# (the order of fp32 sums): these must not move when kernels or time models change.
K_SPLITS = [
    ("i8", 2048, 2048, 1), ("i8", 2048, 6144, 1), ("i8", 6144, 2048, 4), ("i8", 4096, 4096, 2),
    ("i8", 4096, 12288, 2), ("i8", 12288, 4096, 2), ("i8", 2048, 512, 1), ("i8", 8192, 1024, 8),
    ("w4", 2048, 2048, 4), ("w4", 4096, 4096, 2), ("w4", 12288, 4096, 2), ("w4", 2048, 512, 1),
    ("gu8", 2048, 6144, 1), ("gu8", 4096, 12288, 2), ("gu8", 2048, 2048, 4), ("gu8", 1024, 3072, 2),
    ("gu4", 2048, 6144, 1), ("gu4", 4096, 12288, 2), ("gu4", 512, 256, 1),
]


def test_k_splits(tmp_path):
    make = {"i8": D.gemm_i8, "w4": D.gemm_w4, "gu8": D.gate_up_i8, "gu4": D.gate_up_w4}
    # nine rows run on the 16-row tiles: 64 columns without a split, 128 columns x S with
    got = [_grid(r)[2] for r in D.run(tmp_path, [make[k](9, K, N) for k, K, N, _ in K_SPLITS])]
    assert got == [N // 64 if s == 1 else -(-N // 128) * s for _, _, N, s in K_SPLITS]


def test_calls_without_a_split_need_no_workspace(tmp_path):
    for st, events, msg in D.run(tmp_path, [f(M, K, N, ws=0) for M in (9, 64, 512) for f, K, N in
                                            ((D.gemm_i8, 2048, 512), (D.gemm_i8, 2048, 2048), (D.gate_up_w4, 512, 256),
                                             (D.gate_up_w4, 2048, 6144))]):
        assert st == 0 and events, msg


@pytest.mark.parametrize("call,kernel", [
    # gemm_i8 4096x12288 at 96 rows: 28.3 us on 128x128, 36 on the 64-column tiles
    (D.gemm_i8(96, 4096, 12288), "prefill_i8_kernelILi0ELb0ELi0ELi4ELi2E"),
    (D.gemm_i8(512, 12288, 4096), "prefill_i8_kernelILi0ELb0ELi0ELi4ELi2E"),
    # W4 2048x6144 at 129 rows: 19.6 us on the 16-row tiles, 20.5 on 96x64, two rows of tiles
    (D.gemm_w4(129, 2048, 6144), "skinny_kernel"),
    (D.gate_up_i8(64, 2048, 2048), "prefill_i8_kernelILi0ELb0ELi2ELi2ELi1E"),
])
def test_engine_tiles(tmp_path, call, kernel):
    assert kernel in _grid(D.run(tmp_path, [call])[0])[1]


@pytest.mark.parametrize("call", [D.gemm_i8(1, 2048, 2048), D.gemm_w4(4, 2048, 2048), D.gate_up_w4(1, 2048, 2048),
                                  D.proj3_i8(1, 2048, 1024, 512, 512)])
def test_residency_is_asked_of_the_kernel_that_polls(tmp_path, call):
    """A call's split tiles poll their partners, which is safe if every workgroup of the
    launched kernel is resident at once: the occupancy asked for is that kernel's."""
    st, events, msg = D.run(tmp_path, [call])[0]
    assert st == 0, msg
    assert [e[0] for e in events] == ["occupancy", "launch"]
    assert events[0][1] == events[1][1]


@pytest.mark.parametrize("call,kernel", [
    # above the rows that the short-prompt kernel's model is fitted on (512) it was chosen
    # where it is slower: 16.7 us against 15.0, 16.5 / 15.2, 24.9 / 21.1
    (D.linear_w8(1323, 1280, 1248), "prefill_kernel"), (D.linear_w8(1500, 1280, 1248), "prefill_kernel"),
    (D.linear_w4(4000, 2048, 512), "prefill_kernel"),
    # and where it stays the faster one: 8.6 us against 9.5, 16.6 / 18.8
    (D.linear_w8(513, 512, 2048), "prefill_kg_kernel"), (D.linear_w8(1500, 4096, 320), "prefill_kg_kernel"),
    (D.linear_w8(128, 2048, 2048), "prefill_kg_kernel"), (D.linear_w4(128, 6144, 2048), "prefill_kg_kernel"),
])
def test_short_prompt_kernel_choice(tmp_path, call, kernel):
    assert kernel in _grid(D.run(tmp_path, [call])[0])[1]


@pytest.mark.parametrize("K,N,launches", [(8192, 64, 1), (12288, 64, 4), (10240, 1024, 1), (16384, 1024, 4),
                                          (12288, 4096, 1), (16384, 4096, 4), (6144, 8192, 1), (8192, 8192, 4)])
def test_requant_long_columns(tmp_path, K, N, launches):
    """Strips of columns for short columns, four launches over the rows for long ones (K = 16384,
    N = 1024 89 us in strips, 66 in four launches; K = 6144, N = 8192 95 / 106)."""
    st, events, msg = D.run(tmp_path, [D.requant_w8(K, N)])[0]
    assert st == 0 and len(events) == launches, msg


@pytest.mark.parametrize("shape,refused", [(1, False), (2, False), (3, True)])
def test_balanced_schedule_of_the_wide_tile_is_refused(tmp_path, shape, refused):
    """QLIN_PREFILL_SK with the 128x384 tile, which has no balanced schedule, is refused with
    a message before anything is launched (300 rows, 32 K tiles, 37 per workgroup)."""
    st, events, msg = D.run(tmp_path, [D.linear_w8(300, 2048, 1280)],
                            {"QLIN_PREFILL": "tiled", "QLIN_PREFILL_SHAPE": str(shape), "QLIN_PREFILL_SK": "37"})[0]
    assert (st, not events) == ((-2, True) if refused else (0, False)), msg
    assert ("QLIN_PREFILL_SK" in msg) == refused


def test_forced_tiles_are_different_kernels(tmp_path):
    """QLIN_I8_TILE, which the tests of equal bits across tiles set, picks five kernels."""
    calls = [D.gemm_i8(300, 1984, 1280), D.proj3_i8(300, 1984, 1024, 256, 256)]
    seen = [set(), set()]
    for tile in range(5):
        for i, r in enumerate(D.run(tmp_path, calls, {"QLIN_ENGINE_PREFILL": "tiled", "QLIN_I8_TILE": str(tile)})):
            seen[i].add(_grid(r)[1])
    assert [len(s) for s in seen] == [5, 5]
