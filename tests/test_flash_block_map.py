"""The MFMA flash kernel's workgroup -> work map, dumped on the host by the function the kernel itself uses
(ahpc_hip_flash_block_map): whatever the shape and the pairing of query tiles under a causal mask, every
(sequence*head, query tile) must be handled by exactly one workgroup pass, and nothing else may be handled.  A map that misses or repeats a tile computes wrong
attention; one that names a head that does not exist reads outside the tensors."""
import numpy as np
import pytest

ROWS = 128  # query rows per workgroup pass (256 while the tuning value flash_rows says so)


def check_exact_cover(B, N, H, causal, ROWS=ROWS):
    from attention_amd import hip
    bh, t0, t1 = hip.flash_block_map(B, N, H, causal)
    n_tiles = (N + ROWS - 1) // ROWS
    assert len(bh) % 8 == 0
    valid = bh >= 0
    assert ((t0 >= 0) == valid).all() and (t1[~valid] == -1).all()
    assert bh[valid].max() < B * H and t0[valid].max() < n_tiles and t1.max() < n_tiles
    pairs = np.concatenate([bh[valid].astype(np.int64) * n_tiles + t0[valid], (bh.astype(np.int64) * n_tiles + t1)[t1 >= 0]])
    assert len(pairs) == B * H * n_tiles
    assert np.array_equal(np.sort(pairs), np.arange(B * H * n_tiles))
    return bh, t0, t1


SHAPES = [(1, 1, 1), (1, 128, 1), (2, 129, 3), (1, 1000, 3), (2, 2144, 16), (4, 4096, 32), (1, 777, 5), (3, 640, 7),
          (64, 300, 8), (1, 8192, 9), (5, 1152, 13)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,N,H", SHAPES)
def test_default_map_covers_every_tile_once_and_keeps_its_order(B, N, H, causal):
    bh, t0, t1 = check_exact_cover(B, N, H, causal)
    # the default order: consecutive logical ids (= 8 workgroup ids apart) walk one head's tiles, late tiles first
    n_tiles = (N + ROWS - 1) // ROWS
    paired = causal and n_tiles >= 2 and B * H * n_tiles >= 1024
    per_head = (n_tiles + 1) // 2 if paired else n_tiles
    per_xcd = len(bh) // 8
    for block in range(len(bh)):
        logical = (block & 7) * per_xcd + (block >> 3)
        if logical >= B * H * per_head:
            assert bh[block] == -1
            continue
        slot = logical % per_head
        assert bh[block] == logical // per_head and t0[block] == n_tiles - 1 - slot
        want_second = slot if paired and 2 * slot != n_tiles - 1 else -1
        assert t1[block] == want_second


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,N,H", SHAPES)
def test_map_of_256_row_workgroups_covers_every_tile_once(B, N, H, causal):
    from attention_amd import hip
    before = hip.get_tuning("flash_rows")
    hip.set_tuning("flash_rows", 256)
    try:
        check_exact_cover(B, N, H, causal, ROWS=256)
    finally:
        hip.set_tuning("flash_rows", before)


@pytest.mark.parametrize("rows", [128, 256])
@pytest.mark.parametrize("line", [1, 1 << 40])
@pytest.mark.parametrize("B,N,H", SHAPES + [(2, 2048, 12), (4, 1024, 16), (9, 1152, 8), (3, 1000, 32)])
def test_map_covers_every_tile_once_paired_and_single(B, N, H, line, rows):
    """Every map a causal launch can take: which of them it takes is a matter of d, type and shape."""
    from attention_amd import hip
    before = {n: hip.get_tuning(n) for n in ("flash_rows", "flash_pair_min_tiles")}
    hip.set_tuning("flash_rows", rows)
    hip.set_tuning("flash_pair_min_tiles", line)
    try:
        _, _, second = check_exact_cover(B, N, H, True, ROWS=rows)
        assert (second >= 0).any() == (line == 1 and N > rows)
    finally:
        for n, v in before.items():
            hip.set_tuning(n, v)


def test_rejects_bad_shapes_without_a_gpu():
    from attention_amd import hip
    import ctypes as C
    n = C.c_int64(0)
    assert hip.load().ahpc_hip_flash_block_map(0, 16, 4, 0, 0, C.byref(n), None, None, None) == -2
    assert hip.load().ahpc_hip_flash_block_map(1, 16, 4, 0, 0, None, None, None, None) == -1
    buf = np.empty(4, np.int32)
    assert hip.load().ahpc_hip_flash_block_map(4, 4096, 32, 1, 4, C.byref(n), buf.ctypes.data, buf.ctypes.data, buf.ctypes.data) == -2


@pytest.fixture
def pair_line():
    from simt import simt as S
    lib = S.load()
    hip = S.EmulatedHip()
    before = hip.get_tuning("flash_pair_min_tiles")
    yield lambda n, *shape: (hip.set_tuning("flash_pair_min_tiles", n), lib.simt_flash_paired(*shape))[1]
    hip.set_tuning("flash_pair_min_tiles", before)


def test_every_pairing_line_that_is_named_holds(pair_line):
    """512 tiles, which the shape would pair, and 1152: the default's old value, 1024, is a line like any other."""
    assert pair_line(0, 128, 0, 0, 4, 2048, 8) == 1 and pair_line(0, 128, 0, 1, 4, 2048, 8) == 0
    for line in (1023, 1024, 1025):
        for f32, ragged in ((0, 0), (1, 0), (0, 1), (1, 1)):
            assert pair_line(line, 128, f32, ragged, 4, 2048, 8) == 0
            assert pair_line(line, 128, f32, ragged, 9, 2048, 8) == 1
    assert pair_line(1, 128, 0, 1, 1, 129, 1) == 1


# d, fp32?, B, N, H -> are tiles paired?       single    paired, us
PAIRED = [(128, 1, 1, 2958, 16, 1),          # 594       410
          (128, 1, 2, 1106, 32, 0),          # 224       308
          (64, 1, 2, 1337, 16, 1),           # 165       113
          (64, 1, 6, 376, 24, 0),            # 47        69
          (256, 0, 8, 1930, 4, 1),           # 155       105
          (256, 0, 19, 814, 4, 0),           # 83        112
          (128, 0, 2, 3894, 6, 1),           # 86        72
          (128, 0, 2, 552, 40, 0),           # 19        23
          (128, 0, 3, 3101, 8, 0),           # 77        89
          (64, 0, 2, 3779, 8, 1),            # 53        49
          (64, 0, 3, 794, 32, 0),            # 20        23
          (64, 0, 13, 469, 16, 1)]           # 22        19


@pytest.mark.parametrize("d,f32,B,N,H,paired", PAIRED)
def test_the_faster_of_single_and_paired_tiles_is_taken(pair_line, d, f32, B, N, H, paired):
    """Causal launches of the 128-row kernels that were timed both ways."""
    assert pair_line(0, d, f32, 0, B, N, H) == paired
