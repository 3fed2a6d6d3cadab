"""Which automatic decode calls take the grid schedule, and with what scratch (host arithmetic, no GPU)."""
import pytest

from aicomp_amd import _lib

DEFAULT = 32768
BF16, F16, F32, FP8 = _lib.BF16, _lib.F16, _lib.F32, _lib.FP8_E4M3


@pytest.fixture
def lib():
    try:
        lib = _lib.load()
    except _lib.LibraryMissing:
        pytest.skip("library not built")
    prev = lib.aicomp_kv_set_small_decode_tokens(DEFAULT)
    yield lib
    lib.aicomp_kv_set_small_decode_tokens(prev)


def route(lib, rows, hq, hkv, d, tokens, q, kv):
    """(tokens per partition, whether the balanced schedule runs) of an automatic call over a table of `tokens` tokens."""
    args = rows, hq, hkv, d, 16, tokens // 16, q, kv
    ps = lib.aicomp_paged_decode_partition_size(*args)
    need, parts = lib.aicomp_paged_decode_workspace_bytes(*args, 0), -(-tokens // ps)
    split = 0 if parts == 1 else rows * hq * parts * (d + 2) * 4
    return ps, need != split


@pytest.mark.parametrize("rows,hq,hkv,d,q,kv,longest,beyond", [
    # whole rows: the line of few workgroups, then of 128, 256 and 512 pairs of a row and a KV head
    (8, 32, 8, 128, BF16, BF16, 768, 256), (64, 16, 2, 128, BF16, BF16, 896, 256), (32, 32, 8, 128, F16, F16, 1152, 256),
    (64, 32, 8, 128, BF16, BF16, 1664, None), (64, 8, 8, 128, BF16, BF16, 1216, None), (128, 64, 8, 128, BF16, BF16, 1664, None),
    (32, 32, 8, 64, BF16, BF16, 2048, None), (64, 32, 8, 64, BF16, BF16, 3072, None), (128, 32, 8, 64, BF16, BF16, 2048, None),
    (32, 32, 8, 128, BF16, FP8, 1600, None), (64, 32, 8, 128, BF16, FP8, 2880, None), (128, 32, 8, 128, BF16, FP8, 2048, None),
    (96, 16, 2, 64, F16, FP8, 1920, 256), (64, 32, 8, 64, BF16, FP8, 4096, None),
    (48, 32, 8, 128, BF16, BF16, 1280, 256), (48, 32, 8, 64, F16, F16, 2304, None), (48, 64, 8, 128, BF16, FP8, 1920, None),     # 1.5 to a CU
    (32, 32, 8, 64, F32, F32, 928, 256), (64, 32, 8, 64, F32, F32, 1088, None), (64, 32, 8, 128, F32, F32, 640, None),
    (1, 64, 8, 128, F32, F32, 448, 256)])
def test_whole_rows(lib, rows, hq, hkv, d, q, kv, longest, beyond):
    assert route(lib, rows, hq, hkv, d, longest, q, kv) == (-(-longest // 64) * 64, False)
    ps, balanced = route(lib, rows, hq, hkv, d, longest + 16, q, kv)
    assert balanced == (beyond is None) and (balanced or ps == beyond)
    lib.aicomp_kv_set_small_decode_tokens(0)
    assert route(lib, rows, hq, hkv, d, longest, q, kv)[1]
    if rows * longest > DEFAULT - 1:
        lib.aicomp_kv_set_small_decode_tokens(DEFAULT - 1)            # a lower threshold pins the schedule
        assert route(lib, rows, hq, hkv, d, longest, q, kv)[1]


@pytest.mark.parametrize("rows,hkv,d,kv,last", [(16, 8, 128, BF16, 4096), (24, 8, 128, BF16, 2720), (32, 8, 128, BF16, 2048),
                                                (64, 2, 64, BF16, 4096), (24, 8, 128, FP8, 2048), (16, 8, 64, FP8, 3072),
                                                (16, 8, 64, F32, 4096), (4, 8, 128, F32, 8192)])
def test_few_long_rows_are_split(lib, rows, hkv, d, kv, last):
    q = F32 if kv == F32 else BF16
    assert route(lib, rows, 4 * hkv, hkv, d, last, q, kv) == (256, False)
    assert route(lib, rows, 4 * hkv, hkv, d, last + 16, q, kv)[1]


def test_no_call_needs_more_scratch_than_on_the_balanced_schedule(lib):
    """What a caller's scratch, or the library's own 32 MiB, was enough for stays enough."""
    for hq, hkv in ((32, 8), (64, 8), (16, 2), (8, 8), (16, 1), (128, 128), (40, 20)):
        for d in (64, 128):
            for q, kv in ((BF16, BF16), (F16, FP8), (F32, F32)):
                for rows in (1, 2, 5, 17, 33, 65, 129, 300, 1024):
                    for tokens in (256, 640, 656, 784, 1296, 1680, 2064, 2912, 3088, 4096, 4112, 20000):
                        args = rows, hq, hkv, d, 16, tokens // 16, q, kv, 0
                        if rows * tokens <= DEFAULT:
                            continue
                        lib.aicomp_kv_set_small_decode_tokens(0)
                        most = lib.aicomp_paged_decode_workspace_bytes(*args)
                        lib.aicomp_kv_set_small_decode_tokens(DEFAULT)
                        assert lib.aicomp_paged_decode_workspace_bytes(*args) <= most, args


@pytest.mark.parametrize("threshold", [DEFAULT + 1, 131072, 262144, 1 << 20, 1 << 24])
def test_nor_under_a_raised_threshold(lib, threshold):
    """Calls above the threshold in force; the first two outgrew the library's own 32 MiB where the line of the split rose with it."""
    shapes = [(64, 64, 8, 128, BF16, BF16, 4096), (128, 32, 8, 128, BF16, BF16, 4096)]
    shapes += [(rows, hq, hkv, d, q, kv, tokens) for hq, hkv in ((32, 8), (64, 8), (16, 1), (8, 8)) for d in (64, 128)
               for q, kv in ((BF16, BF16), (F16, FP8), (F32, F32)) for rows in (16, 33, 65, 129, 300, 1024)
               for tokens in (784, 1680, 2064, 3088, 4096, 4112, 20000)]
    for rows, hq, hkv, d, q, kv, tokens in shapes:
        if rows * tokens <= threshold:
            continue
        args = rows, hq, hkv, d, 16, tokens // 16, q, kv, 0
        lib.aicomp_kv_set_small_decode_tokens(0)
        most = lib.aicomp_paged_decode_workspace_bytes(*args)
        lib.aicomp_kv_set_small_decode_tokens(threshold)
        assert lib.aicomp_paged_decode_workspace_bytes(*args) <= most, args
