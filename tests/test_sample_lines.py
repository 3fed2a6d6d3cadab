"""Which sampling calls are cut into parts of a row: the scratch the library asks for (host arithmetic, no GPU)."""
import pytest

from aicomp_amd import _lib

F32, BF16, F16 = _lib.F32, _lib.BF16, _lib.F16


@pytest.mark.parametrize("dtype,batch,vocab,top_k,cut", [
    # few kept candidates; 16-bit rows, whose ties are often more than the short merge takes, up to 56 and 60
    (F32, 64, 32000, 64, True), (F32, 64, 32000, 65, False), (BF16, 64, 32000, 56, True), (BF16, 64, 32000, 57, False),
    (F16, 64, 32000, 60, True), (F16, 64, 32000, 61, False), (BF16, 64, 128256, 64, True), (BF16, 65, 128256, 64, False),
    # up to 256 rows are under way together: 512 parts, of five 640
    (BF16, 170, 40000, 20, True), (BF16, 171, 40000, 20, False), (BF16, 256, 32000, 20, True), (BF16, 128, 65536, 50, True),
    (BF16, 129, 65536, 50, False), (F16, 128, 81920, 50, True), (F16, 129, 81920, 50, False), (BF16, 257, 65536, 50, True),
    (BF16, 128, 128256, 50, True), (BF16, 129, 128256, 50, False),
    (F32, 256, 32768, 50, True), (F32, 129, 32768, 51, False), (F32, 128, 32768, 51, True), (F32, 257, 32768, 51, True),
    (F32, 129, 65536, 51, True),
    # one part, more parts than there are, a vocabulary whose rows cannot be read in vectors
    (F32, 8, 16384, 50, False), (F32, 8, 262145, 50, False), (BF16, 64, 50257, 64, True)])
def test_calls_that_are_cut(dtype, batch, vocab, top_k, cut):
    need = _lib.load().aicomp_sample_workspace_bytes(batch, vocab, vocab, 0.8, top_k, 0, dtype)
    assert (need > 0) == cut
