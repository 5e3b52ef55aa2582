"""The rule that sends a decode batch's projection to the library's own kernel or to hipBLASLt: the model's own
projections stay in the own kernel over the decode batch, a large LM head of many rows does not."""
import pytest

from speech_serving import native


@pytest.mark.parametrize("d", [256, 384, 512, 768, 1024, 1280])
@pytest.mark.parametrize("rows", [1, 4, 16, 32, 64, 96, 128])
def test_projections_of_16_bit_layers_stay(d, rows):
    for n, k, gelu in ((3 * d, d, False), (d, d, False), (4 * d, d, True), (d, 4 * d, False)):
        assert native.decode_pays(rows, n, k, False, gelu), (rows, n, k)


@pytest.mark.parametrize("d", [256, 384, 512, 768, 1024, 1280])
@pytest.mark.parametrize("rows", [1, 4, 16, 32])
def test_projections_of_fp32_layers_stay(d, rows):
    for n, k, gelu in ((3 * d, d, False), (d, d, False), (4 * d, d, True), (d, 4 * d, False)):
        assert native.decode_pays(rows, n, k, True, gelu), (rows, n, k)


@pytest.mark.parametrize("n", [51200, 51864])
def test_a_large_lm_head_leaves_where_it_is_slower(n):
    """The rows from which hipBLASLt serves an LM head whose vocabulary the own kernel takes (a multiple of 4)."""
    first = {}
    for wide in (False, True):
        for k in (256, 384, 768, 1024, 1280):
            refused = [m for m in range(1, 129) if not native.decode_pays(m, n, k, wide)]
            assert refused == list(range(refused[0], 129))  # one crossover
            first[wide, k] = refused[0]
    assert all(first[False, k] <= 41 for k in (256, 384, 768, 1024, 1280))
    assert first[False, 1280] <= 17 and all(first[True, k] == 1 for k in (384, 768, 1024, 1280))


def test_fp32_rows_past_4_kib_and_partials():
    assert native.decode_pays(64, 3840, 1280, True) and not native.decode_pays(80, 3840, 1280, True)
    assert native.decode_pays(96, 1280, 1280, True) and not native.decode_pays(128, 1280, 1536, True)
    assert native.decode_pays(32, 5120, 1280, True, True) and not native.decode_pays(32, 5120, 1280, True, False)
    assert not native.decode_pays(64, 5120, 1280, True, True)
    assert native.decode_pays(64, 1280, 5120, True) and not native.decode_pays(96, 1280, 5120, True)
    assert native.decode_pays(128, 1280, 5120, False) and not native.decode_pays(128, 2048, 8192, False)
