"""When an eager call takes the native step, as far as that shows without a GPU."""
import pytest

from bf16_huffman_infer_amd import _lib, functional


class _Taken:
    """In the place of the native step: takes everything."""

    @staticmethod
    def linear(*args):
        return "native"

    weight = linear


@pytest.mark.parametrize("huffman,seams", [(True, ("mv_huffman", "gemv_bf16_huffman", "gemv_bf16_grouped")),
                                           (False, ("mv_ans", "gemv_bf16_ans", "gemv_bf16_grouped"))])
def test_a_wrapper_in_the_place_of_what_would_run_sees_the_call(monkeypatch, huffman, seams):
    monkeypatch.setattr(_lib, "_eager", _Taken)
    for name in seams:
        assert functional._eager(None, None, None, huffman) == "native"
        with monkeypatch.context() as patch:
            patch.setattr(functional, name, lambda *args, **kwargs: None)
            assert functional._eager(None, None, None, huffman) is None, name
    decode = "huffman_decode" if huffman else "ans_decode"
    assert functional._eager_weight(None, huffman) == "native"
    monkeypatch.setattr(functional, decode, lambda *args: None)
    assert functional._eager_weight(None, huffman) is None
