"""When an eager call takes the native step, as far as that shows without a GPU."""
import contextlib
import sys
import types
import warnings

import pytest
import torch

import bf16_huffman_infer_amd
from bf16_huffman_infer_amd import _lib, functional, ops


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


def test_without_the_native_step_the_custom_ops_take_the_calls(monkeypatch):
    """It is missing, or was built for another torch: one warning, and every call goes the way it goes where it is not
    taken.  (The library of kernels has no such substitute.)"""
    monkeypatch.setattr(_lib, "_eager", None)
    monkeypatch.delattr(bf16_huffman_infer_amd, "_bhi_torch", raising=False)
    monkeypatch.setitem(sys.modules, "bf16_huffman_infer_amd._bhi_torch", None)          # import raises ImportError
    with pytest.warns(RuntimeWarning, match="custom ops"):
        assert _lib.eager() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.eager() is None
        assert functional._eager(None, None, None, True) is None and functional._eager_weight(None, False) is None
    # the first op on a device: initialised as before, whether or not there is a step to tell
    monkeypatch.setattr(ops, "_ready_devices", set())
    monkeypatch.setattr(_lib, "load", lambda: types.SimpleNamespace(bhi_device_init=lambda: 0))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "device", lambda index: contextlib.nullcontext())
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 7, raising=False)
    assert ops._stream(types.SimpleNamespace(get_device=lambda: 0)) == 7 and ops._ready_devices == {0}
