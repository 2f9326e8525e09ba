"""The entry points without ctypes in between: same values, and arguments that do not fit are errors."""
import pytest

from litert_amd import capi


def test_calls_agree_with_ctypes():
    lib, calls = capi.load(), capi.calls()
    for batches, depth, out_depth in ((1, 1, 1), (5, 4096, 4096), (33, 8192, 2048), (2048, 16384, 512)):
        assert calls.lrtfc_activation_workspace_bytes(batches, depth) == \
            lib.lrtfc_activation_workspace_bytes(batches, depth)
        for name in ("lrtfc_fc_blockwise_int4_preferred_form",):
            assert getattr(calls, name)(batches, depth, out_depth) == \
                getattr(lib, name)(batches, depth, out_depth)


def test_calls_refuse_arguments_that_do_not_fit():
    calls = capi.calls()
    with pytest.raises(TypeError):
        calls.lrtfc_activation_workspace_bytes(1)
    with pytest.raises(OverflowError):
        calls.lrtfc_activation_workspace_bytes(1 << 31, 64)
    with pytest.raises(TypeError):
        calls.lrtfc_activation_workspace_bytes("1", 64)
