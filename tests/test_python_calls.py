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


def test_extension_is_the_one_of_this_interpreter():
    import sysconfig
    assert capi.CALLS_PATH.endswith("litert_amd_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
    assert capi.calls().__file__ == capi.CALLS_PATH


def test_without_the_extension_calls_go_through_ctypes(monkeypatch):
    """An interpreter that the extension was not built for, or no Python.h to build it with."""
    monkeypatch.setattr(capi, "CALLS_PATH", capi.CALLS_PATH + ".missing")
    monkeypatch.setattr(capi, "_CALLS", None)
    with pytest.warns(UserWarning, match="through ctypes"):
        calls = capi.calls()
    assert calls is capi.load()
    assert calls.lrtfc_activation_workspace_bytes(5, 4096) == \
        capi.load().lrtfc_activation_workspace_bytes(5, 4096)
    # the arguments as ops pass them: integers for addresses, None for absent tensors
    status = calls.lrtfc_fc_int8_packed(None, 4096, None, None, None, 0, None, None, -1, 16, 16, 0, 0,
                                        0, 0, 0)
    assert status != capi.OK
