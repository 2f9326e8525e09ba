"""The entry points without ctypes in between: same values, and arguments that do not fit are errors."""
import ctypes as C

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


def test_output_tensors_are_torch_empty_s(monkeypatch):
    """The native allocation and the one without it: shape, type, device, strides, no gradient; what
    is no tensor or no count is refused."""
    import os
    import torch
    from litert_amd import build
    from litert_amd import fully_connected as fc
    native = fc._empty_functions()
    monkeypatch.setattr(build, "torch_tensors_name", lambda version: "missing.so")
    plain = fc._empty_functions()
    like = torch.zeros((3, 2), dtype=torch.float64, requires_grad=True)
    for functions in (native, plain):
        for empty, dtype in zip(functions, (torch.int8, torch.float32)):
            for shape in ((1, 2048), (0, 7), (5, 0), (77, 5003)):
                out = empty(like, *shape)
                want = torch.empty(shape, dtype=dtype, device=like.device)
                assert (out.shape, out.dtype, out.device, out.stride(), out.requires_grad) == \
                    (want.shape, want.dtype, want.device, want.stride(), False)
            with pytest.raises((TypeError, AttributeError)):
                empty(None, 1, 2)
            with pytest.raises(RuntimeError):
                empty(like, -1, 2)
    monkeypatch.undo()
    if os.path.exists(os.path.join(os.path.dirname(capi.LIB_PATH), build.torch_tensors_name(torch.__version__))):
        assert native[0].__name__ == "empty_int8"


def test_scratch_lives_as_long_as_it_is_held(monkeypatch):
    """Native and plain: distinct memory while both are held, of any size; what is no tensor or no size is
    refused."""
    import torch
    from litert_amd import build
    from litert_amd import fully_connected as fc
    native = fc._empty_functions()[2]
    monkeypatch.setattr(build, "torch_tensors_name", lambda version: "missing.so")
    plain = fc._empty_functions()[2]
    like = torch.zeros(3)
    for scratch in (native, plain):
        held = [scratch(like, size) for size in (1, 1 << 20, 1 << 20, 0)]
        assert len({address for address, _ in held[:3]}) == 3 and held[3][0] == 0
        address, memory = held[1]
        C.memset(address, 7, 1 << 20)
        assert C.string_at(address + (1 << 20) - 1, 1) == b"\x07"
        del held, memory
        with pytest.raises((TypeError, AttributeError)):
            scratch(None, 1)
        with pytest.raises((OverflowError, RuntimeError)):
            scratch(like, -1)


def test_output_allocation_lets_other_threads_run():
    """An allocation that takes its time (here: one that is filled) does not hold the interpreter's lock."""
    import threading
    import time
    import torch
    from litert_amd import fully_connected as fc
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)
    like = torch.zeros(1)
    torch.use_deterministic_algorithms(True)
    thread = threading.Thread(target=tick)
    thread.start()
    try:
        for empty, columns in zip(fc._empty_functions(), (1 << 30, 1 << 28)):
            start = time.perf_counter()
            empty(like, 1, columns)
            took = time.perf_counter() - start
            assert any(start + 0.3 * took < t < start + 0.7 * took for t in ticks), took
    finally:
        torch.use_deterministic_algorithms(False)
        stop.set()
        thread.join()


def test_a_helper_that_does_not_load_is_done_without(monkeypatch, tmp_path):
    """A file of the right name that this torch cannot load (one rebuilt under the same version)."""
    import torch
    from litert_amd import build
    from litert_amd import fully_connected as fc
    broken = tmp_path / "broken.so"
    broken.write_bytes(b"no library")
    monkeypatch.setattr(build, "torch_tensors_name", lambda version: str(broken))
    with pytest.warns(UserWarning, match="torch.empty"):
        empty_int8, empty_float32, scratch = fc._empty_functions()
    like = torch.zeros(1)
    assert empty_int8(like, 2, 3).dtype == torch.int8 and empty_float32(like, 2, 3).dtype == torch.float32
    assert scratch(like, 16)[0] != 0
