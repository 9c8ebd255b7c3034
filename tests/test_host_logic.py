"""Host-side behaviour of the operator that needs no GPU: argument validation and exception
types (reference linear_cross_entropy.py:125-192, cce.py:278-284), the preset table
(cce_utils.py:32-70), and the dense impl="torch_compile" path against the oracle."""

import pytest
import torch

from _util import IGNORE_INDEX, make_inputs
from oracle import dense_lce


def _small():
    e, c, t, bias = make_inputs(24, 32, 16, torch.float32, seed=1, bias=True)
    return e.view(2, 12, 16), c, t.view(2, 12), bias


def test_exports():
    import cut_cross_entropy as cce

    for name in ("LinearCrossEntropy", "LinearCrossEntropyImpl", "linear_cross_entropy", "VocabParallelOptions"):
        assert hasattr(cce, name)
    from cut_cross_entropy.cce_backward import cce_backward_kernel  # noqa: F401
    from cut_cross_entropy.cce_lse_forward import cce_lse_forward_kernel  # noqa: F401
    from cut_cross_entropy.constants import IGNORE_INDEX as pkg_ignore
    from cut_cross_entropy.indexed_dot import indexed_neg_dot_forward_kernel  # noqa: F401
    from cut_cross_entropy.utils import compute_z_loss  # noqa: F401

    assert pkg_ignore == -100


@pytest.mark.parametrize("shift", [-1, 12, 40])
def test_shift_out_of_range_is_value_error(shift):
    from cut_cross_entropy import linear_cross_entropy

    e, c, t, _ = _small()
    with pytest.raises(ValueError, match="Shift must be in the range"):
        linear_cross_entropy(e, c, t, shift=shift, impl="torch_compile")


def test_bias_length_and_shard_size_are_value_errors():
    from cut_cross_entropy import VocabParallelOptions, linear_cross_entropy

    e, c, t, bias = _small()
    with pytest.raises(ValueError, match="Bias has a different number of elements"):
        linear_cross_entropy(e, c, t, bias=bias[:-1], impl="torch_compile")
    with pytest.raises(ValueError, match="Expected c.size"):
        linear_cross_entropy(e, c, t, impl="torch_compile", vocab_parallel_options=VocabParallelOptions(0, 31))


def test_unknown_impl_and_reduction():
    from cut_cross_entropy import linear_cross_entropy

    e, c, t, _ = _small()
    with pytest.raises(NotImplementedError):
        linear_cross_entropy(e, c, t, impl="does_not_exist")
    with pytest.raises(ValueError):
        linear_cross_entropy(e, c, t, impl="torch_compile", reduction="median")


def test_cce_without_gpu_fails_loudly():
    """No silent fallback: the cce implementations need the HIP kernels and a GPU."""
    from cut_cross_entropy import linear_cross_entropy

    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    e, c, t, _ = _small()
    with pytest.raises(RuntimeError):
        linear_cross_entropy(e, c, t, impl="cce")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("moved", ["c", "t", "bias"])
def test_tensors_on_two_devices_are_refused_by_their_devices(dtype, moved):
    """The launchers, which hand on addresses, ask for the devices before anything else: also where there is no GPU."""
    from cut_cross_entropy.cce_lse_forward import loss_forward
    from cut_cross_entropy.fp32_path import fp32_forward

    e, c, t, bias = _small()
    given = {"e": e.to(dtype).flatten(0, -2), "c": c.to(dtype), "t": t.flatten(), "bias": bias.to(dtype)}
    given[moved] = given[moved].to("meta")
    e, c, t, bias = given.values()
    with pytest.raises(RuntimeError, match="on one device"):
        if dtype == torch.float32:
            fp32_forward(e, c, bias, t, None, 0, None, 0)
        else:
            loss_forward(e, c, bias, t, None, 0, None, 0, False)


def test_shape_asserts():
    from cut_cross_entropy.torch_compile import torch_compile_linear_cross_entropy

    e, c, t, _ = _small()
    with pytest.raises(AssertionError):
        torch_compile_linear_cross_entropy(e, c, t[:, :-1])
    with pytest.raises(AssertionError):
        torch_compile_linear_cross_entropy(e, c[:, :-1], t)


def test_preset_table():
    from cut_cross_entropy.cce_utils import CCEPreset, CCEPresets, LinearCrossEntropyImpl

    user = CCEPreset(filter_eps=0.25, accum_e_fp32=False, accum_c_fp32=False, filter_e_grad=False, filter_c_grad=True)
    assert CCEPresets.build_for_impl("cce", user) == user
    for name in ("cce_exact", "cce_kahan_full", "cce_kahan_full_c_full_e"):
        got = CCEPresets.build_for_impl(name, user)
        assert got["filter_eps"] is None and got["accum_e_fp32"] and got["accum_c_fp32"]
        assert got["filter_e_grad"] is False and got["filter_c_grad"] is True  # untouched
    got = CCEPresets.build_for_impl("cce_kahan_full_c", user)
    assert got == dict(filter_eps="auto", accum_e_fp32=True, accum_c_fp32=True, filter_e_grad=True, filter_c_grad=False)
    got = CCEPresets.build_for_impl("cce_kahan_full_e", user)
    assert got == dict(filter_eps="auto", accum_e_fp32=True, accum_c_fp32=True, filter_e_grad=False, filter_c_grad=True)
    with pytest.raises(ValueError):
        CCEPresets.build_for_impl("torch_compile", user)
    names = {v.name.lower() for v in LinearCrossEntropyImpl}
    assert names == {"cce", "torch_compile", "cce_kahan_full_c", "cce_kahan_full_e", "cce_exact",
                     "cce_kahan_full_c_full_e", "cce_kahan_full"}
    assert (names - {"torch_compile"}) <= CCEPresets.names


def test_handle_eps_package():
    from cut_cross_entropy.utils import _handle_eps

    assert _handle_eps("auto", torch.bfloat16) == 2.44140625e-4
    assert _handle_eps(None, torch.bfloat16) is None
    assert _handle_eps(1e-3, torch.bfloat16) == 1e-3
    with pytest.raises(RuntimeError):
        _handle_eps(3, torch.bfloat16)
    with pytest.raises(RuntimeError):
        _handle_eps("never", torch.bfloat16)


@pytest.mark.parametrize("reduction", ["none", "mean", "sum"])
@pytest.mark.parametrize("shift", [0, 2])
@pytest.mark.parametrize("softcap", [None, 10.0])
@pytest.mark.parametrize("invalids", [False, True])
def test_torch_compile_impl_matches_oracle(reduction, shift, softcap, invalids):
    from cut_cross_entropy import linear_cross_entropy

    e, c, t, bias = make_inputs(48, 40, 12, torch.float64, seed=2, bias=True, invalid_frac=0.25 if invalids else 0.0)
    e, t = e.view(4, 12, 12), t.view(4, 12)
    got, got_lse = linear_cross_entropy(e, c, t, bias=bias, softcap=softcap, reduction=reduction, shift=shift,
                                        impl="torch_compile", return_lse=True)
    want, want_lse = dense_lce.dense_linear_cross_entropy(e, c, t, bias, IGNORE_INDEX, softcap, reduction, shift, True)
    # the dense path upcasts to float32 like the reference (torch_compile.py:38-46)
    assert got.shape == want.shape and got.dtype == torch.float32
    assert torch.allclose(got.double(), want, rtol=1e-5, atol=1e-5)
    assert torch.allclose(got_lse.double(), want_lse, rtol=1e-5, atol=1e-5)


def test_torch_compile_shard_matches_oracle():
    from cut_cross_entropy import VocabParallelOptions, linear_cross_entropy

    e, c, t, _ = make_inputs(30, 44, 10, torch.float64, seed=3)
    loss = linear_cross_entropy(e, c[11:33], t, impl="torch_compile", reduction="none",
                                vocab_parallel_options=VocabParallelOptions(11, 33))
    corr, lse = dense_lce.vp_shard_partials(e, c[11:33], t, 11, 33, None, None, torch.float64)
    assert torch.allclose(loss.double(), lse - corr, rtol=1e-5, atol=1e-5)


def test_vocab_parallel_options_and_dtensor_message():
    from cut_cross_entropy import VocabParallelOptions

    o = VocabParallelOptions(3, 9)
    assert (o.start, o.stop, o.group, o.reduce_e_grad) == (3, 9, None, True)


def test_forgotten_measurements_keep_their_word_until_it_has_been_written(monkeypatch):
    """A kernel writes a monitor's pinned word by its address.  After reset_backward_path_memory() the word of a measurement
    in flight stays held; the next backward waits for that measurement, drops it and takes its own."""
    import gc
    import weakref

    from cut_cross_entropy import cce_backward as bw

    class Event:
        waited = 0

        def query(self):
            return False

        def synchronize(self):
            Event.waited += 1

    def measure(mon, lib, tile_max, lse, B, V, filter_eps, dev):
        assert Event.waited == (1 if not seen else Event.waited)  # the one in flight has been waited for
        seen.append(1)
        mon.host[0], mon.pending_cells = 1, 100

    seen = []
    monkeypatch.setattr(bw, "_monitors", {})
    monkeypatch.setattr(bw, "FILTERED_BACKWARD_PATH", "auto")
    monkeypatch.setattr(bw._FlaggedMonitor, "measure", measure)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    mon = object.__new__(bw._FlaggedMonitor)
    mon.host, mon.event = torch.full((1,), 90, dtype=torch.int64), Event()
    mon.pending_cells, mon.fraction, mon.dense, mon.scratch = 100, 0.9, True, {}
    dev = torch.device("cuda", 0)
    bw._monitors[(0, 512, 64, torch.bfloat16)] = mon
    word = weakref.ref(mon.host)
    del mon
    bw.reset_backward_path_memory()
    gc.collect()
    assert word() is not None
    assert bw._filtered_backward_runs_dense(None, None, None, 32, 512, 64, 1e-4, torch.bfloat16, dev) is False
    assert len(seen) == 2 and Event.waited == 2  # its own cells, and those for the backward after it


def test_rows_of_steps_lead_to_the_elements_they_name():
    """Slices, permutations, expansions and dimensions of one entry, up to five dimensions: either the strides answered lead to the
    elements in order, or no one stride does (``view`` to a matrix of dense rows knows)."""
    import itertools

    from cut_cross_entropy.utils import _rows_of_steps

    def check(t):
        rows = _rows_of_steps(t)
        try:
            matrix = t.view(-1, t.size(-1))
        except RuntimeError:
            matrix = None
        if matrix is not None and matrix.stride(1) != 1 and matrix.size(1) > 1:
            matrix = None
        assert (rows is None) == (matrix is None), (t.shape, t.stride())
        if rows is not None:
            n, cols, step = rows
            assert n * cols == t.numel()
            assert torch.equal(t.as_strided((n, cols), (step, 1)), t.reshape(n, cols)), (t.shape, t.stride())

    for ndim in range(1, 6):
        for shape in itertools.product((1, 2, 3), repeat=ndim):
            base = torch.arange(int(torch.tensor(shape).prod())).view(shape)
            for order in itertools.permutations(range(ndim)) if ndim < 5 else [(0, 1, 2, 3, 4), (1, 2, 0, 3, 4), (3, 0, 1, 2, 4), (0, 3, 2, 1, 4)]:
                t = base.permute(order)
                check(t)
                for d in range(ndim):
                    if t.size(d) == 3:
                        check(t.narrow(d, 1, 2))
                        check(t.narrow(d, 2, 1))
                    if t.size(d) == 1:
                        check(t.expand(*t.shape[:d], 2, *t.shape[d + 1 :]))
    # what was read at the wrong places
    check(torch.arange(384).view(4, 1, 12, 8)[:, :, :5])
    check(torch.arange(160).view(5, 4, 1, 8).permute(1, 2, 0, 3))


def test_a_refused_loss_call_leaves_no_count_of_an_earlier_one():
    """The word that receives the count is kept from call to call: -1 after a refusal, so that a workspace too small from the start is
    told from one too small for the rows found.  Nothing is launched: the addresses are never followed."""
    import ctypes

    from cut_cross_entropy import _hip

    lib = _hip.load()
    count, somewhere = ctypes.c_int64(77), ctypes.addressof(ctypes.create_string_buffer(512))
    somewhere = (somewhere + 255) // 256 * 256

    def call(workspace, workspace_bytes, n=64, dtype=0):
        count.value = 77
        return lib.cce_loss_call(somewhere, somewhere, None, somewhere, somewhere, ctypes.addressof(count), somewhere, None, somewhere,
                                 None, workspace, workspace_bytes, n, 64, 512, 128, 128, 128, 1, 0, -100, 0, 0.0, 2, dtype, 0, None)

    assert call(None, 0) == _hip.ERR_WORKSPACE_TOO_SMALL and count.value == -1
    needed = lib.cce_loss_call_workspace_bytes(64, 512, 128, 0, 0)
    assert call(somewhere, needed - 1) == _hip.ERR_WORKSPACE_TOO_SMALL and count.value == -1
    assert call(somewhere + 8, needed) != 0 and count.value == -1
    assert call(somewhere, needed, n=65) != 0 and count.value == -1
    assert call(somewhere, needed, dtype=7) != 0 and count.value == -1
