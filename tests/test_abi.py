"""The C-ABI library loads without a GPU and exports every function the
header declares; host-only entry points behave as documented."""
import ctypes
import os
import re

import pytest

from bitnet_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    names = []
    for header in ("bitlinear_hip.h", "bitnet_decoder_ops.h", "bitlinear_probes.h"):
        text = open(os.path.join(ROOT, "include", header)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names += re.findall(r"\b(bit(?:linear|net)_[a-z0-9_]+)\s*\(", text)
    return names


def test_header_declares_the_drop_in_symbol():
    names = _declared_functions()
    assert "bitlinear_int8xint2" in names
    assert len(names) == len(set(names)) >= 9


def test_library_exports_every_declared_symbol():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built (run python -m bitnet_amd.build)")
    raw = ctypes.CDLL(_lib.LIB_PATH)
    for name in _declared_functions():
        assert hasattr(raw, name), name
    # and the binding table covers exactly the header
    assert set(_lib.SIGNATURES) == set(_declared_functions())


def test_missing_library_fails_loudly(tmp_path):
    with pytest.raises(_lib.BitLinearLibraryError):
        _lib.load_library(str(tmp_path / "nope.so"))


def test_host_only_entry_points():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.load_library()
    # shape table of the reference dispatcher (gpu/bitnet_kernels/bitnet_kernels.cu:4-33)
    table = {(3840, 2560): 3, (2560, 2560): 1, (13824, 2560): 2, (2560, 6912): 1, (4800, 3200): 6,
             (3200, 3200): 1, (20480, 3200): 2, (3200, 10240): 1, (5120, 27648): 1, (55296, 5120): 1}
    for (n, k), v in table.items():
        assert lib.bitlinear_ws_num(n, k) == v
    assert lib.bitlinear_ws_num(1024, 4096) == 1
    # the load-time converter is the identity: the converted weight has the reference's size
    assert lib.bitlinear_repacked_size(2560, 6912) == 2560 * 6912 // 4
    assert lib.bitlinear_repacked_size(100, 2560) == 0 and lib.bitlinear_repacked_size(2560, 100) == 0
    assert lib.bitlinear_repack(None, None, 100, 2560, None) == 1 and lib.bitlinear_repack(None, None, 2560, 2560, None) == 2
    assert lib.bitlinear_quant_absmax_rowsum(None, None, None, None, 1, 2560, 0, None) == 2
    assert lib.bitlinear_status_string(0) == b"ok"
    assert b"shape" in lib.bitlinear_status_string(1)
    assert lib.bitlinear_set_tuning(2, 8, 4, 0) == 0
    assert lib.bitlinear_set_tuning(2, 17, 4, 0) != 0
    assert lib.bitlinear_set_tuning(2, 8, 3, 0) != 0
    assert lib.bitlinear_set_tuning(1, 4, 0, 0) != 0  # no kernel 1
    assert lib.bitlinear_set_tuning(3, 1, 1, 0) != 0
    assert lib.bitlinear_set_tuning(3, 2, 8, 5) == 0
    assert lib.bitlinear_set_tuning(3, 4, 5, 4) != 0
    assert lib.bitlinear_set_tuning(5, 1, 0, 0) == 0
    assert lib.bitlinear_set_tuning(6, 1, 0, 0) == 0
    assert lib.bitlinear_set_tuning(6, 3, 0, 0) != 0
    assert lib.bitlinear_set_tuning(7, 1, 0, 0) == 0
    assert lib.bitlinear_set_tuning(7, 3, 0, 0) != 0
    assert lib.bitlinear_set_tuning(8, 1, 8, 5) == 0 and lib.bitlinear_set_tuning(8, 5, 0, 0) == 0
    assert lib.bitlinear_set_tuning(8, 2, 9, 5) != 0 and lib.bitlinear_set_tuning(8, 1, 8, 6) != 0
    assert lib.bitlinear_set_tuning(9, 2, 0, 0) == 0 and lib.bitlinear_set_tuning(9, 3, 0, 0) != 0
    assert lib.bitlinear_set_tuning(9, 1, 4, 0) == 0 and lib.bitlinear_set_tuning(9, 1, 5, 0) != 0
    assert lib.bitlinear_set_tuning(10, 1, 8, 5) == 0 and lib.bitlinear_set_tuning(10, 2, 0, 0) == 0
    assert lib.bitlinear_set_tuning(10, 1, 8, 6) != 0 and lib.bitlinear_set_tuning(10, 3, 0, 0) != 0
    assert lib.bitlinear_set_tuning(11, 1, 0, 0) == 0 and lib.bitlinear_set_tuning(11, 2, 0, 0) == 0
    assert lib.bitlinear_set_tuning(11, 3, 0, 0) != 0 and lib.bitlinear_set_tuning(12, 0, 0, 0) != 0
    assert lib.bitlinear_set_tuning(0, 0, 0, 0) == 0


def test_argument_checks_need_no_gpu(capfd):
    """Shape and NULL checks run before any HIP call."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.load_library()
    # N not a multiple of 16: the reference's message, nothing launched
    lib.bitlinear_int8xint2(None, None, None, None, None, 1, 100, 2560, None)
    assert lib.bitlinear_last_status() == 1
    assert "required ladder gemm kernel: M 1, N 100, K 2560" in capfd.readouterr().out
    lib.bitlinear_int8xint2(None, None, None, None, None, 1, 2560, 2560, None)
    assert lib.bitlinear_last_status() == 2
    assert lib.bitlinear_quant_absmax(None, None, None, 1, 2560, 0, None) == 2
    assert lib.bitlinear_quant_absmax(None, None, None, 1, 2563, 0, None) == 1
    assert lib.bitlinear_int8xint2_acc_i32(None, None, None, None, None, None, 1, 2560, 100, None) == 1
    # the allocation-free forward: sizes beyond its static scratch, then nulls, before any HIP call
    assert lib.bitlinear_forward_bf16_static(None, None, None, None, 16385, 2560, 64, 0, None) == 5
    assert lib.bitlinear_forward_bf16_static(None, None, None, None, 4096, 2560, 4160, 0, None) == 5
    assert lib.bitlinear_forward_bf16_static(None, None, None, None, 2048, 2560, 6912, 0, None) == 2


def test_decoder_entry_argument_checks_need_no_gpu():
    """The decoder-side entry points refuse bad shapes (1) and null pointers (2)
    before any HIP call."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    lib = _lib.load_library()
    # bitnet_attn_decode: head_dim, group size, split count, nulls
    assert lib.bitnet_attn_decode(None, None, None, None, None, None, None, None, None, 1, 1, 64, 4, 2, 64, None) == 1
    assert lib.bitnet_attn_decode(None, None, None, None, None, None, None, None, None, 1, 1, 64, 6, 2, 128, None) == 1
    assert lib.bitnet_attn_decode(None, None, None, None, None, None, None, None, None, 17, 1, 64, 4, 2, 128, None) == 1
    assert lib.bitnet_attn_decode(None, None, None, None, None, None, None, None, None, 1, 1, 64, 4, 2, 128, None) == 2
    assert lib.bitnet_attn_decode_rows(None, None, None, None, None, None, None, None, None, None, 1, 1, 64, 4, 2, 128, None) == 2
    assert lib.bitnet_attn_decode_workspace_floats(1, 20, 5, 8) == 1 * 5 * 8 * 4 * 130 * 2 + 5 + 2
    assert lib.bitnet_attn_decode_error_index(1, 20, 5, 8) == 1 * 5 * 8 * 4 * 130 * 2 + 5
    assert lib.bitnet_attn_decode_error_index(1, 20, 6, 8) == -1
    assert lib.bitnet_attn_decode_set_spin_limit(5) == 0 and lib.bitnet_attn_decode_set_spin_limit(-1) == 0
    assert len(lib.bitlinear_last_kernel()) > 0  # "none", or whatever an earlier test of this process launched
    assert lib.bitnet_attn_decode_workspace_floats(1, 20, 6, 8) == -1
    # prompt side: start + T beyond the cache, head_dim, nulls
    assert lib.bitnet_attn_prefill(None, None, None, None, 1, 40, 64, 30, 4, 2, 128, None) == 1
    assert lib.bitnet_attn_prefill(None, None, None, None, 1, 40, 64, 0, 4, 2, 64, None) == 1
    assert lib.bitnet_attn_prefill(None, None, None, None, 1, 40, 64, 0, 4, 2, 128, None) == 2
    assert lib.bitnet_rope_cache_tokens(None, None, None, None, None, None, None, 1, 0, 64, 4, 2, 128, None) == 1
    assert lib.bitnet_rope_cache_tokens(None, None, None, None, None, None, None, 1, 8, 64, 4, 2, 128, None) == 2
    assert lib.bitnet_decode_step_begin(None, None, None, None, None, None, None, 1, 100, 250, 64, 128, None) == 1  # dim % 8
    assert lib.bitnet_decode_step_begin(None, None, None, None, None, None, None, 1, 100, 256, 64, 128, None) == 2


def test_host_calls_refuse_bad_arguments_before_any_launch():
    """The native call module checks its operands itself: CPU tensors, non-tensors and wrong argument counts raise here,
    where no GPU exists."""
    import torch

    from bitnet_amd import bitlinear

    if not os.path.exists(_lib.HOST_CALLS_PATH):
        pytest.skip("not built")
    mod = bitlinear.BitLinearKernel(128, 32, seg_ends=(16, 32))
    x = torch.zeros(1, 128, dtype=torch.bfloat16)
    q, s = torch.zeros(1, 128, dtype=torch.int8), torch.ones(1, dtype=torch.bfloat16)
    for call in (lambda: mod(x), lambda: mod.quant_input(x), lambda: bitlinear.quant_input(x),
                 lambda: bitlinear.bitnet_int8xint2_linear(q, mod.weight, s, mod.weight_scale)):
        with pytest.raises(ValueError, match="must live on the GPU"):
            call()
    for call in (lambda: mod(None), lambda: bitlinear.quant_input([1.0]), lambda: _lib.host_calls().forward(x)):
        with pytest.raises(TypeError):
            call()


def _device_tensor(shape, dtype):
    """A tensor that says that it lives on the GPU, on a machine without one."""
    import torch

    class Sub(torch.Tensor):
        @classmethod
        def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
            raise AssertionError(f"no operator is called: {func}")

    return torch.Tensor._make_wrapper_subclass(Sub, shape, dtype=dtype, device="cuda")


@pytest.mark.parametrize("call", ["forward", "forward_segments", "linear", "quant", "pack", "unpack"])
def test_host_calls_refuse_tensors_without_storage(call):
    """What vmap and tracing hand over passes every check of shape, type and device and has no address: an error, in front
    of any allocation, and with the interpreter lock held."""
    import torch

    if not os.path.exists(_lib.HOST_CALLS_PATH):
        pytest.skip("not built")
    host = _lib.host_calls()
    w, ws = _device_tensor((32, 32), torch.int8), _device_tensor((4,), torch.bfloat16)
    shape, dtype, run = {
        "forward": ((2, 128), torch.bfloat16, lambda t: host.forward(t, w, ws, 128, 32, 0, None)),
        "forward_segments": ((2, 128), torch.bfloat16, lambda t: host.forward(t, w, ws, 128, 32, 0, (ctypes.c_int * 2)(16, 32))),
        "linear": ((2, 128), torch.int8, lambda t: host.linear(t, w, _device_tensor((2,), torch.bfloat16), ws, None)),
        "quant": ((2, 128), torch.bfloat16, lambda t: host.quant(t, 0)),
        "pack": ((32, 128), torch.int8, lambda t: host.pack(t)),
        "unpack": ((32, 32), torch.int8, lambda t: host.unpack(t, 32, 128)),
    }[call]
    with pytest.raises(RuntimeError, match="data pointer"):
        torch.vmap(run)(_device_tensor((3, *shape), dtype))


def test_decode_stack_looks_at_what_its_addresses_point_to():
    """The persistent decode kernel gets raw addresses: parameters and caches that it would read as something else leave
    the step to the calls per layer, which refuse them (or take them)."""
    import torch

    from bitnet_amd import decoder

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    args = decoder.ModelArgs(dim=256, n_layers=2, n_heads=2, n_kv_heads=1, vocab_size=32, ffn_dim=128, segment_scales=True)

    def made():
        model = decoder.Transformer(args).to(torch.bfloat16)
        return model, model.make_cache(2, 40, "cpu")

    model, cache = made()
    assert decoder.DecodeStack.applies(model, 2, cache, 3)

    def att(m):
        return m.layers[1].attention

    def norm_of(width):
        return lambda m, c: setattr(att(m).attn_sub_norm.weight, "data", torch.ones(width, dtype=torch.bfloat16))

    def weight_of(t):
        return lambda m, c: setattr(att(m).wqkv.weight, "data", t)

    def scale_of(t):
        return lambda m, c: setattr(att(m).wqkv.weight_scale, "data", t)

    spoiled = {
        "a short norm": norm_of(128), "a long norm": norm_of(257),
        "an unpacked weight": weight_of(torch.zeros(512, 256, dtype=torch.int8)),
        "a weight of few rows": weight_of(torch.zeros(256, 64, dtype=torch.int8)),
        "a weight of another type": weight_of(torch.zeros(512, 64, dtype=torch.float32)),
        "few scales": scale_of(torch.ones(2, dtype=torch.bfloat16)),
        "scales of another type": scale_of(torch.ones(4, dtype=torch.float32)),
        "a module of another width": lambda m, c: setattr(m.layers[0].feed_forward, "w2", decoder.BitLinearKernel(256, 256)),
        "no eps": lambda m, c: setattr(m.layers[0].ffn_norm, "eps", 0.0),
        "an eps that is no number": lambda m, c: setattr(m.layers[0].ffn_norm, "eps", float("nan")),
        "a cache of few rows": lambda m, c: c.__setitem__(1, tuple(t[:, :30].contiguous() for t in c[1])),
        "a cache with gaps": lambda m, c: c.__setitem__(1, tuple(torch.cat((t, t), dim=3)[..., ::2] for t in c[1])),
        "a cache of few layers": lambda m, c: c.pop(),
    }
    for what, spoil in spoiled.items():
        model, cache = made()
        spoil(model, cache)
        assert not decoder.DecodeStack.applies(model, 2, cache, 3), what
