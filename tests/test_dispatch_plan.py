"""Which kernel and launch shape the library picks, pinned over a grid of shapes (no GPU needed): the ten (N, K)
of the reference's dispatch table (gpu/bitnet_kernels/bitnet_kernels.cu:4-33) x ten token counts through the
drop-in product and the forward call, and the decoder's four shapes through the norm-folded calls, against the
committed table tests/golden/dispatch_plan.txt.  A changed threshold or plan shows up as changed rows."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests", "golden"))

import make_dispatch_plan as mk  # noqa: E402

from bitnet_amd import _lib  # noqa: E402


def test_dispatch_matches_the_committed_table():
    want = open(mk.PATH).read().splitlines()
    got = list(mk.rows())
    assert len(got) == len(want) == (2 * 10 + 3 * 4) * 10
    changed = [f"- {w}\n+ {g}" for w, g in zip(want, got) if w != g]
    assert not changed, f"{len(changed)} rows differ (regenerate with tests/golden/make_dispatch_plan.py if intended):\n" + "\n".join(changed[:10])


def test_plan_rows_say_what_the_design_says():
    """A few rows spelled out, so that the table cannot drift as a whole: one token goes through the kernel whose
    waves prepare their own slices, five to eight tokens (short rows) through the kernel whose lanes quantize for their
    own token, up to sixteen through a quantizer kernel plus the product without staging, more than sixteen through the MFMA GEMM, the largest matrix through the streaming kernel."""
    p = _lib.plan_name
    assert p(1, 1, 2560, 2560).startswith("bitlinear_solo_kernel<5, 5, 1, false, 0, false, 1> grid=(160,1,1) block=512")
    assert p(1, 1, 13824, 2560).startswith("bitlinear_solo_kernel<5, 5, 1, false, 0, false, 4> grid=(216,1,1)")
    assert p(2, 1, 3840, 2560).startswith("bitlinear_solo_kernel<5, 1, 1, true, 1, false, 1>")
    assert p(1, 8, 3840, 2560).startswith("bitlinear_solo_tok_kernel<5, 1> grid=(240,1,1) block=512")
    two = p(1, 16, 3840, 2560).split(" + ")
    assert len(two) == 2 and two[0].startswith("quant_absmax_rows_kernel<0, 5>") and two[1].startswith("gemv_i2_solo_kernel<5, 1, false>")
    assert "gemm_i2_prefill_kernel" in p(0, 17, 13824, 2560) and "gemm_i2_prefill_dma_kernel<2, 2, 256>" in p(0, 2048, 13824, 2560)
    # 2048 x 2560 outputs are 320 tiles of 64 x 256: one round of the machine plus a quarter -> tiles of two sizes in one
    # launch (256 + 256 workgroups); 2560 x 2560 outputs (400 tiles) leave too large a rest for that
    assert p(0, 2048, 2560, 6912).startswith("gemm_i2_prefill_mix_kernel<256> grid=(512,1,1) block=256")
    assert "gemm_i2_prefill_mix_kernel" not in p(0, 2560, 2560, 2560) and "gemm_i2_prefill_mix_kernel" not in p(0, 2048, 3840, 2560)
    assert p(0, 1, 55296, 5120).startswith("gemv_i2_stream_kernel<5, true>")
    assert p(0, 1, 20480, 3200).startswith("bitlinear_fused_kernel<")


def test_a_direct_forward_call_quantizes_in_the_products_launch_where_a_recorded_one_does_not():
    """Entries from 16 on stand for calls outside of a capture; only the forward call of 5 to 16 tokens is another one there."""
    p = _lib.plan_name
    for m, n, k, shape in ((16, 2560, 2560, "<5, 1> grid=(160,1,1) block=512"), (8, 2560, 6912, "<7, 1> grid=(160,1,1) block=1024")):
        assert p(17, m, n, k) == f"bitlinear_handed_kernel{shape} lds=0"
        quantizer, product = p(1, m, n, k).split(" + ")
        assert quantizer.startswith("quant_absmax") and product == f"gemv_i2_solo_kernel{shape[:5]}, false>{shape[6:]} lds=0"
    # one token, rows that every workgroup quantizes, many columns, rows that end within a cache line, more than sixteen tokens
    for m, n, k in ((1, 2560, 2560), (8, 3840, 2560), (16, 55296, 5120), (9, 2560, 2112), (17, 2560, 2560)):
        assert p(17, m, n, k) == p(1, m, n, k)
    # the line, 65536 outputs, at one and at several row blocks a wave, and the longest rows
    for m, n, k in ((16, 4096, 2560), (16, 4096, 8192), (15, 4368, 3200), (8, 8192, 4096), (5, 13104, 3328)):
        wider = n + 16 * -(-(65537 - m * n) // (16 * m))
        assert p(17, m, n, k).startswith("bitlinear_handed_kernel<") and p(17, m, wider, k) == p(1, m, wider, k)
    for entry in (0, 2, 3, 4):
        for m in (1, 8, 16, 512):
            assert p(16 + entry, m, 2560, 6912) == p(entry, m, 2560, 6912)


def test_the_gate_is_in_the_epilogue_only_where_that_is_ahead():
    """Against what the separate product would take: the launch with two tile sizes (ahead with 256-k chunks and at most one small
    tile per CU), the split-K kernel (ahead), the kernel with the epilogues (behind)."""
    lib = _lib.load_library()
    seen = set()
    for k in (640, 1152, 2560, 3200, 4096):
        for n in (1024, 2048, 4096, 5120, 8192, 10240, 11264, 13824, 20480):
            for m in (16, 17, 24, 33, 64, 129, 200, 256, 257, 300, 321, 352, 384, 400, 448, 512, 640, 800, 1088, 1300, 2048):
                applies, ahead = lib.bitlinear_norm_epilogue_applies(m, n, k, None, 0), lib.bitlinear_norm_gate_ahead(m, n, k, None, 0)
                product = _lib.plan_name(2, m, n, k).split(" + ")[-1]
                if "gemm_i2_prefill_mix_kernel" in product:
                    groups = int(product.split("grid=(")[1].split(",")[0])
                    rt = -(-m // 64)
                    bigs = min(256 * max(1, -(-n // 256) * rt // 256) // rt, n // 256) * rt
                    # (both kinds are rounded up to eight in the grid)
                    behind = k % 256 == 0 and groups - -(-bigs // 8) * 8 <= 256
                else:
                    behind = "gemv" in product
                want = int(applies and not behind)
                assert ahead == want, (m, n, k, product)
                seen.add((applies, ahead, product.split("<")[0]))
    assert {(1, 0, "gemm_i2_prefill_mix_kernel"), (1, 1, "gemm_i2_prefill_mix_kernel"), (1, 0, "gemv_i2_mfma_kernel"),
            (1, 1, "gemm_i2_prefill_kernel"), (0, 0, "gemm_i2_prefill_mix_kernel")} <= seen, seen
    # the 2B decoder's w13
    assert [lib.bitlinear_norm_gate_ahead(m, 13824, 2560, None, 0) for m in (32, 257, 320, 321, 512, 513)] == [1, 0, 0, 1, 1, 0]


def test_plan_name_argument_checks():
    import ctypes

    lib = _lib.load_library()
    buf = ctypes.create_string_buffer(64)
    assert lib.bitlinear_plan_name(5, 1, 2560, 2560, buf, 64) == 4 and lib.bitlinear_plan_name(0, 1, 2560, 2560, None, 64) == 2
    assert [lib.bitlinear_plan_name(e, 1, 2560, 2560, buf, 64) for e in (-1, 15, 16, 20, 21)] == [4, 4, 0, 0, 4]
    assert lib.bitlinear_plan_name(0, 1, 100, 2560, buf, 64) == 1 and buf.value == b""  # a shape the library refuses
    assert lib.bitlinear_plan_name(0, 1, 2560, 2560, buf, 8) == 0 and len(buf.value) == 7  # truncated, terminated
