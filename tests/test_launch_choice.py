"""Which kernel the launchers take for a shape, read from the launches themselves (recorder.py): the rules over sizes that
no other test would allocate."""
import ctypes

import pytest

from recorder import ptr, recorder

Q8_0 = 8


def rows_form(launches):
    """(waves, blocks an item) of the one launch, where it is the kernel that reads rows in long runs."""
    (one,) = launches
    assert one.kernel == "gemv_rows_kernel", one
    return int(one.params[2]), int(one.params[3])


@pytest.mark.parametrize("n_out", [98304, 128256, 152064, 256000])
@pytest.mark.parametrize("blocks, item", [(13, 1), (14, 2), (16, 2), (17, 2), (18, 0), (19, 2), (20, 2), (32, 2), (72, 2), (73, 1), (80, 1), (94, 1)])
def test_q8_0_matrices_of_many_turns(blocks, item, n_out):
    """Two-block items where their buffers fit LDS, one-block items where they do not: never out of the kernel while those fit
    it.  Of 18 blocks two-block items where the turns are whole (98304 rows on 256 CUs) or many (256000)."""
    want = item or (2 if n_out in (98304, 256000) else 1)
    assert rows_form(recorder().calls("orin_gemv", Q8_0, ptr(1), ptr(2), ptr(3), blocks * 256, n_out)) == (4, want)


Q4_K, Q5_K, Q6_K = 12, 13, 14


@pytest.mark.parametrize("wtype, blocks, pair, two", [
    (Q4_K, 16, True, True), (Q4_K, 15, True, True), (Q4_K, 24, False, True), (Q4_K, 14, False, True), (Q6_K, 14, True, True), (Q8_0, 12, True, True),
    (Q4_K, 14, True, False), (Q4_K, 12, True, False), (Q4_K, 18, False, False), (Q6_K, 20, True, False), (Q8_0, 10, True, False), (Q8_0, 16, False, False),
    (Q4_K, 33, True, False),
])
def test_workgroups_a_cu_of_many_turns(wtype, blocks, pair, two):
    """Two where a row's items come out (nearly) even among four waves, where there are more tiles than three workgroups a CU."""
    def workgroups(tiles):
        n_in, rows = blocks * 256, tiles * (8 if pair else 16)
        (one,) = (recorder().calls("orin_gemv_norm_gate_up_swiglu", wtype, ptr(1), ptr(2), ptr(3), ptr(4), 1e-5, ptr(5), n_in, rows) if pair
                  else recorder().calls("orin_gemv", wtype, ptr(1), ptr(2), ptr(3), n_in, rows))
        return one.grid[0]
    assert workgroups(768) == 768
    few = two and not (pair and blocks <= 16 and wtype != Q8_0)  # (up to four tiles a CU such pairs are 1 to 6 % slower by two)
    assert workgroups(770) == workgroups(1024) == (512 if few else 768)
    assert workgroups(1026) == workgroups(5000) == (512 if two else 768)


@pytest.mark.parametrize("wtype, blocks, pair, three", [
    (Q4_K, 22, False, (6, 8, 10)), (Q4_K, 24, True, (6, 8, 10)), (Q5_K, 23, False, (6, 8, 10)), (Q4_K, 32, False, (8, 10)), (Q5_K, 32, True, (8, 10)),
    (Q4_K, 16, True, (4, 8, 10)), (Q5_K, 15, True, (4, 8, 10)), (Q4_K, 16, False, ()), (Q5_K, 14, False, ()), (Q6_K, 24, False, (6,)), (Q6_K, 22, True, (6,)),
    (Q6_K, 16, True, (4,)), (Q6_K, 30, False, ()), (Q8_0, 12, True, ()), (Q8_0, 16, True, (4,)), (Q8_0, 24, True, ()),
])
def test_two_workgroups_a_cu_only_where_they_were_measured_faster(wtype, blocks, pair, three):
    """Tiles a CU, rounded up, at which three workgroups a CU were measured faster: 2055 launches of 784 to 8000 tiles."""
    def workgroups(tiles):
        n_in, rows = blocks * 256, tiles * (8 if pair else 16)
        (one,) = (recorder().calls("orin_gemv_norm_gate_up_swiglu", wtype, ptr(1), ptr(2), ptr(3), ptr(4), 1e-5, ptr(5), n_in, rows) if pair
                  else recorder().calls("orin_gemv", wtype, ptr(1), ptr(2), ptr(3), n_in, rows))
        return one.grid[0]
    for per_cu in (4, 5, 6, 7, 8, 9, 10, 11, 12, 20):
        want = 768 if per_cu in three else 512
        assert workgroups(256 * per_cu - 254) == workgroups(256 * per_cu) == want, per_cu


@pytest.mark.parametrize("wtype, blocks", [(Q4_K, 16), (Q4_K, 24), (Q6_K, 14), (Q6_K, 30), (Q8_0, 12)])
@pytest.mark.parametrize("pair", [False, True])
def test_the_tallest_matrices_stay_in_the_kernel_that_reads_long_runs(wtype, blocks, pair):
    """A workgroup's turns are counted in six bits: what two workgroups a CU would take in more than 62 is three's."""
    def one(tiles):
        n_in, rows = blocks * 256, tiles * (8 if pair else 16)
        (one,) = (recorder().calls("orin_gemv_norm_gate_up_swiglu", wtype, ptr(1), ptr(2), ptr(3), ptr(4), 1e-5, ptr(5), n_in, rows) if pair
                  else recorder().calls("orin_gemv", wtype, ptr(1), ptr(2), ptr(3), n_in, rows))
        return one.kernel, one.grid[0]
    two = 768 if wtype == Q8_0 and not pair else 512
    assert one(62 * 512 + 510) == ("gemv_rows_kernel", two)
    assert one(63 * 512) == one(62 * 768 + 766) == ("gemv_rows_kernel", 768)


F16 = 1


@pytest.mark.parametrize("n_in, heights, pair, want", [  # (waves, rows a batch, workgroups on 256 CUs)
    (5120, (768,), False, (4, 2, 256)), (5120, (1024,), False, (4, 2, 256)), (5120, (1026,), False, (4, 2, 512)), (5120, (5120, 1280, 1280), False, (4, 2, 512)),
    (5120, (512,), True, (4, 1, 256)), (5120, (513,), True, (4, 1, 512)), (3072, (2048,), False, (4, 4, 256)), (3072, (4096, 1024, 1024), False, (4, 4, 512)),
    (3104, (4096,), False, (4, 4, 256)), (3584, (4096, 512, 512), False, (4, 4, 512)), (4096, (4096,), False, (4, 4, 256)), (6144, (4096,), False, (4, 2, 512)),
    (2048, (2048, 512, 512), False, (4, 8, 384)), (2048, (8192,), False, (4, 8, 256)), (2048, (1536,), True, (4, 4, 384)), (2048, (8192,), True, (4, 4, 256)),
    (28672, (4096,), False, (8, 1, 256)), (28672, (4096,), True, (8, 1, 256)), (18944, (768,), False, (13, 1, 256)), (18944, (769,), False, (13, 2, 256)),
    (18944, (384, 96, 96), False, (13, 1, 256)), (18944, (640, 160, 160), False, (13, 2, 256)), (18944, (512,), True, (13, 1, 256)),
    (1024, (8192,), False, (2, 8, 512)), (512, (16384,), False, (1, 8, 1024)), (14336, (4096,), False, (4, 2, 256)),
])
def test_f16_batches_and_workgroups(n_in, heights, pair, want):
    """Bytes on their way at once and rows of the busiest CU, as measured: both sides of the lines."""
    calls = recorder().calls
    if pair:
        (one,) = calls("orin_gemv_norm_gate_up_swiglu", F16, ptr(1), ptr(2), ptr(3), ptr(4), 1e-5, ptr(5), n_in, heights[0])
    else:
        n, p = len(heights), ctypes.c_void_p * len(heights)
        (one,) = calls("orin_gemv_multi", F16, n, p(*map(ptr, range(1, 1 + n))), p(*[None] * n), p(*map(ptr, range(4, 4 + n))), (ctypes.c_int * n)(*heights), ptr(7), ptr(8), 1e-5, n_in, 0)
    assert one.kernel == "gemv_f16_kernel"
    assert (int(one.params[3]), int(one.params[1]), one.grid[0]) == want and one.block == 64 * want[0]


HEADS = {  # query heads, KV heads, head size
    "qwen1.5b": (12, 2, 128), "qwen7b": (28, 4, 128), "llama8b": (32, 8, 128), "llama1b": (32, 8, 64), "qwen3": (16, 8, 128),
}


def form_of(h, g, d, past, tokens, in_place=False):
    """"short", or the query columns of a workgroup, with the number of KV splits where there are any: "64x4"."""
    attend, *combine = recorder().calls("orin_fa_prefill", ptr(1), ptr(2), ptr(3), ptr(1 if in_place else 4), h, g, d, 32768 + 512, past, tokens, float(d ** -0.5))
    splits = attend.grid[1] // -(-h // g // 8)  # (heads of a group in eights)
    assert (splits > 1) == bool(combine)
    if attend.kernel == "fa_prefill_short_kernel":
        return "short"
    cols = 32 * int(attend.params[1])
    return f"{cols}x{splits}" if splits > 1 else f"{cols}"


def prefill_form(model, past, tokens):
    return form_of(*HEADS[model], past, tokens)


# us a launch of the forms that come near the fastest, as measured on an MI355X: every layer with rows of its own, replayed from a
# graph; a pair: that, and the same behind a write of 600 MB that empties the caches, as the layer's matrices do between two launches.
SHORT_WALKS = [
    ("qwen1.5b", 0, 45, {"short": (3.7, 4.2), "32": (4.9, 5.2)}),
    ("llama1b", 0, 45, {"short": (3.1, 3.8), "32": (4.0, 4.5)}),
    ("qwen1.5b", 0, 200, {"short": (5.7, 6.5), "32": (6.1, 6.6)}),
    ("qwen1.5b", 140, 100, {"short": (5.9, 6.7), "32": (6.2, 6.6)}),
    ("qwen1.5b", 550, 4, {"short": (7.1, 9.0), "32": (7.4, 9.2), "32x4": (8.0, 8.4)}),
    ("qwen1.5b", 0, 512, {"short": (7.3, 9.2), "32": (7.3, 8.3)}),
    ("qwen1.5b", 420, 100, {"short": (7.2, 8.7), "32": (7.2, 7.7)}),
    ("qwen1.5b", 550, 70, {"short": (7.5, 9.1), "32": (7.5, 8.1)}),
    ("qwen3", 550, 70, {"short": (7.5, 9.8), "32": (7.5, 9.0)}),
    ("qwen3", 200, 301, {"short": (7.4, 9.7), "32": (7.3, 8.6)}),
    ("llama8b", 420, 100, {"short": (7.3, 9.5), "32": (7.3, 8.4)}),
]


@pytest.mark.parametrize("model, past, tokens, us", SHORT_WALKS)
def test_short_walks_only_where_they_were_measured_faster(model, past, tokens, us):
    taken = sum(us[prefill_form(model, past, tokens)])
    assert taken <= 1.02 * min(map(sum, us.values()))


# (as above: a turn of the chip and a few workgroups)
PARTIAL_TURNS = [
    ("llama8b", 0, 260, {"short": (6.8, 8.3), "64": (8.3, 9.7), "32": (9.2, 10.6)}),
    ("qwen7b", 0, 280, {"short": (7.1, 8.3), "64": (8.4, 9.7), "32": (9.2, 10.8)}),
    ("qwen7b", 30, 260, {"short": (7.5, 9.0), "64": (8.4, 9.6), "32": (9.6, 11.2)}),
    ("llama8b", 0, 301, {"short": (7.7, 9.5), "64": (8.5, 10.1), "32": (10.0, 11.5)}),
    ("llama8b", 0, 360, {"short": (9.5, 11.6), "64": (9.0, 10.7), "32": (10.9, 12.5)}),
    ("qwen7b", 0, 420, {"short": (10.7, 12.7), "64": (9.4, 11.1), "32": (11.2, 13.1)}),
]


@pytest.mark.parametrize("model, past, tokens, us", PARTIAL_TURNS)
def test_a_partial_turn_costs_what_its_short_walks_take(model, past, tokens, us):
    taken = sum(us[prefill_form(model, past, tokens)])
    assert taken <= 1.02 * min(map(sum, us.values()))


# (us a launch, caches as they are between replays)
HEADS_OF_64 = [
    ("llama1b", 1501, 301, {"32": 11.9, "64": 11.9}),
    ("llama1b", 3584, 280, {"32": 20.7, "64x2": 22.5, "64": 24.0}),
    ("llama1b", 4500, 260, {"32": 24.5, "64": 29.3}),
    ("llama1b", 4500, 301, {"32": 25.0, "64x2": 26.0, "64": 29.1}),
    ("llama1b", 5500, 260, {"64x2": 28.2, "32": 28.4, "64": 34.3}),
    ("llama1b", 8000, 280, {"64x2": 36.2, "64": 48.1}),
    ("llama1b", 8000, 330, {"64x2": 38.7, "64": 48.1}),
    ("llama1b", 900, 420, {"64": 10.1, "32": 10.7}),
    ("llama1b", 420, 512, {"64": 9.1, "32": 10.5}),  # (32 columns: 9.1 to 12.0 from run to run)
    ("llama1b", 4500, 512, {"64": 31.1, "32": 32.2, "64x2": 32.9}),
    ("llama1b", 3584, 512, {"64": 25.9, "32": 27.4}),
]


@pytest.mark.parametrize("model, past, tokens, us", HEADS_OF_64)
def test_forms_of_head_dim_64_at_depth(model, past, tokens, us):
    assert us[prefill_form(model, past, tokens)] <= 1.1 * min(us.values())


FEW_TOKENS_DEEP = [
    ("qwen3", 32000, 24, {"64x16": 32.9, "32x16": 35.3}),
    ("llama8b", 32000, 11, {"64x16": 32.8, "32x16": 35.3}),
    ("llama8b", 16000, 32, {"64x16": 24.0, "64x8": 28.0, "32x8": 30.1}),
    ("qwen7b", 32000, 16, {"64x16": 28.2, "32x16": 30.1, "32x8": 37.4}),
    ("qwen1.5b", 32000, 32, {"32x16": 22.3, "64x16": 25.6, "32x8": 33.1}),
    ("llama1b", 32000, 32, {"64x16": 22.5, "32x8": 30.8, "32x16": 31.8}),
]


@pytest.mark.parametrize("model, past, tokens, us", FEW_TOKENS_DEEP)
def test_few_tokens_deep_in_a_context(model, past, tokens, us):
    assert us[prefill_form(model, past, tokens)] <= 1.07 * min(us.values())


def parameters(test):
    """Every combination of a test's parametrisations, as dictionaries."""
    out = [{}]
    for mark in test.pytestmark:
        if mark.name == "parametrize":
            names = [n.strip() for n in mark.args[0].split(",")]
            out = [{**o, **dict(zip(names, v))} for o in out for v in mark.args[1]]
    return out


def test_the_parity_tests_reach_every_form():
    """The forms of the shapes that test_gpu_parity.py takes on the GPU: each at head_dim 128, in place too; the same comments there."""
    import test_gpu_parity as t

    def forms(test, d, in_place=False):
        return {form_of(p["H"], p["G"], p["d"], p["n_past"], p["batch"], in_place) for p in parameters(test) if p["d"] == d}

    splits, shorts = forms(t.test_prefill_kv_splits, 128), forms(t.test_prefill_short_chunks, 128)
    assert splits | shorts >= {"short", "32"} | {f"{c}x{s}" for c in (32, 64) for s in (2, 4, 8, 16)}
    assert forms(t.test_prefill_short_chunks, 64) | forms(t.test_prefill_kv_splits, 64) >= {"short", "32x4", "32x16", "64x4", "64x8"}
    assert forms(t.test_prefill_in_place, 128, True) >= {"short", "32x2", "32x4", "32x16", "64x2", "64x8"}
    assert forms(t.test_prefill_in_place, 64, True) >= {"short", "32x4"}
    for p in parameters(t.test_short_walks_keep_infinities_and_nans_where_they_belong):
        assert form_of(p["H"], p["G"], p["d"], p["n_past"], p["batch"]) == "short", p


@pytest.mark.parametrize("heads, head_dim, tokens, start, aligned", [(64, 128, 3000001, 7, True), (8, 128, 8388607, 0, True), (3, 100, 8000000, 5, True),
                                                                     (64, 128, 400000, 1, False), (8, 64, 1000, 3, True)])
def test_cache_rows_in_slices_below_two_to_the_31_threads(heads, head_dim, tokens, start, aligned):
    """A launch counts its threads in 32 bits: a longer store goes out as several, one behind the other, that together move every row once."""
    off = 0 if aligned else 2
    launches = recorder().calls("orin_fa_kv_store_batch", ptr(1) + off, ptr(2), ptr(3), ptr(4), heads, head_dim, start + tokens, start, tokens, keep_args=7)
    vec = 8 if aligned and head_dim % 8 == 0 else 1
    done = 0
    for one in launches:
        assert one.kernel == "kv_store_kernel" and one.params == [str(vec), "false"]
        kc, vc, k, v, shape, rows, n = one.args
        threads = one.grid[0] * one.block
        needed = 2 * n * heads * (head_dim // vec)
        assert needed <= threads < needed + one.block and threads < 1 << 31
        assert (kc, vc) == (ptr(1) + off, ptr(2)) and shape == heads | head_dim << 32 and rows == (start + tokens) | (start + done) << 32
        assert (k, v) == (ptr(3) + 4 * done * heads * head_dim, ptr(4) + 4 * done * heads * head_dim)
        done += n
    assert done == tokens
    assert len(launches) == -(-tokens // (0x7fffff00 // (2 * heads * (head_dim // vec))))
