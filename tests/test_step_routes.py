"""Which launches a step of the cache object runs, from its lengths alone (a cache without a device plans as well): over
gathered keys or not, prompts and decoding sequences apart or together.  The lengths on both sides of each rule are ones
whose routes were measured (the times a layer are us on an MI355X, general launches / the other route)."""
import pytest
import torch

from tvm_amd import get_global_func as gf

GENERAL, GATHERED, NEW_TOKEN, APART = 0, 1, 2, 3
NORMAL, INLINE, NONE = 1, 2, 0


def routes(sequences, *, d=128, hq=32, hkv=8, page=16, rope=INLINE, window=0, layer_window=0, dtype=torch.float16):
    """(route of the plain layers, of those with a window) of a step of (cached, new) tokens."""
    kinds = [3, 0] if layer_window else [0]
    tokens = sum(c + n + 2 * page for c, n in sequences)
    config = [len(sequences), tokens, 1 << 17, page, int(window > 0)] + ([layer_window] if layer_window else [])
    cache = gf("vm.builtin.paged_attention_kv_cache_create")(config, [0, len(kinds)], hq, hkv, d, d, kinds, False, rope, 1.0, 1e4, None,
                                                             torch.empty((), dtype=dtype))
    for b, (cached, _) in enumerate(sequences):
        gf("vm.builtin.kv_state_add_sequence")(cache, b)
        if window:
            gf("vm.builtin.attention_kv_cache_enable_sliding_window_for_seq")(cache, b, window, 4)
        if cached:
            gf("vm.builtin.kv_state_begin_forward")(cache, [b], [cached], None)
            gf("vm.builtin.kv_state_end_forward")(cache)
    gf("vm.builtin.kv_state_begin_forward")(cache, list(range(len(sequences))), [n for _, n in sequences], None)
    flags = cache.flags()
    return flags["plain_route"], flags["window_route"]


def many(count, new, cached):
    return [(cached, new)] * count


@pytest.mark.parametrize("sequences,kind,want", [
    # RoPE inside: few row tiles over long keys keep the split of the general launch ...
    (many(1, 64, 30000), dict(d=128), GENERAL),             # 243 / 622
    (many(1, 64, 30000), dict(d=64), GENERAL),              # 150 / 555
    (many(1, 64, 30000), dict(d=96), GENERAL),              # 398 / 581
    (many(1, 64, 30000), dict(d=256, hq=16), GENERAL),      # 711 / 1998
    (many(1, 8, 30000), dict(d=128), GENERAL),              # 100 / 574
    (many(1, 64, 100000), dict(d=128), GENERAL),            # 586 / 2041
    (many(2, 64, 30000), dict(d=128), GENERAL),             # 358 / 668
    (many(1, 256, 30000), dict(d=64), GENERAL),             # 410 / 558
    (many(8, 64, 4000), dict(d=256, hq=16), GENERAL),       # 394 / 420
    (many(1, 64, 20000), dict(d=128, page=24), GENERAL),    # 336 / 419
    (many(1, 64, 30000), dict(d=128, page=24, rope=NORMAL), GENERAL),   # 251 / 618
    (many(4, 64, 30000), dict(d=128, page=24, rope=NORMAL), GENERAL),   # 611 / 751
    (many(32, 16, 3000), dict(d=128, page=24, rope=NORMAL), GENERAL),   # 197 / 251
    # ... and many row tiles, or short keys, rotate or look up every key once
    (many(1, 1024, 30000), dict(d=128), GATHERED),          # 2531 / 657
    (many(1, 1024, 30000), dict(d=64), GATHERED),           # 1505 / 580
    (many(16, 64, 4000), dict(d=128), GATHERED),            # 377 / 212
    (many(1, 8, 1000), dict(d=128), GATHERED),              # 135 / 38
    (many(4, 250, 4000), dict(d=96), GATHERED),             # 568 / 131
    (many(4, 250, 4000), dict(d=256, hq=16), GATHERED),     # 762 / 308
    (many(16, 64, 4000), dict(d=128, page=24, rope=NORMAL), GATHERED),  # 388 / 213
    (many(4, 250, 4000), dict(d=128, window=4096), GATHERED),           # 400 / 140
    (many(1, 512, 4000) + many(31, 1, 4000), dict(d=128), GATHERED),    # 553 / 344
    # windows without rotation on the tuned kernels: nothing to gain
    (many(16, 64, 4000), dict(d=128, window=4096, rope=NONE), GENERAL),  # 128 / 210
    (many(4, 250, 4000), dict(d=64, window=4096, rope=NONE), GENERAL),   # 85 / 103
    # more keys than the gathered rows may take (1 GiB)
    (many(2, 4096, 140000), dict(d=128), GENERAL),
])
def test_steps_over_gathered_keys(sequences, kind, want):
    assert routes(sequences, **kind)[0] == want


LONG_AND_CHUNK = [(6000, 1), (4000, 64)]      # the step is small enough for the general launch to split its keys
LONG_AND_PROMPT = [(30000, 1), (0, 2000)]     # too many row tiles for that: one workgroup walks the long sequence


@pytest.mark.parametrize("sequences,kind,want", [
    (LONG_AND_CHUNK, dict(d=128), GENERAL),                          # 33 / 55
    (LONG_AND_CHUNK, dict(d=64), GENERAL),                           # 28 / 46
    (LONG_AND_CHUNK, dict(d=128, hq=64), GENERAL),                   # 43 / 69
    (LONG_AND_CHUNK, dict(d=128, dtype=torch.float32), GENERAL),     # 182 / 332
    (LONG_AND_CHUNK, dict(d=64, hq=8, dtype=torch.float32), GENERAL),  # 87 / 203
    (LONG_AND_CHUNK, dict(d=72), GENERAL),                           # 120 / 162
    (LONG_AND_CHUNK, dict(d=256, hq=16, page=24), GENERAL),          # 168 / 244
    (many(6, 1, 8000) + many(2, 33, 2000), dict(d=128), GENERAL),    # 64 / 88
    (many(6, 1, 8000) + many(2, 33, 2000), dict(d=64, hq=8, dtype=torch.float32), GENERAL),  # 95 / 159
    (many(3, 1, 30000) + many(1, 64, 3000), dict(d=128), GENERAL),   # 104 / 119
    (many(8, 1, 4000) + many(1, 1000, 0), dict(d=64, hq=8), GENERAL),  # 38 / 53
    (LONG_AND_PROMPT, dict(d=128), APART),                           # 574 / 115
    (LONG_AND_PROMPT, dict(d=64), APART),                            # 601 / 86
    (LONG_AND_PROMPT, dict(d=64, hq=8), APART),                      # 110 / 70
    (LONG_AND_PROMPT, dict(d=128, dtype=torch.float32), APART),      # 2271 / 571
    (LONG_AND_PROMPT, dict(d=72), APART),                            # 654 / 188
    (many(2, 1, 3000) + many(2, 300, 0), dict(d=128, hq=64), APART),  # 74 / 43
    (many(20, 1, 2000) + many(4, 400, 0), dict(d=64, hq=8, dtype=torch.float32), APART),  # 126 / 87
])
def test_steps_that_mix_prompts_and_decoding_sequences(sequences, kind, want):
    assert routes(sequences, **{"rope": NORMAL, **kind})[0] == want
    if kind.get("page") != 24:  # (odd pages could gather as well)
        order = sequences[::-1]
        assert routes(order, **{"rope": NORMAL, **kind})[0] == want


def test_layers_with_a_window_decide_for_themselves():
    # a window that ends the long walk: nothing worth a second launch there
    assert routes(LONG_AND_PROMPT, rope=NORMAL, layer_window=64) == (APART, GENERAL)
    assert routes([(30000, 1), (1500, 2000)], rope=NORMAL, layer_window=1024) == (APART, GENERAL)
    assert routes(LONG_AND_PROMPT, rope=NORMAL, layer_window=16384) == (APART, APART)
    assert routes(LONG_AND_CHUNK, rope=NORMAL, layer_window=1024) == (GENERAL, GENERAL)
    # the generic kernels have no form of it for such layers
    assert routes(LONG_AND_PROMPT, rope=NORMAL, layer_window=16384, dtype=torch.float32) == (APART, GENERAL)


@pytest.mark.parametrize("kind,want", [(dict(window=64), NEW_TOKEN), (dict(window=64, rope=NONE), NEW_TOKEN), (dict(window=64, d=96), GENERAL),
                                       (dict(window=64, page=24), GENERAL), (dict(rope=NORMAL), GENERAL), (dict(), GENERAL)])
def test_decode_steps(kind, want):
    assert routes([(100, 1), (30, 1)], **kind)[0] == want
