"""GPU parity of the whole cache object: the reference's scenario batches through the
HIP-backed cache, checked (a) against the numpy closed form the reference's own test uses,
(b) against the CPU oracle cache on identical seeded inputs, with page tables / append
indices / pool state compared bit for bit."""
import contextlib
import ctypes

import numpy as np
import pytest
import torch

import tvm_amd
from oracle.paged_kv_cache import OraclePagedKVCache
from tests import scenario as S
from tests.gpu_util import DEV, GpuCache, dev, host
from tests.test_host_cache_parity import GLOBAL, PER_DEPTH
from tests.util import assert_close
from tvm_amd import get_global_func as gf
from tvm_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,rope_mode", [(128, S.ROPE_NORMAL), (64, S.ROPE_NORMAL), (128, S.ROPE_NONE), (256, S.ROPE_NORMAL)])
@pytest.mark.parametrize("runner", [S.run_prefill_and_decode, S.run_remove_sequence, S.run_fork_sequence,
                                    S.run_unlimited_depth, S.run_popn])
def test_reference_scenarios_on_the_gpu(runner, d, rope_mode):
    """tests/python/relax/test_runtime_builtin_paged_attention_kv_cache_cpu.py:706-909 of the
    reference with its geometry (32 query / 4 kv heads, page 16, capacity 2048)."""
    layers, hq, hkv = 2, 32, 4
    cache = GpuCache([32, 2048, 512, 16, 0], layers, hq, hkv, d, d, rope_mode=rope_mode)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=rope_mode, seed=5, tol=4e-3)
    runner(sc)


@contextlib.contextmanager
def step_route(route):
    """Steps take this route wherever they can: 1 the general launches, 2 prompts and decoding sequences apart, 3 gathered keys."""
    prev = tvm_amd.set_option("step_route", route)
    try:
        yield
    finally:
        tvm_amd.set_option("step_route", prev)


def joint_launches():
    """Launches of two kinds of work side by side since the process began."""
    count = ctypes.c_uint64()
    check(lib().tvmkv_debug_joint_launches(ctypes.byref(count)))
    return count.value


@contextlib.contextmanager
def launches_apart():
    """A cap on the decode grid that none reaches: the same grids, one kind of work a launch."""
    prev = tvm_amd.set_option("decode_wgs_per_cu", 1 << 20)
    try:
        yield
    finally:
        tvm_amd.set_option("decode_wgs_per_cu", prev)


class Mirror:
    """Feeds the oracle cache and the GPU cache the same calls and the same tensors."""

    def __init__(self, cache_config, layers, hq, hkv, d, rope_mode=1, dtype=np.float16, **rope):
        self.o = OraclePagedKVCache(cache_config, layers, hq, hkv, d, d, rope_mode=rope_mode, dtype=dtype, **rope)
        self.g = GpuCache(cache_config, layers, hq, hkv, d, d, rope_mode=rope_mode, dtype=dtype, **rope)
        self.layers, self.hq, self.hkv, self.d = layers, hq, hkv, d
        self.dtype = dtype
        # float32 storage: what is left is the order of the float32 sums and the device's exp2 / sin / cos
        self.tol = dict(atol=2e-4, rtol=2e-4) if dtype == np.float32 else {}
        self.rng = np.random.default_rng(21)
        self.lengths = {}

    def compare_bookkeeping(self):
        aux = self.o.host.aux
        c = self.g.cache
        flags = c.flags()
        assert flags["num_depths"] == aux["num_depths"]
        assert bool(flags["append_before_attn"]) == aux["append_before_attn"]
        for dd in range(aux["num_depths"]):
            for name in PER_DEPTH:
                assert c.aux(name, dd) == aux[name][dd], f"{name}[{dd}]"
        for name in GLOBAL:
            assert c.aux(name) == aux[name], name
        so, sg = self.o.host.state(), c.state()
        assert sg["free_page_ids"] == so["free_page_ids"] and sg["free_block_idx"] == so["free_block_idx"]
        assert [tuple(b) for b in sg["blocks"]] == [tuple(b) for b in so["blocks"]] and sg["seqs"] == so["seqs"]
        assert c.copy_log() == self.o.host.copies

    def step(self, batch, routes=None):
        """routes: what flags() has to say of the step's plain layers and of those with a window."""
        ids, lens = [], []
        for item, n in batch:
            if isinstance(item, tuple):
                sid, parent, pos = item
                self.o.fork_sequence(parent, sid, pos)
                self.g.fork_sequence(parent, sid, pos)
                self.lengths[sid] = self.lengths[parent] if pos == -1 else pos
            else:
                sid = item
                if sid not in self.lengths:
                    self.o.add_sequence(sid)
                    self.g.add_sequence(sid)
                    self.lengths[sid] = 0
            ids.append(sid)
            lens.append(n)
        self.o.begin_forward(ids, lens)
        self.g.begin_forward(ids, lens)
        self.compare_bookkeeping()
        if routes is not None:
            flags = self.g.cache.flags()
            assert (flags["plain_route"], flags["window_route"]) == routes
        total = sum(lens)
        for layer in range(self.layers):
            qkv = self.rng.standard_normal((total, self.hq + 2 * self.hkv, self.d)).astype(self.dtype)
            eo = np.zeros((total, self.hq, self.d), self.dtype)
            go = np.zeros_like(eo)
            self.o.attention_with_fused_qkv(layer, self.d ** -0.5, qkv, eo)
            self.g.attention_with_fused_qkv(layer, self.d ** -0.5, qkv, go)
            assert_close(go, eo, what=f"layer {layer} output vs oracle cache", **self.tol)
        self.o.end_forward()
        self.g.end_forward()
        for sid, n in zip(ids, lens):
            self.lengths[sid] += n
            L = self.lengths[sid]
            if 3 in self.o.attn_kinds:  # debug_get_kv is for caches whose layers are all plain
                continue
            ek = np.zeros((self.layers, L, self.hkv, self.d), self.dtype)
            ev, gk, gv = np.zeros_like(ek), np.zeros_like(ek), np.zeros_like(ek)
            self.o.debug_get_kv(sid, 0, L, ek, ev)
            self.g.debug_get_kv(sid, 0, L, gk, gv)
            assert np.array_equal(gv, ev), f"cached V of seq {sid}"
            assert_close(gk, ek, atol=1e-3, rtol=2e-3, what=f"cached K of seq {sid}")


@pytest.mark.parametrize("page_size,hq,hkv,d", [(16, 32, 8, 128), (32, 32, 8, 128), (64, 32, 8, 128), (16, 8, 2, 96),
                                                (32, 12, 4, 80), (16, 4, 4, 112)])
def test_identical_inputs_through_oracle_and_gpu_caches(page_size, hq, hkv, d):
    m = Mirror([16, 4096, 1024, page_size, 0], 2, hq, hkv, d)
    m.step([(0, 60), (1, 88), (2, 17), (3, 4)])
    m.step([((4, 3, -1), 35)])
    m.step([((5, 0, 33), 20)])            # fork inside a page -> page copy on the device
    m.step([(0, 1), (1, 1), (2, 1), (4, 1), (5, 1)])
    m.step([((6, 5, -1), 40), (2, 3)])
    m.step([(6, 1), (5, 1), (0, 1)])      # two block depths + merge_state
    m.o.popn(6, 30)
    m.g.popn(6, 30)
    m.lengths[6] -= 30
    m.step([(6, 1), (1, 200)])
    m.step([(i, 1) for i in (0, 1, 2, 4, 5, 6)])


@pytest.mark.parametrize("dtype,page_size,hq,hkv,d", [(np.float32, 16, 8, 2, 128), (np.float32, 16, 32, 4, 64),
                                                      (np.float16, 24, 8, 2, 128), (np.float16, 5, 8, 2, 64),
                                                      (np.float32, 12, 6, 2, 72), (np.float16, 16, 8, 2, 72),
                                                      (np.float16, 48, 20, 1, 128)])
def test_float32_storage_other_page_sizes_and_head_dims_through_both_caches(dtype, page_size, hq, hkv, d):
    """What the reference's kernel factories accept beside the tuned shapes (its tests run float32 storage,
    test_runtime_builtin_paged_attention_kv_cache_cpu.py:269-276; page size and head dim are free parameters of
    every factory): the cache runs these on the generic matrix-core kernels.  Same calls and tensors through the
    oracle cache (the oracle's float32 build for float32 storage), page tables and pool state bit for bit."""
    m = Mirror([16, 2048, 512, page_size, 0], 2, hq, hkv, d, dtype=dtype)
    m.step([(0, 60), (1, 88), (2, 17), (3, 4)])
    m.step([((4, 3, -1), 35)])
    m.step([((5, 0, 33), 20)])            # fork inside a page -> page copy on the device
    m.step([(0, 1), (1, 1), (2, 1), (4, 1), (5, 1)])
    m.step([((6, 5, -1), 40), (2, 3)])
    m.step([(6, 1), (5, 1), (0, 1)])      # two block depths + merge_state
    m.o.popn(6, 30)
    m.g.popn(6, 30)
    m.lengths[6] -= 30
    m.step([(6, 1), (1, 200)])
    m.step([(i, 1) for i in (0, 1, 2, 4, 5, 6)])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("runner", [S.run_prefill_and_decode, S.run_remove_sequence, S.run_fork_sequence,
                                    S.run_unlimited_depth, S.run_popn])
def test_reference_scenarios_float32_storage(runner, d):
    """The float32 rows of the reference's fixture (head dims 64 and 128, RopeMode.NORMAL,
    test_runtime_builtin_paged_attention_kv_cache_cpu.py:269-276) with its geometry, against the numpy closed form."""
    layers, hq, hkv = 2, 32, 4
    cache = GpuCache([32, 2048, 512, 16, 0], layers, hq, hkv, d, d, rope_mode=S.ROPE_NORMAL, dtype=np.float32)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=S.ROPE_NORMAL, seed=5, tol=1e-3, dtype=np.float32)
    runner(sc)


def test_storage_type_of_the_tensors_is_checked():
    cache = GpuCache([4, 64, 32, 16, 0], 1, 8, 2, 128, 128, dtype=np.float32)
    cache.add_sequence(0)
    cache.begin_forward([0], [2])
    qkv = torch.zeros((2, 12, 128), dtype=torch.float16, device=DEV)
    out = torch.zeros((2, 8, 128), dtype=torch.float16, device=DEV)
    with pytest.raises(tvm_amd.KVError, match="stores float32"):
        gf("vm.builtin.attention_kv_cache_attention_with_fused_qkv")(cache.cache, 0, 1.0, qkv, out)


@pytest.mark.parametrize("dtype,page_size,d,tol", [(np.float16, 16, 96, 4e-3), (np.float32, 16, 128, 1e-3),
                                                   (np.float16, 24, 128, 4e-3), (np.float32, 12, 72, 1e-3)])
@pytest.mark.parametrize("runner", [S.run_sliding_window, S.run_sliding_window_fork, S.run_sliding_window_page_reuse])
def test_sliding_window_scenarios_on_the_generic_kernels(runner, dtype, page_size, d, tol):
    """The reference's sliding-window scenarios (attention sinks, window trimming, forks inside the sink, page reuse;
    test_runtime_builtin_paged_attention_kv_cache_cpu.py:912-1022) on caches that the tuned extended kernels do not
    serve: head dim 96, float32 storage, pages of 24 and 12 tokens.  Such a cache rotates inside the attention
    kernels and hands them the (3, batch) length_info."""
    layers, hq, hkv = 2, 8, 2
    cache = GpuCache([32, 2048, 512, page_size, 1], layers, hq, hkv, d, d, rope_mode=S.ROPE_INLINE, dtype=dtype)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=S.ROPE_INLINE, seed=4, tol=tol, dtype=dtype)
    runner(sc)


@pytest.mark.parametrize("dtype,page_size,d", [(np.float16, 16, 80), (np.float32, 16, 64), (np.float16, 40, 128)])
@pytest.mark.parametrize("sliding", [0, 1])
def test_inline_rope_and_forks_on_the_generic_kernels(dtype, page_size, d, sliding):
    """Caches that rotate inside the attention kernels (rope mode 2, with and without sliding-window support) at a
    head dim, a storage type and a page size of the generic kernels, with a frequency variant: prefill (ragged +
    paged + merge), decode, a fork with two block depths, against the oracle cache."""
    rope = dict(rope_theta=5e5, rope_scaling={"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0,
                                              "high_freq_factor": 4.0, "original_max_position_embeddings": 64})
    m = Mirror([8, 2048, 512, page_size, sliding], 2, 8, 2, d, rope_mode=2, dtype=dtype, **rope)
    m.step([(0, 60), (1, 88), (2, 17)])
    m.step([(0, 1), (1, 1), (2, 1)])
    m.step([((3, 1, 40), 25), (0, 2)])
    m.step([(3, 1), (1, 1)])


@pytest.mark.parametrize("page_size,d,hq,hkv,tol", [(16, 128, 8, 2, 4e-3), (16, 64, 8, 8, 4e-3), (32, 256, 4, 2, 4e-3),
                                                   (16, 96, 36, 18, 4e-3), (24, 80, 8, 4, 4e-3), (128, 112, 9, 1, 4e-3)])
def test_prefill_steps_of_windowed_caches_over_gathered_keys(page_size, d, hq, hkv, tol):
    """Prefill steps with enough rows run over keys gathered (and rotated) into one run per sequence: windows of one and
    several runs of 16 keys, with and without sinks, a sequence that is new, one that decodes beside the chunks, chunks
    longer than the window, more kv heads than one workgroup takes, every head dim, small and large pages."""
    layers, tuned = 2, page_size != 24 and d in (64, 128, 256)
    cache = GpuCache([8, 4096, 1024, page_size, 1], layers, hq, hkv, d, d, rope_mode=S.ROPE_INLINE)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=S.ROPE_INLINE, seed=4, tol=tol)
    for sid, (window, sink) in enumerate([(40, 0), (130, 4), (257, 30)]):
        sc.add_with_window(sid, window, sink)
    for batch in ([(0, 17), (1, 128), (2, 200)], [(0, 70), (1, 1), (2, 130)], [(3, 65), (2, 90), (0, 40)],
                  [(0, 33), (1, 129), (2, 1), (3, 16)], [(0, 1), (1, 1), (2, 1), (3, 1)], [(1, 64), (2, 63)]):
        with step_route(3):
            sc.step(list(batch))
        decode = all(n == 1 for _, n in batch)
        assert cache.cache.flags()["plain_route"] == ((2 if tuned else 0) if decode else 1)


@pytest.mark.parametrize("page_size,d,rope_mode", [(24, 128, 1), (5, 64, 1), (12, 256, 1), (40, 96, 0), (16, 128, 2), (16, 112, 2)])
def test_prefill_steps_of_other_caches_over_gathered_keys(page_size, d, rope_mode):
    """The same for caches without windows: pages the tuned kernels do not walk (keys kept rotated or never rotated) and
    RoPE inside the kernels, next to decode steps and forks, against the oracle cache."""
    m = Mirror([8, 2048, 512, page_size, 0], 2, 8, 2, d, rope_mode=rope_mode)
    with step_route(3):
        m.step([(0, 60), (1, 88), (2, 17)], (1, 0))
        m.step([(0, 64), (1, 1), (2, 130)], (1, 0))
        m.step([(0, 1), (1, 1), (2, 1)], (0, 0))
        m.step([(0, 15), (1, 90), (3, 33)], (1, 0))
        m.step([((4, 1, 40), 25), (0, 2)], (0, 0))


def test_gathered_rows_are_allocated_by_the_first_step_that_wants_them():
    """A cache takes no memory for gathered keys when it is created, nor for steps that run without them."""
    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info(0)[0]

    d, heads, tokens = 128, 8, 65536
    rows = (tokens + 16 + 4096) * 2 * heads * d * 2  # the pool's slots and a prefill chunk: 272 MiB
    step = torch.zeros((4096, 3 * heads, d), dtype=torch.float16, device=DEV)
    before = free()
    cache = GpuCache([4, tokens, 4096, 16, 0], 1, heads, heads, d, d, rope_mode=S.ROPE_INLINE)
    created = free()
    # pages, the chunk's q / k / v / output, the step's arrays; the allocator's granularity
    assert before - created < tokens * 2 * heads * d * 2 + 4 * 4096 * heads * d * 2 + (24 << 20)
    cache.add_sequence(0)
    left = []
    for route in (1, 1, 3, 3):  # (a kernel's first launch and split keys take memory of their own)
        with step_route(route):
            cache.begin_forward([0], [4096])
        _attend(cache, step, d)
        cache.end_forward()
        assert cache.cache.flags()["plain_route"] == int(route == 3)
        left.append(free())
    assert left[0] - left[1] < 64 << 20 and left[2] - left[3] < 64 << 20
    assert rows <= left[1] - left[2] < rows + (64 << 20)


@pytest.mark.parametrize("page_size,d", [(16, 128), (24, 64), (16, 96)])
def test_inline_rope_chunks_behind_long_contexts(page_size, d):
    """A chunk of few row tiles behind a long context, by the launch that splits its keys and over gathered keys."""
    for route in (1, 3):
        m = Mirror([4, 2000, 800, page_size, 0], 1, 2, 1, d, rope_mode=S.ROPE_INLINE)
        m.step([(0, 600)])
        m.step([(0, 500), (1, 7)])
        with step_route(route):
            m.step([(0, 33)], (int(route == 3), 0))
            m.step([(0, 3), (1, 20)], (int(route == 3), 0))


@pytest.mark.parametrize("page_size,d,hq,hkv,window", [(16, 128, 8, 2, 0), (16, 64, 8, 8, 0), (64, 128, 20, 1, 100), (16, 64, 8, 2, 1),
                                                      (32, 128, 18, 1, 1024), (16, 128, 4, 4, 1200), (128, 64, 4, 1, 33)])
def test_steps_that_mix_prompts_and_decoding_sequences(page_size, d, hq, hkv, window):
    """Decoding sequences of a mixed step run on the decode kernel with their new token as one more key: long contexts,
    one that ends at a page edge, one of a single token, one without any; prompts with and without cached tokens; layers
    with and without a window (0: none), windows inside one page and longer than some sequences."""
    m = Mirror([12, 6000, 2048, page_size, 0] + ([window] if window else []), 2 if window else 1, hq, hkv, d,
               **({"attn_kinds": [3, 0]} if window else {}))
    apart = (3, 3 if window else 0)
    with step_route(2):
        m.step([(0, 1300), (1, 64), (2, 300)], (0, 0))
        m.step([(3, 1), (1, 1)], (0, 0))
        m.step([(0, 1), (4, 40), (1, 1), (3, 1), (5, 1), (2, 17)], apart)
        m.step([(2, 1), (0, 1), (6, 130)], apart)
        m.step([(4, 3), (0, 1), (2, 1)], apart)
        m.step([(0, 1), (2, 1), (4, 1)], (0, 0))


@pytest.mark.parametrize("dtype,page_size,d,hq,hkv,window", [(np.float32, 16, 128, 8, 2, 0), (np.float32, 24, 64, 4, 4, 70),
                                                            (np.float32, 16, 256, 20, 1, 0), (np.float16, 20, 72, 6, 2, 0),
                                                            (np.float32, 16, 96, 4, 2, 1)])
def test_mixed_steps_on_the_generic_kernels(dtype, page_size, d, hq, hkv, window):
    """The same for storage types, pages and head dims of the generic kernels, whose launches merge into the state of the
    new tokens."""
    m = Mirror([12, 4000, 1024, page_size, 0] + ([window] if window else []), 2 if window else 1, hq, hkv, d, dtype=dtype,
               **({"attn_kinds": [3, 0]} if window else {}))
    with step_route(2):
        m.step([(0, 700), (1, 64), (2, 200)], (0, 0))
        m.step([(0, 1), (4, 40), (1, 1), (3, 1), (5, 1), (2, 17)], (3, 0))
        m.step([(2, 1), (0, 1), (6, 30)], (3, 0))
        m.step([(4, 3), (0, 1), (2, 1), (3, 1)], (3, 0))
        m.step([(0, 1), (2, 1), (4, 1)], (0, 0))


@pytest.mark.parametrize("page_size,d,cached,new", [
    (24, 64, [58, 58, 0], [1, 1, 149]),
    (12, 128, [452, 569, 227, 264, 441, 597, 902, 216, 696, 552, 900, 850, 540] + [0] * 11,
     [1] * 13 + [116, 53, 199, 169, 229, 158, 124, 87, 257, 186, 89])])
def test_mixed_steps_of_generic_caches_that_are_faster_over_gathered_keys(page_size, d, cached, new):
    """Two steps of 64 query and 8 kv heads that take 106 and 374 us for 6 layers over gathered keys, 132 and 510 with prompts
    and decoding sequences apart."""
    cache = GpuCache([len(new), 12000, 8192, page_size, 0], 1, 64, 8, d, d)
    old = [b for b, n in enumerate(cached) if n]
    for b in range(len(new)):
        cache.add_sequence(b)
    cache.begin_forward(old, [cached[b] for b in old])
    cache.end_forward()
    cache.begin_forward(list(range(len(new))), new)
    assert cache.cache.flags()["plain_route"] == 1
    cache.end_forward()


@pytest.mark.parametrize("dtype,page_size,d,hq,hkv,window", [(np.float16, 16, 64, 8, 2, 0), (np.float16, 16, 128, 16, 1, 0), (np.float16, 32, 64, 3, 3, 50),
                                                            (np.float16, 16, 128, 8, 2, 90), (np.float32, 16, 128, 8, 2, 0), (np.float32, 24, 64, 8, 1, 0),
                                                            (np.float16, 20, 72, 12, 2, 0), (np.float16, 12, 64, 8, 2, 0)])
def test_prompts_and_decoding_sequences_in_one_launch(dtype, page_size, d, hq, hkv, window):
    """Steps whose work of either kind is the shorter one by far, a single item, or no multiple of the eight workgroups that
    are dealt out together: new prompts, whose launch is not split, beside long and short decoding sequences (the generic
    kernels': long ones, whose launch is).  The oracle's results, with the bounds of every step of a Mirror."""
    m = Mirror([16, 5000, 1024, page_size, 0] + ([window] if window else []), 2 if window else 1, hq, hkv, d, dtype=dtype,
               **({"attn_kinds": [3, 0]} if window else {}))
    mixed = (3, 3 if window else 0)
    with step_route(2):
        m.step([(0, 900), (1, 64)], (0, 0))
        m.step([(2, 400), (3, 1)], None)
        for batch in ([(4, 2), (0, 1)],  # an item or two of prompts; one sequence
                      [(0, 1), (5, 33), (2, 1), (6, 257), (1, 1), (7, 19)],
                      [(8, 300), (9, 131), (10, 64), (11, 5), (2, 1)],  # few decoding items
                      [(12, 17), (0, 1), (1, 1), (2, 1), (3, 1), (4, 1), (5, 1), (6, 1), (7, 1), (8, 1), (9, 1)]):
            # the generic kernels: where the new tokens' row tiles are of 32 rows and the cached keys are split
            cached = [-(-m.lengths[b] // page_size) * page_size for b, n in batch if n == 1]
            together = dtype == np.float16 and page_size % 16 == 0 or (
                sum(n for _, n in batch) * (hq // hkv) // len(batch) > 16 and sum(cached) // len(cached) >= 256)
            before = joint_launches()
            m.step(batch, mixed)
            assert joint_launches() - before == (m.layers if together else 0)


@pytest.mark.parametrize("dtype,page_size,d,hq,hkv,window", [(np.float16, 16, 128, 8, 2, 0), (np.float16, 16, 64, 8, 2, 1300), (np.float32, 16, 64, 8, 2, 0)])
def test_mixed_steps_of_more_sequences_than_a_wave_has_lanes(dtype, page_size, d, hq, hkv, window):
    """77 sequences, 70 of them decoding, whose order and work items are looked up in two rounds."""
    m = Mirror([80, 30000, 2600, page_size, 0] + ([window] if window else []), 2 if window else 1, hq, hkv, d, dtype=dtype,
               **({"attn_kinds": [3, 0]} if window else {}))
    with step_route(2):
        for first in range(0, 70, 7):  # a quarter of them short
            m.step([(b, 1 + b * 7 % 23 if b % 4 == 0 else 300 + b) for b in range(first, first + 7)])
        m.step([(3, 900), (66, 300)])
        before = joint_launches()
        m.step([(b, 1) for b in range(40)] + [(70 + i, 61 + 50 * i) for i in range(7)] + [(b, 1) for b in range(40, 70)], (3, 3 if window else 0))
    assert joint_launches() - before == m.layers


@pytest.mark.parametrize("page_size,d,hq,hkv,forks,prefix,joint", [(16, 128, 16, 1, 9, 640, 0), (64, 64, 32, 2, 10, 1100, 0), (16, 128, 8, 2, 41, 385, 0),
                                                                  (32, 64, 4, 4, 130, 256, 0), (16, 128, 40, 2, 8, 640, 0), (16, 128, 16, 1, 33, 1290, 1),
                                                                  (32, 128, 8, 2, 41, 2400, 1), (64, 128, 4, 4, 130, 1100, 1), (16, 64, 4, 4, 130, 4100, 1),
                                                                  (64, 64, 32, 2, 33, 1100, 1), (16, 128, 20, 1, 33, 1100, 0)])
def test_decode_step_over_a_shared_prefix_whose_keys_are_split(page_size, d, hq, hkv, forks, prefix, joint):
    """The sequences' own tokens and the shares of the prefix in one launch (from 32 sequences on, where the prefix is a level of
    its own, and 1024 of its keys on, where they are split; up to 16 query heads a kv head): own parts of one token and of
    several chunks, a sequence that is the prefix itself."""
    m = Mirror([forks + 2, prefix + 1500 + forks * 3 * page_size, 1200, page_size, 0], 1, hq, hkv, d)
    for first in range(0, prefix, 1200):
        m.step([(0, min(1200, prefix - first))])
    before = joint_launches()
    m.step([((b, 0, -1), 1) for b in range(1, forks + 1)])
    assert joint_launches() - before == joint
    m.step([(1, 500)])
    m.step([(b, 1) for b in range(1, forks + 1)])
    before = joint_launches()
    m.step([(b, 1) for b in range(forks, 0, -1)])
    assert joint_launches() - before == joint


@pytest.mark.parametrize("d,hq,hkv,page_size", [(128, 32, 8, 16), (64, 16, 2, 32), (128, 4, 4, 64)])
def test_a_prefix_beside_its_sequences_is_the_same_as_apart_and_under_capture(d, hq, hkv, page_size):
    """One launch and two write the same bits; so does every replay of a graph of the step."""
    forks, prefix = 140, 5000
    cache = GpuCache([forks + 2, 2 * prefix + forks * 900, 8192, page_size, 0], 1, hq, hkv, d, d)
    rng = np.random.default_rng(33)
    qkv = dev(rng.standard_normal((forks * 40, hq + 2 * hkv, d)).astype(np.float16))
    attend = gf("vm.builtin.attention_kv_cache_attention_with_fused_qkv")

    def forward(ids, lens):
        cache.begin_forward(ids, lens)
        attend(cache.cache, 0, d ** -0.5, qkv[:sum(lens)], torch.zeros((sum(lens), hq, d), dtype=torch.float16, device=DEV))
        cache.end_forward()

    cache.add_sequence(0)
    forward([0], [prefix])
    ids = list(range(1, forks + 1))
    for b in ids:
        cache.fork_sequence(0, b)
    forward(ids, [1 + 11 * b % 60 for b in ids])
    forward(ids[:3], [700, 800, 900])
    cache.begin_forward(ids, [1] * forks)
    rows = qkv[-forks:]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    cache.cache.set_stream(stream.cuda_stream)
    out = torch.zeros((forks, hq, d), dtype=torch.float16, device=DEV)
    outs = []
    for apart in (False, True):
        out.zero_()
        torch.cuda.synchronize()
        before = joint_launches()
        with launches_apart() if apart else contextlib.nullcontext():
            attend(cache.cache, 0, d ** -0.5, rows, out)
        assert joint_launches() - before == int(not apart)
        torch.cuda.synchronize()
        outs.append(out.clone())
    assert bool(outs[0].any()) and torch.equal(outs[0], outs[1])
    graph = torch.cuda.CUDAGraph()
    before = joint_launches()
    with torch.cuda.graph(graph, stream=stream):
        attend(cache.cache, 0, d ** -0.5, rows, out)
    assert joint_launches() - before == 1
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, outs[0])
        (rows * 2).sum()  # work of the program's own between the replays


def _exact(rows, cached, starts, mask, heads, kv_heads):
    """Attention in 64 bits of one sequence's new tokens (q, k, v rows) over its cached ones and, under `mask`, the new."""
    q, k, v = rows.double().transpose(0, 1).split([heads, kv_heads, kv_heads])
    _, ck, cv = cached.double().transpose(0, 1).split([heads, kv_heads, kv_heads])
    mask = torch.cat([torch.ones((mask.shape[0], starts), dtype=torch.bool), mask], dim=1).to(DEV)
    out = torch.empty((rows.shape[0], heads, rows.shape[2]), dtype=torch.float64, device=DEV)
    for h in range(heads):
        kv = h // (heads // kv_heads)
        keys, values = torch.cat([ck[kv, :starts], k[kv]]), torch.cat([cv[kv, :starts], v[kv]])
        scores = (q[h] @ keys.T.contiguous() * rows.shape[2] ** -0.5).masked_fill(~mask, -torch.inf)
        out[:, h] = torch.softmax(scores, -1) @ values
    return out


def _fill(cache, qkv, lengths, d):
    """Sequence b holds the first lengths[b] rows of qkv."""
    for b, n in enumerate(lengths):
        cache.add_sequence(b)
        if n:
            cache.begin_forward([b], [n])
            _attend(cache, qkv[:n], d)
            cache.end_forward()


def _tree_step_over_unlike_lengths(d, page_size):
    """A cache (no RoPE) whose next step is a verify step of one round of full row tiles, its longest sequence well above
    the mean; the step's rows and the attention of them in 64 bits."""
    heads, nodes, batch = 32, 66, 9
    cache = GpuCache([batch, 16384, 4600, page_size, 0], 1, heads, heads, d, d, rope_mode=S.ROPE_NONE)
    qkv = dev(np.random.default_rng(12).standard_normal((4600, 3 * heads, d)).astype(np.float16))
    lengths = [4600 if b == 4 else 1200 for b in range(batch)]
    _fill(cache, qkv, lengths, d)
    parents = [(i - 1) // 2 if i else -1 for i in range(nodes)]
    sees = torch.eye(nodes, dtype=torch.bool)
    for i in range(1, nodes):
        sees[i] |= sees[parents[i]]
    cache.begin_forward(list(range(batch)), [nodes] * batch, parents * batch)
    rows = qkv[:batch * nodes].flip(0).contiguous()
    exact = torch.cat([_exact(rows[b * nodes:(b + 1) * nodes], qkv, n, sees, heads, heads) for b, n in enumerate(lengths)])
    return cache, rows, exact


def _attend(cache, rows, d):
    out = torch.zeros((rows.shape[0], cache.hq, d), dtype=torch.float16, device=DEV)
    gf("vm.builtin.attention_kv_cache_attention_with_fused_qkv")(cache.cache, 0, d ** -0.5, rows, out)
    return out


def _errors_split_and_whole(cache, rows, exact, d, first=0):
    """Distances from the 64-bit result with the derived split of the keys and without one; they have to differ."""
    outs = []
    for splits in (0, 1):
        prev = tvm_amd.set_option("prefill_kv_splits", splits)
        try:
            outs.append(_attend(cache, rows, d)[first:])
        finally:
            tvm_amd.set_option("prefill_kv_splits", prev)
        assert_close(host(outs[-1]), host(exact.float()), what="split" if splits == 0 else "whole")
    assert not torch.equal(outs[0], outs[1]), "the step did not split"
    return [float((o.double() - exact).norm()) for o in outs]


@pytest.mark.parametrize("d,page_size", [(128, 16), (64, 16), (64, 64)])
def test_tree_steps_over_sequences_of_unlike_lengths(d, page_size):
    """Such a step walks its keys in two shares, whose states are float32: it is as far from the attention in 64 bits as
    the unsplit launch (the same roundings in another order: over two million values the means agree to far below the 2 %
    that are allowed; fp16 shares would be 22 % further off)."""
    cache, rows, exact = _tree_step_over_unlike_lengths(d, page_size)
    split, whole = _errors_split_and_whole(cache, rows, exact, d)
    assert split <= 1.02 * whole


@pytest.mark.parametrize("d", [128, 64])
def test_prompts_of_mixed_steps_lose_no_precision_when_their_keys_are_split(d):
    """Two short chunks behind long cached prompts beside many decoding sequences: a launch of all of them would not split,
    the prompts' own does, with float32 states (fp16 ones: 21 % further off; the bound as above, over half a million values)."""
    heads, kv_heads, new = 32, 8, 64
    lengths = [5000, 4000] + [8000] + [50 + 7 * b for b in range(37)]
    cache = GpuCache([40, 24576, 8000, 16, 0], 1, heads, kv_heads, d, d, rope_mode=S.ROPE_NONE)
    qkv = dev(np.random.default_rng(13).standard_normal((8000, heads + 2 * kv_heads, d)).astype(np.float16))
    _fill(cache, qkv, lengths, d)
    cache.begin_forward(list(range(2, 40)) + [0, 1], [1] * 38 + [new, new])
    rows = qkv[:38 + 2 * new].flip(0).contiguous()
    causal = torch.ones((new, new), dtype=torch.bool).tril()
    exact = torch.cat([_exact(rows[38 + b * new:38 + (b + 1) * new], qkv, lengths[b], causal, heads, kv_heads) for b in range(2)])
    split, whole = _errors_split_and_whole(cache, rows, exact, d, first=38)
    assert split <= 1.02 * whole


def test_captured_tree_step_needs_no_scratch_memory():
    """Under capture the same step runs unsplit: the two shares need scratch memory that a stream without any cannot get
    there."""
    d = 128
    cache, rows, _ = _tree_step_over_unlike_lengths(d, 16)
    eager = _attend(cache, rows, d)
    prev = tvm_amd.set_option("prefill_kv_splits", 1)
    try:
        whole = _attend(cache, rows, d)
    finally:
        tvm_amd.set_option("prefill_kv_splits", prev)
    out = torch.zeros_like(whole)
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    cache.cache.set_stream(stream.cuda_stream)
    with torch.cuda.graph(graph, stream=stream):
        gf("vm.builtin.attention_kv_cache_attention_with_fused_qkv")(cache.cache, 0, d ** -0.5, rows, out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, whole) and not torch.equal(out, eager)
        (rows * 2).sum()  # work of the program's own between the replays


@pytest.mark.parametrize("kinds,dtype", [([0], np.float16), ([3], np.float16), ([0], np.float32)])
def test_a_mixed_step_can_be_captured_once_it_has_run(kinds, dtype):
    """Under capture the general launches run; their scratch memory is there when the step has run eagerly on that stream."""
    d, hq, hkv, lengths, new = 128, 8, 2, [3000, 2500], [1, 40]
    config = [2, 8192, 3000, 16, 0] + ([4096] if 3 in kinds else [])
    qkv = dev(np.random.default_rng(14).standard_normal((3000, hq + 2 * hkv, d)).astype(dtype))
    attend = gf("vm.builtin.attention_kv_cache_attention_with_fused_qkv")
    outs = []
    for route in (1, 2):
        cache = GpuCache(config, 1, hq, hkv, d, d, attn_kinds=kinds, dtype=dtype)
        for b, n in enumerate(lengths):
            cache.add_sequence(b)
            cache.begin_forward([b], [n])
            attend(cache.cache, 0, d ** -0.5, qkv[:n], torch.zeros((n, hq, d), dtype=qkv.dtype, device=DEV))
            cache.end_forward()
        with step_route(route):
            cache.begin_forward([0, 1], new)
        out = torch.zeros((sum(new), hq, d), dtype=qkv.dtype, device=DEV)
        torch.cuda.synchronize()
        stream = torch.cuda.Stream()
        cache.cache.set_stream(stream.cuda_stream)
        attend(cache.cache, 0, d ** -0.5, qkv[:sum(new)], out)
        torch.cuda.synchronize()
        outs.append(out.clone())
    assert not torch.equal(outs[0], outs[1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        attend(cache.cache, 0, d ** -0.5, qkv[:sum(new)], out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, outs[0])
        (outs[1] * 2).sum()


def test_decode_steps_of_windowed_caches_at_the_edges():
    """A decode step of a sequence-window cache takes the new token as one more key: sequences without cached tokens, of
    one token, at the edge of a page and beyond their window, with a prompt's first decode among them; small prefill steps
    of such a cache as well."""
    for d, hq, hkv, rope_mode in ((128, 8, 2, 2), (64, 20, 1, 2), (256, 4, 2, 2), (128, 4, 4, 0)):
        layers = 2
        # the pool is what an earlier cache of the same size left: NaN in every slot
        used = GpuCache([8, 4096, 1024, 16, 1], layers, hq, hkv, d, d, rope_mode=rope_mode)
        for sid in range(4):
            used.add_sequence(sid)
        for _ in range(4):
            used.begin_forward([0, 1, 2, 3], [255] * 4)
            for layer in range(layers):
                used.attention_with_fused_qkv(layer, 1.0, np.full((1020, hq + 2 * hkv, d), np.nan, np.float16),
                                              np.zeros((1020, hq, d), np.float16))
            used.end_forward()
        del used
        cache = GpuCache([8, 4096, 1024, 16, 1], layers, hq, hkv, d, d, rope_mode=rope_mode)
        sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=rope_mode, seed=9, tol=4e-3)
        for sid, (window, sink) in enumerate([(40, 0), (130, 4), (257, 30), (600, 16)]):
            sc.add_with_window(sid, window, sink)
        sc.step([(0, 1), (1, 1), (2, 1)])
        sc.step([(0, 1), (1, 1), (2, 1), (3, 1)])
        # (a chunk longer than its window leaves slots behind the sinks that nothing ever writes)
        sc.step([(0, 14), (1, 29), (2, 300), (3, 500)])
        for _ in range(3):
            sc.step([(0, 1), (1, 1), (2, 1), (3, 1)])
        # a few tokens, and a short chunk beside decoding sequences, by the launches that read the pages themselves
        with step_route(1):
            sc.step([(0, 2), (1, 3), (2, 1), (3, 2)])
            sc.step([(0, 1), (1, 5), (2, 1), (3, 1)])
        sc.step([(0, 1), (1, 1), (2, 1), (3, 1)])


def test_short_chunk_against_a_long_cached_sequence():
    """A chunk of a few tokens against thousands of cached ones is one or two row tiles per kv head: the
    launch splits their keys over several workgroups and merges the states.  Through the cache's one-pass
    chunked prefill and its mixed prefill / decode batches, against the oracle cache."""
    m = Mirror([4, 8192, 2048, 16, 0], 2, 8, 2, 64)
    m.step([(0, 2000), (1, 40)])
    m.step([(0, 1500)])
    m.step([(0, 20), (1, 3)])       # 3520 cached tokens, 20 new ones
    m.step([(0, 1), (1, 2)])        # not a pure decode batch: the prefill kernels again
    m.step([((2, 0, 3000), 7)])     # a fork deep inside the long sequence


@pytest.mark.parametrize("rope", [
    dict(rope_theta=5e5, rope_scaling={"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                                       "original_max_position_embeddings": 8192}),
    dict(rope_scaling={"rope_type": "yarn", "factor": 40.0, "beta_fast": 32, "beta_slow": 1,
                       "original_max_position_embeddings": 4096}),
    dict(rope_scaling={"rope_type": "default", "rotary_dim": 32}),
    dict(rope_scaling={"rope_type": "gptj", "rotary_dim": 64}),
    dict(rope_scaling={"rope_type": "longrope", "max_position_embeddings": 131072, "original_max_position_embeddings": 64},
         rope_ext_factors=np.concatenate([np.linspace(1.0, 8.0, 64), np.linspace(1.0, 1.3, 64)]).astype(np.float32)),
])
def test_rope_frequency_variants_through_the_cache(rope):
    """The model's RoPE variant (what the reference compiles into the split-rotary kernel it hands to the
    cache): prefill, decode and a fork, cached K compared with the oracle cache that rotates the same way.
    The longrope steps have fewer and more rows than original_max_position_embeddings (short / long factors)."""
    m = Mirror([8, 2048, 512, 16, 0], 1, 32, 8, 128, **rope)
    m.step([(0, 60), (1, 88), (2, 17)])   # 165 rows
    m.step([(0, 1), (1, 1), (2, 1)])      # 3 rows
    m.step([((3, 1, 40), 25), (0, 2)])


@pytest.mark.parametrize("rope", [
    dict(rope_theta=5e5, rope_scaling={"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                                       "original_max_position_embeddings": 8192}),
    dict(rope_scaling={"rope_type": "yarn", "factor": 40.0, "beta_fast": 32, "beta_slow": 1,
                       "original_max_position_embeddings": 4096}),
    dict(rope_scaling={"rope_type": "longrope", "max_position_embeddings": 131072, "original_max_position_embeddings": 4096}),
    dict(rope_scaling={"rope_type": "llama4", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                       "original_max_position_embeddings": 8192}),
], ids=lambda r: r["rope_scaling"]["rope_type"])
@pytest.mark.parametrize("sliding", [0, 1])
def test_rope_frequency_variants_in_a_cache_that_rotates_inside_the_attention_kernels(rope, sliding):
    """Inline-RoPE caches (rope mode 2; a sliding-window cache is always one): K is stored unrotated, and every
    attention kernel rotates q and k itself with the model's frequency variant -- prefill (ragged + paged +
    merge), decode and a fork with two block depths, against the oracle cache with the same variant in force."""
    m = Mirror([8, 2048, 512, 16, sliding], 1, 8, 2, 128, rope_mode=2, **rope)
    m.step([(0, 60), (1, 88), (2, 17)])
    m.step([(0, 1), (1, 1), (2, 1)])
    m.step([((3, 1, 40), 25), (0, 2)])
    m.step([(3, 1), (1, 1)])


def test_cfg1_decode_through_the_cache_verbs():
    """BASELINE configs[0] end to end: 1024-page pool, contexts 512/1024/1500/2048 prefilled through
    the real verbs, then one decode step; page table as derived by hand from the reference."""
    m = Mirror([32, 16368, 8192, 16, 0], 1, 32, 8, 128)
    m.step([(0, 512), (1, 1024), (2, 1500), (3, 2048)])
    m.step([(0, 1), (1, 1), (2, 1), (3, 1)])
    c = m.g.cache
    assert c.aux("page_indptr") == [0, 33, 98, 192, 321]
    assert c.aux("append_position_map") == [5088, 5104, 3036, 5120]
    assert c.aux("last_page_len") == [1, 1, 13, 1]
    assert c.aux("q_rope_position_map") == [512, 1024, 1500, 2048]
    assert gf("vm.builtin.attention_kv_cache_get_num_available_pages")(c) == 703


def test_error_paths_on_the_device_cache():
    cache = GpuCache([4, 64, 32, 16, 0], 1, 8, 2, 128, 128)
    c = cache.cache
    cache.add_sequence(0)
    qkv = torch.zeros((4, 12, 128), dtype=torch.float16, device=DEV)
    out = torch.zeros((4, 8, 128), dtype=torch.float16, device=DEV)
    attn = gf("vm.builtin.attention_kv_cache_attention_with_fused_qkv")
    with pytest.raises(tvm_amd.KVError, match="begin_forward has not been called"):
        attn(c, 0, 1.0, qkv, out)
    cache.begin_forward([0], [8])
    with pytest.raises(tvm_amd.KVError, match="fewer than the batch appends"):
        attn(c, 0, 1.0, qkv, out)
    with pytest.raises(tvm_amd.KVError, match="out of range"):
        attn(c, 3, 1.0, torch.zeros((8, 12, 128), dtype=torch.float16, device=DEV),
             torch.zeros((8, 8, 128), dtype=torch.float16, device=DEV))
    cache.add_sequence(1)
    with pytest.raises(tvm_amd.KVError, match="The KV cache is full"):
        cache.begin_forward([1], [80])
    # a kernel's refusal surfaces through the cache call: head_dim 68 is not built (the generic kernels take
    # multiples of 8)
    c2 = GpuCache([4, 64, 32, 16, 0], 1, 8, 2, 68, 68, rope_mode=0)
    c2.add_sequence(0)
    qkv96 = torch.zeros((1, 12, 68), dtype=torch.float16, device=DEV)
    out96 = torch.zeros((1, 8, 68), dtype=torch.float16, device=DEV)
    c2.begin_forward([0], [1])
    with pytest.raises(tvm_amd.KVError, match="is not built"):
        attn(c2.cache, 0, 1.0, qkv96, out96)


@pytest.mark.parametrize("runner", [S.run_sliding_window, S.run_sliding_window_fork, S.run_sliding_window_page_reuse])
def test_sliding_window_scenarios_on_the_gpu(runner):
    """The reference's sliding-window tests (attention sinks, window trimming after every step,
    forks inside the sink; tests/python/relax/test_runtime_builtin_paged_attention_kv_cache_cpu.py:912-1022)
    on the HIP cache: inline RoPE, length_info (3, B), prefill and decode kernels."""
    layers, hq, hkv, d = 2, 8, 2, 128
    cache = GpuCache([32, 2048, 512, 16, 1], layers, hq, hkv, d, d, rope_mode=S.ROPE_INLINE)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=S.ROPE_INLINE, seed=4)
    runner(sc)


@pytest.mark.parametrize("d,rope_mode", [(128, S.ROPE_NORMAL), (64, S.ROPE_NORMAL), (128, S.ROPE_NONE)])
def test_token_tree_scenario_on_the_gpu(d, rope_mode):
    """test_paged_attention_kv_cache_tree_attn of the reference
    (tests/python/relax/test_runtime_builtin_paged_attention_kv_cache_tir.py:1053-1134): tree attention
    over new tokens and over appended tree nodes, commit with the compaction copy, decode after it."""
    layers, hq, hkv = 2, 32, 4
    cache = GpuCache([32, 2048, 512, 16, 0], layers, hq, hkv, d, d, rope_mode=rope_mode)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=rope_mode, seed=8, tol=4e-3)
    S.run_tree_attn(sc)


def test_padded_qkv_rows_are_ignored():
    """qkv / out may carry more rows than the batch appends (src/runtime/vm/paged_kv_cache.cc:1330-1354)."""
    layers, hq, hkv, d = 1, 8, 2, 128
    a = GpuCache([4, 256, 64, 16, 0], layers, hq, hkv, d, d)
    b = GpuCache([4, 256, 64, 16, 0], layers, hq, hkv, d, d)
    rng = np.random.default_rng(3)
    qkv = rng.standard_normal((10, hq + 2 * hkv, d)).astype(np.float16)
    for cache in (a, b):
        cache.add_sequence(0)
        cache.begin_forward([0], [10])
    o_exact = np.zeros((10, hq, d), np.float16)
    a.attention_with_fused_qkv(0, d ** -0.5, qkv, o_exact)
    padded = np.concatenate([qkv, np.full((6, hq + 2 * hkv, d), np.nan, np.float16)])
    o_pad = np.full((16, hq, d), 3.0, np.float16)
    b.attention_with_fused_qkv(0, d ** -0.5, padded, o_pad)
    assert np.array_equal(o_pad[:10], o_exact)


def test_attention_with_shared_kv_reads_the_source_layer():
    """vm.builtin.attention_kv_cache_attention_with_shared_kv (src/runtime/vm/kv_state.cc:97-105,
    paged_kv_cache.cc:1487-1525): a second set of queries attends to the K/V that layer 0 caches plus
    the step's own rows, nothing is appended.  Prefill (self + cross), a second chunk, then decode;
    checked against the oracle cache and against the closed form over layer 0's K/V."""
    from oracle import closed_form as cf
    layers, hq, hkv, d = 2, 8, 2, 128
    cfg = [4, 512, 128, 16, 0]
    gpu = GpuCache(cfg, layers, hq, hkv, d, d, rope_mode=S.ROPE_NONE)
    cpu = OraclePagedKVCache(cfg, layers, hq, hkv, d, d, rope_mode=S.ROPE_NONE)
    rng = np.random.default_rng(17)
    cached_k = {0: np.zeros((0, hkv, d), np.float16), 1: np.zeros((0, hkv, d), np.float16)}
    cached_v = {0: np.zeros((0, hkv, d), np.float16), 1: np.zeros((0, hkv, d), np.float16)}
    for cache in (gpu, cpu):
        cache.add_sequence(0)
        cache.add_sequence(1)
    for lens in ([40, 23], [9, 30], [1, 1], [1, 1]):
        total = sum(lens)
        qkv = rng.standard_normal((total, hq + 2 * hkv, d)).astype(np.float16)
        q2 = rng.standard_normal((total, hq, d)).astype(np.float16)
        k_cur = np.ascontiguousarray(qkv[:, hq:hq + hkv])
        v_cur = np.ascontiguousarray(qkv[:, hq + hkv:])
        outs = []
        for cache in (gpu, cpu):
            cache.begin_forward([0, 1], lens)
            o1 = np.zeros((total, hq, d), np.float16)
            cache.attention_with_fused_qkv(0, d ** -0.5, qkv, o1)
            o2 = np.zeros((total, hq, d), np.float16)
            cache.attention_with_shared_kv(0, d ** -0.5, q2, k_cur, v_cur, o2)
            cache.end_forward()
            outs.append(o2)
        assert_close(outs[0], outs[1], what=f"shared-kv attention vs oracle cache, step {lens}")
        cursor = 0
        for sid, n in enumerate(lens):
            cached_k[sid] = np.concatenate([cached_k[sid], k_cur[cursor:cursor + n]])
            cached_v[sid] = np.concatenate([cached_v[sid], v_cur[cursor:cursor + n]])
            expected, _ = cf.attention(q2[cursor:cursor + n], cached_k[sid], cached_v[sid], d ** -0.5, causal=True)
            assert_close(outs[0][cursor:cursor + n], expected, atol=4e-3, rtol=4e-3,
                         what=f"shared-kv attention vs closed form, seq {sid}")
            cursor += n
    # layer 1 never received anything
    with pytest.raises(tvm_amd.KVError, match="rows"):
        gf("vm.builtin.attention_kv_cache_attention_with_shared_kv")(
            gpu.cache, 0, 1.0, torch.zeros((5, hq, d), dtype=torch.float16, device=DEV),
            torch.zeros((5, hkv, d), dtype=torch.float16, device=DEV),
            torch.zeros((5, hkv, d), dtype=torch.float16, device=DEV),
            torch.zeros((5, hq, d), dtype=torch.float16, device=DEV))


@pytest.mark.parametrize("runner,rope_mode,sliding", [(S.run_fork_sequence, S.ROPE_NORMAL, 0), (S.run_tree_attn, S.ROPE_NORMAL, 0),
                                                      (S.run_sliding_window_fork, S.ROPE_INLINE, 1),
                                                      (S.run_sliding_window_page_reuse, S.ROPE_INLINE, 1)])
def test_reference_scenarios_with_pages_of_32_tokens(runner, rope_mode, sliding):
    """The reference's scenarios on a cache whose pages hold 32 tokens (the kernels walk such pages as
    two runs of 16): forks inside a page, token trees with their commit, sliding windows."""
    layers, hq, hkv, d = 2, 8, 2, 128
    cache = GpuCache([32, 2048, 512, 32, sliding], layers, hq, hkv, d, d, rope_mode=rope_mode)
    sc = S.Scenario(cache, layers, hq, hkv, d, rope_mode=rope_mode, seed=9, tol=4e-3)
    runner(sc)
