"""The matrix prefill's GEMM tiles, splits of K and row kernels at the sizes where they can go wrong:
prompts just past and short of tile edges (64, 128, 256 rows), FFN widths of an odd number of 32s (the
32-wide K steps) and of less than a tile of columns, and products that split K up to 8 ways.

Against the oracle's full causal block, over a stack of 2 layers: layer 1's K and V rows depend on all
of layer 0.  Bars: layer 0's rows within 1 bf16 ulp of the oracle's in 99.9% of elements; layer 1's
with an RMS difference of at most 2^-7 of their RMS.  A bf16 rounding moves a value by up to 2^-9 of
it; about 8 of them lie between the embedding and layer 1's rows, independent ones add to
sqrt(8) 2^-9 = 0.0055.  A wrong tile, row or part of a sum moves the rows by their own size."""

import numpy as np
import pytest
import torch

from oracle import decoder as ref
from tests.test_gpu_prefill import bf16_ulps, kv_rows, oracle_kv_and_logits
from tiles_amd import runtime as R
from tiles_amd.tileplan import package as K
from tiles_amd.tileplan import plan as P
from tiles_amd.tileplan import probe

pytestmark = pytest.mark.gpu


def check(tmp_path, hidden, intermediate, heads, kv_heads, length, std):
    dims = dict(hidden_size=hidden, intermediate_size=intermediate, num_attention_heads=heads, num_key_value_heads=kv_heads,
                head_dim=hidden // heads, max_context=length + 8)
    spec = P.StackSpec(P.BlockSpec(**dims), 2, 512, True)
    path = tmp_path / "pkg"
    K.build_stack_package(spec, K.random_weights(spec, seed=7 + length, std=std), probe.probe_library(), path, "bfloat16")
    packed = K.read_weights(path, spec, "bfloat16")
    width = kv_heads * (hidden // heads)
    prompt = np.random.default_rng(length).integers(0, 512, length).tolist()
    ctx = R.DecoderModel(R.load_plan(path)).create_context()
    snapshot = ctx.collect(ctx.enqueue_prefill(prompt, kv=True))["kv"]
    got = kv_rows(snapshot, K.read_plan(path), 2, length, width)
    want, _ = oracle_kv_and_logits(prompt, packed, ref.Spec(**dims, layers=2, vocab_size=512), 2, width)
    for i, name in enumerate("KV"):
        ulps = bf16_ulps(got[0][i], want[0][i])
        assert float((ulps <= 1).mean()) >= 0.999, name
        rms = lambda a: float(np.sqrt((a.astype(np.float64) ** 2).mean()))  # noqa: E731
        off = rms(got[1][i] - want[1][i]) / rms(want[1][i])
        print(f"{hidden}/{intermediate}, {length} tokens, {name}: layer 0 equal {float((ulps == 0).mean()):.4f}, "
              f"layer 1 off by {off:.5f} of its RMS", flush=True)
        assert off <= 2.0 ** -7, name


@pytest.mark.parametrize("hidden,intermediate,heads,kv_heads,length,std", [
    (256, 512, 4, 1, 3, 0.08),        # the shortest prompt that is prefilled with matrices
    (2048, 8192, 32, 8, 17, 0.02),    # 16 rows
    (256, 544, 4, 1, 65, 0.08),       # 64 rows; down projection over 544 = 17 x 32
    (256, 544, 4, 1, 66, 0.08),       # 65 rows
    (128, 32, 2, 1, 129, 0.12),       # 128 rows; gate/up and down narrower than any tile
    (256, 512, 4, 2, 130, 0.08),      # 129 rows
    (512, 1056, 8, 2, 257, 0.05),     # 256 rows; 33 x 32
    (2048, 8192, 32, 8, 71, 0.02),    # 64-row tiles, K split up to 8 ways
    (2048, 8192, 32, 8, 514, 0.02),   # 128-row tiles, K split
])
def test_matrix_prefill_at_tile_edges(tmp_path, hidden, intermediate, heads, kv_heads, length, std):
    check(tmp_path, hidden, intermediate, heads, kv_heads, length, std)


@pytest.mark.parametrize("hidden,intermediate,heads,kv_heads,length,std", [
    (1024, 256, 16, 16, 1090, 0.03),  # one query head a K/V head; 2 heads and 32 rows a block
    (2048, 256, 32, 16, 2120, 0.02),  # two; 4 heads and 64 rows a block, a last block of 7 rows
    (512, 256, 4, 1, 300, 0.05),      # head_dim 128
    (1024, 256, 8, 4, 90, 0.03),      # head_dim 128, two query heads a K/V head
])
def test_matrix_prefill_attention_forms(tmp_path, hidden, intermediate, heads, kv_heads, length, std):
    """The attention's heads per wave (as many as leave two blocks a CU), query groups smaller than a
    wave takes, and both head widths."""
    check(tmp_path, hidden, intermediate, heads, kv_heads, length, std)


def test_prompt_in_many_parts_then_generation(tmp_path):
    """60 prompts of 4 to 7 tokens queued on one context (each ends with a launch of the logits tasks
    alone, which takes one step's exchange epochs), then 70 generated tokens (two launches), beside a
    context whose every token goes through the worker.  The logits of both after the same 330 + 70
    tokens are within 2^-6 of their RMS: 2 layers' roundings (2^-7, above) on either side."""
    dims = dict(hidden_size=256, intermediate_size=512, num_attention_heads=4, num_key_value_heads=1, head_dim=64, max_context=420)
    spec = P.StackSpec(P.BlockSpec(**dims), 2, 512, True)
    K.build_stack_package(spec, K.random_weights(spec, seed=5, std=0.08), probe.probe_library(), tmp_path / "pkg", "bfloat16")
    model = R.DecoderModel(R.load_plan(tmp_path / "pkg"))
    parts = [np.random.default_rng(i).integers(0, 512, 4 + i % 4).tolist() for i in range(60)]
    matrix, worker = model.create_context(), model.create_context()
    worker.set_matrix_prefill(False)
    tickets = [matrix.enqueue_prefill(p, logits=True) for p in parts]
    last = matrix.collect(tickets[-1])["logits"]
    generated = matrix.wait(matrix.enqueue_generate(70)).generated
    after = matrix.collect(matrix.enqueue_decode(generated[0], logits=True))["logits"]
    for p in parts[:-1]:
        worker.enqueue_prefill(p)
    want = worker.collect(worker.enqueue_prefill(parts[-1], logits=True))["logits"]
    assert np.argmax(last) == generated[0] and len(generated) == 70
    for first in range(0, 70, 64):  # the same tokens, forced
        worker.enqueue_prefill(generated[first:first + 64])
    want_after = worker.collect(worker.enqueue_decode(generated[0], logits=True))["logits"]
    for got, expected in ((last, want), (after, want_after)):
        off = float(np.sqrt(((got - expected) ** 2).mean() / (expected ** 2).mean()))
        print(f"off by {off:.5f} of the RMS", flush=True)
        assert off <= 2.0 ** -6


def test_short_prompts_hold_small_buffers(tmp_path):
    """A context of prompts up to 64 tokens holds buffers for 64 rows (here 1.6 MB; the bar leaves room
    for the allocator's granularity, the long ones take 64 MiB and more), and its rows and logits are
    bit-equal to those of a context that has taken the long ones."""
    dims = dict(hidden_size=256, intermediate_size=512, num_attention_heads=4, num_key_value_heads=1, head_dim=64, max_context=160)
    spec = P.StackSpec(P.BlockSpec(**dims), 2, 512, True)
    K.build_stack_package(spec, K.random_weights(spec, seed=3, std=0.08), probe.probe_library(), tmp_path / "pkg", "bfloat16")
    model = R.DecoderModel(R.load_plan(tmp_path / "pkg"))
    fresh, used = model.create_context(), model.create_context()
    prompt = np.random.default_rng(1).integers(0, 512, 64).tolist()
    used.wait(used.enqueue_prefill(prompt + prompt[:40]))
    used.wait(used.enqueue_reset())
    fresh.wait(fresh.enqueue_decode(1))  # the code of a first launch is loaded
    fresh.wait(fresh.enqueue_reset())
    free = torch.cuda.mem_get_info()[0]
    got = fresh.collect(fresh.enqueue_prefill(prompt, logits=True, kv=True))
    held = free - torch.cuda.mem_get_info()[0]
    want = used.collect(used.enqueue_prefill(prompt, logits=True, kv=True))
    assert held <= 16 << 20, held
    assert np.array_equal(got["kv"], want["kv"]) and np.array_equal(got["logits"], want["logits"])
    for ctx in (fresh, used):
        ctx.wait(ctx.enqueue_reset())
    got, want = (c.collect(c.enqueue_prefill(prompt + prompt[:40], logits=True))["logits"] for c in (fresh, used))
    assert np.array_equal(got, want)
