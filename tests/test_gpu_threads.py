"""Attention calls of several threads on one stream share its workspace: their launches may not
interleave (a call whose global tiles are split launches the attention and then the merge of its chunks)."""

import threading

import pytest
import torch

from tests.helpers import device_paired, oracle_paired, oracle_plan, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["paired", "sparse"])
def test_one_stream(hip_device, entry):
    from hilberta_amd.paired_kernel import paired_attention
    from hilberta_amd.sparse_kernel import sparse_attention

    plan = oracle_plan("1024_t16k3")
    meta = device_paired(oracle_paired(plan, 1), hip_device)
    p = plan["phases"][1]
    ids, counts = (torch.from_numpy(p[f]).to(hip_device) for f in ("kv_indices", "kv_counts"))
    gen = torch.Generator(hip_device).manual_seed(3)
    inputs = [[torch.randn(1, 4, plan["total_tokens"], 128, device=hip_device, generator=gen).to(torch.bfloat16)
               for _ in range(3)] for _ in range(3)]

    def call(qkv):
        if entry == "paired":
            return paired_attention(*qkv, meta)
        return sparse_attention(*qkv, ids, counts, global_tokens=plan["global_tokens"])

    alone = [call(qkv) for qkv in inputs]
    torch.cuda.synchronize()
    outs, start = [[] for _ in inputs], threading.Barrier(len(inputs))

    def work(i):
        start.wait()
        with torch.no_grad():
            outs[i] += [call(inputs[i]) for _ in range(60)]

    say(f"case three threads on one stream, {entry}")
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(inputs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for got, ref in zip(outs, alone):
        assert len(got) == 60 and all(torch.equal(o, ref) for o in got)
