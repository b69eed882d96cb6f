"""CPU tier: the package's functions over registered ops are traced and exported with tensors that have no
memory (fake CUDA tensors), so that nothing outside an op may ask for a pointer."""
import pytest
import torch

from torch._subclasses.fake_tensor import FakeTensorMode


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _calls():
    from smla import compressor, indexer, mla, sparse_attn
    bf = torch.bfloat16
    pair = compressor.project_pair
    yield "pair_fp32", pair, lambda: (_empty(2, 40, 512), _empty(256, 512), _empty(256, 512)), ["linear_pair"]
    yield "pair_bf16", pair, lambda: (_empty(1, 5, 512, dtype=bf), *(_empty(256, 512, dtype=bf) for _ in "ab")), ["linear_pair"]
    yield "pair_mixed", pair, lambda: (_empty(2, 9, 512, dtype=bf), _empty(256, 512), _empty(96, 512)), ["linear"]
    yield ("compressor_prefill", lambda *a: compressor.compressor_prefill(*a)[0],
           lambda: (_empty(1, 40, 512), _empty(1024, 512), _empty(1024, 512), _empty(4, 1024), _empty(512)),
           ["linear_pair", "gated_pool"])
    yield "linear", mla.linear, lambda: (_empty(2, 40, 512), _empty(256, 512)), ["linear"]
    yield ("o_project", mla.o_project,
           lambda: (_empty(40, 64, 512, dtype=bf), torch.zeros(40, dtype=torch.int32, device="cuda"), _empty(64, 32),
                    _empty(64, 32), _empty(8192, 4096, dtype=bf), _empty(4096, 8192, dtype=bf)), ["o_proj"])
    yield ("prefill_attn", lambda q, r, c, s: sparse_attn.prefill_attn(q, r, c, s, 0.04),
           lambda: (_empty(1, 40, 64, 576, dtype=bf), _empty(1, 40, 576, dtype=bf), _empty(1, 10, 576, dtype=bf), _empty(64)),
           ["prefill_attn"])
    yield ("index", lambda q, k, w: indexer.topk(indexer.indexer_score(q, k, None, w), 16),
           lambda: (_empty(1, 4, 64, 128, dtype=bf), _empty(1, 100, 128, dtype=bf), _empty(1, 4, 64)),
           ["indexer_score", "topk"])


@pytest.mark.parametrize("strict", [False, True])
@pytest.mark.parametrize("name,fn,args,ops", list(_calls()), ids=lambda v: v if isinstance(v, str) else "")
def test_exports_as_its_ops(name, fn, args, ops, strict):
    class Call(torch.nn.Module):
        def forward(self, *a):
            return fn(*a)

    with FakeTensorMode(allow_non_fake_inputs=True):
        a = args()
    program = torch.export.export(Call(), a, strict=strict)
    names = [str(n.target) for n in program.graph.nodes if n.op == "call_function" and "smla" in str(n.target)]
    assert names == [f"smla.{op}.default" for op in ops]
