"""The native form of the decode call: the results of the general way, which it leaves everything to that is not plain."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from infer_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture
def call(gpu, monkeypatch):
    assert ops._decode_call is not None
    gen = torch.Generator().manual_seed(0)
    k, v = (torch.randn(9, 64, 2, 128, generator=gen).to(BF16).cuda() for _ in range(2))
    args = {"q": torch.randn(3, 1, 8, 128, generator=gen).to(BF16).cuda(), "k_cache": k, "v_cache": v,
            "cache_seqlens": torch.tensor([5, 100, 192], dtype=torch.int32).cuda(), "block_table": torch.arange(9, dtype=torch.int32).view(3, 3).cuda()}
    ops.flash_attn_with_kvcache(**args)                    # the first call claims the workspace for the stream
    taken = []
    inner = ops._decode_call.decode

    class Counted:
        claim = staticmethod(ops._decode_call.claim)

        @staticmethod
        def decode(*a):
            out = inner(*a)
            taken.append(out is not None)
            return out
    monkeypatch.setattr(ops, "_decode_call", Counted)
    general = torch.empty_like(args["q"][:, 0])
    ops.paged_attn_decode(args["q"][:, 0], k, v, args["block_table"], args["cache_seqlens"], 128 ** -0.5, general)
    return args, taken, general.unsqueeze(1)


def test_a_plain_call_is_taken_and_gives_the_same_bits(call):
    args, taken, want = call
    for scale in (None, 128 ** -0.5):
        got = ops.flash_attn_with_kvcache(**args, softmax_scale=scale)
        assert taken.pop() and torch.equal(got, want) and got.shape == want.shape and got.stride() == want.stride() and not got.requires_grad
    wide = torch.zeros(3, 1, 10, 128, dtype=BF16, device="cuda")
    wide[:, :, 1:9] = args["q"]
    got = ops.flash_attn_with_kvcache(**{**args, "q": wide[:, :, 1:9]})
    assert taken.pop() and torch.equal(got, want)


class Sub(torch.Tensor):
    pass


class Watch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_what_is_not_plain_goes_the_general_way(call):
    args, taken, want = call
    assert torch.equal(ops.flash_attn_with_kvcache(**{**args, "q": args["q"].as_subclass(Sub)}).as_subclass(torch.Tensor), want) and not taken.pop()
    with Watch():
        assert torch.equal(ops.flash_attn_with_kvcache(**args), want) and not taken.pop()
    uniform = ops.flash_attn_with_kvcache(**{**args, "cache_seqlens": 64})
    assert uniform.shape == want.shape and not taken.pop()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        got = ops.flash_attn_with_kvcache(**args)          # claims the workspace for this stream
        assert not taken.pop()
        again = ops.flash_attn_with_kvcache(**args)
        assert taken.pop()
    side.synchronize()
    assert torch.equal(got, want) and torch.equal(again, want)
    assert torch.equal(ops.flash_attn_with_kvcache(**args), want) and not taken.pop()


def test_another_stream_is_refused_while_the_last_call_may_run(call):
    args, taken, want = call
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda._sleep(200_000_000)
    ops.flash_attn_with_kvcache(**args)
    with torch.cuda.stream(side), pytest.raises(RuntimeError, match="another stream"):
        ops.flash_attn_with_kvcache(**args)
    torch.cuda.synchronize()


@pytest.mark.parametrize("wrong", [
    {"q": torch.zeros(3, 2, 8, 128, dtype=BF16)}, {"q": torch.zeros(3, 1, 8, 128)}, {"q": torch.zeros(3, 1, 7, 128, dtype=BF16)},
    {"q": torch.zeros(3, 1, 8, 64, dtype=BF16)}, {"cache_seqlens": torch.zeros(3, dtype=torch.int64)}, {"cache_seqlens": torch.zeros(2, dtype=torch.int32)},
    {"block_table": torch.zeros(3, 0, dtype=torch.int32)}, {"block_table": torch.zeros(2, 3, dtype=torch.int32)}, {"v_cache": torch.zeros(9, 64, 1, 128, dtype=BF16)},
    {"block_table": "strided"},
])
def test_what_was_refused_is_refused(call, wrong):
    args, taken, _ = call
    with pytest.raises((AssertionError, RuntimeError)):
        ops.flash_attn_with_kvcache(**{**args, **{name: args["block_table"].repeat(1, 2)[:, ::2] if isinstance(t, str) else t.cuda() for name, t in wrong.items()}})
    with pytest.raises((AssertionError, RuntimeError)):
        ops.flash_attn_with_kvcache(**{**args, "k_cache": args["k_cache"].cpu(), "v_cache": args["v_cache"].cpu()})
    assert taken == [False, False]


@pytest.mark.parametrize("name,parts", [("q", [(1, 8, 128), (2, 8, 128), (1, 8, 128)]), ("k_cache", [(64, 2, 128), (32, 2, 128)]), ("v_cache", [(64, 2, 128), (32, 2, 128)]),
                                        ("block_table", [(3,), (2,), (3,)])])
def test_nested_tensors_are_refused(call, name, parts):
    """Tensors without sizes: an error of the general way, not one that leaves native code."""
    args, taken, _ = call
    nested = torch.nested.nested_tensor([torch.zeros(s) for s in parts], dtype=torch.int32 if name == "block_table" else BF16, device="cuda")
    with pytest.raises((AssertionError, RuntimeError)):
        ops.flash_attn_with_kvcache(**{**args, name: nested})
    assert taken == [False]
