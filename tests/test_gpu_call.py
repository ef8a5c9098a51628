"""vcx_attention_call: one call gives the bits of its stages."""
import pytest
import torch

import vcx
from helpers import make_qkv
from sageattention_local import forward_prepared, prepare, sageattn_vc
from sageattention_local import vc_fp8
from vc_attention import Config, LayoutCache, attention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("shape", [(2, 3, 257, 400, 128), (1, 2, 2048, 2048, 64), (1, 1, 1, 1, 128)])
@pytest.mark.parametrize("layout", ["HND", "NHD"])
@pytest.mark.parametrize("options", [
    dict(v_smooth=False), dict(v_smooth=False, v_scale_mode="block"), dict(v_smooth=False, kernel_mode="vc9"), dict(v_smooth=False, expcast=False),
    dict(), dict(v_scale_mode="block"), dict(expcast=False, clusters=16), dict(grouping_mode="legacy", sm_scale=0.2),
], ids=lambda o: "_".join("%s-%s" % kv for kv in o.items()) or "default")
def test_one_call_gives_the_bits_of_its_stages(shape, layout, options):
    print("case: one call", shape, layout, options, flush=True)
    q, k, v = (x.to(DEV) for x in make_qkv(*shape, torch.float16, seed=3, kind="outlier"))
    stages = {n: x for n, x in options.items() if n != "kernel_mode"}
    want = forward_prepared(prepare(q, k, v, **stages), kernel_mode=options.get("kernel_mode", "optimized"))
    if layout == "NHD":
        q, k, v, want = (x.transpose(1, 2).contiguous() for x in (q, k, v, want))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        got = sageattn_vc(q, k, v, tensor_layout=layout, **options)
        again = sageattn_vc(q, k, v, tensor_layout=layout, **options)
    stream.synchronize()
    assert got.shape == want.shape and got.is_contiguous()
    assert torch.equal(got, want) and torch.equal(again, want)


@pytest.mark.parametrize("expcast", [True, False])
def test_one_fp8_call_and_cached_steps_give_the_bits_of_their_stages(expcast):
    print("case: one fp8 call, steps", expcast, flush=True)
    q, k, v = (x.to(DEV) for x in make_qkv(1, 3, 300, 1000, 128, torch.bfloat16, seed=5, kind="outlier"))
    want = vc_fp8.forward_prepared(vc_fp8.prepare(q, k, v, expcast=expcast))
    assert torch.equal(vc_fp8.sageattn_vc_fp8(q, k, v, expcast=expcast), want)
    for rotate in (False, True):
        cfg = Config(backend="hip", qk_format="int8", q_block=64, k_quant_block=128, expcast=expcast, v_smooth=True,
                     qk_hadamard=rotate, active_fraction=0.5)
        cache = LayoutCache(cfg)
        for step in range(4):  # steps 2 and 3: no smoothing, K and V still gathered by the layout
            out, counters = attention(q, k, v, cfg, cache=cache, step=step, total_steps=4, request_id="r")
            active, perm = step < 2, cache._layers[0].permutation
            assert counters["smoothing_active"] == active
            q8, qs, k8, ks, _ = vcx.prepare_qk(q, k, perm, hadamard=rotate)
            v8, vs, means = vcx.prepare_v(v, perm, smooth=active)
            assert torch.equal(out, vcx.forward(q8, k8, v8, qs, ks, vs, means, expcast, active, 1, 128 ** -0.5,
                                                affine=expcast and not active))


def test_smoothing_without_a_permutation_keeps_the_tokens_order():
    print("case: smoothing in the given order", flush=True)

    class InOrder(LayoutCache):
        def layout(self, v, **kwargs):
            return None, True, False

    q, k, v = (x.to(DEV) for x in make_qkv(1, 3, 300, 1000, 128, torch.bfloat16, seed=9, kind="outlier"))
    cfg = Config(backend="hip", qk_format="int8", q_block=64, k_quant_block=128, expcast=True, v_smooth=True,
                 qk_hadamard=False)
    out, _ = attention(q, k, v, cfg, cache=InOrder(cfg), request_id="r")
    q8, qs, k8, ks, _ = vcx.prepare_qk(q, k)
    v8, vs, means = vcx.prepare_v(v, smooth=True)
    assert torch.equal(out, vcx.forward(q8, k8, v8, qs, ks, vs, means, True, True, 1, 128 ** -0.5))


def test_one_call_under_capture_replays_to_the_same_bits():
    print("case: one call captured", flush=True)
    q, k, v = (x.to(DEV) for x in make_qkv(1, 2, 300, 700, 128, torch.bfloat16, seed=7, kind="outlier"))
    want = sageattn_vc(q, k, v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sageattn_vc(q, k, v)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(sageattn_vc(q, k, v), want)


def test_one_call_refuses_what_its_stages_refuse():
    q, k, v = (x.to(DEV) for x in make_qkv(1, 2, 64, 130, 64))
    wide = torch.randn(1, 2, 130, 68, device=DEV).to(torch.bfloat16)
    with pytest.raises(vcx.VcxError, match="alignment"):
        sageattn_vc(q, wide[..., 1:65], v, v_smooth=False)
    with pytest.raises(vcx.VcxError, match="multiples"):
        sageattn_vc(q, torch.randn(1, 2, 130, 66, device=DEV).to(torch.bfloat16)[..., :64], v, v_smooth=False)
    with pytest.raises(vcx.VcxError, match="contiguous last dimension"):
        sageattn_vc(q, k, v.transpose(2, 3).contiguous().transpose(2, 3))
    with pytest.raises(vcx.VcxError, match="sm_scale"):
        sageattn_vc(q, k, v, sm_scale=1e-60)
