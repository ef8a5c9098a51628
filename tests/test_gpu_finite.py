"""vcx_check_finite answers for every element of vc_attention's inputs."""
import pytest
import torch

import vcx
from helpers import make_qkv
from vc_attention import Config, attention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("n", [8, 2048, 1024 * 256 * 8 + 8])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_finite_check_sees_every_element(n, dtype):
    print("case: finite", n, dtype, flush=True)
    x = [torch.full((1, 1, n // 8, 8), torch.finfo(dtype).max, dtype=dtype, device=DEV) for _ in range(3)]
    x[1] = -x[1]
    x[2].fill_(torch.finfo(dtype).smallest_normal / 2)
    assert vcx.all_finite(*x)
    for which in range(3):
        for at in {0, 5, n // 2, n - 1}:
            for bad in (float("nan"), float("inf"), -float("inf")):
                keep = x[which].view(-1)[at].item()
                x[which].view(-1)[at] = bad
                assert not vcx.all_finite(*x), (which, at, bad)
                x[which].view(-1)[at] = keep
    assert vcx.all_finite(*x)


def test_finite_check_on_every_layout_and_its_errors():
    print("case: finite layouts", flush=True)
    base = torch.randn(2, 37, 3, 72, device=DEV).to(torch.bfloat16)
    views = {"nhd": base.transpose(1, 2), "cut": base[..., :64].transpose(1, 2), "off": base[..., 1:65],
             "odd": base[:1, :1, :1, :5], "f32": base.float()}
    for name, x in views.items():
        assert vcx.all_finite(x, x, x), name
        y = x.clone() if name != "nhd" else base.clone().transpose(1, 2)
        y[-1, -1, -1, -1] = float("nan")
        assert not vcx.all_finite(x, y, x), name
    q, k, v = (x.to(DEV) for x in make_qkv(1, 2, 100, 130, 64))
    cfg = Config(backend="hip", qk_format="int8", q_block=64, k_quant_block=128)
    v[0, 1, 129, 63] = float("inf")
    with pytest.raises(ValueError, match="must be finite"):
        attention(q, k, v, cfg)
