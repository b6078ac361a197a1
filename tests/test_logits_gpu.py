"""A dense decoder's logits are the product with the vocabulary weight as it is when they are asked for, and torch's own operation under
transforms, at the row counts of decode steps."""
import pytest
import torch

from financial_chatbot_llm_amd.models.configs import get_model_config
from financial_chatbot_llm_amd.models.llama import LlamaModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    m = LlamaModel(get_model_config("llama-tiny"), device="cuda").init_random(seed=5)
    assert m.lm_tiled() is not None               # the copy that the sampler reads
    return m


def rows(*shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(shape[-2])).to(torch.bfloat16).cuda()


@pytest.mark.parametrize("M", [1, 4, 5, 16, 64, 128, 129])
def test_weights_changed_in_place(model, M):
    w, h = model.lm_weight(), rows(M, 256)
    keep = w.clone()
    try:
        for change in (lambda: w.mul_(-2.0), lambda: w.data.copy_(keep.flip(0))):
            change()
            want = h.double() @ w.double().t()
            # one rounding to eight significant bits; f32 sums of 256 products
            size = h.double().abs() @ w.double().abs().t()
            assert ((model.logits(h).double() - want).abs() <= 2.0 ** -8 * want.abs() + 256 * 2.0 ** -24 * size).all()
    finally:
        w.copy_(keep)


@pytest.mark.parametrize("M", [1, 4, 16])
def test_transformed_calls(model, M):
    from torch.autograd import forward_ad as fw
    h, t = rows(3, M, 256), rows(3, M, 256).flip(0)
    w = model.lm_weight()
    want, tangent = torch.nn.functional.linear(h, w).float(), torch.nn.functional.linear(t[0], w).float()
    # the library may take another kernel for another number of rows: a rounding to eight significant bits falls the other way
    same = lambda a, b: bool(((a.float() - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -9 * b.std()).all())      # noqa: E731
    assert same(torch.vmap(model.logits)(h), want)
    with fw.dual_level():
        y, dy = fw.unpack_dual(model.logits(fw.make_dual(h[0], t[0])))
    assert same(y, want[0]) and dy is not None and same(dy, tangent)
    y, dy = torch.func.jvp(model.logits, (h[0],), (t[0],))
    assert same(y, want[0]) and same(dy, tangent)
    traced = torch.jit.trace(model.logits, h[0], check_trace=False)
    assert same(traced(h[1]), want[1])
    with torch.autocast("cuda", dtype=torch.float16):
        assert model.logits(h[0]).dtype == torch.float16
