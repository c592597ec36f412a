"""Which projections' calls a kernel may stand in for: the package's own, with nobody listening; not a class, a forward or a quant method of somebody's
own in their place, whatever it holds."""
import pytest
import torch
from torch import nn

from aphrodite_engine_amd import model as M
from aphrodite_engine_amd.quantization.awq import AWQConfig
from aphrodite_engine_amd.quantization.gptq import ExllamaState, GPTQConfig


class Adapter(M.QuantLinear):
    def forward(self, x, add_bias=True):
        return super().forward(x, add_bias) + 1


class Wrapper(nn.Module):                                    # (none of a projection's attributes)
    def __init__(self, lin):
        super().__init__()
        self.lin = lin

    def forward(self, x):
        return self.lin(x)


def _linear(quant, cls=M.QuantLinear):
    lin = cls(256, [128, 128], quant, torch.float16)
    if isinstance(quant, GPTQConfig):
        lin.exllama_state, lin.g_idx.data = ExllamaState.READY, torch.empty(0, dtype=torch.int32)
    else:
        lin.awq_prepacked = True
    return lin


@pytest.mark.parametrize("quant", [GPTQConfig(4, 128, False), AWQConfig(4, 128, True)])
def test_whose_words_are_multiplied_without_a_call(quant):
    words, x = M.LlamaDecoderLayer._int4_words, torch.zeros(70, 256)
    lin = _linear(quant)
    assert words(lin, x) is not None and words(lin, x[:64]) is None
    assert words(_linear(quant, Adapter), x) is None
    assert words(Wrapper(lin), x) is None
    lin.forward = lambda x, add_bias=True: x
    assert words(lin, x) is None
    del lin.forward
    lin.quant_method.apply = lambda layer, x, bias=None: x
    assert words(lin, x) is None
    del lin.quant_method.apply
    own = lin.quant_method
    lin.quant_method = type("Own", (type(own), ), {"apply": lambda self, layer, x, bias=None: x})(own.quant_config)
    assert words(lin, x) is None
    lin.quant_method = own
    handle = lin.register_forward_hook(lambda module, args, out: out)
    assert words(lin, x) is None
    handle.remove()
    assert words(lin, x) is not None
