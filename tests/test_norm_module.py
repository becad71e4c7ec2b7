"""YvRMSNorm's parameters as the native call gets them: the attributes a user sees, however they
are defined (a plain parameter, a subclass's property, a parametrization)."""
import torch
import torch.nn as nn

from pisceslx_amd import YvRMSNorm


class _Doubled(YvRMSNorm):
    @property
    def weight(self):
        if "weight" not in self._parameters:    # not yet registered
            raise AttributeError("weight")
        return self._parameters["weight"] * 2


class _Plus(nn.Module):
    def forward(self, w):
        return w + 1


def test_parameters_are_the_attributes():
    plain = YvRMSNorm(8, use_bias=True)
    w, b, eps = plain.norm_params()
    assert w.data_ptr() == plain.weight.data_ptr() and b.data_ptr() == plain.bias.data_ptr() and eps == 1e-6
    assert not w.requires_grad and YvRMSNorm(8).norm_params()[1] is None


def test_a_subclass_may_define_them_otherwise():
    m = _Doubled(8)
    assert torch.equal(m.weight, torch.full((8,), 2.0))
    assert torch.equal(m.norm_params()[0], m.weight)


def test_parametrized_weight():
    m = YvRMSNorm(8)
    nn.utils.parametrize.register_parametrization(m, "weight", _Plus())
    assert torch.equal(m.norm_params()[0], torch.full((8,), 2.0))
