"""How pack() stores what the packing kernel returns: like any assignment to the layer's buffers (CPU: the kernel is a stand-in)."""
import subprocess
import sys

import pytest
import torch
import torch.nn as nn

import onebitsparsemul_amd as amd

M, K = 64, 32


class _Weight:
    """what pack() asks of a weight on the GPU"""
    shape, is_cuda, dtype = (M, K), True, torch.float16

    def contiguous(self):
        return self

    def data_ptr(self):
        return 0


class _Binding:
    a, meta = torch.ones((K // 2, M // 8), dtype=torch.uint8), torch.ones((M, K // 16), dtype=torch.int16)

    def pack_weight(self, *_):
        return self.a, self.meta


@pytest.fixture(autouse=True)
def _stand_in(monkeypatch):
    monkeypatch.setattr(amd, "_compiled", _Binding())


def _check(layer):
    layer._prepared = object()
    layer.pack(_Weight())
    assert layer.packed_binary_sparse is _Binding.a and layer.meta is _Binding.meta
    assert layer._buffers["packed_binary_sparse"] is _Binding.a and layer._buffers["meta"] is _Binding.meta
    assert layer.vaild is True and layer._prepared is None


def test_plain_layer():
    _check(amd.BinaryLinear_2_4(K, M))


def test_a_class_that_sets_attributes_its_own_way_sees_them():
    class Watched(amd.BinaryLinear_2_4):
        def __setattr__(self, name, value):
            self.__dict__.setdefault("seen", []).append(name)
            super().__setattr__(name, value)

    layer = Watched(K, M)
    layer.seen.clear()
    _check(layer)
    assert {"packed_binary_sparse", "meta", "vaild"} <= set(layer.seen)


def test_an_attribute_with_a_setter():
    class Property(amd.BinaryLinear_2_4):
        sets = 0

        @property
        def vaild(self):
            return self.__dict__.get("state", False)

        @vaild.setter
        def vaild(self, value):
            type(self).sets += 1
            self.__dict__["state"] = value

    layer = Property(K, M)
    Property.sets = 0
    _check(layer)
    assert Property.sets == 1


def test_registration_hooks_see_the_buffers():
    layer, names = amd.BinaryLinear_2_4(K, M), []
    hook = nn.modules.module.register_module_buffer_registration_hook(lambda module, name, value: names.append(name))
    try:
        _check(layer)
    finally:
        hook.remove()
    assert names == ["packed_binary_sparse", "meta"]


def test_a_torch_that_keeps_the_hooks_elsewhere():
    program = ("import torch.nn.modules.module as m; hooks = m._global_buffer_registration_hooks; "
               "del m._global_buffer_registration_hooks; import onebitsparsemul_amd")
    subprocess.run([sys.executable, "-c", program], check=True, cwd=amd.__file__.rsplit("/", 2)[0])
