"""The packed form a dispatch passes holds to_c()'s bytes, for every payload class
that has one; values past their fields' widths and types other than int go
through to_c(), which wraps or refuses them."""
import random
from dataclasses import fields, replace

import numpy as np
import pytest

from hologram_amd import BufferRef
from hologram_amd import kernel_call as kc


def filled(cls, rng, value):
    args = {}
    for f in fields(cls):
        if f.type in ("MatMulCall", "DecodeAttentionI8Call"):
            args[f.name] = filled(getattr(kc, f.type), rng, value)
        elif f.type == "BufferRef":
            args[f.name] = BufferRef(value(), value(), value())
        elif f.type == "bool":
            args[f.name] = rng.random() < 0.5
        else:
            args[f.name] = value()
    return cls(**args)


@pytest.mark.parametrize("cls", sorted(kc._FLAT, key=lambda c: c.__name__))
def test_packed_form_is_to_c(cls):
    rng = random.Random(cls.__name__)
    packed = 0
    for bits in (8, 16, 32, 64, 70):
        for _ in range(20):
            payload = filled(cls, rng, lambda: rng.randint(0, (1 << bits) - 1))
            call = kc.KernelCall(rng.randint(0, 200), payload)
            form = kc.dispatch_form(call)
            if isinstance(form, bytes):
                packed += 1
                assert form == bytes(call.to_c())
            else:
                assert bytes(form._obj) == bytes(call.to_c())
    assert packed >= 20
    payload = filled(cls, rng, lambda: rng.randint(0, 255))
    last = fields(payload)[-1].name
    for bad in (None, "1", 1.5, np.int64(1), -1):
        call = kc.KernelCall(1, replace(payload, **{last: bad}))
        got = []
        for f in (lambda c: (lambda x: x if isinstance(x, bytes) else bytes(x._obj))(kc.dispatch_form(c)),
                  lambda c: bytes(c.to_c())):
            try:
                got.append(f(call))
            except Exception as e:  # noqa: BLE001 (whatever the conversion raises)
                got.append(type(e))
        assert got[0] == got[1]


def test_other_payloads_go_through_to_c():
    class Sub(kc.UnaryCall):
        pass
    u = kc.KernelCall(1, Sub(BufferRef(0), BufferRef(1), 8))
    assert not isinstance(kc.dispatch_form(u), bytes)
    with pytest.raises(TypeError):
        kc.dispatch_form(kc.KernelCall(1, object()))
