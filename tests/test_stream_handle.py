"""The binding's way to torch's current stream: the raw handle where torch has
the (private) calls for it, the public call where it does not."""
from types import SimpleNamespace

import ssdq


def fake_torch(**private):
    cuda = SimpleNamespace(is_initialized=lambda: True, current_stream=lambda: SimpleNamespace(cuda_stream=0x1234))
    return SimpleNamespace(cuda=cuda, _C=SimpleNamespace(**private))


def call(calls):
    initialised, device, handle = calls
    assert initialised()
    return handle(device())


def test_raw_handle():
    t = fake_torch(_cuda_getDevice=lambda: 3, _cuda_getCurrentRawStream=lambda d: 100 + d)
    assert call(ssdq._stream_calls(t)) == 103


def test_public_call_without_the_private_names():
    assert call(ssdq._stream_calls(fake_torch())) == 0x1234
    assert call(ssdq._stream_calls(fake_torch(_cuda_getDevice=lambda: 3))) == 0x1234


def test_given_stream():
    assert ssdq._stream(SimpleNamespace(cuda_stream=7)) == 7
