"""Scratch of the calls in tessera_amd.rules: two calls in flight at once, on two threads here,
each have a buffer of their own (the kernels of one call hand it from one to the next)."""
import ctypes as C
import threading

import pytest

torch = pytest.importorskip("torch")


def _picked(R):
    R.picked(torch.zeros((300, 64)), torch.zeros((4, 8, 64), dtype=torch.bfloat16), torch.zeros(300, dtype=torch.int32))


def _attend(R):
    k = torch.zeros((4096, 2, 128), dtype=torch.bfloat16)
    z = torch.zeros(1, dtype=torch.int32)
    R.attend_rows(torch.zeros((1, 4, 128)), k, k, z, z, keys=4096, scale=1.0, max_position=4095)


def _step(R):
    k = torch.zeros((4096, 2, 128), dtype=torch.bfloat16)
    z = torch.zeros(1, dtype=torch.int32)
    R.attend_step(torch.zeros((1, 8 * 128)), torch.zeros(128), torch.zeros(128), k, k, z, z, heads=4, keys=4096, scale=1.0,
                  eps=1e-6, theta=1e6, max_position=4095, angles=torch.zeros((4096, 64, 2)))


def _argmax(R):
    R.argmax(torch.zeros((2, 200000)))


def _linear(R):
    R.linear(torch.zeros((16, 8192)), torch.zeros((64, 8192), dtype=torch.bfloat16))


@pytest.mark.parametrize("op", [_picked, _attend, _step, _argmax, _linear])
def test_calls_in_flight_do_not_share_scratch(op, monkeypatch):
    from tessera_amd import abi, rules as R
    seen, both = [], threading.Barrier(2, timeout=20)

    def call(name, args, stream):  # stands where the kernels are enqueued: nothing is launched
        a = args._obj.rows if isinstance(args._obj, abi.StepArgs) else args._obj
        both.wait()  # the other thread's call has its scratch too
        seen.append((a.workspace, a.workspace_bytes))
        both.wait()

    monkeypatch.setattr(R, "_stream", lambda: None)
    monkeypatch.setattr(abi, "call", lambda *a: None)
    op(R)  # what an earlier call may have left behind
    monkeypatch.setattr(abi, "call", call)
    threads = [threading.Thread(target=op, args=(R,)) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(30)
    (a, na), (b, nb) = sorted(seen)
    assert na > 0 and nb > 0
    assert a + na <= b


def test_stream_handle_without_the_raw_call(monkeypatch):
    """A torch without its non-public call for the raw handle: the public one."""
    from types import SimpleNamespace

    from tessera_amd import rules as R
    monkeypatch.setattr(R, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: SimpleNamespace(cuda_stream=1234))
    assert R._stream() == 1234


@pytest.mark.gpu
def test_two_streams_match_serial_calls():
    """Expert products and decode attention enqueued on two streams at once give the bits that
    they give one after the other."""
    from tessera_amd import rules as R
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((600, 256), device="cuda", generator=g)
    w = (torch.randn((16, 128, 256), device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    ids = [torch.randint(0, 16, (600,), device="cuda", generator=g, dtype=torch.int32) for _ in range(2)]
    rows, keys = 4, 4096
    k, v = (torch.randn((rows * keys, 2, 128), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    q = [torch.randn((rows, 4, 128), device="cuda", generator=g) for _ in range(2)]
    slots = torch.arange(rows, dtype=torch.int32, device="cuda")
    pos = torch.full((rows,), keys - 1, dtype=torch.int32, device="cuda")

    def work(i):
        return R.picked(x, w, ids[i]), R.attend_rows(q[i], k, v, slots, pos, keys=keys, scale=128 ** -0.5,
                                                     max_position=keys - 1)

    serial = [work(i) for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for _ in range(10):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                got.append((i, work(i)))
    torch.cuda.synchronize()
    for i, outs in got:
        for a, b in zip(outs, serial[i]):
            assert torch.equal(a, b)
