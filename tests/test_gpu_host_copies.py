"""Copies between NumPy arrays and the device through pinned memory: what a
captured stream is refused, and that calls of other threads do not wait for
each other's streams."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def case(msg):
    print(f"[case] {msg}", flush=True)


@pytest.mark.parametrize("mode", ["relaxed", "global"])
def test_slots_refuse_a_captured_stream(ozk, mode):
    """A copy recorded from a pinned slot would read, on replay, what later
    copies left there.  It is refused under capture before anything is
    recorded, with the other copies of the ring untouched."""
    import torch
    from ozaki_jax_amd import _hip, _lib
    lib = _lib.load()
    st = _hip._stager()
    a = np.random.RandomState(1).randn(1 << 18)
    t = torch.zeros(a.shape, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    case(f"ozk_copy_slots under {mode} capture, up and down")
    for down in (0, 1):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, capture_error_mode=mode):
            rc = lib.ozk_copy_slots(down, t.data_ptr(), a.ctypes.data, a.nbytes, st.up.buf,
                                    st.up.slot, st.up.slots, 0, st.up.ev, 2,
                                    torch.cuda.current_stream().cuda_stream)
            err = ctypes.string_at(lib.ozk_last_error())
            t.zero_()  # the capture itself goes on
        assert rc == _lib.OZK_ERR_HIP and b"capture" in err
        g.replay()
    torch.cuda.synchronize()
    for _ in range(3):
        d = _hip.DeviceArray.from_numpy(a)
        assert np.array_equal(d.numpy(), a)


def test_residual_with_numpy_operands_refuses_capture(ozk):
    """A fused residual of tensors reads no flags; with b as a NumPy array its
    staged upload (16 MiB) is what a capture must refuse."""
    import torch
    from ozaki_jax_amd import _lib
    rng = np.random.RandomState(2)
    A = torch.from_numpy(rng.randn(1 << 21, 8)).cuda()
    x = torch.from_numpy(rng.randn(8)).cuda()
    b = rng.randn(1 << 21)
    want = ozk.residual(A, x, torch.from_numpy(b).cuda(), mode="ozaki")
    case("residual with a NumPy b under capture")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="relaxed"):
        with pytest.raises(_lib.OzakiError, match="capture"):
            ozk.residual(A, x, b, mode="ozaki")
        x.zero_()
    assert torch.equal(ozk.residual(A, x, b, mode="ozaki"), want)


def _busy(stream, seconds):
    """A kernel of about this long on `stream` (one spinning workgroup), and
    the event behind it."""
    import torch
    with torch.cuda.stream(stream):
        e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        e0.record()
        torch.cuda._sleep(1000000)
        e1.record()
        e1.synchronize()
        cycles = int(1000000 * seconds * 1e3 / e0.elapsed_time(e1))
        done = torch.cuda.Event()
        torch.cuda._sleep(cycles)
        done.record()
    return done


def _independent_stream():
    """A stream whose work does not hold up the current stream's: streams
    share the few hardware queues, and those of one queue run in order."""
    import torch
    x = torch.zeros(1 << 20, dtype=torch.float64, device="cuda")
    for _ in range(16):
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        done = _busy(s, 0.05)
        x.add_(1.0).cpu()
        if not done.query():
            torch.cuda.synchronize()
            return s
    pytest.skip("every stream shares the current stream's hardware queue")


@pytest.mark.parametrize("way,mib", [("down", 4), ("down", 48), ("up", 32), ("up", 130)])
def test_copies_do_not_wait_for_another_threads_stream(ozk, way, mib):
    """One thread copies on a stream that is busy for a second; a copy of
    another thread, on an idle stream through the same pinned memory, is done
    long before that."""
    import threading
    import torch
    from ozaki_jax_amd import _device as D
    n = (mib << 20) // 8
    dev = torch.device("cuda", torch.cuda.current_device())
    rng = np.random.RandomState(mib)
    a = [rng.randn(n // 1024, 1024) for _ in range(2)]
    t = [torch.from_numpy(v).cuda() for v in a]
    for i in range(2):  # the pinned memory of this size is there
        assert np.array_equal(D._torch_to_numpy(D._numpy_to_torch(a[i], dev)), a[i])
    busy = _independent_stream()
    case(f"{way} {mib} MiB beside a busy stream")
    done = _busy(busy, 1.0)
    got, inside = {}, threading.Event()

    def first():
        with torch.cuda.stream(busy):
            inside.set()
            got[0] = D._torch_to_numpy(t[0]) if way == "down" else D._numpy_to_torch(a[0], dev)

    th = threading.Thread(target=first)
    th.start()
    inside.wait()
    threading.Event().wait(0.2)  # the first thread's copy has begun
    got[1] = D._torch_to_numpy(t[1]) if way == "down" else D._numpy_to_torch(a[1], dev)
    if way == "up":
        torch.cuda.current_stream().synchronize()
    early = not done.query()
    th.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert np.array_equal(got[i] if way == "down" else got[i].cpu().numpy(), a[i])
    assert early, "the copy waited for the other thread's stream"


def test_f64s_by_place(ozk, monkeypatch):
    """Which uploads are staged, and which of them follow another without a
    wait: sizes around the thresholds, alone and in rows."""
    import torch
    from ozaki_jax_amd import _device as D, _hip
    fam = D.family(False)
    seen = []
    to_device = _hip._Stager.to_device

    def spy(self, ptr, host, stream=None, following=False):
        seen.append((host.nbytes, following))
        return to_device(self, ptr, host, stream, following)

    monkeypatch.setattr(_hip._Stager, "to_device", spy)
    rng = np.random.RandomState(3)
    mib = 1 << 17
    small, one, four, big = (rng.randn(n) for n in (mib - 1, mib, 4 * mib, 16 * mib))
    tensor = torch.ones(2 * mib, dtype=torch.float32, device="cuda")
    rows = [([one], []), ([big], [False]), ([four, small], []),
            ([one, four], [False, True]), ([one, small, four], [False, True]),
            ([four.astype(np.float32), one, big], [False, True, True])]
    rows.append(([one, tensor, four, one], [False, True, False, True]))
    for xs, want in rows:
        del seen[:]
        case(f"f64s of {[x.nbytes if isinstance(x, np.ndarray) else 'tensor' for x in xs]}")
        out = fam.f64s(*xs)
        assert [f for _, f in seen] == want
        for x, t in zip(xs, out):
            x = x if isinstance(x, np.ndarray) else x.cpu().numpy()
            assert np.array_equal(t.numpy(), x.astype(np.float64))
