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
    """A fused residual of tensors reads no flags; with b as a NumPy array of
    1 MiB its upload is what a capture must refuse."""
    import torch
    from ozaki_jax_amd import _lib
    rng = np.random.RandomState(2)
    A = torch.from_numpy(rng.randn(1 << 17, 8)).cuda()
    x = torch.from_numpy(rng.randn(8)).cuda()
    b = rng.randn(1 << 17)
    want = ozk.residual(A, x, torch.from_numpy(b).cuda(), mode="ozaki")
    case("residual with a NumPy b under capture")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="relaxed"):
        with pytest.raises(_lib.OzakiError, match="capture"):
            ozk.residual(A, x, b, mode="ozaki")
        x.zero_()
    assert torch.equal(ozk.residual(A, x, b, mode="ozaki"), want)
