"""Published flag words (ozk_matmul_flag_word, ozk_gram_flag_word) against
ozk_matmul and ozk_gram: the same product bit for bit, the same flags, and a
device word that is zero again, over plane formats, multi-sweep, rectangle
and pairwise schedules, both pipelines and empty products."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def case(msg):
    print(f"[case] {msg}", flush=True)


def device_word(words):
    """The device word once the device is idle."""
    import ctypes
    import torch
    from ozaki_jax_amd import _hip
    torch.cuda.synchronize()
    v = ctypes.c_uint32(7)
    _hip._rt().copy(ctypes.addressof(v), words.dev, 4, _hip._D2H)
    return v.value


# (shape, pipeline, n_hi, n_lo, order, input): orders 0 2Sum, 1 FP64 block,
# 2 host; (6, 1) rectangle sweeps, (9, 1) the pairwise kernel
CASES = [((130, 8192, 70), 0, 4, 1, 0, None), ((130, 8192, 70), 0, 4, 1, 0, "nan"),
         ((64, 8192, 48), 0, 5, 4, 1, "big"), ((64, 6000, 48), 0, 6, 1, 0, "nan"),
         ((64, 300, 48), 0, 9, 1, 0, "nan"), ((65, 65600, 33), 0, 3, 1, 0, "nan"),
         ((100, 300, 90), 0, 3, 1, 0, None), ((1, 1, 1), 0, 4, 1, 0, "nan"),
         ((100, 300, 90), 1, 8, 0, 2, "nan"), ((100, 300, 90), 1, 8, 0, 2, None),
         ((0, 300, 90), 0, 4, 1, 0, None)]


@pytest.mark.parametrize("shape,pipe,nh,nl,order,kind", CASES)
def test_flag_word_matches_matmul(ozk, shape, pipe, nh, nl, order, kind):
    import torch
    from ozaki_jax_amd import _lib, _device as D
    lib = _lib.load()
    dev = torch.device("cuda", 0)
    N, K, M = shape
    rng = np.random.RandomState(N + K + M + nh)
    A, B = rng.randn(N, K), rng.randn(K, M)
    if kind == "nan":
        A[N // 2, K // 3] = np.nan
    elif kind == "big":
        A[1] *= 2.0 ** 110
    At, Bt = torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev)
    wsb = lib.ozk_matmul_workspace_bytes(N, K, M, pipe, nh, nl)
    ws = D.workspace(wsb, dev)

    def args(C):
        return (At.data_ptr(), K, Bt.data_ptr(), M, C.data_ptr(), M, N, K, M, pipe, nh, nl,
                order, ws.data_ptr(), wsb)

    case(f"ozk_matmul_flag_word {shape} pipeline {pipe} ({nh},{nl}) order {order} {kind}")
    C1 = torch.full((N, M), 7.0, dtype=torch.float64, device=dev)
    f1 = torch.full((1,), -559038737, dtype=torch.int32, device=dev)
    _lib.check(lib.ozk_matmul(*args(C1), f1.data_ptr(), D.stream_handle()))
    want = int(f1.item()) & 0xffffffff
    C2 = torch.full((N, M), 7.0, dtype=torch.float64, device=dev)
    words = D.FlagWords(0)
    for _ in range(2):  # the second call relies on the first leaving zeros
        got = words.run(lambda d, h: lib.ozk_matmul_flag_word(*args(C2), d, h, D.stream_handle()),
                        D.stream_handle())
        assert got == want
        assert device_word(words) == 0
    if kind:  # finite inputs on the same words: no flag is left over
        At.copy_(torch.from_numpy(np.where(np.isfinite(A) & (np.abs(A) < 1e9), A, 1.0)))
        C3 = torch.empty_like(C2)
        assert words.run(lambda d, h: lib.ozk_matmul_flag_word(*args(C3), d, h, D.stream_handle()),
                         D.stream_handle()) == 0
    torch.cuda.synchronize()
    assert bool(want & _lib.OZK_FLAG_NONFINITE) == (kind == "nan")
    assert np.array_equal(C1.cpu().numpy(), C2.cpu().numpy(), equal_nan=True)


@pytest.mark.parametrize("rows,cols,nh,nl,kind", [(9000, 200, 4, 1, "nan"), (300, 65, 3, 1, None),
                                                  (3000, 150, 5, 4, "nan"), (300, 0, 4, 1, None)])
def test_gram_flag_word_matches_gram(ozk, rows, cols, nh, nl, kind):
    import torch
    from ozaki_jax_amd import _lib, _device as D
    lib = _lib.load()
    dev = torch.device("cuda", 0)
    A = np.random.RandomState(rows).randn(rows, cols)
    if kind == "nan":
        A[rows // 2, cols // 3] = np.nan
    At = torch.from_numpy(A).to(dev)
    wsb = lib.ozk_gram_workspace_bytes(rows, cols, nh, nl)
    ws = D.workspace(wsb, dev)
    G = [torch.full((cols, cols), 7.0, dtype=torch.float64, device=dev) for _ in range(2)]
    f = torch.full((1,), -559038737, dtype=torch.int32, device=dev)

    def args(i):
        return (At.data_ptr(), max(cols, 1), rows, cols, nh, nl, G[i].data_ptr(), max(cols, 1),
                ws.data_ptr(), wsb)

    case(f"ozk_gram_flag_word ({rows},{cols}) ({nh},{nl}) {kind}")
    _lib.check(lib.ozk_gram(*args(0), f.data_ptr(), D.stream_handle()))
    words = D.FlagWords(0)
    got = words.run(lambda d, h: lib.ozk_gram_flag_word(*args(1), d, h, D.stream_handle()),
                    D.stream_handle())
    assert device_word(words) == 0
    assert got == int(f.item()) & 0xffffffff
    assert bool(got & _lib.OZK_FLAG_NONFINITE) == (kind == "nan")
    assert np.array_equal(G[0].cpu().numpy(), G[1].cpu().numpy(), equal_nan=True)


def test_a_word_that_never_comes_is_an_error(ozk):
    """An idle stream ends the wait with an error, as does a null word."""
    import ctypes
    from ozaki_jax_amd import _lib, _device as D
    lib = _lib.load()
    words = D.FlagWords(0)
    with pytest.raises(_lib.OzakiError, match="never published"):
        words.run(lambda d, h: 0, D.stream_handle())
    with pytest.raises(ValueError, match="null host flag word"):
        _lib.check(lib.ozk_matmul_flag_word(None, 4, None, 4, None, 4, 4, 4, 4, 0, 4, 1, 0, None,
                                            0, None, None, None))
    with pytest.raises(ValueError, match="null pointer"):
        _lib.check(lib.ozk_wait_flag_word(None, None, ctypes.byref(ctypes.c_uint32())))


def test_concurrent_calls_have_words_of_their_own(ozk):
    """Threads with streams of their own, one of them with NaN input: only
    its calls raise."""
    import threading
    import torch
    rng = np.random.RandomState(0)
    A = torch.from_numpy(rng.randn(96, 400)).to("cuda")
    B = torch.from_numpy(rng.randn(400, 64)).to("cuda")
    bad = A.clone()
    bad[3, 5] = float("nan")
    want = ozk.matmul(A, B, pipeline="ondevice")
    torch.cuda.synchronize()
    wrong = []
    case("matmul from four threads, one with NaN")

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                try:
                    C = ozk.matmul(bad if i == 0 else A, B, pipeline="ondevice")
                    if i == 0:
                        wrong.append("no error for NaN")
                    elif not torch.equal(C, want):
                        wrong.append("wrong product")
                except ValueError:
                    if i:
                        wrong.append("error without NaN")

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong, wrong


def test_rejected_calls_give_their_words_back(ozk, monkeypatch):
    """A call that the library refuses before anything is queued leaves its
    words usable: no allocation per rejected call."""
    import torch
    from ozaki_jax_amd import _device as D, _hip
    monkeypatch.setattr(D, "_flag_words_free", {})
    A = torch.from_numpy(np.random.RandomState(0).randn(64, 300)).to("cuda")
    want = ozk.matmul(A, A.T.contiguous(), pipeline="ondevice")  # one pair is there
    rt, got = _hip._rt(), []
    host_malloc = rt.host_malloc
    monkeypatch.setattr(rt, "host_malloc", lambda n: (got.append(n), host_malloc(n))[1])
    case("products and Gram matrices with slice counts that are refused")
    for _ in range(5):
        with pytest.raises(ValueError):
            ozk.matmul(A, A.T.contiguous(), pipeline="ondevice", precision=(40, 1))
        with pytest.raises(ValueError):
            ozk.gram(A, precision=(40, 1), mode="ozaki")
    assert torch.equal(ozk.matmul(A, A.T.contiguous(), pipeline="ondevice"), want)
    assert not got


def test_kept_words_are_released(ozk):
    """What is kept between calls is released by the exit hook, and calls
    after that allocate anew."""
    import torch
    from ozaki_jax_amd import _device as D, _hip
    A = torch.from_numpy(np.random.RandomState(0).randn(64, 300)).to("cuda")
    want = ozk.gram(A, mode="ozaki")
    word, ev, read = D._TorchFamily().early_flags()
    _hip._rt().record(ev)
    read()
    torch.cuda.synchronize()
    assert any(D._flag_words_free.values()) and any(D._early_free.values())
    case("release of the kept words")
    for hook in _hip._exit_hooks:
        hook(_hip._rt().h)
    assert not any(D._flag_words_free.values()) and not any(D._early_free.values())
    assert torch.equal(ozk.gram(A, mode="ozaki"), want)
