"""The host-buffer entry points (qlin_run_f32 / qlin_run_swiglu_f32) through pinned row blocks:
against the device entry point bit for bit at one block, several blocks (more than the slots)
and a ragged last one, at the forms that go through plain copies (K not a multiple of 8, rows
longer than a slot); the error word of a call and of the workspace; several threads at once."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from open_rknpu2_lm_infer_amd import _lib
from open_rknpu2_lm_infer_amd import qlinear as ql
from open_rknpu2_lm_infer_amd import synth
from open_rknpu2_lm_infer_amd._lib import QLIN_ERR_NONFINITE, QLIN_OK, QlinError

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def weights(bits, K, N, seed):
    packed, _, sc = synth.make_linear(N, K, bits, seed, device=DEV)
    return ql.Weights.from_packed_device(bits, K, N, packed, sc)


@pytest.mark.parametrize("bits,K,N,rows", [
    # blocks of 1 MiB of rows: one; the most rows of one, and one more; more blocks than slots
    (4, 2560, 6144, 1), (4, 9728, 2560, 26), (4, 9728, 2560, 27), (8, 4096, 2560, 300), (4, 2560, 2000, 1000),
    (8, 64, 262144, 5),         # one row per block
    (8, 64, 262146, 3),         # a row longer than a slot
    (8, 8192, 28672, 64), (8, 32160, 190, 212),  # weights, or a K, that cost more per block than it saves
    (8, 1001, 98, 40), (4, 1002, 98, 1)])
def test_host_runs_equal_device_runs(bits, K, N, rows):
    w, ws = weights(bits, K, N, 960 + rows), ql.Workspace(rows, K, N)
    for seed in (0, 1):  # a second call goes through the slots the first one used
        A = synth.activations(rows, K, 961 + seed).float().numpy()
        for sw in (False, True):
            want = ql.run(ws, w, torch.from_numpy(A).to(DEV), out_dtype=torch.float32, flags=ql.QLIN_SWIGLU if sw else 0)
            torch.cuda.synchronize()
            got = ql.run_host_f32(ws, w, A, swiglu=sw)
            assert np.array_equal(got.view(np.uint32), want.cpu().numpy().view(np.uint32)), (seed, sw)
    ws.close()
    w.close()


def test_host_run_error_word():
    """A non-finite row in any block fails its call and marks the workspace; the next call, and
    the workspace's word with it, are clean again, also after an asynchronous run set it."""
    K, N, rows = 2560, 2560, 400
    w, ws = weights(4, K, N, 970), ql.Workspace(rows, K, N)
    A = synth.activations(rows, K, 971).float().numpy()
    ref = ql.run_host_f32(ws, w, A)
    for row in (0, 250, rows - 1):
        bad = A.copy()
        bad[row, 7] = np.inf
        with pytest.raises(QlinError) as e:
            ql.run_host_f32(ws, w, bad)
        assert e.value.rc == QLIN_ERR_NONFINITE and ws.status(clear=False) == QLIN_ERR_NONFINITE
        assert np.array_equal(ql.run_host_f32(ws, w, A), ref) and ws.status(clear=False) == QLIN_OK
    x = torch.from_numpy(A).to(DEV)
    x[3, 3] = float("nan")
    ql.run(ws, w, x)
    torch.cuda.synchronize()
    assert np.array_equal(ql.run_host_f32(ws, w, A), ref) and ws.status(clear=False) == QLIN_OK
    ws.close()
    w.close()


def test_host_run_clears_the_word_of_a_run_through_copies():
    """A call whose rows go through plain copies (K = 1002) sets the workspace's word itself; the
    next call through the slots starts clean."""
    w, wide = weights(4, 2560, 256, 975), weights(4, 1002, 256, 976)
    ws = ql.Workspace(4, 2560, 256)
    bad = synth.activations(4, 1002, 977).float().numpy()
    bad[2, 5] = np.inf
    with pytest.raises(QlinError):
        ql.run_host_f32(ws, wide, bad)
    assert ws.status(clear=False) == QLIN_ERR_NONFINITE
    ql.run_host_f32(ws, w, synth.activations(4, 2560, 978).float().numpy())
    assert ws.status(clear=False) == QLIN_OK
    for x in (ws, w, wide):
        x.close()


def test_host_run_over_its_own_input():
    """C at A, with rows out longer than rows in, over several blocks: every row is read first."""
    K, N, rows = 1024, 2048, 500
    w, ws = weights(8, K, N, 985), ql.Workspace(rows, K, N)
    A = synth.activations(rows, K, 986).float().numpy()
    want = ql.run_host_f32(ws, w, A)
    buf = np.zeros(rows * N, np.float32)
    buf[:rows * K] = A.reshape(-1)
    at = buf.ctypes.data_as(ctypes.c_void_p)
    assert _lib.load().qlin_run_f32(ws.handle, w.handle, rows, at, at) == QLIN_OK
    assert np.array_equal(buf.reshape(rows, N), want)
    ws.close()
    w.close()


@pytest.mark.parametrize("mode", ["thread_local", "relaxed"])
def test_host_runs_beside_a_capture(mode):
    """Six host-buffer calls on threads of their own, more than the idle sets kept (so that sets
    are allocated and freed), while this thread records a graph: both give their usual results."""
    K, N = 2560, 2560
    w = weights(4, K, N, 987)
    x, y = synth.activations(64, K, 988).to(DEV), torch.empty((64, N), dtype=torch.float16, device=DEV)
    ws, spaces = ql.Workspace(64, K, N), [ql.Workspace(30, K, N) for _ in range(6)]
    rows = synth.activations(30, K, 989).float().numpy()
    want = ql.run(ws, w, x).clone()
    host = ql.run(spaces[0], w, torch.from_numpy(rows).to(DEV), out_dtype=torch.float32).cpu().numpy()
    torch.cuda.synchronize()
    got, meet = [], threading.Barrier(6)

    def work(space):
        meet.wait()
        got.append(ql.run_host_f32(space, w, rows))

    threads = [threading.Thread(target=work, args=(s,)) for s in spaces]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode=mode):
        ql.run(ws, w, x, out=y)
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert len(got) == 6 and all(np.array_equal(o, host) for o in got)
    for _ in range(2):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    for s in (ws, *spaces, w):
        s.close()


def test_host_runs_on_several_threads():
    """Six threads, a workspace each, more than the idle sets kept: every call gets its own rows."""
    K, N = 2560, 2560
    w = weights(4, K, N, 980)
    rows = [1, 40, 128, 300, 64, 7]
    spaces = [ql.Workspace(r, K, N) for r in rows]
    inputs = [synth.activations(r, K, 981 + r).float().numpy() for r in rows]
    want = [ql.run_host_f32(ws, w, a) for ws, a in zip(spaces, inputs)]
    wrong = []

    def work(i):
        for _ in range(10):
            if not np.array_equal(ql.run_host_f32(spaces[i], w, inputs[i]), want[i]):
                wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(rows))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for ws in spaces:
        ws.close()
    w.close()
