"""The native id-list pass and the packed rows: the same arrays and refusals as the general Python path."""
import threading

import numpy as np
import pytest
import torch

import qwen_warp_amd as q
from qwen_warp_amd import _lib
from qwen_warp_amd import sampling as _sampling
from qwen_warp_amd.sampling import _ids

V = 1000


@pytest.mark.parametrize("n", [0, 1, 7, 5000])
@pytest.mark.parametrize("kind", [list, tuple])
def test_ids_native_pass(n, kind):
    want = np.random.default_rng(n).integers(0, V, n)
    got = _ids(kind(want.tolist()), V, "gen")
    assert got.dtype == np.int64 and np.array_equal(got, want)
    assert np.array_equal(_ids(kind(list(want)), V, "gen"), want)  # numpy integers: the general path


@pytest.mark.parametrize("bad", [-1, V, 2 ** 31, 2 ** 70, True, 1.0, "1", None, np.bool_(True), np.float32(1)])
def test_ids_refusals(bad):
    for at in (0, 3):
        ids = [1, 2, 3, 4]
        ids[at] = bad
        assert _lib.hostpack().ids(ids, V, np.empty(4, np.int64)) == -1
        with pytest.raises(q.ValidationError):
            _ids(ids, V, "gen")


@pytest.mark.parametrize("file", [None, b"not an extension"])
def test_without_the_native_module(file, tmp_path, monkeypatch):
    """A checkout without the module, or with one this interpreter cannot load: the general path, with the same rows and refusals."""
    rows = [q.RowSpec(gen=[1, 2, 2], drafts=(3,), bias={4: 0.5}, stop=[6], min_tokens=9, allowed=[1, 33], repetition=1.1), q.RowSpec(prompt=[V - 1], presence=1.0)]
    want = q.PackedBatch(rows, V, "cpu").dev_buf
    path = tmp_path / _lib.HOSTPACK_PATH.name
    if file:
        path.write_bytes(file)
    monkeypatch.setattr(_lib, "HOSTPACK_PATH", path)
    monkeypatch.setattr(_lib, "_HOSTPACK", None)
    with pytest.warns(RuntimeWarning, match="packed in Python"):
        assert _lib.hostpack() is None
    assert torch.equal(q.PackedBatch(rows, V, "cpu").dev_buf, want) and _ids([], V, "gen").size == 0
    for bad in (-1, V, 2 ** 70, True, 1.0, "1"):
        with pytest.raises(q.ValidationError):
            _ids([1, bad], V, "gen")


def test_ids_buffer_too_small():
    assert _lib.hostpack().ids([1, 2, 3], V, np.empty(2, np.int64)) == -1


def test_packed_rows_fields():
    """The row words as the ctypes structure holds them, a value past its C field included (as the structure converts it)."""
    rows = [q.RowSpec(temperature=0.7, top_k=2 ** 32 + 5, top_p=0.9, min_p=0.1, seed=-1, position=2 ** 33 + 1, row_key=-2, presence=1e39, gen=[1, 2], drafts=[3],
                      bias={4: 0.5, 5: -1.0}, stop=[6, 7], min_tokens=9),
            q.RowSpec(temperature=1.0, gen=[8, 9], repetition=1.5, allowed=[1, 33])]
    p = q.PackedBatch(rows, V, "cpu")
    a, b = p.host_rows[0], p.host_rows[1]
    assert a.top_k == 5 and a.seed == 2 ** 64 - 1 and a.position == 1 and a.row_key == 2 ** 32 - 2 and a.presence == np.inf and a.proc_on == 1
    assert (a.hist_off, a.n_prompt, a.n_gen, a.draft_off, a.n_drafts, a.bias_off, a.n_bias, a.stop_off, a.n_stop, a.ngen) == (0, 0, 2, 0, 1, 0, 2, 0, 2, 2)
    assert (b.hist_off, b.n_gen, b.draft_off, b.mask_mode, b.mask_row, b.state_slot) == (2, 2, 1, _lib.MASK_ALLOWED, 0, -1)
    assert bytes(p.host_rows) == p.rows_t.numpy().tobytes()
    assert p.hist_t.tolist() == [1, 2, 8, 9] and p.bids_t.tolist() == [4, 5] and p.bvals_t.tolist() == [0.5, -1.0] and p.stops_t.tolist() == [6, 7]
    assert p.masks_t[0].tolist()[:2] == [2, 2]
    with pytest.raises(ValueError):
        q.PackedBatch([q.RowSpec(banned=np.zeros(3, np.uint32))], V, "cpu")


@pytest.mark.parametrize("shape", [(1, -1), (-1, 1), (4, -1), (2, -1, 1)])
def test_masks_of_other_shapes(shape):
    """A banned mask of the right number of words is taken in any shape, the same one on every masked row."""
    words = np.random.default_rng(1).integers(0, 1 << 32, 32, dtype=np.uint32)
    flat = q.PackedBatch([q.RowSpec(banned=words), q.RowSpec(), q.RowSpec(banned=~words)], V, "cpu")
    p = q.PackedBatch([q.RowSpec(banned=words.reshape(shape)), q.RowSpec(), q.RowSpec(banned=~words.reshape(shape))], V, "cpu")
    assert torch.equal(p.masks_t, flat.masks_t) and torch.equal(p.dev_buf, flat.dev_buf)
    assert np.array_equal(p.masks_t.numpy().view(np.uint32), np.stack([words, ~words]))
    for rows in ([q.RowSpec(banned=words.reshape(shape)), q.RowSpec(banned=words)], [q.RowSpec(banned=words[:31])], [q.RowSpec(banned=words), q.RowSpec(banned=words[None, :31])]):
        with pytest.raises(ValueError):
            q.PackedBatch(rows, V, "cpu")


@pytest.mark.parametrize("dev,capturing,want", [("cpu", False, False), ("cuda", False, True), ("cuda:0", False, True), ("cuda:1", False, False),
                                                ("cuda", True, False), ("cuda:0", True, False), ("cuda:1", True, False)])
def test_copies_left_unwaited(dev, capturing, want, monkeypatch):
    """Only to the current device (0 here), whose stream's capture state is the one that is asked for, and not under capture."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    copied = []
    monkeypatch.setattr(torch, "empty", lambda n, dtype, pin_memory: copied.append(True) or torch.zeros(n, dtype=dtype))
    monkeypatch.setattr(torch.Tensor, "to", lambda t, d, non_blocking=False: copied.append(non_blocking) or t)
    monkeypatch.setattr(_sampling, "_capture_mode", lambda mode: 0)
    q.PackedBatch([q.RowSpec()], V, dev, ordered=True)
    assert copied == [True, True] if want else copied == [False]


@pytest.mark.gpu
def test_ordered_copies_back_to_back(sampler):
    """Calls that pack their own rows, issued without waiting: each runs on its own rows (staging buffers are not reused early)."""
    Vg = 8 * 4096
    g = torch.Generator().manual_seed(1)
    x = torch.randn(4, Vg, generator=g).cuda()
    batches = [[q.RowSpec(temperature=1.0, top_p=0.9, repetition=1.3, gen=torch.randint(0, Vg, (2000,), generator=g).tolist(), seed=i, row_key=b) for b in range(4)]
               for i in range(24)]
    want = [sampler.run(q.PackedBatch(rows, Vg, "cuda"), x).tolist() for rows in batches]
    got = [sampler.sample(x, rows) for rows in batches]
    assert [t.tolist() for t in got] == want


@pytest.mark.gpu
@pytest.mark.parametrize("own_stream", [False, True])
def test_packing_while_another_thread_captures(sampler, own_stream):
    """Calls that pack their own rows, on one thread, while another captures a graph of the same library: both go on."""
    Vg = 8 * 4096
    x = torch.randn(4, Vg, generator=torch.Generator().manual_seed(1)).cuda()
    rows = [q.RowSpec(temperature=1.0, top_p=0.9, seed=i, row_key=i) for i in range(4)]
    other = [[q.RowSpec(temperature=1.0, top_p=0.9, repetition=1.2, gen=list(range(n + own_stream)), seed=i, row_key=i) for i in range(4)]
             for n in (100, 3000, 20000, 3000)]  # staging buffers of several sizes: taken anew, and again
    packed, out = q.PackedBatch(rows, Vg, "cuda"), torch.empty(4, dtype=torch.int32, device="cuda")
    want, graph_sampler = sampler.run(packed, x).tolist(), q.Sampler("cuda")
    stream, side, graph = torch.cuda.Stream() if own_stream else torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    capturing, packed_all, got = threading.Event(), threading.Event(), []

    def serve():
        try:
            capturing.wait(30)
            with torch.cuda.stream(stream):
                got.extend(sampler.sample(x, r) for r in other)
        except Exception as e:
            got.append(e)
        packed_all.set()

    t = threading.Thread(target=serve)
    t.start()
    with torch.cuda.stream(side):
        graph_sampler.run(packed, x, out_tokens=out)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            capturing.set()
            packed_all.wait(30)
            graph_sampler.run(packed, x, out_tokens=out)
    t.join(30)
    torch.cuda.synchronize()
    assert [g.tolist() for g in got] == [sampler.run(q.PackedBatch(r, Vg, "cuda"), x).tolist() for r in other]
    for _ in range(3):
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert out.tolist() == want
