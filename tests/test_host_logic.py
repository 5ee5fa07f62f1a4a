"""Host-side mirror of the reference's projector helpers (no GPU needed)."""
import numpy as np
import pytest
import torch

from trak_amd import ChunkedCudaProjector, CudaProjector, NoOpProjector, ProjectionType, fast_jl, vectorize
from trak_amd.utils import chunk_sizes_from_numels, get_matrix_mult, get_parameter_chunk_sizes


def test_projection_type_enum():
    # trak/projectors.py:25-27
    assert ProjectionType.normal.value == "normal" and ProjectionType.rademacher.value == "rademacher"
    assert ProjectionType("normal") is ProjectionType.normal and isinstance(ProjectionType.normal, str)


def test_vectorize_dict_order_and_low_rank_params():
    # trak/utils.py:80-110: dict order, params with < 2 dims become one column
    g = {
        "w": torch.arange(2 * 3 * 4, dtype=torch.float32).reshape(2, 3, 4),
        "s": torch.tensor([100.0, 200.0]),
        "b": torch.arange(2 * 5, dtype=torch.float32).reshape(2, 5) + 1000,
    }
    out = vectorize(g, device="cpu")
    assert out.shape == (2, 12 + 1 + 5)
    assert torch.equal(out[:, :12], g["w"].reshape(2, 12))
    assert torch.equal(out[:, 12], g["s"])
    assert torch.equal(out[:, 13:], g["b"])
    arr = torch.zeros(2, 18)
    assert vectorize(g, arr=arr, device="cpu") is arr and torch.equal(arr, out)


def test_chunk_sizes_follow_the_uint32_rule():
    # trak/utils.py:297-331: max_chunk_size = uint32.max // batch_size, greedy grouping
    mx, per = chunk_sizes_from_numels([10, 20, 30], 32)
    assert mx == 4294967295 // 32 == 134217727 and per == [60]
    sizes = [60_000_000, 60_000_000, 60_000_000, 5]
    mx, per = chunk_sizes_from_numels(sizes, 32)
    assert per == [120_000_000, 60_000_005] and sum(per) == sum(sizes)
    mx, per = chunk_sizes_from_numels([100, 100], 4294967295 // 150)
    assert mx == 150 and per == [100, 100]
    model = torch.nn.Sequential(torch.nn.Linear(10, 7), torch.nn.Linear(7, 3))
    mx, per = get_parameter_chunk_sizes(model, 8)
    assert mx == 4294967295 // 8 and per == [10 * 7 + 7 + 7 * 3 + 3]


def test_cuda_projector_rejects_cpu_device():
    # trak/projectors.py:363-365
    with pytest.raises(ValueError, match="only works on a CUDA device"):
        CudaProjector(grad_dim=10, proj_dim=512, seed=0, proj_type=ProjectionType.rademacher, device="cpu", max_batch_size=8)


def test_noop_projector():
    p = NoOpProjector()
    g = torch.randn(3, 7)
    assert p.project(g, model_id=0) is g
    p.free_memory()


def test_fast_jl_namespace_and_input_checks():
    # the six entry points of fast_jl/fast_jl.cu:102-110
    for t in ("rademacher", "normal"):
        for n in (8, 16, 32):
            assert callable(getattr(fast_jl, f"project_{t}_{n}"))
    x = torch.zeros(8, 1000)
    with pytest.raises(RuntimeError, match="CUDA tensor"):   # fast_jl/fast_jl.cu:21
        fast_jl.project_rademacher_8(x, 512, 0, 256)


def test_get_matrix_mult_cpu_path_is_plain_matmul():
    a, b = torch.randn(5, 8), torch.randn(3, 8)
    out = get_matrix_mult(a, b)
    assert out.shape == (5, 3) and torch.allclose(out, a @ b.t())


def test_chunked_projector_bookkeeping_with_a_fake_chunk_projector():
    # packing order, flush rule and summation of trak/projectors.py:470-516, checked on the CPU
    # with a stand-in for the per-chunk projector
    class Fake:
        proj_dim, proj_type = 4, ProjectionType.rademacher

        def __init__(self, scale):
            self.scale, self.seen = scale, []

        def project(self, grads, model_id):
            self.seen.append(grads.clone())
            return torch.full((grads.shape[0], 4), float(grads.sum()) * self.scale)

    fakes = [Fake(1.0), Fake(10.0)]
    proj = ChunkedCudaProjector(fakes, max_chunk_size=7, params_per_chunk=[7, 4], feat_bs=3, device="cpu", dtype=torch.float32)
    g = {"a": torch.ones(2, 2, 2), "b": torch.ones(2, 2) * 2, "c": torch.ones(2) * 3, "d": torch.ones(2, 4) * 5}
    out = proj.project(g, model_id=0)
    assert out.shape == (2, 4)
    assert fakes[0].seen[0].shape == (2, 7) and fakes[1].seen[0].shape == (2, 4)
    assert torch.equal(fakes[0].seen[0][0], torch.tensor([1.0, 1, 1, 1, 2, 2, 3]))
    assert torch.equal(fakes[1].seen[0][0], torch.tensor([5.0, 5, 5, 5]))
    assert torch.allclose(out, torch.full((2, 4), 2 * 11.0 + 10 * 2 * 20.0))
    proj.free_memory()
    assert not proj.input_allocated


def test_out_to_loss_sums_in_half_precision_are_numpys():
    import warnings

    from trak_amd.score_computers import _add_half, _row_factors, _store_rows

    every = np.arange(1 << 16, dtype=np.uint32).astype(np.uint16).view(np.float16)      # subnormals, infinities, NaN
    rng = np.random.default_rng(0)
    same = lambda a, b: np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a[a == 0]), np.signbit(b[b == 0]))
    with warnings.catch_warnings(), np.errstate(all="ignore"):
        warnings.simplefilter("ignore")
        for values in (rng.permutation(every), (rng.standard_normal(1 << 16) * 1e-3).astype(np.float32),
                       (10.0 ** rng.uniform(-9, 6, 1 << 16)).astype(np.float32)):
            got, want = every.copy().reshape(-1, 1), every.copy().reshape(-1, 1)
            values = values.reshape(-1, 1)
            values.flags.writeable = False                                                # as a store opened for reading gives them
            _add_half(got, values)
            want += values
            assert got.dtype == np.float16 and same(got, want)
        for n in (1.0, 2.0, 3.0, 7.0, 50.0, 2049.0, 65504.0, 70000.0):
            for sums in (every.reshape(-1, 1), rng.standard_normal((1000, 1)).astype(np.float32)):
                got = _row_factors(sums.copy(), n)
                assert got.dtype == np.float32 and same(got, (sums / n).astype(np.float32))
    src = torch.arange(12.0).reshape(3, 4)
    for out in (np.zeros((5, 4), np.float32), np.zeros((5, 8), np.float32)[:, ::2], np.zeros((5, 4), np.float32)[:, ::-1]):
        _store_rows(out, 1, 4, src)
        assert np.array_equal(out[1:4], src.numpy()) and not out[[0, 4]].any()
    fixed = np.zeros((5, 4), np.float32)
    fixed.flags.writeable = False
    with pytest.raises(ValueError):
        _store_rows(fixed, 1, 4, src)


@pytest.mark.parametrize("kind", [[("score", "f2"), ("flag", "u1")], [("flag", "u1"), ("score", "f4")], [("flag", "u1"), ("score", "f2"), ("pad", "u1")]])
def test_scores_into_a_field_of_records(kind, tmp_path):
    from trak_amd.score_computers import _store_rows

    # steps of 3, 5 and 4 bytes; an aligned start and two that are not
    src = torch.arange(12.0).reshape(3, 4)
    mapped = np.memmap(tmp_path / "records", mode="w+", dtype=kind, shape=(5, 4))
    for records in (np.zeros((5, 4), kind), mapped):
        out = records["score"]
        _store_rows(out, 1, 4, src.to(torch.float16 if out.dtype == np.float16 else torch.float32))
        assert np.array_equal(out[1:4], src.numpy()) and not out[[0, 4]].any() and not records["flag"].any()


def test_scores_into_arrays_whose_slices_are_copies():
    from trak_amd.score_computers import _store_rows

    class Stored:  # as an array in a file: reading gives a copy, assignment writes
        def __init__(self, shape, dtype):
            self.data, self.shape, self.dtype = np.zeros(shape, dtype), shape, np.dtype(dtype)

        def __getitem__(self, at):
            return self.data[at].copy()

        def __setitem__(self, at, value):
            self.data[at] = value

    src = torch.arange(12.0).reshape(3, 4)
    stored = Stored((5, 4), np.float32)
    _store_rows(stored, 1, 4, src)
    assert np.array_equal(stored.data[1:4], src.numpy()) and not stored.data[[0, 4]].any()
    masked = np.ma.masked_all((5, 4), np.float32)
    _store_rows(masked, 1, 4, src)
    assert np.array_equal(masked[1:4].filled(-1.0), src.numpy()) and masked[[0, 4]].mask.all()


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 9])
def test_scores_into_memory_by_our_own_threads_and_into_files_by_one(rows, tmp_path, monkeypatch):
    from concurrent.futures import ThreadPoolExecutor

    from trak_amd import score_computers as m

    src = torch.arange(4.0 * rows).reshape(rows, 4)
    memory = np.zeros((rows + 2, 4), np.float32)
    mapped = np.lib.format.open_memmap(tmp_path / "scores.npy", mode="w+", dtype=np.float32, shape=(rows + 2, 4))
    monkeypatch.setattr(m.ch, "get_num_threads", lambda: 1)
    assert m._own_threads(memory, m._COPY_BYTES) and not m._own_threads(memory, m._COPY_BYTES - 1)
    for out in (mapped, np.asarray(mapped), mapped[:, ::2]):
        assert not m._in_memory(out) and not m._own_threads(out, m._COPY_BYTES)
    monkeypatch.setattr(m.ch, "get_num_threads", lambda: m._COPY_THREADS)
    assert not m._own_threads(memory, m._COPY_BYTES)
    with ThreadPoolExecutor(m._COPY_THREADS) as pool:
        for out, p in ((memory, pool), (mapped, None)):
            m._store_rows(out, 1, rows + 1, src, p)
            assert np.array_equal(out[1:-1], src.numpy()) and not out[[0, -1]].any()
        memory.flags.writeable = False
        with pytest.raises(ValueError):                                                  # what a thread raises is raised
            m._store_rows(memory, 1, rows + 1, src, pool)
