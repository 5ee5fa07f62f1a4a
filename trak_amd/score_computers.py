"""Score computer plug-in with the interface of the reference's trak/score_computers.py,
running the three GEMMs and the regularized inverse on the GPU through libtrakhip.

`TRAKer(score_computer=BasicScoreComputer)` constructs it as
`cls(dtype=, device=, logging_level=, lambda_reg=)` (trak/traker.py:186-193) and calls
`get_xtx`, `get_x_xtx_inv` and `get_scores` (trak/traker.py:483-485, :667).
"""
import logging
from abc import ABC, abstractmethod
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch
from torch import Tensor

from .utils import (
    gemm_nt,
    gemm_nt16,
    gemm_nt_split,
    gemm_tn,
    get_matrix_mult_blockwise,
    gram16,
    gram16_ok,
    gram_split,
    in_place_alike,
    in_place_pays,
    inverse_of_rejected,
    matmul_nt,
    nt16_ok,
    output_fits_on_device,
    scores_finalize,
    spd_inverse_unchecked,
    split2_rows,
    split_rows,
)

ch = torch


class AbstractScoreComputer(ABC):
    """Interface of trak/score_computers.py:22-91."""

    @abstractmethod
    def __init__(self, dtype, device) -> None:
        self.dtype = dtype
        self.device = device

    @abstractmethod
    def get_xtx(self, grads: Tensor) -> Tensor:
        """X^T X for projected gradients X of shape (n, p)."""

    @abstractmethod
    def get_x_xtx_inv(self, grads: Tensor, xtx: Tensor) -> Tensor:
        """X (X^T X)^-1 of shape (n, p)."""

    @abstractmethod
    def get_scores(self, features: Tensor, target_grads: Tensor, accumulator: Tensor) -> None:
        """accumulator (n, m) += features (n, p) @ target_grads (m, p)^T."""


class BasicScoreComputer(AbstractScoreComputer):
    """GPU implementation of the reference's BasicScoreComputer (trak/score_computers.py:119-189).

    All arithmetic has fp32 accuracy on the device; `dtype` is the type of the returned tensors,
    as in the reference.  Inputs may live on the host: they are moved block by block
    (CUDA_MAX_DIM_SIZE rows at a time), which is what the reference's `block.to(self.device)`
    does.

    `gemm` selects how the three matrix products are computed: "split" (default) splits every
    fp32 operand exactly into three bf16 terms and runs six bf16 MFMAs per k step with fp32
    accumulation (same error as the fp32 instruction, 1.7 times its speed); "fp32" uses the fp32
    MFMA instruction directly; "split2" is an opt-in cheaper split for fp32 operands (rows scaled by a
    power of two, two fp16 planes, three MFMAs per k step: entries keep 22 significand bits relative
    to their row's largest magnitude instead of all 24; 1.75 times the speed of "split").  fp16 / bf16
    operands are multiplied as they are (exact products) under "split" and "split2".  Under "split", products of few
    rows or columns read fp32 operands where they are, on the fp32 instruction (`utils.in_place_pays`); the order in which
    k is added up goes with the numbers of rows and columns, so the last bits of an fp32 row's features or scores may
    differ between calls of other sizes.  All rows of one `get_x_xtx_inv` are added up in one order.

    Differences from the reference that a caller can meet:
      * the device must be a GPU (the reference also runs on "cpu");
      * `X^T X + lambda I` is inverted by a Cholesky factorization.  When that fails - the matrix is
        symmetric but not positive definite, which happens to a Gram matrix that was rounded to fp16
        (TRAKer's default) or has deficient rank (fewer training points than proj_dim with
        lambda_reg = 0) - the matrix is inverted by this library's elimination with partial pivoting
        (`utils.general_inverse`: the pivoting of the LU behind the reference's torch.linalg.inv,
        trak/score_computers.py:163; matrices up to 12288 x 12288) and a warning is logged; an exactly
        singular matrix (a zero pivot) raises torch.linalg.LinAlgError as the reference's call does, an
        inverse with huge or non-finite entries is handed on as it is;
      * sums are kept in fp32 and rounded to `dtype` once.  accumulate_in_dtype=True reproduces the
        reference's arithmetic instead: `X^T X` is the sum over blocks of CUDA_MAX_DIM_SIZE rows of
        block products each rounded to `dtype`, the running sum rounded to `dtype` after every
        block (trak/score_computers.py:147-153), and lambda is added in the dtype of `xtx`
        (:160-162).  It costs one pass per block and only matters for fp16 / bf16 `dtype`.
    """

    def __init__(
        self,
        dtype: torch.dtype,
        device,
        CUDA_MAX_DIM_SIZE: int = 20_000,
        logging_level=logging.INFO,
        lambda_reg: float = 0.0,
        gemm: str = "split",
        accumulate_in_dtype: bool = False,
    ) -> None:
        super().__init__(dtype, device)
        self.accumulate_in_dtype = accumulate_in_dtype
        if gemm not in ("split", "split2", "fp32"):
            raise ValueError('gemm must be "split", "split2" or "fp32"')
        self.gemm = gemm
        self.CUDA_MAX_DIM_SIZE = CUDA_MAX_DIM_SIZE
        self.logger = logging.getLogger("ScoreComputer")
        self.logger.setLevel(logging_level)
        self.lambda_reg = lambda_reg
        dev = ch.device(device)
        if dev.type != "cuda":
            raise ValueError("BasicScoreComputer of trak_amd computes on a GPU; pass a cuda device")
        self._dev = dev

    def _blocks(self, grads):
        if grads.device == self._dev or (grads.is_cuda and self._dev.index is None):
            return [grads]  # resident: one pass, the kernel walks all rows
        return ch.split(grads, split_size_or_sections=self.CUDA_MAX_DIM_SIZE, dim=0)

    def _gram(self, block, out, beta):
        if self.gemm != "fp32" and gram16_ok(block):
            gram16(block, out=out, alpha=1.0, beta=beta)
        elif self.gemm != "fp32":
            # the operand is block^T, read in place; lower-triangle tiles + mirror image
            gram_split(self._split(block, transposed=True), out=out, alpha=1.0, beta=beta)
        else:
            gemm_tn(block, block, out=out, alpha=1.0, beta=beta)

    def get_xtx(self, grads: Tensor) -> Tensor:
        self.proj_dim = grads.shape[1]
        if self.accumulate_in_dtype:
            # trak/score_computers.py:147-153 to the letter: `result += block.T @ block` with both sides
            # in `dtype`, blocks of CUDA_MAX_DIM_SIZE rows wherever the gradients live
            result = ch.zeros(self.proj_dim, self.proj_dim, dtype=self.dtype, device=self._dev)
            product = ch.empty(self.proj_dim, self.proj_dim, dtype=ch.float32, device=self._dev)
            for block in ch.split(grads, split_size_or_sections=self.CUDA_MAX_DIM_SIZE, dim=0):
                self._gram(block.to(self._dev), product, 0.0)
                result += product.to(block.dtype)  # the block product in the gradients' type, as `block.T @ block` returns it
            return result
        blocks = self._blocks(grads)
        if len(blocks) == 1 and self.gemm != "fp32" and self.dtype in (ch.float16, ch.bfloat16):
            blocks = [blocks[0].to(self._dev)]
            if gram16_ok(blocks[0]):
                return gram16(blocks[0], out_dtype=self.dtype)
        result = ch.empty(self.proj_dim, self.proj_dim, dtype=ch.float32, device=self._dev)
        for i, block in enumerate(blocks):
            self._gram(block.to(self._dev), result, 0.0 if i == 0 else 1.0)
        return result.to(self.dtype)

    def get_x_xtx_inv(self, grads: Tensor, xtx: Tensor) -> Tensor:
        # (xtx + lambda I)^-1 in fp32, divided by the mean absolute entry
        # (trak/score_computers.py:160-166)
        xtx, lambda_reg = xtx.to(self._dev), self.lambda_reg
        if self.accumulate_in_dtype:
            # lambda is added in the dtype of xtx (trak/score_computers.py:160-162), then fp32
            xtx = xtx + lambda_reg * ch.eye(xtx.size(dim=0), device=xtx.device, dtype=xtx.dtype)
            lambda_reg = 0.0
        inverse, _, verdict = spd_inverse_unchecked(xtx, lambda_reg, normalize=True)
        result, pivot = self._times_inverse(grads, inverse.to(self.dtype), verdict)
        if pivot is not None:
            del inverse  # (what the first attempt held is given back before the elimination asks for its workspace)
            inverse, _ = inverse_of_rejected(xtx, pivot, lambda_reg, normalize=True)
            result, _ = self._times_inverse(grads, inverse.to(self.dtype))
        return result

    def _times_inverse(self, grads, xtx_inv, verdict=None):
        """(grads @ xtx_inv in `dtype`, None).  `verdict` (see `spd_inverse_unchecked`) is asked behind the product of the first rows,
        which runs while the host waits for the answer; a matrix that was not positive definite gives (None, pivot)."""
        # 16-bit gradients meet the inverse cast to their type (as in the reference) as single planes
        half = grads.dtype == xtx_inv.dtype and grads.dtype in (ch.float16, ch.bfloat16)
        # the sums of a product that reads both in place are rounded as they are stored
        result = ch.empty(grads.shape[0], xtx_inv.shape[1], dtype=self.dtype if half and self.gemm != "fp32" else ch.float32,
                          device=self._dev)
        inv_split = None  # planes of the inverse, made when the first block needs them
        in_place = None  # one route for all blocks of fp32 values: a row's sums do not depend on the block that holds it
        start = 0
        blocks = self._blocks(grads)
        resident = blocks[0] is grads
        if verdict is not None and resident:
            # What the host waits behind is in vain when the answer is bad: of a product of eight rounds of tiles or more, which
            # would add 6 % and more to the elimination, one round (64 us of fp16 rows by 2048 columns, 550 us of fp32 ones by
            # 4096; the rest is enqueued long before it ends).  In two pieces a product takes 9 us longer.
            head = _rows_of_a_round(xtx_inv.shape[1])
            if grads.shape[0] >= 8 * head:
                blocks = [grads[:head], grads[head:]]
        for block in blocks:
            end = start + block.shape[0]
            block = block.to(self._dev)
            if verdict is not None and not resident:  # (it has arrived before the block)
                pivot, verdict = verdict(), None
                if pivot is not None:
                    return None, pivot
            # the inverse is symmetric, so block @ inv == block @ inv^T
            if self.gemm != "fp32":
                if in_place is None:
                    in_place = (self.gemm == "split" and not half and in_place_pays(block, xtx_inv)
                                and (len(blocks) == 1 or in_place_alike({b.shape[0] for b in blocks}, *xtx_inv.shape)))
                if half and nt16_ok(block, xtx_inv):
                    gemm_nt16(block, xtx_inv, out=result[start:end])
                elif in_place:
                    gemm_nt(block, xtx_inv, out=result[start:end], in_place=True)
                else:
                    if inv_split is None:
                        inv_split = self._split(xtx_inv if half else xtx_inv.float())
                    if half:
                        result[start:end] = gemm_nt_split(self._split(block), inv_split)
                    else:
                        gemm_nt_split(self._split(block.float()), inv_split, out=result[start:end])
            else:
                gemm_nt(block, xtx_inv, out=result[start:end])
            start = end
            if verdict is not None:
                pivot, verdict = verdict(), None
                if pivot is not None:
                    return None, pivot
        return result.to(self.dtype), None

    def get_scores(self, features: Tensor, target_grads: Tensor, accumulator: Tensor) -> None:
        train_dim = features.shape[0]
        target_dim = target_grads.shape[0]
        self.logger.debug(f"{train_dim=}, {target_dim=}")
        f, t = features.to(self._dev), target_grads.to(self._dev)
        if (
            accumulator.is_cuda
            and accumulator.device == f.device
            and accumulator.dtype == ch.float32
            and accumulator.dim() == 2
            and accumulator.stride(1) == 1
        ):
            # accumulator on the GPU: the sum over checkpoints happens in the GEMM epilogue and the
            # [N, M] matrix never crosses PCIe per checkpoint (trak/traker.py:641-668 moves it each time)
            self._matmul_nt(f, t, out=accumulator, beta=1.0)
            return
        if not accumulator.is_cuda and not output_fits_on_device(train_dim, target_dim, self._dev):
            # too large for the device: block by block into the host accumulator (trak/utils.py:135-245)
            get_matrix_mult_blockwise(f, t, out=accumulator, accumulate=True,
                                      product=lambda a, b, o: self._matmul_nt(a, b, out=o))
            return
        scores = self._matmul_nt(f, t)
        if accumulator.is_cuda:
            accumulator += scores.to(accumulator.dtype)
        else:
            accumulator += scores.to(accumulator.dtype).detach().cpu()

    def get_scaled_scores(self, features: Tensor, target_grads: Tensor, out_to_loss: Tensor, scale: float = 1.0):
        """scale * (features @ target_grads^T) with row i multiplied by out_to_loss[i], on the
        device: the finalize_scores epilogue of trak/traker.py:670-678 fused into the GEMM."""
        return self._matmul_nt(
            features.to(self._dev), target_grads.to(self._dev), alpha=scale, row_scale=out_to_loss.reshape(-1)
        )

    def _split(self, t, transposed=False):
        """Operand format of the chosen product: 16-bit matrices stay one plane; fp32 ones become three
        exact bf16 planes ("split") or two scaled fp16 planes ("split2")."""
        if self.gemm == "split2" and t.dtype not in (ch.float16, ch.bfloat16):
            return split2_rows(t, transposed=transposed)
        return split_rows(t, transposed=transposed)

    def _matmul_nt(self, a, b, out=None, alpha=1.0, beta=0.0, row_scale=None):
        if self.gemm != "fp32":
            return matmul_nt(a, b, out=out, alpha=alpha, beta=beta, row_scale=row_scale,
                             two_planes=self.gemm == "split2")
        return gemm_nt(a, b, out=out, alpha=alpha, beta=beta, row_scale=row_scale)


def _rows_of_a_round(columns):
    """Rows of a product with this many columns whose 256 x 256 tiles occupy the 256 CUs once."""
    return 256 * max(1, 256 // max(1, -(-columns // 256)))


# The out_to_loss sums in half precision, in the arithmetic of numpy (values widened to fp32, one operation, rounded back),
# by torch: its conversions are vectorized and threaded (50 000 values: 124 -> 24 us the sum, 206 -> 38 us the quotient,
# both between a user's call and the launch that needs them).


def _add_half(sums, values):
    """sums += values for a float16 array and one of float16 or float32 of its shape."""
    if not values.flags.writeable:
        values = values.copy()  # (torch wants to be able to write)
    t = ch.from_numpy(sums)
    t.copy_(t.float().add_(ch.from_numpy(np.ascontiguousarray(values))))


def _row_factors(sums, n):
    """(sums / n).astype(np.float32) for a contiguous array of float16 or float32."""
    if sums.dtype != np.float16:
        return (sums / n).astype(np.float32)
    with np.errstate(over="ignore"):
        divisor = float(np.float16(n))  # a Python number meets an array in the array's type
    return (ch.from_numpy(sums).float() / divisor).half().float().numpy()


# Who copies a block of scores into the store, by the time of a whole `finalize` on the GPU's host (16 CPUs; 10 MB, 260 MB and
# 1 GB of fp16 scores).  Memory: torch's threads where there are as many as _COPY_THREADS or the block is small (16: 0.34, 5.4, 20.6 ms;
# four: 0.33, 5.9, 21.8; one: 0.44, 12.3, 47.5), else as many of our own (under OMP_NUM_THREADS=1: 6.0 and 21.6 ms).  A mapped file: one
# thread.  Its pages are new when scores are written, and threads that ask for them wait for one another (one: 3.1, 31, 114 ms; four
# of our own 4-10, 75-100, 200-300; torch's sixteen 9-10, 151-156, 445-466; written a second time: 0.6, 11, 40-48 ms).
_COPY_THREADS = 4
_COPY_BYTES = 16 << 20


def _in_memory(out):
    """Whether this is an array in memory.  A mapped file is not; and the slices of other kinds of array (in a file, masked, ...) may
    be copies, in which what is written is lost."""
    if type(out) is not np.ndarray:
        return False
    base = out.base
    while isinstance(base, np.ndarray) and not isinstance(base, np.memmap):
        base = base.base
    return not isinstance(base, np.memmap)


def _own_threads(out, block_bytes):
    return block_bytes >= _COPY_BYTES and ch.get_num_threads() < _COPY_THREADS and _in_memory(out)


def _store_rows(out, r0, r1, src, pool=None):
    """out[r0:r1] = src (a CPU tensor), by the _COPY_THREADS threads of `pool` if it is given."""
    if pool is not None:
        values, step = src.numpy(), -(-(r1 - r0) // _COPY_THREADS)

        def assign(at):
            out[r0 + at : min(r1, r0 + at + step)] = values[at : at + step]

        list(pool.map(assign, range(0, r1 - r0, step)))
    # (torch takes no steps backwards or by parts of an element, as a field of records has them)
    elif _in_memory(out) and out.flags.behaved and all(s >= 0 and s % out.itemsize == 0 for s in out.strides):
        ch.from_numpy(out[r0:r1]).copy_(src)
    else:
        out[r0:r1] = src.numpy()


class ScoreAccumulator:
    """The checkpoint loop of TRAKer.finalize_scores (trak/traker.py:641-678) with the score sums
    kept on the GPU.

    The reference adds every checkpoint's [N, M] score matrix into a CPU tensor (one device-to-host
    copy of the whole matrix per checkpoint) and evaluates
    `(_scores / n) * (_avg_out_to_losses / n)` with numpy at the end.  Here `add` accumulates in the
    GEMM epilogue on the device, the out_to_loss sums stay a small host array exactly as in the
    reference, and `finalize` applies the same expression on the device while the matrix is
    written, chunk by chunk through page-locked memory, into the scores store: one crossing of
    PCIe in total.

    Args:
        score_computer: a BasicScoreComputer of this package.
        train_set_size, num_targets: N and M.
        dtype: torch.float16 or torch.float32, the saver's element type (trak/traker.py:127); it
            fixes the type the out_to_loss sums are kept in, as in the reference.
    """

    def __init__(self, score_computer, train_set_size, num_targets, dtype=ch.float32):
        self.score_computer = score_computer
        self.shape = (int(train_set_size), int(num_targets))
        self.dtype = dtype
        self._acc = ch.zeros(self.shape, dtype=ch.float32, device=score_computer._dev)
        self._out_to_loss = np.zeros(
            (self.shape[0], 1), dtype=np.float16 if dtype == ch.float16 else np.float32
        )
        self.num_models = 0

    def add(self, features, target_grads, out_to_loss) -> None:
        """One checkpoint: sums += features @ target_grads^T (trak/traker.py:667) and
        out_to_loss sums += out_to_loss (trak/traker.py:670)."""
        self.score_computer.get_scores(features, target_grads, accumulator=self._acc)
        o = out_to_loss.detach().cpu().numpy() if isinstance(out_to_loss, Tensor) else np.asarray(out_to_loss)
        o = o.reshape(self.shape[0], 1)
        if self._out_to_loss.dtype == np.float16 and o.dtype in (np.float16, np.float32):
            _add_half(self._out_to_loss, o)
        else:
            self._out_to_loss += o
        self.num_models += 1

    def finalize(self, out, chunk_bytes: int = 256 << 20):
        """Writes `(sums / n) * (out_to_loss sums / n)` (trak/traker.py:674-676) into `out`, the
        [N, M] array behind the saver's `<exp>_scores` store (numpy array or memmap of float16 or
        float32) or a tensor (CUDA, or page-locked CPU).  Returns `out`."""
        if self.num_models == 0:
            raise ValueError("no checkpoint was added")
        n = float(self.num_models)
        # the second factor exactly as numpy computes it in the reference, then widened (exact)
        row_factor = _row_factors(self._out_to_loss, n).reshape(-1)
        row_factor = ch.from_numpy(row_factor).to(self._acc.device)
        N, M = self.shape
        if isinstance(out, Tensor):
            scores_finalize(self._acc, n, row_factor, out)
            if not out.is_cuda:
                ch.cuda.current_stream(self._acc.device).synchronize()
            return out
        if tuple(out.shape) != (N, M) or out.dtype not in (np.float16, np.float32):
            raise ValueError(f"out must be a [{N}, {M}] array of float16 or float32")
        tdtype = ch.float16 if out.dtype == np.float16 else ch.float32
        row_bytes = max(1, M * out.dtype.itemsize)
        # four chunks of at least 1 MB or more of them: the copy of one into the store passes under the next one's crossing
        rows = max(1, min(N, int(chunk_bytes) // row_bytes, max(-(-N // 4), (1 << 20) // row_bytes)))
        stage = [ch.empty((rows, M), dtype=tdtype, device="cpu", pin_memory=True) for _ in range(2 if rows < N else 1)]
        pending = [None] * len(stage)
        pool = ThreadPoolExecutor(_COPY_THREADS) if _own_threads(out, rows * row_bytes) else None
        stream = ch.cuda.current_stream(self._acc.device)

        def retire(i):
            if pending[i] is None:
                return
            event, r0, r1 = pending[i]
            event.synchronize()
            _store_rows(out, r0, r1, stage[i][: r1 - r0], pool)
            pending[i] = None

        try:
            for index, r0 in enumerate(range(0, N, rows)):
                i = index % len(stage)
                retire(i)
                r1 = min(N, r0 + rows)
                scores_finalize(self._acc[r0:r1], n, row_factor[r0:r1], stage[i][: r1 - r0])
                event = ch.cuda.Event()
                event.record(stream)
                pending[i] = (event, r0, r1)
            for i in range(len(stage)):
                retire((index + 1 + i) % len(stage))
        finally:
            if pool is not None:
                pool.shutdown()
        return out
