"""Which B an input-gradient GEMM reads (CPU only): the weight as stored where the vector
loaders take both operands, its K-contiguous copy from TRANSPOSE_MIN_ROWS rows of A on where
the product falls to the generic kernel."""
import pytest
import torch

from ops import fused_execution as fx

BF16 = torch.bfloat16


@pytest.fixture(autouse=True)
def copies(monkeypatch):
    monkeypatch.setattr(fx, "transpose", lambda x: x.T.contiguous())


def _a(kind, rows, k):
    if kind == "aligned":
        return torch.empty(rows, k, dtype=BF16)
    if kind == "padded":
        return torch.empty(rows, k + 8, dtype=BF16)[:, :k]
    if kind == "odd stride":
        return torch.empty(rows, k + 1, dtype=BF16)[:, :k]
    if kind == "odd address":
        return torch.empty(rows * k + 8, dtype=BF16)[1:1 + rows * k].view(rows, k)
    if kind == "every other column":
        return torch.empty(rows, 2 * k, dtype=BF16)[:, ::2]
    return torch.empty(k, rows, dtype=BF16).T  # token-major


@pytest.mark.parametrize("kind,rows,k,direct", [
    ("aligned", 2048, 64, True), ("padded", 2048, 64, True), ("aligned", 16376, 64, True),
    ("aligned", 16384, 64, False), ("token-major", 2048, 64, True),
    ("token-major", 16384, 64, True), ("token-major", 2047, 64, False),
    ("aligned", 2048, 65, False), ("aligned", 2048, 60, False), ("odd stride", 2048, 64, False),
    ("odd address", 2048, 64, False), ("every other column", 2048, 64, False)])
def test_weight_is_copied_where_the_generic_kernel_reads_it(kind, rows, k, direct):
    weight = torch.empty(k, 128, dtype=BF16)  # [K, N], N-contiguous
    b = fx.gemm_b(_a(kind, rows, k), weight)
    assert b.shape == weight.shape
    assert (b is weight) == direct
    if not direct:
        assert b.stride(0) == 1


def test_weight_is_copied_for_outputs_off_16_byte_pieces():
    a, weight = _a("aligned", 2048, 64), torch.empty(64, 128, dtype=BF16)
    assert fx.gemm_b(a, weight, vector_out=False).stride(0) == 1


@pytest.mark.parametrize("rows", [1, 1023])
def test_few_rows_never_pay_for_a_copy(rows):
    weight = torch.empty(65, 128, dtype=BF16)
    assert fx.gemm_b(_a("aligned", rows, 65), weight) is weight


@pytest.mark.parametrize("rows,d,vocab,kind,stored,copied", [
    (2048, 64, 1024, "aligned", False, True), (1023, 64, 1024, "aligned", False, False),
    (2048, 64, 1027, "aligned", False, False), (2048, 64, 1028, "aligned", False, False),
    (2048, 64, 1028, "aligned", True, True), (2048, 60, 1027, "aligned", False, True),
    (2048, 64, 1027, "odd stride", False, True), (2048, 64, 1027, "odd address", False, True)])
def test_head_weight_is_copied_where_a_kernel_reads_the_copy(rows, d, vocab, kind, stored, copied):
    """A vocabulary off multiples of 8 with vector operands has padded chunk rows and no copy;
    with any other operands the generic kernel takes it."""
    weight = torch.empty(vocab, d, dtype=BF16)
    copy = fx._head_weight_t(_a(kind, rows, d), weight, stored)
    assert (copy is not None) == copied
    assert copy is None or copy.shape == (d, vocab)
