"""Kernel variants at the sizes where they can go wrong: edges of tiles, remainders, the smallest and largest of a range."""
import pytest
import torch

from helpers import assert_close_rel, bf16_round
from oracle import ops as O

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def dev():
    return torch.device("cuda:0")


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("M,N,K,R", [(1, 1, 4, 0), (64, 64, 32, 32), (65, 63, 36, 4), (31, 130, 100, 36), (200, 70, 644, 128), (129, 640, 640, 32)])
def test_lora_linear_f32_matrix_kernel(M, N, K, R):
    """kh_lora_linear_split_f32: ragged tiles in every dimension, column counts that are no multiple of 4, all K remainders."""
    from katz_amd import ops

    say("lora_linear_split_f32", M, N, K, R)
    g = torch.Generator().manual_seed(M + N)
    x, w, b, res = (torch.randn(*s, generator=g) for s in ((M, K), (N, K), (N,), (M, N)))
    A, Bm = (torch.randn(R, K, generator=g) * 0.1, torch.randn(N, R, generator=g) * 0.1) if R else (None, None)
    d = dev()
    on = lambda t: None if t is None else t.to(d)
    y = ops.lora_linear(on(x), on(w), on(b), on(A), on(Bm), torch.full((R,), 1.5, device=d) if R else None, residual=on(res))
    torch.cuda.synchronize()
    ref = O.lora_linear(x.double(), w.double(), b.double(), [(A.double(), Bm.double(), 1.5)] if R else [], res.double()).float()
    assert_close_rel(y, ref, 1e-5, "fp32 linear")


def test_upload_many_sizes():
    """kh_upload_many: arrays smaller and larger than a staging half, empty gaps, one array, bit for bit."""
    from katz_amd import ops

    say("upload many")
    g = torch.Generator().manual_seed(1)
    for sizes in ([1], [3, 5, 1 << 20, 7], [(9 << 20) + 13, 1, (3 << 20) + 1], [257] * 300):
        src = [torch.randint(0, 256, (n,), generator=g, dtype=torch.uint8) for n in sizes]
        buf, at = ops.upload_many(src, dev())
        torch.cuda.synchronize()
        for t, a in zip(src, at):
            o = a - buf.data_ptr()
            assert torch.equal(buf[o:o + t.numel()].cpu(), t), sizes
