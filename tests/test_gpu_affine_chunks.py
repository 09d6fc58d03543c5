"""The right-affine scan over its split: one chunk and several, whole and partial blocks of steps, every matrix
size the kernel is built for and those between, inputs off the 16-byte grid. The oracle runs in fp64. Bound: a
step adds (D + 2) 2^-24 of its result, the states shrink by about 0.95 a step, so 20 steps' worth adds up: 8e-5."""

import pytest
import torch

import atlas_rnn_amd as am
from _cases import compare
from oracle import affine_scan_sequential

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.mark.parametrize("N,T,R,D,with_prev,offset", [
    (40, 9, 64, 64, True, 0),      # one chunk: the rows fill half the card
    (2, 130, 64, 64, True, 0),     # several chunks, the last one partial
    (2, 131, 17, 64, False, 1),    # rows off the 16-row blocks; inputs 4 bytes off the 16-byte grid
    (5, 97, 33, 48, True, 3),
    (3, 260, 64, 32, True, 0),
    (4, 101, 5, 32, False, 1),
    (9, 75, 64, 16, True, 0),
    (2, 39, 17, 16, False, 2),
    (2, 88, 40, 63, True, 1),      # sizes the kernel is not built for
    (3, 45, 3, 20, True, 0),
    (1, 2, 1, 1, True, 0),
    (1, 700, 2, 64, True, 0),      # many chunks
])
def test_affine_chunks(N, T, R, D, with_prev, offset):
    print(f"affine chunks N={N} T={T} R={R} D={D} prev={with_prev} offset={offset}", flush=True)
    g = torch.Generator().manual_seed(N * 1000 + T)
    A = 0.9 * torch.eye(D) + 0.3 * torch.randn(N, T, D, D, generator=g) / D ** 0.5
    B = torch.randn(N, T, R, D, generator=g)
    prev = torch.randn(N, R, D, generator=g) if with_prev else None
    gout = torch.randn(N, T, R, D, generator=g)
    ins = [t.to(F64).requires_grad_() if t is not None else None for t in (A, B, prev)]
    ref = affine_scan_sequential(ins[0], ins[1], prev=ins[2], remove_prev=True)
    rg = torch.autograd.grad((ref * gout.to(F64)).sum(), [t for t in ins if t is not None])

    def place(t):
        buf = torch.empty(t.numel() + offset, device="cuda")
        v = buf[offset:].view(t.shape)
        v.copy_(t)
        return v.requires_grad_()

    dev = [place(t) if t is not None else None for t in (A, B, prev)]
    out = am.affine_associative_scan(dev[0], dev[1], prev=dev[2], remove_prev=True)
    gg = torch.autograd.grad(out, [t for t in dev if t is not None], gout.cuda())
    compare("affine.out", out.detach().cpu(), ref.detach(), 8e-5)
    for nm, a, b in zip(("dA", "dB", "dprev"), gg, rg):
        compare(f"affine.{nm}", a.cpu(), b, 8e-5)


@pytest.mark.parametrize("N,T,R,D,with_prev,offset", [
    (2, 37, 5, 3, True, 1),        # rows shorter than a group of four
    (3, 50, 2, 2, False, 0),
    (2, 41, 17, 4, True, 1),       # one group a row
    (2, 60, 64, 5, True, 0),       # a row's last group holds one, two and three of its elements
    (3, 33, 16, 6, False, 2),
    (2, 70, 33, 7, True, 3),
    (4, 90, 64, 61, True, 1),
    (40, 20, 64, 62, True, 0),     # one chunk
    (16, 130, 64, 60, True, 0),
    (3, 129, 64, 50, True, 2),
])
def test_affine_sizes_between(N, T, R, D, with_prev, offset):
    test_affine_chunks(N, T, R, D, with_prev, offset)
