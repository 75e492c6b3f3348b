"""Edges of the aggregator's blocks (128 rows, 128 // K whole samples each, waves
of 32 rows): against the fp32 torch restatement, within the tolerances of
test_gpu_aggregator.py (the same bf16 roundings), and its two ways of copying
weights against each other, bit for bit."""
import ctypes

import pytest
import torch

import epcq.csrc as C
from aggregator_ref import random_inputs
from scenes import bits
from test_gpu_aggregator import check, module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 2, 7, 9, 31, 32])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_block_edges(dev, K, extra):
    M = max(1, 3 * (128 // K) + extra)
    print(f"aggregator blocks K={K} M={M}", flush=True)
    check(module(dev, K), random_inputs(M, K, seed=K, empty_every=4), dev)


def test_blocks_without_valid_pairs(dev):
    inputs = list(random_inputs(200, 8, seed=3))
    inputs[5] = inputs[5].clone()
    inputs[5][16:120] = False  # whole blocks, and the end of one
    print("aggregator blocks without valid pairs", flush=True)
    check(module(dev), inputs, dev)


@pytest.mark.parametrize("offset", [1, 4])
def test_weights_at_any_alignment(dev, offset):
    """Weight matrices that start `offset` elements past a 16-byte boundary."""
    mod = module(dev, 5)
    inp = [t.to(dev) for t in random_inputs(300, 5, seed=9)]
    st, keep = mod.packed_params()
    moved, own = type(st)(), []
    for name, _ in type(st)._fields_:
        t = keep[name]
        if t.dtype == torch.bfloat16:
            buf = torch.empty(t.numel() + offset, dtype=t.dtype, device=dev)
            buf[offset:] = t.reshape(-1)
            t = buf[offset:]
            own.append(buf)
        setattr(moved, name, ctypes.c_void_p(t.data_ptr()))
    print(f"aggregator weights at offset {offset}", flush=True)
    with torch.no_grad():
        want = C.aggregator_forward((st, keep), *inp)
        got = C.aggregator_forward((moved, own), *inp)
    for a, b in zip(got, want):
        assert (bits(a.cpu().numpy()) == bits(b.cpu().numpy())).all()
