"""Persistent launches on several streams: their workgroups wait for each other, so a call on another stream is held on the
device until every workgroup of the earlier launches runs."""
import pytest
import torch

from slotstream_spark_amd import _lib
from slotstream_spark_amd.engine.accept import Acceptor
from slotstream_spark_amd.kernels.moe_gemv_affine import moe_decode
from slotstream_spark_amd.memory.synth import verify_logits
from tests.gpu_util import make_pool, rand_ids, rand_weights, rand_x

pytestmark = pytest.mark.gpu

D, V, K = 3, 151936, 8


class Decode:
    """moe_decode with buffers of its own (no allocation in a call)."""

    def __init__(self, pool, seed):
        self.pool, dev = pool, pool.device
        self.x = rand_x(4, pool.hidden, seed).to(dev)
        self.ids, self.w = rand_ids(4, K, pool.experts, seed + 1).to(dev), rand_weights(4, K, seed + 2).to(dev)
        self.h = torch.empty((4, K, pool.inter), device=dev)
        self.o = torch.empty((4, K, pool.hidden), device=dev)
        self.out = torch.empty((4, pool.hidden), device=dev)
        self.want = self().clone()

    def __call__(self):
        return moe_decode(self.x, self.ids, self.w, 0, self.pool.map, self.pool.slot_ptr, self.h, self.o, self.out,
                          experts_per_layer=self.pool.experts)


@pytest.fixture(scope="module")
def pool():
    print("[order] pool H=2048 I=512 E=64", flush=True)
    return make_pool(64, 2048, 512, seed=5)


def test_different_entry_points_on_two_streams(pool):
    """moe_decode on one stream beside the p/q round on another: every result as alone, no bounded wait ran out."""
    print("[order] moe_decode beside the p/q round", flush=True)
    dec, acc = Decode(pool, 31), Acceptor(D, V)
    target, draft = verify_logits(D, V, 7)
    drafts = target[:D].argmax(dim=1).to(torch.int32)
    u = torch.rand(D + 1, generator=torch.Generator().manual_seed(3)).cuda()
    want = acc.pq_async(target, draft, drafts, u, 0.7).clone()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    _lib.device_error()
    got = []
    for _ in range(20):
        with torch.cuda.stream(a):
            got.append((dec().clone(), dec.want))
        with torch.cuda.stream(b):
            got.append((acc.pq_async(target, draft, drafts, u, 0.7).clone(), want))
    torch.cuda.synchronize()
    assert _lib.device_error() == 0
    for i, (g, w) in enumerate(got):
        assert torch.equal(g, w), i


def test_call_while_the_last_stream_is_capturing(pool):
    """Calls on a stream, then a capture on it, and a call on another stream while the capture is open: that call still
    waits for the earlier ones, and a persistent launch recorded in the capture replays as the eager call."""
    print("[order] a call behind an open capture", flush=True)
    first, second = Decode(pool, 41), Decode(pool, 51)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    _lib.device_error()
    for _ in range(3):
        graph = torch.cuda.CUDAGraph()
        second.out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            for _ in range(20):
                first()
            graph.capture_begin()
            first()
            with torch.cuda.stream(b):
                second()
            graph.capture_end()
        torch.cuda.synchronize()
        assert torch.equal(first.out, first.want) and torch.equal(second.out, second.want)
        for _ in range(3):
            first.out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(first.out, first.want)
    assert _lib.device_error() == 0

