"""Device blocks kept between objects: a block given back while work that
reads it is still queued on another stream is not written by its next owner
before that work is done; results stay right over many conversions from two
threads; vkv_workspace_release gives the kept blocks back to the device."""
import threading

import pytest
import torch

import vkv

pytestmark = pytest.mark.gpu


def filled(value, T=4096):
    c = vkv.KVCacheSimple()
    x = torch.full((1, 8, T, 128), value, device="cuda", dtype=torch.bfloat16)
    views = c.update(x, x)
    return c, views


def test_queued_readers_on_another_stream_keep_their_values():
    side = torch.cuda.Stream()
    a = torch.randn((2048, 2048), device="cuda")
    outs = []
    for i in range(48):  # 8 MB buffers: past the bytes at which the pool waits for the device
        c, (k, _) = filled(float(i % 7 + 1))
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(6):
                a = torch.tanh(a @ a)          # keeps the side stream behind
            outs.append((i % 7 + 1, vkv.to_torch(k, stream=side)))
        del c                                   # the reader is still queued
    torch.cuda.synchronize()
    for want, got in outs:
        assert bool((got == want).all())


def test_two_threads_convert_and_rotate():
    bad = []

    def work(seed):
        torch.manual_seed(seed)
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for i in range(24):
                x = torch.full((2, 4, 512 + 32 * (i % 5), 128), float(seed + i), device="cuda").half()
                c = vkv.KVCacheSimple()
                c.update(x, x)
                q = c.to_quantized(64, 8)
                r = vkv.RotatingKVCache(256)
                r.update(x, x)
                _, rv = r.update(x[:, :, :64], x[:, :, :64])
                back = q.to_unquantized().state[0]
                got = vkv.to_torch(rv)
                st.synchronize()
                if not (bool((back == seed + i).all()) and bool((got == seed + i).all())):
                    bad.append((seed, i))
                del c, q, r
    ts = [threading.Thread(target=work, args=(s,)) for s in (1, 100)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_release_empties_the_pool():
    x = torch.empty((8, 8, 4096, 128), device="cuda", dtype=torch.bfloat16)
    c = vkv.KVCacheSimple()
    c.update(x, x)
    del c
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    vkv.workspace_release()
    assert torch.cuda.mem_get_info()[0] >= before + 2 * x.numel() * 2


def test_release_while_another_thread_converts():
    good, done = [], threading.Event()

    def convert():
        st = torch.cuda.Stream()
        try:
            with torch.cuda.stream(st):
                for i in range(60):
                    x = torch.full((2, 4, 512 + 64 * (i % 3), 128), float(i + 1), device="cuda").half()
                    c = vkv.KVCacheSimple()
                    c.update(x, x)
                    back = c.to_quantized(64, 8).to_unquantized().state[0]
                    st.synchronize()
                    good.append(bool((back == i + 1).all()))
        finally:
            done.set()

    def release():
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            while not done.wait(0.002):
                vkv.workspace_release()

    ts = [threading.Thread(target=f) for f in (convert, release)]
    [t.start() for t in ts]
    [t.join(60) for t in ts]
    assert len(good) == 60 and all(good)
