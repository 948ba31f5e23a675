#!/usr/bin/env python3
"""Decode paged-attention microbench: achieved K+V read bandwidth of the
decode kernel at three serving shapes.

Usage:  python tools/bench_decode_attn.py
"""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(__file__), ".."))

SHAPES = [(512, 400), (1024, 300), (256, 1500)]  # (batch, kv_len)
KH, G, D, BS = 8, 4, 128, 16


def run_one():
    import torch
    from kaito_amd import ops

    torch.manual_seed(0)
    dev = "cuda"
    for bs, L in SHAPES:
        blocks_per_seq = (L + BS - 1) // BS
        nblocks = bs * blocks_per_seq + 1
        k_cache = torch.randn(nblocks, KH, BS, D, dtype=torch.bfloat16,
                              device=dev)
        v_cache = torch.randn_like(k_cache)
        q = torch.randn(bs, KH * G, D, dtype=torch.bfloat16, device=dev)
        bt = torch.arange(1, bs * blocks_per_seq + 1, dtype=torch.int32,
                          device=dev).reshape(bs, blocks_per_seq)
        sl = torch.full((bs,), L, dtype=torch.int32, device=dev)
        scale = D ** -0.5

        if bs == SHAPES[0][0]:  # one numerics check
            from kaito_amd.ops import torch_ref
            got = ops.paged_attention(q, k_cache, v_cache, bt, sl, scale)
            want = torch_ref.paged_attention(
                q.float(), k_cache.float(), v_cache.float(), bt, sl, scale)
            err = (got.float() - want).abs().max().item()
            assert err < 2e-2, f"numerics mismatch: {err}"

        for _ in range(20):
            ops.paged_attention(q, k_cache, v_cache, bt, sl, scale)
        torch.cuda.synchronize()
        s, e = torch.cuda.Event(True), torch.cuda.Event(True)
        iters = 100
        s.record()
        for _ in range(iters):
            ops.paged_attention(q, k_cache, v_cache, bt, sl, scale)
        e.record()
        torch.cuda.synchronize()
        us = s.elapsed_time(e) / iters * 1000
        bytes_rd = bs * L * KH * D * 2 * 2  # K+V bf16
        print(f"bs={bs:4d} L={L:4d}: {us:7.1f} us  "
              f"{bytes_rd / us / 1e6:.2f} TB/s", flush=True)


if __name__ == "__main__":
    run_one()
