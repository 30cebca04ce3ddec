"""Short windows in one launch (attn_decode_short): attention, and the fused step of one row, against the oracle at the
edges of the kernel's waves (32 rows of head_dim 64, 8 of 128), its round trips (512 / 128 rows) and its range (512 /
256 rows, one workgroup per CU), on both sides of each, the cache rows past the causal window poisoned with NaN."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import Buffers, assert_parity, bits
from tests.test_gpu_f16kv import download_f16, upload_f16
from tests.test_gpu_parity import cpu_attention

pytestmark = pytest.mark.gpu

# (H, KV, D)
SHAPES = [(14, 2, 64), (32, 4, 64), (5, 5, 64), (32, 8, 64), (24, 8, 128), (4, 1, 128)]


def edges(D):
    return [1, 2, 31, 33, 511, 512, 513] if D == 64 else [1, 7, 9, 127, 129, 255, 256, 257]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("n", [1, 3, 11])
@pytest.mark.parametrize("H,KV,D", SHAPES)
def test_short_windows_match_oracle(backend, H, KV, D, n, f16):
    rng = np.random.default_rng(H + 7 * KV + D + n)
    t = np.float16 if f16 else np.float32
    for rows in edges(D):
        if rows < n:
            continue
        pos0 = rows - n
        q = rng.standard_normal((n, H, D)).astype(np.float32)
        k, v = (rng.standard_normal((rows + 3, KV, D)).astype(t) for _ in range(2))
        kp, vp = k.copy(), v.copy()
        kp[rows:] = np.nan
        vp[rows:] = np.nan
        up = upload_f16 if f16 else (lambda B, a: B.upload(a))
        with Buffers(backend) as B:
            dq, dk, dv, do = B.upload(q), up(B, kp), up(B, vp), B.alloc(q.size)
            (backend.attention_f16kv if f16 else backend.attention)(dq, dk, dv, do, n, pos0, H, KV, D)
            got = backend.download(do, q.shape)
        ref = cpu_attention(q, k[:rows].astype(np.float32), v[:rows].astype(np.float32), pos0, KV)
        assert_parity(got, ref, f"H={H} KV={KV} D={D} n={n} rows={rows} f16={f16}")


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("H,KV,D,neox", [(14, 2, 64, True), (32, 4, 64, False), (24, 8, 128, True)])
def test_short_fused_append(backend, H, KV, D, neox, f16):
    """One row appended and attended in the launch: the cache then holds the rotated row and the output is bitwise that of
    attention over such a cache, row pos0 poisoned before (it is carried in registers, never read)."""
    rng = np.random.default_rng(H + D)
    t = np.float16 if f16 else np.float32
    up = upload_f16 if f16 else (lambda B, a: B.upload(a))
    down = (lambda b, s: download_f16(backend, b, s)) if f16 else backend.download
    name = "_f16kv" if f16 else ""
    for rows in edges(D):
        pos0 = rows - 1
        q = rng.standard_normal((1, H, D)).astype(np.float32)
        kn, vn = (rng.standard_normal((1, KV, D)).astype(np.float32) for _ in range(2))
        k0, v0 = (rng.standard_normal((rows + 2, KV, D)).astype(t) for _ in range(2))
        k0[pos0:], v0[pos0:] = np.nan, np.nan
        # the same step unfused: the cache with the row in it, the rotated query
        qr, kr = oracle.rope(q.copy(), pos0, 1e4, neox, None), oracle.rope(kn.copy(), pos0, 1e4, neox, None)
        k1, v1 = k0.copy(), v0.copy()
        k1[pos0], v1[pos0] = kr[0], vn[0]
        with Buffers(backend) as B:
            dq, dr, dkn, dvn = B.upload(q), B.upload(qr), B.upload(kn), B.upload(vn)
            ck, cv, ck1, cv1 = up(B, k0), up(B, v0), up(B, k1), up(B, v1)
            o1, o2 = B.alloc(q.size), B.alloc(q.size)
            getattr(backend, "append_rope_attention" + name)(dq, ck, cv, dkn, dvn, o1, 1, pos0, H, KV, D, 1e4, neox,
                                                             None)
            getattr(backend, "attention" + name)(dr, ck1, cv1, o2, 1, pos0, H, KV, D)
            r1, r2 = backend.download(o1, q.shape), backend.download(o2, q.shape)
            gk, gv = down(ck, k0.shape), down(cv, v0.shape)
        where = f"H={H} D={D} rows={rows} f16={f16}"
        u = np.uint16 if f16 else np.uint32
        assert np.array_equal(gk[:rows].view(u), k1[:rows].view(u)), f"K cache: {where}"
        assert np.array_equal(gv[:rows].view(u), v1[:rows].view(u)), f"V cache: {where}"
        assert np.all(np.isnan(gk[rows:])) and np.all(np.isnan(gv[rows:])), where
        assert np.array_equal(bits(r1), bits(r2)), f"fused and unfused outputs differ: {where}"
        ref = cpu_attention(qr, k1[:rows].astype(np.float32), v1[:rows].astype(np.float32), pos0, KV)
        assert_parity(r1, ref, where)
