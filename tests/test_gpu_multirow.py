"""The multi-row matrix-core matvec (q8_gemv from 4 rows, layer calls from 2 sequences) against
float64: edges of its row tiles (16, 32, 33 rows), of its column blocks and tiles (64, 320: a partial
256-column tile), of its K ranges (64: one short wave; 160: a range that ends inside a block; 2112: a
wave that lies past K), both layouts, and one workspace shared by calls of different sizes and row
counts.

Bound: the products are exact and the sums f32 over K <= 6144 (a few 2^-24 per partial sum, random
signs: seen 1e-7 to 3e-7); 2e-6 is taken."""
import numpy as np
import pytest
import torch

import q35
from conftest import rel_l2
from gpu_util import dev, host, normal, q8, q8_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["kn", "tiled"])
@pytest.mark.parametrize("K,N,M", [(64, 64, 4), (160, 320, 5), (2112, 320, 6), (2048, 512, 16), (2048, 6144, 17), (6144, 2048, 32),
                                   (2048, 2048, 33), (96, 192, 64)])
def test_q8_gemv_rows(K, N, M, layout):
    print(f"[gemv rows] K={K} N={N} M={M} {layout}", flush=True)
    W = q8(400 + K + N, K, N)
    x = normal(401 + M, (M, K)) * np.exp(normal(402, (M, 1))).astype(np.float32)
    Wd = q8_dev(W, q35.Q35_KN)
    y = host(q35.q8_gemv(dev(x), Wd.tiled() if layout == "tiled" else Wd))
    ref = x.astype(np.float64) @ W.dequant()
    for m in range(M):
        assert rel_l2(y[m], ref[m]) <= 2e-6, m


def test_q8_gemv_rows_share_a_workspace_with_other_sizes():
    """Row counts and widths alternate on the one workspace of q8_gemv: every call's sums start from
    zero whatever ran before, including the one-row kernel's fixed-point words."""
    for K, N, M in [(2048, 512, 8), (2048, 8192, 1), (2048, 6144, 32), (64, 8192, 1), (2048, 512, 1), (2048, 2048, 5)]:
        W = q8(420, K, N)
        x = normal(421 + M, (M, K))
        y = host(q35.q8_gemv(dev(x), q8_dev(W, q35.Q35_KN)))
        assert rel_l2(y, x.astype(np.float64) @ W.dequant()) <= 2e-6, (K, N, M)


def test_q8_gemv_rows_unaligned_input_and_magnitudes():
    """Rows that start 4 bytes past a 16-byte boundary take the one-row kernel; rows of zeros and of
    magnitudes 1e-20 to 1e6 keep their relative precision where the fixed-point sums would not."""
    K, N, M = 2048, 1024, 6
    W = q8(430, K, N)
    x = normal(431, (M, K))
    ref = x.astype(np.float64) @ W.dequant()
    buf = torch.empty(M * K + 1, device="cuda")
    buf[1:] = dev(x).reshape(-1)
    xu = buf[1:].view(M, K)
    assert xu.data_ptr() % 16 != 0
    Wd = q8_dev(W, q35.Q35_KN)
    assert rel_l2(host(q35.q8_gemv(xu, Wd)), ref) <= 2e-6
    mag = np.array([1e-20, 1e-6, 1.0, 0.0, 1e3, 1e6], np.float32)
    y = host(q35.q8_gemv(dev(x * mag[:, None]), Wd))
    for m in range(M):
        if mag[m] == 0:
            np.testing.assert_array_equal(y[m], 0.0)
        else:
            assert rel_l2(y[m], ref[m] * float(mag[m])) <= 2e-6, m


@pytest.mark.parametrize("layout", ["kn", "tiled", "nk"])
@pytest.mark.parametrize("big", [2.0 ** 14, 2.0 ** 24, 2.0 ** 60])
def test_rows_with_one_large_input_keep_f32_products(big, layout):
    """One input per row many times the others, at a k whose weights are all 0: what is left are products
    of ordinary size, as precise as without it (f32 sums as above; nk: the lm_head's rows)."""
    print(f"[one large input] {big:.0e} {layout}", flush=True)
    K, N, M = (512, 32768, 5) if layout == "nk" else (2048, 512, 5)
    x = normal(435, (M, K))
    x[:, 77] = big
    if layout == "nk":
        E = q8(436, N, K)
        E.q[:, 77] = 0
        y, ref = host(q35.q8_lm_head(dev(x), q8_dev(E, q35.Q35_NK))), x.astype(np.float64) @ E.dequant().T
    else:
        W = q8(436, K, N)
        W.q[77] = 0
        Wd = q8_dev(W, q35.Q35_KN)
        y = host(q35.q8_gemv(dev(x), Wd.tiled() if layout == "tiled" else Wd))
        ref = x.astype(np.float64) @ W.dequant()
    for m in range(M):
        assert rel_l2(y[m], ref[m]) <= 1e-6, m


@pytest.mark.parametrize("layout", ["kn", "tiled"])
@pytest.mark.parametrize("N,M", [(512, 4), (4096, 5), (6144, 17)])
def test_k_splits_are_added_in_64_bits(N, M, layout):
    """2^24 from the first rows of K, 1 from the middle and -2^24 from the last, each exact in its own
    split: the sum is 1 as with one row, where 32-bit sums leave 0 (the widths take 16, 8 and 4 splits)."""
    print(f"[64-bit splits] N={N} M={M} {layout}", flush=True)
    K = 2048
    W = q8(437, K, N)
    W.q[:] = 0
    W.s[:] = 1.0
    W.q[0] = W.q[K - 1] = 64
    W.q[K // 2] = 1
    x = np.zeros((M, K), np.float32)
    x[:, 0], x[:, K // 2], x[:, K - 1] = 2.0 ** 18, 1.0, -2.0 ** 18
    Wd = q8_dev(W, q35.Q35_KN)
    Wd = Wd.tiled() if layout == "tiled" else Wd
    for rows in (M, 1):
        np.testing.assert_array_equal(host(q35.q8_gemv(dev(x[:rows]), Wd)), 1.0)


@pytest.mark.parametrize("B", [2, 33])
def test_layers_in_row_groups(B):
    """MLP and attention over one row group and a second one (33 = 32 + 1 rows): each row as by itself."""
    d = q35.dims_2b()
    H, nh, nkv, hd = d.hidden, d.attn_heads, d.kv_heads, d.head_dim
    x = dev(normal(440, (B, H)))
    mlp = q35.MLP(d, *(q8_dev(q8(441 + i, *s), q35.Q35_KN).tiled() for i, s in
                       enumerate([(H, d.ffn), (H, d.ffn), (d.ffn, H)])))
    att = q35.Attention(d, *(q8_dev(q8(445 + i, *s), q35.Q35_KN) for i, s in
                             enumerate([(H, nh * hd * 2), (H, nkv * hd), (H, nkv * hd), (nh * hd, H)])),
                        dev(normal(450, (hd,), 0.1)), dev(normal(451, (hd,), 0.1)))
    tmax = 40
    cs, sn = q35.rope_tables(d, tmax)
    kc, vc = normal(452, (B, nkv, tmax, hd)), normal(453, (B, nkv, tmax, hd))
    pos = (np.arange(B) % tmax).astype(np.int32)
    kd, vd = dev(kc), dev(vc)
    out_m = host(mlp.forward(x, check=True))
    out_a = host(att.forward(x, kd, vd, dev(pos), dev(cs), dev(sn)))
    for b in range(B):
        k1, v1 = dev(kc[b:b + 1]), dev(vc[b:b + 1])
        assert rel_l2(out_m[b], host(mlp.forward(x[b:b + 1]))[0]) <= 3e-6, b
        one = host(att.forward(x[b:b + 1], k1, v1, dev(pos[b:b + 1]), dev(cs), dev(sn)))
        assert rel_l2(out_a[b], one[0]) <= 3e-6, b
        assert rel_l2(host(kd[b]), host(k1[0])) <= 2e-6 and rel_l2(host(vd[b]), host(v1[0])) <= 2e-6


@pytest.mark.parametrize("hidden,ffn,heads", [(512, 1536, 4), (64, 64, 2), (2048, 6144, 16)])
def test_one_row_layers_between_batches(hidden, ffn, heads):
    """One-row MLP and DeltaNet calls equal the same row in a batch of three, call after call, whatever
    sizes other layers of the process have (each size has a workspace of its own)."""
    d = q35.make_dims(hidden=hidden, ffn=ffn, lin_heads=heads)
    vd, cd = heads * 128, 3 * heads * 128
    mlp = q35.MLP(d, *(q8_dev(q8(460 + i, *s), q35.Q35_KN) for i, s in
                       enumerate([(hidden, ffn), (hidden, ffn), (ffn, hidden)])))
    gdn = q35.GatedDeltaNet(d, *(q8_dev(q8(464 + i, *s), q35.Q35_KN).tiled() for i, s in
                                 enumerate([(hidden, cd), (hidden, vd), (vd, hidden)])),
                            dev(normal(468, (hidden, heads), 0.02)), dev(normal(469, (hidden, heads), 0.02)),
                            dev(normal(470, (heads,), 0.5)), dev(np.ones(heads, np.float32)),
                            dev(normal(471, (cd, 4), 0.5)), dev(1 + normal(472, (128,), 0.1)))
    x = dev(normal(473, (3, hidden)))
    cs, S = normal(474, (3, cd, 3)), normal(475, (3, heads, 128, 128), 0.1)
    cs3, S3 = dev(cs), dev(S)
    out_m, out_g = host(mlp.forward(x)), host(gdn.forward(x, cs3, S3))
    for r in (0, 2, 1):
        assert rel_l2(host(mlp.forward(x[r:r + 1], check=True))[0], out_m[r]) <= 3e-6, r
        cs1, S1 = dev(cs[r:r + 1]), dev(S[r:r + 1])
        assert rel_l2(host(gdn.forward(x[r:r + 1], cs1, S1))[0], out_g[r]) <= 3e-6, r
        assert rel_l2(host(S1)[0], host(S3)[r]) <= 3e-6 and rel_l2(host(cs1)[0], host(cs3)[r]) <= 3e-6, r


@pytest.mark.parametrize("N,K,M", [(32768, 256, 2), (32768 + 37, 512, 3), (70001, 1280, 5), (248320, 2048, 4),
                                   (248320, 2048, 8), (40000, 2048, 11)])
def test_lm_head_rows(N, K, M):
    """Rows per pass over a large table: 2 (one-row kernel's form), 3 to 8 on the matrix cores, 11 = 8 + 3; partial last tiles of 64 rows, one and several tiles
    per wave, 4 to 32 scale blocks (20: not a whole number of its groups of 16)."""
    print(f"[lm_head rows] N={N} K={K} M={M}", flush=True)
    rng = np.random.default_rng(N + M)
    q = rng.integers(-127, 128, (N, K), dtype=np.int8)
    s = (rng.random((N, K // 64), dtype=np.float32) + 0.5) * 1e-3
    x = rng.standard_normal((M, K), dtype=np.float32) * np.exp(rng.standard_normal((M, 1))).astype(np.float32)
    E = q35.Q8FTensor(dev(q), dev(s), q35.Q35_NK)
    y = q35.q8_lm_head(dev(x), E)
    for n0 in range(0, N, 1 << 15):
        w = E.q[n0:n0 + (1 << 15)].double().view(-1, K // 64, 64) * E.scale[n0:n0 + (1 << 15)].double()[:, :, None]
        ref = dev(x).double() @ w.view(-1, K).T.contiguous()
        for m in range(M):
            assert rel_l2(host(y[m, n0:n0 + (1 << 15)]), host(ref[m])) <= 1e-6, (m, n0)


def test_lm_head_rows_infinity_as_one_row():
    """A row with an infinity gives what the one-row kernel gives (infinite products, NaN where the
    weight is 0); the other rows are not touched by it."""
    N, K = 32768, 512
    rng = np.random.default_rng(3)
    E = q35.Q8FTensor(dev(rng.integers(-127, 128, (N, K), dtype=np.int8)),
                      dev(rng.random((N, K // 64), dtype=np.float32) * 1e-2), q35.Q35_NK)
    x = rng.standard_normal((3, K), dtype=np.float32)
    x[1, 77] = np.inf
    y = host(q35.q8_lm_head(dev(x), E))
    np.testing.assert_array_equal(y[1], host(q35.q8_lm_head(dev(x[1:2]), E))[0])
    for r in (0, 2):
        assert rel_l2(y[r], host(q35.q8_lm_head(dev(x[r:r + 1]), E))[0]) <= 1e-6


@pytest.mark.parametrize("K,N,M", [(2048, 2048, 33), (6144, 2048, 20), (8192, 16384, 8), (8704, 16384, 8), (64, 64, 4)])
def test_q8_gemv_noalloc_rows_same_bits(K, N, M):
    """The allocation-free entry point takes the rows in smaller groups where its fixed scratch asks for
    it, up to its largest (8704 x 16384 is past it: both entry points keep the one-row kernel), bit for bit."""
    L = q35._lib
    Wd = q8_dev(q8(480, K, N), q35.Q35_KN)
    x = dev(normal(481, (M, K)))
    y = torch.empty(M, N, device="cuda")
    L.check(L.lib().q35_q8_gemv_noalloc(x.data_ptr(), M, Wd.desc(), y.data_ptr(), torch.cuda.current_stream().cuda_stream))
    np.testing.assert_array_equal(host(y), host(q35.q8_gemv(x, Wd)))
