"""Which kernel the dispatch rules choose (no GPU: vnpu_debug_route answers for
256 CUs).  Each row is a call whose two sides were timed on an MI355X: the
route is the faster one.
"""
import re

import pytest

from gpu_ops import route
from test_gpu_parity import DIRECT_I8, FEW_ROWS_F32
from vnpu_mi355x import abi


def attention(pairs, sq, sk, d, fast=False, causal=1, off=0, noalloc=False, mask=None):
    """(kernels, bytes of workspace)"""
    p = [4096 * (i + 1) + off for i in range(4)]
    name, ws = route(abi.OP_ATTENTION_F32, fast, noalloc, Q=p[0], K=p[1], V=p[2], O=p[3], batch=1, heads=pairs,
                     mask=mask, seq_q=sq, seq_k=sk, head_dim=d, causal=causal).split(" ws=")
    return name, int(ws)


@pytest.mark.parametrize("pairs,sq,sk,d,want", [
    # chains against 32-row workgroups, us
    (96, 4, 4000, 128, "exact_decode"),     # 204 / 260
    (96, 3, 4000, 128, "exact_decode"),     # 192 / 260
    (128, 4, 4000, 96, "exact_decode"),     # 227 / 242
    (128, 3, 1500, 128, "exact_decode"),    # 85 / 97
    (192, 2, 1500, 96, "exact_decode"),     # 85 / 93
    (64, 4, 4000, 128, "exact_decode"),     # 114 / 242
    (256, 4, 4000, 64, "exact_rows32"),     # 226 / 201
    (256, 4, 1500, 128, "exact_rows32"),    # 182 / 112
    (256, 4, 300, 128, "exact_rows32"),     # 56 / 29
    (192, 3, 700, 96, "exact_rows32"),      # 66 / 47
    (8, 1, 4000, 128, "exact_decode"), (8, 2, 64, 128, "exact_rows32"), (8, 8, 4000, 64, "exact_decode"),
    (8, 9, 4000, 64, "exact_rows32"), (32, 2048, 2048, 128, "exact_rows128")])
def test_attention_few_rows(pairs, sq, sk, d, want):
    assert attention(pairs, sq, sk, d)[0] == want


def test_attention_few_rows_unaligned():
    """Rows that are not 16-byte aligned: the chains at head sizes 64 and 128, else the row-wise kernel."""
    assert attention(256, 4, 300, 128, off=4)[0] == "exact_decode"
    assert attention(256, 4, 300, 96, off=4)[0] == "rowwise"


@pytest.mark.parametrize("pairs,sq,sk,d,want", [
    # high-throughput device, head sizes without a kernel of its own: general against reference-order, us
    (8, 21, 1986, 8, "general"),            # 27 / 105
    (4, 67, 3819, 24, "general"),           # 54 / 184
    (4, 14, 2006, 80, "general"),           # 43 / 122
    (2, 21, 2294, 112, "general"),          # 66 / 166
    (64, 7, 974, 24, "general"),            # 30 / 51
    (32, 2048, 2048, 80, "exact_rows128"),  # 2580 / 332
    (256, 1, 4096, 80, "exact_decode"),     # 596 / 138
    (32, 64, 99, 72, "exact_rows32"),       # 35 / 13
    (32, 333, 1501, 96, "exact_rows32"),
    # its own kernels keep theirs
    (8, 21, 1986, 64, "split_prefill"), (32, 1, 4096, 128, "stream_decode"), (32, 4, 300, 96, "stream_decode"),
    (4, 20, 300, 160, "general"), (4, 20, 300, 36, "general"), (4, 20, 300, 300, "rowwise")])
def test_attention_high_throughput(pairs, sq, sk, d, want):
    assert attention(pairs, sq, sk, d, fast=True)[0] == want


def test_attention_high_throughput_mask():
    """A mask costs the reference-order kernels more: 64 pairs x 21 rows x 1500 keys of 48, 69 us against 108."""
    assert attention(64, 21, 1500, 48, fast=True, mask=4096)[0] == "general"


@pytest.mark.parametrize("pairs,sq,sk,d", [(96, 1, 4000, 96), (64, 6, 4000, 64), (8, 5, 2000, 128), (8, 4, 4000, 80)])
def test_attention_shared_scratch(pairs, sq, sk, d):
    """On the scratch that all streams share, calls that can do without it do."""
    assert attention(pairs, sq, sk, d)[0] == "exact_decode"
    assert attention(pairs, sq, sk, d, noalloc=True) == ("exact_rows32", 0)
    assert attention(pairs, sq, sk, 8, fast=True, noalloc=True)[0] == attention(pairs, sq, sk, 8, fast=True)[0]


def test_attention_shared_scratch_decode():
    assert attention(32, 1, 4000, 128, noalloc=True) == attention(32, 1, 4000, 128) == ("exact_decode", 32 * 4032 * 4)


@pytest.mark.parametrize("M,K,N", [(331, 4096, 576), (1024, 4096, 256), (781, 8320, 1088), (331, 1376, 5003), (9, 64, 16),
                                   (96, 4096, 1152), (40, 4096, 4111), (2048, 1001, 300)])
def test_matmul_i8_tiles_of_an_xcd(M, K, N):
    """The direct kernel's tiles take no more rounds on any XCD than spread evenly over the eight
    (whole column tiles to the XCDs in turn gave 42 of 168 to one of them for 331 x 4096 x 576)."""
    name, tiles, per = re.fullmatch(r"direct<(.*)> tiles=(\d+) xcd_tiles=(\d+)",
                                    route(abi.OP_MATMUL_I8, A=4096, M=M, K=K, N=N)).groups()
    mg, cb = (int(x) for x in name.split(",")[:2])
    assert int(tiles) == -(-M // (16 * mg)) * -(-N // (16 * cb))
    assert int(tiles) <= 8 * int(per)
    assert -(-int(per) // 32) == -(-int(tiles) // 256)


def test_matmul_i8_direct_instances():
    """The direct kernel's GPU test runs every instance that is built (but the 16 x 16 tiles of weights
    past the last-level cache, which take a depth beyond 400,000)."""
    seen = set()
    for M, K, N, pad, off, _ in DIRECT_I8:
        t = route(abi.OP_MATMUL_I8, A=4096 + off, M=M, K=K, N=N, lda=K + pad)
        if t.startswith("direct"):
            seen.add(t.split()[0])
    narrow = ("1,1,16", "1,2,8", "1,4,8", "2,4,8")
    want = {f"direct<{i}{o}>" for i in narrow for o in ("", ",spread", ",shift", ",shift,spread", ",stream")}
    want.remove("direct<1,1,16,stream>")
    want |= {f"direct<{i}{o}>" for i in ("2,4,4", "4,4,4") for o in ("", ",spread", ",stream")}
    assert seen == want


def matmul_f32(M, K, N, tb=0):
    return route(abi.OP_MATMUL_F32, A=4096, B=4096, C=4096, M=M, K=K, N=N, trans_b=tb)


@pytest.mark.parametrize("M,K,N,tb,splits", [
    # ranges of K against the partial sums that they write and read, us
    (988, 3378, 7616, 0, 1),     # 120 MB in two ranges: 534 / 572
    (382, 1535, 14208, 0, 1),    # 87 MB: 197 / 217
    (670, 939, 1935, 1, 2),      # 21 MB: 65 / 60
    (481, 3808, 1042, 0, 8),     # 32 MB in eight, 16 in four: 70 / 65
    (16, 4096, 4096, 0, 4), (77, 1000, 1001, 0, 4)])
def test_matmul_f32_ranges(M, K, N, tb, splits):
    assert matmul_f32(M, K, N, tb).endswith(f" splits={splits}")


@pytest.mark.parametrize("M,K,N,tb,waves", [
    # 64 x 64 workgroups over a short K, us with the waves here / with eight
    (932, 32, 9408, 1, 2),       # 30 / 46
    (427, 64, 13952, 0, 2),      # 26 / 34
    (700, 32, 2000, 0, 4),       # 8.4 / 11.4
    (796, 128, 7584, 0, 4),      # 37 / 44
    (512, 100, 1243, 0, 8),      # with four 9.1 / 8.0
    (290, 202, 7636, 1, 8)])     # with four 28.0 / 24.9
def test_matmul_f32_waves(M, K, N, tb, waves):
    assert re.fullmatch(rf"skinny<4,4,..,{waves}> splits=1", matmul_f32(M, K, N, tb))


def test_matmul_f32_few_rows_instances():
    """The few-rows kernels' GPU test runs every instance that is built, with K whole and (where it can be) in ranges."""
    seen = set()
    for M, K, N, tb, pad_a, pad_b in FEW_ROWS_F32:
        t = route(abi.OP_MATMUL_F32, A=4096, B=4096, C=4096, M=M, K=K, N=N, trans_b=tb, lda=K + pad_a,
                  ldb=(K if tb else N) + pad_b)
        if t.startswith("skinny"):
            seen.add((t.split()[0], not t.endswith("splits=1")))
        else:
            seen.add(t)
    want = {f"lanes<{m}>" for m in range(1, 9)}
    for b in ("KN", "NK"):
        for mg in (1, 2, 4):
            for cb in (1, 2, 4):
                name = f"skinny<{mg},{cb},{b},{16 if cb == 1 and mg < 4 else 8}>"
                want |= {(name, False), (name, True)}
        want |= {(f"skinny<4,4,{b},{w}>", False) for w in (2, 4)}
    assert not want - seen, sorted(map(str, want - seen))


@pytest.mark.parametrize("M,K,N,want", [
    # direct kernel against the 64-deep staged tiles over a short K, us
    (98, 64, 24512, "gemm"),        # 9.1 / 7.6
    (64, 192, 32000, "gemm"),       # 9.0 / 8.1
    (98, 64, 8192, "direct"),       # 5.1 / 7.0
    (64, 320, 16384, "direct"),     # 6.2 / 8.4
    (256, 192, 8192, "direct"),     # 8.9 / 11.0
    (256, 320, 16384, "gemm")])
def test_matmul_i8_short_depth(M, K, N, want):
    assert route(abi.OP_MATMUL_I8, A=4096, M=M, K=K, N=N).startswith(want)
