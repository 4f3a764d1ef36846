"""Which kernel the dispatch rules choose (no GPU: vnpu_debug_route answers for
256 CUs).  Each row is a call whose two sides were timed on an MI355X: the
route is the faster one.
"""
import ctypes as C

import pytest

from vnpu_mi355x import Session, abi, load_backend


def route(opcode, fast=False, **fields):
    lib = load_backend()
    lib.vnpu_debug_route.restype = C.c_int32
    lib.vnpu_debug_route.argtypes = [C.c_void_p, C.c_uint32, C.c_char_p, C.c_uint32]
    cmd = Session.command(opcode, **fields)
    out = C.create_string_buffer(128)
    assert lib.vnpu_debug_route(C.byref(cmd), int(fast), out, 128) == abi.OK
    return out.value.decode()


def attention(pairs, sq, sk, d, fast=False, causal=1, off=0):
    p = [4096 * (i + 1) + off for i in range(4)]
    return route(abi.OP_ATTENTION_F32, fast, Q=p[0], K=p[1], V=p[2], O=p[3], batch=1, heads=pairs, seq_q=sq, seq_k=sk,
                 head_dim=d, causal=causal)


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
    assert attention(pairs, sq, sk, d) == want


def test_attention_few_rows_unaligned():
    """Rows that are not 16-byte aligned: the chains at head sizes 64 and 128, else the row-wise kernel."""
    assert attention(256, 4, 300, 128, off=4) == "exact_decode"
    assert attention(256, 4, 300, 96, off=4) == "rowwise"
