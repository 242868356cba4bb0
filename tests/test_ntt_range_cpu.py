"""Unreduced values of the forward (DIF) transform passes stay inside the domain
of the reduction that ends a pass (CPU only).

The library's own reduction (csrc/fr29.hpp, compiled for the host) is checked
against integers at the ends of its domain, and inside an integer emulation of
one tile of a pass, limb by limb: stages in pairs, products in the 2^261
Montgomery form, the last two stages by their shorter form, where differences
leave unmultiplied. Inputs that line the signs up (0, c, 0, c, ... and r - 1 at
every fourth place) drive those to their largest magnitude, negative as well as
positive; random inputs stay within a few r.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from pymodel import R

HERE = os.path.dirname(os.path.abspath(__file__))
MASK = (1 << 29) - 1
R8 = R >> 232
NR = (-pow(R, -1, 1 << 29)) % (1 << 29) * R   # = -1 mod 2^29


@pytest.fixture(scope="module")
def red(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("ntt_range") / "ntt_range.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wno-unknown-pragmas", "-shared", "-fPIC", os.path.join(HERE, "cpp", "ntt_range.cpp"),
                    "-o", so], check=True, timeout=300)
    lib = ctypes.CDLL(so)

    def call(name, rows):
        a = np.ascontiguousarray(rows, dtype=np.int32)
        out = np.empty_like(a)
        p = ctypes.POINTER(ctypes.c_int32)
        getattr(lib, name)(a.ctypes.data_as(p), out.ctypes.data_as(p), ctypes.c_long(len(a)))
        return out.tolist()

    return call


def _norm(v):
    """integer -> normalized limbs (limb 8 signed)"""
    return [(v >> (29 * i)) & MASK for i in range(8)] + [v >> 232]


def _value(l):
    return sum(x << (29 * i) for i, x in enumerate(l))


def _check(red, rows):
    for row, got in zip(rows, red("fr_reduce_n", rows)):
        v = _value(row)
        assert all(0 <= x <= MASK for x in got[:8]) and 0 <= _value(got) < 2 * R, (v // R, got)
        assert (_value(got) - v) % R == 0, v // R


def test_reduce_over_its_domain(red):
    rng = np.random.default_rng(1)
    vals = [b * R + o for b in range(-299, 600) for o in (0, 1, -1, R // 2, R - 1)]
    vals += [-300 * R + 1, 600 * R - 1]
    vals += [int.from_bytes(rng.bytes(40), "little") % (900 * R) - 300 * R + 1 for _ in range(2000)]
    _check(red, [_norm(v) for v in vals])
    # limbs 0..7 of a sum of four normalized values, or of differences
    rows = []
    for lo in (-4 * MASK, 4 * MASK, -2 * MASK, 2 * MASK):
        for top in (-298, -259, -64, -48, 0, 300, 515, 597):
            rows.append([lo] * 8 + [top * R8])
    _check(red, rows)
    can = [0, 1, R - 1, R, R + 1, 2 * R - 1]
    for v, got in zip(can, red("fr_canonical_n", [_norm(v) for v in can])):
        assert _value(got) == v % R


def _mul(a, b):
    """limbs29's product: eight digits by NR, the last by R"""
    acc = _value(a) * b
    for k in range(8):
        acc += ((acc >> (29 * k)) & MASK) * NR << (29 * k)
    m = ((acc >> 232) & MASK) * ((-pow(R, -1, 1 << 29)) % (1 << 29)) & MASK
    return _norm((acc + (m * R << 232)) >> 261)


def _add(a, b):
    r = [x + y for x, y in zip(a, b)]
    assert all(-(1 << 31) <= x < 1 << 31 for x in r)
    return r


def _sub(a, b):
    return _add(a, [-x for x in b])


def _dif_tile(red, x, tw):
    """One tile of R = len(tw) stages over all of x: chunks of two stages, values reduced after six in a longer pass."""
    n, stages = len(x), len(x).bit_length() - 1
    v = [_norm(a) for a in x]
    nrm = lambda l: _norm(_value(l))
    for s in range(0, stages - stages % 2, 2):
        if stages > 8 and s == 6:
            v = red("fr_reduce_n", v)
        h, last = n >> (s + 1), s + 2 == stages
        q = h // 2
        for base in range(0, n, 2 * h):
            for j in range(q):
                i = [base + j, base + j + q, base + j + h, base + j + h + q]
                a, b, c, d = (v[k] for k in i)
                if last:   # twiddles 1, 1, the fourth root of unity
                    s0, s1, d0, p = _add(a, c), _add(b, d), _sub(a, c), _mul(_sub(b, d), tw[n // 4])
                    v[i[0]], v[i[1]], v[i[2]], v[i[3]] = _add(s0, s1), _sub(s0, s1), _add(d0, p), _sub(d0, p)
                else:
                    w0, w1, w2 = tw[j << s], tw[(j + q) << s], tw[j << (s + 1)]
                    s0, s1, d0, d1 = _add(a, c), _add(b, d), _mul(_sub(a, c), w0), _mul(_sub(b, d), w1)
                    v[i[0]], v[i[1]] = nrm(_add(s0, s1)), _mul(_sub(s0, s1), w2)
                    v[i[2]], v[i[3]] = nrm(_add(d0, d1)), _mul(_sub(d0, d1), w2)
    if stages % 2:
        for i in range(0, n, 2):
            a, b = v[i], v[i + 1]
            v[i], v[i + 1] = nrm(_add(a, b)), _mul(_sub(a, b), tw[0])
    worst = [min(_value(l) for l in v) / R, max(_value(l) for l in v) / R]
    assert -300 < worst[0] and worst[1] < 600, worst
    return [_value(l) for l in red("fr_canonical_n", red("fr_reduce_n", v))]


def _dft_bitrev(x):
    n, w = len(x), pow(5, (R - 1) // len(x), R)
    out, h, s = list(x), len(x) // 2, 1
    while h:
        for base in range(0, n, 2 * h):
            for j in range(h):
                a, b = out[base + j], out[base + j + h]
                out[base + j], out[base + j + h] = (a + b) % R, (a - b) * pow(w, j * s, R) % R
        h, s = h // 2, s * 2
    return out


@pytest.mark.parametrize("log_n", [6, 7, 8, 9, 10])
@pytest.mark.parametrize("top", [R - 1, 2 * R - 1])   # a call's values, and those that an earlier pass leaves
def test_pass_on_structured_values(red, log_n, top):
    n = 1 << log_n
    w = pow(5, (R - 1) // n, R)
    tw = [pow(w, e, R) * pow(2, 261, R) % R for e in range(n // 2)]
    minus_one = R - pow(2, 256, R)
    pats = [[top], [0, top], [top, 0], [0, 0, top, 0], [0, top, 0, 0], [0, 0, 0, top], [1, R - 1], [0, minus_one], [top, 0, 0, top],
            [0, 2], [0, 7]]
    for pat in pats:
        x = (pat * n)[:n]
        assert _dif_tile(red, x, tw) == _dft_bitrev([v % R for v in x]), pat
