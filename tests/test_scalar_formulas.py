"""Scalar formulas of the kernels (newton_amd/csrc/vbd_scalar.h) on the CPU, over the ranges where they can go wrong."""

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("scalar") / "scalar_check.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-o", str(so),
                    str(HERE / "scalar_check.cpp")], check=True)
    return ctypes.CDLL(str(so))


def _screen(lib, blocks):
    blocks = np.ascontiguousarray(blocks, np.float32)
    out = np.zeros(len(blocks), np.int32)
    lib.screen(len(blocks), blocks.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p))
    return out == 1, blocks.astype(np.float64)


def _condition(blocks):
    """||H||_F ||adj H||_F / |det H| in double precision from the stored entries: what the block solve compares with
    1e6."""
    adj = np.stack([np.cross(blocks[:, 1], blocks[:, 2]), np.cross(blocks[:, 2], blocks[:, 0]),
                    np.cross(blocks[:, 0], blocks[:, 1])], axis=1)
    det = np.abs(np.sum(blocks[:, 0] * adj[:, 0], axis=1))
    norm = lambda a: np.sqrt((a.reshape(-1, 9) ** 2).sum(axis=1))  # noqa: E731
    return norm(blocks) * norm(adj) / np.maximum(det, 1e-300)


def _blocks(rng, n, condition, scale, symmetric):
    u = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0]
    v = u if symmetric else np.linalg.qr(rng.normal(size=(n, 3, 3)))[0]
    lo = 1.0 / condition
    mid = np.exp(rng.uniform(np.log(lo), 0.0, n))
    s = np.stack([np.ones(n), mid, lo * np.ones(n)], axis=1)
    return scale * np.einsum("nij,nj,nkj->nik", u, s, v)


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("scale", [0.1, 1.0, 1.0e4, 1.0e9, 1.0e12, 3.0e12, 1.0e13, 1.0e15, 1.0e18, 3.0e19])
def test_screen_never_clears_an_ill_conditioned_block(lib, scale, symmetric):
    """Conditions on both sides of 1e6, scales up to where the determinant, then the squared norm, overflow."""
    rng = np.random.default_rng(7)
    for condition in (1.0e5, 3.0e5, 1.0e6, 3.0e6, 1.0e7, 1.0e9):
        cleared, blocks = _screen(lib, _blocks(rng, 4000, condition, scale, symmetric))
        assert not np.any(cleared & (_condition(blocks) > 1.0e6)), condition


@pytest.mark.parametrize("diagonal", [(1e16, 1e16, 1e7), (1e15, 1e15, 1e9), (1e16, 1e15, 3e8), (1e18, 1e18, 1.0)])
def test_screen_leaves_an_overflowed_determinant_to_double_precision(lib, diagonal):
    cleared, blocks = _screen(lib, np.diag(diagonal)[None])
    assert _condition(blocks)[0] > 1.0e6 and not cleared[0]


@pytest.mark.parametrize("scale", [1.0, 1.0e4, 1.0e9, 1.0e12])
def test_screen_clears_ordinary_blocks(lib, scale):
    """Conditions up to 1e4 with the middle stiffness high are cleared: the screen spares their estimate."""
    rng = np.random.default_rng(8)
    for condition in (1.0, 10.0, 1.0e3, 1.0e4):
        u = np.linalg.qr(rng.normal(size=(2000, 3, 3)))[0]
        s = np.array([1.0, 1.0, 1.0 / condition])
        cleared, _ = _screen(lib, scale * np.einsum("nij,j,nkj->nik", u, s, u))
        assert cleared.all(), condition


def _sigmoid(lib, z):
    z = np.ascontiguousarray(z, np.float32)
    out = np.full(len(z), 7.0, np.float32)
    lib.sigmoid(len(z), z.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p))
    return out


def test_sigmoid_within_its_range(lib):
    """Against 64 bits: exp2 (an ulp), the product's and the sum's roundings and the reciprocal's leave about three
    ulps; half an ulp of the argument of exp2 that the low part restores would be worth 40 of them at z = -80."""
    z = np.concatenate([np.linspace(-87.33, 88.0, 200001), np.random.default_rng(1).normal(0, 3, 100000)])
    z = z.astype(np.float32)
    with np.errstate(over="ignore"):
        ref = 1.0 / (1.0 + np.exp(-z.astype(np.float64)))
    assert np.max(np.abs(_sigmoid(lib, z) - ref) / ref) <= 4.0 * 2.0 ** -23


def test_sigmoid_far_outside_its_range(lib):
    """0 below 2^-126 and 1 above, up to infinity, as 1 / (1 + expf(-z)) gives them (its denormals aside); the order
    is kept all the way."""
    far = np.array([-np.inf, -3.4e38, -1e30, -1e12, -1e10, -3.3e8, -3.0e7, -1e4, -104.0, -89.0], np.float32)
    assert np.all(_sigmoid(lib, far) == 0.0) and np.all(_sigmoid(lib, -far) == 1.0)
    z = np.sort(np.concatenate([far, -far, np.linspace(-90, 20, 4001)]).astype(np.float32))
    s = _sigmoid(lib, z)
    assert np.all(np.diff(s) >= -2.0 ** -23 * s[1:]) and np.all((s >= 0.0) & (s <= 1.0 + 2.0 ** -23))
