"""Shared helpers of the GPU parity tests: seeded EXL3 weights and the tolerance bar."""

from __future__ import annotations

import numpy as np
import torch

# Tolerance bar of the matmul outputs: max-abs-err <= 2e-2 * rms(ref)
# and cosine >= 0.9999 against an fp32-accumulated reference on the same inputs.
MAX_ABS_REL_RMS = 2e-2
MIN_COSINE = 0.9999

CB_IDS = {"3inst": 0, "mcg": 1, "mul1": 2}


def make_weight(k: int, n: int, K: int, seed: int):
    """Seeded EXL3 weight: uniform random int16 trellis (every 16-bit state reachable)
    and +-1 fp16 sign vectors.  numpy arrays."""
    rng = np.random.default_rng(seed)
    trellis = rng.integers(-32768, 32768, size=(k // 16, n // 16, 16 * K), dtype=np.int64).astype(np.int16)
    suh = np.where(rng.random(k) < 0.5, -1.0, 1.0).astype(np.float16)
    svh = np.where(rng.random(n) < 0.5, -1.0, 1.0).astype(np.float16)
    return trellis, suh, svh


def make_x(m: int, k: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed + 7919)
    return rng.standard_normal((m, k)).astype(np.float16)


def to_dev(*arrs, device="cuda"):
    return [torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in arrs]


def check_close(out: np.ndarray, ref: np.ndarray, what: str = "") -> dict:
    out = np.asarray(out, dtype=np.float64).reshape(-1)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1)
    assert np.all(np.isfinite(out)), f"{what}: non-finite output"
    rms = float(np.sqrt(np.mean(ref * ref)))
    err = float(np.max(np.abs(out - ref)))
    cos = float(np.dot(out, ref) / (np.linalg.norm(out) * np.linalg.norm(ref) + 1e-300))
    assert err <= MAX_ABS_REL_RMS * rms, f"{what}: max-abs-err {err:.4g} > {MAX_ABS_REL_RMS} * rms {rms:.4g}"
    assert cos >= MIN_COSINE, f"{what}: cosine {cos:.6f} < {MIN_COSINE}"
    return {"max_abs_err": err, "rms": rms, "cos": cos}


def weight64(trellis: torch.Tensor, K: int, cb: int) -> torch.Tensor:
    """The trellis's entries [k, n] in float64, a codebook value not rounded (MCG and 3INST: the exact sum of
    its two fp16 halves; mul1: the exact affine map of the byte sum)."""
    kt, nt, kw = trellis.shape
    v = trellis.reshape(-1, kw // 2, 2).to(torch.int64) & 0xFFFF
    words = v[..., 0] | (v[..., 1] << 16)
    t = torch.arange(256, device=trellis.device)
    start = ((t + 257) * K - 16) % (256 * K)
    last = (start + 15) // 32
    pair = (words[:, start // 32] << 32) | words[:, last % (kw // 2)]
    s = np.arange(65536, dtype=np.uint64)
    if cb == 2:
        x = (s * 0x83DCD12D) & 0xFFFFFFFF
        total = ((x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + (x >> 24)).astype(np.float64)
        half = np.array([0x1EEE, 0xC931], dtype=np.uint16).view(np.float16).astype(np.float64)
        values = (1024.0 + total) * half[0] + half[1]
    else:
        x = s * 89226354 + 64248484 if cb == 0 else s * 0xCBAC1FED
        x = ((x & 0x8FFF8FFF) ^ 0x3B603B60).astype(np.uint32)
        values = x.view(np.float16).astype(np.float64).reshape(-1, 2).sum(axis=1)
    val = torch.from_numpy(values).to(trellis.device)[(pair >> ((last + 1) * 32 - start - 16)) & 0xFFFF]
    lane, j = t >> 3, t & 7
    pos = (2 * (lane & 3) + (j & 1) + 8 * ((j >> 1) & 1)) * 16 + (lane >> 2) + 8 * (j >> 2)
    tile = torch.empty_like(val)
    tile[:, pos] = val
    return tile.view(kt, nt, 16, 16).permute(0, 2, 1, 3).reshape(kt * 16, nt * 16)


def _rotate64(x: torch.Tensor) -> torch.Tensor:
    h = torch.ones((1, 1), dtype=torch.float64, device=x.device)
    while h.shape[0] < 128:
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return (x.reshape(-1, 128) @ (h / 128.0 ** 0.5)).view(x.shape)


def product64(x: torch.Tensor, trellis: torch.Tensor, suh: torch.Tensor, svh: torch.Tensor, K: int,
              cb: int) -> torch.Tensor:
    """x @ W in float64 from the input rotated in fp16, as every kernel takes it, and unrounded weights: what is
    left of a kernel's error is its own (the output's rounding, and its weights' if it rounds them)."""
    xr = _rotate64((x.half() * suh).double()).half().double()
    return _rotate64(xr @ weight64(trellis, K, cb)) * svh.double()


def rel_error(got: torch.Tensor, want: torch.Tensor) -> float:
    return float((got.double() - want).norm() / want.norm())


# Relative error of fp16 outputs: their rounding alone is 2^-11 / sqrt(3) of the value's binade, 2.0e-4 of the norm
# for random outputs; weights rounded to fp16 add as much again (2.2e-4), 3.0e-4 together.
EXACT_WEIGHTS_REL = 2.5e-4
