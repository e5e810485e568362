"""GEMM tile autotuning for gfx950 (CDNA4).

Flow as in the reference autotuner (``tensorjit/runtime/autotune.py:83-118``):
an analytic cost model ranks the candidate tile configurations, only the
best ``top_k`` are compiled and timed on real buffers, and the winner is
persisted in ``AutotuneStore`` so later processes start warm.

The model is re-derived for MI355X instead of the reference's GPU branch
(``autotune.py:73-79``): times fitted to measurements for the ring, direct-to-LDS and decode
schedules, and for register-staged tiles the slowest of

* MFMA time: 2*M*N*K at the dense matrix-core peak, scaled by how well the
  tile grid fills 256 CUs (tail rounds of workgroups) and by edge waste;
* LDS time: every wave re-reads its A and B fragments from LDS each K step
  (128 B/clk/CU);
* L2 time: each workgroup streams a (BM + BN) x K panel;
* HBM time: A, B and C once at 8 TB/s.

It rejects staged tiles that exceed 160 KiB of double-buffered LDS or 512 VGPRs
(accumulators + fragments + staging) per lane.
"""
from __future__ import annotations

import math
import os
import time
from dataclasses import dataclass
from typing import Callable, Sequence

from .cache import AutotuneStore

# MI355X (gfx950) figures used by the model.
CU_COUNT = 256
CLOCK_HZ = 2.4e9
LDS_BYTES_PER_CU = 160 * 1024
LDS_BYTES_PER_CLK = 128
MFMA_FLOP_PER_CLK_BF16 = 4096   # per CU: 2.5 PF / 256 CU / 2.4 GHz
MFMA_FLOP_PER_CLK_F32 = 256     # per CU: 157.3 TF / 256 CU / 2.4 GHz
HBM_BYTES_PER_S = 8.0e12
L2_BYTES_PER_S = 16.0e12


@dataclass(frozen=True)
class MatmulConfig:
    """A GEMM tiling: block tile TM x TN, K step TK, ``num_warps`` waves of 64 lanes.

    ``WM`` x ``WN`` is the wave grid inside the workgroup (``WM * WN == num_warps``)
    and ``MI`` the MFMA tile edge (32 -> 32x32 blocks, 16 -> 16x16 blocks).
    ``SPLIT_K`` > 1 splits K across the waves of a workgroup (skinny GEMMs).
    """

    TM: int
    TN: int
    TK: int = 0
    num_warps: int = 4
    WM: int = 2
    WN: int = 2
    MI: int = 32
    SPLIT_K: int = 1
    GROUP_M: int = 8        # tile rows per group of the XCD-aware tile order (0 = plain row-major order)
    PINGPONG: int = 0       # two wave groups alternate MFMA and memory phases: 1/2 = loads 2/3 K steps ahead, 3 = K-split tiles
    INTERLEAVE: int = 0     # 1: one wave per SIMD, memory instructions threaded between its MFMAs
    DIRECT: int = 0         # 1: one wave per SIMD, tiles loaded straight into LDS (buffer_load_dwordx4 ... lds)
    KSPLIT: int = 1         # > 1: K split over that many workgroups, partials summed by the last of them
    PERSIST: int = 0        # > 0 (DIRECT only): that many workgroups (one per CU) loop over the output tiles
    STAGES: int = 0         # > 0: ring of that many LDS stages filled by DMA (small tiles, NT and NN, any KSPLIT)

    def as_dict(self) -> dict:
        return {"TM": self.TM, "TN": self.TN, "TK": self.TK, "num_warps": self.num_warps,
                "WM": self.WM, "WN": self.WN, "MI": self.MI, "SPLIT_K": self.SPLIT_K, "GROUP_M": self.GROUP_M,
                "PINGPONG": self.PINGPONG, "INTERLEAVE": self.INTERLEAVE, "DIRECT": self.DIRECT, "KSPLIT": self.KSPLIT,
                "PERSIST": self.PERSIST, "STAGES": self.STAGES}

    @staticmethod
    def from_dict(d: dict) -> "MatmulConfig":
        return MatmulConfig(d["TM"], d["TN"], d.get("TK", 0), d.get("num_warps", 4), d.get("WM", 2),
                            d.get("WN", 2), d.get("MI", 32), d.get("SPLIT_K", 1), d.get("GROUP_M", 8),
                            d.get("PINGPONG", 0), d.get("INTERLEAVE", 0), d.get("DIRECT", 0), d.get("KSPLIT", 1),
                            d.get("PERSIST", 0), d.get("STAGES", 0))


# bf16 / fp16 candidates (MFMA 32x32x16 or 16x16x32)
HIP_CANDIDATES: list[MatmulConfig] = [
    # persistent direct-to-LDS kernels: one workgroup per CU looping over the output tiles
    MatmulConfig(256, 256, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1, 1, CU_COUNT),
    MatmulConfig(256, 128, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1, 1, CU_COUNT),
    MatmulConfig(256, 256, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(256, 128, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    # 192-row and 192-column tiles: where 256 leaves a nearly empty last round of workgroups
    # (bf16 2000 x 11008 x 4096 with bias and gelu, kernel on repeated buffers: 344 tiles of
    # 256x256 174 us, 464 of 256x192 144)
    MatmulConfig(256, 192, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(192, 256, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(192, 192, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(192, 128, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(128, 192, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(256, 256, 64, 4, 2, 2, 32, 1, 8, 0, 0, 1),
    MatmulConfig(256, 128, 64, 4, 2, 2, 32, 1, 8, 0, 0, 1),
    # mid-size products (a few hundred 256x256 tiles or fewer): smaller direct tiles fill the CUs
    MatmulConfig(128, 128, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(128, 64, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(64, 128, 64, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(256, 256, 64, 8, 2, 4, 32, 1, 8, 3),
    MatmulConfig(256, 256, 64, 8, 4, 2, 32, 1, 8, 3),
    MatmulConfig(256, 256, 32, 8, 2, 4, 32, 1, 8, 2),
    MatmulConfig(256, 256, 32, 8, 4, 2, 32, 1, 8, 2),
    MatmulConfig(256, 256, 32, 8, 2, 4, 32, 1, 8, 1),
    MatmulConfig(256, 256, 32, 8, 4, 2, 32, 1, 8, 1),
    MatmulConfig(256, 128, 32, 8, 4, 2, 32, 1, 8, 2),
    MatmulConfig(256, 128, 32, 8, 4, 2, 32, 1, 8, 1),
    MatmulConfig(256, 256, 64, 8, 2, 4, 32),
    MatmulConfig(256, 256, 32, 8, 2, 4, 32),
    MatmulConfig(256, 128, 64, 8, 4, 2, 32),
    MatmulConfig(256, 256, 64, 4, 2, 2, 32, 1, 8, 0, 1),
    MatmulConfig(256, 256, 32, 4, 2, 2, 32, 1, 8, 0, 1),
    MatmulConfig(256, 128, 64, 4, 2, 2, 32),
    MatmulConfig(128, 256, 64, 4, 2, 2, 32),
    MatmulConfig(128, 128, 64, 4, 2, 2, 32),
    MatmulConfig(128, 128, 32, 4, 2, 2, 32),
    MatmulConfig(128, 64, 64, 4, 2, 2, 32),
    MatmulConfig(64, 128, 64, 4, 2, 2, 32),
    MatmulConfig(64, 64, 64, 4, 2, 2, 16),
    MatmulConfig(64, 64, 32, 4, 2, 2, 16),
    MatmulConfig(32, 64, 64, 4, 2, 2, 16),
    # skinny (M <= 16 / 32): one MI x MI tile per workgroup, K split over its waves
    MatmulConfig(16, 32, 64, 4, 1, 1, 16, 4, 0),
    MatmulConfig(16, 32, 128, 4, 1, 1, 16, 4, 0),
    MatmulConfig(16, 32, 128, 2, 1, 1, 16, 2, 0),
    MatmulConfig(32, 32, 64, 4, 1, 1, 32, 4, 0),
    MatmulConfig(16, 32, 256, 8, 1, 1, 16, 8, 0),
    MatmulConfig(16, 64, 256, 8, 1, 1, 16, 8, 0),
    MatmulConfig(16, 32, 128, 16, 1, 1, 16, 16, 0),
    MatmulConfig(16, 64, 128, 16, 1, 1, 16, 16, 0),
    MatmulConfig(16, 16, 256, 8, 1, 1, 16, 8, 0),
    MatmulConfig(32, 32, 128, 8, 1, 1, 32, 8, 0),
    MatmulConfig(32, 64, 64, 16, 1, 1, 32, 16, 0),
]

# fp32 candidates (MFMA 32x32x2 / 16x16x4 f32)
HIP_F32_CANDIDATES: list[MatmulConfig] = [
    # direct-to-LDS (32-deep K tiles: the bf16 kernel's 128-byte rows), 16x16x4 MFMAs
    MatmulConfig(128, 128, 32, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(128, 256, 32, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(256, 128, 32, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(128, 128, 32, 4, 2, 2, 16, 1, 8, 0, 0, 1, 1, CU_COUNT),
    MatmulConfig(64, 64, 32, 4, 2, 2, 16, 1, 8, 0, 0, 1),
    MatmulConfig(128, 128, 16, 4, 2, 2, 32),
    MatmulConfig(128, 128, 32, 4, 2, 2, 32),
    MatmulConfig(128, 64, 32, 4, 2, 2, 32),
    MatmulConfig(64, 128, 32, 4, 2, 2, 32),
    MatmulConfig(64, 64, 32, 4, 2, 2, 16),
    MatmulConfig(64, 64, 16, 4, 2, 2, 16),
    MatmulConfig(32, 32, 32, 4, 2, 2, 16),
    MatmulConfig(32, 64, 32, 4, 2, 2, 16),
    MatmulConfig(64, 32, 32, 4, 2, 2, 16),
    MatmulConfig(32, 32, 64, 4, 2, 2, 16),
    # K split over workgroups (few output tiles, long K: config 1's 512x768x3072)
    MatmulConfig(64, 64, 32, 4, 2, 2, 16, 1, 8, 0, 0, 0, 8),
    MatmulConfig(64, 64, 32, 4, 2, 2, 16, 1, 8, 0, 0, 0, 4),
    MatmulConfig(32, 32, 64, 4, 2, 2, 16, 1, 8, 0, 0, 0, 4),
    MatmulConfig(32, 64, 64, 4, 2, 2, 16, 1, 8, 0, 0, 0, 4),
]


def ring_candidates(M: int, N: int, K: int, batch: int, itemsize: int) -> list[MatmulConfig]:
    """Ring-schedule tilings of one product: the tiles below with K split over 1-12
    workgroups, as far as the split still has work (two K tiles per part) and the grid is not
    full without it (four workgroups per CU)."""
    tk = 128 // itemsize
    kt = -(-K // tk)
    out = []
    for tm, tn, waves, wm, wn, stages in RING_TILES:
        if tm > 32 and tm >= 2 * M:
            continue
        tiles = -(-M // tm) * -(-N // tn) * batch
        for s in (1, 2, 3, 4, 6, 8, 12):
            if s > 1 and (tiles * s > 4 * CU_COUNT or kt < 2 * s):
                break
            out.append(MatmulConfig(tm, tn, tk, waves, wm, wn, 16, 1, 8, 0, 0, 0, s, 0, stages))
    return out


# (TM, TN, waves, WM, WN, STAGES): 32 KiB (32x32) to 128 KiB (128x128) of LDS.  Of these the small tiles
# win while the grid leaves CUs idle, 128x128 with 8 waves (two per SIMD, one workgroup per CU)
# once it is full.
RING_TILES = [
    (32, 32, 4, 2, 2, 4), (32, 64, 4, 2, 2, 4), (32, 64, 4, 2, 2, 3), (32, 128, 4, 1, 4, 4),
    (64, 64, 4, 2, 2, 4), (64, 64, 4, 2, 2, 3), (64, 128, 4, 2, 2, 3), (128, 64, 4, 2, 2, 3),
    (128, 128, 8, 4, 2, 4),
]


def _hbm_us(M: int, N: int, K: int, batch: int, elem: int, mats: tuple[int, int] | None = None) -> float:
    """``mats``: distinct A and B matrices of the batch (a weight shared by all is read once)."""
    na, nb = mats or (batch, batch)
    return (M * K * na + N * K * nb + M * N * batch) * elem * 1e-6


def _ring_cost(cfg: MatmulConfig, M: int, N: int, K: int, batch: int, elem: int,
               mats: tuple[int, int] | None = None) -> float:
    """Microseconds of a ring-schedule product.  The busiest CU runs ``w`` workgroups, ``occ`` at
    a time; each K tile costs its MFMAs, its DMA bytes and a latency share; HBM once; each round
    an epilogue; a K split its partials.  The constants are fitted to measured times of decode,
    prompt and MLP shapes; over 165 other products, chosen where schedules are close, the
    estimate is off by 21% rms in 16 bits (with the factors of ``cost_model``), 6% in fp32 and
    28% where a batch shares its weight, and the schedule it chooses is within 4% of the best
    measured one in 154."""
    tm, tn, S = cfg.TM, cfg.TN, cfg.KSPLIT
    per = -(-(-(-K // cfg.TK)) // S)
    wgs = -(-M // tm) * -(-N // tn) * batch * S
    occ = max(1, min(LDS_BYTES_PER_CU // (cfg.STAGES * (tm + tn) * 128 + 64), 32 // cfg.num_warps))
    w = -(-wgs // CU_COUNT)
    rounds, conc = -(-w // occ), min(w, occ)
    mflop = tm * tn * cfg.TK * 2e-6 * (0.2465 if elem == 2 else 2.04) * (0.88 if cfg.num_warps == 8 else 1.0)
    t_mfma = w * per * mflop
    t_dma = w * per * (tm + tn) * 0.128 * 0.0085
    t_lat = rounds * per * 0.1 / (cfg.STAGES - 1) ** 0.89
    mem = _hbm_us(M, N, K, batch, elem, mats)
    t_hbm = mem / 9.42
    edge = 4.0 if N % (16 // elem) else 1.0                       # element-wise stores of ragged rows
    t_epi = rounds * (0.62 + tm * tn * 1e-3 * 0.104 * conc * edge)
    t_split = 1.35 + 0.02 * S * tm * tn * 0.004 * max(1.0, w / S) if S > 1 else 0.0
    t_loop = (t_mfma ** 3.1 + t_dma ** 3.1 + t_lat ** 3.1 + t_hbm ** 3.1) ** (1 / 3.1)
    return 1.5 + max(t_loop + rounds * per * 0.034, mem / 7.0) + t_epi + t_split


# 16-bit direct-to-LDS tiles: (microseconds per K tile of a round with one workgroup per CU,
# with all that fit, microseconds of a full round's epilogue), workgroups per CU; fitted to
# prompt and MLP products without a batch (2000 x 11008 x 4096 plain: estimate 130, measured 134;
# the calls around such a kernel take 172, with new buffers each)
DIRECT_US = {
    (64, 128): (0.467, 0.704, 8.9, 3), (128, 64): (0.418, 0.790, 1.5, 3), (128, 128): (0.570, 0.815, 3.0, 2),
    (128, 192): (0.663, 1.034, 7.8, 2), (192, 128): (0.651, 1.044, 7.25, 2), (192, 192): (0.736, 0.736, 8.2, 1),
    (192, 256): (0.818, 0.818, 12.0, 1), (256, 192): (0.817, 0.817, 11.9, 1), (256, 128): (0.751, 0.751, 6.25, 1),
    (256, 256): (0.989, 0.989, 16.9, 1),
}
PERSIST_US = {(256, 256): (0.879, 25.3), (256, 128): (0.737, 9.3)}


def _direct_cost(cfg: MatmulConfig, M: int, N: int, K: int, batch: int, elem: int,
                 mats: tuple[int, int] | None = None) -> float:
    """Microseconds of a direct-to-LDS product: whole rounds of ``occ`` workgroups per CU, then
    the last round at the concurrency it has left."""
    tm, tn = cfg.TM, cfg.TN
    per = -(-K // cfg.TK)
    wgs = -(-M // tm) * -(-N // tn) * batch
    if elem == 2 and (tm, tn) in DIRECT_US:
        one, full, epi, occ = DIRECT_US[(tm, tn)]
        if cfg.PERSIST and (tm, tn) in PERSIST_US:
            one = full = PERSIST_US[(tm, tn)][0]
            epi = PERSIST_US[(tm, tn)][1]
    else:
        occ = 1 if cfg.PERSIST else max(1, min(LDS_BYTES_PER_CU // (2 * (tm + tn) * 128), 2))
        mflop = tm * tn * cfg.TK * 2e-6 * (0.14 if elem == 2 else 2.0)
        one, epi = mflop + (tm + tn) * 1e-3 * 0.396, tm * tn * 1e-3 * 0.2156 * occ
        full = one * occ
    if cfg.MI == 32:
        one, full = one * 1.1, full * 1.1                         # lower clock on random data
    if N % (16 // elem):
        epi *= 4.0                                                # element-wise stores of ragged rows
    rounds = -(-wgs // (CU_COUNT * occ))
    last = -(-(wgs - (rounds - 1) * CU_COUNT * occ) // CU_COUNT)
    step = one + (full - one) * (last - 1) / (occ - 1) if occ > 1 else full
    t = (rounds - 1) * (per * full + epi) + per * step + epi * last / occ
    return 1.5 + max(t, _hbm_us(M, N, K, batch, elem, mats) / 7.0)


# The register-staged tilings that still beat the ring where no direct-to-LDS tile applies:
# 256x256 with 8 waves, K step 32 or 64.  (NT, PINGPONG) -> us per K step of a round, us per
# round beside its K loop, and the loss (M, N) from a last tile that is cut.  us, 16-bit, ring
# (128x128) / the best of these:
#   NN 8192^3 1005 / 921, 16384 x 4096 x 4096 519 / 485, 1000 x 16384 x 4096 136 / 125, 64 of
#   512^3 38.5 / 25.9; but 2048 x 4096 x 4096 66 / 77, 2048 x 11008 x 4096 188 / 209, 6000^3
#   462 / 531 (half-empty rounds of workgroups)
#   NT with K no multiple of 64: 8192 x 8192 x 8200 1254 / 916, 2048 x 11008 x 4104 242 / 192,
#   900 x 11008 x 4104 121 / 107; but 1500 x 11008 x 2056 108 / 116
# No smaller staged tile, and none in fp32, was the fastest of 63 shapes.  Of 60 further random
# shapes at which the two estimates are close, the choice is the slower one at 7, always the
# ring: by 7-15%, and at 84 x 1152 x 184 x 496 62 / 43.
STAGED_US = {
    (False, 1): (0.915, 6.6, 1.0, 1.0), (False, 2): (0.910, 6.6, 1.17, 1.17), (False, 3): (2.3, 9.0, 1.5, 1.5),
    (True, 1): (0.96, 4.0, 1.0, 1.0), (True, 2): (0.968, 8.0, 1.12, 1.12), (True, 3): (1.66, 10.0, 1.08, 1.3),
}


def beside_ring(cfg: MatmulConfig) -> bool:
    """A register-staged tiling that is kept where the ring schedule applies too."""
    return cfg.PINGPONG > 0 and (cfg.TM, cfg.TN, cfg.WM, cfg.TK) == (256, 256, 2, 64 if cfg.PINGPONG == 3 else 32)


def _staged_us(cfg: MatmulConfig, M: int, N: int, K: int, batch: int, tb: bool) -> float:
    """Microseconds of a ``beside_ring`` tiling: whole rounds of one workgroup per CU; a last
    round that is not full runs at a higher clock and rate."""
    step, epi, cut_m, cut_n = STAGED_US[(tb, cfg.PINGPONG)]
    wgs = -(-M // cfg.TM) * -(-N // cfg.TN) * batch
    rounds = -(-wgs // CU_COUNT)
    last = 0.7 + 0.3 * (wgs - (rounds - 1) * CU_COUNT) / CU_COUNT
    cut = max(cut_m if M % cfg.TM else 1.0, cut_n if N % cfg.TN else 1.0)
    # what the estimate misses: a launch's start, few K steps, output rows off the 128-byte lines
    lead = (1.24 if not tb and N % 64 else 1.0) / (0.93 if K < 256 else 1.0)
    epi += 13.0 if N % 8 else 0.0                                 # element-wise stores
    return ((rounds - 1 + last) * (-(-K // cfg.TK) * step + epi) * cut + 2.0) * lead


def _skinny_cost(cfg: MatmulConfig, M: int, N: int, K: int, batch: int, elem: int,
                 mats: tuple[int, int] | None = None) -> float:
    """Streaming kernel (M <= 16 / 32), from 35 shapes of 1-16 rows on MI355X: HBM, or rounds
    of one workgroup per CU whose waves each run K / SPLIT_K serially (8 waves of 16 columns
    0.83 ns per k, 4 or 2 waves of 32 columns 1.9)."""
    if M > cfg.TM or elem != 2:
        return math.inf
    rounds = -(-(-(-N // cfg.TN) * batch) // CU_COUNT)
    per_k = 0.00083 if cfg.TN == 16 else 0.0019
    if cfg.SPLIT_K == 8 and (K // cfg.SPLIT_K) % 256:
        per_k *= 1.3                                              # A is read in fragments, not through LDS
    if cfg.TM == 32:
        per_k *= 2.2
    if mats and mats[1] < batch:
        # a batch that shares its weight: [64, 1, 4096] x 4096 242 us where the ring takes 88,
        # [2, 1, 4096] x 4096 9.6 (8.2), [16, 16, 1024] x 1024 5.8 (4.0)
        per_k *= 1.7
    extra = {4: 1.0, 2: 1.04, 8: 1.06, 16: 1.1}.get(cfg.SPLIT_K, 1.2) * (1.0 if cfg.TN <= 32 else 1.05)
    return 1.5 + max(rounds * K * per_k, _hbm_us(M, N, K, batch, elem, mats) / 6.85) * extra


def _sched_factor(cfg: MatmulConfig) -> float:
    """Relative MFMA-phase cost of a register-staged loop schedule, from bf16 NT 8192^3 runs on
    MI355X (the plain double-buffered loop ~9% behind ping-pong with K-split tiles)."""
    if cfg.INTERLEAVE:
        return 1.15
    return {3: 1.0, 2: 1.04, 1: 1.05}.get(cfg.PINGPONG, 1.09)


def _hip_cost(cfg: MatmulConfig, M: int, N: int, K: int, batch: int, elem: int,
              mats: tuple[int, int] | None = None) -> float:
    if cfg.SPLIT_K > 1:
        return _skinny_cost(cfg, M, N, K, batch, elem, mats)
    if cfg.STAGES:
        return _ring_cost(cfg, M, N, K, batch, elem, mats)
    if cfg.DIRECT:
        return _direct_cost(cfg, M, N, K, batch, elem, mats)
    tm, tn, tk = cfg.TM, cfg.TN, cfg.TK or 32
    waves = cfg.num_warps
    if tm % (cfg.WM * cfg.MI) or tn % (cfg.WN * cfg.MI):
        return math.inf
    pad = 16 // elem
    lds = 2 * (tm + tn) * (tk + pad) * elem
    if lds > LDS_BYTES_PER_CU:
        return math.inf
    acc = tm * tn / (64 * waves)
    frags = 2 * (tm / cfg.WM + tn / cfg.WN) / cfg.MI * (4 if elem == 2 else 1)  # double-buffered
    staging = (tm + tn) * tk * elem / (64 * waves * 4)                      # staged K step per lane, 4 B per VGPR
    regs = acc + frags + staging + 32
    if regs > 512:
        return math.inf
    # workgroups per CU: LDS, and registers (a SIMD holds 512 per lane; waves spread over 4 SIMDs)
    occ = max(1, min(LDS_BYTES_PER_CU // lds, int(512 // regs) * 4 // waves, 32 // waves))
    S = cfg.KSPLIT
    tiles = -(-M // tm) * -(-N // tn) * batch * S                  # a K split multiplies the workgroups
    kt = K / S                                                     # ... each over 1/S of K
    slots = CU_COUNT * occ
    rounds = -(-tiles // slots)
    fill = tiles / (rounds * slots)
    busy_cus = min(1.0, tiles / CU_COUNT)
    edge = (M / (-(-M // tm) * tm)) * (N / (-(-N // tn) * tn))
    flops = 2.0 * M * N * K * batch
    peak = (MFMA_FLOP_PER_CLK_BF16 if elem == 2 else MFMA_FLOP_PER_CLK_F32) * CU_COUNT * CLOCK_HZ
    t_mfma = flops / (peak * max(fill, 1e-3) * max(busy_cus, 1e-3) * edge) * _sched_factor(cfg)
    # LDS: per K step each wave reads (tm/WM + tn/WN) x tk elements; per CU per tile
    lds_bytes_tile = waves * (tm / cfg.WM + tn / cfg.WN) * kt * elem
    lds_bytes_tile += (tm + tn) * kt * elem                        # the global->LDS writes
    t_lds = tiles * lds_bytes_tile / (LDS_BYTES_PER_CLK * CLOCK_HZ * min(CU_COUNT, tiles))
    t_l2 = tiles * (tm + tn) * kt * elem / L2_BYTES_PER_S
    t_hbm = (M * K + N * K + M * N) * batch * elem / HBM_BYTES_PER_S
    # a workgroup writes its output tile after its K loop; with one workgroup per CU
    # nothing overlaps that store, which matters when the output dominates (small K)
    t_out = M * N * batch * (4 * S if S > 1 else elem) / HBM_BYTES_PER_S / occ
    # split K: the S fp32 partials are read back and the output written after the last
    # split finishes (in the tile's last workgroup, ~2.3 us of tail at config 1, or a second launch)
    t_sum = ((S * 4 + elem) * M * N * batch / HBM_BYTES_PER_S + 4e-6) if S > 1 else 0.0
    t = max(t_mfma, t_lds, t_l2, t_hbm) + t_out + t_sum
    return t * 1e6


def fp32_factor(cfg: MatmulConfig, M: int, N: int, batch: int) -> float:
    """Measured time of an fp32 tiling of a full grid over its estimate: 0.73-0.87 for the
    direct-to-LDS tiles (64x64 to 128x256, 15 NT shapes), 0.83-0.89 for the ring's 4-wave tiles
    two and more to a CU (14 shapes), 1 for its 128x128."""
    if cfg.DIRECT:
        return 0.79
    wgs = -(-M // cfg.TM) * -(-N // cfg.TN) * batch * cfg.KSPLIT
    return 0.86 if cfg.STAGES and cfg.num_warps == 4 and wgs >= 2 * CU_COUNT else 1.0


def cost_model(cfg: MatmulConfig, M: int, N: int, K: int, backend: str, batch: int = 1,
               ring_nt: bool | None = None, mats: tuple[int, int] | None = None) -> float:
    """Lower is better.  ``backend``: "hip" (bf16/fp16) or "hip_f32"; CPU kinds
    "c" / "c_dot" keep the reference's register-pressure heuristic.  ``ring_nt``: whether B is
    stored [N][K], given where ring and register-staged tilings compete; ``mats``: distinct A
    and B matrices of the batch (default: as many as products)."""
    if backend == "hip" and ring_nt is not None:
        if cfg.PINGPONG:
            return _staged_us(cfg, M, N, K, batch, ring_nt)
        if cfg.STAGES:
            # the ring beside these: 0.91 of its model, or where B's rows start inside a
            # 128-byte line 1.13 (NT) and 1.06 (NN)
            return _hip_cost(cfg, M, N, K, batch, 2, mats) * (1.13 if ring_nt else 1.06 if N % 64 else 0.91)
    if backend in ("hip", "hip_f32"):
        return _hip_cost(cfg, M, N, K, batch, 2 if backend == "hip" else 4, mats)
    tm, tn = cfg.TM, cfg.TN
    tk = cfg.TK or K
    cost = (4.0 * (tm * tk + tk * tn)) / (2.0 * tm * tn * tk)
    cost /= (M / (-(-M // tm) * tm)) * (N / (-(-N // tn) * tn))
    if backend == "c_dot":
        regs = tm * tn + tm
        if regs > 14:
            cost *= (regs / 14.0) ** 2
    elif backend == "c":
        regs = tm * tn / 8.0
        if regs > 12:
            cost *= 1.0 + (regs - 12) / 4.0
    if M / tm < 2 * (os.cpu_count() or 1):
        cost *= 1.3
    return cost


def _wall_timer(run: Callable[[], None], warmup: int, iters: int) -> float:
    for _ in range(warmup):
        run()
    t0 = time.perf_counter()
    for _ in range(iters):
        run()
    return (time.perf_counter() - t0) / iters * 1e3


def autotune(
    key: str,
    candidates: Sequence[MatmulConfig],
    build: Callable[[MatmulConfig], Callable[[], None]],
    shape: tuple,
    backend: str,
    top_k: int = 4,
    store: AutotuneStore | None = None,
    warmup: int = 2,
    iters: int = 5,
    timer: Callable[[Callable[[], None], int, int], float] | None = None,
    rounds: int = 1,
    rank: Callable[[MatmulConfig], float] | None = None,
) -> MatmulConfig:
    """Fastest candidate by measurement; ``build(cfg)`` returns a runner for ``timer``.

    ``timer(run, warmup, iters) -> ms`` measures one runner (device-event timing for
    GPU kernels).  All runners are built first, then timed in ``rounds`` interleaved
    passes keeping each candidate's best time, so clock ramp-up or a noisy
    neighbour cannot favour whichever candidate happened to run last.  Candidates
    whose build or run raises are skipped.  ``rank`` replaces the cost model's order.
    """
    store = store or AutotuneStore()
    M, N, K = shape[:3]
    batch = shape[3] if len(shape) > 3 else 1
    rank = rank or (lambda c: cost_model(c, M, N, K, backend, batch))
    if os.environ.get("TENSORJIT_NO_AUTOTUNE") == "1":
        return min(candidates, key=rank)
    cached = store.get(key)
    if cached is not None:
        return MatmulConfig.from_dict(cached["config"])
    ranked = [c for c in sorted(candidates, key=rank) if math.isfinite(rank(c))][:top_k]
    if not ranked:
        ranked = [min(candidates, key=rank)]
    timer = timer or _wall_timer
    runners = []
    for cfg in ranked:
        try:
            runners.append((cfg, build(cfg)))
        except Exception:  # invalid for this shape: skip it
            continue
    best_of = {}
    for _ in range(max(1, rounds)):
        for cfg, run in runners:
            try:
                ms = timer(run, warmup, iters)
            except Exception:
                continue
            best_of[cfg] = min(ms, best_of.get(cfg, math.inf))
    if not best_of:
        best, best_ms = ranked[0], math.inf
    else:
        best = min(best_of, key=best_of.get)
        best_ms = best_of[best]
    store.put(key, best.as_dict(), best_ms)
    return best


__all__ = ["MatmulConfig", "HIP_CANDIDATES", "HIP_F32_CANDIDATES", "cost_model", "autotune"]
