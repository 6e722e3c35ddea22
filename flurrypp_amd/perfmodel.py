"""Algorithmic work of each libflurry_hip kernel (FP64 fused path), for roofline fractions.

Bytes count every array a kernel must read or write once at its storage
precision (FP64 state, metrics and fluxes; int32 face indices); flops count
the arithmetic of the operator contractions only (flux formulas are a few
hundred flops per point and never bound these kernels).  Counts are per
launch of the kernel on a mesh with E elements and nFF face flux points of
which nFFb lie on boundaries.
"""
from __future__ import annotations

from dataclasses import dataclass

B8, B4 = 8, 4  # bytes per double / int32


@dataclass
class Work:
    bytes: float
    flops: float


def fused_work(D: int, P: int, E: int, nFF: int, nFFb: int, viscous: bool, nRK: int, time_type: int) -> dict:
    """Per-launch algorithmic bytes/flops of the fused-path kernels."""
    N, P1 = D + 2, P + 1
    S = P1 ** D
    F = 2 * D * P1 ** (D - 1)
    nFFi = nFF - nFFb
    out = {}
    # volume: U, the metric terms
    rd = E * (N * S + D * D * S)
    fl = E * N * (D * S * 2 * P1 + F * D * 2 * P1)   # divergence + normal-flux extrapolation
    if viscous:
        # 1/detJ; U across, normal, dA, side/partner code at the flux points;
        # the corrected divergence, each side's part of the LDG flux and the
        # last stage's wave speeds out
        rd += E * S + 2 * nFFi * N + E * F * (D + 1 + B4 / B8)
        wr = E * N * S + 2 * nFFi * N + nFF / nRK
        fl += E * N * (D * S * 2 * P1 + D * S * 2 * 2 * D + (D + 1) * F * 2 * P1)
        out["fused_volume_viscous"] = Work((rd + wr) * B8, fl)
    else:
        # inviscid runs: one stage kernel, which also forms the common flux and
        # applies the RK update (below); divF, the common and the discontinuous
        # normal flux stay on chip, U at the element's flux points and across
        # is read instead (with the normal, dA and the side code)
        vol_rd = rd + E * 2 * N * F + E * F * (D + 1 + B4 / B8)
        vol_wr = nFF / nRK                           # the wave speeds of the last stage
    # rk update, averaged over the stages of one step
    per_stage = []
    for st in range(nRK):
        rd = E * S                                   # detJ
        if viscous:
            # divF; the partners' LDG parts, dA, partner code
            rd += E * N * S + 2 * nFFi * N + E * F * (1 + B4 / B8)
        wr = E * (N * S + N * F)                     # U, U at the faces
        if time_type >= 5:
            rd += E * N * S                          # U0
        elif nRK == 1:
            rd += E * N * S                          # U
        elif st == 0:
            rd += E * N * S                          # U (the step's U0: stages before the last write a stage copy)
            wr += E * N * S                          # Uacc
        elif st == nRK - 1:
            rd += E * N * S                          # Uacc
        else:
            rd += 2 * E * N * S                      # U0, Uacc
            wr += E * N * S                          # Uacc
        # (divF_spts[0] is stored by the last step of an update call only, not
        # per step: not counted)
        per_stage.append((rd + wr) * B8)
    rk = Work(sum(per_stage) / len(per_stage), E * N * S * 2 * 2 * D)
    if viscous:
        out["fused_rk_update"] = rk
    else:
        out["fused_stage"] = Work((vol_rd + vol_wr) * B8 + rk.bytes, fl + rk.flops)
    return out


def mixed_work(D: int, P: int, E: int, nFF: int, nFFb: int, viscous: bool, nRK: int, time_type: int) -> dict:
    """Per-launch algorithmic bytes of the mixed-path kernels: FP32 face and
    volume intermediates, fluxes, U at the flux points, stage copy of U and
    stored stage residuals, FP32 copies of the geometry; FP64 state, stage-0
    copy, detJ and wave speeds.  Flops as for the FP64 kernels."""
    N, P1 = D + 2, P + 1
    S = P1 ** D
    F = 2 * D * P1 ** (D - 1)
    nFFi = nFF - nFFb
    f4, d8, i4 = 4, 8, 4
    fp = fused_work(D, P, E, nFF, nFFb, viscous, nRK, time_type)
    out = {}
    # volume: U (stage copy), metric terms (inviscid runs, the stage kernel:
    # with U at the flux points and across, normal, dA and side code, and the
    # last stage's wave speeds)
    rd = E * f4 * (N * S + D * D * S)
    if not viscous:
        rd += E * F * (f4 * (2 * N + D + 1) + i4) + nFF * d8 / nRK
    if viscous:
        # 1/detJ; U across, normal, dA, side code; divF, the flux jump, the LDG
        # side parts and the last stage's wave speeds out
        rd += E * (f4 * (S + D * F + F) + i4 * F) + f4 * 2 * nFFi * N
        wr = E * f4 * (N * S + N * F) + f4 * 2 * nFFi * N + nFF * d8 / nRK
        out["mixed_volume_viscous"] = Work(rd + wr, fp["fused_volume_viscous"].flops)
    # classical RK stages keep their residuals in FP32 (the form without a
    # multigrid source); the FP64 state, written at the last stage only, is
    # also the step's U0; Jameson-form stages read it and write the state last
    per_stage = []
    for st in range(nRK):
        rd_ = E * d8 * S                               # detJ
        if viscous:
            # divF, the flux jump, dA, code; the partner's LDG part
            rd_ += E * (f4 * (N * S + N * F + F) + i4 * F) + f4 * 2 * nFFi * N
        wr_ = E * (f4 * N * F + f4 * N * S)            # U at the faces, stage copy of U
        if time_type >= 5:
            rd_ += E * d8 * N * S                      # U0
            if st == nRK - 1:
                wr_ += E * d8 * N * S                  # U
        elif nRK == 1:
            rd_ += E * d8 * N * S
            wr_ += E * d8 * N * S
        elif st == 0:
            rd_ += E * d8 * N * S                      # U (the step's U0 until the last stage writes it)
            wr_ += E * f4 * N * S                      # residual of stage 0
        elif st == nRK - 1:
            rd_ += E * (d8 * N * S + f4 * N * S * (nRK - 1))  # U0, stored residuals
            wr_ += E * d8 * N * S                      # U
        else:
            rd_ += E * d8 * N * S                      # U0
            wr_ += E * f4 * N * S                      # residual of this stage
        per_stage.append(rd_ + wr_)
    rk = sum(per_stage) / len(per_stage)
    if viscous:
        out["mixed_rk_update"] = Work(rk, fp["fused_rk_update"].flops)
    else:
        out["mixed_stage"] = Work(rd + rk, fp["fused_stage"].flops)
    return out


def hbm_bound(w: Work, peak_tf: float = 78.6, peak_bw: float = 8.0) -> bool:
    """True when the kernel's intensity is under the FP64 ridge point."""
    if w.bytes == 0:
        return False
    return (w.flops / w.bytes) < (peak_tf / peak_bw)
