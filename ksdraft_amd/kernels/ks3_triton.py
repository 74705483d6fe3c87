"""``project_fused`` under the reference's module name (ksdraft/kernels/ks3_triton.py).

The reference's Triton kernel fuses the down-projection GEMM, the Horner spine, ReLU^2 and
the per-group requantization (ks3_triton.py:100-156), following the fused kernel's own
arithmetic contract, not the composed one.

* 'int8' (NL == 2) with group 128, where _one_launch_pays: ksd_ks3_project_fused. Up to 256
  rows (decode and short prefill) it keeps the GEMM's accumulator in its workspace and runs the
  fused contract on it (fp32 coordinates and LUT index, no truncation, group pre-scale, second
  requantization): at d 1536, F 5888 on MI355X 9 us at M = 1 and 23 at M = 256. Past them it is
  the reference's single-kernel form, a GEMM whose epilogue runs the contract on each finished
  tile, with no accumulator in memory. The accumulator is the unsplit ordered sum over all K
  groups, so the entry is taken only where the standalone GEMM would not split K either: the
  outputs are then identical to the other form's.
* 'int8' otherwise: ksd_w8a8_gemm_nt (fp32 accumulator out), then ksd_ks3_spine_fused, the
  same per-element arithmetic. ``one_launch`` forces either form. The single kernel gathers
  the per-chart table (128 KB per 128-chart tile) from L2, as it cannot sit in LDS beside the
  GEMM's operand ring.
* 'fp16' and 'fp32' (NL == 1, 0; ks3_triton.py:76-98): ksd_ks3_spine_float on the
  accumulator (the coordinates not rounded to fp16, the warp scalars in fp16), every
  fp16/fp32 op of the Triton source rounded separately.
"""

from __future__ import annotations

import torch

from .. import _lib
from .gemm import _prepare, gemm_splits, w8a8_gemm
from .ks3_int8 import spine_float, spine_fused_int8

FP16 = torch.float16
TANH_DOMAIN = 3.2


def project_fused(
    a_codes: torch.Tensor, a_scales: torch.Tensor,
    w_codes: torch.Tensor, w_scales: torch.Tensor,
    spine_codes: torch.Tensor, spine_scale: torch.Tensor,
    warp_scale: torch.Tensor, warp_shift: torch.Tensor,
    tanh_lut: torch.Tensor,
    group: int, nonlinear: str, *, one_launch: bool | None = None,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Input projection + Horner spine + requant (ks3_triton.py:159-195).

    warp_scale/warp_shift: dequantized fp16 per-chart scalars. one_launch: None picks the
    form by shape (see above); True forces ksd_ks3_project_fused ('int8', group 128 only),
    False the GEMM and the spine. Returns (h_codes int8 (M, N), h_scales fp16 (M, ceil(N/group)))."""
    if group & (group - 1):
        raise ValueError("group must be a power of two (32 or 128)")
    nl = {"fp32": 0, "fp16": 1, "int8": 2}[nonlinear]
    if one_launch and (nl != 2 or group != 128):
        raise ValueError("one_launch: 'int8' with group 128 only")
    if one_launch is None:
        one_launch = nl == 2 and group == 128 and _one_launch_pays(a_codes, w_codes)
    if one_launch:
        out = _project_fused_int8(a_codes, a_scales, w_codes, w_scales, spine_codes, spine_scale,
                                  warp_scale.to(FP16), warp_shift.to(FP16), tanh_lut)
        if out is not None:
            return out
    acc = w8a8_gemm(a_codes, a_scales, w_codes, w_scales, group)
    if nl == 2:
        return spine_fused_int8(acc, spine_codes, spine_scale, warp_scale.to(FP16),
                                warp_shift.to(FP16), tanh_lut, group)
    _, hq, hs = spine_float(acc, spine_codes, spine_scale, warp_scale.to(FP16).float(),
                            warp_shift.to(FP16).float(), nonlinear, group)
    return hq, hs


# Largest M for which project_fused may take ksd_ks3_project_fused by default.
ONE_LAUNCH_MAX_ROWS = 1024
# Largest M for which that entry is the GEMM and the table-free spine, the accumulator in its table
# workspace (the entry's own limit: 256 values a chart); past it, the single GEMM launch.
_ACC_ROWS = 256


def _one_launch_pays(a_codes: torch.Tensor, w_codes: torch.Tensor) -> bool:
    """Whether ksd_ks3_project_fused is the faster form, at a GEMM shape the standalone launch
    would not split along K (so both forms compute the same ordered accumulator).

    Up to 256 rows it is the same two kernels in one call. Past them it is the single launch: its
    time goes with the rounds of 128 x 128 tiles over the CUs (256), N (the table) and K, and
    hardly with the M N values, which the GEMM and the spine store and read, more slowly in rows
    that are not 16-byte aligned (N % 4). The lines below are least squares over 642 shapes (M 257
    to 1024, K 128 to 2048, N 1536 to 8192; us saved against us spent, sizes in thousands, values in
    millions): the form they pick is within 11 percent of the faster one. Both sides (us, single and
    two, M x K -> N): 512 x 1536 -> 5888 34, 29; 1024 x 128 -> 4096 24, 33; 1024 x 1536 -> 4096 35,
    36; 512 x 128 -> 3001 20, 19; 1024 x 128 -> 3001 22, 29; 512 x 768 -> 5001 25, 28; 1024 x 1536
    -> 5001 56, 52; 1024 x 768 -> 6869 53, 55; 1024 x 128 -> 6912 41, 47; 1024 x 512 -> 6912 49, 47."""
    if a_codes.dim() != 2 or w_codes.dim() != 2:
        return False
    M, K = a_codes.shape
    N = w_codes.shape[0]
    K128 = -(-K // 128) * 128
    if not (0 < M <= ONE_LAUNCH_MAX_ROWS and N > 0 and K128 > 0 and gemm_splits(M, N, K128) == 1):
        return False
    if M <= _ACC_ROWS:
        return True
    rounds = -(-(-(-M // 128) * -(-N // 128)) // 256)
    n, k, values = N / 1e3, K128 / 1e3, M * N / 1e6
    if rounds == 1:
        if N % 4:
            return values * (5.4 - 0.85 * k) > 7.8 + 0.75 * n + 0.15 * k
        return values * (5.0 - 0.8 * k) > 9.3 + 0.9 * n + 0.25 * k
    if rounds == 2 and N % 4:
        return values * (4.1 + 0.55 * k) > 8.4 + 2.1 * n + 4.5 * k
    return rounds == 2 and K128 <= 256 and values > 5.6


def _project_fused_int8(a_codes, a_scales, w_codes, w_scales, spine_codes, spine_scale,
                        warp_scale16, warp_shift16, tanh_lut):
    """GEMM + spine + requantization in one call (group 128, 'int8'); None for K = 0,
    which the two-launch path covers (its GEMM returns zeros)."""
    dev, M, N, K, a, as_, w, ws = _prepare(a_codes, a_scales, w_codes, w_scales, 128)
    if K == 0:
        return None
    dev = _lib.require_gpu(spine_codes, spine_scale, warp_scale16, warp_shift16, tanh_lut)
    if spine_codes.numel() != 6 * N or spine_scale.numel() != N:
        raise ValueError(f"spine buffers do not match {N} charts")
    if warp_scale16.numel() != N or warp_shift16.numel() != N:
        raise ValueError(f"warp scalars do not match {N} charts")
    if tanh_lut.numel() != 256:
        raise ValueError("tanh_lut must have 256 entries")
    hq = torch.empty((M, N), dtype=torch.int8, device=dev)
    hs = torch.empty((M, -(-N // 128)), dtype=FP16, device=dev)
    if M == 0 or N == 0:
        return hq, hs
    table = torch.empty((N, 256), dtype=torch.float32, device=dev)
    sc, ps = spine_codes.reshape(N, 6).contiguous(), spine_scale.reshape(N).contiguous()
    wsc, wsh = warp_scale16.reshape(N).contiguous(), warp_shift16.reshape(N).contiguous()
    lut = tanh_lut.contiguous()
    _lib.call("ksd_ks3_project_fused", a.data_ptr(), as_.data_ptr(), w.data_ptr(), ws.data_ptr(),
              M, N, K, sc.data_ptr(), ps.data_ptr(), wsc.data_ptr(), wsh.data_ptr(),
              lut.data_ptr(), 128, hq.data_ptr(), hs.data_ptr(), table.data_ptr(),
              _lib.stream_ptr(dev))
    return hq, hs
