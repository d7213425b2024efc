"""Layer calibration on the HIP backend.

Same contract as actune/calibration.py:7-16 and :42-93:

* ``activation_reference(value, bits, group_size=64)`` returns the group-64
  dequantized activations codes * scale. The codes and scales come from the
  library's group-64 quantizer (the exact codebook of inference); the
  product codes * scale is the same fp32 multiply the reference performs.
* ``calibrate_linear(linear, inputs, row_weights=None, *, budget, group_size,
  clip_grid)`` fits the activation-guided channel scale (5 alphas), then the
  per-row clip ratio of every weight version over the clip grid, and the
  weighted error per (W, A) pair. Every candidate output is evaluated by the
  inference kernels themselves: x / scale quantized by the group-64
  quantizer and multiplied by the packed candidate weights in the packed
  GEMM, with fp32 output. The reference evaluates the same quantized
  operands with a float GEMM (F.linear of dequantized activations and
  weights); both are fp32 evaluations of the same exact sums, so scores
  differ only in the last bits and the selected scale and clips agree except
  on exact near-ties. All clip ratios of a pair are evaluated together: their
  packed weights stand one below the other, so one launch forms the codes, one
  GEMM the outputs and one kernel the losses.
* Weight codebooks are torch's on the layer's device, as the reference
  evaluates them (quantizers.py:23-94): on a GPU the divisions by the
  constants 7 and 127 are reciprocal multiplies there as well.

Calibration runs on the GPU only: CPU tensors raise ValueError (the
reference's own module remains the CPU path). jacobian_row_weights, the
RNG-driven Hutchinson estimate (calibration.py:19-39), stays with the
reference's offline tooling.
"""
from __future__ import annotations

import torch

from . import _native

_CLIP_GRID = (1., .975, .95, .925, .9, .875, .85, .8, .75)


def _require_gpu(t, what):
    if not t.is_cuda:
        raise ValueError(f"{what}: the HIP calibration path needs CUDA tensors")


def _unpack_codes(packed, bits, k):
    """u8 [M, K*bits/8] -> int8 codes [M, K] (code j of byte b at bits (j*bits))."""
    if bits == 8:
        return packed.view(torch.int8)
    per = 8 // bits
    fields = [(packed >> (j * bits)) & ((1 << bits) - 1) for j in range(per)]
    u = torch.stack(fields, dim=-1).reshape(packed.shape[0], k).to(torch.int16)
    half = 1 << (bits - 1)
    return ((u ^ half) - half).to(torch.int8)


def activation_reference(value, bits, group_size=64):
    """The exact symmetric group-64 codebook used by inference, dequantized
    (calibration.py:7-16)."""
    if bits not in (2, 4, 8) or value.shape[-1] % group_size:
        raise ValueError("Unsupported activation width or unaligned input")
    if group_size != 64:
        raise ValueError("the HIP backend quantizes groups of 64")
    _require_gpu(value, "activation_reference")
    shape = value.shape
    flat = value.reshape(-1, shape[-1]).contiguous()
    packed, scales = _native.quantize_groups(flat, bits)
    codes = _unpack_codes(packed, bits, shape[-1]).float()
    deq = codes.reshape(flat.shape[0], -1, 64) * scales[:, :, None]
    return deq.reshape(shape)


def _outputs(a_codes, weight, w, a, ratios):
    """fp32 outputs [M, R * N] of the packed GEMM for the codes of x against
    the weight candidates of every ratio, one below the other."""
    a_packed, a_scales = a_codes
    packed, scale = _native.weight_candidates(weight, ratios, w, a)
    return _native.grouped_linear(a_packed, a_scales, packed, scale, None, (a_packed.shape[0], weight.shape[1]), w, a,
                                  out_dtype=torch.float32)


# fp32 outputs and packed weights of the candidates evaluated at a time
_CANDIDATE_BYTES = 512 << 20


def _best_candidates(a_codes, weight, w, a, grid, reference):
    """(loss, ratio) per row of the first candidate of the lowest loss over
    the ratios of the f32 device tensor `grid`, and the last losses."""
    m, n = reference.shape
    best = torch.full((n,), float("inf"), device=reference.device)
    chosen, losses = torch.ones_like(best), None
    if w == 8 and a != 4:
        grid = grid[:1]  # plain W8 takes no clip: every candidate is the first
    step = max(1, _CANDIDATE_BYTES // (n * max(4 * m, weight.shape[1] * w // 8)))
    for i in range(0, len(grid), step):
        ratios = grid[i:i + step]
        losses = _native.candidate_select(_outputs(a_codes, weight, w, a, ratios), reference, ratios, best, chosen)
    return best, chosen, losses


@torch.no_grad()
def calibrate_linear(linear, inputs, row_weights=None, *, budget="w4a4", group_size=64, clip_grid=_CLIP_GRID):
    """Fit activation-guided scales, row clips and weighted errors per pair
    (calibration.py:42-93), with every candidate evaluated by the inference
    quantizer and packed GEMM."""
    if budget not in ("w4a4", "w4a8"):
        raise ValueError("Unknown precision budget")
    x = inputs.detach().reshape(-1, linear.in_features).to(linear.weight.device, linear.weight.dtype)
    if not len(x) or not torch.isfinite(x).all() or linear.in_features % group_size:
        raise ValueError("Nonempty finite aligned fitting inputs required")
    if group_size != 64:
        raise ValueError("the HIP backend quantizes groups of 64")
    _require_gpu(x, "calibrate_linear")
    gains = torch.ones(linear.out_features, device=x.device) if row_weights is None \
        else row_weights.to(x.device).float()
    if gains.shape != (linear.out_features,) or not torch.isfinite(gains).all() or (gains < 0).any():
        raise ValueError("Invalid action-Jacobian weights")
    if not bool(gains.sum()):
        gains = torch.ones_like(gains)
    reference = torch.nn.functional.linear(x.float(), linear.weight.float())
    base_a = 4 if budget == "w4a4" else 8
    moment = x.float().abs().mean(0).clamp_min(1e-4)
    x, unclipped = x.contiguous(), torch.ones(1, device=x.device)
    candidates, scores = [], []
    for alpha in (0., .25, .5, .75, 1.):
        scale = moment.pow(alpha)
        scale = (scale / (scale.max() * scale.min()).sqrt()).clamp(1 / 16, 16).to(x.dtype)
        weight = (linear.weight * scale[None, :]).to(x.dtype).contiguous()
        _, _, losses = _best_candidates(_native.quantize_groups(x, base_a, scale), weight, 4, base_a, unclipped,
                                        reference)
        candidates.append((scale, weight))
        scores.append((losses[0] * gains).sum())
    scores = torch.stack(scores).tolist()
    chosen = 0
    for i, score in enumerate(scores):
        if score < scores[chosen]:
            chosen = i
    scale, weight = candidates[chosen]
    widths = (8,) if budget == "w4a8" else (2, 4, 8)
    a_codes = {a: _native.quantize_groups(x, a, scale) for a in widths}
    grid = tuple(clip_grid)
    if not all(0 < ratio <= 1 for ratio in grid):
        raise ValueError("Clip ratios must lie in (0, 1]")
    grid = torch.tensor([float(ratio) for ratio in grid], dtype=torch.float32, device=x.device)
    totals, clips = {}, {}
    for w in (2, 4, 8):
        for a in widths:
            mode = f"w{w}a{a}"
            row_error, clips[mode], _ = _best_candidates(a_codes[a], weight, w, a, grid, reference)
            totals[mode] = (row_error * gains).sum()
    errors = dict(zip(totals, torch.stack(list(totals.values())).tolist()))
    return dict(channel_scale=scale, clips=clips, errors=errors, group_size=group_size)
