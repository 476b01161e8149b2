"""Anneal-window helpers (reference: src/pytorch_modules/utils.py)."""
import math

import torch

from . import _native


def cosine_easing_window(num_freqs, alpha):
    """Eases the levels in one by one with a cosine as ``alpha`` goes from 0 to ``num_freqs``.

    ``win[k] = 0.5 * (1 + cos(pi * clip(alpha - k, 0, 1) + pi))``: exactly 1 for fully eased-in
    levels, exactly 0 for levels not yet started (reference: utils.py:5-16).
    """
    # The same natively, for a plain step number and where nothing observes the tensor operations (None); the bools, arrays
    # and symbols that are numbers too take the operations' own rules, and a compiler sees only these.
    if type(num_freqs) is int and type(alpha) in (int, float) and not torch.compiler.is_dynamo_compiling():
        native = _native._bridge or _native.bridge_if_built()
        window = native.cosine_window(num_freqs, alpha) if native is not None else None
        if window is not None:
            return window
    x = torch.clip(alpha - torch.arange(num_freqs, dtype=torch.float32), 0.0, 1.0)
    return 0.5 * (1 + torch.cos(math.pi * x + math.pi))


def map_range_val(input_val, input_start, input_end, output_start, output_end):
    """Clamps ``input_val`` to [input_start, input_end] and maps it linearly (reference: utils.py:19-23)."""
    input_clamped = max(input_start, min(input_end, input_val))
    return output_start + ((output_end - output_start) / (input_end - input_start)) * (input_clamped - input_start)
