"""WKV7Runner: the runner's prefill / decode control flow at the WKV-op level.

Mirrors RWKV7Runner (wkvm/runner/runner.py:23-89) with the model forward
reduced to its WKV7 op: callers hand in the per-layer projected vectors
(r, w, k, v, a, b) that the RWKV-7 time-mix produces, instead of token ids.
The control flow is the reference's:

* ``prefill`` walks the prompt in ``prefill_chunk`` slices and, inside each
  slice, every layer; the state round-trips through the slot between slices
  exactly as a preempted request's would (runner.py:12-14, 52-62);
* ``decode_step`` advances a batch of slots by one token through every layer
  (runner.py:65-89);
* ``mixed_step`` is one scheduler step with decode rows and ragged prefill
  rows together, one decode launch plus one varlen prefill launch per layer
  (the split Engine._execute makes, wkvm/engine.py:142-160, laid out with
  MixedBatchMetadata-style offsets, wkvm/core/mixed_batch.py:213-270).

Errors mirror the reference: ``ValueError`` for ``prefill_chunk < 1``, an
empty prompt and a batch / input length mismatch.
"""

from __future__ import annotations

from typing import Sequence

import torch

from . import ops
from .state import RWKV7StateBank

LayerInputs = Sequence[torch.Tensor]  # (r, w, k, v, a, b)


class WKV7Runner:
    """The WKV7 work of whole requests over a bank, every layer at once: each
    call takes all layers' vectors and launches one kernel over them. (A model
    whose next layer needs this one's output has one layer's vectors at a time;
    it calls the bank's ``decode_wkv`` / ``prefill_wkv`` per layer, or keeps
    whole time-mix blocks in a ``TimeMixDecodeGraph``.)"""

    # Chunks at least this long run segmented when ``prefill_segments`` is a
    # count (one layer's segments are faster from about 2k tokens on).
    SEGMENT_MIN_TOKENS = 2048

    def __init__(self, bank: RWKV7StateBank, prefill_chunk: int = 512,
                 prefill_segments: int | str | None = None) -> None:
        """``prefill_segments``: cut each prefill chunk of at least
        ``SEGMENT_MIN_TOKENS`` tokens into that many segments that run side by
        side (``ops.wkv7_prefill_segments``), a layer at a time; ``"auto"``
        picks the count from the compute units one layer's chunk leaves idle
        (``ops.auto_segments``), for banks of so few layers that it pays;
        ``None`` runs every chunk in one pass. Results agree to the
        scan's rounding (``ops.wkv7_prefill_segments``)."""
        if prefill_chunk < 1:
            raise ValueError("prefill_chunk must be >= 1")
        if prefill_segments is not None and prefill_segments != "auto" and (
                not isinstance(prefill_segments, int) or prefill_segments < 1):
            raise ValueError("prefill_segments must be >= 1, 'auto' or None")
        self.bank = bank
        self.prefill_chunk = prefill_chunk
        self.prefill_segments = prefill_segments
        self.device = bank.device

    def _check_layers(self, layer_inputs: Sequence[LayerInputs]) -> None:
        if len(layer_inputs) != self.bank.layout.n_layer:
            raise ValueError(f"expected inputs for {self.bank.layout.n_layer} layers, "
                             f"got {len(layer_inputs)}")

    @torch.inference_mode()
    def prefill(self, layer_inputs: Sequence[LayerInputs], slots: dict[str, int],
                out_dtype: torch.dtype = torch.bfloat16) -> list[torch.Tensor]:
        """Run a prompt's ``[T, H, 64]`` vectors through every layer in chunks,
        leaving the final state in ``slots``; returns per-layer ``y [T, H, 64]``."""
        self._check_layers(layer_inputs)
        T = int(layer_inputs[0][0].shape[0])
        if T == 0:
            raise ValueError("empty prompt")
        H = self.bank.layout.num_heads
        ys = [torch.empty((T, H, 64), dtype=out_dtype, device=self.device)
              for _ in layer_inputs]
        ids = ops.device_ids([slots["wkv"]], self.bank.num_slots + 1, self.device, "slots",
                             wait=False)
        # device plans (offsets 0, n and the one-sequence order), uploaded once
        # per chunk length rather than once per layer
        plans: dict[int, torch.Tensor] = {}
        # the first layer's r says how many tokens there are, longer vectors are
        # read up to there
        layer_inputs = [xs if all(x.shape[0] == T for x in xs) else [x[:T] for x in xs]
                        for xs in layer_inputs]
        ptrs = None
        for start in range(0, T, self.prefill_chunk):
            n = min(self.prefill_chunk, T - start)
            if n not in plans:
                plans[n] = ops.upload_ints([0, n, 0], self.device, wait=False)
            plan = plans[n]
            G = self._segments(n, H)
            if G > 1:
                for layer, xs in enumerate(layer_inputs):
                    ops.wkv7_prefill_segments(self.bank.wkv[layer], [slots["wkv"]], [0, n],
                                              *[x[start:start + n] for x in xs], segments=G,
                                              out=ys[layer][start:start + n])
            else:
                if ptrs is None:
                    ptrs, keep = ops.layer_vectors(layer_inputs, (T, H, 64),
                                                   self.bank.wkv.device, "prefill")
                ops.wkv7_prefill_layers(self.bank.wkv, ids, plan[:2], ptrs, ys, start, n,
                                        seq_order=plan[2:])
        return ys

    def _segments(self, n: int, H: int) -> int:
        if self.prefill_segments is None or n < self.SEGMENT_MIN_TOKENS:
            return 1
        if self.prefill_segments == "auto":
            G = ops.auto_segments(H, [n], self.device)
            L = self.bank.layout.n_layer
            # One launch runs all layers side by side, the segmented form one
            # after the other, each with about twice the arithmetic and 70 us of
            # launches and upload. us, segmented against one launch: 16,384 tokens
            # x 12 heads in 8 segments, 3 layers 462 / 542, 12 layers 1839 / 743;
            # x 32 heads in 4, 2 layers 598 / 724, 3 layers 832 / 684; 4,096 tokens
            # x 32 heads in 4, 1 layer 106 / 150, 2 layers 195 / 198.
            return G if L == 1 or (2 * L <= G and n >= 512 * L * G) else 1
        return self.prefill_segments

    @torch.inference_mode()
    def decode_step(self, slot_batch: list[dict[str, int]],
                    layer_inputs: Sequence[LayerInputs],
                    out_dtype: torch.dtype = torch.bfloat16) -> list[torch.Tensor]:
        """Advance every slot in ``slot_batch`` by one token through every
        layer; ``layer_inputs[l]`` holds ``[B, H, 64]`` vectors. Returns
        per-layer ``y [B, H, 64]``."""
        self._check_layers(layer_inputs)
        if any(int(x.shape[0]) != len(slot_batch) for xs in layer_inputs for x in xs):
            raise ValueError("slot_batch and last_tokens length mismatch")
        return ops.wkv7_decode_layers(self.bank.wkv, ops.ids_list(slot_batch, "wkv"),
                                      layer_inputs, out_dtype=out_dtype)

    @torch.inference_mode()
    def mixed_step(self, decode_batch: list[dict[str, int]],
                   decode_inputs: Sequence[LayerInputs],
                   prefill_batch: list[dict[str, int]], prefill_lens: Sequence[int],
                   prefill_inputs: Sequence[LayerInputs], *, zero_init: bool = False,
                   out_dtype: torch.dtype = torch.bfloat16, concurrent: bool = True):
        """One scheduler step over decode rows (one token each) and ragged
        prefill rows (``prefill_lens`` tokens each, packed along dim 0).
        Returns ``(decode_ys, prefill_ys)`` per layer.

        One prefill launch and one decode launch over all layers, both on the
        caller's stream: with one launch per kind there is one ragged tail to
        fill instead of one per layer, and decode workgroups on a second stream
        take units from the prefill's next workgroups (two layers of 64 prompts
        and 448 decode rows, 1.5B shape: 1175 us on one stream, 1220 us on two).
        ``concurrent``, which asked for that second stream, is still accepted
        and has no effect."""
        self._check_layers(decode_inputs)
        self._check_layers(prefill_inputs)
        if len(prefill_lens) != len(prefill_batch):
            raise ValueError("prefill_batch and prefill_lens length mismatch")
        if any(int(n) < 1 for n in prefill_lens):
            raise ValueError("prefill rows need at least one token")
        cu = [0]
        for n in prefill_lens:
            cu.append(cu[-1] + int(n))
        if prefill_batch and any(int(x.shape[0]) != cu[-1] for xs in prefill_inputs for x in xs):
            raise ValueError("prefill inputs do not hold sum(prefill_lens) tokens")
        rows = self.bank.num_slots + 1
        dec_ids, dec_order = ops.decode_plan(ops.ids_list(decode_batch, "wkv"), rows, self.device,
                                             wait=False)
        pre_ids = ops.device_ids(ops.ids_list(prefill_batch, "wkv"), rows, self.device, "prefill",
                                 wait=False)
        if set(ops.ids_list(decode_batch, "wkv")) & set(ops.ids_list(prefill_batch, "wkv")):
            raise ValueError("a slot cannot decode and prefill in the same step")
        # offsets and the longest-first start order in one upload
        nseq = len(prefill_batch)
        plan = ops.upload_ints(cu + ops.longest_first(cu), self.device, wait=False)
        cu_t, pre_order = plan[:nseq + 1], plan[nseq + 1:]
        L, H = self.bank.layout.n_layer, self.bank.layout.num_heads
        dec_ys, pre_ys = [None] * L, [None] * L
        if prefill_batch:
            ptrs, keep = ops.layer_vectors(prefill_inputs, (cu[-1], H, 64), self.bank.wkv.device,
                                           "prefill")
            pre_ys = [torch.empty((cu[-1], H, 64), dtype=out_dtype, device=self.device)
                      for _ in range(L)]
            ops.wkv7_prefill_layers(self.bank.wkv, pre_ids, cu_t, ptrs, pre_ys, 0, cu[-1],
                                    zero_init=zero_init, seq_order=pre_order)
        if decode_batch:
            dec_ys = ops.wkv7_decode_layers(self.bank.wkv, dec_ids, decode_inputs,
                                            out_dtype=out_dtype, row_order=dec_order)
        return dec_ys, pre_ys
