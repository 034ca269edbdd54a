"""The sampler step behind lm_head: host mirror of `sampleGreedy` (rtp_llm/models_py/bindings/core/CudaSampleOp.cc:619-800) over the
MI355 kernels -- same parameter record (bindings/core/OpData.h:260-286, the fields this path reads), same order of operations
and the same host-side shortcuts:

  1. temperature, only when some row has T != 1                          (:633-645)
  2. repetition / presence / frequency penalties, only when some row is off-default   (:648-685)
  2b. no_repeat_ngram_size, only when some decoder row has one                          (:242-283)
  3. every top_k == 1 and no probabilities wanted: arg-max of the logits (:688-700)
  4. softmax in place, top_p == 0 reads as 1                             (:703-736)
  5. every top_k == 1: arg-max of the probabilities; otherwise top-k / top-p filter, renormalise, draw   (:739-786)
  6. the drawn ids go into the last column of token_ids                 (:797-799)

Randomness is explicit: where the reference consumes `generator` inside torch.multinomial, the caller passes one uniform in
[0, 1) per row (`uniform`), so a run is reproducible and checkable against the oracle.  `cum_log_probs` / `output_log_probs`
are not on this path (the reference's ROCm branch does not update them per token either)."""
from dataclasses import dataclass
from typing import Optional

import numpy as np
import torch

from . import ops


@dataclass
class GreedyParams:
    logits: torch.Tensor              # [batch_size, vocab_size] fp32, GPU, modified in place (penalties, then probabilities)
    input_lengths: torch.Tensor       # [batch_size] int32
    sequence_lengths: torch.Tensor    # [decoder_batch_size] int32
    token_ids: torch.Tensor           # [batch_size, step + 1] int32; column `step` receives the new token
    step: int
    top_k: torch.Tensor               # [batch_size] int32
    top_p: torch.Tensor               # [batch_size] fp32
    temperature: torch.Tensor         # [batch_size] fp32
    repetition_penalty: Optional[torch.Tensor] = None
    presence_penalty: Optional[torch.Tensor] = None
    frequency_penalty: Optional[torch.Tensor] = None
    no_repeat_ngram_size: Optional[torch.Tensor] = None   # [decoder_batch_size] int32, 0 = off
    output_all_probs: Optional[torch.Tensor] = None     # [batch_size, vocab_size] fp32 GPU: receives the probabilities
    return_original_all_probs: bool = False
    uniform: Optional[torch.Tensor] = None              # [batch_size] fp32 in [0, 1): the draw (see the module docstring)


def _host(t: torch.Tensor, dtype) -> torch.Tensor:
    return t.detach().to(device="cpu", dtype=dtype)


def _off(t: torch.Tensor, default) -> bool:
    return bool((t.numpy() != default).any())


def _softmax_in_place(logits: torch.Tensor) -> torch.Tensor:
    # the kernel may overwrite its input; host tensors reach this flow only with another `ops`, which need not
    return ops.softmax_rows(logits, out=logits) if logits.is_cuda else logits.copy_(ops.softmax_rows(logits))


def _upload(tensors, device):
    """The named host tensors of 32-bit values on the device, contiguous: packed into one buffer and sent in one copy."""
    if not tensors:
        return {}
    host = np.concatenate([t.numpy().reshape(-1).view(np.int32) for t in tensors.values()])
    flat = torch.from_numpy(host).to(device)
    out, at = {}, 0
    for name, t in tensors.items():
        n = t.numel()
        out[name] = flat[at:at + n].view(t.dtype).view(t.shape)
        at += n
    return out


def sample_greedy(params: GreedyParams) -> torch.Tensor:
    """-> the new token ids [batch_size] int32 on the GPU (also written to params.token_ids[:, step])."""
    logits = params.logits
    B, V = logits.shape
    dev = logits.device
    step = int(params.step)
    if params.token_ids.shape != (B, step + 1):
        raise ValueError("sample_greedy: token_ids must be [batch_size, step + 1]")
    # vectors and history on the host, nothing between the penalties and the draw: the whole step in one native call, where some row has a filter.  Where none has, what was seen serves below,
    # and the step costs what it did without the question
    penalties = (params.repetition_penalty, params.presence_penalty, params.frequency_penalty)
    seen = None
    if logits.is_cuda and params.uniform is not None and params.output_all_probs is None and (params.no_repeat_ngram_size is None or params.sequence_lengths.numel() == 0) and \
            (penalties[0] is None or (penalties[1] is not None and penalties[2] is not None)):
        seen = ops.sampler_filters(params.top_k, params.top_p, V)
        host = None
        if seen is None or (seen[1] and not seen[0]):
            host = ops.sampler_vectors(logits, params.token_ids, params.temperature, None if penalties[0] is None else penalties, params.top_k, params.top_p, params.uniform,
                                       params.input_lengths, params.sequence_lengths, seen)
        if host is not None:
            return ops.sampling_draw(logits, None, None, params.uniform, host=host)
    temperature = _host(params.temperature, torch.float32)
    scale = _off(temperature, 1.0)
    penalise = False
    if params.repetition_penalty is not None:
        if params.presence_penalty is None or params.frequency_penalty is None:
            raise ValueError("sample_greedy: repetition_penalty comes with presence_penalty and frequency_penalty")
        rep, pres, freq = (_host(t, torch.float32) for t in (params.repetition_penalty, params.presence_penalty, params.frequency_penalty))
        penalise = _off(rep, 1.0) or _off(pres, 0.0) or _off(freq, 0.0)
    top_k = _host(params.top_k, torch.int32)
    all_greedy = not _off(top_k, 1) if seen is None else seen[0]
    draw = not all_greedy
    if draw and params.uniform is None:
        raise ValueError("sample_greedy: sampling rows need params.uniform (one value in [0, 1) per row)")
    ngram = None
    if params.no_repeat_ngram_size is not None and params.sequence_lengths.numel() > 0:
        ngram = _host(params.no_repeat_ngram_size, torch.int32)
        if not _off(ngram[:params.sequence_lengths.numel()], 0):
            ngram = None
    # logits -> probabilities in two launches, unless something else comes between
    together = logits.is_cuda and ngram is None and step < 2048 and B <= 65535 and not (all_greedy and params.output_all_probs is None)

    # everything the step needs on the device that is on the host: one buffer, one copy
    up = {}
    if scale:
        up["temperature"] = temperature
    if penalise:
        lengths = _host(params.input_lengths, torch.int32).clone()
        nd = params.sequence_lengths.numel()
        if nd > 0:
            lengths[:nd] = _host(params.sequence_lengths, torch.int32)
        up.update(rep=rep, pres=pres, freq=freq, lengths=lengths)
        if params.token_ids.device.type == "cpu":
            history = params.token_ids.to(torch.int32)                                    # [batch_size, step + 1]
            up["history"] = history if together else history.t()
    if draw:
        top_p = _host(params.top_p, torch.float32).clone()
        p = top_p.numpy()
        p[np.abs(p) < 1e-7] = 1.0
        if seen is not None:
            filtered = seen[1]
        else:
            filtered = bool((p != 1.0).any()) or (_off(top_k, 0) and bool(((top_k.numpy() > 0) & (top_k.numpy() < V)).any()))
        up.update(top_k=top_k, top_p=top_p)
        if params.uniform.device.type == "cpu":
            up["uniform"] = params.uniform.to(torch.float32)
    up = _upload(up, dev)

    if together:
        vectors = {}
        if penalise:
            vectors = dict(repetition_penalty=up["rep"], presence_penalty=up["pres"], frequency_penalty=up["freq"], input_lengths=up["lengths"], max_input_length=step + 1,
                           step=step + 1, token_ids=up["history"] if "history" in up else params.token_ids.to(device=dev, dtype=torch.int32).contiguous())
        # and the draw behind them, where a row has a filter: with none the histograms that name its threshold are for nothing (64 rows of 152064 56 us in two calls, 65 in one; with
        # top-p 0.8 to 0.95 125 and 52)
        if not all_greedy and filtered and params.output_all_probs is None:
            u = up["uniform"] if "uniform" in up else params.uniform.to(device=dev, dtype=torch.float32).contiguous()
            ids = ops.sampling_draw(logits, up["top_k"], up["top_p"], u, up.get("temperature"), **vectors)
            params.token_ids[:, step] = ids.to(params.token_ids.device)
            return ids
        probs = ops.sampling_probs(logits, up.get("temperature"), **vectors)
    else:
        if scale:
            ops.apply_penalties(logits, temperature=up["temperature"])
        if penalise:
            transposed = up["history"] if "history" in up else params.token_ids.to(device=dev, dtype=torch.int32).t().contiguous()
            ops.apply_penalties(logits, repetition_penalty=up["rep"], presence_penalty=up["pres"], frequency_penalty=up["freq"], output_ids=transposed,
                                input_lengths=up["lengths"], max_input_length=step + 1, step=step + 1)
        if ngram is not None:
            # the kernel takes the index of the last valid token and adds one itself (CudaSampleOp.cc:262-265)
            nd = params.sequence_lengths.numel()
            tokens = params.token_ids.to(device=dev, dtype=torch.int32).contiguous()
            ops.ban_repeat_ngram(logits, tokens[:nd], _host(params.sequence_lengths, torch.int32) - 1, ngram[:nd])

    if all_greedy and params.output_all_probs is None:
        ids = ops.argmax(logits)
    else:
        if not together:
            probs = _softmax_in_place(logits)
        want_renorm = params.output_all_probs is not None and not params.return_original_all_probs
        if all_greedy:
            ids = ops.argmax(probs)
            if want_renorm:   # top_k_renorm_probs with k = 1: the mass of the maximum (ties share it)
                _, renorm = ops.top_k_top_p_sample(probs, top_k, None, torch.zeros(B, device=dev), return_probs=True)
                params.output_all_probs.copy_(renorm)
        else:
            u = up["uniform"] if "uniform" in up else params.uniform.to(device=dev, dtype=torch.float32).contiguous()
            if want_renorm:
                ids, renorm = ops.top_k_top_p_sample(probs, up["top_k"], up["top_p"], u, return_probs=True)
                params.output_all_probs.copy_(renorm)
            else:
                ids = ops.top_k_top_p_sample(probs, up["top_k"], up["top_p"], u)
        if params.return_original_all_probs and params.output_all_probs is not None:
            params.output_all_probs.copy_(probs)
    params.token_ids[:, step] = ids.to(params.token_ids.device)
    return ids
