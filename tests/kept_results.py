"""What a plain decoder gave, kept for the calls that follow with the same model and requests: a test in the other dtype, the same
sequence with and without a change.  Everything that the decoder reads is part of the key, so no result depends on it."""
import functools
import hashlib
import json
from collections import OrderedDict

import torch

KEPT = 48


def kept(reference):
    """`reference(cfg, tensors, requests, rnd=None)`, which gives {request: logits}, with its latest results."""
    results = OrderedDict()

    @functools.wraps(reference)
    def of(cfg, tensors, requests, rnd=None):
        read = hashlib.blake2b(json.dumps([cfg, list(requests.items())], sort_keys=True).encode())
        for name in sorted(tensors):
            t = tensors[name].detach().cpu().contiguous()
            read.update(f"{name} {t.dtype} {tuple(t.shape)}".encode())
            read.update(t.reshape(-1).view(torch.uint8).numpy())
        key = (read.digest(), rnd)
        if key not in results:
            results[key] = reference(cfg, tensors, requests, rnd)
            while len(results) > KEPT:
                results.popitem(last=False)
        results.move_to_end(key)
        return {request: logits.clone() for request, logits in results[key].items()}

    return of
