"""Host-side token selection of globals.js:47-74."""
import math
import random

import numpy as np


def selectTopK(probs, top_k):
    """Stable descending sort by value, first top_k (globals.js:66-74): ties keep the
    lower index first. Of a long array only what can be among the first top_k is sorted: the values not below
    the top_k-th largest of the maxima of runs of 64 (50257 values, top_k = 40: 8 ms for all of them in a list, 0.1 ms so)."""
    if isinstance(probs, np.ndarray) and probs.ndim == 1 and probs.dtype in (np.float16, np.float32, np.float64):
        a = probs
    else:  # any sequence of what float() takes
        a = np.array([float(probs[i]) for i in range(len(probs))], np.float64)
    runs = a.size // 64
    order = None
    if top_k is not None and 0 < top_k < runs:
        tops = a[:64 * runs].reshape(runs, 64).max(axis=1)
        order = np.flatnonzero(a >= np.partition(tops, runs - top_k)[runs - top_k])
        if order.size < top_k:  # NaN among them
            order = None
    if order is None:
        order = np.arange(a.size)
    order = order[np.argsort(-a[order], kind="stable")][:top_k]
    return {"topKIndices": [int(i) for i in order], "topKProbs": [float(v) for v in a[order]]}


def cpuSoftmax(logits, temperature=1.0):
    """float64 softmax with the temperature inside the exponent (globals.js:59-64)."""
    m = max(logits)
    e = [math.exp((x - m) / temperature) for x in logits]
    s = 0.0
    for v in e:
        s += v
    return [v / s for v in e]


def sampleFromDistribution(probs, rand=None):
    """Inverse-CDF sampling (globals.js:47-57)."""
    r = random.random() if rand is None else rand
    c = 0.0
    for i, p in enumerate(probs):
        c += p
        if r < c:
            return i
    return len(probs) - 1
