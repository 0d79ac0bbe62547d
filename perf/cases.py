"""The work a program has this framework do, as cases that can be measured.

Every case goes through the public entry points of tao_attention:

* request: a new state, its prompt (in one call or in chunks) and the first
  generated tokens, as a server runs one request through one layer;
* decode: one route period (24 tokens) of generation from a long prompt;
* batch: the same for many requests of one layer, one batched call per token;
* full: tao_attention without gradients (scoring, evaluation);
* train: tao_attention forward and backward, every gradient.

Operands are N(0, 1), as the tests and bench.py have them: raw_q / raw_k are
projections before the caller's transform, and a normalised hidden state
projected at unit gain has about that distribution. Fusion parameters are fp32
at 0.02, a trained layer's scale; alpha is 0.5.
"""
import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "tao-memory_amd"))

ALPHA = 0.5
BLOCK, KEEP, GROUP, PERIOD = 256, 512, 8, 24
FIRST = BLOCK + KEEP                       # first position with a sealed fine
PIECE = 16384                              # tokens of one prompt call and one random draw


def _case(kind, heads, width, tokens, **more):
    case = dict(kind=kind, heads=heads, width=width, tokens=tokens, batch=1, steps=0, chunk=0,
                values=False, writer="softmax", graph=False, dtype="bf16")
    case.update(more)
    return case


def listed():
    return [
        # A chat turn on a small layer, default configuration: everything is
        # launch and host latency.
        dict(_case("request", 12, 64, 200, steps=16, values=True), name="request-200"),
        # An ordinary prompt past the first page, with a ragged end.
        dict(_case("request", 12, 64, 2700, steps=2, values=True), name="request-2700"),
        # Chunked prefill, as a server interleaves a prompt with other work.
        dict(_case("request", 8, 128, 7000, steps=2, chunk=1999, values=True),
             name="request-chunked"),
        # A long prompt at the headline width.
        dict(_case("request", 32, 128, 16384, steps=2), name="request-16k"),
        # The regularized association writer in the stream.
        dict(_case("request", 8, 128, 5000, steps=2, writer="regularized_association"),
             name="request-regularized"),
        # Generation at the headline context and width.
        dict(_case("decode", 32, 128, 131072, steps=PERIOD), name="decode-128k"),
        # Generation in one layer of the published 12-layer model's shape,
        # graph preset.
        dict(_case("decode", 6, 128, 32768, steps=PERIOD, graph=True), name="decode-32k-graph"),
        # A server's batch of ragged requests.
        dict(_case("batch", 32, 128, 32768, batch=32, steps=PERIOD), name="batch-32"),
        # A long document scored in one call.
        dict(_case("full", 8, 128, 16384, values=True), name="full-16k"),
        # fp32 operands, the reference's CPU-eager shape.
        dict(_case("full", 4, 64, 2048, dtype="fp32", values=True), name="full-2k-fp32"),
        # A training step of the published shape.
        dict(_case("train", 12, 64, 8192, batch=2, values=True), name="train-8k"),
        # A training step of a feature-mass layer at an odd length.
        dict(_case("train", 8, 64, 3001, writer="feature_mass_association", values=True),
             name="train-mass"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random):
    kind = rng.choice(["request", "request", "decode", "batch", "full", "train"])
    width = rng.choice([64, 128])
    values = rng.random() < 0.5
    if kind == "request":
        heads, tokens = _log(rng, 1, 32), _log(rng, 16, 16384)
        chunk = 0 if rng.random() < 0.6 else max(64, _log(rng, tokens / 8, tokens))
        writer = "softmax" if rng.random() < 0.8 else "regularized_association"
        return _case(kind, heads, width, tokens, steps=rng.randint(1, 16), chunk=chunk,
                     values=values, writer=writer)
    if kind == "decode":
        return _case(kind, _log(rng, 1, 32), width, _log(rng, 100, 131072), steps=PERIOD,
                     values=values, graph=not values and rng.random() < 0.5)
    if kind == "batch":
        return _case(kind, _log(rng, 1, 32), width, _log(rng, 1000, 32768),
                     batch=rng.randint(2, 32), steps=PERIOD, values=values)
    heads, batch = _log(rng, 1, 16), rng.randint(1, 2)
    if kind == "full":
        if rng.random() < 0.25:
            return _case(kind, min(heads, 8), width, _log(rng, 200, 4096), dtype="fp32",
                         values=values)
        tokens = min(_log(rng, 200, 16384), 16777216 // (heads * width * batch))
        return _case(kind, heads, width, tokens, batch=batch, values=values)
    tokens = min(_log(rng, 300, 8192), 12582912 // (heads * width * batch))
    writer = rng.choice(["softmax"] * 5 + ["regularized_association", "feature_mass_association",
                                           "structured_gram_association"])
    return _case(kind, heads, width, tokens, batch=batch, values=values, writer=writer)


# ---- inputs -----------------------------------------------------------------

def _config(case):
    from tao_attention import TaoConfig
    from tao_attention.presets import index_only_page_memo
    if case["kind"] in ("decode", "batch") and not case["values"]:
        return index_only_page_memo(graph=case["graph"])
    return TaoConfig(coarse_index_only=not case["values"], fine_writer=case["writer"],
                     q1_page_normalization_memo=not case["values"] and case["writer"] == "softmax")


def _tokens(case, batch, count, g):
    """(q, k, v, raw_q, raw_k), each [batch, count, heads, width]."""
    dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
    return [torch.randn((batch, count, case["heads"], case["width"]), generator=g,
                        device="cuda").to(dtype) for _ in range(5)]


def _fusion(case, g):
    return [torch.randn((case["heads"], case["width"], 3), generator=g, device="cuda") * 0.02
            for _ in range(2)]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _lengths(case, seed):
    """Prompt lengths of a batch's requests: half to all of case["tokens"]."""
    rng = random.Random(seed)
    return [rng.randint(case["tokens"] // 2, case["tokens"]) for _ in range(case["batch"])]


def _pieces(case, length, g):
    for at in range(0, length, PIECE):
        yield _tokens(case, 1, min(PIECE, length - at), g)


def _named(xs, fusion):
    q, k, v, raw_q, raw_k = xs
    return (q, k, v), dict(raw_q=raw_q, raw_k=raw_k, fusion_a=fusion[0], fusion_b=fusion[1],
                           alpha=ALPHA)


def _each(xs, start, count):
    """One-token operands of `count` steps from token `start`."""
    return [[x[:, i:i + 1].contiguous() for x in xs] for i in range(start, start + count)]


def prepare(case, seed):
    from tao_attention import new_state, tao_attention_prefill
    g = _generator(seed)
    state = dict(case=case, config=_config(case), fusion=_fusion(case, g))
    kind = case["kind"]
    if kind == "request":
        xs = _tokens(case, 1, case["tokens"] + case["steps"], g)
        width = case["chunk"] or case["tokens"]
        cuts = range(0, case["tokens"], width)
        state["chunks"] = [[x[:, c:min(c + width, case["tokens"])].contiguous() for x in xs]
                           for c in cuts]
        state["decode"] = _each(xs, case["tokens"], case["steps"])
    elif kind in ("decode", "batch"):
        # The prompts are part of what the program already has: their states.
        lengths = [case["tokens"]] if kind == "decode" else _lengths(case, seed)
        state["states"] = []
        for length in lengths:
            s = new_state(0, state["config"])
            for xs in _pieces(case, length, g):
                ops, named = _named(xs, state["fusion"])
                _, s = tao_attention_prefill(*ops, **named, state=s, position=s.get_pos())
            state["states"].append(s)
        xs = _tokens(case, len(lengths), case["steps"], g)
        state["decode"] = _each(xs, 0, case["steps"])
    else:
        state["xs"] = _tokens(case, case["batch"], case["tokens"], g)
        if kind == "train":
            state["leaves"] = [x.requires_grad_(True) for x in state["xs"] + state["fusion"]]
            state["grad"] = torch.randn(state["xs"][0].shape, generator=g,
                                        device="cuda").to(state["xs"][0].dtype)
    return state


# ---- one pass ---------------------------------------------------------------

def _decode(steps, fusion, s, copy):
    from tao_attention import tao_attention_decode
    outs = []
    for xs in steps:
        ops, named = _named(xs, fusion)
        out, s = tao_attention_decode(*ops, **named, state=s, position=s.get_pos())
        # The graph preset's next step overwrites its output buffer.
        outs.append(out.clone() if copy else out)
    return outs


def run(state):
    from tao_attention import (new_state, tao_attention, tao_attention_decode_batch,
                               tao_attention_prefill)
    case, fusion, kind = state["case"], state["fusion"], state["case"]["kind"]
    if kind == "request":
        s, outs = new_state(0, state["config"]), []
        for xs in state["chunks"]:
            ops, named = _named(xs, fusion)
            out, s = tao_attention_prefill(*ops, **named, state=s, position=s.get_pos())
            outs.append(out)
        return outs + _decode(state["decode"], fusion, s, False)
    if kind == "decode":
        return _decode(state["decode"], fusion, state["states"][0], case["graph"])
    if kind == "batch":
        outs = []
        for xs in state["decode"]:
            ops, named = _named(xs, fusion)
            out, _ = tao_attention_decode_batch(*ops, **named, states=state["states"])
            outs.append(out)
        return outs
    ops, named = _named(state["xs"], fusion)
    if kind == "full":
        with torch.no_grad():
            return tao_attention(*ops, **named, config=state["config"])
    out = tao_attention(*ops, **named, config=state["config"])
    return [out, *torch.autograd.grad(out, state["leaves"], state["grad"])]


# ---- what a pass cannot do without ------------------------------------------

def _fines(position):
    return 0 if position < FIRST else (position - FIRST) // BLOCK + 1


def _budget(n):
    return min(n, math.isqrt(2 * n - 1) + 1 + 2) if n > 0 else 0


def _routed(fines):
    """(pages chosen, fines read) of `fines` sealed ones."""
    done, pending = divmod(fines, GROUP)
    pages = min(done, -(-2 * _budget(GROUP * done) // GROUP))
    return pages, min(GROUP * pages + pending, _budget(fines))


def work(case):
    kind, d, heads = case["kind"], case["width"], case["heads"]
    size = 4 if case["dtype"] == "fp32" else 2
    row = heads * d * size
    matrix = heads * d * d * size
    if kind in ("decode", "batch"):
        # Per token the window and the operands, per pass the selected
        # matrices (a pass holds one route per request).
        lengths = [case["tokens"]] if kind == "decode" else [
            case["tokens"] // 2 + (2 * r + 1) * case["tokens"] // (4 * case["batch"])
            for r in range(case["batch"])]
        nbytes = flops = 0
        for n in lengths:
            window = n if n < FIRST else KEEP + (n - FIRST) % BLOCK
            m = _routed(_fines(n))[1]
            nbytes += case["steps"] * (2 * window + 6) * row + m * matrix
            flops += case["steps"] * heads * (4 * window * d + (2 * d * d if m else 0))
        return {"bytes": nbytes, "flops": flops}
    tokens = case["tokens"] + case["steps"]
    local = read = 0
    for start in range(0, tokens, BLOCK):
        n = min(BLOCK, tokens - start)
        local += n * min(start, KEEP) + n * (n + 1) // 2
        read += n * _routed(_fines(start))[1]
    fines = _fines(tokens)
    flops = 4 * d * local + 2 * d * d * (read + BLOCK * fines)
    nbytes = 6 * tokens * row
    if case["writer"] != "softmax":       # Gram matrix, factor and solve of each fine
        flops += fines * (2 * BLOCK * d * d + 2 * d ** 3 // 3 + 2 * d ** 3)
    if kind == "request":
        nbytes += fines * matrix
    if kind == "train":
        flops, nbytes = 3.5 * flops, 12 * tokens * row
    scale = case["batch"] * heads
    return {"bytes": nbytes * case["batch"], "flops": flops * scale}


def tolerance(case):
    # About four times the distance from exact() measured over these ranges:
    # 4e-7 in fp32, 4e-3 for bf16 heads (their own rounding is 1.6e-3), 6e-3
    # for the bf16 gradient of raw_q.
    if case["dtype"] == "fp32":
        return {"rel": 2e-6, "max": 2e-4}
    return {"rel": 0.022 if case["kind"] == "train" else 0.015, "max": 0.5}


# ---- the same in 64 bits ----------------------------------------------------
# Routes are whole numbers that follow from rounded descriptors and scores, so
# those are rounded where the operator defines it; everything that is summed
# or read is in 64 bits.

class _Exact:
    def __init__(self, case):
        self.case = case
        self.low = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        self.feature = case["writer"] in ("feature_mass_association",
                                          "structured_gram_association")

    def r(self, x):
        return x.to(self.low).double()

    def pinned(self, x, rounded):
        """The rounded value, with the unrounded one's derivative."""
        return x + (rounded - x).detach()

    def lse(self, x, dim):
        """logsumexp as separate rounded operations."""
        r = self.r
        top = x.detach().amax(dim, keepdim=True)
        total = r(r((r(x.detach() - top)).exp()).sum(dim))
        return self.pinned(torch.logsumexp(x, dim), r(r(total.log()) + top.squeeze(dim)))

    def solve(self, first, cross, mass, count):
        d = cross.shape[-1]
        if self.case["writer"] == "structured_gram_association":
            # (diag(var + ridge) - var var^T / sum(var) + mass mass^T / count)^-1 cross
            var = (first - mass * mass / count).clamp_min(0)
            ridge = first.sum(-1, keepdim=True) / d
            system = (torch.diag_embed(var + ridge)
                      - var.unsqueeze(-1) * var.unsqueeze(-2) / var.sum(-1)[..., None, None]
                      + mass.unsqueeze(-1) * mass.unsqueeze(-2) / count)
        else:
            ridge = first.diagonal(dim1=-2, dim2=-1).mean(-1)
            system = first + ridge[..., None, None] * torch.eye(d, dtype=first.dtype,
                                                                device=first.device)
        return torch.linalg.solve(system, cross)

    def write(self, raw_k, v, fines):
        """Descriptors, matrices and page matrices; raw_k, v [B, H, T, D]."""
        b, h, _, d = raw_k.shape
        kb = raw_k[:, :, :fines * BLOCK].reshape(b, h, fines, BLOCK, d)
        vb = v[:, :, :fines * BLOCK].reshape(b, h, fines, BLOCK, d)
        pages = fines // GROUP

        def grouped(x):
            return x[:, :, :pages * GROUP].unflatten(2, (pages, GROUP)).sum(3)

        soft = torch.softmax(kb, 3)
        self.z, self.mass, self.page_c = self.lse(kb, 3), None, None
        if self.case["writer"] == "softmax":
            self.c = soft.transpose(-1, -2) @ vb
        else:
            u = torch.softmax(kb, -1)
            u = self.pinned(u, self.r(u))
            cross, mass = u.transpose(-1, -2) @ vb, u.sum(3)
            first = ((u * u).sum(3) if self.case["writer"].startswith("structured")
                     else u.transpose(-1, -2) @ u)
            self.c = self.solve(first, cross, mass, BLOCK)
            if self.feature:
                self.mass = mass
                self.z = self.pinned(mass.log(), self.r(mass.log()))
            if pages:
                self.page_c = self.solve(grouped(first), grouped(cross), grouped(mass),
                                         GROUP * BLOCK)
        self.page_z = [self.page(p * GROUP, (p + 1) * GROUP) for p in range(pages)]
        if self.case["writer"] == "softmax" and pages and self.case["values"]:
            w = (self.z[:, :, :pages * GROUP].unflatten(2, (pages, GROUP))
                 - torch.stack(self.page_z, 2).unsqueeze(3)).exp().flatten(2, 3)
            self.page_c = grouped(w.unsqueeze(-1) * self.c[:, :, :pages * GROUP])

    def page(self, low, high):
        if self.feature:
            x = self.mass[:, :, low:high].sum(2).log()
            return self.pinned(x, self.r(x))
        return self.lse(self.z[:, :, low:high], 2)

    def pages_at(self, fines):
        done, pending = divmod(fines, GROUP)
        pz = self.page_z[:done] + ([self.page(done * GROUP, fines)] if pending else [])
        return torch.stack(pz, 2)

    @torch.no_grad()
    def select(self, raw_q, fines):
        """0/1 [B, H, Q, fines]: the fines that each query of raw_q routes to."""
        r = self.r
        pz = self.pages_at(fines)
        of = torch.arange(fines, device=pz.device) // GROUP
        sw = r(r(self.z[:, :, :fines] - pz[:, :, of]).exp())
        hv = r(r(torch.softmax(raw_q, -1)).unsqueeze(3) * r(torch.softmax(pz, 2)).unsqueeze(2))
        done = fines // GROUP
        pages, m = _routed(fines)
        mass = r(hv.sum(-1))[..., :done]
        chosen = mass.argsort(dim=-1, descending=True, stable=True)[..., :pages]
        open_ = torch.zeros_like(mass, dtype=torch.bool).scatter_(-1, chosen, True)
        open_ = torch.cat([open_, torch.ones_like(hv[..., 0][..., :1], dtype=torch.bool)], -1)
        score = torch.stack([r(r(hv[..., f // GROUP, :] * sw[:, :, None, f]).sum(-1))
                             for f in range(fines)], -1)
        score = score.masked_fill(~open_[..., of], -math.inf)
        best = score.argsort(dim=-1, descending=True, stable=True)[..., :m]
        return torch.zeros_like(score).scatter_(-1, best, 1.0)

    def mixture(self, h, z, c, mask=None):
        mass = h @ z.exp().transpose(-1, -2)
        mass = mass if mask is None else mass * mask
        w = mass / mass.sum(-1, keepdim=True)
        return sum((w[..., f:f + 1] * h) @ c[:, :, f] for f in range(c.shape[2]))

    def history(self, h, mask, fines):
        """(fine, coarse or None) read by the queries h [B, H, Q, D]."""
        done = fines // GROUP
        coarse, values = None, self.case["values"] and done > 0
        if self.feature:
            fine = self.mixture(h, self.z[:, :, :fines], self.c[:, :, :fines], mask)
            if values:
                coarse = self.mixture(h, torch.stack(self.page_z[:done], 2),
                                      self.page_c[:, :, :done])
            return fine, coarse
        pz = self.pages_at(fines)
        pw = torch.softmax(pz, 2)
        num, den = 0, 0
        for f in range(fines):
            p = f // GROUP
            w = pw[:, :, p] * (self.z[:, :, f] - pz[:, :, p]).exp()
            a = h * w.unsqueeze(2) * mask[..., f:f + 1]
            num, den = num + a @ self.c[:, :, f], den + a.sum(-1, keepdim=True)
        if values:
            cw = torch.softmax(pz[:, :, :done], 2)
            coarse = h @ (cw.unsqueeze(-1) * self.page_c[:, :, :done]).sum(2)
        return num / den, coarse

    def outputs(self, q, k, v, raw_q, raw_k, fusion, first, routed):
        """Heads [B, T - first, H, D] from position `first` on; operands
        [B, T, H, D]; routed: a route for every query and not for each turn."""
        q, k, v, raw_q, raw_k = (x.transpose(1, 2).double() for x in (q, k, v, raw_q, raw_k))
        fa, fb = (x.double().unsqueeze(1) for x in fusion)             # [H, 1, D, 3]
        total, d = q.shape[2], q.shape[3]
        if _fines(total - 1):
            self.write(raw_k, v, _fines(total - 1))
        parts, mask = [], None
        began = max(0, first - PERIOD) // BLOCK * BLOCK    # the turn that `first` reads under
        for start in range(began, total, BLOCK):
            end = min(total, start + BLOCK)
            at = max(0, start - KEEP)
            rows = torch.arange(start, end, device=q.device)
            fines = _fines(start)
            if fines and routed:
                mask = self.select(raw_q[:, :, start:end], fines)
            elif fines:
                turns = [p for p in range(start, end) if (p - FIRST) % PERIOD == 0]
                old = torch.zeros_like(q[:, :, :1, :1]).expand(-1, -1, 1, fines).clone()
                if mask is not None:
                    old[..., :mask.shape[-1]] = mask[:, :, -1:]
                picked = torch.cat([old, self.select(raw_q[:, :, turns], fines)], 2)
                upto = torch.tensor([sum(t <= p for t in turns) for p in range(start, end)],
                                    device=q.device)
                mask = picked[:, :, upto]
            if end <= first:
                continue
            s = q[:, :, start:end] @ k[:, :, at:end].transpose(-1, -2) / math.sqrt(d)
            seen = torch.arange(at, end, device=q.device) <= rows[:, None]
            out = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, :, at:end]
            if fines:
                rq = raw_q[:, :, start:end]
                # Queries before the oldest turn considered are not returned.
                used = mask if routed else mask.index_fill(2, (rows < first).nonzero()[:, 0], 1.0)
                fine, coarse = self.history(torch.softmax(rq, -1), used, fines)
                score = fa * rq.unsqueeze(-1) + fb
                score = score + torch.tensor(
                    [math.log(2) if coarse is not None else 0.0,
                     0.0 if coarse is not None else -math.inf, 0.0], device=q.device).double()
                rho = torch.softmax(score, -1)
                out = 2 * rho[..., 0] * out + 2 * ALPHA * rho[..., 2] * fine
                if coarse is not None:
                    out = out + 2 * ALPHA * rho[..., 1] * coarse
            parts.append(out[:, :, max(0, first - start):])
        return torch.cat(parts, 2).transpose(1, 2)


def exact(case, seed):
    g = _generator(seed)
    fusion = _fusion(case, g)
    kind, steps = case["kind"], case["steps"]
    if kind == "request":
        xs = _tokens(case, 1, case["tokens"] + steps, g)
        out = _Exact(case).outputs(*xs, fusion, 0, False)
        width = case["chunk"] or case["tokens"]
        return [out[:, c:min(c + width, case["tokens"])]
                for c in range(0, case["tokens"], width)] + [
            out[:, i:i + 1] for i in range(case["tokens"], case["tokens"] + steps)]
    if kind in ("decode", "batch"):
        lengths = [case["tokens"]] if kind == "decode" else _lengths(case, seed)
        prompts = []
        for length in lengths:
            pieces = list(_pieces(case, length, g))
            prompts.append([torch.cat([p[i] for p in pieces], 1) for i in range(5)])
        new = _tokens(case, len(lengths), steps, g)
        outs = []
        for r, (length, prompt) in enumerate(zip(lengths, prompts)):
            xs = [torch.cat([a, b[r:r + 1]], 1) for a, b in zip(prompt, new)]
            outs.append(_Exact(case).outputs(*xs, fusion, length, False))
        out = torch.cat(outs, 0)
        return [out[:, i:i + 1] for i in range(steps)]
    xs = _tokens(case, case["batch"], case["tokens"], g)
    if kind == "full":
        with torch.no_grad():
            return _Exact(case).outputs(*xs, fusion, 0, True)
    grad = torch.randn(xs[0].shape, generator=g, device="cuda").to(xs[0].dtype)
    leaves = [x.double().requires_grad_(True) for x in xs + fusion]
    out = _Exact(case).outputs(*leaves[:5], leaves[5:], 0, True)
    grads = torch.autograd.grad(out, leaves, grad.double(), allow_unused=True)
    return [out.detach(), *(torch.zeros_like(x) if d is None else d
                            for x, d in zip(leaves, grads))]
