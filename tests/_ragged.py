"""A ragged step on a device, from its lengths."""
import torch

from light_vllm_amd.utils.context import RaggedStep


def ragged_step(new, ctx, page, device, seed=0):
    """(step, number of pages): sequences of new[b] tokens behind ctx[b], pages in random order, state slots reversed."""
    cu, tok = [0], []
    for b, n in enumerate(new):
        cu.append(cu[-1] + n)
        tok += [b] * n
    need = [max(1, -(-(n + c) // page)) for n, c in zip(new, ctx)]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).tolist()
    tables, at = [], 0
    for k in need:
        tables.append(perm[at:at + k])
        at += k
    wide, B = max(need), len(new)
    i32 = dict(dtype=torch.int32, device=device)
    slots = list(reversed(range(B)))
    return RaggedStep(torch.tensor(cu, **i32), torch.tensor(ctx, **i32), torch.tensor(slots, **i32), torch.tensor(tok, **i32),
                      torch.tensor([t + [-1] * (wide - len(t)) for t in tables], **i32), new, ctx, slots, tables), sum(need)


def close(got, want, dtype):
    """f32 results within a few dozen roundings of each other; bf16 ones a rounding apart."""
    want = want.float()
    tol = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -18
    err = (got.cpu().float() - want).abs()
    return bool((err <= tol * want.abs() + tol * 1e-2).all())
