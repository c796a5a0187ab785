"""Host copy of the plan rules of tomocupy_amd/csrc (common.hip, fft_lds.h,
fourierrec.hip, filter.hip): which passes a transform length runs."""

MAX_PRIME, REG_PRIME, VALS = 127, 17, 20
COMPILED = {256, 512, 768, 1024, 1280, 1536, 2048, 2304, 2560, 3072, 3840, 4096, 4608, 5120,
            6144, 8192}
# compiled lengths of the separate filter's rows
ROWS16 = {256, 512, 1024, 2048, 4096, 8192, 16384}
ROWS32 = ROWS16 | COMPILED | {7680, 9216, 10240, 12288, 15360}
LDS = 160 * 1024


def rule(n):
    """FftPlan::radices: the radix sequence by which lengths are accepted."""
    if n > 16384:
        return None
    r, m = [], n
    for p in [16, 8, 4, 2] + list(range(3, MAX_PRIME + 1)):
        while m % p == 0:
            r.append(p)
            m //= p
    return r if m == 1 else None


def maxb(radix):
    """rt_maxb"""
    return 8 if radix == 2 else VALS // radix if radix <= VALS // 2 else 1


def is_prime_pass(radix):
    return radix > VALS or radix == 19


_COST = [0, 0, 3, 4.5, 4, 6.5, 6, 10, 6, 8, 8.5, 15, 8, 18, 12, 10, 9.5, 24, 10, -1, 9.5]


def plan(n, lg=0):
    """fft_rt_radices: (radices, cost), or (None, 0)."""
    fixed, m = [], n
    for p in range(MAX_PRIME, REG_PRIME, -1):
        if all(p % q for q in range(2, int(p ** 0.5) + 1)):
            while m % p == 0:
                fixed.append(p)
                m //= p
    best = {1: (0.0, 1)}
    for v in [v for v in range(2, m + 1) if m % v == 0]:
        b = (1e30, 0)
        for r in range(2, VALS + 1):
            if r == 19 or v % r or (n // r) << lg > 1024 * maxb(r) or v // r not in best:
                continue
            c = best[v // r][0] + 11 + 24 / r + _COST[r]
            if c < b[0]:
                b = (c, r)
        if b[1]:
            best[v] = b
    if m not in best:
        return None, 0.0
    rest, v = [], m
    while v > 1:
        rest.append(best[v][1])
        v //= best[v][1]
    rest.sort(key=lambda r: (r & -r, -r))
    return fixed + rest, best[m][0]


def _waves(nb, p, g):
    return (nb + 63) // 64 * (((p - 1) // 2 + g - 1) // g)


def pairs(nb, p):
    """rt_prime_pairs"""
    return 8 if _waves(nb, p, 8) <= 16 else 12 if _waves(nb, p, 12) <= 16 else 16


def threads(n, radices, lg=0, one_each=True):
    """fft_rt_threads"""
    t = one = 64
    for r in radices:
        nb = (n // r) << lg
        if is_prime_pass(r):
            t = max(t, 64 * _waves(nb, r, pairs(nb, r)))
        else:
            t, one = max(t, -(-nb // maxb(r))), max(one, nb)
    if one_each and n <= 1024 and one <= 512:
        t = max(t, one)
    t = (t + 63) // 64 * 64
    return t if t <= 1024 else -1


def wide(n, radices, lg=0):
    """fft_rt_wide"""
    return any(is_prime_pass(r) and pairs((n // r) << lg, r) == 16 for r in radices)


def rule_threads(radices, elems, ept=16):
    """fft_threads"""
    per = ept
    for r in radices:
        if r <= 8 or r == 16 or (r <= 17 and r <= ept):
            per = min(per, ept // r * r)
    t = (-(-elems // per) + 63) // 64 * 64
    return max(t, 256) if t <= 1024 else -1


def width_ok(n):
    """fr_fft_shapes_ok"""
    r1, r2 = rule(n), rule(2 * n)
    if n % 2 or n < 20 or r1 is None or r2 is None:
        return False
    m = n
    for p in (2, 3):
        while m % p == 0:
            m //= p
    shapes = ((r1, n, 16), (r2, 2 * n, 16), (r2, 2 * n, 32 if m == 1 else 16))
    return all(0 < rule_threads(r, e, ept) <= 512 for r, e, ept in shapes)


def row_ok(ne):
    """flt_create's lengths"""
    r = rule(ne)
    return ne % 2 == 0 and r is not None and rule_threads(r, ne) > 0


def column_plan(n):
    """fr_create: (radices, lg) of a run-time column pass."""
    n2 = 2 * n
    r, cost = plan(n2)
    lg = 0
    while (lg < 4 and (8 * n2) << (lg + 1) <= LDS and threads(n2, r, lg + 1) > 0
           and not wide(n2, r, lg + 1)):
        lg += 1
    if lg < 3 and (8 * n2) << (lg + 1) <= LDS:
        more, c = plan(n2, lg + 1)
        if (more and c <= 1.1 * cost and threads(n2, more, lg + 1) > 0
                and not wide(n2, more, lg + 1)):
            return more, lg + 1
    return r, lg


def kinds(radices):
    """The pass instances a plan of lds_fft runs: (radix, first or later)."""
    return {('prime' if is_prime_pass(r) else r, 'first' if i == 0 else 'later')
            for i, r in enumerate(radices)}


def rule_kinds(radices):
    """The same of lds_fft_rule: padded output, padded input, plain."""
    pad = len(radices) > 1 and radices[1] <= REG_PRIME and radices[0] % 2 == 0
    return {('prime' if is_prime_pass(r) else r, ('out', 'in')[i] if pad and i < 2 else 'plain')
            for i, r in enumerate(radices)}
