"""The run-time plans of every accepted length, by the host copy of their rules
(no GPU): each fits a workgroup of 1024 threads and its LDS, none of a detector
width needs the 16-pair prime passes that only the separate filter's kernels have,
and the lengths of test_gpu_runtime_radices.py reach every pass instance that an
accepted length reaches."""
import runtime_plans as rp
from test_gpu_runtime_radices import ROWS16, ROWS32, WIDTHS


def test_widths():
    count = 0
    for n in range(20, 4097, 2):
        if not rp.width_ok(n):
            continue
        count += 1
        for m in (n, 2 * n):
            r, _ = rp.plan(m)
            assert r and 0 < rp.threads(m, r) and not rp.wide(m, r), m
        r, lg = rp.column_plan(n)
        assert 0 < rp.threads(2 * n, r, lg) and not rp.wide(2 * n, r, lg), n
        assert (16 * n) << lg <= rp.LDS
    assert count > 1000


def test_filter_lengths():
    for ne in range(20, 16385, 2):
        if not rp.row_ok(ne):
            continue
        for r, one in ((rp.plan(ne)[0], True), (rp.rule(ne), False)):
            assert len(r) <= 16 and 0 < rp.threads(ne, r, one_each=one), ne
        assert 8 * (ne + ne // 16) <= rp.LDS


def test_gpu_lengths_reach_every_pass():
    image, rows16, rows32 = set(), set(), set()
    for n in range(20, 4097, 2):
        if rp.width_ok(n) and 2 * n not in rp.COMPILED:
            for r in (rp.plan(n)[0], rp.plan(2 * n)[0], rp.column_plan(n)[0]):
                image |= rp.kinds(r)
    for ne in range(20, 16385, 2):
        if rp.row_ok(ne) and ne not in rp.ROWS16:
            rows16 |= rp.kinds(rp.plan(ne)[0])
        if rp.row_ok(ne) and ne not in rp.ROWS32:
            rows32 |= rp.rule_kinds(rp.rule(ne))
    run = set()
    for n in WIDTHS:
        for r in (rp.plan(n)[0], rp.plan(2 * n)[0], rp.column_plan(n)[0]):
            run |= rp.kinds(r)
    assert image <= run
    assert rows16 <= set().union(*(rp.kinds(rp.plan(ne)[0]) for ne in ROWS16))
    assert rows32 <= set().union(*(rp.rule_kinds(rp.rule(ne)) for ne in ROWS32))
