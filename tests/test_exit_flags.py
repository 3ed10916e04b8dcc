"""Kernels of several workgroups decide their early exit alike in all
wavefronts of a workgroup: a wavefront must not test on its own a field of the
solver state that another workgroup of the same launch writes, or some of a
workgroup's wavefronts leave while the others go into its barriers.  Read from
the sources: the conditions of the returns before a kernel's first reduction
or barrier, against the fields that the kernel or its helpers write."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "parcel-legacy_amd", "csrc")
BARRIER = re.compile(r"__syncthreads|column_barrier|reduce_part|block_sum|store_partials")


def functions(src, head):
    for m in re.finditer(head + r"[^;{}]*?\b(\w+)\(([^{};]*)\)\s*\{", src):
        depth, i = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(src[i], 0)
            i += 1
        yield m.group(1), src[m.end():i]


def closure(body, helpers):
    seen, text, todo = set(), body, [body]
    while todo:
        for name in set(re.findall(r"\b(\w+)\(", todo.pop())) & set(helpers) - seen:
            seen.add(name)
            text += helpers[name]
            todo.append(helpers[name])
    return text


@pytest.mark.parametrize("name", ["bicg.hip", "gmres.hip", "ddcg.hip", "cg_kernels.hpp"])
def test_no_wavefront_tests_a_field_its_own_launch_writes(name):
    src = re.sub(r"//[^\n]*|__launch_bounds__\(\w+\)", "", open(os.path.join(CSRC, name)).read())
    helpers = dict(functions(src, r"__device__"))
    kernels = dict(functions(src, r"__global__"))
    assert len(kernels) > 3
    for k, body in kernels.items():
        launches = re.findall(r"hipLaunchKernelGGL\(\(?%s\b(?:<[^>]*>)?\)?,\s*(dim3\(1\)|\w+)" % k, src)
        if launches and all(g == "dim3(1)" for g in launches):
            continue
        first = BARRIER.search(body)
        before = body[:first.start()] if first else body
        conds = " ".join(re.findall(r"if \((.*)\) return;", before))
        tested = set(re.findall(r"st->(\w+)", closure(conds, helpers)))
        written = set(re.findall(r"st->(\w+)(?:\s*=[^=]|, \d|, \(unsigned)", closure(body, helpers)))
        assert not tested & written, (name, k, tested & written)
