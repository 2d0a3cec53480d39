"""Shared fixtures for the parity tests: seeded layers, the tolerance of the
benchmark definition, and device/oracle runners over the same bytes."""
from __future__ import annotations

import ctypes as C
import functools
import os
import subprocess
import tempfile

import numpy as np

from oracle import oracle as O
from shrike_amd import synth as S
from tests.conftest import ROOT

ABS_TOL, REL_TOL = 2e-3, 1e-3   # FFN outputs: max-abs 2e-3 / relative 1e-3 (benchmark definition)


def f16(bits: np.ndarray) -> np.ndarray:
    return S.f16_bits_to_f32(bits)


def assert_ffn_close(dev_bits: np.ndarray, ref_bits: np.ndarray, what: str = "", rel: float = REL_TOL):
    a, b = f16(dev_bits).astype(np.float64), f16(ref_bits).astype(np.float64)
    assert np.all(np.isfinite(b)), f"{what}: the oracle's output is not finite; the fixture is unusable"
    err = np.abs(a - b)
    bound = ABS_TOL + rel * np.abs(b)
    worst = int(np.argmax(err - bound))
    assert np.all(err <= bound), (
        f"{what}: element {worst}: device {a[worst]} vs oracle {b[worst]} "
        f"(|diff| {err[worst]:.3e} > {bound[worst]:.3e}); {int(np.sum(err > bound))} of {a.size} out of tolerance")


def assert_rel_close(dev_bits: np.ndarray, ref_bits: np.ndarray, what: str = "", tol: float = REL_TOL):
    """The reference's own metric (sources/ShrikeValidation/Support/Tolerance/RelError.swift:7-19):
    max |a - b| / max(max |b|, 1e-6). Used end to end, where fp16 roundings between the stages
    (gate/up -> act -> down) make single elements of a cancelling sum move by more than 2e-3."""
    a, b = f16(dev_bits).astype(np.float64), f16(ref_bits).astype(np.float64)
    assert np.all(np.isfinite(b)), f"{what}: the oracle's output is not finite"
    rel = np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-6)
    assert rel <= tol, f"{what}: relative error {rel:.3e} > {tol:.1e}"


class Layer:
    """One synthetic MoE layer: E routed expert blobs, router, optional shared expert."""

    def __init__(self, seed, d, f, num_experts, top_k, bits=4, meta=S.META_BF16, router_bits=0,
                 shared_f=0, shared_bits=None, additive_biases=False, label="layer.0", distinct=None):
        """distinct: of the experts' blobs, where making them all would take long; expert e has number e % distinct."""
        self.d, self.f, self.ne, self.k = d, f, num_experts, top_k
        self.bits, self.meta, self.router_bits = bits, meta, router_bits
        self.additive = additive_biases
        tree = S.SeedTree(seed)
        self.tree = tree
        self.off, self.stride = S.expert_offsets(d, f, bits, additive_biases)
        made = [S.expert_blob(tree, f"{label}.expert.{e}", d, f, bits, meta, additive_biases) for e in range(distinct or num_experts)]
        self.blobs = [made[e % len(made)] for e in range(num_experts)]
        # router
        if router_bits == 0:
            self.router_w = S.router_f16(tree, f"{label}.router.w", num_experts, d)
            self.router_s = self.router_b = None
        else:
            dense = tree.key(f"{label}.router.w").normal(num_experts * d, std=0.02).reshape(num_experts, d)
            self.router_w, self.router_s, self.router_b = S.quantize_affine(dense, router_bits, meta)
        self.eff_scale = S.f32_to_bf16_bits(np.ones(d, np.float32))
        self.expert_scale = S.f32_to_bf16_bits(np.ones(num_experts, np.float32))
        self.logit_bias = S.f32_to_bf16_bits(np.zeros(num_experts, np.float32))
        self.x = S.activations_f16(tree, f"{label}.x", d)
        self.hidden = S.activations_f16(tree, f"{label}.hidden", d)
        # shared expert as separate resident tensors
        self.shared_f = shared_f
        self.shared_bits = shared_bits or bits
        if shared_f:
            sb = self.shared_bits
            self.shared = {name: S.affine_matrix(tree.key(f"{label}.shared.{name}"), rows, n, sb, meta)
                           for name, rows, n in (("gate", shared_f, d), ("up", shared_f, d), ("down", d, shared_f))}

    def oracle_offsets(self):
        off, stride = O.expert_offsets(self.d, self.f, self.bits, self.additive)
        assert stride == self.stride
        return off

    def router_dict(self):
        return dict(weights=self.router_w, scales=self.router_s, biases=self.router_b,
                    kind=self.router_bits, eff_scale=self.eff_scale, expert_scale=self.expert_scale,
                    bias=self.logit_bias, meta=self.meta)


@functools.lru_cache(maxsize=None)
def ffn_rules() -> C.CDLL:
    """csrc/decode_rules.h, ffn_rules.h and router_rules.h, compiled for the host."""
    with tempfile.TemporaryDirectory() as where:
        lib = os.path.join(where, "rules.so")
        source = """
#include "decode_rules.h"
#include "ffn_rules.h"
#include "router_rules.h"
extern "C" uint32_t readable_records(uint32_t bound, uint64_t pairs, uint32_t experts) { return shrike::readable_records(bound, pairs, experts); }
extern "C" const char *routed_shape(uint64_t pairs, uint32_t experts, uint32_t d, uint32_t f, uint32_t bits) {
    static const char *const names[] = {"split", "tile", "deep", "wide"};
    return names[int(shrike::routed_shape(pairs, experts, d, f, bits))];
}
extern "C" bool takes_lines(uint64_t pairs, uint32_t experts, uint32_t d, uint32_t f, uint32_t bits, uint64_t align) {
    const shrike::FfnShape shape = shrike::routed_shape(pairs, experts, d, f, bits);
    return shrike::lines_shape(shape, pairs, experts, d, f, bits, align) == shrike::FfnShape::kLines;
}
extern "C" uint32_t logits_lds(uint32_t router_bits, uint32_t d) {
    return router_bits == 0 ? shrike::LogitsLds<0>::bytes(d) : router_bits == 8 ? shrike::LogitsLds<8>::bytes(d) : shrike::LogitsLds<4>::bytes(d);
}
extern "C" uint32_t phase1_row_steps(uint64_t workgroups, uint32_t d, uint32_t bits) { return shrike::phase1_row_steps(workgroups, d, bits); }
extern "C" bool past_the_cache(uint64_t experts, uint32_t d, uint32_t f, uint32_t bits) { return shrike::past_the_cache(experts, d, f, bits); }
"""
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{ROOT}/shrike_amd/csrc", "-x", "c++", "-", "-o", lib],
                       input=source.encode(), check=True)
        rules = C.CDLL(lib)
    rules.readable_records.argtypes, rules.readable_records.restype = [C.c_uint32, C.c_uint64, C.c_uint32], C.c_uint32
    rules.routed_shape.argtypes, rules.routed_shape.restype = [C.c_uint64, *[C.c_uint32] * 4], C.c_char_p
    rules.takes_lines.argtypes, rules.takes_lines.restype = [C.c_uint64, *[C.c_uint32] * 4, C.c_uint64], C.c_bool
    rules.logits_lds.argtypes, rules.logits_lds.restype = [C.c_uint32] * 2, C.c_uint32
    rules.phase1_row_steps.argtypes, rules.phase1_row_steps.restype = [C.c_uint64, C.c_uint32, C.c_uint32], C.c_uint32
    rules.past_the_cache.argtypes, rules.past_the_cache.restype = [C.c_uint64, *[C.c_uint32] * 3], C.c_bool
    return rules
