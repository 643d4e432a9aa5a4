"""Performance cases of the gate-bootstrapping engine: the calls that programs built on it make, with the
keys, sizes and gate mixes that its benchmark, tests and circuits use.

A case's "path" is one of
  gate        one gate per launch on the caller's stream (the plain form), or `n` gates on `n` streams
  plan        a batch of gates over a device pool of wires, planned once and run again and again
  annihilate  annihilation key switching of a batch of TRLWEs
  serve       layered circuits submitted to the continuous-batching server (host ciphertexts in and out)

Every output is the torus words of ciphertexts. The lvl1 arithmetic is exact (FP64 products stay below 2^50 and
round to the integer, the NTT is modular) and every lvl2 NTT result is exact too. The lvl2 FFT rotation rounds in
FP64, but no tolerance between "the same words" and "all words differ" exists for it: one gadget digit that
rounds the other way replaces the whole (uniform) mask of the result. So every case is compared exactly.
"""
import ctypes

import numpy as np
import torch

import cufhe_amd as C
from cufhe_amd.circuits import BINARY, random_circuit

N0, N1, N2 = C.N0, C.N1, C.N2
STEPS = N0 // 2  # key-bundle steps of a rotation

# level, backend, rotation variant and subset key switch of a key set; the ones that the benchmark and the tests
# load. A program loads one lvl1 set and, for the lvl02 API, one lvl2 set beside it.
KEYS = {
    "lvl1-kb": (1, C.BACKEND_FFT, C.BR_KEY_BUNDLE, False),
    "lvl1-plain": (1, C.BACKEND_FFT, C.BR_PLAIN, False),
    "lvl1-ntt-bb": (1, C.BACKEND_NTT, C.BR_BLOCK_BINARY, True),
    "lvl2-kb": (2, C.BACKEND_FFT, C.BR_KEY_BUNDLE, False),
    "lvl2-ntt-kb": (2, C.BACKEND_NTT, C.BR_KEY_BUNDLE, False),
}

_host = {}    # host keys by name, generated once
_loaded = {}  # level -> name of the key set on the GPU


def _secret(block_binary):
    if ("secret", block_binary) not in _host:
        _host["secret", block_binary] = C.secret_key_gen(11, block_binary=block_binary)
    return _host["secret", block_binary]


def _secret_of(name):
    return _secret(KEYS[name][2] == C.BR_BLOCK_BINARY)


def _use_keys(name):
    """Loads the key set unless it is the one on the GPU."""
    level, backend, variant, subset = KEYS[name]
    if _loaded.get(level) == name:
        return
    k0, k1, k2 = _secret_of(name)
    kt = k1 if level == 1 else k2
    bundle = variant == C.BR_KEY_BUNDLE
    tag = (level, bundle, variant == C.BR_BLOCK_BINARY)
    if tag not in _host:
        _host[tag] = C.bk_gen(level, bundle, 12, k0, kt), C.ksk_gen(level, 13, kt, k0, subset=subset)
    bk, ksk = _host[tag]
    C.check(C.lib().cufhe_initialize(), "cufhe_initialize")
    if level == 1:
        C.initialize_lvl01(bk, ksk, backend=backend, variant=variant, subset=subset)
    else:
        C.initialize_lvl02(bk, ksk, backend=backend, key_bundle=bundle)
    _loaded[level] = name


def _use_annihilation_key(level):
    if _loaded.get(("annihilate", level)):
        return
    key = _secret(False)[level]
    C.check(C.lib().cufhe_initialize(), "cufhe_initialize")
    C.annihilate_key_load(level, C.annihilate_key_gen(level, 14, key))
    _loaded["annihilate", level] = True


class _Wires:
    """Device memory of a program: a torch tensor and the pointer that the engine takes."""

    def __init__(self, host):
        self.tensor = torch.from_numpy(host).cuda()
        self.ptr = ctypes.c_void_p(self.tensor.data_ptr())
        self.row_bytes = self.tensor.stride(0) * self.tensor.element_size()

    def at(self, row):
        return ctypes.c_void_p(self.ptr.value + row * self.row_bytes)


# ------------------------------------------------------------------- cases

def listed():
    return [
        # one gate for a caller that waits for it: the reference's form of use
        {"name": "gate_nand", "path": "gate", "keys": "lvl1-kb", "api": 1, "op": "NAND", "n": 1},
        # the reference's throughput form: gates on streams of their own
        {"name": "gate_streams24", "path": "gate", "keys": "lvl1-kb", "api": 1, "op": "XOR", "n": 24},
        # the lvl02 API's one gate, of the two-rotation kind
        {"name": "gate_lvl02_mux", "path": "gate", "keys": "lvl2-kb", "api": 2, "op": "MUX", "n": 1},
        # one layer of one circuit request (an AES-128 layer holds up to 304 gates)
        {"name": "layer_150", "path": "plan", "keys": "lvl1-kb", "api": 1, "n": 150, "mux": 0.1, "graph": False},
        # a layer of several requests together; odd, more than one job per CU
        {"name": "layer_1011", "path": "plan", "keys": "lvl1-kb", "api": 1, "n": 1011, "mux": 0.1, "graph": True},
        # the benchmark's batch: 4096 binary gates
        {"name": "batch_4096", "path": "plan", "keys": "lvl1-kb", "api": 1, "n": 4096, "mux": 0.0, "graph": True},
        # keys without the bundle (one CMUX per key bit), lvl0 wires: half the key memory
        {"name": "plain_keys_500", "path": "plan", "keys": "lvl1-plain", "api": 0, "n": 500, "mux": 0.1,
         "graph": False},
        # the benchmark's exact backend: block-binary keys, subset key switch
        {"name": "ntt_bb_4096", "path": "plan", "keys": "lvl1-ntt-bb", "api": 1, "n": 4096, "mux": 0.0,
         "graph": True},
        # the benchmark's lvl2 mix: 1536 binary gates and 512 MUX
        {"name": "lvl02_mix_2048", "path": "plan", "keys": "lvl2-kb", "api": 2, "n": 2048, "mux": 0.25,
         "graph": True},
        # TRLWE packing support: lvl1 and lvl2 batches
        {"name": "annihilate_4096", "path": "annihilate", "level": 1, "n": 4096},
        {"name": "annihilate_lvl2_1000", "path": "annihilate", "level": 2, "n": 1000},
        # small circuits from several callers at once
        {"name": "serve_6", "path": "serve", "keys": "lvl1-kb", "requests": 6, "width": 40, "depth": 4},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    path = rng.choice(["gate", "plan", "plan", "plan", "annihilate", "serve"])
    if path == "gate":
        keys = rng.choice(["lvl1-kb", "lvl1-kb", "lvl1-plain", "lvl1-ntt-bb", "lvl2-kb"])
        api = 2 if keys == "lvl2-kb" else rng.choice([0, 1])
        return {"path": path, "keys": keys, "api": api, "op": rng.choice(BINARY + ["MUX", "NMUX"]),
                "n": rng.choice([1, 1, 1, _log_int(rng, 2, 24)])}
    if path == "plan":
        keys = rng.choice(["lvl1-kb", "lvl1-kb", "lvl1-kb", "lvl1-plain", "lvl1-ntt-bb", "lvl2-kb", "lvl2-ntt-kb"])
        most = {"lvl1-plain": 2048, "lvl2-kb": 1536, "lvl2-ntt-kb": 60}.get(keys, 4096)
        api = 2 if keys.startswith("lvl2") else rng.choice([1, 1, 0])
        return {"path": path, "keys": keys, "api": api, "n": _log_int(rng, 2, most),
                "mux": rng.choice([0.0, 0.1, 0.25]), "graph": rng.random() < 0.5}
    if path == "annihilate":
        level = rng.choice([1, 2])
        return {"path": path, "level": level, "n": _log_int(rng, 1, 4096 if level == 1 else 1024)}
    return {"path": path, "keys": "lvl1-kb", "requests": rng.randint(1, 8), "width": _log_int(rng, 4, 64),
            "depth": rng.randint(2, 5)}


# ---------------------------------------------------------- before the call

def _wire_level(api):
    return 1 if api == 1 else 0  # lvl0 wires for the lvl0 and the lvl02 API


def _gates(rng, n, mux_share, ops=None):
    """n gates over n + 2 input wires: (op, out, in0, in1, inc) with the outputs behind the inputs."""
    if ops is None:
        ops = rng.choice(BINARY, n).tolist()
        for i in rng.choice(n, int(round(mux_share * n)), replace=False):
            ops[i] = "MUX" if rng.random() < 0.5 else "NMUX"
    inputs = n + 2
    wires = rng.integers(0, inputs, (n, 3))
    return inputs, [(ops[i], inputs + i, int(wires[i, 0]), int(wires[i, 1]), int(wires[i, 2])) for i in range(n)]


def _encrypted(name, level, seed, count, spare):
    """`count` encryptions of random bits and `spare` rows for results."""
    bits = np.random.default_rng(seed + 1).integers(0, 2, count).astype(np.uint8)
    host = np.zeros((count + spare, C.tlwe_words(level)), np.uint32)
    host[:count] = C.encrypt_bits(level, seed, _secret_of(name)[level], bits)
    return host


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    path = case["path"]
    if path == "annihilate":
        level, n = case["level"], case["n"]
        _use_annihilation_key(level)
        # uniform words: what a TRLWE looks like without the key (here, encryptions of uniform polynomials)
        words = 2 * (N1 if level == 1 else N2)
        signed, width = (np.int32, 32) if level == 1 else (np.int64, 64)
        host = rng.integers(-(1 << (width - 1)), 1 << (width - 1), (n, words), dtype=signed)
        src = torch.from_numpy(host).cuda()
        return {"path": path, "level": level, "n": n, "words": words, "src": src, "out": torch.empty_like(src)}
    _use_keys(case["keys"])
    if path == "serve":
        requests = []
        for r in range(case["requests"]):
            circuit = random_circuit(rng, case["width"], case["depth"])
            requests.append((circuit, _encrypted(case["keys"], 1, seed * 16 + r, circuit.n_inputs, 0)))
        return {"path": path, "server": C.Server(pool_bytes=64 << 20), "requests": requests}
    api, n = case["api"], case["n"]
    if path == "gate":
        inputs, gates = _gates(rng, n, 0.0, [case["op"]] * n)
    else:
        inputs, gates = _gates(rng, n, case["mux"])
    wires = _Wires(_encrypted(case["keys"], _wire_level(api), seed, inputs, n).view(np.int32))
    state = {"path": path, "api": api, "wires": wires, "out": wires.tensor[inputs:]}
    if path == "plan":
        state["plan"] = C.Plan(gates, wires, use_graph=case["graph"], level=api)
    else:
        launch = {0: C.lib().cufhe_gate_lvl0, 1: C.lib().cufhe_gate_lvl1, 2: C.lib().cufhe_gate_lvl02}[api]
        streams = [C.Stream() for _ in gates] if n > 1 else [None]
        state["streams"] = streams
        state["calls"] = [(launch, C.GATES[op], wires.at(out), wires.at(in0), wires.at(in1), wires.at(inc),
                           s.handle if s else None) for (op, out, in0, in1, inc), s in zip(gates, streams)]
    return state


# ----------------------------------------------------------------- the call

def run(state):
    path = state["path"]
    if path == "plan":
        state["plan"].run()
        return state["out"]
    if path == "gate":
        for launch, op, out, in0, in1, inc, stream in state["calls"]:
            C.check(launch(op, out, in0, in1, inc, stream), "gate")
        return state["out"]
    if path == "annihilate":
        C.check(C.lib().cufhe_annihilate_key_switch_batch(
            state["level"], state["out"].data_ptr(), state["words"], state["src"].data_ptr(), state["words"],
            state["n"], None), "cufhe_annihilate_key_switch_batch")
        return state["out"]
    server = state["server"]
    ids = [server.submit(circuit, inputs) for circuit, inputs in state["requests"]]
    return [server.result(i).view(np.int32) for i in ids]


# --------------------------------------------------------------- what it is

def _fft(h):
    return 5 * h * (h.bit_length() - 1)


# one rotation: bytes of its key and operations. FFT: folded transforms of the digits and of the two results, and
# per bin the bundle (three complex products and sums, where there is one) and the product with it. NTT:
# butterflies of three operations, and a product and a sum per key word and digit word.
def _rotation(keys):
    if keys == "lvl1-kb":
        return 62521344, STEPS * (6 * _fft(512) + 8 * 512 * 32)
    if keys == "lvl1-plain":
        return 41680896, N0 * (6 * _fft(512) + 8 * 512 * 8)
    if keys == "lvl1-ntt-bb":
        return 20840448, N0 // 4 * (6 * 3 * 512 * 10 + 8 * 1024 * 2 * 5)
    if keys == "lvl2-kb":
        return 250085376, STEPS * (10 * _fft(1024) + 16 * 1024 * 32)
    return 250085376, STEPS * (10 * 3 * 1024 * 11 + 16 * 2048 * 2 * 4)


def _key_switch(keys):
    rows = {"lvl1-ntt-bb": N1 - N0}.get(keys, N2 if keys.startswith("lvl2") else N1) * 7
    return rows * 2 * (N0 + 1) * 4, rows * (N0 + 1)


def work(case):
    path = case["path"]
    if path == "annihilate":
        big, size, rounds, digits, bits = ((N1, 4, 10, 2, 327680) if case["level"] == 1 else (N2, 8, 11, 4, 1441792))
        per = rounds * ((digits + 2) * _fft(big // 2) + 2 * digits * (big // 2) * 8)
        return {"bytes": case["n"] * 2 * 2 * big * size + bits, "flops": case["n"] * per}
    if path == "serve":
        rotations = case["requests"] * case["width"] * case["depth"] * 1.1
        wires, words = case["requests"] * case["width"] * 2, N1 + 1
    elif path == "gate":
        rotations = case["n"] * (2 if case["op"] in ("MUX", "NMUX") else 1)
        wires, words = 2 * case["n"] + 2, N1 + 1 if case["api"] == 1 else N0 + 1
    else:
        rotations = case["n"] + int(round(case["mux"] * case["n"]))
        wires, words = 2 * case["n"] + 2, N1 + 1 if case["api"] == 1 else N0 + 1
    rotation, switch = _rotation(case["keys"]), _key_switch(case["keys"])
    return {"bytes": rotation[0] + switch[0] + wires * words * 4, "flops": rotations * (rotation[1] + switch[1])}


def tolerance(case):
    return "exact"
