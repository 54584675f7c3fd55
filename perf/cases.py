"""Performance cases of the data-tiled matmul microkernels.

Every case is one pass of work that a program hands to iree_uk_pack, iree_uk_mmt4d
and iree_uk_unpack, over the sizes, element types, tile shapes and options they are
called with. Device operands are torch tensors and the calls are enqueued on torch's
current stream; the host cases leave the library in its default mode, where operands
lie in host memory and a call returns with its result. A case has a "kind":

  mmt4d   one product on operands that are tiled already
  chain   row-major activations -> pack -> mmt4d with weights packed beforehand -> unpack
  copy    pack, unpack, or one after the other
  host    one product whose operands are ordinary host memory

Logical sizes: an m x k matrix times a k x n matrix. Where a case is "mmt4d" or "host",
m, n and k are whole tiles; "chain" and "copy" take any size and pad.
"""
import ctypes as C
import math

import torch

from iree_amd import abi, library

# Per type: (mmt4d flag, lhs, rhs and result element types; None is two 4-bit values a byte).
_TYPES = {
    "s8": (abi.MMT4D_TYPE_S8S8S32, torch.int8, torch.int8, torch.int32),
    "s8s4": (abi.MMT4D_TYPE_S8S4S32, torch.int8, None, torch.int32),
    "f16": (abi.MMT4D_TYPE_F16F16F32, torch.float16, torch.float16, torch.float32),
    "bf16": (abi.MMT4D_TYPE_BF16BF16F32, torch.bfloat16, torch.bfloat16, torch.float32),
    "bf16_out16": (abi.MMT4D_TYPE_BF16BF16BF16 | abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS,
                   torch.bfloat16, torch.bfloat16, torch.bfloat16),
    "f32": (abi.MMT4D_TYPE_F32F32F32, torch.float32, torch.float32, torch.float32),
}

# The tile shapes (M0, N0, K0) that products of many rows come in: what
# iree_uk_query_tile_sizes_2d returns, the benchmark's own, and those of modules compiled
# for x86-64 and Arm; one-row tiles are row-major activations passed as they are.
_TILES = {
    "s8": [(16, 16, 64), (8, 8, 4), (16, 16, 2), (8, 8, 8), (1, 16, 64)],
    "s8s4": [(16, 16, 32)],
    "f16": [(16, 16, 16), (16, 16, 1), (1, 16, 16)],
    "bf16": [(16, 16, 16), (16, 16, 8), (16, 16, 2), (8, 8, 4)],
    "bf16_out16": [(16, 16, 16), (16, 16, 2)],
    "f32": [(16, 16, 4), (16, 16, 1)],
}

# N0 and K0 of few-row products; their M0 is the number of rows.
_DECODE_TILES = {
    "s8": [(16, 64), (16, 2)],
    "s8s4": [(16, 32)],
    "f16": [(16, 16), (16, 1)],
    "bf16": [(16, 8), (16, 2)],
}

_PACK_FLAGS = {"f32": (abi.PACK_TYPE_F32F32, torch.float32), "f16": (abi.PACK_TYPE_F16F16, torch.float16),
               "bf16": (abi.PACK_TYPE_BF16BF16, torch.bfloat16), "s8": (abi.PACK_TYPE_I8I8, torch.int8),
               "s32": (abi.PACK_TYPE_I32I32, torch.int32)}
_UNPACK_FLAGS = {"f32": abi.UNPACK_TYPE_F32F32, "f16": abi.UNPACK_TYPE_F16F16, "bf16": abi.UNPACK_TYPE_BF16BF16,
                 "s32": abi.UNPACK_TYPE_I32I32}
# Tile shapes of packed operands per element type (rows x columns of the row-major matrix).
_COPY_TILES = {
    "f32": [(16, 1), (16, 4), (16, 16)],
    "s32": [(16, 16), (8, 8)],
    "f16": [(16, 16), (16, 1)],
    "bf16": [(16, 16), (16, 8), (16, 2)],
    "s8": [(16, 64), (8, 4), (16, 2)],
}

_MAX_FLOPS = 2 * 4096 ** 3
_MAX_BYTES = 1 << 30
_MAX_F32_FLOPS = 2 * 1024 * 2048 * 2048
_MAX_HOST_BYTES = 48 << 20


def _mmt4d(name, type, m, n, k, tile, accumulate=False, kind="mmt4d"):
    return {"name": name, "kind": kind, "type": type, "m": m, "n": n, "k": k,
            "m0": tile[0], "n0": tile[1], "k0": tile[2], "accumulate": accumulate}


def listed():
    return [
        # A small quantised layer on a few tokens, everything odd: three calls whose kernels
        # take microseconds, so what counts is what a call costs.
        {"name": "chain_s8_tiny", "kind": "chain", "type": "s8", "m": 33, "n": 300, "k": 257},
        # The small square product that parity is stated on; a quarter of the chip's tiles.
        _mmt4d("s8_1024", "s8", 1024, 1024, 1024, (8, 8, 4)),
        # The headline product.
        _mmt4d("s8_4096", "s8", 4096, 4096, 4096, (8, 8, 4)),
        # A product that adds onto what the result holds (a K loop outside, a residual).
        _mmt4d("f16_4096_accumulate", "f16", 4096, 4096, 4096, (16, 16, 16), accumulate=True),
        # Prefill of 512 tokens against a weight matrix quantised to four bits.
        _mmt4d("s8s4_prefill_512", "s8s4", 512, 11008, 4096, (16, 16, 32)),
        # One decoded token through a feed-forward up-projection: streams the weights once.
        _mmt4d("bf16_decode_1", "bf16", 1, 14336, 4096, (1, 16, 8)),
        # One decode step of 64 sequences through the same weights.
        _mmt4d("bf16_decode_64", "bf16", 64, 14336, 4096, (16, 16, 8)),
        # One token against four-bit weights, a matrix small enough for latency to show.
        _mmt4d("s8s4_decode_1", "s8s4", 1, 11008, 4096, (1, 16, 32)),
        # A layer on a ragged batch of row-major activations: pack, product, unpack.
        {"name": "chain_bf16_ragged", "kind": "chain", "type": "bf16", "m": 777, "n": 4100, "k": 4095},
        # Tiled and back, both ways at sizes that no tile divides: bound by memory.
        {"name": "copy_f32_both_ways", "kind": "copy", "type": "f32", "rows": 8191, "cols": 8190, "t0": 16, "t1": 1,
         "inner": False, "outer": False, "way": "both"},
        # A [k][n] weight matrix into the layout the product reads, transposing tiles and their order.
        {"name": "copy_bf16_weights", "kind": "copy", "type": "bf16", "rows": 4096, "cols": 14336, "t0": 16, "t1": 16,
         "inner": True, "outer": True, "way": "pack"},
        # A drop-in call of a module compiled for x86-64: its tiles, its host buffers, result on return.
        _mmt4d("host_s8", "s8", 512, 2048, 2048, (16, 16, 2), kind="host"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _up(v, to):
    return -(-v // to) * to


def _draw_once(rng):
    family = rng.choice(["decode", "batch", "prefill", "chain", "chain", "copy", "copy", "host"])
    if family == "decode":
        t = rng.choice(sorted(_DECODE_TILES))
        n0, k0 = rng.choice(_DECODE_TILES[t])
        m = rng.choice([1, 1, 2, 4, 8, 16])
        return _mmt4d("", t, m, _up(_log(rng, 512, 28672), n0), _up(_log(rng, 512, 14336), k0), (m, n0, k0))
    if family in ("batch", "prefill"):
        t = rng.choice(sorted(_TILES))
        tile = rng.choice(_TILES[t])
        m = _log(rng, 17, 511) if family == "batch" else _log(rng, 512, 4096)
        return _mmt4d("", t, _up(m, tile[0]), _up(_log(rng, 256, 14336), tile[1]), _up(_log(rng, 256, 8192), tile[2]),
                      tile, accumulate=rng.random() < 0.25)
    if family == "chain":
        return {"kind": "chain", "type": rng.choice(["s8", "f16", "bf16", "f32"]), "m": _log(rng, 1, 4096),
                "n": _log(rng, 64, 14336), "k": _log(rng, 64, 8192)}
    if family == "copy":
        t = rng.choice(sorted(_COPY_TILES))
        tile = rng.choice(_COPY_TILES[t])
        way = "pack" if t == "s8" else rng.choice(["pack", "unpack", "both"])
        return {"kind": "copy", "type": t, "rows": _log(rng, 16, 16384), "cols": _log(rng, 16, 16384), "t0": tile[0],
                "t1": tile[1], "inner": rng.random() < 0.5, "outer": rng.random() < 0.5, "way": way}
    t = rng.choice(["s8", "bf16", "f32"])
    tile = {"s8": (16, 16, 2), "bf16": (16, 16, 2), "f32": (16, 16, 1)}[t]
    return _mmt4d("", t, _up(_log(rng, 16, 4096), tile[0]), _up(_log(rng, 64, 4096), tile[1]),
                  _up(_log(rng, 64, 4096), tile[2]), tile, accumulate=rng.random() < 0.25, kind="host")


def draw(rng):
    while True:
        case = _draw_once(rng)
        case.pop("name", None)
        w = work(case)
        if w["flops"] > (_MAX_F32_FLOPS if case["type"] == "f32" else _MAX_FLOPS) or w["bytes"] > _MAX_BYTES:
            continue
        if case["kind"] == "host" and w["bytes"] > _MAX_HOST_BYTES:
            continue
        return case


def _size(dtype):
    return torch.empty(0, dtype=dtype).element_size()


def work(case):
    if case["kind"] == "copy":
        e = _size(_PACK_FLAGS[case["type"]][1])
        plain = case["rows"] * case["cols"]
        tiled = _up(case["rows"], case["t0"]) * _up(case["cols"], case["t1"])
        pack, unpack = (plain + tiled) * e, 2 * plain * e
        return {"bytes": {"pack": pack, "unpack": unpack, "both": pack + unpack}[case["way"]], "flops": 0}
    _, lhs, rhs, out = _TYPES[case["type"]]
    m, n, k = case["m"], case["n"], case["k"]
    weights = n * k * _size(rhs) if rhs else n * k // 2
    passes = 2 if case.get("accumulate") else 1
    return {"bytes": m * k * _size(lhs) + weights + passes * m * n * _size(out), "flops": 2 * m * n * k}


def tolerance(case):
    if case["kind"] == "copy" or case["type"] in ("s8", "s8s4"):
        return "exact"
    if case["type"] == "bf16_out16":
        # One rounding to 8 significant bits, which another order of summation can tip.
        return {"rel": 4e-3, "max": 1e-2}
    # Sums of up to 14336 products in 32 bits, in any order.
    return {"rel": 1e-5, "max": 1e-3}


def _values(gen, count, dtype, sigma, device):
    if dtype in (torch.int8, None):
        return torch.randint(-128, 128, (count,), generator=gen, device=device, dtype=torch.int8)
    if dtype == torch.int32:
        return torch.randint(-2 ** 20, 2 ** 20, (count,), generator=gen, device=device, dtype=torch.int32)
    return (torch.randn(count, generator=gen, device=device) * sigma).to(dtype)


def _pack_params(src, rows, cols, dst, t0, t1, flags):
    """Row-major [rows, cols] -> tiles of t0 x t1 (of rows x columns), in the order the flags ask for."""
    outer, tile = [-(-rows // t0), -(-cols // t1)], [t0, t1]
    if flags & abi.PACK_TRANSPOSE_OUTER:
        outer.reverse()
    if flags & abi.PACK_TRANSPOSE_INNER:
        tile.reverse()
    p = abi.PackParams()
    p.in_buffer, p.in_stride0, p.in_stride1 = src.data_ptr(), cols, 1
    p.out_buffer, p.out_stride0, p.out_stride1 = dst.data_ptr(), outer[1] * t0 * t1, t0 * t1
    p.in_size0, p.in_size1 = rows, cols
    p.out_size0, p.out_size1, p.out_size2, p.out_size3 = outer + tile
    p.flags = flags
    return p


def _unpack_params(src, dst, rows, cols, t0, t1, flags):
    outer, tile = [-(-rows // t0), -(-cols // t1)], [t0, t1]
    if flags & abi.UNPACK_TRANSPOSE_OUTER:
        outer.reverse()
    if flags & abi.UNPACK_TRANSPOSE_INNER:
        tile.reverse()
    p = abi.UnpackParams()
    p.in_buffer, p.in_stride0, p.in_stride1 = src.data_ptr(), outer[1] * t0 * t1, t0 * t1
    p.out_buffer, p.out_stride0, p.out_stride1 = dst.data_ptr(), cols, 1
    p.in_size0, p.in_size1, p.in_size2, p.in_size3 = outer + tile
    p.out_size0, p.out_size1 = rows, cols
    p.flags = flags
    return p


def _mmt4d_params(lhs, rhs, out, tiles, tile, flags):
    p = abi.Mmt4dParams()
    p.M, p.N, p.K = tiles
    p.M0, p.N0, p.K0 = tile
    p.lhs_buffer, p.rhs_buffer, p.out_buffer = lhs.data_ptr(), rhs.data_ptr(), out.data_ptr()
    p.lhs_stride0, p.rhs_stride0, p.out_stride0 = p.K * p.M0 * p.K0, p.K * p.N0 * p.K0, p.N * p.M0 * p.N0
    p.flags = flags
    return p


def _queried_tile(lib, type):
    op = {"s8": abi.QTS_OP_MATMUL_I8I8I32, "f16": abi.QTS_OP_MATMUL_F16F16F32, "bf16": abi.QTS_OP_MATMUL_BF16BF16F32,
          "f32": abi.QTS_OP_MATMUL_F32F32F32}[type]
    sizes = []
    for role in (abi.QTS_ROLE_LHS, abi.QTS_ROLE_RHS):
        q, o = abi.QueryTileSizes2dParams(flags=op | role), abi.QueryTileSizes2dOutParams()
        lib.iree_uk_query_tile_sizes_2d(C.byref(q), C.byref(o))
        sizes.append((o.tile_size0, o.tile_size1))
    return sizes[0][0], sizes[1][0], sizes[0][1]


def _prepare_product(lib, case, device, gen):
    flag, lhs_t, rhs_t, out_t = _TYPES[case["type"]]
    m, n, k = case["m"], case["n"], case["k"]
    tile = case["m0"], case["n0"], case["k0"]
    lhs = _values(gen, m * k, lhs_t, 1.0 / math.sqrt(k) if case["type"] == "f16" else 1.0, device)
    rhs = _values(gen, n * k if rhs_t else n * k // 2, rhs_t, 1.0 if case["type"] == "f16" else 0.02, device)
    out = (_values(gen, m * n, out_t, 1.0, device) if case["accumulate"]
           else torch.zeros(m * n, dtype=out_t, device=device))
    flags = flag | (abi.MMT4D_ACCUMULATE if case["accumulate"] else 0)
    p = _mmt4d_params(lhs, rhs, out, (m // tile[0], n // tile[1], k // tile[2]), tile, flags)
    return [(lib.iree_uk_mmt4d_p, p)], [out], [lhs, rhs]


def _prepare_chain(lib, case, gen):
    flag, in_t, _, out_t = _TYPES[case["type"]]
    m, n, k = case["m"], case["n"], case["k"]
    m0, n0, k0 = _queried_tile(lib, case["type"])
    tiles = -(-m // m0), -(-n // n0), -(-k // k0)
    activations = _values(gen, m * k, in_t, 1.0, "cuda")
    weights = _values(gen, k * n, in_t, 0.02, "cuda")  # row-major [k][n], packed here once
    lhs = torch.empty(tiles[0] * tiles[2] * m0 * k0, dtype=in_t, device="cuda")
    rhs = torch.empty(tiles[1] * tiles[2] * n0 * k0, dtype=in_t, device="cuda")
    acc = torch.empty(tiles[0] * tiles[1] * m0 * n0, dtype=out_t, device="cuda")
    out = torch.empty(m, n, dtype=out_t, device="cuda")
    pack_flag = _PACK_FLAGS[case["type"]][0]
    pack_rhs = _pack_params(weights, k, n, rhs, k0, n0,
                            pack_flag | abi.PACK_TRANSPOSE_INNER | abi.PACK_TRANSPOSE_OUTER)
    lib.iree_uk_pack_p(C.byref(pack_rhs))
    calls = [
        (lib.iree_uk_pack_p, _pack_params(activations, m, k, lhs, m0, k0, pack_flag)),
        (lib.iree_uk_mmt4d_p, _mmt4d_params(lhs, rhs, acc, tiles, (m0, n0, k0), flag)),
        (lib.iree_uk_unpack_p, _unpack_params(acc, out, m, n, m0, n0,
                                              _UNPACK_FLAGS["s32" if case["type"] == "s8" else "f32"])),
    ]
    return calls, [out], [activations, weights, lhs, rhs, acc]


def _prepare_copy(lib, case, gen):
    rows, cols, t0, t1 = case["rows"], case["cols"], case["t0"], case["t1"]
    pack_flag, dtype = _PACK_FLAGS[case["type"]]
    order = (abi.PACK_TRANSPOSE_INNER if case["inner"] else 0) | (abi.PACK_TRANSPOSE_OUTER if case["outer"] else 0)
    plain = _values(gen, rows * cols, dtype, 1.0, "cuda")
    tiled = torch.empty(_up(rows, t0) * _up(cols, t1), dtype=dtype, device="cuda")
    pack = (lib.iree_uk_pack_p, _pack_params(plain, rows, cols, tiled, t0, t1, pack_flag | order))
    if case["way"] == "pack":
        return [pack], [tiled], [plain]
    back = torch.zeros(rows, cols, dtype=dtype, device="cuda")
    unpack = (lib.iree_uk_unpack_p, _unpack_params(tiled, back, rows, cols, t0, t1, _UNPACK_FLAGS[case["type"]] | order))
    if case["way"] == "both":
        return [pack, unpack], [tiled, back], [plain]
    lib.iree_uk_pack_p(C.byref(pack[1]))
    return [unpack], [back], [plain, tiled]


def prepare(case, seed):
    lib = library.load()
    if lib.iree_uk_mi355x_init(torch.cuda.current_device()) != 0:
        raise RuntimeError("the current device is not a gfx950 part")
    on_host = case["kind"] == "host"
    lib.iree_uk_mi355x_set_stream(torch.cuda.current_stream().cuda_stream, 0 if on_host else 1)
    device = "cpu" if on_host else "cuda"
    gen = torch.Generator(device=device).manual_seed(seed)
    if case["kind"] == "chain":
        calls, outputs, kept = _prepare_chain(lib, case, gen)
    elif case["kind"] == "copy":
        calls, outputs, kept = _prepare_copy(lib, case, gen)
    else:
        calls, outputs, kept = _prepare_product(lib, case, device, gen)
    return {"calls": [(f, C.byref(p)) for f, p in calls], "outputs": outputs, "kept": kept}


def run(state):
    for function, params in state["calls"]:
        function(params)
    return state["outputs"]
