"""The work this framework's speed is judged by: matrix products through the C ABI and through the IR builder, the training
step of a linear layer, fused attention and the row-wise ops of the dialect, each called as a user's program calls it.

A case is a dict of plain values: its `family` and the sizes, element types and options of one call (or of the calls of
one step).  `listed` holds the named ones, `draw` gives more of the same ranges.
"""
import torch

import frisk_amd  # noqa: F401  (puts the builder package on the path)
import frisk as F
from frisk_amd import runtime as R

TORCH = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16, "int8": torch.int8, "e4m3": torch.float8_e4m3fn}


def listed():
    return [
        # the smallest product a program issues on its own: launch and host time are most of it
        gemm("f16_128x128x128_nn", "fp16", 128, 128, 128),
        # fp32 product written with the IR builder and launched by the builder's runtime (the program of the design sketch)
        dict(family="builder", name="builder_f32_1024", dtype="fp32", M=1024, N=1024, K=1024, tile_m=128, tile_n=128, tile_k=32),
        # the ordinary dense product, operands row-major as they come
        gemm("f16_4096_nn", "fp16", 4096, 4096, 4096),
        # W8A8 inference: int8 operands, int32 sums, per-row and per-column scales, fp16 result
        gemm("i8_4096_w8a8", "int8", 4096, 4096, 4096),
        # the largest dense product: a projection with its weights stored [N][K]
        gemm("bf16_8192_nt", "bf16", 8192, 8192, 8192, transB=True),
        # decoding: a batch of 32 token rows against 8-bit weights streamed from memory
        gemm("e4m3_decode_32x8192x8192_nt", "e4m3", 32, 8192, 8192, transB=True),
        # decoding with 16-bit weights stored [K][N] and a row count that fills no tile
        gemm("f16_decode_48x8192x8192_nn", "fp16", 48, 8192, 8192),
        # a K that is no multiple of any K tile, everything else in order
        gemm("f16_ragged_4096x4096x4000_nn", "fp16", 4096, 4096, 4000),
        # nothing in order: every size odd, so that no row but the first starts on a 16-byte boundary
        gemm("f16_odd_1999x4099x3001_nn", "fp16", 1999, 4099, 3001),
        # forward and backward of a linear layer over a packed batch of 3000 tokens
        dict(family="linear", name="bf16_linear_step_3000x4096x11008", dtype="bf16", tokens=3000, n_in=4096, n_out=11008),
        # attention of one long sequence, 32 heads
        attention("attention_f16_1x32x4096x4096", "fp16", 1, 32, 4096, 4096),
        # row-wise ops on activations: cast, mean, scale and shift, softmax
        dict(family="rows", name="row_ops_f16_8192x8192", dtype="fp16", rows=8192, cols=8192),
    ]


def gemm(name, dtype, M, N, K, transA=False, transB=False, pad=False):
    """`pad`: the rows of all three matrices are padded to a multiple of 16 bytes"""
    return dict(family="gemm", name=name, dtype=dtype, M=M, N=N, K=K, transA=transA, transB=transB, pad=pad)


def attention(name, dtype, batch, heads, seq_q, seq_k, k_transposed=False):
    return dict(family="attention", name=name, dtype=dtype, batch=batch, heads=heads, seq_q=seq_q, seq_k=seq_k, k_transposed=k_transposed)


def between(rng, lo, hi, step=1):
    """a multiple of `step` in [lo, hi], spread over the logarithm"""
    x = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(x / step)) * step))


def draw(rng):
    kind = rng.choice(["small", "builder", "dense", "dense", "dense", "decode", "decode", "ragged", "ragged", "linear", "attention", "attention", "rows"])
    if kind == "small":
        c = gemm("", rng.choice(["fp16", "bf16", "fp32"]), between(rng, 16, 512), between(rng, 16, 512), between(rng, 16, 512), rng.random() < 0.3, rng.random() < 0.5)
    elif kind == "builder":
        tile = dict(tile_m=128, tile_n=128, tile_k=32)
        c = dict(family="builder", dtype=rng.choice(["fp32", "fp16"]), M=between(rng, 128, 2048, 128), N=between(rng, 128, 2048, 128), K=between(rng, 128, 2048, 128), **tile)
    elif kind == "dense":
        # weights [K][N] or [N][K]; A stored [K][M] as in a weight gradient
        c = gemm("", rng.choice(["fp16", "bf16", "int8", "e4m3"]), between(rng, 512, 8192, 64), between(rng, 512, 8192, 64), between(rng, 512, 8192, 128),
                 rng.random() < 0.25, rng.random() < 0.5)
    elif kind == "decode":
        c = gemm("", rng.choice(["fp16", "bf16", "int8", "e4m3"]), between(rng, 1, 64), between(rng, 2048, 16384, 64), between(rng, 2048, 8192, 128), False, rng.random() < 0.6)
    elif kind == "ragged":
        c = gemm("", rng.choice(["fp16", "bf16", "int8", "e4m3"]), between(rng, 512, 4096), between(rng, 512, 4096), between(rng, 512, 4096), rng.random() < 0.25,
                 rng.random() < 0.5, rng.random() < 0.5)
    elif kind == "linear":
        c = dict(family="linear", dtype=rng.choice(["bf16", "fp16"]), tokens=between(rng, 256, 3000), n_in=between(rng, 1024, 4096, 64), n_out=between(rng, 1024, 11008, 64))
    elif kind == "attention":
        c = attention("", rng.choice(["fp16", "bf16"]), rng.choice([1, 1, 2, 4]), rng.choice([8, 16, 32]), between(rng, 256, 4096, 256), between(rng, 256, 4096, 64), rng.random() < 0.25)
        while c["batch"] * c["heads"] * c["seq_q"] * c["seq_k"] > 32 * 4096 * 4096:
            c["batch"] //= 2
    else:
        c = dict(family="rows", dtype=rng.choice(["fp16", "bf16", "fp32"]), rows=between(rng, 64, 16384), cols=between(rng, 128, 16384))
        c["rows"] = min(c["rows"], 8192 * 8192 // c["cols"])
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ preparation
class State:
    """what a program has in hand before the call: operands, outputs, descriptors, workspaces"""


def rounded(n, dtype, pad):
    per = 16 // torch.empty(0, dtype=TORCH[dtype]).element_size()
    return (n + per - 1) // per * per if pad else n


def operand(g, dtype, rows, ld, scale):
    """`rows` rows of `ld` elements, N(0,1) * scale (int8: uniform; e4m3: spread over its range)"""
    if dtype == "int8":
        return torch.randint(-127, 128, (rows, ld), device="cuda", dtype=torch.int8, generator=g)
    x = torch.randn(rows, ld, device="cuda", generator=g)
    if dtype == "e4m3":
        return (x * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (x * scale).to(TORCH[dtype])


def workspace(nbytes):
    return torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda"), nbytes


class Product:
    """one matrix product: descriptor, output and workspace, laid out once"""

    def __init__(self, dtype, M, N, K, A, B, out, transA=False, transB=False, lda=None, ldb=None, clear=True, scales=None, epilogue=R.EPI_NONE):
        self.A, self.B, self.C, self.scales = A, B, out, scales
        codes = {torch.float32: R.F32, torch.float16: R.F16, torch.bfloat16: R.BF16}
        self.desc = R.make_desc(R.DTYPE_NAMES[dtype], M, N, K, dtype_out=codes[out.dtype], transA=transA, transB=transB, lda=lda, ldb=ldb, ldc=out.shape[1], clear_accum=clear,
                                epilogue=epilogue)
        self.ws, self.ws_bytes = workspace(R.workspace_bytes(self.desc))

    def __call__(self, stream):
        sa, sb = (None, None) if self.scales is None else (self.scales[0].data_ptr(), self.scales[1].data_ptr())
        R.gemm(self.desc, self.A.data_ptr(), self.B.data_ptr(), self.C.data_ptr(), sa, sb, self.ws.data_ptr(), self.ws_bytes, stream)


def prepare_gemm(case, g, s):
    dt, M, N, K, ta, tb, pad = (case[k] for k in ("dtype", "M", "N", "K", "transA", "transB", "pad"))
    lda, ldb = rounded(M if ta else K, dt, pad), rounded(K if tb else N, dt, pad)
    A = operand(g, dt, K if ta else M, lda, K ** -0.5)
    B = operand(g, dt, N if tb else K, ldb, 1.0)
    out_dtype = {"int8": "fp16", "e4m3": "bf16"}.get(dt, dt)
    C = torch.zeros(M, rounded(N, out_dtype, pad), device="cuda", dtype=TORCH[out_dtype])
    scales, epilogue = None, R.EPI_NONE
    if dt == "int8":
        scales, epilogue = [torch.rand(n, device="cuda", generator=g) * 0.019 + 0.001 for n in (M, N)], R.EPI_ROW_COL_SCALE
    elif dt == "e4m3":
        scales, epilogue = [torch.rand(1, device="cuda", generator=g) * 0.01 + 0.005 for _ in range(2)], R.EPI_TENSOR_SCALE
    s.product = Product(dt, M, N, K, A, B, C, ta, tb, lda, ldb, scales=scales, epilogue=epilogue)


def prepare_builder(case, g, s):
    M, N, K, dt = case["M"], case["N"], case["K"], case["dtype"]
    s.session = F.create_session()
    s.kernel = s.session.tiled_gemm("matmul", M, N, K, dt, tile=(case["tile_m"], case["tile_n"], case["tile_k"]), threads=256)
    scale = 1.0 if dt == "fp32" else K ** -0.5
    s.A = ((torch.rand(M, K, device="cuda", generator=g) * 2 - 1) * scale).to(TORCH[dt])
    s.B = (torch.rand(K, N, device="cuda", generator=g) * 2 - 1).to(TORCH[dt])
    s.C = torch.zeros(M, N, device="cuda", dtype=TORCH[dt])


def prepare_linear(case, g, s):
    dt, T, n_in, n_out = case["dtype"], case["tokens"], case["n_in"], case["n_out"]
    X = operand(g, dt, T, n_in, 1.0)
    W = operand(g, dt, n_out, n_in, n_in ** -0.5)
    dY = operand(g, dt, T, n_out, T ** -0.5)
    s.dY, s.code, s.T, s.n_in, s.n_out = dY, R.DTYPE_NAMES[dt], T, n_in, n_out
    s.Y, s.dX = (torch.zeros(T, n, device="cuda", dtype=TORCH[dt]) for n in (n_out, n_in))
    s.dW = torch.zeros(n_out, n_in, device="cuda")
    s.db = torch.zeros(n_out, device="cuda", dtype=TORCH[dt])
    s.forward = Product(dt, T, n_out, n_in, X, W, s.Y, transB=True)
    s.input_gradient = Product(dt, T, n_in, n_out, dY, W, s.dX)
    s.weight_gradient = Product(dt, n_out, n_in, T, dY, X, s.dW, transA=True, clear=False)
    s.ws, s.ws_bytes = workspace(R.reduce_workspace_bytes(s.code, T, n_out, 0))


def prepare_attention(case, g, s):
    b, h, sq, sk = (case[k] for k in ("batch", "heads", "seq_q", "seq_k"))
    dt = TORCH[case["dtype"]]
    s.desc = R.make_attention_desc(R.DTYPE_NAMES[case["dtype"]], b, h, sq, sk, 128, k_transposed=case["k_transposed"])
    s.Q, s.K, s.V = (torch.randn(b * h, n, 128, device="cuda", generator=g).to(dt) for n in (sq, sk, sk))
    if case["k_transposed"]:
        s.K = s.K.transpose(1, 2).contiguous()
    s.O = torch.zeros(b, h, sq, 128, device="cuda", dtype=dt)
    s.lse = torch.zeros(b, h, sq, device="cuda")


def prepare_rows(case, g, s):
    rows, cols, dt = case["rows"], case["cols"], TORCH[case["dtype"]]
    s.code, s.rows, s.cols = R.DTYPE_NAMES[case["dtype"]], rows, cols
    s.src = torch.randn(rows, cols, device="cuda", generator=g) + 0.5
    s.x, s.y, s.p = (torch.zeros(rows, cols, device="cuda", dtype=dt) for _ in range(3))
    s.sums = torch.zeros(rows, device="cuda", dtype=dt)
    s.gain = (torch.rand(cols, device="cuda", generator=g) + 0.5).to(dt)
    s.shift = torch.randn(cols, device="cuda", generator=g).to(dt)
    # y = (x - sum / cols) * gain + shift: a per-row operand and two per-column ones beside x
    program = [("input", 0), ("input", 1), ("const", 1.0 / cols), "mul", "sub", ("input", 2), "mul", ("input", 3), "add"]
    s.block = R.make_elementwise_desc(program, [(s.code, cols, 1), (s.code, 1, 0), (s.code, 0, 1), (s.code, 0, 1)], s.code, rows, cols)
    s.ws, s.ws_bytes = workspace(R.reduce_workspace_bytes(s.code, rows, cols, 1))
    s.ws2, s.ws2_bytes = workspace(R.softmax_workspace_bytes(s.code, rows, cols))


PREPARE = {"gemm": prepare_gemm, "builder": prepare_builder, "linear": prepare_linear, "attention": prepare_attention, "rows": prepare_rows}


def prepare(case, seed):
    s = State()
    s.family = case["family"]
    PREPARE[s.family](case, torch.Generator(device="cuda").manual_seed(seed), s)
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    stream = torch.cuda.current_stream().cuda_stream
    if s.family == "gemm":
        s.product(stream)
        return s.product.C
    if s.family == "builder":
        F.runtime.launch(s.kernel, [s.A.data_ptr(), s.B.data_ptr(), s.C.data_ptr()], stream)
        return s.C
    if s.family == "linear":
        R.fill(R.F32, s.dW.data_ptr(), s.n_out, s.n_in, s.n_in, 0.0, stream)  # zero the gradient, then accumulate into it
        s.forward(stream)
        s.input_gradient(stream)
        s.weight_gradient(stream)
        R.reduce(s.code, s.dY.data_ptr(), s.T, s.n_out, s.n_out, 0, "add", True, s.db.data_ptr(), s.ws.data_ptr(), s.ws_bytes, stream)
        return {"y": s.Y, "dx": s.dX, "dw": s.dW, "db": s.db}
    if s.family == "attention":
        R.attention(s.desc, s.Q.data_ptr(), s.K.data_ptr(), s.V.data_ptr(), s.O.data_ptr(), s.lse.data_ptr(), stream)
        return {"out": s.O, "lse": s.lse}
    R.copy(R.F32, s.src.data_ptr(), s.cols, s.code, s.x.data_ptr(), s.cols, s.rows, s.cols, stream)
    R.reduce(s.code, s.x.data_ptr(), s.rows, s.cols, s.cols, 1, "add", True, s.sums.data_ptr(), s.ws.data_ptr(), s.ws_bytes, stream)
    R.elementwise(s.block, [s.x.data_ptr(), s.sums.data_ptr(), s.gain.data_ptr(), s.shift.data_ptr()], s.y.data_ptr(), stream)
    R.softmax(s.code, s.y.data_ptr(), s.cols, s.p.data_ptr(), s.cols, s.rows, s.cols, stream=stream, workspace_ptr=s.ws2.data_ptr(), workspace_bytes=s.ws2_bytes)
    return {"x": s.x, "sums": s.sums, "y": s.y, "p": s.p}


# ------------------------------------------------------------------ what a pass cannot do without, and how exact it is
SIZE = {"fp32": 4, "fp16": 2, "bf16": 2, "int8": 1, "e4m3": 1}


def work(case):
    es = SIZE[case["dtype"]]
    if case["family"] in ("gemm", "builder"):
        M, N, K = case["M"], case["N"], case["K"]
        scales = {"int8": 4 * (M + N), "e4m3": 8}.get(case["dtype"], 0)
        return {"bytes": (M * K + K * N) * es + M * N * (2 if es == 1 else es) + scales, "flops": 2 * M * N * K}
    if case["family"] == "linear":
        T, i, o = case["tokens"], case["n_in"], case["n_out"]
        # X, W and dY read, Y, dX, dW and db written
        return {"bytes": (T * i + o * i + T * o) * es + (T * o + T * i + o) * es + o * i * 4, "flops": 3 * 2 * T * i * o + T * o}
    if case["family"] == "attention":
        bh, sq, sk = case["batch"] * case["heads"], case["seq_q"], case["seq_k"]
        return {"bytes": bh * (2 * sq + 2 * sk) * 128 * es + bh * sq * 4, "flops": 4 * bh * sq * sk * 128}
    n, r, c = case["rows"] * case["cols"], case["rows"], case["cols"]
    return {"bytes": n * 4 + 3 * n * es + (r + 2 * c) * es, "flops": 10 * n}


def tolerance(case):
    # four times or so what the outputs measure against the same step in 64 bits, relative: fp16 2.1e-4 (attention 2.9e-4), bf16 1.7e-3 (one
    # rounding to the output type after fp32 sums), fp32 products at most 6e-7 (K = 1024; twice that leaves room for the order of a longer sum)
    dt = case["dtype"]
    if case["family"] == "gemm" and dt == "int8":
        return "exact"
    if dt == "fp32":
        return {"rel": 5e-6}
    return {"rel": 1e-3 if dt == "fp16" else 7e-3}
