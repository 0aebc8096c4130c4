"""Which kernel a call is given, on the CPU: the library over the stand-in runtime of fake_hip.cpp, which says what was launched."""
import pytest

import test_k_order as k_order
import test_large_tiles as large
from test_f32_tiles import ODD_SIZES, SIZES, SMALLEST
from test_host_copies import fake_hip  # noqa: F401 - a fixture

BF16 = 1

LAUNCHED = """
import importlib
lang, nn = cg.lang, cg.nn
fake.fake_hip_launched.restype = fake.fake_hip_products.restype = ctypes.c_char_p

def launched(f):
    be.sync()
    fake.fake_hip_launched()
    be.realize(f())
    be.sync()
    return [n for n in fake.fake_hip_launched().decode().split("\\n") if "gem" in n]

def operand(*shape):
    n = int(np.prod(shape))
    if int(sys.argv[2]):
        return be.from_bf16_bits(np.zeros(n, np.uint16), shape)
    return be.tensor(np.zeros(n, np.float32).reshape(shape))

def product(m, n, k, along_k=True, batch=1, residual=False):
    lead, r = ((), 2) if batch == 1 else ((batch,), 3)
    x, w = operand(*lead, m, k), operand(*lead, *((n, k) if along_k else (k, n)))
    res = be.reshape(be.tensor(np.zeros(batch * m * n, np.float32)), lead + (m, n)) if residual else None
    def f():
        y = be.matmul(x, be.transpose(w, r - 2, r - 1) if along_k else w)
        return be.add(res, y) if residual else y
    return launched(f)

class Term(lang.Module):
    def __init__(self, n_in, f): self.n_in, self.f = n_in, f
    def path(self): return lang.path(["choice"])
    def sort(self): return [lang.TENSOR] * self.n_in, [lang.TENSOR]
    def def_(self, b, args): return [self.f(b, *args)]

def run(f, *args):
    return cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Term(len(args), f).term(), list(args))[0]

def linear(b, x, w, n, k):
    return lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, k, n), lang.transpose(b, 0, 1, w)))
"""


def test_no_kernel_with_fixed_places_in_lds_beside_variables_of_its_own(fake_hip):  # noqa: F811
    fake_hip(LAUNCHED + """
fake.fake_hip_static_lds(64)
assert fails(lambda: product(4096, 4096, 384))
fake.fake_hip_static_lds(0)
assert ["gemm_bf16_ring" in n for n in product(4096, 4096, 384)] == [True]
""", BF16)


def test_products_on_256_x_256_tiles(fake_hip):  # noqa: F811
    """The sizes that test_large_tiles.py gives its edges, and batches: eight wavefronts for few k-steps, four beyond and for a residual."""
    fake_hip(LAUNCHED + """
four, eight = "gemm_bf16_ring_kernelILi0ELi2E", "gemm_bf16_dma_kernelILi256ELi256ELi2ELi4ELb0ELi2E"
for m, n, k, kernel in ((4096, 4096, 128, eight), (4090, 4093, 192, eight), (3841, 3843, 256, eight), (8001, 2046, 320, eight), (255, 65299, 448, four),
                        (4096, 4093, 384, four), (8192, 4096, 512, eight), (8192, 4096, 576, four), (4096, 8192, 512, four), (8192, 2048, 512, four)):
    names = product(m, n, k)
    assert len(names) == 1 and kernel in names[0], (m, n, k, names)
for b, m, n, k in ((1, 3841, 3843, 128), (1, 4090, 4093, 192), (1, 8001, 2046, 256), (16, 1000, 1002, 128)):
    for residual in (False, True):
        names = product(m, n, k, batch=b, residual=residual)
        assert len(names) == 1 and (four if residual else eight) in names[0], (b, m, n, k, names)
""", BF16)


def test_a_round_of_192_rows(fake_hip):  # noqa: F811
    """Four wavefronts from ten k-steps on, eight below."""
    fake_hip(LAUNCHED + """
for m, n, k, waves in ((2305, 2049, 64, 8), (6000, 700, 256, 8), (2303, 2049, 576, 8), (2303, 2049, 640, 4), (2305, 2048, 2048, 4)):
    for residual in (False, True):
        names = product(m, n, k, residual=residual)
        assert len(names) == 1 and "gemm_bf16_dma_kernelILi192ELi128ELi2ELi%dELb0E" % (waves // 2) in names[0], (m, n, k, names)
        assert names[0].endswith("ELb%dEEEvNS_8GemmDescE" % residual), names
""", BF16)


def test_gated_products(fake_hip):  # noqa: F811
    """gate and up stacked: one and two k-steps on eight wavefronts unless whole rounds of 256 rows are ahead, four wavefronts beyond."""
    fake_hip(LAUNCHED + """
class Gated(lang.Module):
    def __init__(self, m, f, k): self.m, self.f, self.k = m, f, k
    def path(self): return lang.path(["gated", "%d" % self.m, "%d" % self.f, "%d" % self.k])
    def sort(self): return [lang.TENSOR] * 4, [lang.TENSOR]
    def def_(self, b, args):
        def linear(x, w, n, k): return lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, k, n), lang.transpose(b, 0, 1, w)))
        x, g, u, d = args
        return [linear(nn.silu(b, linear(x, g, self.f, self.k)) * linear(x, u, self.f, self.k), d, 64, self.f)]

wide, tall, four, four128 = ("gemm_bf16_dma_kernelILi128ELi256ELi2ELi4ELb1ELi3ELb1E", "gemm_bf16_dma_kernelILi256ELi256ELi2ELi4ELb1ELi2ELb1E",
                             "gemm_bf16_ring_kernelILi2ELi2E", "gemm_bf16_ring_kernelILi2ELi1E")
for m, f, k, kernel in ((4100, 2056, 64, tall), (4200, 2600, 128, tall), (4100, 1256, 128, four), (4200, 2600, 192, four128),
                        (1000, 3000, 64, wide), (1030, 2184, 128, wide), (1030, 2184, 192, four128)):
    xs = [operand(1, m, k), operand(f, k), operand(f, k), operand(64, f)]
    be.sync()
    fake.fake_hip_launched()
    be.realize(cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Gated(m, f, k).term(), xs)[0])
    be.sync()
    names = [n for n in fake.fake_hip_launched().decode().split("\\n") if "gem" in n]
    assert kernel in names[0], (m, f, k, names)
""", BF16)


def test_less_than_a_round(fake_hip):  # noqa: F811
    """A quarter of a 128 x 128 tile from four k-steps on, half of one below or where the quarters are more than the CUs."""
    fake_hip(LAUNCHED + """
for m, n, k, tile in ((140, 700, 192, "Li128ELi64E"), (300, 300, 256, "Li64ELi64E"), (900, 700, 64, "Li128ELi64E"), (1200, 700, 256, "Li64ELi64E"),
                      (1000, 1100, 256, "Li128ELi64E")):
    for residual in (False, True):
        names = product(m, n, k, residual=residual)
        assert len(names) == 1 and "gemm_bf16_dma_kernelI" + tile in names[0], (m, n, k, names)
""", BF16)


def test_one_column(fake_hip):  # noqa: F811
    """A wave to a row unless few k of very many rows, or of one tile's worth, are quicker on 64 x 64 tiles."""
    fake_hip(LAUNCHED + """
for b, m, k, column in ((1, 17, 72, 0), (1, 17, 160, 1), (1, 65, 72, 1), (1, 6000, 64, 1), (1, 6001, 176, 0), (1, 6001, 192, 1), (1, 16384, 504, 0),
                        (1, 16384, 512, 1), (1, 70000, 1016, 0), (1, 70000, 1024, 1), (100, 66, 192, 0), (20, 66, 64, 1)):
    names = product(m, 1, k, batch=b)
    assert len(names) == 1 and ("gemm_bf16_column" if column else "gemm_bf16_nt_kernelILi64ELi64E") in names[0], (b, m, k, names)
""", BF16)


def test_one_column_and_a_sigmoid(fake_hip):  # noqa: F811
    """In the column kernel's launch, and a launch of its own behind the tiles, which have none, from either order of the column."""
    fake_hip(LAUNCHED + """
class Sigmoid(lang.Module):
    def __init__(self, along_k): self.along_k = along_k
    def path(self): return lang.path(["sigmoid", str(self.along_k)])
    def sort(self): return [lang.TENSOR] * 2, [lang.TENSOR]
    def def_(self, b, args): return [nn.sigmoid(b, lang.matmul(b, args[0], lang.transpose(b, 0, 1, args[1]) if self.along_k else args[1]))]

for m, k, column in ((17, 72, 0), (17, 160, 1), (65, 72, 1), (6001, 176, 0), (6001, 192, 1)):
    for along_k in (True, False):
        x, w = operand(m, k), operand(*((1, k) if along_k else (k, 1)))
        be.sync()
        fake.fake_hip_launched()
        be.realize(cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Sigmoid(along_k).term(), [x, w])[0])
        be.sync()
        names = [n for n in fake.fake_hip_launched().decode().split("\\n") if "gem" in n or "ew_" in n]
        assert len(names) == 2 - column and ("gemm_bf16_column" if column else "gemm_bf16_nt_kernelILi64ELi64E") in names[0], (m, k, along_k, names)
""", BF16)


def test_less_than_64_columns(fake_hip):  # noqa: F811
    """32 x 32 tiles of the whole of k, or 64 x 64 ones through registers and, deep, in slices."""
    fake_hip(LAUNCHED + """
direct, registers = "gemm_bf16_dma_kernelILi32ELi32E", "gemm_bf16_nt_kernelILi64ELi64E"
for b, m, n, k, kernel in ((1, 17, 60, 256, registers), (1, 17, 60, 320, direct), (1, 65, 33, 384, registers), (1, 65, 33, 448, direct),
                                     (1, 512, 60, 256, registers), (1, 512, 60, 320, direct), (1, 4096, 60, 320, direct), (1, 4097, 60, 384, registers),
                                     (1, 8192, 60, 448, direct), (1, 8193, 60, 512, registers), (3, 4096, 60, 512, registers), (1, 512, 60, 3072, direct), (1, 512, 60, 3136, registers), (1, 513, 60, 3584, direct),
                                     (1, 1024, 60, 4096, registers), (1, 1023, 63, 4096, direct), (1, 3072, 60, 4096, direct), (1, 200, 60, 4160, registers)):
    for residual in (False, True):      # (32 x 32 tiles add it as they are stored)
        names = product(m, n, k, batch=b, residual=residual)
        assert len(names) == 1 and kernel in names[0], (b, m, n, k, names)
        assert kernel != direct or names[0].endswith("ELb%dEEEvNS_8GemmDescE" % residual), names
""", BF16)


def test_f32_tiles(fake_hip):  # noqa: F811
    """Every height of tile, with both layouts of the right operand, for the sizes of test_f32_tiles.py; 32 x 32 tiles where these are ahead."""
    fake_hip(LAUNCHED + f"""
for rows, b, m, n, k in {SIZES}:
    for along_k in (True, False):
        names = product(m, n, k, along_k, b)
        assert len(names) == 1 and "gemm_f32_dma_kernelILi%dE" % rows in names[0] and names[0].split("ELb")[1][0] == "10"[along_k], (b, m, n, k, along_k, names)
for b, m, n, k in ((1, 64, 256, 128), (1, 33, 132, 1044), (3, 70, 260, 100), (1, 10, 512, 2048), (1, 2000, 20, 2000), (1, 4455, 18, 2700), (1, 4191, 23, 2860), (3, 1355, 11, 2792), (5, 469, 20, 3576)):
    names = product(m, n, k, batch=b)
    assert len(names) == 1 and "gemm_small_f32_kernel" in names[0], (b, m, n, k, names)
for b, m, n, k in {SMALLEST}:
    for along_k in (True, False):
        names = product(m, n, k, along_k, b)
        assert len(names) == 1 and "gemm_small_f32_kernel_16" in names[0], (b, m, n, k, names)
for b, m, n, k in ((1, 33, 132, 1044), (1, 10, 512, 2048), (1, 2000, 40, 256)):     # (deep; more tiles than CUs)
    names = product(m, n, k, batch=b)
    assert len(names) == 1 and "gemm_small_f32_kernelI" in names[0], (b, m, n, k, names)
for b, m, n, k in ((1, 4129, 24, 3200), (1, 4129, 40, 3200), (3, 326, 17, 7488)):     # (deeper, of more columns, of four slices)
    names = product(m, n, k, batch=b)
    assert len(names) == 1 and "gemm_f32_dma_kernel" in names[0], (b, m, n, k, names)
""")


def test_attention_with_heads_of_128(fake_hip):  # noqa: F811
    """Two wavefronts to 32 queries up to one workgroup of 128 queries a CU, with a mask and without; one beyond."""
    fake_hip("""
import importlib
lang, nn = cg.lang, cg.nn
helpers = importlib.import_module("catgrad-rs_amd.llm.helpers")
fake.fake_hip_launched.restype = ctypes.c_char_p

class Attention(lang.Module):
    def __init__(self, shape, causal): self.shape, self.causal = shape, causal
    def path(self): return lang.path(["attention", str(self.causal)])
    def sort(self): return [lang.TENSOR] * 3, [lang.TENSOR]
    def def_(self, b, args):
        q, k, v = (lang.reshape(b, lang.make_shape(b, *self.shape), x) for x in args)
        q, k, v = q + q - q, helpers.repeat_kv(b, 1, k + k - k), helpers.repeat_kv(b, 1, v + v - v)
        s = lang.matmul(b, q, lang.transpose(b, 2, 3, k))
        sh = lang.shape(b, s)
        s = s / lang.constant(b, 11.0, sh)
        if self.causal: s = s + lang.broadcast(b, helpers.causal_mask(b, lang.to_nat(b, self.shape[2])), sh)
        return [lang.matmul(b, nn.softmax(b, s), v)]

for shape, wide in (((1, 16, 2048, 128), 1), ((1, 16, 2049, 128), 0), ((4, 16, 512, 128), 1), ((2, 16, 1100, 128), 0)):
    for causal in (False, True):
        q, k, v = (be.tensor(np.zeros(int(np.prod(shape)), np.float32)) for _ in range(3))
        be.sync()
        fake.fake_hip_launched()
        be.realize(cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Attention(shape, causal).term(), [q, k, v])[0])
        be.sync()
        names = [n for n in fake.fake_hip_launched().decode().split("\\n") if "attn_prefill" in n]
        assert len(names) == 1 and "attn_prefill_kernelILi128ELi64ELi4ELi1ELi%dE" % (wide + 1) in names[0], (shape, causal, names)
""", BF16)


def test_attention_over_one_step_of_keys(fake_hip):  # noqa: F811
    """Heads of 64: a wavefront to a tile up to 64 keys, with a mask and without; the keys of four beyond, and where tiles of 64 queries fill the CUs."""
    fake_hip("""
import importlib
lang, nn = cg.lang, cg.nn
helpers = importlib.import_module("catgrad-rs_amd.llm.helpers")
fake.fake_hip_launched.restype = ctypes.c_char_p

class Attention(lang.Module):
    def __init__(self, shape, causal): self.shape, self.causal = shape, causal
    def path(self): return lang.path(["attention", str(self.causal)])
    def sort(self): return [lang.TENSOR] * 3, [lang.TENSOR]
    def def_(self, b, args):
        q, k, v = (lang.reshape(b, lang.make_shape(b, *self.shape), x) for x in args)
        q, k, v = q + q - q, helpers.repeat_kv(b, 1, k + k - k), helpers.repeat_kv(b, 1, v + v - v)
        s = lang.matmul(b, q, lang.transpose(b, 2, 3, k))
        sh = lang.shape(b, s)
        s = s / lang.constant(b, 11.0, sh)
        if self.causal: s = s + lang.broadcast(b, helpers.causal_mask(b, lang.to_nat(b, self.shape[2])), sh)
        return [lang.matmul(b, nn.softmax(b, s), v)]

for shape, kernel in (((1, 32, 37, 64), "keysplit_kernelILi64ELi64ELi1E"), ((1, 32, 64, 64), "keysplit_kernelILi64ELi64ELi1E"),
                      ((1, 32, 65, 64), "keysplit_kernelILi64ELi64ELi4E"), ((20, 32, 64, 64), "attn_prefill_kernelILi64E")):
    for causal in (False, True):
        q, k, v = (be.tensor(np.zeros(int(np.prod(shape)), np.float32)) for _ in range(3))
        be.sync()
        fake.fake_hip_launched()
        be.realize(cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Attention(shape, causal).term(), [q, k, v])[0])
        be.sync()
        names = [n for n in fake.fake_hip_launched().decode().split("\\n") if "attn_prefill" in n]
        assert len(names) == 1 and kernel in names[0], (shape, causal, names)
""", BF16)


def test_masks_that_are_read_as_they_are(fake_hip):  # noqa: F811
    """Rows of a multiple of four keys are copied to longer ones for the kernel of one step alone; others always."""
    fake_hip("""
import importlib
lang, nn = cg.lang, cg.nn
helpers = importlib.import_module("catgrad-rs_amd.llm.helpers")
fake.fake_hip_launched.restype = ctypes.c_char_p

class Attention(lang.Module):
    def __init__(self, shape): self.shape = shape
    def path(self): return lang.path(["attention"])
    def sort(self): return [lang.TENSOR] * 3, [lang.TENSOR]
    def def_(self, b, args):
        q, k, v = (lang.reshape(b, lang.make_shape(b, *self.shape), x) for x in args)
        q, k, v = q + q - q, helpers.repeat_kv(b, 1, k + k - k), helpers.repeat_kv(b, 1, v + v - v)
        s = lang.matmul(b, q, lang.transpose(b, 2, 3, k))
        sh = lang.shape(b, s)
        s = s / lang.constant(b, 11.0, sh) + lang.broadcast(b, helpers.causal_mask(b, lang.to_nat(b, self.shape[2])), sh)
        return [lang.matmul(b, nn.softmax(b, s), v)]

for shape, padded in (((1, 32, 36, 64), 1), ((1, 32, 64, 64), 0), ((1, 32, 68, 64), 0), ((1, 32, 70, 64), 1), ((20, 32, 60, 64), 0),
                      ((1, 16, 36, 128), 0), ((1, 16, 37, 128), 1), ((1, 4, 60, 256), 0), ((1, 4, 61, 256), 1), ((4, 16, 32, 128), 0)):
    q, k, v = (be.tensor(np.zeros(int(np.prod(shape)), np.float32)) for _ in range(3))
    be.sync()
    fake.fake_hip_launched()
    be.realize(cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Attention(shape).term(), [q, k, v])[0])
    be.sync()
    names = fake.fake_hip_launched().decode().split("\\n")
    assert sum("attn_prefill" in n for n in names) == 1 and sum("mask_pad" in n for n in names) == padded, (shape, names)
""", BF16)


def test_sum_of_two_slots_of_the_same_experts(fake_hip):  # noqa: F811
    """The launch that realises one addend of `y0 + y1` makes the other as well: nothing is left of the product to add to."""
    fake_hip("""
import importlib
lang, nn, vectors = cg.lang, cg.nn, importlib.import_module("tests.vectors")

def total(b, x, idx, wg, wu, wd):
    def slot(i):
        of = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, lang.get(b, 1, i, idx), w))
        return lang.matmul(b, nn.silu(b, lang.matmul(b, x, of(wg))) * lang.matmul(b, x, of(wu)), of(wd))
    return slot(0) + slot(1)
for s in (1, 5, 20, 200):
    up = np.zeros((3, 192, 128), np.float32)
    (got,) = vectors.run(be, total, 1, np.zeros((s, 1, 128), np.float32), np.zeros((s, 2), np.uint32), up, up + 1, np.zeros((3, 128, 192), np.float32))
    assert got.shape == (s, 1, 128)
""", BF16)


def test_f32_tiles_of_odd_heights(fake_hip):  # noqa: F811
    """16 rows more than a multiple of 32 for up to 512 rows; none beyond, nor for few k."""
    fake_hip(LAUNCHED + f"""
for rows, b, m, n, k in {ODD_SIZES}:
    for along_k in (True, False):
        (name,) = [x for x in product(m, n, k, along_k, b) if "gemm" in x and "splitk" not in x]
        assert "gemm_f32_dma_kernelILi%dE" % rows in name and name.endswith("ELb%dELb1EEEvNS_8GemmDescE" % (not along_k)), (b, m, n, k, along_k, name)
for b, m, n, k in ((1, 700, 2048, 8192), (1, 1000, 8192, 2048), (1, 130, 7312, 52), (1, 220, 30000, 100)):
    assert all(x.endswith("ELb0EEEvNS_8GemmDescE") for x in product(m, n, k) if "dma" in x)
""")


def test_tiles_of_128_x_256(fake_hip):  # noqa: F811
    """One round of them where 128 x 128 are two to a CU and 192 rows more than a round, from 16 k-steps on; the sizes of test_large_tiles.py."""
    fake_hip(LAUNCHED + """
for m, n, k, half in ((3100, 2050, 1024, True), (3333, 2049, 1088, True), (2300, 3001, 2048, True), (1000, 6143, 1152, True), (4096, 2048, 4160, True),
                      (3100, 2050, 960, False), (2900, 2048, 2048, False), (4100, 2050, 2048, False)):
    for residual in (False, True):
        names = product(m, n, k, residual=residual)
        assert len(names) == 1 and ("gemm_bf16_ring_kernelILi0ELi1E" in names[0]) == half, (m, n, k, names)
""", BF16)


def test_where_column_tiles_start_at_different_k(fake_hip):  # noqa: F811
    """The lists of test_k_order.py: kernel, slices of k, and the order as the kernel is told of it."""
    fake_hip(LAUNCHED + f"""
def products(f, *args):     # (kernel, slices, values to a slice, order)
    be.sync()
    fake.fake_hip_products()
    be.realize(run(f, *args))
    be.sync()
    lines = [line.rsplit(" ", 3) for line in fake.fake_hip_products().decode().splitlines()]
    return [(name, int(s), int(k), int(o)) for name, s, k, o in lines if "route" not in name]

def check(what, got, kernel, slices, on):
    assert (kernel % 0 if "%d" in kernel else kernel) in got[0] and got[1] == slices and got[3] == on, (what, got)

for on, sizes in ((1, {k_order.PRODUCTS}), (0, {k_order.OTHER_PRODUCTS})):
    for m, n, k, kernel, slices in sizes:
        (got,) = products(lambda b, x, w: linear(b, x, w, n, k), operand(1, m, k), operand(n, k))
        check((m, n, k), got, kernel, slices, on)
for on, sizes in ((1, {k_order.PARTS_OF_ROWS}), (0, {k_order.OTHER_PARTS_OF_ROWS})):
    for m, n, k, apart, kernel, slices in sizes:
        (got,) = products(lambda b, x, w: linear(b, x, lang.slice(b, 1, 64, k, w), n, k), operand(1, m, k), operand(n, apart))
        check((m, n, k, apart), got, kernel, slices, on)
        assert got[2] // 64 % 2 == 1 or not on, got
for m, n, k, kernel in {k_order.SIGMOIDS}:
    (got,) = products(lambda b, x, w: nn.sigmoid(b, linear(b, x, w, n, k)), operand(1, m, k), operand(n, k))
    check((m, n, k), got, kernel % 1, 1, 1)
for on, sizes in ((1, {k_order.GATED}), (0, {k_order.OTHER_GATED})):
    for m, f, k, kernel in sizes:
        got = products(lambda b, x, g, u, d: linear(b, nn.silu(b, linear(b, x, g, f, k)) * linear(b, x, u, f, k), d, 64, f),
                       operand(1, m, k), operand(f, k), operand(f, k), operand(64, f))
        check((m, f, k), got[0], kernel % 2 if "%d" in kernel else kernel, 1, on)

def experts(b, x, idx, gs, us, ds):
    x, total = x + x - x, None
    for i in range(2):
        slot = lang.get(b, 1, i, idx)
        of = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, slot, w))
        y = lang.matmul(b, nn.silu(b, lang.matmul(b, x, of(gs))) * lang.matmul(b, x, of(us)), of(ds))
        total = y if total is None else total + y
    return total
for s, kernel, on in {k_order.EXPERTS}:
    for f, h in ((192, 2048), (2048, 192)):
        got = products(experts, operand(s, 1, h), be.tensor(np.zeros((s, 2), np.uint32)), operand(5, f, h), operand(5, f, h), operand(5, h, f))
        assert len(got) == 2 and all(kernel in g[0] and g[3] == (on if g[2] == 2048 else 0) for g in got), (s, f, h, got)
""", BF16)


def test_tiles_of_256_x_288(fake_hip):  # noqa: F811
    """Where they need fewer rounds, plain with and without a residual, in a batch, stacked; the sizes of test_large_tiles.py."""
    fake_hip(LAUNCHED + f"""
tall, wide = "gemm_bf16_ring_kernelILi%dELi2ELb0E", "gemm_bf16_ring_kernelILi%dELi2ELb1E"
for kernel, sizes in ((wide, {large.WIDE}), (tall, {large.NOT_WIDE}), (wide, [(16384, 1152, 1024)]), (tall, [(8192, 1152, 6912), (4096, 4096, 2048)])):
    for m, n, k in sizes:
        for residual in (False, True):
            (name,) = product(m, n, k, residual=residual)
            assert kernel % 0 in name or (m, n, k) == (8192, 1152, 6912), (m, n, k, name)
            assert (wide % 0 in name) == (kernel is wide), (m, n, k, name)
b, m, n, k = {large.WIDE_BATCH}
for residual in (False, True):
    (name,) = product(m, n, k, batch=b, residual=residual)
    assert wide % 0 in name, name
for kernel, sizes in ((wide, {large.WIDE_GATED}), (tall, [(4096, 2048, 320)])):
    for m, f, k in sizes:
        for kind, act in ((2, nn.silu), (3, nn.gelu)):
            (first, *_) = launched(lambda: run(lambda b, x, g, u, d: linear(b, act(b, linear(b, x, g, f, k)) * linear(b, x, u, f, k), d, 64, f),
                                               operand(1, m, k), operand(f, k), operand(f, k), operand(64, f)))
            assert kernel % kind in first, (m, f, k, first)
""", BF16)


def test_tiles_of_192_x_256(fake_hip):  # noqa: F811
    """Gate and up from eight k-steps on, and q / k / v, where 256 rows to a tile, or 128, put in as many rounds, or a few less and the grid is
    dealt evenly; the sizes of test_large_tiles.py."""
    fake_hip(LAUNCHED + f"""
sys.path.insert(0, "tests")
import test_large_tiles as large
short, ring = "gemm_bf16_ring_kernelILi%dELi2ELb0ELb1E", "gemm_bf16_ring_kernelILi%dE"
for m, f, k, on in ((700, 8192, 512, True), (577, 7688, 576, True), (768, 6920, 640, True), (1153, 8200, 512, True), (2100, 8192, 2048, True),
                    (700, 8192, 448, False), (512, 8192, 2048, False), (769, 8192, 2048, False), (2900, 8192, 2048, False),
                    # more rounds than on other tiles, a grid of a multiple of eight tiles and others; as many rounds
                    (6144, 6912, 1152, True), (5900, 6912, 1152, False), (6208, 6912, 1152, False), (5153, 8192, 2048, True), (1601, 6912, 1152, True)):
    for kind, act in ((2, nn.silu), (3, nn.gelu)):
        (first, *_) = launched(lambda: run(lambda b, x, g, u, d: linear(b, act(b, linear(b, x, g, f, k)) * linear(b, x, u, f, k), d, 64, f),
                                           operand(1, m, k), operand(f, k), operand(f, k), operand(64, f)))
        assert ring % kind in first and (short % kind in first) == on, (m, f, k, first)
for on, sizes in ((True, {large.ROTATED_LARGE}), (False, {large.ROTATED_256}), (False, {large.ROTATED_HALF})):
    for hd, batch, s, heads, kv, k, bias, norm in sizes:
        if hd == 256: continue
        ns, kind = [heads * hd, kv * hd, kv * hd], {{64: 4, 128: 6}}[hd] + bias
        args = [operand(1, batch * s, k)] + [operand(n, k) for n in ns] + [be.tensor(np.zeros(n, np.float32)) for n in ns]
        (name,) = launched(lambda: run(lambda b, x, *p: large.attention_of_projections(b, x + x - x, p, hd, batch, s, heads, kv, k, bias, norm)[0], *args))
        assert ring % kind in name and (short % kind in name) == on, (hd, batch, s, name)
""", BF16)


def test_q_k_v_that_rotate_on_large_tiles(fake_hip):  # noqa: F811
    """256 x 256 and 128 x 256 tiles for the sizes of test_large_tiles.py, with biases and norm; smaller ones, and no rotation, beyond."""
    fake_hip(LAUNCHED + f"""
sys.path.insert(0, "tests")
import test_large_tiles as large
ring = "gemm_bf16_ring_kernelILi%dELi%dE"

def names(hd, batch, s, heads, kv, k, bias, norm, gamma=True):
    ns = [heads * hd, kv * hd, kv * hd]
    args = [operand(1, batch * s, k)] + [operand(n, k) for n in ns]
    args += [be.tensor(np.zeros(n, np.float32)) for n in ns + ([hd] * 2 if gamma else [])]
    return launched(lambda: run(lambda b, x, *p: large.attention_of_projections(b, x + x - x, p, hd, batch, s, heads, kv, k, bias, norm)[0], *args))

for height, sizes in ((2, {large.ROTATED_LARGE}), (1, {large.ROTATED_HALF})):
    for c in sizes:
        hd, bias, norm = c[0], c[6], c[7]
        kind = {{64: 4, 128: 6, 256: 8}}[hd] + (bias or norm)
        for gamma in (True, False) if norm else (True,):
            got = names(*c, gamma=gamma)
            assert len(got) == 1 and ring % (kind, height) in got[0], (c, got)
for c in ((64, 1, 703, 20, 20, 768, False, False), (128, 1, 1202, 16, 16, 704, False, False)):       # few rows; few k
    (got,) = names(*c)
    assert "gemm_bf16_dma_kernel" in got, (c, got)
(got,) = names(256, 4, 257, 4, 1, 768, False, True)
assert "ring_kernelILi9E" not in got, got
""", BF16)


DEPENDENT = LAUNCHED + """
helpers = importlib.import_module("catgrad-rs_amd.llm.helpers")
def rows_of(b, y): return lang.transpose(b, 1, 2, lang.max(b, lang.transpose(b, 1, 2, y)))     # the largest of every column, a row
def column(b, q): return lang.transpose(b, 1, 2, q)
def graph(f, *args):
    for outputs in range(2):
        be.realize(run(lambda b, *a: f(b, *a)[outputs], *args))
        both = cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(Both(len(args), f).term(), list(args))
        for o in both[::-1] if outputs else both: be.realize(o)
    be.sync()

class Both(Term):
    def sort(self): return [lang.TENSOR] * self.n_in, [lang.TENSOR] * 2
    def def_(self, b, args): return self.f(b, *args)
"""


@pytest.mark.parametrize("rows", [4, 16, 300, 512])
@pytest.mark.parametrize("columns", [8, 40])
def test_a_column_that_comes_from_another_product_of_the_same_rows(fake_hip, rows, columns):  # noqa: F811
    """A narrow product takes others of the same rows along, unless their matrices wait for a product: for itself, or for a third."""
    fake_hip(DEPENDENT + f"""
rows, n, k = {rows}, {columns}, 512
x, w, v, u = operand(1, rows, k), operand(n, k), operand(n, k), operand(k, n)
f32 = lambda x: x + x - x
def pooled(b, x, w, u):
    x = f32(x)
    y = linear(b, x, w, n, k)
    return [lang.matmul(b, x, column(b, linear(b, rows_of(b, y), u, k, n))), y]
def largest(b, x, w):
    x = f32(x)
    y = linear(b, x, w, n, rows)
    return [lang.matmul(b, x, lang.reshape(b, lang.make_shape(b, 1, rows, 1), lang.max(b, y))), y]
def third(b, x, w, v, u):
    x = f32(x)
    y, p = linear(b, x, w, n, k), linear(b, x, v, n, k)
    return [y + y, lang.matmul(b, x, column(b, linear(b, rows_of(b, p), u, k, n)))]
graph(pooled, x, w, u)
graph(third, x, w, v, u)
graph(largest, operand(1, rows, rows), operand(n, rows))
""", BF16)


@pytest.mark.parametrize("flags", [0, BF16])
@pytest.mark.parametrize("rows", [1, 4, 16, 300])
def test_matrices_and_biases_that_come_from_another_product_of_the_same_rows(fake_hip, rows, flags):  # noqa: F811
    """The readers of a norm that is computed on the way in, of a gated pair's rows, of q / k / v with biases: none joins that waits for a product."""
    fake_hip(DEPENDENT + f"""
rows, n, k = {rows}, 256, 512
x, w, v, u, one = operand(1, rows, k), operand(n, k), operand(n, k), operand(k, n), operand(1, k)
norm = lambda b, x: helpers.rmsnorm_raw(b, 1e-5, x + x)
def normed(b, x, w, u):
    h = norm(b, x)
    y = linear(b, h, w, n, k)
    return [lang.matmul(b, h, column(b, linear(b, rows_of(b, y), u, k, n))), y]
def third(b, x, w, v, u):
    h = norm(b, x)
    y, p = linear(b, h, w, n, k), linear(b, h, v, n, k)
    return [y + y, lang.matmul(b, h, column(b, linear(b, rows_of(b, p), u, k, n)))]
def biased(rows_in):
    def f(b, x, w, v):
        h = rows_in(b, x)
        y, z, t = linear(b, h, w, n, k), linear(b, h, v, n, k), linear(b, h, v, n, k)
        return [z + lang.broadcast(b, lang.reshape(b, lang.make_shape(b, n), rows_of(b, y)), lang.shape(b, z)), y * t]
    return f
def gated(b, x, w, v, u, one):      # a gated pair and a column that comes from its gate's weights, or they from the column
    h = norm(b, x)
    c = linear(b, h, one, 1, k)
    pair = nn.silu(b, linear(b, h, w, n, k)) * linear(b, h, v, n, k)
    late = lang.matmul(b, h, column(b, linear(b, rows_of(b, lang.broadcast(b, c, lang.shape(b, pair))), u, k, n)))
    return [pair, c + late]
def gated_late(b, x, w, v, u, one):
    h = norm(b, x)
    c = linear(b, h, one, 1, k)
    row = linear(b, rows_of(b, lang.broadcast(b, c, lang.make_shape(b, 1, rows, n))), u, k, n)
    w = lang.transpose(b, 0, 1, w) + lang.broadcast(b, lang.reshape(b, lang.make_shape(b, k, 1), row), lang.make_shape(b, k, n))
    pair = nn.silu(b, lang.matmul(b, h, lang.reshape(b, lang.make_shape(b, 1, k, n), w))) * linear(b, h, v, n, k)
    return [pair, c]
graph(normed, x, w, u)
graph(third, x, w, v, u)
graph(biased(norm), x, w, v)
graph(biased(lambda b, x: x + x - x), x, w, v)
graph(gated, x, w, v, u, one)
graph(gated_late, x, w, v, u, one)
""", flags)


@pytest.mark.parametrize("flags", [0, BF16])
@pytest.mark.parametrize("rows", [1, 4, 20, 300])
def test_experts_chosen_by_another_expert(fake_hip, rows, flags):  # noqa: F811
    """Routed experts' products of the same rows join each other's launches, unless their indices or matrices wait for an expert's product."""
    fake_hip(DEPENDENT + f"""
s, f, k = {rows}, 256, 512
x, idx = be.tensor(np.zeros((s, 1, k), np.float32)), be.tensor(np.zeros((s, 2), np.uint32))
up, down = [operand(5, f, k) for i in range(2)], operand(5, k, f)
of = lambda b, i, w: lang.transpose(b, 1, 2, lang.index(b, 0, i, w))
first = lambda b, idx: lang.reshape(b, lang.make_shape(b, s), lang.get(b, 1, 0, idx))
def plain(b, x, idx, w):
    y = lang.matmul(b, x, of(b, first(b, idx), w))
    return [y + lang.matmul(b, x, of(b, lang.reshape(b, lang.make_shape(b, s), lang.argmax(b, y)), w)), y]
def matrices(b, x, idx, w):
    y = lang.matmul(b, x, of(b, first(b, idx), w))
    t = lang.broadcast(b, lang.slice(b, 0, 0, 1, y), lang.make_shape(b, 5, k, f))
    return [lang.matmul(b, x, of(b, first(b, idx), lang.transpose(b, 1, 2, t))), y]
def whole(b, x, idx, g, u, d):
    expert = lambda i: lang.matmul(b, nn.silu(b, lang.matmul(b, x, of(b, i, g))) * lang.matmul(b, x, of(b, i, u)), of(b, i, d))
    y = expert(first(b, idx))
    return [y + expert(lang.reshape(b, lang.make_shape(b, s), lang.argmax(b, y))), y]
graph(plain, x, idx, up[0])
graph(matrices, x, idx, up[0])
graph(whole, x, idx, *up, down)
""", flags)


def test_a_dense_expert_in_the_routed_experts_launches(fake_hip):  # noqa: F811
    """Up to 3072 tokens; launches of its own beyond."""
    fake_hip(LAUNCHED + """
sys.path.insert(0, "tests")
import test_dense_expert as dense
e, f, h, fs = 5, 768, 1280, 320
weights = [operand(*s) for s in ((e, f, h), (e, f, h), (e, h, f), (fs, h), (fs, h), (h, fs))]
for s, joined in ((300, True), (3072, True), (3073, False)):
    be.sync()
    fake.fake_hip_launched()
    term = type("Layer", (Term,), {"sort": lambda self: ([lang.TENSOR] * 8, [lang.TENSOR] * 2), "def_": lambda self, b, args: dense.layer("silu", 2, f, h, fs)(b, *args)})
    for t in cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(term(8, None).term(), [operand(1, s, h), be.tensor(np.zeros((s, 2), np.uint32))] + weights):
        be.realize(t)
    be.sync()
    names = [n for n in fake.fake_hip_launched().decode().split("\\n") if "gem" in n or "moe_ring" in n]
    assert sum("moe_ring" in n for n in names) == 2 and (len(names) == 2) == joined, (s, names)
""", BF16)


def test_a_product_and_a_column_that_start_at_different_k(fake_hip):  # noqa: F811
    """The sizes of test_large_tiles.py: one launch of 32 x 32 tiles, up to 128 rows of whole multiples of 4 KB with an order of their own."""
    fake_hip(LAUNCHED + f"""
for m, n, k, joined in {large.WITH_COLUMN}:
    both = lambda b, x, w, c: [linear(b, x, w, n, k), linear(b, x, c, 1, k)]
    term = type("Both", (Term,), {{"sort": lambda self: ([lang.TENSOR] * 3, [lang.TENSOR] * 2), "def_": lambda self, b, a: both(b, a[0] + a[0] - a[0], *a[1:])}})
    be.sync()
    fake.fake_hip_products()
    for t in cg.Interpreter(be, cg.stdlib(), cg.Parameters()).run(term(3, None).term(), [operand(1, m, k), operand(n, k), operand(1, k)]):
        be.realize(t)
    be.sync()
    lines = [line.rsplit(" ", 3) for line in fake.fake_hip_products().decode().splitlines()]
    assert (len(lines) == 1) == joined, (m, n, k, lines)
    if joined:
        assert "gemm_bf16_dma_kernelILi32ELi32E" in lines[0][0] and int(lines[0][3]) == (m <= 128 and k >= 2048 and k % 2048 == 0), (m, n, k, lines)
""", BF16)


@pytest.mark.parametrize("flags", [0, BF16])
@pytest.mark.parametrize("shared", [True, False])
def test_layers_of_experts_that_wait_for_each_other(fake_hip, flags, shared):  # noqa: F811
    """Nothing is realised between three layers: with matrices of their own or the same in each (whose experts' products look alike), a few tokens
    and many.  The experts' launch of a few tokens finds their experts itself, as where the layer in front is there."""
    fake_hip(LAUNCHED + f"""
helpers = importlib.import_module("catgrad-rs_amd.llm.helpers")
k, f, fs, e, top, shared, flags = 512, 256, 1024, 60, 4, {shared}, {flags}
def chain(rows, layers):
    re = lambda b, x, *shape: lang.reshape(b, lang.make_shape(b, *shape), x)
    def layer(b, x, wr, wg, wu, wd, sg, su, sd, gate):
        h = helpers.rmsnorm_raw(b, 1e-5, x)
        values, idx = lang.topk(b, top, nn.softmax(b, re(b, linear(b, h, wr, e, k), rows, e)))
        each, total = re(b, h, rows, 1, k), None
        for i in range(top):
            slot = lang.get(b, 1, i, idx)
            of = lambda w: lang.transpose(b, 1, 2, lang.index(b, 0, slot, w))
            y = lang.matmul(b, nn.silu(b, lang.matmul(b, each, of(wg))) * lang.matmul(b, each, of(wu)), of(wd))
            y = y * lang.broadcast(b, re(b, lang.get(b, 1, i, values), rows, 1, 1), lang.shape(b, y))
            total = y if total is None else total + y
        y = linear(b, nn.silu(b, linear(b, h, sg, fs, k)) * linear(b, h, su, fs, k), sd, k, fs)
        y = y * lang.broadcast(b, nn.sigmoid(b, linear(b, h, gate, 1, k)), lang.shape(b, y))
        return re(b, total, 1, rows, k) + y
    def all_of_them(b, x, *ws):
        x = x + x - x
        for i in range(layers): x = layer(b, x, *(ws if shared else ws[8 * i:8 * i + 8]))
        return x
    shapes = ((e, k), (e, f, k), (e, f, k), (e, k, f), (fs, k), (fs, k), (k, fs), (1, k))
    args = [operand(1, rows, k)] + [operand(*s) for s in shapes * (1 if shared else layers)]
    be.sync()
    fake.fake_hip_launched()
    be.realize(run(all_of_them, *args))
    be.sync()
    return [n for n in fake.fake_hip_launched().decode().split("\\n") if n]
for rows in (1, 4, 9, 20, 300):
    one, three = chain(rows, 1), chain(rows, 3)
    if rows < 9:
        assert not any("softmax_topk" in n for n in three), (rows, three)
""", flags)


@pytest.mark.parametrize("flags", [0, BF16])
def test_what_a_product_adds_lies_in_memory(fake_hip, flags):  # noqa: F811
    """`linear(x) + bias` of a value that is such a sum itself, and of residuals: a bias vector is not read as a matrix, whatever was realised
    on the way to it."""
    fake_hip(LAUNCHED + f"""
helpers = importlib.import_module("catgrad-rs_amd.llm.helpers")
fake.fake_hip_outside.restype = ctypes.c_char_p
k = 512
def biased(b, x, w, bias, n):
    y = linear(b, x, w, n, k)
    return y + lang.broadcast(b, bias, lang.shape(b, y))
between = {{"nothing": lambda b, y, x: y, "gelu": lambda b, y, x: nn.gelu(b, y), "silu": lambda b, y, x: nn.silu(b, y), "sigmoid": lambda b, y, x: nn.sigmoid(b, y),
           "norm": lambda b, y, x: helpers.rmsnorm_raw(b, 1e-5, y), "residual": lambda b, y, x: x + y, "softmax": lambda b, y, x: nn.softmax(b, y)}}
for rows in (1, 2, 4, 8, 9, 16, 20, 100, 300, 1000):
    for n in (512, 40):
        for what, act in between.items():
            def chain(b, x, w1, b1, w2, b2, w3, b3):
                x = x + x - x
                y = act(b, biased(b, x, w1, b1, k), x)
                return biased(b, act(b, biased(b, y, w2, b2, k), x), w3, b3, n)
            args = [operand(1, rows, k)]
            for m in (k, k, n): args += [operand(m, k), be.tensor(np.zeros(m, np.float32))]
            be.realize(run(chain, *args))
            be.sync()
            assert not fake.fake_hip_outside(), (rows, n, what)
""", flags)
