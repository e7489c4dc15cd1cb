"""Subnormal, infinite and NaN operands through every projection that runs on
depth-1 FP32 MFMA: the catalog's and the packed projection's tiles against the
oracle, the decode projections of three to eight rows and the exact prompt
pass against the one-row decode step (vector-ALU FMAs, itself equal to the
oracle).  An MFMA element is one FMA with a single rounding and subnormals
kept, so results are equal bit for bit, and a special value in one row leaves
the other rows as they are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HIDDEN = 4096


def special_rows(rng, rows, width):
    """FP32 rows, one kind after the other; row 0 and every sixth are plain."""
    x = rng.standard_normal((rows, width)).astype(np.float32)
    for r in range(rows):
        at = rng.integers(0, width, 3)
        kind = r % 6
        if kind == 1:
            x[r] *= 1e-39  # subnormal inputs
        elif kind == 2:
            x[r] *= 1e-20  # subnormal products with the weights of 1e-20
        elif kind == 3:
            x[r, at[0]] = np.inf
        elif kind == 4:
            x[r, at[0]] = np.nan
        elif kind == 5:
            x[r, at] = 3e38, -np.inf, 3e38
    return x


def special_weights(rng, outputs, width):
    w = (0.05 * rng.standard_normal((outputs, width))).astype(np.float32)
    w[1::5] *= 1e-20
    w[2::5] *= 1e-38  # subnormal
    w[3::7, rng.integers(0, width)] = -np.inf
    w[4::11, rng.integers(0, width)] = 3e38
    return w


def check_mix(bits):
    """The case holds what it is for: finite, infinite, NaN and subnormal results."""
    exponent, fraction = bits & 0x7f80, bits & 0x7f
    assert ((exponent == 0x7f80) & (fraction == 0)).any() and ((exponent == 0x7f80) & (fraction != 0)).any()
    assert ((exponent == 0) & (fraction != 0)).any() and (exponent < 0x7f80).any()


# (16- and 32-row tiles) x (16 and 32 partials).
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("rows,in_w,out_w", [(18, 512, 1040), (12, 512, 64), (102, 512, 1040), (99, 4352, 64)])
def test_projection_tiles(device, queue, oracle, packed, rows, in_w, out_w):
    from dolittle_amd import _lib
    rng = np.random.default_rng(rows + in_w)
    x, w = (oracle.bf16_from_f32(a.reshape(-1)) for a in (special_rows(rng, rows, in_w), special_weights(rng, out_w, in_w)))
    want = oracle.projection(x, w, rows, in_w, out_w)
    check_mix(want)
    bx, bw, by = (device.upload_array(queue, a) for a in (x, w, np.zeros(rows * out_w, np.uint16)))
    if packed:
        weights = device.allocate(w.nbytes)
        _lib.call("dl_projection_pack", queue.handle, bw.ptr(), weights.ptr(), out_w, in_w)
        _lib.call("dl_projection_packed", queue.handle, bx.ptr(), weights.ptr(), by.ptr(), rows, in_w, out_w, None)
    else:
        _lib.call("dl_projection", queue.handle, 1, bx.ptr(), bw.ptr(), by.ptr(), rows, in_w, out_w, None)
    queue.drain()
    assert np.array_equal(queue.read(by, np.uint16, want.size), want)


@pytest.fixture(scope="module", params=["tiny weights", "infinite gain"])
def model(request, device, queue, oracle):
    """Two blocks whose projections have outputs of 1e-20 and subnormal
    weights among the ordinary ones; or an infinite norm gain, so that every
    row of the first projections has an infinite input."""
    from dolittle_amd.qwen3 import Qwen3Config, Qwen3Model
    m = Qwen3Model(device, queue, Qwen3Config(layers=2, vocab=2048))
    m.fill_synthetic(77, 0.02)
    if request.param == "infinite gain":
        gain = np.ascontiguousarray(m.read("input_norm", 0).reshape(-1))
        gain[9] = 0x7f80
        m.write("input_norm", 0, gain)
        return m
    for role, layer in [(r, l) for r in ("q", "k", "v", "o", "gate", "up", "down") for l in (0, 1)] + [("lm_head", 0)]:
        w = oracle.f32_from_bf16(m.read(role, layer).reshape(-1)).reshape(m.config.shape(role)).copy()
        w[1::5] *= 1e-20
        w[2::5] *= 1e-37
        m.write(role, layer, oracle.bf16_from_f32(w.reshape(-1)))
    return m


def special_row(oracle, kind):
    rng = np.random.default_rng(3)
    row = (0.02 * rng.standard_normal(HIDDEN)).astype(np.float32)
    if kind == "subnormal":
        row *= 1e-37
    elif kind == "nan":
        row[100] = np.nan
    elif kind == "inf":
        row[200] = np.inf
    return oracle.bf16_from_f32(row)


def caches(plan, count, seq=0):
    return [a for layer in (0, 1) for a in plan.read_cache(layer, 0, count, seq)]


@pytest.mark.parametrize("batch", [3, 8])
@pytest.mark.parametrize("kind", ["subnormal", "nan", "inf"])
def test_decode_rows(model, oracle, kind, batch):
    """The last position of one sequence takes a special embedding row; every
    sequence equals the one-sequence step with and without that row."""
    from dolittle_amd.qwen3 import Plan
    ids, special = np.array([7, 300], np.uint32), batch - 2
    want = []
    for mask in (0, 1):
        one = Plan(model, batch=1, capacity=8)
        if mask:
            one.set_embedding_override(1, special_row(oracle, kind), 1)
        one.forward(ids)
        want.append([one.hidden(0), one.logits(0), *caches(one, 2)])
    many = Plan(model, batch=batch, capacity=8)
    many.set_embedding_override(1, special_row(oracle, kind), 1 << special)
    many.forward(ids)
    for b in range(batch):
        for got, expected in zip([many.hidden(b), many.logits(b), *caches(many, 2, b)], want[b == special]):
            assert np.array_equal(got, expected), b


@pytest.mark.parametrize("kind", ["subnormal", "nan", "inf"])
def test_exact_prompt_rows(model, oracle, kind):
    """33 positions in one chunk of the many-row GEMM, the last one special;
    their K/V rows of both blocks equal those of the token loop."""
    from dolittle_amd.qwen3 import Plan
    prompt = np.random.default_rng(5).integers(0, 2048, 34).astype(np.uint32)
    plans = [Plan(model, batch=1, capacity=48) for _ in range(2)]
    for plan in plans:
        plan.set_embedding_override(32, special_row(oracle, kind), 1)
    plans[0].prefill(prompt)
    plans[1].forward(prompt[:33])
    for got, expected in zip(caches(plans[0], 33), caches(plans[1], 33)):
        assert np.array_equal(got, expected)
