"""Performance cases of the FK20 library: what its users have it do, through its public entry
points (the `fk20_amd` package over the C ABI of include/fk20.h), from one row to full batches.

Points leave every case in a canonical encoding -- 48-byte compressed points (the prover's
output format) or canonical affine coordinates (fk20_g1p_to_affine) -- because that is what a
program stores, sends or compares: a projective representative is not unique.

Every output is whole numbers, so there is no floating-point value for it (`exact`).
"""
import ctypes
import math
import os
import sys

import torch  # before the library, so that both use one HIP runtime

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fk20-cuda_amd"))
from fk20_amd import lib, synthetic  # noqa: E402
from fk20_amd.prover import Prover  # noqa: E402

SIZES = (1024, 2048, 4096)


def listed():
    return [
        # one blob of the full size: the latency a single request sees
        {"name": "prove_1_of_4096", "do": "prove", "groups": "4096:1", "window": 8, "out": "affine"},
        # a small batch of small blobs at a ragged row count, proofs as they are sent
        {"name": "prove_37_of_1024", "do": "prove", "groups": "1024:37", "window": 10, "out": "compressed"},
        # an ordinary batch, not a multiple of a wave
        {"name": "prove_200_of_2048", "do": "prove", "groups": "2048:200", "window": 12, "out": "affine"},
        # the benchmark batch: 512 rows of 4096 coefficients
        {"name": "prove_512_of_4096", "do": "prove", "groups": "4096:512", "window": 12, "out": "compressed"},
        # what a serving loop packs into one pass: three setups, uneven groups, sampling order
        {"name": "prove_uneven", "do": "prove", "groups": "1024:150,2048:75,4096:301", "window": 8,
         "out": "compressed_da"},
        # the drop-in call without a resident setup: one row, and an odd batch
        {"name": "plain_1_of_4096", "do": "plain", "N": 4096, "rows": 1},
        {"name": "plain_100_of_2048", "do": "plain", "N": 2048, "rows": 100},
        # the stages on their own: column sums over a caller's points, the G1 transforms in both
        # directions, the scalar transform of a batch's Toeplitz rows
        {"name": "msm_300_of_512", "do": "msm", "n": 512, "rows": 300},
        {"name": "g1_fft_512_of_512", "do": "g1_fft", "n": 512, "count": 512, "inverse": False},
        {"name": "g1_ift_65_of_128", "do": "g1_fft", "n": 128, "count": 65, "inverse": True},
        {"name": "fr_fft_8192_of_512", "do": "fr_fft", "n": 512, "count": 8192, "inverse": False},
        # commitments of a batch, the step before its proofs
        {"name": "commit_512_of_4096", "do": "commit", "N": 4096, "rows": 512, "window": 10},
    ]


def _rows(rng, hi):
    return max(1, min(hi, int(round(math.exp(rng.uniform(0.0, math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prove", "prove", "prove", "plain", "msm", "g1_fft", "fr_fft", "commit"])
    if kind == "prove":
        sizes = list(SIZES)
        rng.shuffle(sizes)
        sizes = sorted(sizes[:rng.choice([1, 1, 1, 2, 3])])
        top = 512 // len(sizes)
        return {"do": "prove", "groups": ",".join("%d:%d" % (N, _rows(rng, top)) for N in sizes),
                "window": rng.choice([8, 9, 10, 11] if len(sizes) > 1 else [8, 9, 10, 11, 12]),
                "out": rng.choice(["affine", "affine_da", "compressed", "compressed_da"])}
    if kind == "plain":
        return {"do": "plain", "N": rng.choice(SIZES), "rows": _rows(rng, 200)}
    if kind == "msm":
        return {"do": "msm", "n": rng.choice([128, 256, 512]), "rows": _rows(rng, 512)}
    if kind == "g1_fft":
        return {"do": "g1_fft", "n": rng.choice([128, 256, 512]), "count": _rows(rng, 512),
                "inverse": rng.random() < 0.5}
    if kind == "fr_fft":
        return {"do": "fr_fft", "n": rng.choice([128, 256, 512]), "count": _rows(rng, 8192),
                "inverse": rng.random() < 0.5}
    return {"do": "commit", "N": rng.choice(SIZES), "rows": _rows(rng, 512), "window": rng.choice([8, 9, 10])}


# ---------------------------------------------------------------- inputs

# top 64-bit word of r: a word below it makes the value less than r
_R_TOP = 0x73EDA753299D7D48


def _scalars(gen, *shape):
    """Scalars below r, uniform but for the last 2^-62 of the range: (..., 4) words on the GPU."""
    w = torch.randint(-2**63, 2**63 - 1, shape + (4,), generator=gen, dtype=torch.int64)
    w[..., 3] = torch.randint(0, _R_TOP, shape, generator=gen, dtype=torch.int64)
    return w.cuda()


def _field(gen, n):
    """Non-zero residues below p: (n, 6) words on the GPU."""
    w = torch.randint(-2**63, 2**63 - 1, (n, 6), generator=gen, dtype=torch.int64)
    w[:, 5] = torch.randint(1, 0x1A0111EA397FE69A, (n,), generator=gen, dtype=torch.int64)
    return w.cuda()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _points(gen, n):
    """n points of G1 as projective triples with independent z (what earlier stages hand on):
    multiples of the generator, brought to x, y and scaled by z."""
    k = _scalars(gen, n)
    g = torch.tensor(synthetic.G1_GEN.astype("int64")).cuda().expand(n, 18).contiguous()
    p = torch.empty(n, 18, dtype=torch.int64, device="cuda")
    xy = torch.empty(n, 12, dtype=torch.int64, device="cuda")
    z = _field(gen, n)
    s = _stream()
    lib.call("fk20_g1p_op", 3, p.data_ptr(), g.data_ptr(), None, k.data_ptr(), n, s)
    lib.call("fk20_g1p_to_affine", xy.data_ptr(), p.data_ptr(), n, s)
    zz = z.repeat_interleave(2, 0).contiguous()
    lib.call("fk20_fp_op", 2, xy.data_ptr(), xy.data_ptr(), zz.data_ptr(), 2 * n, s)
    torch.cuda.synchronize()
    return torch.cat([xy, z], 1).contiguous()


def _words(gen):
    return int(torch.randint(1, 2**62, (1,), generator=gen))


def _secret(gen):
    return (_words(gen) | _words(gen) << 62 | _words(gen) << 124) + 1


def _empty(*shape, dtype=torch.int64):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _groups(case):
    return [tuple(int(v) for v in g.split(":")) for g in case["groups"].split(",")]


class _State:
    """What a program holds between calls; its prover's tables are freed with it."""
    prover = None

    def __del__(self):
        if self.prover is not None:
            self.prover.close()
            self.prover = None


def prepare(case, seed):
    gen = torch.Generator().manual_seed(seed)
    st = _State()
    st.case = case
    kind = case["do"]
    if kind == "prove":
        st.prover = Prover()
        st.prover.set_output({"affine": "g1p", "affine_da": "g1p_da"}.get(case["out"], case["out"]))
        st.affine = case["out"].startswith("affine")
        st.items, st.keep, st.out = [], [], []
        for N, rows in _groups(case):
            xext = synthetic.device_setup(N, _secret(gen))
            sid = st.prover.load_setup(xext, N, case["window"])
            xext.free()
            st.prover.reserve(rows, N)
            poly = _scalars(gen, rows, N)
            h = _empty(rows, N // 8, 18) if st.affine else _empty(rows, N // 8, 48, dtype=torch.uint8)
            st.items.append((sid, rows, poly.data_ptr(), h.data_ptr()))
            st.keep.append((poly, h))
            st.out.append(_empty(rows, N // 8, 12) if st.affine else h)
    elif kind == "plain":
        N, rows = case["N"], case["rows"]
        st.xext = synthetic.device_setup(N, _secret(gen))
        st.poly = _scalars(gen, rows, N)
        st.h = _empty(rows, N // 8, 18)
        st.xy = _empty(rows, N // 8, 12)
    elif kind == "msm":
        n, rows = case["n"], case["rows"]
        st.tc = _scalars(gen, rows, 16, n)
        st.x = _points(gen, 16 * n)
        st.h = _empty(rows, n, 18)
        st.xy = _empty(rows, n, 12)
    elif kind == "g1_fft":
        n, count = case["n"], case["count"]
        st.x = _points(gen, count * n)
        st.y = _empty(count, n, 18)
        st.xy = _empty(count, n, 12)
    elif kind == "fr_fft":
        st.x = _scalars(gen, case["count"], case["n"])
        st.y = torch.empty_like(st.x)
    else:
        N, rows = case["N"], case["rows"]
        st.prover = Prover()
        srs = synthetic.device_srs(N, _secret(gen))
        st.sid = st.prover.load_commit_setup(srs, N, case["window"])
        srs.free()
        st.poly = _scalars(gen, rows, N)
        st.c = _empty(rows, 18)
        st.xy = _empty(rows, 12)
    torch.cuda.synchronize()
    return st


def _affine(xy, pts):
    lib.call("fk20_g1p_to_affine", xy.data_ptr(), pts.data_ptr(), pts.numel() // 18, _stream())
    return xy


def run(st):
    case = st.case
    kind = case["do"]
    s = ctypes.c_void_p(_stream())
    if kind == "prove":
        if len(st.items) == 1:
            sid, rows, poly, h = st.items[0]
            st.prover.prove_device(sid, h, poly, rows, s)
        else:
            st.prover.prove_batch_device(st.items, s)
        if st.affine:
            for (_, h), xy in zip(st.keep, st.out):
                _affine(xy, h)
        return st.out
    if kind == "plain":
        lib.call("fk20_poly2h_fft", st.h.data_ptr(), st.poly.data_ptr(), st.xext.ptr, case["rows"], case["N"], s)
        return _affine(st.xy, st.h)
    if kind == "msm":
        lib.call("fk20_msm", st.h.data_ptr(), st.tc.data_ptr(), st.x.data_ptr(), case["rows"], case["n"], s)
        return _affine(st.xy, st.h)
    if kind == "g1_fft":
        lib.call("g1p_ift" if case["inverse"] else "g1p_fft", st.y.data_ptr(), st.x.data_ptr(), case["count"],
                 case["n"], s)
        return _affine(st.xy, st.y)
    if kind == "fr_fft":
        lib.call("fr_ift" if case["inverse"] else "fr_fft", st.y.data_ptr(), st.x.data_ptr(), case["count"],
                 case["n"], s)
        return st.y
    st.prover.commit_device(st.sid, st.c.data_ptr(), st.poly.data_ptr(), case["rows"], s)
    return _affine(st.xy, st.c)


# ---------------------------------------------------------------- work

# 32 x 32-bit multiply-adds of a product in Fp (12 words) and Fr (8 words), operand and
# Montgomery half; the group operations of the library's algorithms in Fp products
_FP, _FR = 2 * 12 * 12, 2 * 8 * 8
_ADD, _MIXED, _DBL = 12, 11, 7
_TWIDDLE = 124 * _DBL + 43 * _MIXED


def _transform(n):
    """Fp products of one G1 transform: radix-2^2, twiddles on 3/4 of the points per two stages."""
    lg = n.bit_length() - 1
    return n * lg // 2 * 2 * _ADD + 3 * n // 4 * (lg // 2) * _TWIDDLE


def work(case):
    """Points and scalars in and out once; one product = 2 operations per multiply-add."""
    kind = case["do"]
    if kind == "prove":
        out = 96 if case["out"].startswith("affine") else 48
        nbytes = fp = fr = 0
        for N, rows in _groups(case):
            n = N // 8
            nbytes += rows * (N * 32 + n * out)
            fp += rows * (16 * n * -(-256 // case["window"]) * _MIXED + 2 * _transform(n))
            fr += rows * 16 * n // 2 * (n.bit_length() - 1)
    elif kind == "plain":
        n, rows = case["N"] // 8, case["rows"]
        nbytes = rows * (case["N"] * 32 + n * 96) + 16 * n * 144
        fp = rows * (n * (252 * _DBL + 16 * 43 * _ADD) + 2 * _transform(n))
        fr = rows * 16 * n // 2 * (n.bit_length() - 1)
    elif kind == "msm":
        n, rows = case["n"], case["rows"]
        nbytes = rows * n * (16 * 32 + 96) + 16 * n * 144
        fp, fr = rows * n * (252 * _DBL + 16 * 43 * _ADD), 0
    elif kind == "g1_fft":
        n, count = case["n"], case["count"]
        nbytes = count * n * (144 + 96)
        fp, fr = count * _transform(n), 0
    elif kind == "fr_fft":
        n, count = case["n"], case["count"]
        nbytes = count * n * 64
        fp, fr = 0, count * n // 2 * (n.bit_length() - 1)
    else:
        N, rows = case["N"], case["rows"]
        nbytes = rows * (N * 32 + 96)
        fp, fr = rows * N * -(-256 // case["window"]) * _MIXED, 0
    return {"bytes": nbytes, "flops": 2 * (fp * _FP + fr * _FR)}


def exact(case, seed):
    """Every output is whole numbers (residues and encoded points), equal or wrong."""
    return None
