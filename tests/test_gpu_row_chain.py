"""The products of a layer in one launch: sizes at the edges of its rows, of
the pieces of K and of its ways of bringing x, against the same in 64 bits,
and what a wave computes for blocks that are not there."""

import pytest
import torch

pytestmark = pytest.mark.gpu

U8, BF, F32 = torch.uint8, torch.bfloat16, torch.float32


@pytest.fixture(scope="module")
def ho():
    from llm_np_cp_amd.ops import hip_ops
    return hip_ops


def rand(seed, *shape, scale=1.0):
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda") * scale


def weight(ho, wt, seed, N, K):
    """As it is multiplied, and its values in 64 bits."""
    w = rand(seed, N, K, scale=K ** -0.5).bfloat16()
    if wt == 0:
        return (w, None, None), w.double()
    if wt == 1:
        q = torch.empty(N, K, dtype=U8, device="cuda")
        s = torch.empty(N, device="cuda")
        ho.quant_fp8(w, q, s)
        return (q, s, None), q.view(torch.float8_e4m3fn).double() * \
            s.double()[:, None]
    q = torch.empty(N, K // 2, dtype=U8, device="cuda")
    e = torch.empty(N, K // 32, dtype=U8, device="cuda")
    ho.quant_fp4(w, q, e)
    grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0],
                        dtype=torch.float64, device="cuda")
    nib = torch.stack([q & 15, q >> 4], -1).reshape(N, K).long()
    v = grid[nib & 7] * torch.where(nib > 7, -1.0, 1.0)
    return (q, None, e), v * torch.exp2(e.double() - 127.0) \
        .repeat_interleave(32, 1)


class Layer:
    """att -> o -> gate and up -> down -> q, k and v of the next layer, each
    from what the one before it left in memory (so that a rounding in one is
    no error of the next)."""

    def __init__(self, ho, wt, H, I, A, Q, gemma=False, last=False, seed=0,
                 head=0.0):
        self.ho, self.gemma, self.last, self.head = ho, gemma, last, head
        act = F32 if wt else BF
        self.W = [weight(ho, wt, seed + 1, H, A), weight(ho, wt, seed + 2,
                  2 * I, H), weight(ho, wt, seed + 3, H, I),
                  weight(ho, wt, seed + 4, Q, H)]
        self.att = rand(seed + 5, A).bfloat16()
        self.h = rand(seed + 6, H).bfloat16()
        self.bias = rand(seed + 7, Q).bfloat16()
        self.g = [1 + 0.1 * rand(seed + 8 + i, H) for i in range(4)]
        kinds = (H, BF), (I, act), (H, BF)
        size = [ho.chain_room(*k) for k in kinds]
        self.buf = torch.zeros(sum(size), dtype=U8, device="cuda")
        o, mid, dn = (ho.chain_part(self.buf, sum(size[:k]), *v)
                      for k, v in enumerate(kinds))
        self.o, self.mid, self.dn = o, mid, dn
        self.qkv = torch.zeros(Q + 8, dtype=F32 if head else BF,
                               device="cuda")
        self.hout = torch.zeros(H, dtype=BF, device="cuda")
        gu = dict(W=self.W[1][0], x=o, y=mid, glu=True)
        down = dict(W=self.W[2][0], x=mid, y=dn)
        st = [dict(W=self.W[0][0], x=self.att, y=o), gu, down]
        qkv = dict(W=self.W[3][0], x=dn, y=self.qkv, softcap=head,
                   add=None if head else self.bias)
        if gemma:
            gu.update(kind=ho.CHAIN_NORM2, h=self.h, g=self.g[0],
                      g2=self.g[1])
            qkv.update(kind=ho.CHAIN_NORM2, g=self.g[2], g2=self.g[3],
                       hout=self.hout)
            if last:
                gu.update(hout=self.hout)
        else:
            st[0].update(add=self.h)
            gu.update(kind=ho.CHAIN_NORM, g=self.g[0])
            down.update(add=o)
            qkv.update(kind=ho.CHAIN_NORM, g=self.g[1])
        self.chain = ho.Chain(st + [qkv] * (not last), wt, int(gemma), 1e-5)
        self.wt = wt

    def run(self, **kw):
        self.buf.fill_(255)
        self.chain.run(**kw)
        torch.cuda.synchronize()
        return [t.clone() for t in (self.o, self.mid, self.dn, self.qkv,
                                    self.hout)]

    def check(self, out):
        """Each product's error by the roundings on its way: bf16 x and y
        (2^-9 each), sums in 32 bits, the factors of a norm and of the gate
        (some 2^-20)."""
        o, mid, dn, qkv, hout = (t.double() for t in out)
        W = [w for _, w in self.W]

        def norm(x):
            return x / torch.sqrt((x * x).mean() + 1e-5)

        def near(got, x, w, factor=None, add=None, bf=True, xbf=False):
            want = w @ x
            far = w.abs() @ x.abs() * (2.0 ** -9 * (xbf and self.wt == 0) +
                                       x.numel() * 2.0 ** -23 + 2.0 ** -19)
            if factor is not None:
                want, far = factor(want, far)
            if add is not None:
                want = want + add
            far = far + want.abs() * 2.0 ** -8 * bf + 1e-30
            assert ((got - want).abs() <= far).all(), \
                ((got - want).abs() / far).max()

        near(o, self.att.double(), W[0],
             add=None if self.gemma else self.h.double())
        if self.gemma:
            h1 = (self.h.double() + norm(o) * self.g[0].double()) \
                .bfloat16().double()
            x = norm(h1) * self.g[1].double()
        else:
            x = norm(o) * self.g[0].double()

        def gate(z, far):
            I = mid.numel()
            a, b = z[:I], z[I:]
            t = a.clone().requires_grad_()
            s = torch.nn.functional.gelu(t, approximate="tanh") \
                if self.gemma else torch.nn.functional.silu(t)
            s.sum().backward()
            s = s.detach()
            return s * b, (t.grad.abs() * far[:I] + far[:I] ** 2) * \
                (b.abs() + far[I:]) + s.abs() * (far[I:] + 2.0 ** -18 *
                                                 b.abs())

        # the gemma stream may round to its other neighbour here and there:
        # 2^-8 of it, in place of the exact value above
        slack = 2.0 ** -8 if self.gemma else 0.0
        W1 = W[1]
        near(mid, x, W1, lambda z, far: gate(z, far + slack * (
            W1.square() @ x.square()).sqrt()), bf=self.wt == 0, xbf=True)
        near(dn, mid, W[2], add=None if self.gemma else o)
        if self.gemma and not self.last:
            h2 = h1 + norm(dn) * self.g[2].double()
            assert ((hout - h2).abs() <= h2.abs() * 2.0 ** -8 +
                    h1.abs() * 2.0 ** -7).all()
            x = norm(hout) * self.g[3].double()
        elif self.gemma:
            assert ((hout - h1).abs() <= h1.abs() * 2.0 ** -7).all()
        else:
            x = norm(dn) * self.g[1].double()
        if not self.last:
            n = self.bias.numel()
            if self.head:                     # |d cap tanh(z / cap)| <= |dz|
                near(qkv[:n], x, W[3], lambda z, far: (
                    self.head * torch.tanh(z / self.head),
                    far + self.head * 2.0 ** -20), bf=False, xbf=True)
            else:
                near(qkv[:n], x, W[3], add=self.bias.double(), xbf=True)
            assert (qkv[n:] == 0).all()       # nothing behind its end


# blocks without rows, with one, four and five, ends of rows inside a piece
# and on its edge, x by 2, 4 and 8 quads a thread, rings of 8 to 4 slots
SIZES = [
    (128, 256, 128, 192),
    (256, 512, 64, 130),
    (1024, 1280, 1024, 1536),
    (1152, 2048, 640, 1290),
    (2048, 8192, 2048, 3072),
    (2304, 4608, 2048, 2310),
    (3584, 9472, 3584, 4608),
    (4096, 14336, 4096, 6144),
]


@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("gemma", [False, True])
@pytest.mark.parametrize("H,I,A,Q", SIZES)
def test_chain(ho, wt, gemma, H, I, A, Q):
    if wt == 2 and any(k % 128 for k in (H, I, A)):
        pytest.skip("rows of MXFP4 that are no multiple of 128")
    l = Layer(ho, wt, H, I, A, Q, gemma)
    assert l.chain.fits()
    first = l.run()
    l.check(first)
    for _ in range(3):                        # a pass gives the same bits
        for a, b in zip(first, l.run()):
            assert torch.equal(a, b)


# more rows a block than threads that finish them, one each, and a rest
@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("gemma", [False, True])
@pytest.mark.parametrize("V", [512, 32768, 66000, 128256])
def test_head(ho, wt, gemma, V):
    l = Layer(ho, wt, 256, 768, 256, V, gemma, head=30.0)
    assert l.chain.fits()
    l.check(l.run())


@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("gemma", [False, True])
def test_last_layer(ho, wt, gemma):
    l = Layer(ho, wt, 256, 768, 256, 64, gemma, last=True)
    l.check(l.run())


# limit 0: a wave computes by itself whatever is not there at its first read
@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("gemma", [False, True])
@pytest.mark.parametrize("H,I,A,Q", [(128, 256, 128, 192),
                                     (1152, 1152, 640, 1290),
                                     (2304, 2560, 2048, 2310)])
def test_what_is_missing_is_computed(ho, wt, gemma, H, I, A, Q):
    l = Layer(ho, wt, H, I, A, Q, gemma)
    for a, b in zip(l.run(), l.run(limit=0)):
        assert torch.equal(a, b)


def claims(ho, absent=()):
    """A word a block, of ones; without bit 2 it leaves its rows to others."""
    c = torch.full((ho.CHAIN_BLOCKS,), -1, dtype=torch.int32, device="cuda")
    c[list(absent)] = ~4
    return c


# blocks that do nothing, as where another stream's kernels hold their CUs:
# the first (the stream's), the last, half, all but a few, all but one
@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("gemma", [False, True])
@pytest.mark.parametrize("absent", [(), (0,), (255, 7), range(0, 256, 2),
                                    range(8, 256), range(1, 256)])
@pytest.mark.parametrize("H,I,A,Q", [(128, 256, 128, 192),
                                     (1152, 2048, 640, 1290),
                                     (2304, 2560, 2048, 2310)])
def test_rows_are_taken_over(ho, wt, gemma, absent, H, I, A, Q):
    l = Layer(ho, wt, H, I, A, Q, gemma)
    want = l.run()
    l.chain._claims = c = claims(ho, absent)
    for a, b in zip(want, l.run()):
        assert torch.equal(a, b)
    # bit 0: it has started; bit 1: another block has its rows
    assert not (c & 1).any()
    gone = torch.zeros(256, dtype=torch.bool, device="cuda")
    gone[list(absent)] = True
    assert ((c & 2 == 0) == gone).all()


@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("V", [130, 66000])
def test_outputs_are_taken_over(ho, wt, V):
    """And the largest of their shares."""
    l = Layer(ho, wt, 256, 768, 256, V, head=30.0)
    want = l.run()
    tops = torch.full((ho.CHAIN_TOPS,), 1e9, device="cuda")
    l.chain._stages[3].tops = tops.data_ptr()
    for absent in ((), (1, 255), range(0, 256, 2), range(16, 256)):
        tops.fill_(1e9)
        l.chain._claims = claims(ho, absent)
        for a, b in zip(want, l.run()):
            assert torch.equal(a, b)
        per = -(-V // ho.CHAIN_BLOCKS)
        for b in (0, 1, 2, 64, 255):
            rows = want[3][b * per:max(b * per, min(V, (b + 1) * per))]
            assert tops.view(-1, 4)[b].max() == \
                (rows.max() if rows.numel() else float("-inf"))


def test_refused(ho):
    l = Layer(ho, 0, 128, 256, 128, 192)
    long = Layer(ho, 0, 4352, 256, 128, 192)  # a norm of more than 4096
    assert not long.chain.fits()
    with pytest.raises(RuntimeError):
        long.chain.run()
    with pytest.raises(RuntimeError):
        l.chain.run(limit=-1)
    l.chain._stages[1].y = None
    with pytest.raises(RuntimeError):
        l.chain.run()


# the middle that leaves a ring three slots, and two: right but slower than a
# launch for each product
@pytest.mark.parametrize("wt,three,two", [(0, 45056, 52224),
                                          (1, 23552, 27648),
                                          (2, 21504, 25600)])
def test_few_slots(ho, wt, three, two):
    for I, slots in ((three, 3), (two, 2)):
        l = Layer(ho, wt, 4096, I, 256, 192)
        assert ho.lib().chain_slots(l.chain._stages, 4, wt) == slots
        assert l.chain.fits() == (slots == 3)
        l.check(l.run())


def test_values_that_are_no_numbers(ho):
    """inf and NaN go through, and end no wait."""
    for bad in (float("inf"), float("nan")):
        for wt in (0, 1):
            l = Layer(ho, wt, 256, 512, 256, 192)
            l.att[3] = bad
            o, mid, dn, qkv, _ = l.run()
            assert not o.isfinite().any()
            assert mid.isnan().all() and dn.isnan().all()
            assert qkv[:192].isnan().all()


def test_chain_in_a_graph(ho):
    l = Layer(ho, 0, 2048, 2048, 2048, 3072)
    want = l.run()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        l.buf.fill_(255)
        l.chain.run()
    for i in range(4):
        l.qkv.zero_()
        l.buf.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(l.qkv, want[3])
        rand(i, 1000).sum().item()


def test_two_at_a_time(ho):
    """Blocks of two launches share the CUs: each ends, with its own bits."""
    ls = [Layer(ho, wt, 1024, 2048, 1024, 1536, seed=30 * wt)
          for wt in (0, 1)]
    want = [l.run() for l in ls]
    streams = [torch.cuda.Stream() for _ in ls]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for _ in range(20):
        for l, s in zip(ls, streams):
            with torch.cuda.stream(s):
                l.buf.fill_(255)
                l.chain.run()
    torch.cuda.synchronize()
    for l, w in zip(ls, want):
        for a, b in zip(w, (l.o, l.mid, l.dn, l.qkv)):
            assert torch.equal(a, b)


def test_engines_on_two_streams(ho):
    """Two models at once, each in a thread with a stream of its own: what
    each answers alone."""
    import threading

    import llm_np_cp_amd as L
    from llm_np_cp_amd.io.loader import random_weights
    from llm_np_cp_amd.models.engine import GPUModel

    ms = []
    for hidden, dtype in ((1024, "bf16"), (2048, "fp8")):
        cfg = L.ModelConfig(
            model_type="llama", vocab_size=512, hidden_size=hidden,
            intermediate_size=2 * hidden, num_hidden_layers=3,
            num_attention_heads=8, num_key_value_heads=4, head_dim=128)
        ms.append(GPUModel(cfg, random_weights(cfg, seed=3), max_seq=700,
                           dtype=dtype))
        assert ms[-1]._chains is not None

    def answer(m, to):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                ids = m.generate_tokens([3, 1, 4, 1, 5], 200)
                to.append((ids, m.b_logits.clone()))
            torch.cuda.synchronize()

    got = [[], [], [], []]
    for m, to in zip(ms, got):
        answer(m, to)
    ts = [threading.Thread(target=answer, args=a) for a in zip(ms, got[2:])]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for alone, beside in zip(got[:2], got[2:]):
        for (i, z), (j, y) in zip(alone, beside):
            assert i == j and torch.equal(z, y)


class Experts(Layer):
    """Routed experts between W_o and the next layer's q, k and v."""

    def __init__(self, ho, wt, H, I, E, top, seed=0, tie=False):
        super().__init__(ho, wt, H, I, 256, 192, seed=seed)
        st = self.chain._held
        act = F32 if wt else BF
        self.E, self.top = E, top
        self.wg = rand(seed + 20, E, H, scale=H ** -0.5).bfloat16()
        if tie:
            self.wg[:] = self.wg[0]
        up, dn = weight(ho, wt, seed + 21, E * 2 * I, H), \
            weight(ho, wt, seed + 22, E * H, I)
        self.Wup, self.Wdn = up[1].view(E, 2 * I, H), dn[1].view(E, H, I)
        kinds = [(H, BF), (H, BF)] + [(I, act)] * top + [(H, F32)] * (top - 1)
        size = [ho.chain_room(*k) for k in kinds]
        self.buf = torch.zeros(sum(size), dtype=U8, device="cuda")
        self.o, self.dn, *rest = (
            ho.chain_part(self.buf, sum(size[:k]), *v)
            for k, v in enumerate(kinds))
        self.mids, self.parts = rest[:top], rest[top:]
        new = [dict(st[0], y=self.o)]
        for j in range(top):
            new.append(dict(W=up[0], x=self.o, y=self.mids[j], glu=True,
                            kind=ho.CHAIN_NORM, g=self.g[0], experts=E,
                            slot=j + 1))
        new[1].update(route=self.wg, top=top)
        for j in range(top):
            last = j == top - 1
            new.append(dict(W=dn[0], x=self.mids[j], experts=E, slot=j + 1,
                            y=self.dn if last else self.parts[j], scaled=True,
                            add=self.o if last else None,
                            add2=self.parts[0] if last and top > 1 else None))
        new.append(dict(st[3], x=self.dn))
        self.chain = ho.Chain(new, wt, 0, 1e-5)

    def run(self, **kw):
        super().run(**kw)
        return [t.clone() for t in [self.o, self.dn, self.qkv] + self.mids +
                self.parts]

    def check(self, out):
        top, wt = self.top, self.wt
        o, dn, qkv, *rest = (t.double() for t in out)
        mids, parts = rest[:top], rest[top:]

        def norm(x):
            return x / torch.sqrt((x * x).mean() + 1e-5)

        def near(got, want, far, bf):
            far = far + want.abs() * 2.0 ** -8 * bf + 1e-30
            assert ((got - want).abs() <= far).all(), \
                ((got - want).abs() / far).max()

        def dot(w, x, bf=True):               # and its error, as in Layer
            return w @ x, w.abs() @ x.abs() * (
                2.0 ** -9 * (bf and wt == 0) + x.numel() * 2.0 ** -23 +
                2.0 ** -19)

        z, far = dot(self.W[0][1], self.att.double(), False)
        near(o, z + self.h.double(), far, True)
        x = norm(o) * self.g[0].double()
        p = torch.softmax(self.wg.double() @ x, 0)
        pw, pe = torch.sort(p, descending=True, stable=True)
        pw, pe = pw[:top] / pw[:top].sum(), pe[:top].tolist()
        want, err = self.o.double() * 0, 0
        for j in range(top):
            I = mids[j].numel()
            z, far = dot(self.Wup[pe[j]], x)
            t = z[:I].clone().requires_grad_()
            s = torch.nn.functional.silu(t)
            s.sum().backward()
            s = s.detach()
            near(mids[j], s * z[I:], (t.grad.abs() * far[:I] + far[:I] ** 2) *
                 (z[I:].abs() + far[I:]) + s.abs() * (
                     far[I:] + 2.0 ** -18 * z[I:].abs()), wt == 0)
            z, far = dot(self.Wdn[pe[j]], mids[j], False)
            want, err = want + pw[j] * z, err + pw[j] * far + \
                2.0 ** -16 * z.abs()
            if j < top - 1:
                near(parts[j], want, err, False)
        near(dn, want + o, err, True)
        z, far = dot(self.W[3][1], norm(dn) * self.g[1].double())
        near(qkv[:192], z + self.bias.double(), far, True)


@pytest.mark.parametrize("wt", [0, 1])
@pytest.mark.parametrize("H,I,E,top", [
    (256, 512, 8, 2), (1152, 640, 3, 2), (2048, 4096, 8, 2),
    (2304, 1280, 5, 1), (4096, 2048, 8, 2), (128, 256, 1, 1)])
def test_experts(ho, wt, H, I, E, top):
    for seed in (0, 100, 200):
        l = Experts(ho, wt, H, I, E, top, seed)
        assert l.chain.fits()
        first = l.run()
        l.check(first)
        for kw in ({}, dict(limit=0)):
            for a, b in zip(first, l.run(**kw)):
                assert torch.equal(a, b)


@pytest.mark.parametrize("wt", [0, 1])
@pytest.mark.parametrize("E,top", [(8, 2), (3, 2), (5, 1)])
def test_experts_are_taken_over(ho, wt, E, top):
    l = Experts(ho, wt, 1152, 640, E, top)
    want = l.run()
    for absent in ((0,), range(1, 256, 2), range(16, 256)):
        l.chain._claims = claims(ho, absent)
        for a, b in zip(want, l.run()):
            assert torch.equal(a, b)


def test_experts_alike(ho):
    """The first of equals, as ``moe_route`` has it; and none that is not
    there where the router's input is no number."""
    l = Experts(ho, 0, 256, 512, 8, 2, tie=True)
    l.check(l.run())
    l.att[3] = float("nan")
    o, dn, qkv, *rest = l.run()
    assert not dn.isfinite().any() and qkv[:192].isnan().all()


def test_experts_refused(ho):
    for field, bad in (("experts", 9), ("top", 3), ("top", 0), ("slot", 2),
                       ("kind", 0)):
        l = Experts(ho, 0, 256, 512, 8, 2)
        setattr(l.chain._stages[1], field, bad)
        with pytest.raises(RuntimeError):
            l.chain.run()


# blocks of many rows, of a few, with none; waves without a row
@pytest.mark.parametrize("wt", [0, 1, 2])
@pytest.mark.parametrize("V", [130, 512, 66000, 128256])
def test_largest_outputs(ho, wt, V):
    l = Layer(ho, wt, 256, 768, 256, V, head=30.0)
    tops = torch.full((ho.CHAIN_TOPS,), 1e9, device="cuda")
    l.chain._stages[3].tops = tops.data_ptr()
    out = l.run()
    l.check(out)
    assert tops.max() == out[3][:V].max()
    per = -(-V // ho.CHAIN_BLOCKS)            # a block's rows, its waves'
    for b in (0, 1, V // per - 1, ho.CHAIN_BLOCKS - 1):
        rows = out[3][b * per:min(V, (b + 1) * per)]
        assert tops.view(-1, 4)[b].max() == \
            (rows.max() if rows.numel() else float("-inf"))
    l.chain._stages[0].tops = tops.data_ptr()  # of the last, in fp32
    with pytest.raises(RuntimeError):
        l.chain.run()


# one trip of a block through its logits and more; shares of none
@pytest.mark.parametrize("V,n", [(1, 1), (7, 3), (2048, 1024), (2049, 1024),
                                 (32000, 1024), (300001, 1024)])
@pytest.mark.parametrize("temperature", [1.0, 0.3])
def test_picks_by_shares(ho, V, n, temperature):
    """The picks that a pass through all logits ahead gives, and the counter
    that it leaves."""
    logits = 3 * rand(V, V)
    for bad in (None, float("-inf"), float("nan")):
        if bad is not None:
            logits[V // 2] = bad
        tops = torch.full((n,), float("-inf"), device="cuda")
        for i, share in enumerate(logits.chunk(n)):
            tops[i] = share[~share.isnan()].max() if \
                (~share.isnan()).any() else float("-inf")
        got = []
        for kw in ({}, dict(tops=tops)):
            st = [torch.zeros(k, dtype=dt, device="cuda") for k, dt in (
                (1, torch.int64), (1, torch.int64), (1, torch.int64),
                (1, torch.int32), (64, torch.int32), (1, torch.int32),
                (1, torch.int32))]
            for _ in range(40):
                ho.sample(logits, 0.1, False, 5, *st, bump_len=True,
                          temperature=temperature, **kw)
            got.append(st)
        for a, b in zip(*got):
            assert torch.equal(a, b)
        assert got[0][0].item() == 40


def test_shares_of_more_rows_refused(ho):
    z = [torch.zeros(2, dtype=dt, device="cuda") for dt in (
        torch.int64, torch.int64, torch.int64, torch.int32, torch.int32,
        torch.int32, torch.int32, torch.int32)]
    with pytest.raises(RuntimeError):
        ho.sample(torch.zeros(2, 64, device="cuda"), 0.1, False, 5, *z[:7],
                  cnt=z[7], batch=2, tops=torch.zeros(4, device="cuda"))
