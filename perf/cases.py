"""Workloads of the ZeRO-1 shard update, each one pass through the package's public entry points: what is timed and
compared when a kernel or a launch path changes.

A case is a dict of plain values.  ``kind`` says which program it stands for:

  shard    the flat-shard optimizer: clip_grad_norm(1.0) + step() on one GPU's FlatShard (or, with trainer, the
           trainer's sync-free update with its sample-size factor, flags and clip metric)
  owner    the same behind the owner-side sum: reduce_clip() over the ranks' BF16 contributions, then step()
  dropin   the reference's seams: CEReduce._sum per backward phase in the slot-major staging, the owned gradients as
           views of ``out``, zero1_fast.clip_grad_norm(1.0) and zero1_fast.step() through the fairseq stand-ins
  ampc     the reference's unfused sequence: one scale_up per tensor, then FusedAdamCast with amp_C's signature
  embed    the embedding owner's token gradient, in its three call forms

The model of the first four is ``layers`` blocks of ([dim, dim], [hidden, dim], [dim]), then [dim, dim] and, with
extra, a 1-D tensor of that many elements.  Inputs follow the distributions of the benchmark's configurations:
p ~ N(0, 0.02), m ~ N(0, 1e-4), v = |N(0, 1e-8)|, gradients N(0, 1e-4) or, with heavy, Student-t(2) x 1e-3.
"""
import math

import torch

LR, BETAS, EPS, WD, MAX_NORM, STEP = 3e-4, (0.9, 0.95), 1e-8, 0.1, 1.0, 1000
DEV = 'cuda'


def _f32(x):
    """A Python number as the kernels receive it: rounded once to fp32."""
    return float(torch.tensor(x, dtype=torch.float32))


# ------------------------------------------------------------------------------------------------------- the cases
def listed():
    c2 = dict(layers=12, dim=3072, hidden=8192, extra=5_952_768)         # 430,662,912 parameters in 38 tensors
    return [
        # the smallest update (the smoke test's 36,928 parameters): launches and host calls are all of it
        dict(name='shard 37k fp32', kind='shard', layers=1, dim=64, hidden=256, extra=12_288, grad='fp32',
             trainer=False, heavy=False),
        # a small odd-sized model in the trainer's form: BF16 gradients, every row a ragged tail and a gap
        dict(name='shard 1.8M odd bf16 trainer', kind='shard', layers=3, dim=391, hidden=1003, extra=30_011,
             grad='bf16', trainer=True, heavy=False),
        # the benchmark's plumbing configuration: 9,438,208 parameters
        dict(name='shard 9.4M fp32', kind='shard', layers=1, dim=1024, hidden=4096, extra=3_145_728, grad='fp32',
             trainer=False, heavy=False),
        # the headline: one GPU's share of YOCO-3B
        dict(name='shard 431M fp32', kind='shard', grad='fp32', trainer=False, heavy=False, **c2),
        # a middle-sized shard fed by four ranks, sizes off every boundary
        dict(name='owner 26M odd x4', kind='owner', layers=6, dim=1001, hidden=3001, extra=777_777, world=4),
        # the headline shard fed by the eight ranks' contributions
        dict(name='owner 431M x8', kind='owner', world=8, **c2),
        # the reference's own call sequence on a small model with odd sizes: parameters packed without padding
        dict(name='dropin 14M odd x8', kind='dropin', layers=8, dim=777, hidden=1333, extra=12_345, world=8, rank=3),
        # the same on the headline shard
        dict(name='dropin 431M x8', kind='dropin', world=8, rank=3, **c2),
        # scale pass per tensor + amp_C's Adam call, a quarter-width model
        dict(name='ampc 44M', kind='ampc', layers=20, dim=768, hidden=2048, extra=0),
        # the token gradient of the training recipe: 8 ranks x 2048 tokens, vocabulary 100,288
        dict(name='embed 16384x3072 uniform', kind='embed', rows=16_384, dim=3072, vocab=100_288, ids='uniform',
             form='owner', world=8, pad=1),
        # the same with text's skewed token frequencies, in the copy-engine path's order
        dict(name='embed 16384x3072 zipf', kind='embed', rows=16_384, dim=3072, vocab=100_288, ids='zipf', form='ce',
             world=8, pad=1),
        # a short batch on a small model: few rows (aten's other summation order), output and workspace kept
        dict(name='embed 2000x768 few', kind='embed', rows=2000, dim=768, vocab=32_000, ids='zipf', form='kept',
             world=4, pad=-1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_model(rng, lo, hi):
    """A model of lo to hi parameters: its width follows from a drawn size, depth and aspect ratio."""
    n, layers, ratio = _log_int(rng, lo, hi), rng.randint(1, 32), rng.uniform(1.5, 4.0)
    dim = max(8, int(math.sqrt(n / (layers * (1 + ratio) + 1))))
    if rng.random() < 0.6:
        dim = max(16, dim // 16 * 16)
    hidden = max(8, int(dim * ratio))
    if dim % 16 == 0:
        hidden = max(16, hidden // 16 * 16)
    extra = rng.choice([0, rng.randint(1, max(2, n // 50))])
    return dict(layers=layers, dim=dim, hidden=hidden, extra=extra)


def draw(rng):
    kind = rng.choice(['shard', 'shard', 'owner', 'dropin', 'ampc', 'embed'])
    if kind == 'shard':
        return dict(kind=kind, grad=rng.choice(['fp32', 'bf16']), trainer=rng.random() < 0.3, heavy=rng.random() < 0.3,
                    **_draw_model(rng, 3e4, 3.8e8))
    if kind == 'owner':
        return dict(kind=kind, world=rng.choice([2, 3, 4, 5, 8, 8]), **_draw_model(rng, 1e5, 3.8e8))
    if kind == 'dropin':
        world = rng.choice([2, 4, 7, 8])
        return dict(kind=kind, world=world, rank=rng.randrange(world), **_draw_model(rng, 1e5, 3.8e8))
    if kind == 'ampc':
        return dict(kind=kind, **_draw_model(rng, 1e5, 1.5e8))
    dim = _log_int(rng, 64, 4096)
    if rng.random() < 0.8:
        dim = dim // 8 * 8
    return dict(kind=kind, rows=_log_int(rng, 100, 32_768), dim=dim, vocab=_log_int(rng, 1000, min(131_072, 3e8 / dim)),
                ids=rng.choice(['uniform', 'zipf']), form=rng.choice(['owner', 'ce', 'kept']),
                world=rng.choice([2, 4, 8]), pad=rng.choice([-1, 1]))


def _shapes(case):
    d, h = case['dim'], case['hidden']
    s = [(d, d), (h, d), (d,)] * case['layers'] + [(d, d)]
    return s + [(case['extra'],)] if case['extra'] else s


def _numels(case):
    return [math.prod(s) for s in _shapes(case)]


# ------------------------------------------------------------------------------------------------------- the inputs
def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 64 + stream)
    return g


def _normal(n, std, gen, dtype=torch.float32):
    out = torch.empty(n, dtype=dtype, device=DEV)
    for i in range(0, n, 1 << 26):
        k = min(1 << 26, n - i)
        out[i:i + k] = torch.randn(k, generator=gen, device=DEV) * std
    return out


def _student(n, scale, gen):
    out = torch.empty(n, device=DEV)
    for i in range(0, n, 1 << 26):
        u = torch.rand(min(1 << 26, n - i), dtype=torch.float64, device=DEV, generator=gen)
        u.clamp_(2.0 ** -30, 1.0 - 2.0 ** -30)
        out[i:i + u.numel()] = (2.0 * u - 1.0) / torch.sqrt(2.0 * u * (1.0 - u)) * scale
    return out


def _state(case, seed):
    """p, m, v of the whole model, its tensors one after the other."""
    n = sum(_numels(case))
    return (_normal(n, 0.02, _gen(seed, 0)), _normal(n, 1e-4, _gen(seed, 1)),
            _normal(n, 1e-8, _gen(seed, 2)).abs_())


def _grad(case, seed):
    """The gradient of shard (fp32 values, rounded to BF16 for a BF16 shard) and ampc (BF16)."""
    n = sum(_numels(case))
    g = _student(n, 1e-3, _gen(seed, 3)) if case.get('heavy') else _normal(n, 1e-4, _gen(seed, 3))
    return g if case.get('grad') == 'fp32' else g.to(torch.bfloat16)


def _contribution(case, seed, k):
    return _normal(sum(_numels(case)), 1e-4, _gen(seed, 16 + k), torch.bfloat16)


SAMPLE_SIZE, NUMER, FACTOR = 1000.0, 8, 0.37


def _tokens(case, seed):
    gen = _gen(seed, 4)
    if case['ids'] == 'uniform':
        return torch.randint(0, case['vocab'], (case['rows'],), generator=gen, device=DEV)
    w = torch.arange(1, case['vocab'] + 1, dtype=torch.float64, device=DEV) ** -1.2
    return torch.multinomial(w, case['rows'], replacement=True, generator=gen)


def _token_grads(case, seed):
    return _normal(case['rows'] * case['dim'], 1e-2, _gen(seed, 5), torch.bfloat16).view(case['rows'], case['dim'])


# ------------------------------------------------------------------------------------------------------- prepare
def _spread(numels):
    """Offsets of separately allocated tensors within one buffer that holds them: each on 512 bytes of fp32, as torch's
    allocator places blocks, with a gap after it, so that a pass returns them as one tensor."""
    off, pos = [], 0
    for n in numels:
        off.append(pos)
        pos += (n + 127) // 128 * 128 + 128
    return off, pos


def _spread_copy(flat, numels, dtype=torch.float32):
    off, total = _spread(numels)
    buf = torch.zeros(total, dtype=dtype, device=DEV)
    pos = 0
    for o, n in zip(off, numels):
        if flat is not None:
            buf[o:o + n] = flat[pos:pos + n]
        pos += n
    return buf, [buf[o:o + n] for o, n in zip(off, numels)]


def _prepare_shard(case, seed):
    from faster_yoco_amd import shard, trainer_glue
    bf16 = case['kind'] == 'owner' or case['grad'] == 'bf16'
    sh = shard.FlatShard(_shapes(case), DEV, grad_dtype=torch.bfloat16 if bf16 else torch.float32)
    flats = dict(zip('pmv', _state(case, seed)))
    if case['kind'] == 'shard':
        flats['g'] = _grad(case, seed)
    for name, flat in flats.items():
        pos = 0
        for view in sh.views(name):
            view.copy_(flat[pos:pos + view.numel()].view_as(view))
            pos += view.numel()
    sh.p16.copy_(sh.p)
    opt = shard.Zero1ShardOptimizer(sh, lr=LR, betas=BETAS, eps=EPS, weight_decay=WD)
    opt.set_step(STEP - 1)
    st = dict(case=case, shard=sh, opt=opt)
    if case['kind'] == 'owner':
        st['contribs'] = []
        for k in range(case['world']):
            flat, c, pos = _contribution(case, seed, k), torch.zeros(sh.total, dtype=torch.bfloat16, device=DEV), 0
            for o, n in zip(sh.offsets, sh.numels):
                c[o:o + n] = flat[pos:pos + n]
                pos += n
            st['contribs'].append(c)
    elif case['trainer']:
        st['trainer'] = trainer_glue.TrainerUpdate(opt, clip_norm=MAX_NORM, numer=NUMER)
        st['sample_size'] = torch.full((1,), SAMPLE_SIZE, device=DEV)
    return st


def _phase_layout(numels):
    """CEReduce's layout of the owner's gradient: three backward phases (the model's last third first), each its
    tensors in model order.  (offset of each tensor, phase bounds)"""
    t = len(numels)
    phase = [2 if i < t // 3 else 1 if i < 2 * t // 3 else 0 for i in range(t)]
    where, bounds, pos = [0] * t, [[0, 0] for _ in range(3)], 0
    for ph in range(3):
        bounds[ph][0] = pos
        for i in range(t):
            if phase[i] == ph:
                where[i] = pos
                pos += numels[i]
        bounds[ph][1] = pos
    return where, bounds


def _prepare_dropin(case, seed):
    from faster_yoco_amd import ce_reduce, layout, standins, zero1_fast
    shapes, numels = _shapes(case), _numels(case)
    zero1_fast.configure(ENABLED=True, ALLGATHER=True, PARAM_VIEWS=True, REDUCE_OWNER=True, ONE_PASS=True,
                         SCALE_KERNEL=True, FUSED_ADAM=True, CE_ALLGATHER=False, FOLD_SCALE=False)
    mixin = type('Mixin', (standins.FakeMixin,), {})
    zero1_fast.install(mixin)
    p, m, v = _state(case, seed)
    params, pos = [], 0
    for s, n in zip(shapes, numels):
        params.append(torch.nn.Parameter(p[pos:pos + n].to(torch.bfloat16).view(s)))
        pos += n
    placed = layout.place_params(params, 1)
    zero1_fast._PLACED.clear()
    zero1_fast._PLACED.update(placed)
    opt = type('Opt', (mixin, standins.FakeFP16Optimizer), {})(params, lr=LR, betas=BETAS, eps=EPS, weight_decay=WD)
    bufs = {}
    bufs['p'], ps = _spread_copy(p, numels)
    bufs['m'], ms = _spread_copy(m, numels)
    bufs['v'], vs = _spread_copy(v, numels)
    bufs['g'], gs = _spread_copy(None, numels)
    adam = opt.fp32_optimizer.optimizer.optim
    adam.param_groups[0]['step'] = STEP - 1
    for p32, s, a, b, c, d in zip(opt.fp32_params, shapes, ps, ms, vs, gs):
        p32.data, p32.grad = a.view(s), d.view(s)
        adam.state[p32] = {'exp_avg': b.view(s), 'exp_avg_sq': c.view(s)}
    opt.zero_grad()                          # the optimizer's plan is made here, on this model's placement
    G, W, r = sum(numels), case['world'], case['rank']
    where, bounds = _phase_layout(numels)
    staging, out = torch.empty((W - 1) * G, dtype=torch.bfloat16, device=DEV), None
    for k in range(W):
        flat, pos = _contribution(case, seed, k), 0
        row = out = torch.empty(G, dtype=torch.bfloat16, device=DEV) if k == r else out
        if k != r:
            slot = k if k < r else k - 1
            row = staging[slot * G:(slot + 1) * G]
        for o, n in zip(where, numels):
            row[o:o + n] = flat[pos:pos + n]
            pos += n
    ce = ce_reduce.install(type('CEReduce', (standins.FakeCEReduce,), {}))(staging, out, G, bounds, r, W)
    views = [out[o:o + n].view(s) for o, n, s in zip(where, numels, shapes)]
    return dict(case=case, opt=opt, params=params, ce=ce, views=views, bufs=bufs, flat=placed['flat'])


def _prepare_ampc(case, seed):
    from faster_yoco_amd import fused_adam_cast
    numels = _numels(case)
    bufs, lists = {}, {}
    for name, flat in zip('pmv', _state(case, seed)):
        bufs[name], lists[name] = _spread_copy(flat, numels)
    bufs['g'], lists['g'] = _spread_copy(None, numels)
    bufs['p16'], p16 = _spread_copy(None, numels, torch.bfloat16)
    _, g16 = _spread_copy(_grad(case, seed), numels, torch.bfloat16)
    dest = {a.data_ptr(): b for a, b in zip(lists['p'], p16)}
    return dict(case=case, bufs=bufs, lists=lists, g16=g16, adam=fused_adam_cast.FusedAdamCast(dest),
                factor=torch.full((1,), FACTOR, device=DEV), step=STEP - 1)


def _prepare_embed(case, seed):
    from faster_yoco_amd import embedding
    st = dict(case=case, grad=_token_grads(case, seed), ids=_tokens(case, seed))
    if case['form'] == 'kept':
        st['call'] = embedding.OwnerEmbeddingGrad(case['rows'], case['dim'], case['vocab'], case['pad'], case['world'],
                                                  DEV)
    return st


def prepare(case, seed):
    import faster_yoco_amd  # noqa: F401
    with torch.no_grad():
        return dict(shard=_prepare_shard, owner=_prepare_shard, dropin=_prepare_dropin, ampc=_prepare_ampc,
                    embed=_prepare_embed)[case['kind']](case, seed)


# ------------------------------------------------------------------------------------------------------- one pass
def run(st):
    kind = st['case']['kind']
    if kind in ('shard', 'owner'):
        sh, opt = st['shard'], st['opt']
        out = {}
        if kind == 'owner':
            out['grad_norm'] = opt.reduce_clip(st['contribs'], MAX_NORM)
            opt.step()
            out['avg'] = sh.g
        elif 'trainer' in st:
            out['grad_norm'], out['clip'] = st['trainer'](st['sample_size'])
        else:
            out['grad_norm'] = opt.clip_grad_norm(MAX_NORM)
            opt.step()
        out.update(p=sh.p, m=sh.m, v=sh.v, p16=sh.p16)
        return out
    if kind == 'dropin':
        ce, opt = st['ce'], st['opt']
        for ph in range(3):
            ce._sum(ph)
        for p, g in zip(st['params'], st['views']):
            p.grad = g
        grad_norm = opt.clip_grad_norm(MAX_NORM)
        opt.step()
        opt.zero_grad()
        return dict(grad_norm=grad_norm, avg=ce.out, p16=st['flat'], **st['bufs'])
    if kind == 'ampc':
        from faster_yoco_amd.fused_adam_cast import scale_up
        ls = st['lists']
        for g16, g32 in zip(st['g16'], ls['g']):
            scale_up(g16, g32, st['factor'])
        st['step'] += 1
        st['adam'](2048 * 32, None, [ls['g'], ls['p'], ls['m'], ls['v']], LR, BETAS[0], BETAS[1], EPS, st['step'], 1, 1,
                   WD)
        st['adam'].cast.clear()
        return dict(st['bufs'])
    from faster_yoco_amd import embedding
    c = st['case']
    if c['form'] == 'kept':
        return st['call'](st['grad'], st['ids'])
    fn = embedding.owner_embedding_grad if c['form'] == 'owner' else embedding.ce_owner_embedding_grad
    return fn(st['grad'], st['ids'], c['vocab'], c['pad'], c['world'])


# ------------------------------------------------------------------------------------------------------- work
def work(case):
    """Every input read once and every output written once: p, m, v in and out (24 bytes a parameter), the BF16 copy
    (2), the gradient or the contributions in, and what the form returns beside them."""
    if case['kind'] == 'embed':
        r, d, v = case['rows'], case['dim'], case['vocab']
        return dict(bytes=r * d * 2 + r * 8 + v * d * 2, flops=r * d)
    n = sum(_numels(case))
    per = {'shard': 4 if case.get('grad') == 'fp32' else 2,
           'owner': 2 * case.get('world', 0) + 2,                 # contributions in, the average out
           'dropin': 2 * case.get('world', 0) + 2 + 4,            # and the FP32 master gradients out
           'ampc': 2 + 4}[case['kind']]
    return dict(bytes=n * (26 + per), flops=n * (20 + case.get('world', 0)))


# Against the sums taken in another order (contributions in reverse rank order; a token's occurrences in one running
# sum) no BF16 result in 2 million moved, and a norm one fp32 ulp off moves the moments by 1e-8 of their size: what is
# stated is four times a flip in ten thousand BF16 values, and for single values about two flips (2^-8 each).  At most
# 3072 rows a token's sum is rounded to BF16 after every 16 rows, so its error is that of BF16 running sums.
def tolerance(case):
    if case['kind'] == 'embed':
        return dict(rel=4e-3, max=0.04) if case['rows'] <= 3072 else dict(rel=1e-4, max=0.01)
    return dict(rel=2e-5 if case['kind'] in ('owner', 'dropin') else 1e-5, max=0.01)


# ------------------------------------------------------------------------------------------------------- in 64 bits
def _exact_update(case, seed, g, factor=1.0, clip=True):
    """The update of the whole model in float64 (its tensors one after the other): dict of p, m, v, g' and grad_norm.
    The hyperparameters are the fp32 numbers the kernels take."""
    p, m, v = (x.double() for x in _state(case, seed))
    out, f = {}, factor
    if clip:
        out['grad_norm'] = f * float(g.square().sum().sqrt())
        f = f * min(MAX_NORM / (out['grad_norm'] + 1e-6), 1.0)
    b1, b2 = _f32(BETAS[0]), _f32(BETAS[1])
    bc1, bc2 = _f32(1 - BETAS[0] ** STEP), _f32(1 - BETAS[1] ** STEP)
    g = g * f
    m.mul_(b1).add_(g, alpha=1 - b1)
    v.mul_(b2).addcmul_(g, g, value=1 - b2)
    upd = (m / bc1).div_((v / bc2).sqrt_().add_(_f32(EPS))).add_(p, alpha=_f32(WD))
    p.sub_(upd, alpha=_f32(LR))
    out.update(p=p, m=m, v=v, g=g)
    return out


def _place(flat, numels, offsets, total):
    out, pos = torch.zeros(total, dtype=flat.dtype, device=DEV), 0
    for o, n in zip(offsets, numels):
        out[o:o + n] = flat[pos:pos + n]
        pos += n
    return out


def _average(case, seed):
    """The owner sum's BF16 average: the sum in float64, rounded once (the values every later stage reads)."""
    acc = torch.zeros(sum(_numels(case)), dtype=torch.float64, device=DEV)
    for k in range(case['world']):
        acc += _contribution(case, seed, k)
    return acc.div_(case['world']).to(torch.bfloat16)


@torch.no_grad()
def exact(case, seed):
    if case['kind'] == 'embed':
        ids = _tokens(case, seed)
        out = torch.zeros(case['vocab'], case['dim'], dtype=torch.float64, device=DEV)
        out.index_add_(0, ids, _token_grads(case, seed).double())
        if case['pad'] >= 0:
            out[case['pad']] = 0
        return out.div_(case['world'])
    numels = _numels(case)
    if case['kind'] in ('shard', 'owner'):
        off, pos = [], 0
        for n in numels:                     # FlatShard's layout: every tensor on a 64-element boundary
            pos = (pos + 63) // 64 * 64
            off.append(pos)
            pos += n
        total = pos
        if case['kind'] == 'owner':
            avg = _average(case, seed)
            u = _exact_update(case, seed, avg.double())
        else:
            u = _exact_update(case, seed, _grad(case, seed).double(),
                              _f32(NUMER / SAMPLE_SIZE) if case['trainer'] else 1.0)
        out = dict(grad_norm=u['grad_norm'])
        if case['kind'] == 'owner':
            out['avg'] = _place(avg.double(), numels, off, total)
        elif case['trainer']:
            out['clip'] = 100.0 if u['grad_norm'] > MAX_NORM else 0.0
        for k in 'pmv':
            out[k] = _place(u[k], numels, off, total)
        out['p16'] = out['p']
        return out
    off, total = _spread(numels)
    if case['kind'] == 'dropin':
        avg = _average(case, seed).double()
        u = _exact_update(case, seed, avg)
        where, _ = _phase_layout(numels)
        out = dict(grad_norm=u['grad_norm'], avg=_place(avg, numels, where, sum(numels)), p16=u['p'])
    else:
        u = _exact_update(case, seed, _grad(case, seed).double(), _f32(FACTOR), clip=False)
        out = dict(p16=_place(u['p'], numels, off, total))
    for k in 'pmvg':
        out[k] = _place(u[k], numels, off, total)
    return out
