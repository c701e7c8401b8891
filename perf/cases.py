"""The work that users of this framework have it do, as measurable cases.

A pass is one training step without the optimizer's own update (zero the gradients, register the model and the loss call,
``forward_and_backward()``), or, for a user who holds Kronecker factors already, the damped inverses and the
product with a gradient.  The models are the architectures of the benchmark and the tests at random initialisation; the
ranges behind ``draw`` go from layers of a few units to 4096 x 4096 and from 16 rows to 8192.

Keys of a case:
  kind       'kfac' | 'shampoo' (gradient makers), 'kron' (factors in hand: Kron.update_inv + Kron.mvp)
  model      'mlp' | 'resnet' (CIFAR stem, basic blocks) | 'resnet50' (bottlenecks) | 'decoder'
  widths     layer widths of an MLP, 'in-hidden-...-out'; of 'kron', the (A, B) sizes of each layer 'AxB-AxB'
  refresh    True: curvature and its inverses / roots are renewed in the pass; False: a step between two renewals
"""
import torch
import torch.nn as nn
import torch.nn.functional as F

from asdl_amd import (FISHER_EMP, FISHER_MC, KfacGradientMaker, Kron, PreconditioningConfig, ShampooGradientMaker)

NEVER = 10 ** 9
MOST_OUTPUTS = 64
NEWTON_STEPS = 18        # of the coupled iteration at the ridge and tolerance used here


# ------------------------------------------------------------------------------------------------ models
class _Basic(nn.Module):
    def __init__(self, cin, cout, stride):
        super().__init__()
        self.conv1, self.bn1 = nn.Conv2d(cin, cout, 3, stride, 1, bias=False), nn.BatchNorm2d(cout)
        self.conv2, self.bn2 = nn.Conv2d(cout, cout, 3, 1, 1, bias=False), nn.BatchNorm2d(cout)
        self.short = nn.Sequential()
        if stride != 1 or cin != cout:
            self.short = nn.Sequential(nn.Conv2d(cin, cout, 1, stride, bias=False), nn.BatchNorm2d(cout))

    def forward(self, x):
        y = self.bn2(self.conv2(F.relu(self.bn1(self.conv1(x)))))
        return F.relu(y + self.short(x))


class _Bottleneck(nn.Module):
    def __init__(self, cin, width, stride):
        super().__init__()
        cout = 4 * width
        self.conv1, self.bn1 = nn.Conv2d(cin, width, 1, bias=False), nn.BatchNorm2d(width)
        self.conv2, self.bn2 = nn.Conv2d(width, width, 3, stride, 1, bias=False), nn.BatchNorm2d(width)
        self.conv3, self.bn3 = nn.Conv2d(width, cout, 1, bias=False), nn.BatchNorm2d(cout)
        self.short = nn.Sequential()
        if stride != 1 or cin != cout:
            self.short = nn.Sequential(nn.Conv2d(cin, cout, 1, stride, bias=False), nn.BatchNorm2d(cout))

    def forward(self, x):
        y = F.relu(self.bn2(self.conv2(F.relu(self.bn1(self.conv1(x))))))
        return F.relu(self.bn3(self.conv3(y)) + self.short(x))


class _Resnet(nn.Module):
    def __init__(self, block, expansion, base, depths, classes, imagenet_stem):
        super().__init__()
        self.pool = imagenet_stem
        self.conv1 = nn.Conv2d(3, base, 7, 2, 3, bias=False) if imagenet_stem else nn.Conv2d(3, base, 3, 1, 1, bias=False)
        self.bn1 = nn.BatchNorm2d(base)
        cin, stages = base, []
        for i, depth in enumerate(depths):
            width = base << i
            for j in range(depth):
                stages.append(block(cin, width, 2 if i and not j else 1))
                cin = width * expansion
        self.body, self.fc = nn.Sequential(*stages), nn.Linear(cin, classes)

    def forward(self, x):
        x = F.relu(self.bn1(self.conv1(x)))
        if self.pool:
            x = F.max_pool2d(x, 3, 2, 1)
        return self.fc(F.adaptive_avg_pool2d(self.body(x), 1).flatten(1))


class _DecoderBlock(nn.Module):
    def __init__(self, d, heads):
        super().__init__()
        self.heads = heads
        self.ln_1, self.c_attn, self.c_proj = nn.LayerNorm(d), nn.Linear(d, 3 * d), nn.Linear(d, d)
        self.ln_2, self.c_fc, self.c_out = nn.LayerNorm(d), nn.Linear(d, 4 * d), nn.Linear(4 * d, d)

    def forward(self, x):
        b, t, d = x.shape
        q, k, v = (z.view(b, t, self.heads, d // self.heads).transpose(1, 2) for z in self.c_attn(self.ln_1(x)).split(d, 2))
        y = F.scaled_dot_product_attention(q, k, v, is_causal=True)
        x = x + self.c_proj(y.transpose(1, 2).reshape(b, t, d))
        return x + self.c_out(F.gelu(self.c_fc(self.ln_2(x))))


class _Decoder(nn.Module):
    """Token embedding and output head are frozen, so that no statistic is as wide as the vocabulary."""

    def __init__(self, vocab, d, layers, heads, context):
        super().__init__()
        self.wte, self.wpe = nn.Embedding(vocab, d), nn.Parameter(torch.empty(context, d))
        self.h = nn.Sequential(*(_DecoderBlock(d, heads) for _ in range(layers)))
        self.ln_f, self.head = nn.LayerNorm(d), nn.Linear(d, vocab, bias=False)
        for m in self.modules():
            if isinstance(m, (nn.Linear, nn.Embedding)):
                nn.init.normal_(m.weight, std=0.02)
        nn.init.normal_(self.wpe, std=0.02)
        self.wte.weight.requires_grad_(False)
        self.head.weight.requires_grad_(False)

    def forward(self, idx):
        return self.head(self.ln_f(self.h(self.wte(idx) + self.wpe[:idx.shape[1]]))).flatten(0, 1)


def _widths(case):
    return [int(w) for w in case['widths'].split('-')]


def _model(case):
    if case['model'] == 'mlp':
        w = _widths(case)
        layers = []
        for i, (a, b) in enumerate(zip(w, w[1:])):
            layers += [nn.Linear(a, b)] + ([nn.ReLU()] if i < len(w) - 2 else [])
        return nn.Sequential(*layers)
    if case['model'] == 'resnet':
        return _Resnet(_Basic, 1, case['base'], [case['blocks']] * case['stages'], case['classes'], False)
    if case['model'] == 'resnet50':
        return _Resnet(_Bottleneck, 4, 64, [3, 4, 6, 3], case['classes'], True)
    return _Decoder(case['classes'], case['d'], case['layers'], case['heads'], case['tokens'])


def _input_shape(case):
    if case['model'] == 'mlp':
        return (case['batch'], _widths(case)[0])
    if case['model'] == 'decoder':
        return (case['batch'], case['tokens'])
    return (case['batch'], 3, case['image'], case['image'])


def _classes(case):
    return _widths(case)[-1] if case['model'] == 'mlp' else case['classes']


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    mlp = dict(kind='kfac', model='mlp', widths='784-512-512-10', batch=128, fisher='mc', bf16=False, ema=-1.0, damping=1e-3,
               refresh=True, norms=False, swift=False)
    linear = dict(mlp, widths='4096-4096', batch=8192, bf16=True, ema=0.95)
    net = dict(kind='kfac', fisher='mc', ema=-1.0, damping=1e-3, refresh=True, norms=False, swift=False)
    resnet18 = dict(net, model='resnet', base=64, stages=4, blocks=2, classes=10, image=32, batch=128, bf16=False)
    resnet50 = dict(net, model='resnet50', classes=1000, image=224, batch=64, bf16=True, damping=3e-2)
    decoder = dict(net, model='decoder', d=768, heads=12, layers=2, tokens=1024, batch=8, classes=50257, bf16=True, ema=0.95,
                   norms=True, fisher='emp', damping=1e-2)
    shampoo = dict(kind='shampoo', model='decoder', d=768, heads=12, layers=12, tokens=1024, batch=8, classes=50257, bf16=True,
                   ema=-1.0, damping=1e-6)
    return [
        # the smallest step in use: most steps of a run lie between two renewals and only precondition
        dict(mlp, name='kfac_mlp_between_renewals', refresh=False),
        # the same network with everything renewed in the step: dozens of small launches
        dict(mlp, name='kfac_mlp'),
        # widths of tabular data: nothing a multiple of anything, moving average, empirical Fisher
        dict(mlp, name='kfac_mlp_ragged', widths='1021-677-301-17', batch=1000, fisher='emp', ema=0.95),
        # one large layer: the widest factors and inverses of the range
        dict(linear, name='kfac_linear4096'),
        # the CIFAR network in fp32, NCHW
        dict(resnet18, name='kfac_resnet18_fp32'),
        # the headline: ImageNet network, bf16 autocast, channels last
        dict(resnet50, name='kfac_resnet50_bf16'),
        # fewer samples than columns: factors kept as row matrices, with the 2 x 2 blocks of the BatchNorm layers
        dict(resnet18, name='skfac_resnet18', batch=64, swift=True, norms=True),
        # transformer layers with their LayerNorm blocks, moving average
        dict(decoder, name='kfac_decoder'),
        # Shampoo on a small network, roots renewed in the step
        dict(shampoo, name='shampoo_mlp', model='mlp', widths='784-512-512-10', batch=128, bf16=False, refresh=True),
        # Shampoo on a decoder of GPT-2-small shape: a step that renews the roots, and one between two renewals
        dict(shampoo, name='shampoo_decoder_roots', refresh=True),
        dict(shampoo, name='shampoo_decoder_between_roots', refresh=False),
        # factors in hand (loaded, or accumulated elsewhere): inverses and product, layer by layer
        dict(name='kron_inverse_and_product', kind='kron', widths='1153x512-577x1000-300x75-64x10', damping=1e-3),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(['kfac mlp', 'kfac mlp', 'kfac resnet', 'kfac decoder', 'shampoo mlp', 'shampoo decoder', 'kron'])
    if kind == 'kron':
        pairs = [(_log_int(rng, 8, 2500), _log_int(rng, 8, 1500)) for _ in range(rng.randint(1, 6))]
        return dict(kind='kron', widths='-'.join('%dx%d' % p for p in pairs), damping=rng.choice([1e-2, 1e-3]))
    maker, model = kind.split()
    case = dict(kind=maker, model=model, bf16=rng.random() < 0.5, ema=rng.choice([-1.0, 0.95]), refresh=rng.random() < 0.75)
    if maker == 'kfac':
        case.update(fisher=rng.choice(['mc', 'emp']), damping=rng.choice([1e-2, 1e-3]), norms=rng.random() < 0.5, swift=False)
    else:
        case.update(damping=1e-6)
    if model == 'mlp':
        widths = [_log_int(rng, 12, 2048) for _ in range(rng.randint(2, 5))]
        case.update(widths='-'.join(map(str, widths)), batch=_log_int(rng, 16, 4096))
    elif model == 'resnet':
        case.update(base=rng.choice([16, 20, 24, 32, 48, 64]), stages=rng.randint(1, 3), blocks=rng.randint(1, 2), classes=_log_int(rng, 10, 200),
                    image=rng.randint(14, 40), batch=_log_int(rng, 8, 128), swift=rng.random() < 0.25)
        if case['swift']:
            case.update(ema=-1.0, bf16=False)
        elif case['bf16']:
            case.update(damping=3e-2, refresh=True)
    else:
        heads = rng.randint(2, 12)
        case.update(heads=heads, d=64 * heads, layers=rng.randint(1, 3), tokens=_log_int(rng, 33, 1024), batch=rng.randint(1, 8), classes=_log_int(rng, 500, 20000))
    return case


# ------------------------------------------------------------------------------------------------ a user's program
def _spectrum(d, rng):
    """A covariance as a layer's rows give it: a few strong directions over a floor."""
    rows = torch.randn(2 * d, d, device='cuda', generator=rng) * torch.logspace(0, -2, d, device='cuda')
    return rows.t() @ rows / (2 * d)


def prepare(case, seed):
    rng = torch.Generator('cuda').manual_seed(seed)
    if case['kind'] == 'kron':
        layers = []
        for pair in case['widths'].split('-'):
            da, db = map(int, pair.split('x'))
            layers.append((Kron(_spectrum(da, rng), _spectrum(db, rng)), torch.randn(db, da, device='cuda', generator=rng),
                           torch.randn(db, device='cuda', generator=rng)))
        return dict(case=case, layers=layers)
    torch.manual_seed(seed)
    with torch.device('cuda'):
        model = _model(case)
    shape, classes = _input_shape(case), _classes(case)
    if case['model'] == 'decoder':
        x = torch.randint(0, classes, shape, device='cuda', generator=rng)
        t = torch.randint(0, classes, (case['batch'] * case['tokens'],), device='cuda', generator=rng)
    else:
        x = torch.randn(shape, device='cuda', generator=rng)
        t = torch.randint(0, classes, (case['batch'],), device='cuda', generator=rng)
    if len(shape) == 4 and case['bf16']:
        model, x = model.to(memory_format=torch.channels_last), x.contiguous(memory_format=torch.channels_last)

    def forward(inputs):
        with torch.autocast('cuda', dtype=torch.bfloat16, enabled=case['bf16']):
            return model(inputs).float()

    every = 1 if case['refresh'] else NEVER
    if case['kind'] == 'shampoo':
        maker = ShampooGradientMaker(model, PreconditioningConfig(
            damping=case['damping'], ema_decay=case['ema'], curvature_upd_interval=1, preconditioner_upd_interval=every))
        shown = [p for p in model.parameters() if p.requires_grad and p.ndim > 1]
    else:
        ignore = [] if case['norms'] else [nn.BatchNorm2d, nn.LayerNorm]
        maker = KfacGradientMaker(model, PreconditioningConfig(
            data_size=t.numel(), damping=case['damping'], ema_decay=case['ema'], preconditioner_upd_interval=every,
            ignore_modules=ignore), fisher_type=FISHER_MC if case['fisher'] == 'mc' else FISHER_EMP, seed=1, swift=case['swift'])
        shown = [p for m in maker.modules_for_curvature for p in m.parameters() if p.requires_grad]
    optimizer = torch.optim.SGD([p for p in model.parameters() if p.requires_grad], lr=0.1)
    state = dict(case=case, model=model, maker=maker, optimizer=optimizer, forward=forward, x=x, t=t, shown=shown)
    if not case['refresh']:
        run(state)              # the step that renewed the curvature lies behind
    return state


def _curvature(maker):
    """What a checkpoint would hold of the maker, as the live tensors."""
    if isinstance(maker, ShampooGradientMaker):
        return [q for p in maker.preconditioners for q in p.statistics + p.preconditioners]
    found = []
    for m in maker.modules_for_curvature:
        for part, names in ((m.fisher.kron, ('A', 'B', 'A_inv', 'B_inv')), (m.fisher.unit, ('data', 'inv'))):
            if part is not None:
                found += [getattr(part, n) for n in names if getattr(part, n) is not None]
    return found


def _noisy(case):
    """bf16 convolutions of the framework below add in another order on every run.  The activations differ in their last bit,
    some change sides at a ReLU, and the gradients of a random initialisation, sums of mostly cancelling terms, differ by a
    third between two runs of the same code; the damped inverses differ by a percent and are what can be compared."""
    return case['bf16'] and case['model'].startswith('resnet')


def run(state):
    case = state['case']
    if case['kind'] == 'kron':
        out = []
        for kron, weight, bias in state['layers']:
            kron.update_inv(case['damping'])
            out += [kron.A_inv, kron.B_inv, *kron.mvp(weight, bias, use_inv=True)]
        return out
    maker = state['maker']
    state['optimizer'].zero_grad()
    if case['kind'] == 'shampoo' and case['refresh']:
        torch.manual_seed(1)    # the start vectors of the power iteration
    logits = maker.setup_model_call(state['forward'], state['x'])
    maker.setup_loss_call(F.cross_entropy, logits, state['t'])
    _, loss = maker.forward_and_backward()
    out = [loss.detach()]
    if not _noisy(case):
        out += [p.grad for p in state['shown']]
    curvature = _curvature(maker)
    if _noisy(case) and len(out) + len(curvature) > MOST_OUTPUTS:
        return out + [torch.cat([c.flatten() for c in curvature])]      # packed, as for an exchange between ranks
    # the gradients depend on all of the curvature; it is shown too where the outputs are not too many
    return out + curvature if len(out) + len(curvature) <= MOST_OUTPUTS else out


# ------------------------------------------------------------------------------------------------ what a pass needs
def _layers(case):
    """(columns of A, columns of B, rows of A, rows of B, bias, trained) of every Linear / Conv2d of the model."""
    found = []
    with torch.device('meta'):
        model = _model(case)
        x = torch.zeros(_input_shape(case), dtype=torch.long) if case['model'] == 'decoder' else torch.zeros(_input_shape(case))

    def note(m, _, y):
        rows = y.numel() // (y.shape[1] if y.ndim == 4 else y.shape[-1])
        found.append((m.weight[0].numel(), m.weight.shape[0], rows, m.bias is not None, m.weight.requires_grad))
    for m in model.modules():
        if isinstance(m, (nn.Linear, nn.Conv2d)):
            m.register_forward_hook(note)
    with torch.no_grad():
        model(x)
    return model, found


def work(case):
    """Bytes: inputs, parameters, gradients, and the curvature that a pass reads and writes.  FLOP: the model's passes,
    symmetric statistics counted once (M d (d + 1)), d^3 per damped inverse, 4 n^3 per Newton step of a root (symmetric products)."""
    if case['kind'] == 'kron':
        pairs = [tuple(map(int, p.split('x'))) for p in case['widths'].split('-')]
        return {'bytes': sum(4 * (2 * a * a + 2 * b * b + 2 * a * b + 2 * b) for a, b in pairs),
                'flops': sum(a ** 3 + b ** 3 + 2 * a * b * (a + b) + 2 * b * b for a, b in pairs)}
    model, layers = _layers(case)
    params = sum(p.numel() for p in model.parameters())
    trained = sum(p.numel() for p in model.parameters() if p.requires_grad)
    size = 8 if case['model'] == 'decoder' else 4
    n_in = 1
    for s in _input_shape(case):
        n_in *= s
    flops, nbytes, fresh = 0, 4 * (params + trained) + size * n_in, case['refresh']
    for a, b, rows, bias, learns in layers:
        flops += rows * a * b * (6 if learns else 4)
        if not learns:
            continue
        if case['kind'] == 'shampoo':
            flops += a * b * (a + b + 2)                       # both statistics
        elif fresh:
            flops += rows * (a * (a + 1) + b * (b + 1))        # both factors
            if case['fisher'] == 'mc':
                flops += rows * a * b * 2                      # the sampled backward pass
        swift = case['kind'] == 'kfac' and case['swift']
        for d in (a, b):
            low = swift and case['batch'] < d                  # a row matrix: Gram matrix, its inverse, one product
            if fresh:
                if case['kind'] == 'shampoo':
                    flops += 4 * NEWTON_STEPS * d ** 3
                else:
                    flops += case['batch'] ** 3 + 3 * case['batch'] * d * d if low else d ** 3
            moved = (2 if case['kind'] == 'shampoo' else 2 if fresh and case['ema'] > 0 else 0) + 1
            nbytes += 4 * moved * d * d
        flops += 2 * a * b * (a + b) + (2 * b * b if bias else 0)
    return {'bytes': nbytes, 'flops': flops}


def tolerance(case):
    if case.get('bf16'):
        return {'rel': 2e-2 if _noisy(case) else 1e-2}      # activations, output gradients and their products round to 8 bits
    if case['kind'] == 'shampoo':
        return {'rel': 5e-3}      # inverse 4th roots of rank-deficient statistics in fp32, condition 1e6 after the ridge
    return {'rel': 1e-3}          # fp32 inverses of factors with a condition of up to about 1e4
