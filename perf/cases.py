"""Performance cases of the ASRN framework: what its users run, through the public API, over the sizes they run it at.

Kinds of case (the key 'tipo'):
  capa      one ASRN layer's forward and backward (ASRNLayer), the hot path of training
  bloque    one local block's forward and backward (BloqueLocal), the model's other half
  perdida   the loss over a vocabulary, forward and backward (ops.cross_entropy)
  entreno   a whole training step replayed by PasoGrafado (forward, loss, backward, clipping, AdamW)
  prompt    a model's prompt through ModelWriter and the first generated step after it
  paso      one layer's O(1) generation step (LayerWriter with its graph)
  escribir  whole generation calls (escribir) with sampling

The layer and block steps are captured once in a HIP graph and replayed, as PasoGrafado does with a whole step: that is
how a training loop on this framework runs them, and the launches stay in the measured time while Python does not.
Weights are moved off their neutral starts (synth.move_params), tokens are the benchmark's synthetic text (uniform
or Zipf ids with copied spans). exact() restates every path in float64 with plain torch.
"""
import math

import torch
import torch.nn.functional as F

import asrn_amd
from asrn_amd import ops, synth

DEV = 'cuda'
C, T, NB, TC, CF, K, N_VISTOS = 32, 8, 14, 4, 16, 4, 4      # the layer's default options


def listed():
    return [
        # the smallest call: one short text at the default width (a unit test, a toy model): launches count
        dict(name='capa_minima', tipo='capa', B=1, L=200, d=64, V=256, bits=32),
        # the layer benchmark's shape: byte-level text, float32
        dict(name='capa_media', tipo='capa', B=8, L=4096, d=256, V=256, bits=32),
        # texts of an odd length at a width that is no power of two
        dict(name='capa_irregular', tipo='capa', B=3, L=1537, d=384, V=8000, bits=32),
        # long texts in bf16: what the layer's constant cost per token is for
        dict(name='capa_larga', tipo='capa', B=2, L=32768, d=512, V=32000, bits=16),
        # a local block of the d = 768 model at its training batch, bf16
        dict(name='bloque_ancho', tipo='bloque', B=8, L=2048, d=768, ff=1536, bits=16),
        # a local block in float32 on ragged texts
        dict(name='bloque_irregular', tipo='bloque', B=5, L=1001, d=256, ff=512, bits=32),
        # the loss of a language model over its vocabulary, bf16 logits
        dict(name='perdida', tipo='perdida', N=8192, V=32768, bits=16),
        # the quick-start model's training step: small kernels only
        dict(name='entreno_pequeno', tipo='entreno', B=8, L=256, d=64, V=256, n_capas=2, bits=32),
        # a d = 768 language model's training step in bf16, two blocks deep
        dict(name='entreno_ancho', tipo='entreno', B=8, L=2048, d=768, V=32768, n_capas=2, bits=16),
        # serving: the prompts of a batch and the first generated token
        dict(name='prompt', tipo='prompt', B=4, L=3000, d=768, V=32768, n_capas=4),
        # serving: a generated token of one layer, 16 sequences
        dict(name='paso', tipo='paso', B=16, L=1024, d=768, V=32768),
        # serving: a whole generation call of the '12m' size with the default sampling
        dict(name='escribir', tipo='escribir', B=4, L=300, d=256, V=8000, n_capas=16, nuevos=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _alineado(L, bits):
    """16-bit batches come padded to a multiple of 16 positions."""
    return (L + 15) // 16 * 16 if bits == 16 else L


def draw(rng):
    tipo = rng.choice(['capa', 'capa', 'capa', 'bloque', 'bloque', 'perdida', 'entreno', 'prompt', 'paso'])
    d = rng.choice([64, 96, 256, 384, 512, 768])          # the widths of the named sizes, the benchmark and the tests
    V = rng.choice([256, 1000, 8000, 32000, 32768])
    bits = rng.choice([16, 32])
    if tipo == 'capa':
        fichas = _log(rng, 200, 32768)
        B = rng.choice([1, 2, 3, 4, 8])
        return dict(tipo=tipo, B=B, L=_alineado(max(16, fichas // B), bits), d=d, V=V, bits=bits)
    if tipo == 'bloque':
        fichas = _log(rng, 200, 16384)
        B = rng.choice([1, 2, 5, 8, 16])
        return dict(tipo=tipo, B=B, L=max(8, fichas // B), d=d, ff=2 * d, bits=bits)
    if tipo == 'perdida':
        return dict(tipo=tipo, N=_log(rng, 256, 8192), V=rng.randint(2000, 32768), bits=bits)
    if tipo == 'entreno':
        fichas = _log(rng, 500, 8192)
        B = rng.choice([2, 4, 8])
        return dict(tipo=tipo, B=B, L=_alineado(fichas // B, bits), d=rng.choice([64, 128, 256, 512]),
                    V=rng.choice([256, 1000, 8000]), n_capas=2, bits=bits)
    if tipo == 'prompt':
        return dict(tipo=tipo, B=rng.randint(1, 8), L=_log(rng, 30, 1500), d=rng.choice([64, 256, 512, 768]), V=8000,
                    n_capas=rng.choice([2, 3, 4]))
    return dict(tipo=tipo, B=rng.randint(1, 16), L=_log(rng, 50, 1024), d=d, V=V)


# ---------------------------------------------------------------------------------------------------------------------
# what a program has in hand
# ---------------------------------------------------------------------------------------------------------------------

def _fichas(B, L, V, seed):
    zipf = 1.1 if V > 1000 else None
    span = (min(8, max(1, L // 16)), min(64, max(2, L // 4)))
    return synth.tokens(B, L, V, frac=0.25, span=span, zipf=zipf, seed=seed).to(DEV)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _autocast(bits):
    return torch.autocast('cuda', dtype=torch.bfloat16, enabled=bits == 16, cache_enabled=False)


def _modelo(case, seed):
    m = asrn_amd.crear_modelo(case['V'], d=case['d'], n_capas=case['n_capas'], semilla=seed)
    for capa in m.largos:
        synth.move_params(capa, seed)
    return m.to(DEV)


def _capa(case, seed):
    torch.manual_seed(seed)
    return synth.move_params(asrn_amd.ASRNLayer(case['d']), seed).to(DEV)


def _entradas_capa(case, seed, L):
    x = _fichas(case['B'], L, case['V'], seed)
    g = _gen(seed + 100)
    E = torch.randn(case['V'], case['d'], generator=g, device=DEV)[x]
    h = torch.randn(case['B'], L, case['d'], generator=g, device=DEV)
    return x, E, h, torch.randn(case['B'], L, case['d'], generator=g, device=DEV)


def _bloque(case, seed):
    torch.manual_seed(seed)
    b = asrn_amd.BloqueLocal(case['d'], ff=case['ff']).to(DEV)
    g = _gen(seed + 100)
    forma = (case['B'], case['L'], case['d'])
    return b, torch.randn(forma, generator=g, device=DEV), torch.randn(forma, generator=g, device=DEV)


def _logits(case, seed):
    g = _gen(seed)
    lg = 2.0 * torch.randn(case['N'], case['V'], generator=g, device=DEV)
    y = torch.randint(0, case['V'], (case['N'],), generator=g, device=DEV)
    return lg.to(torch.bfloat16 if case['bits'] == 16 else torch.float32), y


def _con_gradiente(m, bits):
    """The parameters whose gradients a training step's case returns: all in float32. In 16 bits the matrices: a
    scalar's gradient there is a sum over every position of 16-bit terms that nearly cancel (up to 0.3 off float64)."""
    return {n: p for n, p in m.named_parameters() if bits == 32 or p.numel() >= 2048}


def _grabar(paso):
    """paso() captured in a HIP graph after two ordinary runs on a side stream: (graph, its outputs)."""
    lado = torch.cuda.Stream()
    lado.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(lado):
        for _ in range(2):
            paso()
    torch.cuda.current_stream().wait_stream(lado)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        salida = paso()
    return g, salida


def _paso_modulo(modulo, entradas, fijas, gy, bits):
    """Forward and backward of a module on inputs that need gradients (and others that do not): a function giving the
    output, the inputs' gradients and the parameters'."""
    nombres, ps = zip(*modulo.named_parameters())
    entradas = [t.requires_grad_() for t in entradas]

    def paso():
        with _autocast(bits):
            y = modulo(*entradas, *fijas)
        gs = torch.autograd.grad(y, entradas + list(ps), gy.to(y.dtype))
        out = {'y': y.detach(), 'entradas': list(gs[:len(entradas)])}
        out.update(zip(nombres, gs[len(entradas):]))
        return out
    return paso


def prepare(case, seed):
    tipo = case['tipo']
    if tipo == 'capa':
        x, E, h, gy = _entradas_capa(case, seed, case['L'])
        capa = _capa(case, seed)               # the graph reads the weights and the inputs in place: the state keeps them
        g, salida = _grabar(_paso_modulo(capa, [E, h], [x], gy, case['bits']))
        return dict(tipo=tipo, grafo=g, salida=salida, vivos=(capa, x, E, h, gy))
    if tipo == 'bloque':
        b, h, gy = _bloque(case, seed)
        g, salida = _grabar(_paso_modulo(b, [h], [], gy, case['bits']))
        return dict(tipo=tipo, grafo=g, salida=salida, vivos=(b, h, gy))
    if tipo == 'perdida':
        lg, y = _logits(case, seed)
        return dict(tipo=tipo, lg=lg.requires_grad_(), y=y)
    if tipo == 'entreno':
        m = _modelo(case, seed).train()
        opt = asrn_amd.crear_optimizador(m, lr=1e-6, capturable=True)
        paso = asrn_amd.PasoGrafado(m, opt, case['B'], case['L'], precision='bf16' if case['bits'] == 16 else 'fp32')
        w = _fichas(case['B'], case['L'] + 1, case['V'], seed)
        x, y = w[:, :-1].contiguous(), w[:, 1:].contiguous()
        for _ in range(4):                     # the ordinary steps and the capture, with the weights left as they are
            paso(x, y, lr=0.0)
        return dict(tipo=tipo, paso=paso, x=x, y=y, params=_con_gradiente(m, case['bits']))
    if tipo == 'prompt':
        w = _fichas(case['B'], case['L'] + 1, case['V'], seed)
        return dict(tipo=tipo, m=_modelo(case, seed).eval(), x=w[:, :-1].contiguous(), sig=w[:, -1].contiguous())
    if tipo == 'paso':
        x, E, h, _ = _entradas_capa(case, seed, case['L'] + 1)
        esc = asrn_amd.LayerWriter(_capa(case, seed).eval(), memoria_de_lo_ajeno=False, grafo=True)
        with torch.no_grad():
            esc.inicio(E[:, :-2].contiguous(), h[:, :-2].contiguous(), x[:, :-2].contiguous(), capacidad=16384)
            esc.paso(E[:, -2], h[:, -2], x[:, -2])             # the first step runs op by op, the next is captured
        return dict(tipo=tipo, esc=esc, e=E[:, -1].contiguous(), h=h[:, -1].contiguous(), x=x[:, -1].contiguous())
    if tipo == 'escribir':
        return dict(tipo=tipo, m=_modelo(case, seed).eval(), x=_fichas(case['B'], case['L'], case['V'], seed),
                    nuevos=case['nuevos'], semilla=seed)
    raise ValueError(f'tipo={tipo!r}')


def run(state):
    tipo = state['tipo']
    if tipo in ('capa', 'bloque'):
        state['grafo'].replay()
        return state['salida']
    if tipo == 'perdida':
        p = ops.cross_entropy(state['lg'], state['y'])
        return {'perdida': p.detach(), 'dlogits': torch.autograd.grad(p, state['lg'])[0]}
    if tipo == 'entreno':
        perdida, norma, _ = state['paso'](state['x'], state['y'], lr=1e-6)      # the warm-up's first rate
        return {'perdida': perdida, 'norma': norma, 'grad': {n: p.grad for n, p in state['params'].items()}}
    if tipo == 'prompt':
        esc = asrn_amd.ModelWriter(state['m'], memoria_de_lo_ajeno=False)
        ultimo = esc.inicio(state['x'])
        return {'prompt': ultimo, 'paso': esc.paso(state['sig'])}
    if tipo == 'paso':
        return state['esc'].paso(state['e'], state['h'], state['x'])
    texto, logits = asrn_amd.escribir(state['m'], state['x'], n_nuevos=state['nuevos'], semilla=state['semilla'])
    return {'texto': texto, 'logits': logits}


# ---------------------------------------------------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------------------------------------------------

M_HASH = 64          # hidden units of each hash MLP


def _pesos_capa(d):
    return 3 * M_HASH * d + 2 * M_HASH * (T * NB // 2) + 2 * d * d + 2 * CF * d + 8 * d


def _trabajo_capa(fichas, d, b):
    """(bytes, flops) of a layer's forward: E and h in, h' out, the weights; the products, and the candidates' scores
    and value sums (about 20 distinct candidates a query)."""
    return (8 * d + b * d) * fichas + 4 * _pesos_capa(d), 2 * fichas * (_pesos_capa(d) - d * d + 20 * (T * NB + CF + d))


def _trabajo_bloque(fichas, d, ff):
    pesos = 4 * d * d + 2 * d * ff
    return 8 * d * fichas + 4 * pesos, 2 * fichas * pesos


def work(case):
    tipo = case['tipo']
    b = case.get('bits', 32) // 8
    if tipo == 'perdida':
        return dict(bytes=2 * b * case['N'] * case['V'], flops=6 * case['N'] * case['V'])
    d = case['d']
    fichas = case['B'] * (1 if tipo == 'paso' else case['L'])
    if tipo == 'capa':
        by, fl = _trabajo_capa(fichas, d, 4)
        return dict(bytes=3 * by, flops=3 * fl)
    if tipo == 'bloque':
        by, fl = _trabajo_bloque(fichas, d, case['ff'])
        return dict(bytes=3 * by, flops=3 * fl)
    if tipo == 'paso':
        by, fl = _trabajo_capa(fichas, d, 4)
        return dict(bytes=by + 4 * case['B'] * 20 * (T * NB + CF + d), flops=fl)
    n, V = case['n_capas'], case['V']
    largos = len(range(0, n - 1, 2))
    bc, fc = _trabajo_capa(fichas, d, 4)
    bb, fb = _trabajo_bloque(fichas, d, 2 * d)
    pesos = n * (4 * d * d + 4 * d * d) + largos * _pesos_capa(d) + V * d
    if tipo == 'entreno':
        return dict(bytes=3 * (n * bb + largos * bc + 2 * b * fichas * V) + 28 * pesos,
                    flops=3 * (n * fb + largos * fc + 2 * fichas * V * d))
    if tipo == 'prompt':
        return dict(bytes=n * bb + largos * bc + 4 * pesos, flops=n * fb + largos * fc + 4 * case['B'] * V * d)
    q = case['nuevos']
    return dict(bytes=n * bb + largos * bc + 4 * (q + 1) * pesos,
                flops=n * fb + largos * fc + 2 * q * case['B'] * pesos)


def tolerance(case):
    """About four times what the paths differ by from float64 over several seeds (the worst output of a case: in the
    layer and the training step a scalar parameter's gradient, a sum over all positions that nearly cancels)."""
    tipo = case['tipo']
    if case.get('bits') == 16:
        return {'capa': {'rel': 0.03, 'max': 0.7}, 'bloque': {'rel': 0.018, 'max': 0.1},
                'perdida': {'rel': 0.008, 'max': 0.016}, 'entreno': {'rel': 0.03, 'max': 0.99}}[tipo]
    # the layer, alone or in a model: a hash output within rounding of 0 may fall on either side, about one a pass at
    # the layer benchmark's shape, and the positions of that token then sit in another bucket (6e-5 to 3e-3 seen)
    if tipo in ('capa', 'entreno'):
        return {'rel': 1e-2, 'max': 0.9}
    return {'rel': {'bloque': 8e-6, 'paso': 5e-6}.get(tipo, 1e-5)}


# ---------------------------------------------------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------------------------------------------------

def _hash64(p, E, f=torch.float64):
    """The hash MLPs' outputs (B, L, T * NB) in the type f."""
    lin = lambda x, n: F.linear(x, p[n + '.weight'].to(f), p[n + '.bias'].to(f))
    E = E.to(f)
    clave = torch.cat([E, F.pad(E, (0, 0, 1, 0))[:, :E.shape[1]]], -1)
    return torch.cat([lin(F.gelu(lin(E, 'afin_palabra.0')), 'afin_palabra.2'),
                      lin(F.gelu(lin(clave, 'afin_contexto.0')), 'afin_contexto.2')], -1)


def _recurrencia(a, b):
    """S_i = a_i S_{i-1} + b_i over the last axis, by doubling."""
    s = 1
    while s < b.shape[-1]:
        b = torch.cat([b[..., :s], b[..., s:] + a[..., s:] * b[..., :-s]], -1)
        a = torch.cat([a[..., :s], a[..., s:] * a[..., :-s]], -1)
        s *= 2
    return b


def _sufijo(x):
    """(B, L, K): the tokens before each position, -1 before the text."""
    return torch.stack([F.pad(x, (j, 0), value=-1)[:, :x.shape[1]] for j in range(1, K + 1)], -1)


def _repeticion64(p, x, beta, Bt, log_alfa):
    B, L = x.shape
    s = x.double()
    clave, claves = torch.zeros_like(s), []
    for j in range(N_VISTOS):
        clave = clave + F.pad(s, (j, 0), value=float('nan'))[:, :L] * p['c_vistos'][j]
        claves.append(clave)
    k = torch.stack(claves, 1)                                                             # (B, n, L)
    ks, orden = torch.sort(k, dim=-1, stable=True)
    rep = F.pad((ks[..., 1:] == ks[..., :-1]), (1, 0)).double()
    Bo = torch.gather(Bt.unsqueeze(1).expand(-1, N_VISTOS, -1), -1, orden)
    ao = torch.gather(log_alfa.exp().unsqueeze(1).expand(-1, N_VISTOS, -1), -1, orden)
    dB = F.pad((Bo[..., 1:] - Bo[..., :-1]).clamp(min=0), (1, 0))
    a = rep * torch.exp(-p['log_kappa'].exp().unsqueeze(-1) * dB)
    lam = _recurrencia(a, a * F.pad(ao[..., :-1], (1, 0)))
    hawkes = torch.zeros_like(lam).scatter(-1, orden, lam).transpose(1, 2)
    vistos = torch.zeros_like(rep).scatter(-1, orden, rep).transpose(1, 2)
    r = vistos[..., -1]
    return vistos, hawkes, _recurrencia(r * torch.exp(-p['log_kappa_racha'].exp() * beta), r)


def _tabla64(q, k, v, Qc, Kc, Bt, log_alfa, w_suf, tasa, t, pos, ok, suf):
    """One table's attention of the queries t over their candidates pos (n, C): (n, d), the best score and weight."""
    n, c = pos.shape
    fila = lambda m: m.index_select(0, pos.reshape(-1)).view(n, c, -1)
    sc = (fila(k) @ q[t].unsqueeze(-1)).squeeze(-1) / math.sqrt(T * NB)
    sc = sc + (fila(Kc) @ Qc[t].unsqueeze(-1)).squeeze(-1) * CF ** -0.5
    ell = (suf[t].unsqueeze(1) == suf[pos]).logical_and(suf[pos] >= 0).long().cumprod(-1).sum(-1)
    sc = sc + w_suf[ell] + log_alfa[pos] + (Bt[pos] - Bt[t].unsqueeze(-1)) * tasa
    hay = ok.any(-1, keepdim=True)
    sc = sc.masked_fill(~ok, -math.inf).masked_fill(~hay, 0.0)
    att = torch.softmax(sc, -1) * hay
    out = (att.unsqueeze(1) @ fila(v)).squeeze(1)
    return out, sc.detach().amax(-1), att.detach().amax(-1)


def _candidatos64(phi, ids, V, Qc, Kc, Bt, log_alfa, x, w_suf, gamma):
    B, L, _ = phi.shape
    suf = _sufijo(x)
    salida, sen = [], []
    paso = 8192
    for b in range(B):
        filas = []
        for t0 in range(0, L, paso):
            t = torch.arange(t0, min(L, t0 + paso), device=x.device)
            suma, pt, pc, pico = 0.0, 0.0, 0.0, 0.0
            mejor = torch.full((len(t),), -1e9, dtype=torch.float64, device=x.device)
            for tau in range(T):
                orden = torch.argsort(ids[b, :, tau], stable=True)
                rango = torch.empty_like(orden).scatter_(0, orden, torch.arange(L, device=x.device))
                i = rango[t].unsqueeze(-1) - torch.arange(1, C + 1, device=x.device)
                pos = orden[i.clamp(min=0)]
                ok = (i >= 0) & (ids[b, :, tau][pos] == ids[b, t, tau].unsqueeze(-1))
                out, mx, pk = torch.utils.checkpoint.checkpoint(
                    _tabla64, phi[b], phi[b], V[b], Qc[b], Kc[b], Bt[b], log_alfa[b], w_suf, gamma[tau] / C, t, pos, ok,
                    suf[b], use_reentrant=False)
                hay = ok.any(-1)
                suma, pt, pico = suma + out, pt + hay.double(), pico + pk * hay
                mejor = torch.where(hay, torch.maximum(mejor, mx), mejor)
                pc = pc + hay.double() * (tau >= T - TC)
            filas.append((suma, torch.stack([pt, mejor, pico, pc], -1)))
        salida.append(torch.cat([f[0] for f in filas]))
        sen.append(torch.cat([f[1] for f in filas]))
    return torch.stack(salida), torch.stack(sen)


def _capa64(p, E, h, x, ids16):
    """The layer in float64. ids16: the buckets from 16-bit products, as under autocast (a sign near 0 is whatever the
    rounding says); the values are not rounded."""
    hh = F.layer_norm(h, h.shape[-1:], p['ln_ctx.weight'], p['ln_ctx.bias'])
    Qc, Kc = F.linear(hh, p['cq.weight']), F.linear(hh, p['ck.weight'])
    u = F.linear(hh, p['w_reloj'], p['b_reloj'])
    beta = F.softplus(u[..., 0]).clamp(max=1e4)
    log_alfa = (F.logsigmoid(u[..., 1]) + math.log(2)).clamp(min=-30.0)
    Bt = beta.cumsum(1)
    phi = _hash64(p, E)
    with torch.no_grad():
        bits = (_hash64(p, E, torch.bfloat16) if ids16 else phi).view(*phi.shape[:2], T, NB) > 0
        ids = (bits.long() << torch.arange(NB, device=x.device)).sum(-1)
    V = F.pad(F.linear(E, p['v.weight']), (0, 0, 0, 1))[:, 1:]
    salida, sen = _candidatos64(phi, ids, V, Qc, Kc, Bt, log_alfa, x, p['w_sufijo'], p['gamma'])
    vistos, hawkes, racha = _repeticion64(p, x, beta, Bt, log_alfa)
    pt = sen[..., :1]
    mejor = torch.where(pt > 0, sen[..., 1:2], torch.zeros_like(pt)).clamp(-1e4, 1e4)
    s = torch.cat([pt / T, mejor, sen[..., 2:3] / pt.clamp(min=1), sen[..., 3:] / TC], -1)
    logit = F.linear(h, p['g.weight'], p['g.bias']) + F.linear(s, p['g_conf.weight'], p['g_conf.bias'])
    logit = logit + (vistos * p['w_vistos']).sum(-1, keepdim=True)
    logit = logit + (torch.log1p(hawkes) * p['u_hawkes']).sum(-1, keepdim=True)
    dr = p['d_racha']
    r = (torch.log1p(racha) / (math.log1p(256) / (len(dr) - 1))).clamp(max=len(dr) - 1)
    i = r.detach().floor().long().clamp(0, len(dr) - 2)
    logit = logit + (dr.cumsum(0)[i] + (r - i) * dr[1:][i]).unsqueeze(-1)
    return h + torch.sigmoid(logit) * F.linear(salida / pt.clamp(min=1), p['o.weight'])


def _bloque64(p, h):
    d = h.shape[-1]
    z = F.layer_norm(h, (d,), p['ln1.weight'], p['ln1.bias'])
    w = p['conv.weight']
    k = w.shape[-1]
    zp = F.pad(z, (0, 0, k - 1, 0))
    c = sum(F.linear(zp[:, j:j + z.shape[1]], w[..., j]) for j in range(k)) + p['conv.bias']
    h = h + F.gelu(c)
    y = F.layer_norm(h, (d,), p['ln2.weight'], p['ln2.bias'])
    return h + F.linear(F.gelu(F.linear(y, p['ff.0.weight'], p['ff.0.bias'])), p['ff.2.weight'], p['ff.2.bias'])


def _de(p, prefijo):
    return {n[len(prefijo):]: v for n, v in p.items() if n.startswith(prefijo)}


def _logits64(p, x, n_capas, ids16):
    """The model's state before the head's product, and the head's matrix."""
    E = p['emb.weight'][x]
    h, j = E, 0
    for i in range(n_capas):
        h = _bloque64(_de(p, f'bloques.{i}.'), h)
        if i % 2 == 0 and i < n_capas - 1:
            h = _capa64(_de(p, f'largos.{j}.'), E, h, x, ids16)
            j += 1
    return F.layer_norm(h, h.shape[-1:], p['ln_f.weight'], p['ln_f.bias'])


def _doble(m, grad):
    p = {n: v.detach().double() for n, v in m.state_dict().items() if n != 'head.weight'}
    for n, v in m.named_parameters():
        if n in p:
            p[n].requires_grad_(grad)
    return p


def _exacto_modulo(f, modulo, entradas, gy):
    p = _doble(modulo, True)
    entradas = [t.double().requires_grad_() for t in entradas]
    y = f(p, *entradas)
    nombres = [n for n, _ in modulo.named_parameters()]
    gs = torch.autograd.grad(y, entradas + [p[n] for n in nombres], gy.double())
    out = {'y': y.detach(), 'entradas': list(gs[:len(entradas)])}
    out.update(zip(nombres, gs[len(entradas):]))
    return out


def exact(case, seed):
    tipo = case['tipo']
    if tipo == 'capa':
        x, E, h, gy = _entradas_capa(case, seed, case['L'])
        return _exacto_modulo(lambda p, E, h: _capa64(p, E, h, x, case['bits'] == 16), _capa(case, seed), [E, h], gy)
    if tipo == 'bloque':
        b, h, gy = _bloque(case, seed)
        return _exacto_modulo(_bloque64, b, [h], gy)
    if tipo == 'perdida':
        lg, y = _logits(case, seed)
        lg = lg.double().requires_grad_()
        p = F.cross_entropy(lg, y)
        return {'perdida': p.detach(), 'dlogits': torch.autograd.grad(p, lg)[0]}
    if tipo == 'entreno':
        m = _modelo(case, seed)
        p = _doble(m, True)
        w = _fichas(case['B'], case['L'] + 1, case['V'], seed)
        h = _logits64(p, w[:, :-1].contiguous(), case['n_capas'], case['bits'] == 16)
        perdida = F.cross_entropy(F.linear(h, p['emb.weight']).flatten(0, 1), w[:, 1:].reshape(-1))
        nombres = [n for n, _ in m.named_parameters()]
        gs = torch.autograd.grad(perdida, [p[n] for n in nombres])
        norma = torch.stack([g.square().sum() for g in gs]).sum().sqrt()
        gs = [g * (1.0 / (norma + 1e-6)).clamp(max=1.0) for g in gs]
        gs = dict(zip(nombres, gs))
        return {'perdida': perdida.detach(), 'norma': norma, 'grad': {n: gs[n] for n in _con_gradiente(m, case['bits'])}}
    with torch.no_grad():
        if tipo == 'prompt':
            m = _modelo(case, seed)
            p = _doble(m, False)
            w = _fichas(case['B'], case['L'] + 1, case['V'], seed)
            h = _logits64(p, w, case['n_capas'], False)
            lg = F.linear(h[:, -2:], p['emb.weight'])
            return {'prompt': lg[:, 0], 'paso': lg[:, 1]}
        if tipo == 'paso':
            x, E, h, _ = _entradas_capa(case, seed, case['L'] + 1)
            return _capa64(_doble(_capa(case, seed), False), E.double(), h.double(), x, False)[:, -1]
    return None                # sampled text: a draw has no float64 value
