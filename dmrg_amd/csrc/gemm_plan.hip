// Operand descriptions of the pipelined GEMM: how K is cut into chunks and stages, which way the 16-byte units run, and
// the order in which a load's lanes walk memory.
#include "gemm_plan.hpp"

namespace dmrg {
namespace pipe {
namespace {

bool is_plain(const Idx2 &x) { return x.c == PLAIN; }
Idx2 scaled(Idx2 x, int64_t f) { return Idx2{x.s0 * f, x.s1 * f, x.c}; }
bool separable(const Idx2 &x, uint32_t ext) { return is_plain(x) || x.c % ext == 0 || ext % x.c == 0; }
// Whether u consecutive indices are contiguous from every multiple of u on (element strides).
bool unit_run(const Idx2 &x, int64_t ext, int u) { return u == 1 || (x.s0 == 1 && ext % u == 0 && (is_plain(x) || x.c % u == 0)); }

// How K is walked: nout chunks of nin consecutive values at strides in (and out from chunk to chunk) for both operands;
// or, where a small chunk divides the stage (ratio), as one chunk with the map's own offsets inside a stage.
struct Walk {
    int64_t nin, nout, a_in, a_out, b_in, b_out;
    bool    ratio;
};
// 128-byte lines that the 64 units of a load touch, walking K (korder) or the non-K index first.
int lines(const Idx2 &r, const Idx2 &k, bool korder, int ru, int ku, int kn) {
    const int nk = korder ? kn : 4, nr = 64 / nk;
    int64_t   slot[128], ro[64];
    std::fill(slot, slot + 128, int64_t(-1));
    for(int i = 0; i < nr; ++i) ro[i] = idx_off(r, i * ru);
    int count = 0;
    for(int j = 0; j < nk; ++j) {
        const int64_t ko = idx_off(k, j * ku);
        for(int i = 0; i < nr; ++i) {
            const int64_t line = (ro[i] + ko) / 128;
            uint32_t      h    = static_cast<uint32_t>(line ^ (line >> 7)) & 127;
            while(slot[h] != -1 && slot[h] != line) h = (h + 1) & 127;
            count += slot[h] == -1 ? 1 : 0;
            slot[h] = line;
        }
    }
    return count;
}

// es: element size; maps r (extent R) and k in elements; in/out: the walk's strides of this operand.
bool operand(Operand &o, const void *p, int64_t batch, const Idx2 &r, const Idx2 &k, const Walk &w, int64_t in, int64_t out, int64_t R, bool conj,
             bool ro, int es, int RT, int BK) {
    const int u = 16 / es;
    o.p         = p;
    o.batch     = batch * es;
    o.r         = scaled(r, es);
    o.R         = static_cast<int32_t>(R);
    o.sign      = conj ? -1.0f : 1.0f;
    if(w.ratio && !is_plain(k)) {
        o.k     = scaled(k, es);
        o.kstep = BK / static_cast<int64_t>(k.c) * o.k.s1;
        o.kwrap = 0;
    } else {
        o.k                  = Idx2{in * es, 0, PLAIN};
        const int64_t stages = (w.nin + BK - 1) / BK;
        o.kstep              = BK * o.k.s0;
        o.kwrap              = out * es - stages * o.kstep;
    }
    magic(o.r.c, o.rmul, o.rsh);
    magic(o.k.c, o.kmul, o.ksh);
    o.sep_r  = separable(o.r, static_cast<uint32_t>(RT));
    return span(o.r, o.sep_r ? std::min<int64_t>(R, RT) : R) + span(o.k, BK) + 16 < static_cast<int64_t>(0x7fffffff);
}

// The order that touches fewer lines.
void set_order(Operand &o, bool ro, int u, int BK) {
    const int kn = ro ? BK : BK / u;
    o.korder     = lines(o.r, o.k, true, ro ? u : 1, ro ? 1 : u, kn) <= lines(o.r, o.k, false, ro ? u : 1, ro ? 1 : u, kn);
}

// All of a description but its operands' orders.
bool describe_units(const GemmDesc &g, const ShapeInfo &s, int ksplit, Launch &out, bool k_units) {
    const int  es = static_cast<int>(dtype_size(g.dtype)), u = 16 / es;
    const Idx2 am = normal(g.am, g.M), ak = normal(g.ak, g.K), bk = normal(g.bk, g.K), bn = normal(g.bn, g.N);
    for(const Idx2 &x : {am, ak, bk, bn})
        if(x.s0 < 0 || x.s1 < 0) return false;
    if(g.K <= 0 || g.M <= 0 || g.N <= 0) return false;
    Walk w{g.K, 1, ak.s0, 0, bk.s0, 0, false};
    if(!is_plain(ak) || !is_plain(bk)) {
        const uint32_t c = is_plain(ak) ? bk.c : ak.c;
        if(!is_plain(ak) && !is_plain(bk) && ak.c != bk.c) return false;
        if(g.K % c != 0) return false;
        const int64_t a1 = is_plain(ak) ? ak.s0 * c : ak.s1, b1 = is_plain(bk) ? bk.s0 * c : bk.s1, n = g.K / c;
        if(c < static_cast<uint32_t>(s.BK) && s.BK % c == 0) w.ratio = true;
        else if(static_cast<int64_t>(c) >= n) w = Walk{c, n, ak.s0, a1, bk.s0, b1, false};
        else w = Walk{n, c, a1, ak.s0, b1, bk.s0, false}; // the longer index inside: fewer padded stages
    }
    // Orientation: along K where units are contiguous there, else along the non-K index; else loads of 4 bytes.
    auto along_k = [&](const Idx2 &k, int64_t in) { return u == 1 || (w.nin % u == 0 && (w.ratio ? unit_run(k, g.K, u) : in == 1)); };
    const bool aK = along_k(ak, w.a_in), bK = along_k(bk, w.b_in);
    const bool aR = !k_units && s.TM % u == 0 && unit_run(am, g.M, u), bR = !k_units && s.TN % u == 0 && unit_run(bn, g.N, u);
    out.W  = (aK || aR) && (bK || bR) && reinterpret_cast<uintptr_t>(g.A) % 4 == 0 && reinterpret_cast<uintptr_t>(g.B) % 4 == 0 ? 16 : 4;
    out.ar = out.W == 16 && !aK;
    out.br = out.W == 16 && !bK;
    Desc &d = out.d;
    if(!operand(d.a, g.A, g.a_batch, am, ak, w, w.a_in, w.a_out, g.M, g.conjA != 0, out.ar, es, s.BM, s.BK)) return false;
    if(!operand(d.b, g.B, g.b_batch, bn, bk, w, w.b_in, w.b_out, g.N, g.conjB != 0, out.br, es, s.BN, s.BK)) return false;
    d.C                = g.C;
    d.cm               = normal(g.cm, g.M);
    d.cn               = normal(g.cn, g.N);
    d.c_batch          = g.c_batch;
    d.part             = g.part;
    d.M                = g.M;
    d.N                = g.N;
    d.accumulate       = g.accumulate;
    d.xcd_remap        = g.xcd_remap;
    d.wide             = out.W == 16;
    d.Kin              = static_cast<int32_t>(w.nin);
    d.stages_per_chunk = static_cast<int32_t>((w.nin + s.BK - 1) / s.BK);
    const int64_t st   = d.stages_per_chunk * w.nout;
    if(st >= (int64_t(1) << 30)) return false;
    d.stages           = static_cast<int32_t>(st);
    d.stages_per_slice = (d.stages + ksplit - 1) / ksplit;
    d.ksplit           = (d.stages + d.stages_per_slice - 1) / d.stages_per_slice;
    return true;
}

} // namespace

bool describe(const GemmDesc &g, const ShapeInfo &s, int ksplit, Launch &out, bool k_units) {
    if(!describe_units(g, s, ksplit, out, k_units)) return false;
    const int u = 16 / static_cast<int>(dtype_size(g.dtype));
    set_order(out.d.a, out.ar, u, s.BK);
    set_order(out.d.b, out.br, u, s.BK);
    return true;
}

int load_bytes(const GemmDesc &g, const ShapeInfo &s) {
    Launch l;
    return describe_units(g, s, 1, l, false) ? l.W : 4;
}

} // namespace pipe
} // namespace dmrg
