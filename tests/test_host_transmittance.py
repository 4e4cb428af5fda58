"""The exponents of the hits' transmittance factors (traverse.hip: set_factors, transmittance), from their
own source on the host, against 64 bits: every combination of LONG and SHORT queries and beams, photons,
grey and coloured media from thin to very thick (sigma_t 80, lengths to 2)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def cut(src, start, end):
    src = src[src.index(start):]
    return src[:src.index(end) + len(end)]


def test_exponents_against_64_bits(tmp_path):
    src = open(os.path.join(ROOT, "smallupbp_amd", "csrc", "traverse.hip")).read()
    body = cut(src, "struct SegState {", "\n};") + "\n" + cut(src, "__device__ __forceinline__ float pick3", "}\n")
    body += cut(src, "struct Trans {", "s.x2 * dq))};\n}\n")
    # u = 2^-24, E = sigma_t log2(e) in 64 bits, kLog2e within 0.25 u of log2(e). A LONG length's coefficient
    # is -E_c (1 + 1.25 u); a SHORT one's E_k - E_c to 2.25 u of itself, or where the other length is LONG
    # to 1.25 u (E_k + E_c) and one more rounding. The product and the sum round once more each: at most
    # 4 u E_c per LONG length (LONG beam, SHORT query: and 4 u E_k) and 5 u (E_k + E_c) per SHORT one, the
    # sum's rounding included. For c = k every SHORT coefficient is exactly 0 and a LONG one -E_k (1 + 1.25 u):
    # 4 u E_k per LONG length and nothing per SHORT length.
    code = """
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_exp2f(x) (x)  // the exponent itself
static const float kLog2e = 1.4426950408889634f;
%s
int main() {
    std::mt19937 rng(3);
    const auto uni = [&] { return rng() * (1.0f / 4294967296.0f); };
    const double u = std::ldexp(1.0, -24), log2e = 1.4426950408889634074;
    for (float thick : {0.5f, 3.f, 20.5f, 80.f})
        for (int n = 0; n < 200000; ++n) {
            float st[3];
            for (float& v : st) v = thick * (0.02f + uni());
            if (n %% 3 == 0) st[1] = st[2] = st[0];
            const int k = st[1] < st[0] ? (st[2] < st[1] ? 2 : 1) : (st[2] < st[0] ? 2 : 0);
            const float dq = 2.f * uni(), t2 = 2.f * uni();
            for (int mode = 0; mode < 6; ++mode) {
                const bool photon = mode >= 4, sq = mode & 1, sb = !photon && (mode & 2);
                SegState s;
                set_factors(s, st[0], st[1], st[2], k, sq);
                const Trans t = photon ? transmittance(s, dq) : transmittance(s, dq, t2, short_diff(sb, sq));
                const float got[3] = {t.c0, t.c1, t.c2};
                for (int c = 0; c < 3; ++c) {
                    const double Ec = st[c] * log2e, Ek = st[k] * log2e;
                    const double lb = photon ? 0.0 : (double)t2;
                    const double want = (sq ? Ek - Ec : -Ec) * dq + (sb ? Ek - Ec : -Ec) * lb;
                    const double lng = (sq ? 0.0 : dq) + (sb ? 0.0 : lb), sht = (sq ? dq : 0.0) + (sb ? lb : 0.0);
                    double bound = 4 * u * Ec * lng;
                    if (st[c] != st[k]) bound += 5 * u * (Ek + Ec) * sht + (sq && !sb ? 4 * u * Ek * lb : 0.0);
                    if (!(std::fabs(got[c] - want) <= bound)) {
                        std::printf("sigma_t %%g of %%g, mode %%d, lengths %%g %%g: %%.9g, not %%.9g within %%.3g\\n",
                                    st[c], st[k], mode, dq, t2, got[c], want, bound);
                        return 1;
                    }
                }
            }
        }
    return 0;
}
""" % body
    exe = str(tmp_path / "factors")
    (tmp_path / "factors.cpp").write_text(code)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", str(tmp_path / "factors.cpp"), "-o", exe])
    assert subprocess.call([exe]) == 0
