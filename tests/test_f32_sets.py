"""Which of the two sets of fp32 kernels the launches of a problem go to.  (Host code alone: the selection of sjvp_f32.hip is compiled
and run here, with launches that note the set.)"""
import random
import subprocess

from semicat_amd import build

MAIN = r"""
#include <cstdio>
#include "sjvp_f32.hip"
namespace sjvp {
static char used;  // p: three bf16 parts, u: fp32 unit
int fwd_f32x3(const FwdParamsF32&, int, bool, int, hipStream_t) { used = 'p'; return SJVP_OK; }
int bwd_f32x3(const BwdParamsF32&, int, bool, bool, int, int, hipStream_t) { used = 'p'; return SJVP_OK; }
}
extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { sjvp::used = 'u'; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* n, hipDeviceAttribute_t, int) { *n = 256; return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { return nullptr; }  // there is no device code
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}
int main() {
    int BH, Lq, Lk, D;
    while (scanf("%d %d %d %d", &BH, &Lq, &Lk, &D) == 4) {
        sjvp::FwdParamsF32 f{};
        sjvp::BwdParamsF32 b{};
        f.H = b.H = 1, f.Lq = b.Lq = Lq, f.Lk = b.Lk = Lk, f.D = b.D = D, f.Lr = b.Lr = (Lq + 127) / 128 * 128;
        char sets[9] = {}, *s = sets;
        for (bool tangents : {true, false}) sjvp::fwd_f32(f, BH, tangents, nullptr), *s++ = sjvp::used;
        for (int cot : {3, 2, 1})  // dO and dTO, dTO, dO
            for (int part : {SJVP_BWD_ROW, SJVP_BWD_COL}) sjvp::bwd_f32(b, BH, cot & 1, cot & 2, part, nullptr), *s++ = sjvp::used;
        puts(sets);
    }
}
"""


def test_all_launches_of_a_shape_come_from_one_set(tmp_path):
    (tmp_path / "sets.hip").write_text(MAIN)
    subprocess.run([build.hipcc_path(), "-std=c++20", "-O0", "-w", "--cuda-host-only", "-Wl,--unresolved-symbols=ignore-all",
                    "-I" + build.CSRC, "-x", "hip", str(tmp_path / "sets.hip"), "-o", str(tmp_path / "sets")], check=True, capture_output=True)
    rng = random.Random(1)
    shapes = [(256, 200, 32, 100), (249, 172, 172, 128), (120, 76, 76, 80), (768, 128, 128, 64), (8, 256, 256, 64), (1, 1, 1, 16)]
    for _ in range(6000):
        size = [int(round(2 ** rng.uniform(a, b))) for a, b in ((0, 11), (3, 12), (3, 12))]
        size[2] = size[1] if rng.random() < 0.5 else size[2]
        shapes.append((*size, rng.choice((16, 20, 21, 32, 36, 48, 64, 67, 80, 96, 100, 128))))
    out = subprocess.run([str(tmp_path / "sets")], input="".join("%d %d %d %d\n" % s for s in shapes), check=True, capture_output=True, text=True)
    sets = dict(zip(shapes, out.stdout.split(), strict=True))
    assert set(sets.values()) == {"p" * 8, "u" * 8}, [s for s in sets.items() if len(set(s[1])) > 1][:5]
    assert sets[(768, 128, 128, 64)] == "p" * 8 and sets[(8, 256, 256, 64)] == sets[(1, 1, 1, 16)] == "u" * 8
