// Driver for the CPU emulation of k_carry_groups; the kernel's source is cut out
// of bluecrunch_amd/csrc/kernels.h by tests/test_carry_emulation.py into
// carry_cpu.h. LDS starts filled with a pattern, as a workgroup finds it on the
// device, and every index is checked against its size.
//   drv in out      in: C b K ng CL addl cover lds, group sums, addend
#include <fstream>

#include "carry_cpu.h"

int main(int argc, char **argv) {
  if (argc < 3) return 2;
  std::ifstream in(argv[1]);
  int C, b, K, cover;
  size_t ng, CL, addl, lds;
  in >> C >> b >> K >> ng >> CL >> addl >> cover >> lds;
  const int stride = (K + 3) & ~3;
  std::vector<uint4> sums(ng * stride / 4);
  std::vector<uint32_t> add(addl), out(CL, 0xabababab);
  uint32_t *y = reinterpret_cast<uint32_t *>(sums.data());
  for (size_t i = 0; i < ng * stride; i++) in >> y[i];
  for (uint32_t &x : add) in >> x;
  CarryArgs a{};
  a.bits = b;
  a.out = out.data();
  a.CL = CL;
  a.wpb = GCT * GWPT;
  a.nblk = (CL + a.wpb - 1) / a.wpb;
  std::vector<unsigned char> fn(a.nblk);
  a.blk_fn = fn.data();
  a.add = addl ? add.data() : nullptr;
  a.addl = addl;
  a.ybuf = y;
  a.gC = C;
  a.gK = K;
  a.gKs = stride;
  a.ng = (long long)ng;
  for (unsigned k = 0; k < a.nblk; k++) {
    g_lds.assign(lds, 0xdeadbeefu);
    run_grid(1, GCT, [&] {
      blockIdx.x = k;
      if (cover <= 2) k_carry_groups<2>(a);
      else if (cover == 3) k_carry_groups<3>(a);
      else k_carry_groups<4>(a);
    });
  }
  std::ofstream o(argv[2]);
  for (uint32_t w : out) o << w << '\n';
  for (unsigned char f : fn) o << (f >> 2) << '\n';  // open blocks
  return 0;
}
