// The single-body velocity-stepping kernel's LDS layout on the host: in a
// workgroup of one to four waves, which of a wave's two programs (four and
// eight lanes an instance) a wave has reached does not depend on the other
// waves, so every value of either program has to lie in a part of LDS that no
// other wave uses, and rows and parked states of one program must not overlap.
// Prints the faults found and returns 1 if there are any.
#include "../../gorilla-physics_amd/csrc/gp_vstep_body.hip"

#include <vector>

namespace gp {
namespace {

constexpr int kNobody = -1;

template <int L>
int check(int block, std::vector<int>& wave_of) {
  const int total = (int)(body_lds_bytes<L>(block) / sizeof(double));
  int bad = 0;
  std::vector<int> owner(total, kNobody);  // of this program's values
  auto take = [&](int at, int n, int who, int wave) {
    for (int k = at; k < at + n; ++k) {
      if (k < 0 || k >= total) {
        ++bad;
        continue;
      }
      if (owner[k] != kNobody && owner[k] != who) ++bad;
      owner[k] = who;
      if (wave_of[k] != kNobody && wave_of[k] != wave) ++bad;
      wave_of[k] = wave;
    }
  };
  for (int t = 0; t < block; ++t) {
    take((int)body_row_at<L>(t), body_lds_pitch<L>(), t, t / 64);
    take((int)body_stash_at<L>(t), kStash, block + t / L, t / 64);
  }
  if (body_lds_bytes<L>(block) > (160u << 10)) ++bad;
  if (bad) std::printf("%d lanes an instance, workgroup of %d: %d faults\n", L, block, bad);
  return bad;
}

}  // namespace
}  // namespace gp

int main() {
  int bad = 0;
  for (int block : {64, 128, 192, 256}) {
    std::vector<int> wave_of(gp::body_lds_bytes<4>(block) / sizeof(double), gp::kNobody);
    bad += gp::check<4>(block, wave_of) + gp::check<8>(block, wave_of);
  }
  std::vector<int> wave_of(gp::body_lds_bytes<1>(gp::kLoneLanes) / sizeof(double), gp::kNobody);
  bad += gp::check<1>(gp::kLoneLanes, wave_of);
  return bad ? 1 : 0;
}
