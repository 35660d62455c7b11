// Where the launches of concurrent contexts start (XcdStart): the first eight
// on XCDs of their own, halves apart first, the next on the first free again,
// and each device counted by itself.
#include <cstdio>
#include <memory>
#include <vector>

#include "../../mprgp_amd/csrc/mprgp_host.h"

using mprgp::XcdStart;

static int fails = 0;
static void expect(bool ok, const char *what) {
  if (!ok) std::printf("%s\n", what), ++fails;
}

int main() {
  std::vector<std::unique_ptr<XcdStart>> s;
  unsigned seen = 0;
  for (int i = 0; i < 8; ++i) {
    s.emplace_back(new XcdStart());
    s.back()->take(0);
    seen |= 1u << s.back()->xcd();
  }
  expect(seen == 0xff, "eight contexts, eight XCDs");
  expect(s[0]->xcd() == 0 && s[1]->xcd() == 4, "the second half the card away");
  expect((s[2]->xcd() & 1) == 0 && (s[3]->xcd() & 1) == 0, "then quarters");
  XcdStart other;
  other.take(1);
  expect(other.xcd() == 0, "another device");
  const int freed = s[5]->xcd();
  s[5].reset();
  XcdStart again;
  again.take(0);
  expect(again.xcd() == freed, "a freed XCD first");
  XcdStart ninth;
  ninth.take(0);
  expect(ninth.xcd() == 0, "shared from the first on");
  ninth.take(0);
  expect(ninth.xcd() == 0, "taken again in its own place");
  for (int i = 0; i < 1000; ++i) {
    XcdStart t;
    t.take(1);
    expect(t.xcd() == 4, "short-lived contexts leave nothing");
  }
  return fails != 0;
}
