// The page table's changed entries across recordings (kv_pages.hpp), as
// hymt_hip.cpp drives it: exit 0, or the line of the first check that fails.
#include "../../hymt2sharp_amd/csrc/kv_pages.hpp"

#define CHECK(x) \
    if (!(x)) return __LINE__ & 0xFF

using hymt::KvPages;
typedef std::vector<int> Ints;

int main() {
    KvPages p(640);
    p.ensure_written(0, 320);
    CHECK((p.take_dirty() == Ints{0, 1, 2, 3, 4}));  // an eager call: on the device now
    CHECK(p.end_recording().empty() && !p.has_dirty());

    // a recording maps page 5, another of its calls page 6; it is dropped
    p.ensure_written(320, 1);
    CHECK((p.take_dirty(true) == Ints{5}));
    p.ensure_written(320, 65);
    CHECK((p.take_dirty(true) == Ints{6}));
    CHECK(!p.has_dirty());  // not recorded twice
    CHECK((p.end_recording() == Ints{5, 6}));

    // the update is still to do: a second recording takes it up again, and
    // an eager call after that one
    CHECK((p.take_dirty(true) == Ints{5, 6}));
    const Ints kept = p.end_recording();
    CHECK((p.take_dirty() == Ints{5, 6}));
    CHECK(!p.has_dirty() && p.end_recording().empty());

    // the table moves on, and a replay writes the recorded entries again
    p.set_len(320);
    CHECK((p.take_dirty() == Ints{5, 6}));
    p.mark_dirty(kept);
    p.mark_dirty(kept);  // two replays
    CHECK((p.take_dirty() == Ints{5, 6}));
    CHECK(p.phys(5) == -1 && p.phys(6) == -1);

    // before another recording, which writes entry 5 itself, runs: the entries
    // that name a page, and not its own
    p.ensure_written(320, 192);  // 5, 6, 7
    p.take_dirty();
    p.mark_dirty({3, 5, 6});
    p.set_len(385);  // 7 given back
    CHECK((p.take_mapped({5}) == Ints{3, 6}));
    CHECK((p.take_dirty() == Ints{5, 7}));

    // entries of a larger context's recording are none of this table's
    p.mark_dirty({-1, 10, 1000});
    CHECK(!p.has_dirty());
    return 0;
}
