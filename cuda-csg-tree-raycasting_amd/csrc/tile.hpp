// Classification of a tile's 64 rays at once (included by render.hip, inside
// its anonymous namespace).
//
// A wave takes an 8x8 tile, one ray a lane, and walks the tree once for all
// of them: the walk is the same for every lane (the records come through the
// scalar cache and the branches are scalar), and each lane holds its own
// ray's crossings.  An operator is entered when any lane's ray hits a child's
// box; a child is evaluated for the lanes whose rays hit it.  Evaluating a
// node leaves, for each lane, the node's solid along that ray as a list of
// crossings (time, hit bits), ascending, alternating Enter and Exit (the
// first is an Exit when the ray starts inside); lists lie on a per-lane stack
// in LDS ([slot][lane]), a left child's under its right sibling's, so an
// operator combines the two topmost lists in place.  The root's first
// crossing is the ray's hit.
//
// It returns what the state machine (Trace) returns.  Evaluating a subtree
// at a tmin is the machine's eval(X, tmin): the subtree's next crossing
// beyond tmin.  By induction over the tree, where eval of both children
// returns the next crossing of their lists beyond tmin, Compute's loops find
// the next change of the combination, so eval of the operator returns the
// next crossing of the combined list -- with these exceptions, which are
// found ray by ray and handed to the cooperative kernel instead:
//   * ties: the machine compares the children's next times with a strict <,
//     so two equal times at one operator may end the search (CombineLists).
//     The crossings it compares are exactly those of the two lists an
//     operator combines; in a Union group, whose members it pairs up in some
//     order, two equal Enters or Exits of any members count;
//   * in a Union group or a stretch, a primitive whose crossings are not
//     (Enter, Exit) or a lone Exit, and an operator in a Union group whose list
//     is not a solid's (two Enters or two Exits in a row, or no Exit at its
//     end, as a tie or a zone leaves it): the group counts the members a ray is
//     inside of;
//   * a tilted cylinder that leaves its box: the machine enters a primitive's
//     operator only by its boxes, so re-entered at a tmin beyond the box's
//     exit b it takes the cylinder for missed although its own exit x > b is
//     still to come (a box missed at tmin 0 is missed for good, as here).
//     Operators are re-entered at crossing times of their own or their
//     ancestors' results only, so the ray is exact unless one of these lists
//     has a crossing in [b, x): the zone, kept with the list as one interval
//     around all the zones in it and tested at every operator above.  With
//     one at t, that list is sure up to and including t, and what its next
//     crossing is depends on when the machine asks.  So the operator above is
//     sure up to its last crossing at or before t, if it has one, and so on
//     to the root, whose first crossing is the answer if it is still sure
//     (most zones lie on the far side of what the ray hits).  An empty list
//     keeps its zone, as an operand missed there may let the other one appear,
//     unless an empty operand without a zone empties it.  A mixed tree of
//     200 at 1023x1023 hands over 70 rays so, 2234 if any such list fails, none
//     with the zones' ends bounded by the other operand's;
//   * more crossings than the stack holds.
// A subtree is skipped for lanes whose answer cannot depend on it: an
// Intersection's or a Difference's right child where the left list is empty
// (Compute returns Miss whatever the other record is), and an Intersection's
// left child where the right box is missed.
//
// In exact mode the boxes are the reference's and a primitive of any kind may
// leave its box by a rounding error, so each one's exit is compared with its
// box's, and zones are kept as for tilted cylinders; Union groups, whose
// boxes are the fast mode's, are not used.  512 spheres taken from a cube at
// 640x360 take 910 us per lane and 781 us so, at 1920x1080 2232 and 1144 us, a
// mixed tree of 200 at 640x360 974 and 373 us, a chain of 41 325 and 101 us.
//
// Union groups (walkOps, scene.hpp) test the boxes of their chunks and
// members one box a lane against the bundle of the tile's rays (an interval
// of directions an axis), and each member some ray may meet is then
// intersected by all lanes; the members' crossings are gathered unordered,
// sorted in registers and swept with a count.

typedef uint32_t U32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));
#define CSG_SCALAR __attribute__((address_space(4))) const
// (inlined before the optimiser splits up the variables they capture)
#define CSG_INLINE __attribute__((always_inline))

// Wave-uniform reads through the scalar cache (the scene and the job table
// do not change during a launch).
__device__ __forceinline__ U32x16 ScalarRecord(const float4* p, uint32_t at) {
  return *reinterpret_cast<CSG_SCALAR U32x16*>(reinterpret_cast<uintptr_t>(p + at));
}
__device__ __forceinline__ float4 ScalarF4(const float4* p, uint32_t at) {
  const U32x4 v = *reinterpret_cast<CSG_SCALAR U32x4*>(reinterpret_cast<uintptr_t>(p + at));
  return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}

__device__ __forceinline__ float Uniform(float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(AsU(x))); }

// The slab test of BoxHit at tmin 0, also returning where the ray leaves the
// box.
template <bool kFast>
__device__ __forceinline__ bool BoxHitExit(const RayF& r, float lx, float ly, float lz, float hx, float hy, float hz,
                                           float& tmx) {
  float tmn;
  if (kFast) {
    const float t1 = fmaf(lx, r.ix, r.nox), t2 = fmaf(hx, r.ix, r.nox);
    const float t3 = fmaf(ly, r.iy, r.noy), t4 = fmaf(hy, r.iy, r.noy);
    const float t5 = fmaf(lz, r.iz, r.noz), t6 = fmaf(hz, r.iz, r.noz);
    tmn = fmaxf(fmaxf(fminf(t1, t2), fminf(t3, t4)), fminf(t5, t6));
    tmx = fminf(fminf(fmaxf(t1, t2), fmaxf(t3, t4)), fmaxf(t5, t6));
  } else {
    Slab<false>(r, lx, ly, lz, hx, hy, hz, tmn, tmx);
  }
  return !(tmx < 0) & !(tmn > tmx) & !((tmn <= 0.0f) & (tmx <= 0.0f));
}

// A list entry as one double: the time's bits above the hit bits.  Times are
// positive, so entries order by time (the low word only orders ties), and
// every bit pattern met here is a finite double (a float's exponent 255 is
// an ordinary exponent of a double).
__device__ __forceinline__ double EntryOf(float t, uint32_t bits) {
  return __hiloint2double(static_cast<int>(AsU(t)), static_cast<int>(bits));
}
__device__ __forceinline__ uint32_t EntryBits(double e) { return static_cast<uint32_t>(__double2loint(e)); }
__device__ __forceinline__ uint32_t EntryTime(double e) { return static_cast<uint32_t>(__double2hiint(e)); }
// Bits of an entry during a combination: its side (1 left, 2 right) and, two
// bits up, its side again when the next entry of its list is an Exit.
constexpr uint32_t kSideShift = 11, kNextShift = 13, kMarkBits = 0xFu << kSideShift;
constexpr uint32_t kTileFlip = kFlip | kExit | kEnter;

// (bare v_min_f64 / v_max_f64: without a NaN among them the canonicalising
// copies that fmin and fmax add are not needed)
__device__ __forceinline__ void Order(double& a, double& b) {
  double lo, hi;
  asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
  asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  a = lo;
  b = hi;
}

// Batcher's odd-even merge sort (for S that is no power of two, the next
// one's network without the comparisons past the end).
template <int S>
__device__ __forceinline__ void Sort(double (&v)[S]) {
#pragma unroll
  for (int p = 1; p < S; p *= 2) {
#pragma unroll
    for (int k = p; k > 0; k /= 2) {
#pragma unroll
      for (int j = k % p; j + k < S; j += 2 * k) {
#pragma unroll
        for (int i = 0; i < k; i++)
          if (i + j + k < S && (i + j) / (2 * p) == (i + j + k) / (2 * p)) Order(v[i + j], v[i + j + k]);
      }
    }
  }
}

// Above every entry; of no side.
__device__ __forceinline__ double NoEntry() { return __hiloint2double(0x7FE00000, 0); }

// The walk below has no divergent branch: the wave's control stays scalar.
// A lane with nothing to store stores to the first of two spare rows past the
// lists, one with nothing to load reads a row of its own and ignores it.
struct TileList {
  double* col;  // this lane's column: row i at col[64 i]
  int spare;    // the spare row
  int top;      // the last row of the lists
  __device__ __forceinline__ double Get(int row) const { return col[min(row, top) * 64]; }
  // (a list's ends and the rows after them: two rows follow the lists)
  __device__ __forceinline__ double At(int row) const { return col[row * 64]; }
  __device__ __forceinline__ void Put(bool on, int row, double e) const { col[(on ? row : spare) * 64] = e; }
};

// Whether two of the n first of the sorted entries have one time.
template <int S>
__device__ __forceinline__ bool HasTie(const double (&v)[S], int n) {
  uint32_t gap = ~0u;
#pragma unroll
  for (int j = 0; j + 1 < S; j++) {
    const uint32_t g = EntryTime(v[j + 1]) - EntryTime(v[j]);
    gap = min(gap, j + 1 < n ? g : ~0u);
  }
  return gap == 0;
}

template <int S>
__device__ __forceinline__ void StoreEntries(const TileList& l, int base, int n, const double (&v)[S]) {
#pragma unroll
  for (int j = 0; j < S; j++) l.Put(j < n, base + j, v[j]);
}

// Sorts the n entries from `base` on in LDS (insertion; lists longer than
// the register sorts take, nearly always two sorted runs).
__device__ __forceinline__ void SortInPlace(const TileList& l, int base, int n) {
#pragma unroll 1
  for (int i = 1; __ballot(i < n) != 0; i++) {
    int k = i;
    const double e = l.Get(base + i);
    for (;;) {
      const double f = l.Get(base + max(k - 1, 0));
      const bool up = (i < n) & (k > 0) & (f > e);
      if (__ballot(up) == 0) break;
      l.Put(up, base + k, f);
      k -= up ? 1 : 0;
    }
    l.Put(i < n, base + k, e);
  }
}

// `table` has bit s set when an operator's solid holds a point inside the
// children of the bits of s (1 left, 2 right).
__device__ __forceinline__ uint32_t SolidTable(uint32_t op) {
  return op == kOpUnion ? 0xEu : (op == kOpDifference ? 0x2u : 0x8u);
}

// Entry `e`, the last of its list or followed there by `next`, marked for a
// combination (a Difference's right list with its bits flipped).
__device__ __forceinline__ double MarkEntry(double e, bool right, bool last, double next, bool diff) {
  const uint32_t side = right ? 2u : 1u;
  const uint32_t bits = EntryBits(e) ^ ((right & diff) ? kTileFlip : 0u);
  const bool inside = !last & ((EntryBits(next) & kExit) != 0);
  return EntryOf(__uint_as_float(EntryTime(e)),
                 bits | side << kSideShift | (inside ? side << kNextShift : 0u));
}

// Combines two lists into one.  The machine knows a child by its next record:
// the ray is inside the child where that is an Exit, and the closer of the
// two records is returned where consuming it changes the solid, else Compute
// loops into that child.  So, over the entries in order of time: `s`, the
// children whose next entry is an Exit, changes with each entry of a child
// to what its next one says (for a solid's alternating crossings, it
// toggles), and an entry is one of the combination's when the solid differs
// with its child's bit toggled.
__device__ __forceinline__ bool TakesEntry(uint32_t bits, uint32_t table, uint32_t& s) {
  const uint32_t side = (bits >> kSideShift) & 3u, next = (bits >> kNextShift) & 3u;
  const bool change = (((table >> s) ^ (table >> (s ^ side))) & 1u) != 0;
  s = (s & ~side) | next;
  return change;
}

// The combination of two lists of at most two entries each (nL from `base`
// on, nR from `mid` on); false, with nothing changed, when two have one time.
__device__ __forceinline__ bool CombinePairs(const TileList& l, int base, int mid, int nL, int nR, bool diff,
                                             uint32_t table, int& len) {
  const double l0 = l.At(base), l1 = l.At(base + 1), r0 = l.At(mid), r1 = l.At(mid + 1);
  const bool two = nL > 1, twoR = nR > 1;
  const uint32_t flip = diff ? kTileFlip : 0u;
  // marked as MarkEntry does
  const uint32_t a0 = EntryBits(l0) | 1u << kSideShift | ((two & ((EntryBits(l1) & kExit) != 0)) ? 1u << kNextShift : 0u);
  const uint32_t a1 = EntryBits(l1) | 1u << kSideShift;
  const uint32_t b0 = (EntryBits(r0) ^ flip) | 2u << kSideShift |
                      ((twoR & ((EntryBits(r1) & kExit) != 0)) ? 2u << kNextShift : 0u);
  const uint32_t b1 = (EntryBits(r1) ^ flip) | 2u << kSideShift;
  double v[4];
  v[0] = nL > 0 ? EntryOf(__uint_as_float(EntryTime(l0)), a0) : NoEntry();
  v[1] = two ? EntryOf(__uint_as_float(EntryTime(l1)), a1) : NoEntry();
  v[2] = nR > 0 ? EntryOf(__uint_as_float(EntryTime(r0)), b0) : NoEntry();
  v[3] = twoR ? EntryOf(__uint_as_float(EntryTime(r1)), b1) : NoEntry();
  uint32_t s = ((EntryBits(l0) & kExit) ? 1u : 0u) | ((EntryBits(r0) & kExit) ? 2u : 0u);
  // two ascending pairs merged
  Order(v[0], v[2]);
  Order(v[1], v[3]);
  Order(v[1], v[2]);
  if (__ballot(HasTie<4>(v, nL + nR)) != 0) return false;
  int w = base;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const bool change = TakesEntry(EntryBits(v[j]), table, s);
    l.Put(change, w, EntryOf(__uint_as_float(EntryTime(v[j])), EntryBits(v[j]) & ~kMarkBits));
    w += change ? 1 : 0;
  }
  len = w - base;
  return true;
}

// The combination of the n = nL + nR <= S entries from `base` on (the left
// list, then the right one), `s` as above before them.  False, with the
// entries marked and sorted in place, when two have one time.
template <int S>
__device__ __forceinline__ bool Combine(const TileList& l, int base, int nL, int n, bool diff, uint32_t s,
                                        uint32_t table, int& len) {
  double v[S];
  double e = l.Get(base);
#pragma unroll
  for (int j = 0; j < S; j++) {
    const double next = j + 1 < S ? l.Get(base + j + 1) : e;
    const double m = MarkEntry(e, j >= nL, (j + 1 == nL) | (j + 1 >= n), next, diff);
    v[j] = j < n ? m : NoEntry();
    e = next;
  }
  Sort<S>(v);
  if (__ballot(HasTie<S>(v, n)) != 0) {
    StoreEntries<S>(l, base, n, v);
    return false;
  }
  int w = base;
#pragma unroll
  for (int j = 0; j < S; j++) {
    const bool change = TakesEntry(EntryBits(v[j]), table, s);
    l.Put(change, w, EntryOf(__uint_as_float(EntryTime(v[j])), EntryBits(v[j]) & ~kMarkBits));
    w += change ? 1 : 0;
  }
  len = w - base;
  return true;
}

// Marks the entries in place, for the lists Combine does not take.
__device__ __forceinline__ void MarkInPlace(const TileList& l, int base, int nL, int n, bool diff) {
#pragma unroll 1
  for (int i = 0; __ballot(i < n) != 0; i++)
    l.Put(i < n, base + i,
          MarkEntry(l.Get(base + i), i >= nL, (i + 1 == nL) | (i + 1 >= n), l.Get(base + i + 1), diff));
}

// The same from marked, sorted entries in LDS, with two cases more.
//
// Two entries at one time, taken as the machine takes them, comparing times
// with a strict <: where the two together leave the solid as it was, Compute
// loops into one child and then the other, and no crossing results; where
// they change it, neither is closer and Compute returns Miss.  The list then
// ends there (`cutAt`, else `te`), as the machine sees it until it comes back
// at a later tmin.  (At the end `te` of a stretch, where lists are cut off
// together, they simply end.)  `bad`: a tied Enter with no Exit after it in
// its list, which the machine's order decides.
//
// A child (side `own`, 0: none) that is a cylinder leaving its box, with the
// zone [zlo, zhi): once this operator has returned a crossing in the zone, it
// is entered again by its boxes, and the cylinder missed.  Its other entries
// then do not count, and the zone ends at that crossing.
__device__ __forceinline__ int CombineSpecial(const TileList& l, int base, int n, uint32_t s, uint32_t table,
                                              uint32_t te, uint32_t own, float zlo, float& zhi, bool& bad,
                                              uint32_t& cutAt) {
  int w = base;
  bool live = true, tied = false;
  uint32_t before = s;  // the state before the entries at this time
  uint32_t gone = 0;    // the side missed from here on
#pragma unroll 1
  for (int i = 0; __ballot(i < n) != 0; i++) {
    const double e = l.Get(base + i), f = l.Get(base + i + 1);
    const uint32_t t = EntryTime(e), bits = EntryBits(e), side = (bits >> kSideShift) & 3u;
    const bool valid = (i < n) & ((side & gone) == 0), tieNext = (i + 1 < n) & (EntryTime(f) == t);
    const uint32_t both = tied ? before ^ 3u : before ^ side;
    const bool differs = (((table >> before) ^ (table >> both)) & 1u) != 0;
    const bool change = valid & !tieNext & live & differs, ends = change & tied & (t != te);
    bad |= valid & live & (tied | tieNext) & (t != te) &
           ((((s ^ (bits >> kNextShift)) & side) == 0) | (own != 0));
    uint32_t after = s;
    TakesEntry(bits, table, after);
    s = valid ? after : s;
    const bool put = change & !ends;
    l.Put(put, w, EntryOf(__uint_as_float(t), bits & ~kMarkBits));
    w += put ? 1 : 0;
    const bool drop = put & (own != 0) & (__uint_as_float(t) >= zlo) & (__uint_as_float(t) < zhi);
    gone = drop ? own : gone;
    s = drop ? s & ~own : s;
    zhi = drop ? __uint_as_float(t) : zhi;
    cutAt = ends ? t : cutAt;
    live &= !ends;
    before = tieNext ? before : s;
    tied = tieNext;
  }
  return w - base;
}

// The union of the n <= S crossings from `base` on, in any order: sorted and
// swept with a count of the members the ray is inside of.  Every member's list
// alternates and ends with an Exit (NoSolid fails the rays of others), so the
// members the ray starts inside of are the surplus of Exits.
// False, with the entries sorted in place, when two have one time.
template <int S>
__device__ __forceinline__ bool Unite(const TileList& l, int base, int n, int& len) {
  double v[S];
#pragma unroll
  for (int j = 0; j < S; j++) {
    const double e = l.Get(base + j);
    v[j] = j < n ? e : NoEntry();
  }
  Sort<S>(v);
  if (__ballot(HasTie<S>(v, n)) != 0) {
    StoreEntries<S>(l, base, n, v);
    return false;
  }
  int depth = 0;  // minus the sum of the entries' steps, +1 for an Enter
#pragma unroll
  for (int j = 0; j < S; j++) depth -= static_cast<int>(EntryBits(v[j]) & kEnter) - 1;
  depth -= S - n;  // (a NoEntry counted as an Exit)
  int w = base;
#pragma unroll
  for (int j = 0; j < S; j++) {
    const int before = depth;
    depth += static_cast<int>(EntryBits(v[j]) & kEnter) - 1;
    const bool change = min(before, depth) == 0;  // (after the last entry the count runs below 0)
    l.Put(change, w, v[j]);
    w += change ? 1 : 0;
  }
  len = w - base;
  return true;
}

// Whether the list in rows [from, to) is not a solid's: two Enters or two Exits
// in a row, or an Enter at its end.
__device__ __forceinline__ bool NoSolid(const TileList& l, int from, int to) {
  bool odd = false;
  uint32_t bits = EntryBits(l.Get(from));
#pragma unroll 1
  for (int i = from; __ballot(i < to) != 0; i++) {
    const uint32_t next = i + 1 < to ? EntryBits(l.Get(i + 1)) : kEnter;
    odd |= (i < to) & (((bits ^ next) & kEnter) == 0);
    bits = next;
  }
  return odd;
}

// The same from sorted entries in LDS with equal times among them: an Enter
// and an Exit at one time leave the union as it was however the machine pairs
// the members; two Enters or two Exits make the ray `bad` (but at `te`).
__device__ __forceinline__ int UniteTies(const TileList& l, int base, int n, uint32_t te, bool& bad) {
  int depth = 0;
#pragma unroll 1
  for (int i = 0; __ballot(i < n) != 0; i++) {
    const int step = (EntryBits(l.Get(base + i)) & kEnter) ? -1 : 1;
    depth += i < n ? step : 0;
  }
  int w = base, before = depth;
  bool tied = false;
#pragma unroll 1
  for (int i = 0; __ballot(i < n) != 0; i++) {
    const double e = l.Get(base + i), f = l.Get(base + i + 1);
    const bool valid = i < n, enter = (EntryBits(e) & kEnter) != 0;
    const bool tieNext = (i + 1 < n) & (EntryTime(e) == EntryTime(f));
    depth += valid ? (enter ? 1 : -1) : 0;
    bad |= tieNext & (EntryTime(e) != te) & (tied | (enter == ((EntryBits(f) & kEnter) != 0)));
    const bool change = valid & !tieNext & ((before == 0) != (depth == 0));
    l.Put(change, w, e);
    w += change ? 1 : 0;
    before = tieNext ? before : depth;
    tied = tieNext;
  }
  return w - base;
}

// The bundle of a tile's rays, direction D = forward + nx right + ny up over
// the tile's rectangle, as factors of the slab test on interval bounds: per
// axis, with box limits p, q from the origin, every ray that enters the slab
// does so after p a and after q b, and every ray that leaves it does so
// before max(p c, q c) + k (k infinite where D's sign varies over the tile).
struct TileBundle {
  float a[3], b[3], c[3], k[3];
};
// Bounds of 1 / |D| over the tile: a stretch of a ray's distances times these
// is one of D's multiples.
struct TileScale {
  float lo, hi;
};

// Whether some ray of the bundle may meet the box between the multiples `from`
// and `to` of its D, the box widened by far more than the rounding of any
// ray's own slab test.
__device__ __forceinline__ bool BundleMeets(const TileBundle& f, const float* o, float lx, float ly, float lz,
                                            float hx, float hy, float hz, float from = 0.0f,
                                            float to = __builtin_inff()) {
  const float l[3] = {lx, ly, lz}, h[3] = {hx, hy, hz};
  float en = from, ex = to;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float pad = 1e-5f * (fabsf(o[i]) + fabsf(l[i]) + fabsf(h[i]));
    const float p = (l[i] - pad) - o[i], q = (h[i] + pad) - o[i];
    en = fmaxf(en, fmaxf(p * f.a[i], q * f.b[i]));
    ex = fminf(ex, fmaxf(p * f.c[i], q * f.c[i]) + f.k[i]);
  }
  return !(en > ex);
}

// The bundle of tile (x0, y0): its pixels' sample points lie in
// [x0, x0 + 8] x [y0, y0 + 8].
__device__ __forceinline__ TileBundle BundleOf(const Job& jb, int x0, int y0, TileScale& scale) {
  const float kx = (static_cast<float>(jb.width) / static_cast<float>(jb.height)) * jb.tanHalf, ky = jb.tanHalf;
  const float iw = __builtin_amdgcn_rcpf(static_cast<float>(jb.width - 1));
  const float ih = __builtin_amdgcn_rcpf(static_cast<float>(jb.height - 1));
  const float u0 = (2.0f * (static_cast<float>(x0) * iw) - 1.0f) * kx;
  const float u1 = (2.0f * (static_cast<float>(x0 + 8) * iw) - 1.0f) * kx;
  const float v0 = (1.0f - 2.0f * (static_cast<float>(y0) * ih)) * ky;
  const float v1 = (1.0f - 2.0f * (static_cast<float>(y0 + 8) * ih)) * ky;
  // |D|^2 = 1 + nx^2 + ny^2: the camera's axes are unit vectors at right angles
  // but for rounding, which the margins cover
  const float au = fmaxf(fabsf(u0), fabsf(u1)), av = fmaxf(fabsf(v0), fabsf(v1));
  const float bu = u0 * u1 > 0.0f ? fminf(fabsf(u0), fabsf(u1)) : 0.0f;
  const float bv = v0 * v1 > 0.0f ? fminf(fabsf(v0), fabsf(v1)) : 0.0f;
  scale.lo = 0.9999f * __builtin_amdgcn_rsqf(1.0f + au * au + av * av);
  scale.hi = 1.0001f * __builtin_amdgcn_rsqf(1.0f + bu * bu + bv * bv);
  TileBundle f;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float r0 = jb.right[i] * u0, r1 = jb.right[i] * u1, s0 = jb.up[i] * v0, s1 = jb.up[i] * v1;
    const float pad = 1e-5f * (1.0f + fabsf(r0) + fabsf(r1) + fabsf(s0) + fabsf(s1));
    const float lo = jb.forward[i] + fminf(r0, r1) + fminf(s0, s1) - pad;
    const float hi = jb.forward[i] + fmaxf(r0, r1) + fmaxf(s0, s1) + pad;
    // 1/lo and 1/hi, widened over the reciprocal's rounding; a sign that may
    // vary leaves that side of the slab out of reach or without a bound
    const float ilo = __builtin_amdgcn_rcpf(lo), ihi = __builtin_amdgcn_rcpf(hi);
    f.a[i] = hi > 0.0f ? 0.999999f * ihi : 1e30f;
    f.b[i] = lo < 0.0f ? 0.999999f * ilo : -1e30f;
    f.c[i] = lo > 0.0f ? 1.000001f * ilo : (hi < 0.0f ? 1.000001f * ihi : 0.0f);
    f.k[i] = lo > 0.0f || hi < 0.0f ? 0.0f : __builtin_inff();
  }
  return f;
}

// CubeAt with CubeNormalAxis's division, where some lane's quotient lies in
// the band that needs it, behind one scalar branch.
__device__ __forceinline__ Hit TileCubeAt(const RayF& r, const float4& a, uint32_t prim, float t) {
  constexpr float kBias = 1.00001f;
  const float half = a.w / 2, rh = __builtin_amdgcn_rcpf(half);
  const float p[3] = {(r.ox + t * r.dx) - a.x, (r.oy + t * r.dy) - a.y, (r.oz + t * r.dz) - a.z};
  float n[3];
  bool band[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float x = p[k] * rh * kBias, ax = fabsf(x);
    n[k] = copysignf(ax < 1.0f ? 0.0f : 1.0f, x);
    band[k] = !((ax < 1.0f - 4e-6f) | ((ax > 1.0f + 4e-6f) & (ax < 2.0f - 8e-6f)));
  }
  if (__ballot(band[0] | band[1] | band[2]) != 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float d = TruncInt(p[k] / half * kBias);
      n[k] = band[k] ? d : n[k];
    }
  }
  const float dn = n[0] * r.dx + n[1] * r.dy + n[2] * r.dz;
  return Hit{t, HitBits(dn <= 0 ? kEnter : kExit, kCubeT, prim)};
}

// Crossings beyond 0 of a wave-uniform primitive, as PrimCrossings reports
// them: `c` of them, the last in `x` and, of two, the first in `e`.
template <bool kFast>
__device__ __forceinline__ uint32_t TilePrimCrossings(const Job& jb, const RayF& r, uint32_t desc, const float4& pa, Hit& e,
                                                      Hit& x) {
  const uint32_t type = DescType(desc), prim = DescIndex(desc);
  if (type == kSphereT) {
    float t0, t1;
    const bool hit = RootsOfSphere<kFast>(r, pa, t0, t1) & (t1 > 0.0f);
    e = SphereAt(r, pa, prim, t0);
    x = SphereAt(r, pa, prim, t1);
    return !hit ? 0u : ((t0 > 0.0f) & (t1 > t0) ? 2u : 1u);
  }
  if (type == kCubeT) {
    float tmn, tmx;
    const bool hit = CubeSlab<kFast>(r, pa, tmn, tmx) & (tmx > 0.0f);
    e = TileCubeAt(r, pa, prim, tmn);
    x = TileCubeAt(r, pa, prim, tmx);
    return !hit ? 0u : ((tmn > 0.0f) & (tmx > tmn) ? 2u : 1u);
  }
  CylinderRoots roots;
  const bool hit = RootsOfCylinder<kFast>(r, pa, ScalarF4(jb.sc.primB, prim), roots);
  // the first root beyond 0, then the second if it lies beyond that
  const bool in0 = !((roots.t[0] <= 0.0f) | roots.skip[0]);
  const float beyond = in0 ? roots.t[0] : 0.0f;
  const bool in1 = !((roots.t[1] <= beyond) | roots.skip[1]);
  e = CylinderAt(r, roots, prim, 0);
  const Hit last = CylinderAt(r, roots, prim, 1);
  x = Hit{in1 ? last.t : e.t, in1 ? last.bits : e.bits};
  return hit ? (in0 ? 1u : 0u) + (in1 ? 1u : 0u) : 0u;
}

// LDS of one wave (TileLds): the list stack, `slots` x 64 x 8 B, and two
// spare rows; the tile's bundle (kept here for the groups that use it: 12
// registers); a group's hit chunks, 64 x 2 B, and a spare entry; per level
// and lane where its list starts, 1 B.
struct TileLdsView {
  double* lists;
  float4* bundle;
  uint16_t* chunks;
  uint8_t* bounds;
};

// Where the walk goes on after a child's list is complete.
constexpr uint32_t kTileLeft = 0, kTileRight = 1, kTileGroup = 2, kTileEnter = 3, kTileReturn = 4;

// Evaluates the root over the rays' stretch [ts, te) for the lanes in
// `active`; returns in `fail` the lanes the machine must trace, in `full`
// those whose lists overflowed, and in `h` the other active lanes' first
// crossings in the stretch.  Over the whole ray (te infinite) subtrees are
// skipped as said above and zones kept; over a shorter stretch (`cut`) a
// list is cut off at te by an Exit there, an empty list only says that the
// ray is outside throughout the stretch, so every child whose box is hit is
// evaluated (a tie anywhere on the ray counts) and every zone kept.
template <bool kFast, bool kGroups>
__device__ __forceinline__ void TileTrace(const Job& jb, const RayF& r, uint64_t active, const float4* ops,
                                          const TileLdsView& lds, int slots, int lane, float ts, float te, Hit& h,
                                          uint64_t& fail, uint64_t& full) {
  constexpr bool kWide = kGroups || !kFast;  // lists of up to 16 crossings a pair sort in registers
  const bool cut = kGroups && (te < __builtin_inff() || ts > 0.0f);
  const uint32_t teBits = AsU(te);
  const float4* groups = jb.sc.walkOps;
  const TileList list{lds.lists + lane, slots, slots - 1};
  const uint64_t me = uint64_t{1} << lane;
  int sp = 0;           // this lane's list stack top
  full = 0;
  uint64_t dead = 0;  // lanes no longer followed: failed or full
  float zlo = __builtin_inff(), zhi = -__builtin_inff();  // the current list's zone
  uint64_t zoneLevels = 0;                                // levels whose left list's zone is saved
  int limit = slots;    // rows the lists may take; those above hold saved zones
  bool zones = false;   // some lane has met a zone
  // A list with a crossing in its zone at `sure`, its operator's level and
  // whether some lane has one: what the machine finds beyond is in doubt.
  float sure = __builtin_inff();
  int sureLevel = 0;
  bool doubts = false;
  // frames of the entered operators: lane i holds level i's
  uint32_t fOp = 0, fRight = 0, fMl = 0, fMh = 0, fRl = 0, fRh = 0;
  int d = 0;
  uint32_t X = 0;
  uint64_t M = active;

  auto wl = [&](uint32_t& reg, uint32_t v) CSG_INLINE {
    reg = lane == d ? v : reg;
  };
  auto rl = [&](uint32_t reg) CSG_INLINE { return static_cast<uint32_t>(__builtin_amdgcn_readlane(reg, d)); };

  // Pushes a primitive's crossings in the stretch for the lanes in `mask`,
  // whose rays leave its box at `tmx`.
  auto leaf = [&](uint32_t desc, const float4& pa, uint64_t mask, float tmx, bool strict) CSG_INLINE {
    Hit a, b;
    uint32_t c = TilePrimCrossings<kFast>(jb, r, desc, pa, a, b);
    c = (mask & me) != 0 ? c : 0u;
    // (Enter, Exit) or (Exit) alone, unless its records are combined one by
    // one (Combine); at finite times
    const bool two = c == 2;
    const bool odd = !(b.bits & kExit) | (two & !(a.bits & kEnter));
    const bool bad = (c != 0) & (!(b.t < __builtin_inff()) | (odd & strict));
    dead |= __ballot(bad);
    if (!kFast || DescType(desc) == kCylinderT) {
      const bool out = (c != 0) & !(b.t <= tmx);
      if (__ballot(out) != 0) {
        zones = true;
        zlo = out ? fminf(zlo, tmx) : zlo;
        zhi = out ? fmaxf(zhi, b.t) : zhi;
      }
    }
    const bool enters = two & (a.t >= ts);  // its Enter lies in the stretch
    int n = (c != 0) & !bad & (b.t >= ts) & !(two & (a.t >= te)) ? (enters ? 2 : 1) : 0;
    const bool over = sp + n > limit;
    full |= __ballot(over);
    dead |= full;
    n = over ? 0 : n;
    const double last = EntryOf(fminf(b.t, te), b.bits);
    const double head = EntryOf(enters ? a.t : fminf(b.t, te), enters ? a.bits : b.bits);
    list.Put(n >= 1, sp, head);
    list.Put(n == 2, sp + 1, last);
    sp += n;
  };
  // Whether this lane, if in `mask`, has a crossing of its current list (from
  // `base` on) in its zone, and the first such time.
  auto inZone = [&](uint64_t mask, int base, float& at) CSG_INLINE {
    const bool has = ((mask & me) != 0) & (zhi > zlo);
    bool in = false;
    if (__ballot(has) != 0) {
#pragma unroll 1
      for (int i = base; __ballot(has & (i < sp)) != 0; i++) {
        const float t = __uint_as_float(EntryTime(list.Get(i)));
        const bool here = has & (i < sp) & (t >= zlo) & (t < zhi);
        at = here & !in ? t : at;
        in |= here;
      }
    }
    return in;
  };
  // Saves the current zones with level d's pending list.
  auto saveZones = [&]() CSG_INLINE {
    if (!zones) return;
    const uint64_t has = __ballot(zhi > zlo);
    if (has == 0) return;
    // in the topmost free row of the lists; a lane whose list reaches it
    // cannot keep one
    const bool room = limit > 1;
    const uint64_t high = __ballot((sp >= limit) | !room);
    dead |= high & has;
    limit -= room ? 1 : 0;
    list.Put((high & me) == 0, limit, EntryOf(zhi, AsU(zlo)));
    zoneLevels |= static_cast<uint64_t>(room) << d;
    zlo = __builtin_inff();
    zhi = -__builtin_inff();
  };
  U32x16 q;                  // X's record, when it is entered
  uint32_t cur = 0, rDesc = 0;  // X's operator type and which children are primitives; its right child
  auto qf = [&](int k) CSG_INLINE { return __uint_as_float(q[k]); };
  int base = 0, mid = 0;
  float exitR = 0.0f;  // where the ray leaves the right child's box
  uint64_t mR = 0;
  // a Union group's walk: chunk round, member round, hit chunks of the chunk
  // round, members of the member round still to visit, and the lane's member
  uint32_t cr = 0, mr = 0, nHit = 0, skip = 0;
  uint64_t todo = 0;
  float4 m0 = make_float4(0, 0, 0, 0), m1 = m0, m2 = m0;
  // what comes next: kTileLeft, kTileRight and kTileGroup go on with operator
  // X after a child; kTileEnter enters X for the lanes M; kTileReturn: X's
  // list is complete
  uint32_t state = kTileEnter;
  for (;;) {
    uint32_t leafDesc = kNone;
    float4 leafA = make_float4(0, 0, 0, 0);
    uint64_t leafMask = 0;
    float leafExit = 0.0f;
    // enters child operator `k` for `lanes`, to come back in state `next`
    auto enter = [&](uint32_t k, uint64_t lanes, uint32_t next, uint64_t keep) CSG_INLINE {
      wl(fOp, X | next << 15 | cur << 17);
      wl(fMl, static_cast<uint32_t>(M));
      wl(fMh, static_cast<uint32_t>(M >> 32));
      if (next != kTileRight) {
        wl(fRl, static_cast<uint32_t>(keep));
        wl(fRh, static_cast<uint32_t>(keep >> 32));
      }
      // (entered on the left, a child's list starts where X's does)
      if (next == kTileLeft) wl(fRight, rDesc);
      else lds.bounds[d * 64 + lane] = static_cast<uint8_t>(base);
      X = k;
      M = lanes;
      d++;
      state = kTileEnter;
    };
    if (state == kTileReturn) {
      if (d == 0) break;
      d--;
      const uint32_t f = rl(fOp);
      X = f & 0x7FFFu;
      state = (f >> 15) & 3u;
      cur = f >> 17;
      M = (static_cast<uint64_t>(rl(fMh)) << 32 | rl(fMl));
      mR = (static_cast<uint64_t>(rl(fRh)) << 32 | rl(fRl));
      mid = base;
      if (state == kTileLeft) {
        rDesc = rl(fRight);
        if (kFast ? DescType(rDesc) == kCylinderT : DescType(rDesc) >= kSphereT) {
          q = ScalarRecord(ops, 4 * X);
          BoxHitExit<kFast>(r, qf(3), qf(7), qf(8), qf(9), qf(10), qf(11), exitR);
        }
      } else {
        base = lds.bounds[d * 64 + lane];
        if (state == kTileRight) mR = ~uint64_t{0};  // (its right list was evaluated)
      }
      if (kGroups && state == kTileGroup) {
        // (the member's list lies in rows [mid, sp))
        dead |= __ballot(NoSolid(list, mid, sp));
        q = ScalarRecord(ops, 4 * X);
        // this member round again, past the member it left off at
        cr = static_cast<uint32_t>(mR) >> 8;
        mr = (static_cast<uint32_t>(mR) >> 6) & 3u;
        skip = static_cast<uint32_t>(mR) & 63u;
        nHit = 0;
        todo = 0;
        if ((zoneLevels >> d) & 1) {
          // (a lane that could not keep its zone then reads another entry of
          // its list for one: at worst it fails)
          zoneLevels &= ~(uint64_t{1} << d);
          const double z = list.At(limit);
          limit++;
          zlo = fminf(zlo, __uint_as_float(EntryBits(z)));
          zhi = fmaxf(zhi, __uint_as_float(EntryTime(z)));
        }
      }
    }
    if (state == kTileEnter) {
      M &= ~dead;
      q = ScalarRecord(ops, 4 * X);
      base = sp;
      mid = sp;
      if (kGroups && (q[14] & kWalkGroupFlag)) {
        state = kTileGroup;
        cr = mr = nHit = skip = 0;
        todo = 0;
      } else {
        const bool gL = BoxHitExit<kFast>(r, qf(0), qf(1), qf(2), qf(4), qf(5), qf(6), leafExit);
        const bool gR = BoxHitExit<kFast>(r, qf(3), qf(7), qf(8), qf(9), qf(10), qf(11), exitR);
        const uint32_t op = q[14] & 0xFFu;
        uint64_t mL = __ballot(gL) & M;
        mR = __ballot(gR) & M;
        if (op != kOpUnion) mR &= mL;
        if (op > kOpDifference) mL = mR;
        const bool opL = DescType(q[12]) < kSphereT, opR = DescType(q[13]) < kSphereT;
        rDesc = q[13];
        cur = op | (opL ? 0u : 4u) | (opR ? 0u : 8u);
        state = kTileLeft;
        if ((mL | mR) == 0) {
          state = kTileReturn;
        } else if (mR == 0 && opL) {
          // the left child's list is the operator's: on to it in its place
          X = DescIndex(q[12]);
          M = mL;
          state = kTileEnter;
        } else if (mL == 0 && opR) {
          X = DescIndex(q[13]);
          M = mR;
          state = kTileEnter;
        } else if (mL != 0) {
          if (opL) {
            enter(DescIndex(q[12]), mL, kTileLeft, mR);
          } else {
            leafDesc = q[12];
            leafA = ScalarF4(jb.sc.primA, DescIndex(q[12]));
            leafMask = mL;
          }
        }
      }
    } else if (state == kTileLeft) {
      mid = sp;
      if ((cur & 3u) != kOpUnion && !cut) mR &= __ballot(sp > base);
      mR &= ~dead;
      state = kTileRight;
      if (mR != 0) {
        saveZones();
        if (cur & 8u) {
          leafDesc = rDesc;
          leafA = ScalarF4(jb.sc.primA, DescIndex(rDesc));
          leafMask = mR;
          leafExit = exitR;
        } else {
          enter(DescIndex(rDesc), mR, kTileRight, 0);
        }
      }
    } else if (state == kTileRight) {
      // combine the two lists of the lanes in M
      const uint32_t op = cur & 3u;
      const bool on = (M & me) != 0;
      const int nL = mid - base, nR = sp - mid;
      const bool both = on & (nL > 0) & (nR > 0);
      // Each list's zone; where only one has one and that list is a
      // primitive's, the side it is on (CombineSpecial).
      uint32_t own = 0;
      bool gone = false;  // empty for good: an operand without a zone is, and empties the combination
      // Whether some lane has a zone or a doubt here (in exact mode, where nearly
      // every tile has zones, the test costs 8 % of 181 spheres at 1722x1722).
      bool zoned = zones && (!kFast || doubts || ((zoneLevels >> d) & 1) != 0 || __ballot(zhi > zlo) != 0);
      if (zoned) {
        float l0 = __builtin_inff(), l1 = -__builtin_inff();
        if ((zoneLevels >> d) & 1) {
          zoneLevels &= ~(uint64_t{1} << d);
          const double z = list.At(limit);
          const bool low = mid <= limit;
          limit++;
          l0 = low ? __uint_as_float(EntryBits(z)) : l0;
          l1 = low ? __uint_as_float(EntryTime(z)) : l1;
        } else if (mR == 0) {  // no right list: the current zone is the left one's
          l0 = zlo;
          l1 = zhi;
          zlo = __builtin_inff();
          zhi = -__builtin_inff();
        }
        const bool hasL = l1 > l0, hasR = zhi > zlo;
        own = hasL & !hasR & ((cur & 4u) != 0) ? 1u : 0u;
        own = hasR & !hasL & ((cur & 8u) != 0) ? 2u : own;
        own = on & !cut ? own : 0u;
        gone = (op != kOpUnion) & (nL == 0 ? !hasL : ((op > kOpDifference) & (nR == 0) & !hasR));
        zlo = fminf(zlo, l0);
        zhi = fmaxf(zhi, l1);
        // Past the last crossing of an operand without a zone that the solid
        // lies in, the combination is empty whatever the other one is.
        if (op != kOpUnion && !cut && __ballot(both & (hasL != hasR)) != 0) {
          const float lastL = __uint_as_float(EntryTime(list.At(max(mid - 1, 0))));
          const float lastR = __uint_as_float(EntryTime(list.At(max(sp - 1, 0))));
          zhi = both & !hasL ? fminf(zhi, lastL) : zhi;
          zhi = both & (op > kOpDifference) & !hasR ? fminf(zhi, lastR) : zhi;
        }
      }
      if (__ballot(both) != 0) {
        const uint32_t table = SolidTable(op);
        const bool diff = op == kOpDifference, special = __ballot(own != 0) != 0;
        const int n = both ? nL + nR : 0;
        int len = 0;
        bool done = false;
        if (!special && __ballot(both & ((nL > 2) | (nR > 2))) == 0)
          done = CombinePairs(list, base, mid, both ? nL : 0, both ? nR : 0, diff, table, len);
        if (!done) {
          // inside a child where its next entry is an Exit
          const uint32_t s = ((EntryBits(list.At(base)) & kExit) ? 1u : 0u) |
                             ((EntryBits(list.At(mid)) & kExit) ? 2u : 0u);
          const float end = fmaxf(__uint_as_float(EntryTime(list.At(max(mid - 1, 0)))),
                                  __uint_as_float(EntryTime(list.At(max(sp - 1, 0)))));
          if (special || __ballot(n > (kWide ? 16 : 8)) != 0) {
            MarkInPlace(list, base, nL, n, diff);
            SortInPlace(list, base, n);
          } else if (__ballot(n > 8) == 0) {
            done = Combine<8>(list, base, nL, n, diff, s, table, len);
          } else if (kWide) {
            done = Combine<16>(list, base, nL, n, diff, s, table, len);
          }
          if (!done) {
            bool bad = false;
            uint32_t cutAt = teBits;
            len = CombineSpecial(list, base, n, s, table, teBits, own, zlo, zhi, bad, cutAt);
            const bool ended = both & (cutAt != teBits);
            // seen whole again from `cutAt` on: a zone up to the later list's end
            zlo = ended ? fminf(zlo, __uint_as_float(cutAt)) : zlo;
            zhi = ended ? fmaxf(zhi, end) : zhi;
            bad |= ended & cut;
            zoned |= __ballot(ended) != 0;
            zones |= zoned;
            dead |= __ballot(bad);
          }
        }
        sp = both ? base + len : sp;
      }
      // an Intersection with one list empty, a Difference with the left one
      const bool none = on & !both & ((op > kOpDifference) | ((op == kOpDifference) & (nL == 0)));
      sp = none ? base : sp;
      if (zoned) {
        // an only list with its own zone: once its Enter is returned in the
        // zone, its Exit is not seen (CombineSpecial)
        const float t0 = __uint_as_float(EntryTime(list.At(base)));
        const bool drop = !both & (own != 0) & (sp == base + 2) & (t0 >= zlo) & (t0 < zhi);
        sp = drop ? base + 1 : sp;
        zhi = drop ? t0 : zhi;
        // missed, a primitive that the solid lies in leaves it empty too
        gone |= (sp == base) & ((own == 1 && op != kOpUnion) | (own == 2 && op > kOpDifference));
        // (a zone no longer than a point is none: it must not widen the next one)
        gone = (gone & on & !cut) | !(zhi > zlo);
        zlo = gone ? __builtin_inff() : zlo;
        zhi = gone ? -__builtin_inff() : zhi;
        // the last crossing a child's doubt leaves sure; none of an empty
        // list that the other child alone has emptied
        bool low = false;
        if (doubts) {
          low = on & (sureLevel > d);
          if (__ballot(low) != 0) {
            float last = -1.0f;
#pragma unroll 1
            for (int i = base; __ballot(low & (i < sp)) != 0; i++) {
              const float t = __uint_as_float(EntryTime(list.Get(i)));
              last = low & (i < sp) & (t <= sure) ? t : last;
            }
            const bool clear = low & none & !cut;
            dead |= __ballot(low & !clear & (last < 0.0f));
            sure = low ? (clear ? __builtin_inff() : last) : sure;
            sureLevel = low ? (clear ? 0 : d) : sureLevel;
            low &= !clear;
          }
        }
        float at = 0.0f;
        const bool in = inZone(M, base, at);
        doubts |= __ballot(in) != 0;
        // (one doubt a lane: with another pending, of a list beside this one, it fails)
        dead |= __ballot(in & !low & (sure < __builtin_inff()));
        sure = in ? fminf(sure, at) : sure;
        sureLevel = in ? d : sureLevel;
      }
      state = kTileReturn;
    } else if (kGroups && state == kTileGroup) {
      // chunks of the group 64 a round, the members of the hit chunks
      // 64 a round, the members some ray may meet one by one
      const uint32_t first = q[12], count = q[13];
      const uint32_t nChunks = (count + kWalkChunk - 1) / kWalkChunk, mfirst = first + 2 * nChunks;
      constexpr uint32_t kPerRound = 64 / kWalkChunk;
      TileBundle bundle{};
      float from = 0.0f, to = __builtin_inff();
      if (todo == 0) {
        // only members that lie in the stretch: each is wholly inside its box
        // (or marked, and taken in every stretch)
        if (cut) {
          const float4 sc = lds.bundle[3];
          from = ts * sc.x;
          to = te * sc.y;
        }
        const float4 u = lds.bundle[0], v = lds.bundle[1], w = lds.bundle[2];
        bundle = TileBundle{{u.x, u.y, u.z}, {u.w, v.x, v.y}, {v.z, v.w, w.x}, {w.y, w.z, w.w}};
      }
      while (todo == 0 && (mr * kPerRound < nHit || cr * 64 < nChunks)) {
        if (nHit == 0) {
          const uint32_t ci = cr * 64 + static_cast<uint32_t>(lane);
          const uint32_t ca = first + 2 * min(ci, nChunks - 1);
          const float4 c0 = groups[ca], c1 = groups[ca + 1];
          const bool all = AsU(c1.w) != 0;
          const bool hit = (ci < nChunks) & BundleMeets(bundle, jb.pos, c0.x, c0.y, c0.z, c0.w, c1.x, c1.y,
                                                        all ? 0.0f : from, all ? __builtin_inff() : to);
          const uint64_t hm = __ballot(hit);
          lds.chunks[hit ? LanesBelow(hm) : 64u] = static_cast<uint16_t>(ci);
          nHit = static_cast<uint32_t>(__popcll(hm));
          WaveSync();
        }
        if (mr * kPerRound < nHit) {
          const uint32_t k = mr * kPerRound + static_cast<uint32_t>(lane) / kWalkChunk;
          const uint32_t mi = lds.chunks[min(k, nHit - 1)] * kWalkChunk + static_cast<uint32_t>(lane) % kWalkChunk;
          const uint32_t ma = mfirst + 2 * min(mi, count - 1);
          m0 = groups[ma];
          m1 = groups[ma + 1];
          // (an operator member's lane reads some primitive's record and ignores it)
          const uint32_t md = AsU(m1.z);
          m2 = jb.sc.primA[DescType(md) >= kSphereT ? DescIndex(md) : 0u];
          const bool meets = (k < nHit) & (mi < count) &
                             BundleMeets(bundle, jb.pos, m0.x, m0.y, m0.z, m0.w, m1.x, m1.y,
                                         AsU(m1.w) != 0 ? 0.0f : from, AsU(m1.w) != 0 ? __builtin_inff() : to);
          todo = __ballot(meets) & (~uint64_t{0} << skip);
          skip = 0;
          if (todo == 0) mr++;
        }
        if (todo == 0 && mr * kPerRound >= nHit) {
          // on to the next chunk round
          cr++;
          mr = 0;
          nHit = 0;
        }
      }
      if (todo != 0) {
        const int l = __ffsll(static_cast<unsigned long long>(todo)) - 1;
        todo &= todo - 1;
        auto u = [&](float f) CSG_INLINE { return __uint_as_float(__builtin_amdgcn_readlane(AsU(f), l)); };
        const bool g = BoxHitExit<kFast>(r, u(m0.x), u(m0.y), u(m0.z), u(m0.w), u(m1.x), u(m1.y), leafExit);
        const uint64_t mm = __ballot(g) & M & ~dead;
        const uint32_t md = __builtin_amdgcn_readlane(AsU(m1.z), l);
        // where to go on after this member: its round's next lane, or the
        // round after it
        const uint32_t here = cr << 8 | mr << 6 | static_cast<uint32_t>(l + 1);
        if (todo == 0) {
          mr++;
          if (mr * kPerRound >= nHit) {
            cr++;
            mr = 0;
            nHit = 0;
          }
        }
        if (mm != 0) {
          if (DescType(md) >= kSphereT) {
            leafDesc = md;
            leafA = make_float4(u(m2.x), u(m2.y), u(m2.z), u(m2.w));
            leafMask = mm;
          } else {
            saveZones();
            enter(DescIndex(md), mm, kTileGroup, todo != 0 ? here : (cr << 8 | mr << 6));
          }
        }
      } else {
        const bool on = (M & me) != 0;
        if (zones) {
          float at;
          const bool in = inZone(M, base, at);
          dead |= __ballot(in | (on & (sureLevel > d)));
        }
        int n = on ? sp - base : 0;
        // one member's (Enter, Exit) or lone Exit is a list already
        const bool sorts = (n > 2) | ((n == 2) & !(EntryBits(list.At(base)) & kEnter));
        if (__ballot(sorts) != 0) {
          n = sorts ? n : 0;
          int len = 0;
          const bool done = __ballot(n > 8) == 0 ? Unite<8>(list, base, n, len)
                                                 : Unite<kTileSlots>(list, base, n, len);
          if (!done) {
            bool bad = false;
            len = UniteTies(list, base, n, teBits, bad);
            dead |= __ballot(bad);
          }
          sp = sorts ? base + len : sp;
        }
        state = kTileReturn;
      }
    }
    if (leafDesc != kNone) leaf(leafDesc, leafA, leafMask, leafExit, kGroups && (cut | (state == kTileGroup)));
  }
  const double e = list.At(0);
  const bool found = (sp > 0) & (EntryTime(e) != teBits);
  h = MissRecord();
  h.t = found ? __uint_as_float(EntryTime(e)) : h.t;
  h.bits = found ? EntryBits(e) : h.bits;
  full &= active;
  fail = dead & active & ~full;
}

// Tile coordinates and sample plane of a job's `local`-th tile.
struct TilePlace {
  uint32_t tx, ty, sample;
};
__device__ __forceinline__ TilePlace PlaceOf(const Job& jb, uint32_t local, bool morton) {
  uint32_t perSample = static_cast<uint32_t>(jb.tiles), sample = 0, t = local;
  if (jb.spp > 1) {
    perSample /= static_cast<uint32_t>(jb.spp);
    sample = local / perSample;
    t = local - sample * perSample;
  }
  const uint32_t tilesX = static_cast<uint32_t>(jb.tilesX);
  if (morton && tilesX == perSample / tilesX && (tilesX & (tilesX - 1)) == 0)
    return TilePlace{Compact1By1(t), Compact1By1(t >> 1), sample};
  uint32_t ty;
  if (t < 1u << 22) {
    // exact in floats but for one step either way
    ty = static_cast<uint32_t>(static_cast<float>(t) * __builtin_amdgcn_rcpf(static_cast<float>(tilesX)));
    ty = ty * tilesX > t ? ty - 1 : ty;
    ty = (ty + 1) * tilesX <= t ? ty + 1 : ty;
  } else {
    ty = t / tilesX;
  }
  return TilePlace{t - ty * tilesX, ty, sample};
}

// The job whose tiles hold queue index `q`: the last with tileBase <= q, by
// one 64-way step over every 16th job and one over the 16 that remain.
__device__ __forceinline__ uint32_t JobOfTile(const Job* jobs, uint32_t n, uint32_t q, int lane) {
  static_assert(kMaxBatchJobs <= 1024, "two steps of 64 and 16");
  const uint32_t a = 16u * static_cast<uint32_t>(lane);
  const bool le = a < n && static_cast<uint32_t>(jobs[a].tileBase) <= q;
  const uint32_t first = 16u * (static_cast<uint32_t>(__popcll(__ballot(le))) - 1u);
  const uint32_t b = first + (static_cast<uint32_t>(lane) & 15u);
  const bool le2 = lane < 16 && b < n && static_cast<uint32_t>(jobs[b].tileBase) <= q;
  return first + static_cast<uint32_t>(__popcll(__ballot(le2))) - 1u;
}

// Walks a tile's rays may take.
constexpr int kTilePasses = 24;
// State-machine steps a failed ray takes in its lane before the cooperative
// kernel gets it, in launches without groups whose trees have 8 operators or
// more (others finish it in its lane, or hand it over at once).  Each step
// holds the whole wave up for about a microsecond, and a launch that hands
// nothing over saves one ray's chain there, which small trees take with a few
// more steps.  0, 16, 32 and 64 steps: a union of 20 cubes on a grid at 640x360 67,
// 66, 45 and 45 us, of 30 223, 218, 214 and 267, of 64 cylinders 137, 145, 155
// and 186; a mixed tree of 200 at 1023x1023 393, 393, 402 and 427; a plate with 8
// holes at 1920x1080, exact mode, 75, 67, 68 and 67; 48 random trees in a batch
// 1426, 1422, 1422 and 1438.
constexpr int kTileSteps = 16, kTileSmallOps = 32, kTileSmallSteps = 32;

// Whether the cooperative kernel has been handed fewer rays than it has waves.
// Such rays are traced side by side, where a tile's stretches follow one
// another: a union of 1143 at 292x164 takes 427 to 637 us so, 630 to 1276 with
// stretches alone (30 rays overflow a list), at 1280x720 420 to 578 and 507 to
// 1034; of 4095 at 1920x1080, 4 samples, 8.1 and 7.7 ms (190 ms with all rays
// handed over).
__device__ __forceinline__ bool HandsOverFew(const RenderParams& p) {
  const uint32_t n = __hip_atomic_load(p.queue + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return p.heavyCap != 0 && __builtin_amdgcn_readfirstlane(n) < p.coopWaves;
}

// One wave, one tile.  kGroups: some scene of the launch has Union groups;
// without, the code is half as long and takes half the registers, and shorter
// lists do (4 waves a SIMD instead of 2).  Workgroups come from the hardware's
// dispatcher, which starts one every 0.2 ns over the chip: a grid of resident
// waves that claim their tiles pays an atomic for each, at 2.7 ns over the
// chip whatever the number of counters (two spheres taken from a cube at
// 1920x1080, 32,400 tiles: 72 us with claims, 26 us without).
template <bool kFast, bool kBatch, bool kGroups>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kGroups ? 2 : !kFast ? 3 : 4)))
TileKernel(RenderParams p) {
  extern __shared__ uint4 ldsBase[];
  __shared__ uint16_t table[kDecisionEntries];
  const int lane = threadIdx.x;
  TileLdsView lds;
  lds.lists = reinterpret_cast<double*>(ldsBase);
  lds.bundle = reinterpret_cast<float4*>(lds.lists + 64 * (p.tileSlots + 2));
  lds.chunks = reinterpret_cast<uint16_t*>(lds.bundle + 4);
  lds.bounds = reinterpret_cast<uint8_t*>(lds.chunks + 72);
  const uint32_t q = blockIdx.x;
  if (q >= static_cast<uint32_t>(p.numTiles)) return;
  uint32_t jobIndex = 0, local = q;
  if (kBatch) {
    jobIndex = __builtin_amdgcn_readfirstlane(JobOfTile(p.jobs, static_cast<uint32_t>(p.numJobs), q, lane));
  }
  const Job& jb = kBatch ? *(const Job*)(CSG_SCALAR Job*)(p.jobs + jobIndex) : p.job;
  if (kBatch) local = q - static_cast<uint32_t>(jb.tileBase);
  const TilePlace at = PlaceOf(jb, local, p.morton != 0);
  const int x0 = static_cast<int>(at.tx) * 8, y0 = static_cast<int>(at.ty) * 8;
  const int x = x0 + (lane & 7), y = y0 + (lane >> 3);
  const bool inside = x < jb.width && y < jb.height;
  TileScale scale;
  const TileBundle bundle = BundleOf(jb, x0, y0, scale);
  const bool rootOp = DescType(jb.sc.rootDesc) < kSphereT;
  bool meets = true;
  if (kFast && rootOp) {
    // a tile whose rays all miss the root's children's boxes (odd lanes
    // test the right one) is background
    const U32x16 o = ScalarRecord(kGroups ? jb.sc.tileOps : jb.sc.ops, 0);
    if (!(o[14] & kWalkGroupFlag)) {
      auto b = [&](int l, int rr) CSG_INLINE { return __uint_as_float((lane & 1) ? o[rr] : o[l]); };
      meets = __ballot(BundleMeets(bundle, jb.pos, b(0, 3), b(1, 7), b(2, 8), b(4, 9), b(5, 10), b(6, 11))) != 0;
    }
  }
  const uint32_t pixel = static_cast<uint32_t>(y) * static_cast<uint32_t>(jb.width) + static_cast<uint32_t>(x);
  float ox = 0.5f, oy = 0.5f;
  if (jb.spp > 1) {
    ox = JitterUnit(JitterHash(jb.seed, pixel, at.sample, 0));
    oy = JitterUnit(JitterHash(jb.seed, pixel, at.sample, 1));
  }
  RayF r{};
  if (meets) r = MakeRay<kFast>(jb, x, y, ox, oy);
  const size_t out = static_cast<size_t>(pixel) * static_cast<size_t>(jb.spp) + at.sample;
  const SceneView sv{jb.sc.ops, jb.sc.primA, jb.sc.primB, jb.sc.ops, 0u};
  Counts n{0, 0, 0, 0, 0, 0};
  Hit h = MissRecord();
  uint64_t fail = 0;
  const uint64_t active = __ballot(inside);
  if (!meets) {
  } else if (!rootOp) {
    // a primitive root, as in Trace
    h = Intersect<kFast, false>(sv, r, jb.sc.rootDesc, 0.0f, MissRecord(), n);
    if (Flags(h.bits) & kMissBit) h = MissRecord();
  } else if (!kGroups) {
    uint64_t failed, full;
    TileTrace<kFast, false>(jb, r, active, jb.sc.ops, lds, p.tileSlots, lane, 0.0f, __builtin_inff(), h, failed,
                            full);
    fail = failed | full;
  } else {
    lds.bundle[0] = make_float4(bundle.a[0], bundle.a[1], bundle.a[2], bundle.b[0]);
    lds.bundle[1] = make_float4(bundle.b[1], bundle.b[2], bundle.c[0], bundle.c[1]);
    lds.bundle[2] = make_float4(bundle.c[2], bundle.k[0], bundle.k[1], bundle.k[2]);
    lds.bundle[3] = make_float4(scale.lo, scale.hi, 0.0f, 0.0f);
    WaveSync();
    // The whole ray first.  Rays that fail, on a tie in a Union group for
    // the most part, go to the cooperative kernel; without one, they are walked
    // again through the tree as it is, where every comparison is the
    // machine's own (a walk of all 512 spheres for one ray kept the frame of
    // some views 700 us instead of 200).  Then the lanes whose lists overflow,
    // unless the cooperative kernel has room (HandsOverFew), again over
    // consecutive stretches of the ray (half its extent in the root's
    // children's boxes, halved while a list overflows, grown after each
    // that fits, the last one open-ended), to its end.  (Where all primitives
    // stay in their boxes the cooperative kernel merges intervals, which is
    // always faster: the 512-sphere frame 209 us, 306 with stretches.)
    uint64_t todo = active, over = 0;
    float ts = 0.0f, te = __builtin_inff(), w = 0.0f, end = 0.0f;
    const float4* ops = jb.sc.tileOps;
    uint32_t stage = 0;  // 0, 1 the whole ray (1: without groups), 2 stretches
    for (int pass = 0; pass < kTilePasses; pass++) {
      uint64_t failed, full;
      Hit first;
      TileTrace<kFast, true>(jb, r, todo, ops, lds, p.tileSlots, lane, ts, te, first, failed, full);
      const bool mine = ((todo & ~failed & ~full) >> lane) & 1u;
      if (stage < 2) {
        h.t = mine ? first.t : h.t;
        h.bits = mine ? first.bits : h.bits;
        over |= full;
        if (stage == 0 && failed != 0 && ops != jb.sc.ops && p.heavyCap == 0) {
          ops = jb.sc.ops;
          todo = failed;
          stage = 1;
          continue;
        }
        fail |= failed;
        todo = over;
        if (jb.sc.conservative || over == 0 || HandsOverFew(p)) break;
        const U32x16 o = ScalarRecord(jb.sc.tileOps, 0);
        float nL, xL, nR, xR;
        Slab<true>(r, __uint_as_float(o[0]), __uint_as_float(o[1]), __uint_as_float(o[2]), __uint_as_float(o[4]),
                   __uint_as_float(o[5]), __uint_as_float(o[6]), nL, xL);
        Slab<true>(r, __uint_as_float(o[3]), __uint_as_float(o[7]), __uint_as_float(o[8]), __uint_as_float(o[9]),
                   __uint_as_float(o[10]), __uint_as_float(o[11]), nR, xR);
        float t0 = (over >> lane) & 1u ? fmaxf(0.0f, fminf(nL, nR)) : __builtin_inff();
        float t1 = (over >> lane) & 1u ? fmaxf(xL, xR) : 0.0f;
        for (int off = 32; off > 0; off >>= 1) {
          t0 = fminf(t0, __shfl_xor(t0, off, 64));
          t1 = fmaxf(t1, __shfl_xor(t1, off, 64));
        }
        t0 = Uniform(t0);
        end = Uniform(t1);
        if (!(end > t0) || !(end < __builtin_inff())) break;
        w = Uniform(0.5f * (end - t0));
        te = Uniform(t0 + w);
        ops = jb.sc.tileOps;
        stage = 2;
      } else if (full != 0) {
        fail |= failed;
        todo &= ~failed;
        w = Uniform(0.5f * w);
        te = Uniform((ts > 0.0f ? ts : te - 2.0f * w) + w);
      } else {
        fail |= failed;
        todo &= ~failed;
        const bool take = mine & ((Flags(h.bits) & kMissBit) != 0);
        h.t = take ? first.t : h.t;
        h.bits = take ? first.bits : h.bits;
        if (!(te < __builtin_inff())) {
          todo = 0;
          break;
        }
        ts = te;
        w = Uniform(1.5f * w);
        te = Uniform(ts + w);
      }
      if (te >= end) te = __builtin_inff();
      if (todo == 0 || !(te > ts)) break;
    }
    fail |= todo;  // not resolved
  }
  bool store = inside;
  if (fail != 0) {
    if (lane < kDecisionEntries) table[lane] = kDecisions.v[lane];
    WaveSync();
    // The state machine, its stacks in the lists' place, as many lanes at a
    // time as fit; a ray it does not finish in kTileSteps goes to the
    // cooperative kernel, or, if there is none or its list is full, is
    // finished here.
    const int depth = max(p.stackSlots, 1), cols = min(64, 64 * (p.tileSlots + 2) / depth);
    bool need = (fail >> lane) & 1u;
    const int handSteps = kGroups ? 0 : (p.coopOps < kTileSmallOps ? kTileSmallSteps : kTileSteps);
    for (int steps = p.heavyCap != 0 ? handSteps : 0x7FFFFFFF;; steps = 0x7FFFFFFF) {
      bool left = steps == 0;
      for (int first = 0; first < 64 && steps != 0; first += cols) {
        if (need & (lane >= first) & (lane < first + cols))
          h = Trace<kFast, false>(sv, r, jb.sc.rootDesc, reinterpret_cast<uint2*>(lds.lists) + (lane - first), cols,
                                  depth, table, n, steps, nullptr, nullptr, 0, left);
      }
      need &= left;
      if (__ballot(need) == 0) break;
      if (need) {
        const uint32_t slot = atomicAdd(p.queue + 2, 1u);
        if (slot < p.heavyCap) {
          const bool dir = slot < DirCap(p);
          p.heavy[slot] = make_uint2(jobIndex | (dir ? kDirFlag : 0u), static_cast<uint32_t>(out));
          if (dir) Directions(p)[slot] = make_uint4(AsU(r.dx), AsU(r.dy), AsU(r.dz), 0u);
          store = false;
          need = false;
        }
      }
      if (__ballot(need) == 0) break;
    }
  }
  if (store) ShadeAndStore<kFast>(jb, sv, r, h, out);
}
