// Collapses an SBVH into four-wide nodes; see wide_nodes.hpp.
#include "wide_nodes.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <future>
#include <limits>
#include <system_error>
#include <thread>

namespace phx {
namespace {

// Runs task(0) to task(count - 1) on up to `threads` threads, this one among them.
template <class Task>
void runTasks(uint32_t count, uint32_t threads, const Task& task)
{
	std::atomic<uint32_t> next{0};
	auto work = [&] {
		for (uint32_t i = next++; i < count; i = next++) task(i);
	};
	std::vector<std::future<void>> others;
	for (uint32_t t = 1; t < std::min(threads, count); t++) {
		try {
			others.push_back(std::async(std::launch::async, work));
		} catch (const std::system_error&) {
			break;  // no more threads to be had
		}
	}
	work();
	for (std::future<void>& o : others) o.get();
}

// A binary tree, and a flag per node whose child boxes stick out of its own (none: empty).
struct Tree {
	const PhxBVHNode* nodes;
	std::vector<uint8_t> loose;
	bool isLoose(int32_t node) const { return !loose.empty() && loose[node]; }
};

bool sticksOut(const PhxBVHNode* nodes, const PhxBVHNode& nd, int c)
{
	const float *b = nd.fData + 6 * c, *f = nodes[nd.iData[c]].fData;
	bool inside = true;
	for (int k = 0; k < 3; k++)
		inside &= f[k] >= b[k] && f[k + 6] >= b[k] && f[k + 3] <= b[k + 3] && f[k + 9] <= b[k + 3];
	return !inside;
}

// Whether every child box lies within +-2^126 and is not inverted (false for NaN too); sets tree.loose.
bool eligible(Tree& tree, uint32_t n, uint32_t threads)
{
	constexpr uint32_t kRange = 8192;
	std::atomic<bool> bad{false}, anyLoose{false};
	runTasks((n + kRange - 1u) / kRange, threads, [&](uint32_t range) {
		bool good = true, out = false;
		for (uint32_t i = range * kRange; i < std::min(n, (range + 1u) * kRange); i++) {
			const PhxBVHNode& nd = tree.nodes[i];
			for (int c = 0; c < 2; c++) {
				const float* b = nd.fData + 6 * c;
				for (int k = 0; k < 3; k++)
					good &= std::fabs(b[k]) <= 0x1p126f && std::fabs(b[k + 3]) <= 0x1p126f && b[k] <= b[k + 3];
				if (nd.iData[2 + c] == 0) out |= sticksOut(tree.nodes, nd, c);
			}
		}
		if (!good) bad = true;
		if (out) anyLoose = true;
	});
	if (bad) return false;
	if (anyLoose) {
		tree.loose.resize(n);
		for (uint32_t i = 0; i < n; i++)
			for (int c = 0; c < 2; c++)
				if (tree.nodes[i].iData[2 + c] == 0 && sticksOut(tree.nodes, tree.nodes[i], c))
					tree.loose[tree.nodes[i].iData[c]] = 1;
	}
	return true;
}

// One slot while a wide node is put together: a leaf, or an inner binary node.
struct Slot {
	const float* box;
	uint32_t ref;    // leaf: the finished reference; inner: the binary node's index
	bool leaf;
	bool loose;      // inner: kWideLoose
	float area;      // half surface area of an inner slot that may be opened, else negative
};

float halfArea(const float* b)
{
	const float x = b[3] - b[0], y = b[4] - b[1], z = b[5] - b[2];
	return x * y + y * z + z * x;
}

// Whether a wide node may hold the children of binary node `node` in place of it, whose box is `b`: no ray
// passes a child's box that does not pass b (wide_nodes.hpp: flat boxes), and no child is loose, which has
// to be decided when this node is taken.
bool mayOpen(const Tree& t, int32_t node, const float* b)
{
	const PhxBVHNode& nd = t.nodes[node];
	if (!t.loose.empty())
		for (int c = 0; c < 2; c++)
			if (t.loose[node] || (nd.iData[2 + c] == 0 && t.loose[nd.iData[c]])) return false;
	for (int c = 0; c < 2; c++)
		for (int k = 1; k < 3; k++) {
			const float* f = nd.fData + 6 * c;
			if (f[k] == f[k + 3] && f[k] == b[k + 3] && b[k] < b[k + 3]) return false;
		}
	return true;
}

// The slots of binary node `node` in castRay's order (see wide_nodes.hpp); returns how many (2).
int expand(const Tree& tree, uint32_t node, Slot out[2])
{
	const PhxBVHNode& nd = tree.nodes[node];
	int k = 0;
	for (int c = 0; c < 2; c++)
		if (nd.iData[2 + c] != 0) {
			const uint32_t cnt = uint32_t(nd.iData[2 + c]);
			uint32_t ref = kWideLeaf | uint32_t(~nd.iData[c]) | ((cnt <= 3u ? cnt : 0u) << kWideCountShift);
			if (c == 0 && nd.iData[3] != 0) ref |= kWidePair;
			out[k++] = Slot{nd.fData + 6 * c, ref, true, false, 0.0f};
		}
	for (int c = 1; c >= 0; c--)
		if (nd.iData[2 + c] == 0) {
			const float* b = nd.fData + 6 * c;
			const int32_t at = nd.iData[c];
			out[k++] = Slot{b, uint32_t(at), false, tree.isLoose(at), mayOpen(tree, at, b) ? halfArea(b) : -1.0f};
		}
	return k;
}

// A wide node's slots: binary node `root` with the inner slots of largest area opened in place
// until four are used.
int collapse(const Tree& tree, uint32_t root, Slot s[4])
{
	int k = expand(tree, root, s);
	while (k < 4) {
		int best = -1;
		for (int i = 0; i < k; i++)
			if (!s[i].leaf && s[i].area >= 0.0f && (best < 0 || s[i].area > s[best].area)) best = i;
		if (best < 0) break;
		Slot two[2];
		expand(tree, s[best].ref, two);
		for (int i = k; i > best + 1; i--) s[i] = s[i - 1];
		s[best] = two[0];
		s[best + 1] = two[1];
		k++;
	}
	return k;
}

WideNode emptyNode()
{
	WideNode w;
	const float nan = std::numeric_limits<float>::quiet_NaN();
	for (WideNode::Slot& s : w.slot) s = WideNode::Slot{{nan, nan, nan}, 0u, {nan, nan, nan}, nan};
	return w;
}

void setSlot(WideNode::Slot& s, const float* box, uint32_t ref)
{
	std::memcpy(s.min, box, sizeof(s.min));
	std::memcpy(s.max, box + 3, sizeof(s.max));
	s.ref = ref;
}

uint32_t innerRef(uint32_t at, bool isLoose) { return at | (isLoose ? kWideLoose : 0u); }

// A node to fill: the binary node whose subtree it covers and the slots pending beside it.
struct Item {
	uint32_t at, node, pending;
};

// The wide node of `it`, its inner slots numbered from firstChild on; they are appended to `next`.
WideNode fill(const Tree& tree, const Item& it, uint32_t firstChild, std::vector<Item>& next, uint32_t& maxPending)
{
	Slot t[4];
	const int k = collapse(tree, it.node, t);
	maxPending = std::max(maxPending, it.pending + uint32_t(k - 1));
	WideNode w = emptyNode();
	for (int i = 0; i < k; i++) {
		setSlot(w.slot[i], t[i].box, t[i].leaf ? t[i].ref : innerRef(firstChild, t[i].loose));
		if (!t[i].leaf) next.push_back(Item{firstChild++, t[i].ref, it.pending + uint32_t(k - 1 - i)});
	}
	return w;
}

// Adds `base` to a node's inner references and sets lastMax.
void finish(WideNode& w, uint32_t base)
{
	for (int i = 0; i < 4; i++)
		if (!(w.slot[i].ref & kWideLeaf) && w.slot[i].min[0] == w.slot[i].min[0]) w.slot[i].ref += base;
	for (int i = 0; i < 3; i++) w.slot[i].lastMax = w.slot[3].max[i];
}

}  // namespace

std::vector<WideNode> buildWide(const PhxBVHNode* nodes, uint32_t numNodes, uint32_t topCap, bool* loose)
{
	std::vector<WideNode> out;
	// (At least 8,192 nodes a thread.)
	const uint32_t threads = std::min(std::min(8u, std::max(1u, numNodes / 8192u)), std::max(1u, std::thread::hardware_concurrency()));
	Tree tree{nodes, {}};
	const bool fits = eligible(tree, numNodes, threads);
	if (loose) *loose = fits && !tree.loose.empty();
	if (!fits || (!loose && !tree.loose.empty())) return out;

	std::vector<Item> queue;  // breadth first up to topCap nodes
	if (threads == 1u) out.reserve(size_t(numNodes) / 2 + 8);
	out.push_back(emptyNode());
	uint32_t maxPending = 0;

	// The root: its slots become nodes 1..k. Leaves get a node that holds just them.
	Slot s[4];
	const int rootSlots = collapse(tree, 0, s);
	struct RootSlot {
		int first, count;  // range of s
	};
	RootSlot rs[4];
	int numRoot = 0;
	for (int i = 0; i < rootSlots; i++) {
		const int count = s[i].leaf && (s[i].ref & kWidePair) ? 2 : 1;
		rs[numRoot++] = RootSlot{i, count};
		i += count - 1;
	}
	for (int j = 0; j < numRoot; j++) {
		const Slot& a = s[rs[j].first];
		setSlot(out[0].slot[j], a.box, innerRef(uint32_t(j + 1), a.loose));
		if (rs[j].count == 2) {
			const Slot& b = s[rs[j].first + 1];
			for (int k = 0; k < 3; k++) {
				out[0].slot[j].min[k] = std::min(a.box[k], b.box[k]);
				// (A float more: flat at the maximum, a leaf may be passed by a ray that does not pass there.)
				out[0].slot[j].max[k] = std::nextafter(std::max(a.box[k + 3], b.box[k + 3]), HUGE_VALF);
			}
		}
		out.push_back(emptyNode());
		const uint32_t pending = uint32_t(numRoot - 1 - j);
		if (a.leaf) {
			for (int i = 0; i < rs[j].count; i++)
				setSlot(out[size_t(j) + 1].slot[i], s[rs[j].first + i].box, s[rs[j].first + i].ref);
			maxPending = std::max(maxPending, pending + 1u);
		} else {
			queue.push_back(Item{uint32_t(j + 1), a.ref, pending});
		}
	}
	maxPending = std::max(maxPending, uint32_t(numRoot - 1));

	size_t head = 0;
	while (head < queue.size() && out.size() < topCap) {
		const Item it = queue[head++];
		const size_t before = queue.size();
		const WideNode w = fill(tree, it, uint32_t(out.size()), queue, maxPending);
		out[it.at] = w;
		out.resize(out.size() + (queue.size() - before));
	}

	// The rest depth first: a node's children are numbered when it is filled (siblings side by side), the
	// first slot's subtree before the next one's. The subtrees of a run of queue items follow one another
	// in the array, so runs are built by themselves, each from its own index 0 on (one run: in `out`).
	struct Run {
		std::vector<WideNode> nodes;
		uint32_t maxPending = 0, base = 0;
	};
	const uint32_t items = uint32_t(queue.size() - head);
	std::vector<Run> runs(std::min(items, threads == 1u ? 1u : 8u * threads));
	const bool one = runs.size() == 1u;
	auto firstOf = [&](uint32_t run) { return head + size_t(items) * run / runs.size(); };
	runTasks(uint32_t(runs.size()), threads, [&](uint32_t r) {
		Run& run = runs[r];
		std::vector<WideNode>& built = one ? out : run.nodes;
		std::vector<Item> stack, kids;
		for (size_t i = firstOf(r); i < firstOf(r + 1u); i++) {
			bool top = true;  // the item's own node is in `out`
			stack.push_back(queue[i]);
			while (!stack.empty()) {
				const Item it = stack.back();
				stack.pop_back();
				kids.clear();
				const WideNode w = fill(tree, it, uint32_t(built.size()), kids, run.maxPending);
				(top ? out : built)[it.at] = w;
				top = false;
				built.resize(built.size() + kids.size());
				stack.insert(stack.end(), kids.rbegin(), kids.rend());
			}
		}
	});
	size_t total = out.size();
	for (Run& run : runs) {
		run.base = one ? 0u : uint32_t(total);
		total += run.nodes.size();
		maxPending = std::max(maxPending, run.maxPending);
	}
	if (maxPending > kWideMaxPending || total > kWideIndex) return {};
	if (one || runs.empty()) {
		for (WideNode& w : out) finish(w, 0u);
		return out;
	}
	const size_t tops = out.size();
	out.resize(total);
	std::vector<uint8_t> moved(tops, 0);  // filled by a run: its references count from the run's base
	runTasks(uint32_t(runs.size()), threads, [&](uint32_t r) {
		Run& run = runs[r];
		for (size_t i = firstOf(r); i < firstOf(r + 1u); i++) {
			finish(out[queue[i].at], run.base);
			moved[queue[i].at] = 1;
		}
		for (size_t i = 0; i < run.nodes.size(); i++) {
			finish(run.nodes[i], run.base);
			out[run.base + i] = run.nodes[i];
		}
		run.nodes = {};
	});
	for (size_t i = 0; i < tops; i++)
		if (!moved[i]) finish(out[i], 0u);
	return out;
}

}  // namespace phx
