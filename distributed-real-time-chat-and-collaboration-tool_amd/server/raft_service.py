"""``raft.RaftNode`` gRPC service: the chat application over Raft.

RPC semantics, response messages and log-entry payloads follow the reference
handlers (server/raft_node.py:1401-2347); deliberate fixes are
numbered by the quirk of the reference they address:

  Q1  writes are acknowledged after majority commit (RaftConfig.local_commit
      restores leader-local commit);
  Q3  AI calls run OUTSIDE every lock, with a circuit breaker instead of a
      3 s re-probe per call when the LLM service is down;
  Q6  tokens verify by signature + replicated user (valid on every node,
      survive failover) unless ``token_mode="reference"``;
  Q8  an auto-join on SendMessage is replicated (JOIN_CHANNEL), not local;
  Q9  GetMessages / GetDirectMessages honour ``offset``;
  Q11 the default users/channels are seeded through the log (genesis entries
      proposed once by the first leader of a fresh cluster: identical bcrypt
      hashes, ids and timestamps on every replica) unless ``seed_mode="local"``
      restores the reference's per-node seeding;
  --  logout is replicated (REVOKE_TOKEN), so a logged-out token stays invalid
      on every node and across failover;
  --  writes carrying the optional ``request_id`` (an additive proto field)
      are idempotent: the id becomes the message / DM / file id, which the
      state machine already de-duplicates, so a client retry after a
      DEADLINE_EXCEEDED cannot duplicate the write.
"""
from __future__ import annotations

import datetime as _dt
import hashlib
import logging
import mimetypes
import threading
import time
import uuid
from dataclasses import dataclass, field

import grpc

from ..protos import LLM_SERVICE, llm_pb, make_stub, raft_pb
from ..raft.core import NotLeaderError, RaftConfig
from ..raft.node import RaftRuntime
from ..utils import auth
from ..utils.metrics import METRICS
from ..raft.state_machine import DEFAULT_USERS as DEFAULT_USERS_ALL

log = logging.getLogger(__name__)

DEFAULT_PUBLIC = ("general", "random", "tech")

# canned AI fallbacks (server/raft_node.py:1997-2205)
FB_SMART_DOWN = ["I agree", "That's interesting", "Tell me more"]
FB_SMART_ERR = ["Sounds good", "I understand", "Interesting"]
FB_SUGGEST_DOWN = (["continue the thought", "ask a question", "share more"],
                   ["current topic", "related discussion"])
FB_SUGGEST_ERR = (["continue the conversation", "ask for details", "share thoughts"],
                  ["current discussion"])
LLM_DOWN_ANSWER = ("LLM service is not available. Please start the LLM server: "
                   "python -m drtc_amd.llm.server")


@dataclass
class NodeConfig:
    node_id: int = 1
    port: int = 50051
    peers: dict = field(default_factory=dict)       # id -> "host:port" (may include self)
    data_root: str = "."
    storage: str = "native"                         # native | pickle
    raft: RaftConfig = field(default_factory=RaftConfig)
    llm_address: str | None = "localhost:50055"
    jwt_secret: str = "raft-chat-secret-key"
    token_ttl_hours: float = 24.0
    token_mode: str = "replicated"                  # replicated | reference
    bcrypt_rounds: int = 12
    write_timeout: float = 5.0
    grpc_workers: int = 32
    advertise_host: str = "localhost"
    fsync: bool = True   # durable votes / log appends before acknowledging (Raft safety)
    seed_defaults: bool = True
    seed_mode: str = "log"                          # log (replicated genesis) | local (reference)
    snapshot_every: int = 0                         # compact the log every N applied entries (0: never)
    llm_timeouts: dict = field(default_factory=lambda: {
        "smart": 20.0, "summary": 10.0, "answer": 10.0, "suggest": 20.0})
    # per-feature LLM services (None: ``llm_address``, the reference's single LLM server,
    # ref server/raft_node.py:372).  One node can route each AI RPC to the engine group
    # serving that feature's model (for instance Gemma-2B smart reply, 8B summarize, 70B ask,
    # Mixtral suggestions) - ref call sites :2018 / :2084 / :2126 / :2187.
    llm_smart: str | None = None
    llm_summary: str | None = None
    llm_ask: str | None = None
    llm_suggest: str | None = None
    forward_timeout_s: float = 5.0                  # follower -> leader forwarded calls

    def llm_routes(self) -> dict:
        """feature -> LLM service address (the per-feature override or ``llm_address``)."""
        return {"smart": self.llm_smart or self.llm_address,
                "summary": self.llm_summary or self.llm_address,
                "answer": self.llm_ask or self.llm_address,
                "suggest": self.llm_suggest or self.llm_address}


class LLMClient:
    """Node -> llm.LLMService client (one HTTP/2 connection) with a circuit breaker."""

    def __init__(self, address: str | None, cooldown: float = 5.0):
        self.address = address
        self.cooldown = cooldown
        self._down_until = 0.0
        self.stub = None
        if address:
            opts = [("grpc.keepalive_time_ms", 30000), ("grpc.keepalive_timeout_ms", 5000)]
            self.channel = grpc.insecure_channel(address, options=opts)
            self.stub = make_stub(self.channel, LLM_SERVICE)

    def available(self) -> bool:
        return self.stub is not None and time.monotonic() >= self._down_until

    def call(self, method: str, req, timeout: float):
        try:
            return getattr(self.stub, method)(req, timeout=timeout)
        except grpc.RpcError as e:
            if e.code() in (grpc.StatusCode.UNAVAILABLE,):
                self._down_until = time.monotonic() + self.cooldown
            raise


class ChatNode:
    """All 25 raft.RaftNode RPCs. Consensus RPCs delegate to RaftRuntime."""

    def __init__(self, cfg: NodeConfig):
        self.cfg = cfg
        self.sessions: dict[str, dict] = {}
        # node-local fast path for logouts (token -> exp), pruned as tokens
        # expire; the replicated REVOKE_TOKEN record is authoritative
        self.revoked: dict[str, int] = {}
        self.local_lock = threading.Lock()

        def seed(state):
            if cfg.seed_defaults:
                salt = lambda: auth.bcrypt_gensalt(cfg.bcrypt_rounds)  # noqa: E731
                state.seed_defaults(lambda pw: auth.bcrypt_hashpw(pw, salt()))

        local_seed = cfg.seed_defaults and cfg.seed_mode == "local"
        self.rt = RaftRuntime(cfg.node_id, cfg.port, cfg.peers, cfg.data_root, cfg.storage,
                              cfg.raft, fsync=cfg.fsync, seed_defaults=seed if local_seed else None,
                              snapshot_every=cfg.snapshot_every)
        self.state = self.rt.state
        # one client (channel + circuit breaker) per distinct address; features that share
        # an address share its client
        by_addr: dict = {}
        self.llms = {}
        for f, a in cfg.llm_routes().items():
            if a not in by_addr:
                by_addr[a] = LLMClient(a)
            self.llms[f] = by_addr[a]
        self.llm = self.llms["smart"]
        self.genesis_done = threading.Event()
        if not (cfg.seed_defaults and cfg.seed_mode == "log"):
            self.genesis_done.set()
        self._running = False

    # ------------------------------------------------------------ helpers
    def start(self):
        self.rt.start()
        self._running = True
        if not self.genesis_done.is_set():
            threading.Thread(target=self._genesis_loop, name=f"genesis-{self.cfg.node_id}",
                             daemon=True).start()
        return self

    def stop(self):
        self._running = False
        self.rt.stop()

    def _genesis_loop(self) -> None:
        """Seed the default users/channels through the log: once
        this node leads and has applied its whole log (its NOOP committed, so
        every earlier entry is in the state), propose whatever default record
        is still missing.  Apply is idempotent by username / channel id, so a
        leader change halfway through only completes the set."""
        while self._running and not self.genesis_done.is_set():
            time.sleep(0.02)
            info = self.rt.leader_info()
            with self.rt.state_lock:
                have = all(n in self.st.users for n, _ in DEFAULT_USERS_ALL) and all(
                    c in self.st.channels for c in DEFAULT_PUBLIC)
            if have:
                self.genesis_done.set()
                return
            if not info["is_leader"] or self.rt.core.last_applied < info["log"] - 1:
                continue
            salt = lambda: auth.bcrypt_gensalt(self.cfg.bcrypt_rounds)  # noqa: E731
            with self.rt.state_lock:
                entries = self.st.genesis_entries(lambda pw: auth.bcrypt_hashpw(pw, salt()))
            for cmd, data in entries:
                if self._propose(cmd, data) is not None:
                    break  # lost leadership / timeout: re-evaluate

    def _await_genesis(self, timeout: float = 5.0) -> None:
        """Early requests on a fresh cluster wait briefly for the defaults."""
        if not self.genesis_done.is_set():
            self.genesis_done.wait(timeout)

    @staticmethod
    def _token_hash(token: str) -> str:
        return hashlib.sha256(token.encode()).hexdigest()

    @property
    def st(self):
        return self.state

    def _token(self, user_id: str, username: str) -> str:
        payload = {"user_id": user_id, "username": username,
                   "exp": _dt.datetime.now(_dt.timezone.utc) + _dt.timedelta(hours=self.cfg.token_ttl_hours)}
        if self.cfg.token_mode != "reference":
            # a random token id: logins within the same second (same exp) must not mint
            # the token a logout just revoked (replicated revocation is by token hash);
            # an extra claim, so reference verifiers (PyJWT) still accept it
            payload["jti"] = uuid.uuid4().hex
        return auth.jwt_encode(payload, self.cfg.jwt_secret)

    def _verify(self, token: str) -> dict | None:
        try:
            payload = auth.jwt_decode(token, self.cfg.jwt_secret)
        except auth.InvalidTokenError:
            return None
        name = payload.get("username")
        with self.rt.state_lock:
            user = self.st.users.get(name) if name else None
            if user is None:
                return None
            if self.cfg.token_mode == "reference":
                if user.get("active_token") == token or token in self.sessions:
                    return payload
                return None
        if token in self.revoked:
            return None
        with self.rt.state_lock:
            if self.st.revoked_tokens and self._token_hash(token) in self.st.revoked_tokens:
                return None
        return payload

    def _propose(self, command: str, data: dict) -> str | None:
        """None on success, else an error message."""
        try:
            ok = self.rt.propose(command, data, self.cfg.write_timeout)
        except NotLeaderError:
            return "Not the leader"
        METRICS.inc(f"raft.propose.{command}")
        return None if ok else "Replication failed"

    # ------------------------------------------------------------ consensus
    def RequestVote(self, request, context):
        return self.rt.RequestVote(request, context)

    def AppendEntries(self, request, context):
        return self.rt.AppendEntries(request, context)

    def GetLeaderInfo(self, request, context):
        info = self.rt.leader_info()
        lid = info["leader_id"]
        if info["is_leader"]:
            addr = f"{self.cfg.advertise_host}:{self.cfg.port}"
        elif lid is not None and lid in self.rt.peers:
            addr = self.rt.peers[lid]
        else:
            addr = ""
        return raft_pb.GetLeaderResponse(is_leader=info["is_leader"],
                                         leader_id=lid if lid is not None else -1,
                                         leader_address=addr, term=info["term"], state=info["state"])

    # ------------------------------------------------------------ auth
    def Signup(self, request, context):
        username = request.username.strip()
        self._await_genesis()
        with self.rt.state_lock:
            if username in self.st.users:
                return raft_pb.SignupResponse(success=False, message="Username already exists")
        if not self.rt.is_leader():
            return raft_pb.SignupResponse(success=False, message="Not the leader")
        user_id = str(uuid.uuid4())
        hashed = auth.bcrypt_hashpw(request.password.encode(), auth.bcrypt_gensalt(self.cfg.bcrypt_rounds))
        display = request.display_name or username
        data = {"user_id": user_id, "username": username, "password": hashed.decode("latin1"),
                "email": request.email, "display_name": display, "is_admin": False}
        err = self._propose("CREATE_USER", data)
        if err:
            return raft_pb.SignupResponse(success=False, message=err)
        info = raft_pb.UserInfo(user_id=user_id, username=username, display_name=display,
                                email=request.email, is_admin=False, status="offline")
        return raft_pb.SignupResponse(success=True, message="Account created!", user_info=info)

    def Login(self, request, context):
        username = request.username.strip()
        self._await_genesis()
        with self.rt.state_lock:
            user = self.st.users.get(username)
            stored = user["password"] if user else None
        if user is None:
            return raft_pb.LoginResponse(success=False, message="Invalid credentials")
        if isinstance(stored, str):
            stored = stored.encode("latin1")
        if not auth.bcrypt_checkpw(request.password.encode("utf-8"), stored):
            return raft_pb.LoginResponse(success=False, message="Invalid credentials")
        token = self._token(user["id"], username)
        now = _dt.datetime.now(_dt.timezone.utc)
        with self.rt.state_lock:
            self.sessions[token] = {"user_id": user["id"], "username": username, "login_time": now}
            user["active_token"] = token
            user["token_issued_at"] = now.isoformat()
            user["status"] = "online"
            self.st.online_users.add(username)
            self.st.dirty.add("users")
            general = self.st.channel_by_name("general")
            need_join = general is not None and user["id"] not in general["members"]
        if need_join and self.rt.is_leader():
            self._propose("JOIN_CHANNEL", {"channel_id": general["id"], "user_id": user["id"]})
        info = raft_pb.UserInfo(user_id=user["id"], username=username,
                                display_name=user.get("display_name", username),
                                email=user.get("email", ""), is_admin=user.get("is_admin", False),
                                status="online")
        return raft_pb.LoginResponse(success=True, token=token, message="Login successful",
                                     user_info=info)

    def Logout(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.StatusResponse(success=False, message="Invalid token")
        name = p["username"]
        # replicated through the leader, like every other write: the token then stays
        # invalid on every node and after failover.  The reference logs out on ANY node
        # (ref server/raft_node.py:1751) and its CLI neither redirects a logout nor keeps its
        # session when one fails (client/chat_client.py:568), so a follower forwards the
        # call to the leader; either way it drops the session and the presence locally.
        if not self.rt.is_leader():
            return self._forward_logout(request, name)
        err = self._propose("REVOKE_TOKEN", {"username": name,
                                             "token_hash": self._token_hash(request.token),
                                             "exp": int(p.get("exp", 0)), "ts": int(time.time())})
        with self.rt.state_lock:
            self.sessions.pop(request.token, None)
            now = int(time.time())
            for t in [t for t, exp in self.revoked.items() if exp < now]:
                del self.revoked[t]
            self.revoked[request.token] = int(p.get("exp", 0)) or now + 86400
            u = self.st.users.get(name)
            if u is not None:
                u["active_token"] = None
                u["status"] = "offline"
                self.st.online_users.discard(name)
                self.st.dirty.add("users")
        if err:  # revoked on this node; the replicated revocation did not commit
            return raft_pb.StatusResponse(success=False, message=f"Logout not replicated: {err}")
        return raft_pb.StatusResponse(success=True, message="Logged out")

    def _drop_session(self, token: str, name: str) -> None:
        with self.rt.state_lock:
            self.sessions.pop(token, None)
            u = self.st.users.get(name)
            if u is not None:
                u["status"] = "offline"
                self.st.online_users.discard(name)
                self.st.dirty.add("users")

    def _forward_logout(self, request, name: str):
        """Logout received by a follower: relay it to the current leader (which replicates
        the revocation to every node, this one included); the local session goes either way."""
        info = self.rt.leader_info()
        lid = info.get("leader_id")
        stub = self.rt.stubs.get(lid) if lid is not None else None
        self._drop_session(request.token, name)
        if stub is None:
            return raft_pb.StatusResponse(success=False,
                                          message="Logout not replicated: no leader known")
        try:
            return stub.Logout(request, timeout=self.cfg.forward_timeout_s)
        except grpc.RpcError as e:
            return raft_pb.StatusResponse(
                success=False, message=f"Logout not replicated: leader unreachable ({e.code().name})")

    # ------------------------------------------------------------ channels
    def CreateChannel(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.StatusResponse(success=False, message="Invalid token")
        if not self.rt.is_leader():
            return raft_pb.StatusResponse(success=False, message="Not the leader")
        name = request.channel_name.strip()
        with self.rt.state_lock:
            for ch in self.st.channels.values():
                if ch["name"].lower() == name.lower():
                    return raft_pb.StatusResponse(success=False, message=f"Channel #{name} already exists")
        cid = str(uuid.uuid4())
        data = {"channel_id": cid, "name": name,
                "description": request.description or f"Channel {name}",
                "is_private": request.is_private, "members": [p["user_id"]], "admins": [p["user_id"]],
                "created_at": _dt.datetime.now(_dt.timezone.utc).isoformat()}
        err = self._propose("CREATE_CHANNEL", data)
        if err:
            return raft_pb.StatusResponse(success=False, message=err)
        return raft_pb.StatusResponse(success=True, channel_id=cid,
                                      message=f"Channel #{name} created! You are now in the channel.")

    def GetChannels(self, request, context):
        if not self._verify(request.token):
            return raft_pb.ChannelListResponse(success=False, channels=[])
        with self.rt.state_lock:
            chans = [raft_pb.Channel(channel_id=c["id"], name=c["name"], description=c["description"],
                                     is_private=c["is_private"], member_count=len(c["members"]))
                     for c in self.st.channels.values()]
        return raft_pb.ChannelListResponse(success=True, channels=chans)

    def JoinChannel(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.StatusResponse(success=False, message="Invalid token")
        with self.rt.state_lock:
            ch = self.st.channels.get(request.channel_id)
            if ch is None:
                return raft_pb.StatusResponse(success=False, message="Channel not found")
            name, member = ch["name"], p["user_id"] in ch["members"]
        if name.lower() in DEFAULT_PUBLIC:
            if member:
                return raft_pb.StatusResponse(success=True, message="Already in #general")
            err = self._propose("JOIN_CHANNEL", {"channel_id": request.channel_id, "user_id": p["user_id"]})
            if err:
                return raft_pb.StatusResponse(success=False, message=err)
            return raft_pb.StatusResponse(success=True, message=f"Joined #{name}")
        return raft_pb.StatusResponse(
            success=False,
            message=f" Cannot join #{name} directly. Ask a channel admin to add you using: "
                    f"add_user {p['username']}")

    def GetChannelMembers(self, request, context):
        if not self._verify(request.token):
            return raft_pb.ChannelMembersResponse(success=False, members=[], total_count=0)
        with self.rt.state_lock:
            ch = self.st.channels.get(request.channel_id)
            if ch is None:
                return raft_pb.ChannelMembersResponse(success=False, members=[], total_count=0)
            out = []
            for uid in ch["members"]:
                name = self.st.users_by_id.get(uid)
                u = self.st.users.get(name) if name else None
                if u is None:
                    continue
                out.append(raft_pb.ChannelMember(user_id=uid, username=name,
                                                 display_name=u.get("display_name", name),
                                                 is_admin=uid in ch.get("admins", set()),
                                                 status=u.get("status", "offline")))
        return raft_pb.ChannelMembersResponse(success=True, members=out, total_count=len(out))

    def _admin_change(self, request, add: bool):
        p = self._verify(request.token)
        if not p:
            return raft_pb.StatusResponse(success=False, message="Invalid token")
        target = request.target_username.strip()
        with self.rt.state_lock:
            ch = self.st.channels.get(request.channel_id)
            if ch is None:
                return raft_pb.StatusResponse(success=False, message="Channel not found")
            u = self.st.users.get(target)
            if u is None:
                return raft_pb.StatusResponse(success=False, message=f"User '{target}' not found")
            cname, is_member = ch["name"], u["id"] in ch["members"]
            is_admin = p["user_id"] in ch["admins"]
            n_admins = len(ch["admins"])
        if add and is_member:
            return raft_pb.StatusResponse(success=False, message=f"{target} is already a member of #{cname}")
        if not add and not is_member:
            return raft_pb.StatusResponse(success=False, message=f"{target} is not a member of #{cname}")
        if not is_admin:
            verb = "add" if add else "remove"
            return raft_pb.StatusResponse(
                success=False, message=f" Only admins of #{cname} can {verb} users. You are not an admin.")
        if not add and u["id"] == p["user_id"] and n_admins == 1:
            return raft_pb.StatusResponse(
                success=False,
                message=" Cannot remove yourself as you are the only admin. Add another admin first.")
        err = self._propose("JOIN_CHANNEL" if add else "LEAVE_CHANNEL",
                            {"channel_id": request.channel_id, "user_id": u["id"]})
        if err:
            return raft_pb.StatusResponse(success=False, message=err)
        if add:
            return raft_pb.StatusResponse(success=True, message=f" Added {target} to #{cname}")
        return raft_pb.StatusResponse(success=True, message=f" Removed {target} from #{cname}")

    def AddUserToChannel(self, request, context):
        return self._admin_change(request, True)

    def RemoveUserFromChannel(self, request, context):
        return self._admin_change(request, False)

    # ------------------------------------------------------------ messaging
    def SendMessage(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.StatusResponse(success=False, message="Invalid token")
        if not self.rt.is_leader():
            return raft_pb.StatusResponse(success=False, message="Not the leader")
        cid = request.channel_id
        with self.rt.state_lock:
            ch = self.st.channels.get(cid) if cid else None
            if ch is None:
                return raft_pb.StatusResponse(success=False, message=f"Channel not found: {cid}")
            member = p["user_id"] in ch["members"]
        if not member:  # Q8: the auto-add is replicated
            err = self._propose("JOIN_CHANNEL", {"channel_id": cid, "user_id": p["user_id"]})
            if err:
                return raft_pb.StatusResponse(success=False, message=err)
        msg = {"id": self._write_id(request, p["user_id"]), "sender_id": p["user_id"],
               "sender_name": p["username"], "channel_id": cid, "content": request.content,
               "timestamp": int(time.time() * 1000)}
        err = self._propose("SEND_MESSAGE", msg)
        if err:
            return raft_pb.StatusResponse(success=False, message=err)
        return raft_pb.StatusResponse(success=True, message="Message sent")

    # namespace of the record ids derived from (sender, request_id)
    _WRITE_NS = uuid.UUID("6f1c2d0e-9a57-4c1b-8e43-2b7d0c5a9e11")

    @classmethod
    def _write_id(cls, request, sender_id: str) -> str:
        """Record id of a write.  With a client request_id it is
        uuid5(sender_id, request_id): a retry of the same write by the same
        user maps onto the same record (the apply de-duplicates it), while two
        users that happen to pick the same request_id (counters, or an id
        copied from GetMessages) get different records.  Without one: a fresh
        uuid4 as in the reference (server/raft_node.py:1837)."""
        rid = getattr(request, "request_id", "")
        if rid and len(rid) <= 64:
            return str(uuid.uuid5(cls._WRITE_NS, f"{sender_id}:{rid}"))
        return str(uuid.uuid4())

    @staticmethod
    def _window(items, limit: int, offset: int):
        limit = limit if limit > 0 else 50
        offset = max(0, offset)
        end = len(items) - offset
        if end <= 0:
            return []
        return items[max(0, end - limit):end]

    def GetMessages(self, request, context):
        if not self._verify(request.token):
            return raft_pb.MessageListResponse(success=False, messages=[])
        with self.rt.state_lock:
            msgs = self._window(self.st.channel_messages.get(request.channel_id, []),
                                request.limit, request.offset)
            out = [raft_pb.Message(message_id=m["id"], sender_id=m["sender_id"],
                                   sender_name=m["sender_name"], channel_id=m["channel_id"],
                                   content=m["content"], timestamp=m["timestamp"]) for m in msgs]
        return raft_pb.MessageListResponse(success=True, messages=out)

    def SendDirectMessage(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.StatusResponse(success=False, message="Invalid token")
        if not self.rt.is_leader():
            return raft_pb.StatusResponse(success=False, message="Not the leader")
        with self.rt.state_lock:
            rec = self.st.users.get(request.recipient_username)
            if rec is None:
                return raft_pb.StatusResponse(success=False, message="User not found")
            rid = rec["id"]
        dm = {"id": self._write_id(request, p["user_id"]), "sender_id": p["user_id"], "sender_name": p["username"],
              "recipient_id": rid, "recipient_name": request.recipient_username,
              "content": request.content, "timestamp": int(time.time() * 1000), "is_read": False}
        err = self._propose("SEND_DM", dm)
        if err:
            return raft_pb.StatusResponse(success=False, message=err)
        return raft_pb.StatusResponse(success=True, message="DM sent")

    def GetDirectMessages(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.DirectMessageListResponse(success=False, messages=[])
        with self.rt.state_lock:
            if request.other_username not in self.st.users:
                return raft_pb.DirectMessageListResponse(success=False, messages=[])
            conv = self.st.conversation(p["username"], request.other_username)
            msgs = self._window(conv, request.limit, request.offset)
            out = [raft_pb.DirectMessage(message_id=d["id"], sender_id=d["sender_id"],
                                         sender_name=d["sender_name"], recipient_id=d["recipient_id"],
                                         recipient_name=d["recipient_name"], content=d["content"],
                                         timestamp=d["timestamp"], is_read=d["is_read"]) for d in msgs]
        return raft_pb.DirectMessageListResponse(success=True, messages=out)

    def GetOnlineUsers(self, request, context):
        if not self._verify(request.token):
            return raft_pb.UserListResponse(success=False, users=[])
        with self.rt.state_lock:
            users = [raft_pb.UserInfo(user_id=u["id"], username=n, display_name=u.get("display_name", n),
                                      email=u.get("email", ""), is_admin=u.get("is_admin", False),
                                      status=u.get("status", "offline"))
                     for n, u in self.st.users.items()]
        return raft_pb.UserListResponse(success=True, users=users)

    def ListConversations(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.ConversationsResponse(success=False, conversations=[])
        uid = p["user_id"]
        with self.rt.state_lock:
            partners, unread = {}, {}
            for d in self.st.dms_of_user(uid):
                other = d["recipient_id"] if d["sender_id"] == uid else d["sender_id"]
                partners[other] = True
                if d["recipient_id"] == uid and d["sender_id"] == other and not d.get("is_read", False):
                    unread[other] = unread.get(other, 0) + 1
            out = []
            for pid in partners:
                name = self.st.users_by_id.get(pid)
                u = self.st.users.get(name) if name else None
                if u is None:
                    continue
                out.append(raft_pb.Conversation(username=name, display_name=u.get("display_name", name),
                                                unread_count=unread.get(pid, 0)))
        return raft_pb.ConversationsResponse(success=True, conversations=out)

    # ------------------------------------------------------------ files
    def UploadFile(self, request, context):
        p = self._verify(request.token)
        if not p:
            return raft_pb.FileUploadResponse(success=False, message="Invalid token")
        if not self.rt.is_leader():
            return raft_pb.FileUploadResponse(success=False, message="Not the leader")
        fid = self._write_id(request, p["user_id"])
        mime = request.mime_type or mimetypes.guess_type(request.file_name)[0] or "application/octet-stream"
        data = {"file_id": fid, "name": request.file_name, "data": request.file_data.hex(),
                "size": len(request.file_data), "mime_type": mime, "uploader_id": p["user_id"],
                "uploader_name": p["username"], "channel_id": request.channel_id or None,
                "recipient": request.recipient_username or None, "description": request.description}
        err = self._propose("UPLOAD_FILE", data)
        if err:
            return raft_pb.FileUploadResponse(success=False, message=err)
        return raft_pb.FileUploadResponse(success=True, message="File uploaded successfully",
                                          file_id=fid, file_url=f"file://{fid}")

    def DownloadFile(self, request, context):
        if not self._verify(request.token):
            return raft_pb.FileDownloadResponse(success=False, file_name="", file_data=b"")
        with self.rt.state_lock:
            f = self.st.files.get(request.file_id)
        if f is None:
            return raft_pb.FileDownloadResponse(success=False, file_name="Not found", file_data=b"",
                                                mime_type="text/plain")
        data = f["data"]
        if isinstance(data, str):
            data = bytes.fromhex(data)
        return raft_pb.FileDownloadResponse(success=True, file_name=f["name"], file_data=data,
                                            mime_type=f["mime_type"])

    def ListFiles(self, request, context):
        if not self._verify(request.token):
            return raft_pb.FileListResponse(success=False, files=[])
        with self.rt.state_lock:
            files = [raft_pb.FileMetadata(file_id=fid, file_name=f["name"], uploader_name=f["uploader_name"],
                                          file_size=f["size"], mime_type=f["mime_type"],
                                          channel_id=request.channel_id)
                     for fid, f in self.st.files.items() if f.get("channel_id") == request.channel_id]
        return raft_pb.FileListResponse(success=True, files=files)

    # ------------------------------------------------------------ AI proxy
    def _recent(self, channel_id: str, count: int) -> list:
        with self.rt.state_lock:
            msgs = self.st.channel_messages.get(channel_id, [])
            return [llm_pb.Message(sender=m["sender_name"], content=m["content"])
                    for m in msgs[-count:]] if count > 0 else []

    def GetSmartReply(self, request, context):
        if not self._verify(request.token):
            return raft_pb.SmartReplyResponse(success=False, suggestions=[])
        recent = self._recent(request.channel_id, request.recent_message_count or 5)
        if not self.llms["smart"].available():
            return raft_pb.SmartReplyResponse(success=True, suggestions=FB_SMART_DOWN)
        try:
            t0 = time.perf_counter()
            r = self.llms["smart"].call("GetSmartReply", llm_pb.SmartReplyRequest(
                request_id=str(uuid.uuid4()), recent_messages=recent), self.cfg.llm_timeouts["smart"])
            METRICS.observe("ai.smart_reply.latency_s", time.perf_counter() - t0)
            return raft_pb.SmartReplyResponse(success=True, suggestions=list(r.suggestions))
        except Exception as e:
            log.error("LLM smart reply error: %s", e)
            return raft_pb.SmartReplyResponse(success=True, suggestions=FB_SMART_ERR)

    def SummarizeConversation(self, request, context):
        if not self._verify(request.token):
            return raft_pb.SummarizeResponse(success=False, summary="", key_points=[])
        recent = self._recent(request.channel_id, request.message_count or 20)
        if not recent:
            return raft_pb.SummarizeResponse(success=True, summary="No messages to summarize", key_points=[])
        parts = list({m.sender for m in recent})
        if not self.llms["summary"].available():
            return raft_pb.SummarizeResponse(
                success=True,
                summary=f"Conversation with {len(recent)} messages between {', '.join(parts[:3])}",
                key_points=[f"{len(recent)} messages exchanged", f"{len(parts)} participants",
                            "💡 Tip: Start LLM server for AI-powered summaries: python -m drtc_amd.llm.server"])
        try:
            r = self.llms["summary"].call("SummarizeConversation", llm_pb.SummarizeRequest(
                request_id=str(uuid.uuid4()), messages=recent, max_length=200),
                self.cfg.llm_timeouts["summary"])
            return raft_pb.SummarizeResponse(success=True, summary=r.summary, key_points=list(r.key_points))
        except Exception as e:
            log.error("LLM summarize error: %s", e)
            return raft_pb.SummarizeResponse(success=True, summary=f"Discussion between {', '.join(parts)}",
                                             key_points=[f"{len(recent)} messages", "Active conversation"])

    def GetLLMAnswer(self, request, context):
        if not self._verify(request.token):
            return raft_pb.LLMResponse(success=False, answer="Invalid token")
        if not self.llms["answer"].available():
            return raft_pb.LLMResponse(success=False, answer=LLM_DOWN_ANSWER)
        try:
            r = self.llms["answer"].call("GetLLMAnswer", llm_pb.LLMRequest(
                request_id=str(uuid.uuid4()), query=request.query, context=list(request.context)),
                self.cfg.llm_timeouts["answer"])
            return raft_pb.LLMResponse(success=True, answer=r.answer)
        except Exception as e:
            log.error("LLM answer error: %s", e)
            return raft_pb.LLMResponse(success=False, answer=f"Error: {e}")

    def GetContextSuggestions(self, request, context):
        if not self._verify(request.token):
            return raft_pb.ContextSuggestionsResponse(success=False, suggestions=[], topics=[])
        recent = self._recent(request.channel_id, request.context_message_count or 5)
        if not self.llms["suggest"].available():
            s, t = FB_SUGGEST_DOWN
            return raft_pb.ContextSuggestionsResponse(success=True, suggestions=s, topics=t)
        try:
            r = self.llms["suggest"].call("GetContextSuggestions", llm_pb.ContextRequest(
                request_id=str(uuid.uuid4()), context=recent, current_input=request.current_input),
                self.cfg.llm_timeouts["suggest"])
            return raft_pb.ContextSuggestionsResponse(success=True, suggestions=list(r.suggestions),
                                                      topics=list(r.topics))
        except Exception as e:
            log.error("Context suggestions error: %s", e)
            s, t = FB_SUGGEST_ERR
            return raft_pb.ContextSuggestionsResponse(success=True, suggestions=s, topics=t)
